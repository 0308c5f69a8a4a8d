"""The compiled route of the operators (csrc/binding.cpp) against the route through the checks of ops.py: the same results
for strided, shared and contiguous operands and every way to name a stream, the same refusals."""
import numpy as np
import pytest
import torch

from vectorsparse_amd import ops
from vectorsparse_amd import colvec_csr as cv

pytestmark = pytest.mark.gpu

V, HEADS, SEQ, D = 4, 3, 192, 64


class _Unusual:
    """In the binding's place: nothing is ordinary, every call goes through ops.py."""

    def __getattr__(self, name):
        return lambda *args: -1


@pytest.fixture(params=["compiled", "checked"])
def route(request, monkeypatch):
    if request.param == "checked":
        monkeypatch.setattr(ops, "_native", _Unusual())
    return request.param


def _problem():
    rng = np.random.default_rng(1)
    lengths = rng.integers(0, 60, SEQ // V)
    lengths[5] = 190
    ro, ci = cv._pattern_from_lengths(rng, SEQ // V, SEQ, lengths)
    return ops.DeviceProblem(cv.ColVecCSR(SEQ // V, SEQ, V, ro, ci))


def _calls(prob):
    """name -> (operands by name, the written one last; call(operands, stream))"""
    idx = (prob.row_indices, prob.row_offsets, prob.column_indices)
    parts, slots = prob.row_parts(64)[:2]
    spmm_ws = torch.zeros(ops.spmm_row_parts_workspace_bytes(V, D, parts.n_split, parts.parts_max, batch=HEADS), dtype=torch.uint8, device="cuda")
    soft_ws = torch.zeros(ops.sparse_softmax_row_parts_workspace_bytes(V, parts.n_split, parts.parts_max, batch=HEADS), dtype=torch.uint8, device="cuda")
    nnz, m = prob.nnz_vec, SEQ // V
    scores, dense = (nnz, V), (SEQ, D)
    return {
        "spmm_batched": ((scores, dense, dense), lambda a, s: ops.spmm_batched(m, V, D, SEQ, *idx, *a, stream=s)),
        "spmm_batched cuda": ((scores, dense, dense), lambda a, s: ops.spmm_batched(m, V, D, SEQ, *idx, *a, kernel="cuda", stream=s)),
        "spmm_softmax_batched": ((scores, dense, dense), lambda a, s: ops.spmm_softmax_batched(m, V, D, SEQ, *idx, *a, scale=0.125, stream=s)),
        "sddmm_batched": ((dense, dense, scores), lambda a, s: ops.sddmm_batched(m, D, SEQ, nnz, *idx, *a, V, stream=s)),
        "sddmm_batched cuda": ((dense, dense, scores), lambda a, s: ops.sddmm_batched(m, D, SEQ, nnz, *idx, *a, V, kernel="cuda", stream=s)),
        "sparse_softmax": ((scores, scores), lambda a, s: ops.sparse_softmax(m, V, *idx[:2], *a, scale=0.125, stream=s)),
        "sparse_attention": ((dense, dense, dense, dense), lambda a, s: ops.sparse_attention(m, V, SEQ, *idx, *a, stream=s)),
        "spmm_row_parts": ((scores, dense, dense), lambda a, s: ops.spmm_row_parts(V, D, SEQ, parts, slots, nnz, idx[2], *a, spmm_ws, s)),
        "sddmm_row_parts": ((dense, dense, scores), lambda a, s: ops.sddmm_row_parts(D, SEQ, parts, slots, nnz, idx[2], *a, V, s)),
        "softmax_row_parts": ((scores, scores), lambda a, s: ops.sparse_softmax_row_parts(V, parts, slots, *a, 0.125, soft_ws, s)),
    }


NAMES = ("spmm_batched", "spmm_batched cuda", "spmm_softmax_batched", "sddmm_batched", "sddmm_batched cuda", "sparse_softmax",
         "sparse_attention", "spmm_row_parts", "sddmm_row_parts", "softmax_row_parts")


def _tensors(shapes, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    made = [torch.randn((HEADS,) + s, device="cuda", generator=g).half() for s in shapes]
    made[-1].fill_(7.0)
    return made


def _spread(t):
    """The same problems with 256 elements between them (the last one ends with its buffer)."""
    each = t[0].numel()
    room = torch.full((HEADS * (each + 256) - 256,), 3.0, dtype=t.dtype, device=t.device)
    out = room.as_strided(t.shape, (each + 256, t.shape[2], 1))
    out.copy_(t)
    return room, out


@pytest.mark.parametrize("name", NAMES)
def test_strided_shared_and_contiguous_operands(gpu, name, route):
    shapes, call = _calls(_problem())[name]
    operands = _tensors(shapes, 2)
    want = operands[-1]
    call(operands, None)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for stream in (None, side, side.cuda_stream):
        out = torch.full_like(want, 7.0)
        torch.cuda.synchronize()
        call(operands[:-1] + [out], stream)
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    spread = [_spread(t) for t in operands[:-1] + [torch.full_like(want, 7.0)]]
    call([t for _, t in spread], None)
    torch.cuda.synchronize()
    assert torch.equal(spread[-1][1], want)
    each = want[0].numel()
    for h in range(HEADS - 1):
        assert bool((spread[-1][0][h * (each + 256) + each:(h + 1) * (each + 256)] == 3.0).all())
    if "softmax" not in name or name == "spmm_softmax_batched":     # the first problem's inputs shared by all of them
        out = torch.full_like(want, 7.0)
        call([t if name == "sparse_attention" else t[0] for t in (u[:1].expand(HEADS, -1, -1) for u in operands[:-1])] + [out], None)
        expanded = torch.full_like(want, 7.0)
        call([t[:1].expand(HEADS, -1, -1) for t in operands[:-1]] + [expanded], None)
        torch.cuda.synchronize()
        for h in range(HEADS):
            assert torch.equal(out[h], want[0]) and torch.equal(expanded[h], want[0])


@pytest.mark.parametrize("name", NAMES)
def test_refused_layouts_types_and_places(gpu, name, route):
    shapes, call = _calls(_problem())[name]
    operands = _tensors(shapes, 3)
    last = operands[-1]
    for i, t in enumerate(operands):
        wide = torch.zeros(t.shape[:2] + (2 * t.shape[2],), dtype=t.dtype, device="cuda")
        for bad in (wide[..., :t.shape[2]], t.transpose(1, 2).contiguous().transpose(1, 2), t.cpu()):
            with pytest.raises(ValueError):
                call(operands[:i] + [bad] + operands[i + 1:], None)
        with pytest.raises(TypeError):
            call(operands[:i] + [t.float()] + operands[i + 1:], None)
    torch.cuda.synchronize()
    assert bool((last == 7.0).all())


@pytest.mark.parametrize("name", ["spmm_row_parts", "sddmm_row_parts", "softmax_row_parts"])
def test_problems_that_overlap_are_not_written(gpu, name, route):
    shapes, call = _calls(_problem())[name]
    operands = _tensors(shapes, 4)
    one = torch.full((HEADS,) + shapes[-1], 7.0, dtype=torch.float16, device="cuda")
    each = one[0].numel()
    flat = one.view(-1)
    for stride in (0, V, each - 8):
        with pytest.raises(ValueError):
            call(operands[:-1] + [flat.as_strided(one.shape, (stride, one.shape[2], 1))], None)
    if name == "softmax_row_parts":     # in place
        with pytest.raises(ValueError):
            call([flat.as_strided(one.shape, (0, one.shape[2], 1)), None], None)
    torch.cuda.synchronize()
    assert bool((one == 7.0).all())
