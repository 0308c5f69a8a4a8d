"""Softmax in place and SpMM in one launch (vs_wmma_softmax_spmm_f16_batched) against the exact definition and the two launches."""
import numpy as np
import pytest
import torch

from vectorsparse_amd import _lib, ops
from vectorsparse_amd import colvec_csr as cv

pytestmark = pytest.mark.gpu

# around the steps of 32 and 64, the 256 scores a wave holds and the 512 up to which one launch is the default
LENGTHS = (0, 1, 31, 32, 33, 64, 65, 127, 200, 0, 255, 256, 257, 511, 512, 17)
N = 640


def _pattern(V, lengths, seed):
    lengths = np.array(lengths, dtype=np.int64)
    ro, ci = cv._pattern_from_lengths(np.random.default_rng(seed), len(lengths), N, lengths)
    return cv.random_values(cv.ColVecCSR(len(lengths), N, V, ro, ci), seed=seed)


@pytest.mark.parametrize("steps", (0, 2))
@pytest.mark.parametrize("k, heads, longer", ((64, 3, ()), (128, 40, ()), (100, 1, ()), (4, 2, (513, 600)), (64, 1, (640,)), (7, 2, ()), (192, 2, ())))
@pytest.mark.parametrize("V", (1, 2, 4, 8))
def test_one_launch(gpu, V, k, heads, longer, steps):
    pat = _pattern(V, LENGTHS + longer, 7 + V)
    prob = ops.DeviceProblem(pat, sort=True)
    nnz, scale = pat.nnz_vec, 0.3
    g = torch.Generator(device="cuda").manual_seed(k)
    gap = 64 * V
    room = torch.full((heads * (nnz * V + gap),), 3.0, dtype=torch.float16, device="cuda")
    values = room.as_strided((heads, nnz, V), (nnz * V + gap, V, 1))
    scores = (torch.randn((heads, nnz, V), device="cuda", generator=g) * 4).half()
    scores[:, 5::11] = float("-inf")    # masked: probability 0, unless the row holds nothing else
    ro = pat.row_offsets
    scores[:, ro[1]] = 0.5              # (the row of a single vector)
    rhs = torch.randn((heads, N, k), device="cuda", generator=g).half()

    def run(route):
        values.copy_(scores)
        out = torch.full((heads, pat.m, k), 7.0, dtype=torch.float16, device="cuda")
        with _lib.thread_options(softmax_spmm=route, spmm_steps=steps):
            ops.softmax_spmm_batched(pat.m_vec, V, k, N, prob.row_indices, prob.row_offsets, prob.column_indices, values, rhs, out,
                                     scale, nonzeros_vec=nnz, longest_row_vec=prob.longest_row_vec)
        torch.cuda.synchronize()
        assert bool((room.as_strided((heads, gap), (nnz * V + gap, 1), nnz * V) == 3.0).all())
        return values.double().cpu().numpy(), out.double().cpu().numpy()

    x, w = scores.double().cpu().numpy() * scale, rhs.double().cpu().numpy()
    for route in (1, 2, 0):
        p, out = run(route)
        for h in range(heads):
            for i in range(pat.m_vec):
                lo, hi = ro[i], ro[i + 1]
                if lo == hi:
                    assert (out[h, i * V:(i + 1) * V] == 0).all()
                    continue
                e = np.exp(x[h, lo:hi] - x[h, lo:hi].max(axis=0, keepdims=True))
                want = e / e.sum(axis=0, keepdims=True)
                # rounded once to fp16 (2^-11, below the normal range 2^-25), and fp32 arithmetic: an argument of up to 32 with an
                # error of 2^-23 of itself, exp2, sum and product a few 2^-23 more
                assert (np.abs(p[h, lo:hi] - want) <= want * (2.0 ** -11 + 2.0 ** -17) + 2.0 ** -25).all(), (route, h, i)
                rows = w[h][pat.column_indices[lo:hi]]
                got, exact = out[h, i * V:(i + 1) * V], p[h, lo:hi].T @ rows
                # products of halves are exact in fp32, each of their sums and the result's rounding are not
                bound = (hi - lo) * 2.0 ** -23 * (p[h, lo:hi].T @ np.abs(rows)) + 2.0 ** -11 * np.abs(exact) + 2.0 ** -24
                assert (np.abs(got - exact) <= bound).all(), (route, h, i)


def test_nan_and_infinity_stay_in_their_row(gpu):
    V, k, heads = 2, 64, 2
    pat = _pattern(V, (40, 40, 40, 300, 40), 3)
    prob = ops.DeviceProblem(pat)
    ro = pat.row_offsets
    scores = torch.randn((heads, pat.nnz_vec, V), device="cuda").half()
    scores[0, ro[1] + 3, 0] = float("nan")
    scores[0, ro[2] + 3, 1] = float("inf")
    scores[1, ro[3]:ro[4], 0] = float("-inf")
    rhs = torch.randn((heads, N, k), device="cuda").half()
    results = []
    for route in (1, 2):
        values, out = scores.clone(), torch.empty((heads, pat.m, k), dtype=torch.float16, device="cuda")
        with _lib.thread_options(softmax_spmm=route):
            ops.softmax_spmm_batched(pat.m_vec, V, k, N, prob.row_indices, prob.row_offsets, prob.column_indices, values, rhs, out,
                                     0.5, nonzeros_vec=pat.nnz_vec, longest_row_vec=prob.longest_row_vec)
        torch.cuda.synchronize()
        results.append((values, out))
    for one, two in zip(*results):
        assert torch.equal(one.isnan(), two.isnan()) and torch.equal(one.isinf(), two.isinf())
    nan = results[0][1].isnan().all(dim=2).cpu()
    assert nan.sum() == 3 and nan[0, 2] and nan[0, 5] and nan[1, 6]


def test_capture_and_replay(gpu):
    V, heads, k = 4, 2, 64
    pat = _pattern(V, LENGTHS, 9)
    prob = ops.DeviceProblem(pat, sort=True)
    scores = torch.randn((heads, pat.nnz_vec, V), device="cuda").half()
    rhs = torch.randn((heads, N, k), device="cuda").half()
    values, out = scores.clone(), torch.empty((heads, pat.m, k), dtype=torch.float16, device="cuda")

    def call():
        values.copy_(scores)
        ops.softmax_spmm_batched(pat.m_vec, V, k, N, prob.row_indices, prob.row_offsets, prob.column_indices, values, rhs, out, 0.5,
                                 nonzeros_vec=pat.nnz_vec, longest_row_vec=prob.longest_row_vec)

    call()
    torch.cuda.synchronize()
    want = values.clone(), out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for _ in range(3):
        values.fill_(9.0), out.fill_(9.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(values, want[0]) and torch.equal(out, want[1])


def test_problems_that_share_values_are_refused(gpu):
    """(they are replaced in place: several problems would normalise the same scores)"""
    V, heads, k = 4, 3, 64
    pat = _pattern(V, LENGTHS, 9)
    prob = ops.DeviceProblem(pat, sort=True)
    scores = torch.randn((heads, pat.nnz_vec, V), device="cuda").half()
    rhs, out = torch.randn((heads, N, k), device="cuda").half(), torch.empty((heads, pat.m, k), dtype=torch.float16, device="cuda")

    def call(values, out=out):
        return ops.softmax_spmm_batched(pat.m_vec, V, k, N, prob.row_indices, prob.row_offsets, prob.column_indices, values, rhs[:out.shape[0]],
                                        out, 0.5, nonzeros_vec=pat.nnz_vec, longest_row_vec=prob.longest_row_vec)

    kept = scores.clone()
    overlapping = scores.view(-1).as_strided((heads, pat.nnz_vec, V), (8 * V, V, 1))
    for values in (scores[0], scores[:1], scores[:2], scores[:1].expand(heads, -1, -1), overlapping):
        with pytest.raises(ValueError, match="values of its own"):
            call(values)
    torch.cuda.synchronize()
    assert torch.equal(scores, kept)
    one = call(scores[0], out=out[:1]).clone()      # (a single problem may be two-dimensional)
    scores.copy_(kept)
    assert torch.equal(call(scores)[:1], one)
