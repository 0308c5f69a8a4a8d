"""Split attention launches (long row blocks streamed by several workgroups): against dense masked attention in float64."""
import numpy as np
import pytest
import torch

from vectorsparse_amd import _lib, ops
from vectorsparse_amd import colvec_csr as cv
from test_gpu_attention import _check_layer, _dense_attention

pytestmark = pytest.mark.gpu


def _mask(kind, seq, V, tokens=24, half_width=40):
    start = (seq // 2 - 8) // V * V     # the tokens' rows lie in two row blocks
    rows = []
    for i in range(seq // V):
        c = i * V + V // 2
        cols = np.arange(max(0, c - half_width), min(seq, c + half_width + 1))
        if kind == "empty rows" and i % 7 == 3:
            cols = cols[:0]
        if kind != "band" and start <= i * V < start + tokens:
            cols = np.arange(seq)
        elif kind == "global":
            cols = np.union1d(cols, np.arange(start, start + tokens))
        rows.append(cols)
    ro = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    return cv.ColVecCSR(seq // V, seq, V, ro, np.concatenate(rows).astype(np.int32))


def _operands(heads, seq, d, d_v, seed=1):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn((heads, seq, w), device="cuda", generator=g).half() for w in (d, d, d_v)]


@pytest.mark.parametrize("V", [1, 2, 4, 8])
@pytest.mark.parametrize("kind,seq,d,d_v,rounds,scale", [
    ("global", 520, 64, 64, 1, None), ("global", 776, 32, 64, 2, None), ("global", 520, 128, 32, 3, None),
    ("global", 640, 64, 128, 1, -0.2), ("empty rows", 520, 64, 64, 2, None), ("empty rows", 264, 16, 24, 1, 0.0),
    ("band", 520, 64, 64, 1, None), ("global", 1032, 64, 64, 32, None)])
def test_split_launches_match_dense_attention(gpu, kind, seq, d, d_v, rounds, scale, V):
    mask = _mask(kind, seq, V)
    layer = ops.SparseAttention(mask)
    heads = 2
    q, k, v = _operands(heads, seq, d, d_v)
    pad = torch.full((heads, seq + 2, d_v), 7.0, dtype=torch.float16, device="cuda")
    out = pad[:, 1:-1]
    layer.forward(q, k, v, out=out, scale=scale, fused=("split", rounds))
    torch.cuda.synchronize()
    assert bool((pad[:, 0] == 7.0).all()) and bool((pad[:, -1] == 7.0).all())
    slots = layer._splits[d, d_v, rounds][0]
    assert (slots.n_merges > 0) == (rounds < 4 or seq > 4096)
    ref = _dense_attention(mask, q.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), d ** -0.5 if scale is None else scale)
    _check_layer(out.cpu().numpy(), ref, "%s V%d rounds %d" % (kind, V, rounds))


def test_blocks_beyond_the_plan_and_foreign_plans_take_the_per_row_path(gpu):
    V, heads, d = 8, 1, 32
    mask = _mask("global", 4352, V)     # blocks of 4352 distinct columns: more than a split plan holds
    layer = ops.SparseAttention(mask)
    q, k, v = _operands(heads, 4352, d, d)
    out = layer.forward(q, k, v, fused=("split", 4))
    ref = _dense_attention(mask, q.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), d ** -0.5)
    _check_layer(out.cpu().numpy(), ref, "beyond the plan")
    mask = _mask("global", 520, V)
    layer = ops.SparseAttention(mask)
    q, k, v = _operands(heads, 520, d, d)
    slots, device_slots, plan = layer._split(d, d, 1)
    out = torch.empty_like(q)
    ops.sparse_attention_split(layer.prob, slots, device_slots, torch.zeros_like(plan), q, k, v, out, d ** -0.5)
    ref = _dense_attention(mask, q.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), d ** -0.5)
    _check_layer(out.cpu().numpy(), ref, "a plan of zeros")


def test_the_automatic_route_splits_and_replays(gpu):
    V, heads, seq, d = 1, 4, 1500, 64
    mask = _mask("global", seq, V, tokens=64)
    layer = ops.SparseAttention(mask)
    q, k, v = _operands(heads, seq, d, d)
    fresh = ops.SparseAttention(mask)
    route = layer._route(d, d, heads)
    assert route[0] == "split"
    assert torch.equal(layer.forward(q, k, v), layer.forward(q, k, v, fused=route))
    want = layer.forward(q, k, v)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    other = layer.forward(q, k, v, stream=side)
    side.synchronize()
    assert torch.equal(other, want)
    out = torch.empty_like(want)
    fresh.plan(d, d, heads)     # (makes what the route needs: the first pass can be captured)
    for one in (layer, fresh):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            one.forward(q, k, v, out=out)
        for _ in range(3):
            out.fill_(3.0)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)


def test_refused_arguments(gpu):
    mask = _mask("global", 520, 8)
    layer = ops.SparseAttention(mask)
    q, k, v = _operands(2, 520, 64, 64)
    slots, device_slots, plan = layer._split(64, 64, 1)
    out = torch.empty_like(q)
    whole = torch.empty(slots.n_partials * 2 * 128 * 66, dtype=torch.float32, device="cuda")
    for bad_plan, workspace in ((plan[:-16], None), (plan, whole[:-1])):
        with pytest.raises(_lib.VSparseError, match=r"vs_sparse_attention_f16_split.*invalid"):
            ops.sparse_attention_split(layer.prob, slots, device_slots, bad_plan, q, k, v, out, 0.125, workspace)
    # (the same call with all of the plan and exactly the room it needs)
    ops.sparse_attention_split(layer.prob, slots, device_slots, plan, q, k, v, out, 0.125, whole)
    assert torch.equal(out, layer.forward(q, k, v, scale=0.125, fused=("split", 1)))
    with pytest.raises(TypeError):
        ops.sparse_attention_split(layer.prob, slots, device_slots, plan, q.float(), k, v, out, 0.125)


def _layer_in_float64(mask, q, k, v, scale):
    """Softmax attention over each row's own columns alone (a repeated column counts as often as it is listed)."""
    out = np.zeros((q.shape[0], mask.m, v.shape[2]))
    q, k, v = (x.double().cpu().numpy() for x in (q, k, v))
    V, ro = mask.vec_length, mask.row_offsets
    with np.errstate(invalid="ignore"):
        for h in range(q.shape[0]):
            for i in range(mask.m_vec):
                cols = mask.column_indices[ro[i]:ro[i + 1]]
                if len(cols):
                    s = (q[h, i * V:(i + 1) * V] @ k[h, cols].T) * scale
                    p = np.exp(s - s.max(axis=1, keepdims=True))
                    out[h, i * V:(i + 1) * V] = (p / p.sum(axis=1, keepdims=True)) @ v[h, cols]
    return out


def test_slots_that_start_behind_the_plan_are_left_to_the_first_one(gpu):
    """Parts of a block of more columns than a plan lists, as a caller of the C entry point may dispatch them: the first takes
    the per-row path for all of the block, the others read nothing behind its record.  Blocks of 8192 columns, parts that
    start at sub-rounds 0, 4 .. 60; the last block is among them."""
    V, seq, d = 8, 8192, 32
    rows = [np.arange(max(0, i * V - 20), min(seq, i * V + 28)) for i in range(seq // V)]
    rows[3] = rows[-2] = np.arange(seq)
    mask = cv.ColVecCSR(seq // V, seq, V, np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32),
                        np.concatenate(rows).astype(np.int32))
    layer = ops.SparseAttention(mask)
    q, k, v = _operands(1, seq, d, d)
    unions = layer._block_unions()
    assert unions[0] == unions[-1] == seq and sorted(unions)[-3] < 512
    listed = ops.AttentionSlots(unions, 4)
    assert listed.n_partials == listed.n_merges == 0
    cut = ops.AttentionSlots(unions, 4)
    cut.slots = np.array([(block, start, start + 4, i * 16 + start // 4) for i, block in enumerate((0, len(unions) - 1)) for start in range(0, 64, 4)]
                         + [slot for slot in listed.slots.tolist() if slot[0] not in (0, len(unions) - 1)]
                         + [(0, 0, 16, 0), (len(unions) - 1, 16, 16, 0)], dtype=np.int32)
    cut.n_slots, cut.n_merges, cut.n_partials = len(cut.slots) - 2, 2, 32
    plan = layer._split(d, d, 4)[2]
    ref = _layer_in_float64(mask, q, k, v, d ** -0.5)
    for slots in (listed, cut):
        out = torch.full_like(q, 7.0)
        ops.sparse_attention_split(layer.prob, slots, torch.from_numpy(slots.slots).cuda(), plan, q, k, v, out, d ** -0.5)
        _check_layer(out.double().cpu().numpy(), ref, "%d partial tiles" % slots.n_partials)


@pytest.mark.parametrize("V", [1, 2, 4, 8])
@pytest.mark.parametrize("route,d,d_v,scale", [
    (("split", 1), 64, 64, None), (("split", 2), 32, 24, -0.2), (("split", 32), 64, 64, None), (("split", 1), 128, 64, 0.0),
    (("split", 2), 64, 128, None), ("layer", 64, 64, None), ("layer", 128, 128, -0.2), (None, 64, 64, None)])
def test_infinities_and_nans_reach_the_rows_that_attend_to_them_alone(gpu, route, d, d_v, scale, V):
    seq, heads, tokens = 776, 2, 24
    mask = _mask("global", seq, V, tokens=tokens)
    start = (seq // 2 - 8) // V * V     # (the tokens, see _mask)
    lonely, ro, ci = 40 // V, mask.row_offsets, mask.column_indices
    cols = [ci[ro[i]:ro[i + 1]] for i in range(mask.m_vec)]
    cols[lonely] = np.array([300], dtype=np.int32)      # a row whose only score is -infinity below
    mask = cv.ColVecCSR(mask.m_vec, seq, V, np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32), np.concatenate(cols))
    q, k, v = _operands(heads, seq, d, d_v)
    q[:, :, 0] = q[:, :, 0].abs() + 0.1
    sign = -1.0 if scale is not None and scale < 0 else 1.0
    k[0, 100, 0] = sign * np.inf
    k[0, 150, 1] = -np.inf
    k[0, 200, 2] = np.nan
    k[0, 300] = 0.0
    k[0, 300, 0] = -sign * np.inf
    v[0, 500, 3] = np.inf
    v[0, 600, d_v - 1] = np.nan
    v[1, 640, 0] = -np.inf
    touched = [100, 150, 200, 300, 500, 600, 640]
    assert not set(touched) & set(range(start, start + tokens))     # (else every row attends to them)
    if route == "layer":
        layer = ops.SparseAttention(mask)
        out = torch.empty((heads, seq, d_v), dtype=torch.float16, device="cuda")
        plan = ops.sparse_attention_plan(mask.m_vec, V, seq, d, d_v, 128 // V, layer.prob.row_offsets, layer.prob.column_indices)
        ops.sparse_attention(mask.m_vec, V, seq, layer.prob.row_indices, layer.prob.row_offsets, layer.prob.column_indices, q, k, v,
                             out=out, scale=scale, rows_per_workgroup=128 // V, plan=plan)
    else:
        out = ops.SparseAttention(mask).forward(q, k, v, scale=scale, fused=route)
    got = out.double().cpu().numpy()
    ref = _layer_in_float64(mask, q, k, v, d ** -0.5 if scale is None else scale)
    finite = np.isfinite(ref)
    assert np.isnan(ref[0, lonely * V:(lonely + 1) * V]).all() and 0.3 < finite.mean() < 1.0
    # (a probability that rounds to zero in fp16 makes a NaN of an infinite product, in every route)
    assert np.array_equal(np.isfinite(got), finite)
    _check_layer(np.where(finite, got, 0.0), np.where(finite, ref, 0.0), "non-finite K and V, V%d %s" % (V, route))


@pytest.mark.parametrize("V", [1, 8])
def test_the_default_counts_a_repeated_column_as_often_as_it_is_listed(gpu, V):
    """(the union of a block's columns holds it once)"""
    heads, seq, d = 4, 1500 // V * V, 64
    mask = _mask("global", seq, V, tokens=64)
    assert ops.SparseAttention(mask)._route(d, d, heads)[0] == "split"
    ro, ci = mask.row_offsets, mask.column_indices.copy()
    ci[ro[:-1] + 2] = ci[ro[:-1] + 1]
    mask = cv.ColVecCSR(mask.m_vec, seq, V, ro, ci)
    q, k, v = _operands(heads, seq, d, d)
    out = ops.SparseAttention(mask).forward(q, k, v)
    _check_layer(out.double().cpu().numpy(), _layer_in_float64(mask, q, k, v, d ** -0.5), "repeated columns V%d" % V)


def test_the_default_leaves_the_probabilities_in_a_callers_buffer(gpu):
    """Masks with global tokens: the default on row parts leaves them there, and a buffer asks for it."""
    V, heads, seq, d = 1, 4, 1500, 64
    mask = _mask("global", seq, V, tokens=64)
    layer = ops.SparseAttention(mask)
    q, k, v = _operands(heads, seq, d, d)
    assert layer._route(d, d, heads)[0] == "split"
    scores = torch.full((heads, mask.nnz_vec, V), 7.0, dtype=torch.float16, device="cuda")
    out = layer.forward(q, k, v, scores=scores)
    want = torch.empty_like(scores)
    assert torch.equal(out, layer.forward(q, k, v, scores=want, fused="parts"))
    assert torch.equal(scores, want)
    sums = scores.double().cpu().numpy()[0, :, 0]
    sums = np.add.reduceat(sums, mask.row_offsets[:-1])
    assert (np.abs(sums - 1.0) < 2.0 ** -11 * 4).all()


def test_a_first_pass_inside_a_capture_takes_what_needs_no_preparation(gpu):
    """A layer that has served another head count, captured at one whose split launch was never planned: the plan cannot be
    made there, the routes that need none can be captured.  The next eager pass makes it."""
    V, seq, d = 4, 776, 64
    layer = ops.SparseAttention(_mask("global", seq, V))
    assert layer._route(d, d, 4) is True and layer._route(d, d, 8) == ("split", 2)
    layer.forward(*_operands(4, seq, d, d))
    q, k, v = _operands(8, seq, d, d)
    out, scores = torch.empty_like(q), torch.empty((8, layer.prob.nnz_vec, V), dtype=torch.float16, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        layer.forward(q, k, v, out=out)
    assert not layer._splits
    want = layer.forward(q, k, v, scores=scores, fused=True)
    for _ in range(3):
        out.fill_(3.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    split = layer.forward(q, k, v)
    assert torch.equal(split, layer.forward(q, k, v, fused=("split", 2))) and not torch.equal(split, want)


def test_partial_tiles_lie_in_memory_of_the_stream_that_uses_them(gpu):
    """A pass on one stream gives its partial tiles back while it still runs; a pass on another stream that is not ordered
    behind it must not get the same memory."""
    V, heads, seq, d = 8, 2, 776, 64
    layer = ops.SparseAttention(_mask("global", seq, V))
    q, k, v = _operands(heads, seq, d, d)
    want = layer.forward(q, k, v, fused=("split", 1))
    torch.cuda.synchronize()
    side, handed = torch.cuda.Stream(), []
    empty = torch.empty

    def watched(*args, **kwargs):
        t = empty(*args, **kwargs)
        if t.dtype == torch.float32:
            handed.append((torch.cuda.current_stream().cuda_stream, t.data_ptr()))
        return t

    out = [torch.zeros_like(want) for _ in range(9)]
    torch.empty = watched
    try:
        for i, one in enumerate(out):
            layer.forward(q, k, v, out=one, fused=("split", 1), stream=(None, side, side.cuda_stream)[i % 3])
    finally:
        torch.empty = empty
    torch.cuda.synchronize()
    assert all(torch.equal(one, want) for one in out)
    here, there = torch.cuda.current_stream().cuda_stream, side.cuda_stream
    assert [stream for stream, _ in handed] == [here, there, there] * 3
    assert not {p for s, p in handed if s == here} & {p for s, p in handed if s == there}
