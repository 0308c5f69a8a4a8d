"""Attention with a workgroup per vector row in one launch (csrc/sparse_attention_rows.hip) against the exact definition: rows at the
edges of groups, steps and waves, rows longer than the launch was made for, its probabilities, what it refuses and its default route."""
import numpy as np
import pytest
import torch

from vectorsparse_amd import _lib, ops
from vectorsparse_amd import colvec_csr as cv

pytestmark = pytest.mark.gpu

# around the groups of 16, the steps of 32 and the 64 and 128 nonzeros that a wave holds
LENGTHS = (0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 0, 200, 256, 257, 300)


def _pattern(V, lengths, n, seed, shuffled=False):
    rng = np.random.default_rng(seed)
    ro, ci = cv._pattern_from_lengths(rng, len(lengths), n, np.array(lengths, dtype=np.int64))
    if shuffled:        # any order, columns twice
        for i in range(len(lengths)):
            ci[ro[i]:ro[i + 1]] = rng.integers(0, n, ro[i + 1] - ro[i])
    return cv.ColVecCSR(len(lengths), n, V, ro, ci)


def _rows(prob, q, k, v, out, kept, scale, longest=None):
    heads, d = q.shape[0], q.shape[2]
    return ops._native.sparse_attention_rows(heads, prob.m_vec, prob.vec_length, prob.n, d, v.shape[2], prob.nnz_vec, longest or prob.longest_row_vec,
                                             prob.row_indices, prob.row_offsets, prob.column_indices, q, k, v, out, kept, float(scale), None)


def _check(pat, q, k, v, scale, out, kept, what):
    q, k, v, out = (x.double().cpu().numpy() for x in (q, k, v, out))
    ro, ci, V, d = pat.row_offsets, pat.column_indices, pat.vec_length, q.shape[2]
    for h in range(q.shape[0]):
        for i in range(pat.m_vec):
            rows, cols = slice(i * V, (i + 1) * V), ci[ro[i]:ro[i + 1]]
            if len(cols) == 0:
                assert (out[h, rows] == 0).all(), (what, h, i)
                continue
            x = q[h, rows] @ k[h, cols].T * scale
            e = np.exp(x - x.max(axis=1, keepdims=True))
            want = e / e.sum(axis=1, keepdims=True)
            # a score's sum of d exact products in fp32, and the argument of the exponential of up to 32
            off = d * 2.0 ** -23 * abs(scale) * (np.abs(q[h, rows]) @ np.abs(k[h, cols]).T).max(axis=1, keepdims=True) + 32 * 2.0 ** -23
            near = want * (np.expm1(2 * off) + 2.0 ** -17)
            if kept is not None:
                p = kept[h, ro[i]:ro[i + 1]].double().cpu().numpy().T
                assert (np.abs(p - want) <= near + want * 2.0 ** -11 + 2.0 ** -25).all(), (what, h, i)
                want, near = p, 0.0
            else:
                near = near + want * 2.0 ** -11 + 2.0 ** -25
            # products of halves are exact in fp32, each of their sums and the result's rounding are not
            exact, size = want @ v[h, cols], want @ np.abs(v[h, cols])
            bound = len(cols) * 2.0 ** -23 * size + 2.0 ** -11 * np.abs(exact) + 2.0 ** -24 + (near @ np.abs(v[h, cols]) if kept is None else 0.0)
            assert (np.abs(out[h, rows] - exact) <= bound).all(), (what, h, i)


@pytest.mark.parametrize("waves", [2, 3, 4, 5])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("V", [1, 2, 4, 8])
def test_rows_match_the_definition(gpu, V, d, waves):
    n, heads, scale = 420, 3, 0.2
    for shuffled in (False, True):
        pat = _pattern(V, LENGTHS, n, V + d, shuffled)
        prob = ops.DeviceProblem(pat, sort=shuffled)
        g = torch.Generator(device="cuda").manual_seed(d + V)
        q, k, v = (torch.randn((heads, rows, d), device="cuda", generator=g).half() for rows in (pat.m, n, n))
        gap = 64 * V
        room = torch.full((heads * (pat.nnz_vec * V + gap),), 3.0, dtype=torch.float16, device="cuda")
        kept = room.as_strided((heads, pat.nnz_vec, V), (pat.nnz_vec * V + gap, V, 1))
        for keep in (kept, None):
            pad = torch.full((heads, pat.m + 16, d), 7.0, dtype=torch.float16, device="cuda")
            with _lib.thread_options(attention_rows=waves):
                assert _rows(prob, q, k, v, pad[:, 8:-8], keep, scale) == 0
            torch.cuda.synchronize()
            assert bool((pad[:, :8] == 7.0).all()) and bool((pad[:, -8:] == 7.0).all())
            assert bool((room.as_strided((heads, gap), (pat.nnz_vec * V + gap, 1), pat.nnz_vec * V) == 3.0).all())
            _check(pat, q, k, v, scale, pad[:, 8:-8], keep, (shuffled, keep is not None))


def test_a_scale_below_zero_and_scores_beyond_fp16(gpu):
    pat = _pattern(4, (40, 200, 8), 300, 5)
    prob = ops.DeviceProblem(pat)
    q, k, v = (torch.randn((2, rows, 64), device="cuda").half() for rows in (pat.m, 300, 300))
    for scale, size in ((-0.3, 1.0), (0.0, 1.0), (2.0 ** -14, 100.0)):
        out, kept = torch.empty_like(q), torch.empty((2, pat.nnz_vec, 4), dtype=torch.float16, device="cuda")
        big = (q * size).half(), (k * size).half()
        with _lib.thread_options(attention_rows=3):
            assert _rows(prob, *big, v, out, kept, scale) == 0
        _check(pat, *big, v, scale, out, kept, scale)


def test_nan_and_infinity_stay_in_their_row(gpu):
    pat = _pattern(2, (40, 40, 40, 300, 40), 400, 3)
    prob = ops.DeviceProblem(pat)
    q, k, v = (torch.randn((2, rows, 64), device="cuda").half() for rows in (pat.m, 400, 400))
    q[0, 2, 5] = float("nan")       # scalar row 2: vector row 1
    only = int(np.setdiff1d(pat.column_indices[pat.row_offsets[3]:pat.row_offsets[4]],
                            np.delete(pat.column_indices, np.r_[pat.row_offsets[3]:pat.row_offsets[4]]))[0])
    v[1, only, 7] = float("inf")    # a column of vector row 3 alone
    for waves in (2, 3, 4, 5):
        out = torch.empty_like(q)
        with _lib.thread_options(attention_rows=waves):
            assert _rows(prob, q, k, v, out, None, 0.1) == 0
        bad = ~torch.isfinite(out)
        want = torch.zeros_like(bad)
        want[0, 2], want[1, 6:8, 7] = True, True
        assert torch.equal(bad, want)


def test_a_wave_of_nan_is_the_whole_rows(gpu):
    """A row longer than announced, with NaN wherever one of two waves looks: its probabilities are NaN at the other's nonzeros too."""
    pat = _pattern(4, (300, 40), 400, 3)
    prob = ops.DeviceProblem(pat)
    q, k, v = (torch.randn((1, rows, 64), device="cuda").half() for rows in (pat.m, 400, 400))
    k[0, torch.from_numpy(np.r_[pat.column_indices[:128], pat.column_indices[256:300]]).cuda().long()] = float("nan")
    out, kept = torch.empty_like(q), torch.empty((1, pat.nnz_vec, 4), dtype=torch.float16, device="cuda")
    with _lib.thread_options(attention_rows=3):
        assert _rows(prob, q, k, v, out, kept, 0.1, longest=40) == 0
    assert bool(torch.isnan(kept[0, :300]).all()) and bool(torch.isnan(out[0, :4]).all())


def test_the_default_route(gpu):
    """8 heads x 1024, V = 8, 96 %: the operators that keep the probabilities and the default without a caller's scores run in one
    launch, other layers and scores that a caller asked for as they did; replays of a capture give the eager bits."""
    V, heads, seq, d = 8, 8, 1024, 64
    layer = ops.SparseAttention(cv.binomial_pattern(seq // V, seq, 0.96, seed=3, vec_length=V))
    q, k, v = (torch.randn((heads, seq, d), device="cuda").half() for _ in range(3))
    kept, raw = (torch.empty((heads, layer.prob.nnz_vec, V), dtype=torch.float16, device="cuda") for _ in range(2))
    got = layer.forward(q, k, v, fused=False, scores=kept)
    out, want = torch.empty_like(got), torch.empty_like(kept)
    assert _rows(layer.prob, q, k, v, out, want, d ** -0.5) == 0
    assert torch.equal(got, out) and torch.equal(kept, want)
    assert _rows(layer.prob, q, k, v, out, None, d ** -0.5) == 0 and torch.equal(layer.forward(q, k, v, fused=True), out)
    with _lib.thread_options(attention_rows=1):
        operators = layer.forward(q, k, v, fused=False, scores=want)
        two = layer.forward(q, k, v, fused=True, scores=raw)
    assert not torch.equal(operators, got)
    again = torch.empty_like(raw)
    assert torch.equal(layer.forward(q, k, v, fused=True, scores=again), two) and torch.equal(again, raw)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        layer.forward(q, k, v, fused=False, scores=kept, out=out)
    for _ in range(3):
        out.fill_(3.0)
        kept.fill_(3.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, got)
    narrow = tuple(x[..., :32].contiguous() for x in (q, k, v))
    assert _rows(layer.prob, *narrow, torch.empty_like(narrow[0]), None, 1.0) == 801
    assert _rows(layer.prob, q, k, v, out, None, 1.0, longest=513) == 801
    assert _rows(layer.prob, q, k, v, out[:1].expand(heads, -1, -1), None, 1.0) == -1     # (problems that share outputs)


def test_outputs_in_the_place_of_inputs(gpu):
    """Other workgroups still gather k and v while one writes: an output there takes two launches, as without this kernel; in the place
    of q it is the same launch, and side by side with the inputs in one tensor too."""
    V, heads, seq, d = 8, 8, 1024, 64
    layer = ops.SparseAttention(cv.binomial_pattern(seq // V, seq, 0.96, seed=3, vec_length=V))
    q, k, v = (torch.randn((heads, seq, d), device="cuda").half() for _ in range(3))
    kept = torch.empty((heads, layer.prob.nnz_vec, V), dtype=torch.float16, device="cuda")
    one = layer.forward(q, k, v, fused=True)
    assert _rows(layer.prob, q, k, v, torch.empty_like(q), None, d ** -0.5) == 0
    with _lib.thread_options(attention_rows=1):
        two, operators = layer.forward(q, k, v, fused=True), layer.forward(q, k, v, fused=False, scores=kept)
    assert not torch.equal(one, two)
    over = k.clone()
    assert _rows(layer.prob, q, over, v, over, None, d ** -0.5) == 801
    assert torch.equal(layer.forward(q, over, v, out=over, fused=True), two)
    over = k.clone()
    assert torch.equal(layer.forward(q, over, v, out=over, fused=False, scores=kept), operators)
    over = q.clone()
    assert torch.equal(layer.forward(over, k, v, out=over, fused=True), one)
    room = torch.stack((q, k, v, torch.zeros_like(q)), dim=1)
    side = [room[:, i] for i in range(4)]
    assert _rows(layer.prob, *side, None, d ** -0.5) == 0 and torch.equal(side[3], one)
    assert _rows(layer.prob, side[0], side[1], side[2], room.reshape(heads, 4 * seq, d)[:, 3 * seq - V:4 * seq - V], None, d ** -0.5) == 801
