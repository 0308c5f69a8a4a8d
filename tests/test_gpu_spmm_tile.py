"""SpMM on dense tiles (csrc/spmm_tile.hip): every shape at the edges of tiles, chunks, windows and rows against the C
oracle, whatever the order of a row's columns, and against the gathering kernel where a dense product would differ (zeros
times infinities)."""
import numpy as np
import pytest
import torch

from oracle import c_oracle as co
from vectorsparse_amd import _lib, ops
from vectorsparse_amd import colvec_csr as cv
from util import assert_parity

pytestmark = pytest.mark.gpu


def _pattern(kind, m_vec, n, V):
    rng = np.random.default_rng(m_vec + n + V)
    if kind == "dense and empty rows":      # more nonzeros of a row in a chunk than its windows hold
        lengths = np.where(np.arange(m_vec) % 2 == 0, n, 0)
        return cv.ColVecCSR(m_vec, n, V, *cv._pattern_from_lengths(rng, m_vec, n, lengths))
    if kind == "one row":
        lengths = np.where(np.arange(m_vec) == m_vec // 2, max(1, n // 2), 0)
        return cv.ColVecCSR(m_vec, n, V, *cv._pattern_from_lengths(rng, m_vec, n, lengths))
    if kind == "clustered columns":         # chunks without a nonzero
        rows = [np.sort(rng.choice(np.r_[0:17, n - 9:n], 20, replace=False)) for _ in range(m_vec)]
        return cv.ColVecCSR(m_vec, n, V, (np.arange(m_vec + 1) * 20).astype(np.int32), np.concatenate(rows).astype(np.int32))
    if kind == "a nonzero":
        ro = np.zeros(m_vec + 1, dtype=np.int32)
        ro[m_vec // 2 + 1:] = 1
        return cv.ColVecCSR(m_vec, n, V, ro, np.array([n - 1], dtype=np.int32))
    pat = cv.binomial_pattern(m_vec, n, 0.6, seed=3, vec_length=V)
    if kind == "uniform":
        return pat
    cols = pat.column_indices.copy()
    for i in range(0, m_vec, 3 if kind == "a row in three shuffled" else 1):
        beg, end = pat.row_offsets[i], pat.row_offsets[i + 1]
        if kind == "repeated columns":      # (ascending, some twice)
            cols[beg:end] = np.sort(rng.integers(0, n, end - beg))
        else:
            rng.shuffle(cols[beg:end])
    return cv.ColVecCSR(m_vec, n, V, pat.row_offsets, cols)


@pytest.mark.parametrize("tile", [2, 3, 4])
@pytest.mark.parametrize("V", [1, 2, 4, 8])
@pytest.mark.parametrize("kind,rows,n,N", [
    ("uniform", 1, 1, 4), ("uniform", 128, 256, 128), ("uniform", 136, 257, 132), ("uniform", 24, 767, 60),
    ("uniform", 296, 769, 64), ("uniform", 120, 1601, 260), ("dense and empty rows", 144, 1600, 68), ("one row", 64, 3000, 64),
    ("clustered columns", 200, 2500, 136), ("a nonzero", 64, 400, 64), ("shuffled columns", 96, 900, 96),
    ("a row in three shuffled", 136, 500, 132), ("repeated columns", 136, 800, 64)])
def test_dense_tiles_match_the_oracle(gpu, kind, rows, n, N, V, tile):
    m_vec = max(1, rows // V)
    pat = cv.random_values(_pattern(kind, m_vec, n, V), 5)
    B = cv.dense_uniform(n, N, seed=6)
    prob = ops.DeviceProblem(pat)
    assert prob.columns_distinct == (kind not in ("shuffled columns", "a row in three shuffled", "repeated columns"))
    ref = co.spmm_host_ref_f32(pat.m_vec, V, N, n, pat.row_offsets, pat.column_indices, pat.values, B)
    pad = torch.full((pat.m + 32, N), 7.0, dtype=torch.float16, device="cuda")
    for kernel in ("wmma", "cuda"):
        with _lib.thread_options(spmm_tile=tile):
            prob.spmm(torch.from_numpy(B).cuda(), kernel=kernel, out=pad[16:16 + pat.m])
        torch.cuda.synchronize()
        assert bool((pad[:16] == 7.0).all()) and bool((pad[16 + pat.m:] == 7.0).all())
        assert_parity(pad[16:16 + pat.m].cpu().numpy(), ref.reshape(pat.m, N), "%s %s" % (kind, kernel))


@pytest.mark.parametrize("tile", [2, 3, 4])
def test_infinities_and_nans_stay_where_the_nonzeros_put_them(gpu, tile):
    """Rows of rhs that hold an infinity or a NaN meet the zeros of every other row of a tile."""
    V, m_vec, n, N = 4, 50, 700, 132
    pat = cv.random_values(cv.binomial_pattern(m_vec, n, 0.9, seed=7, vec_length=V), 8)
    B = cv.dense_uniform(n, N, seed=9)
    B[11, 5], B[13, 70], B[690, 131], B[n - 1, 0] = np.inf, np.nan, -np.inf, 65504.0
    prob = ops.DeviceProblem(pat)
    rhs = torch.from_numpy(B).cuda()
    with _lib.thread_options(spmm_tile=1):
        want = prob.spmm(rhs).cpu().numpy()
    with _lib.thread_options(spmm_tile=tile):
        got = prob.spmm(rhs).cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    assert np.isnan(want).any() and np.isinf(want).any() and np.isfinite(want).mean() > 0.9
    both = np.isfinite(want)
    assert_parity(got[both], want[both], "finite outputs")


def test_dense_tiles_batched(gpu):
    V, heads, n, N = 2, 3, 190, 72
    pat = cv.random_values(cv.binomial_pattern(75, n, 0.6, seed=8, vec_length=V), 9)
    prob = ops.DeviceProblem(pat)
    g = torch.Generator(device="cuda").manual_seed(1)
    values = torch.randn((heads, pat.nnz_vec, V), device="cuda", generator=g).half()
    B = torch.randn((heads, n, N), device="cuda", generator=g).half()
    out = torch.empty((heads, pat.m, N), dtype=torch.float16, device="cuda")
    for tile in (2, 3, 4):
        with _lib.thread_options(spmm_tile=tile):
            ops.spmm_batched(pat.m_vec, V, N, n, prob.row_indices, prob.row_offsets, prob.column_indices, values, B, out)
        for h in range(heads):
            ref = co.spmm_host_ref_f32(pat.m_vec, V, N, n, pat.row_offsets, pat.column_indices, values[h].cpu().numpy(), B[h].cpu().numpy())
            assert_parity(out[h].cpu().numpy(), ref.reshape(pat.m, N), "head %d" % h)


def test_the_automatic_route_and_its_replays(gpu):
    """V = 1, 1024 x 1024 at 50 %, 512 columns: tiles by themselves where the columns ascend strictly and outputs are fp16,
    gathered else; captured launches give the eager bits."""
    pat = cv.random_values(cv.binomial_pattern(1024, 1024, 0.5, seed=3, vec_length=1), 4)
    B = torch.from_numpy(cv.dense_uniform(1024, 512, seed=5)).cuda()
    prob = ops.DeviceProblem(pat)
    gathered, tiles = {}, {}
    for kernel in ("wmma", "cuda"):
        with _lib.thread_options(spmm_tile=1):
            gathered[kernel] = prob.spmm(B, kernel=kernel)
        tiles[kernel] = prob.spmm(B, kernel=kernel)
        assert torch.equal(prob.spmm(B, kernel=kernel, row_length_hint=True), tiles[kernel])
        with _lib.thread_options(spmm_tile=1):
            f32 = prob.spmm(B, kernel=kernel, out_dtype=torch.float32)
        assert torch.equal(prob.spmm(B, kernel=kernel, out_dtype=torch.float32), f32)
    assert torch.equal(tiles["wmma"], tiles["cuda"])
    assert not torch.equal(tiles["wmma"], gathered["wmma"]) and not torch.equal(tiles["cuda"], gathered["cuda"])
    raw = torch.empty_like(gathered["wmma"])
    ops.spmm.wmmaSpmm(prob.m_vec, 1, 512, 1024, prob.row_indices, prob.row_offsets, prob.column_indices, prob.values, B, raw)
    assert torch.equal(raw, gathered["wmma"])
    swapped = pat.column_indices.copy()
    swapped[:2] = swapped[1::-1]
    other = ops.DeviceProblem(cv.ColVecCSR(1024, 1024, 1, pat.row_offsets, swapped, pat.values))
    with _lib.thread_options(spmm_tile=1):
        want = other.spmm(B)
    assert torch.equal(other.spmm(B), want)
    out = torch.empty_like(tiles["wmma"])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        prob.spmm(B, out=out)
    for _ in range(3):
        out.fill_(3.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, tiles["wmma"])


def _ascending_but_for(V, n, rows, row, at, kind, tight, rng):
    """Rows of ascending columns (next to each other, or anywhere) with the given numbers of nonzeros, but for one pair:
    nonzero `at` of row `row` repeats its predecessor's column, or lies in front of all of the row's others."""
    cols = []
    for i, length in enumerate(rows):
        c = np.arange(4, 4 + length) if tight else np.sort(rng.choice(np.arange(4, n), length, replace=False))
        if i == row:
            c[at] = c[at - 1] if kind == "repeated" else 1
        cols.append(c)
    ro = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
    return cv.random_values(cv.ColVecCSR(len(rows), n, V, ro, np.concatenate(cols).astype(np.int32)), 5)


@pytest.mark.parametrize("tile", [2, 3, 4])
@pytest.mark.parametrize("V", [1, 2, 4, 8])
def test_a_single_pair_out_of_order_is_noticed(gpu, V, tile):
    """One repeated or misplaced column in a pattern that ascends otherwise, at the edges of what a lane fetches, of windows
    and of the pattern's end: nothing else makes a workgroup go nonzero by nonzero."""
    threads, tile_rows, each = 256, 32 << (tile - 2), {2: (8, 8, 4, 4), 3: (8, 8, 4, 4), 4: (8, 4, 4, 2)}[tile][V.bit_length() - 1]
    window = min(64, threads * V // tile_rows) * each
    rng = np.random.default_rng(10 * V + tile)
    n, N, missed = 1700, 32, []
    B = cv.dense_uniform(n, N, seed=6)
    rhs, exact = torch.from_numpy(B).cuda(), B.astype(np.float64)
    lengths = sorted({*range(2, 2 * each + 2), window - 1, window, window + 1, window + each + 1, 2 * window, 2 * window + 1, 3 * window + 2})
    for length in lengths:
        places = {1, length // 2, length - 1, length - 2, (length - 1) // each * each, window, 2 * window}
        for at in sorted(p for p in places if 0 < p < length):
            # the last row, or a row of one nonzero behind it
            for kind, tight, behind in ((k, t, b) for k in ("repeated", "misplaced") for t in (True, False) for b in ((), (1,))):
                rows = (3, length) + behind
                pat = _ascending_but_for(V, n, rows, 1, at, kind, tight, rng)
                prob = ops.DeviceProblem(pat)
                assert not prob.columns_distinct
                with _lib.thread_options(spmm_tile=tile):
                    got = prob.spmm(rhs).double().cpu().numpy()
                ro, ci = pat.row_offsets, pat.column_indices
                values = pat.values.astype(np.float64)
                want = np.concatenate([values[ro[i]:ro[i + 1]].T @ exact[ci[ro[i]:ro[i + 1]]] for i in range(pat.m_vec)])
                size = np.concatenate([np.abs(values[ro[i]:ro[i + 1]].T) @ np.abs(exact[ci[ro[i]:ro[i + 1]]]) for i in range(pat.m_vec)])
                # products of halves are exact in fp32; each of their sums and the result's rounding are not
                if not (np.abs(got - want) <= length * 2.0 ** -23 * size + 2.0 ** -11 * np.abs(want) + 2.0 ** -24).all():
                    missed.append((rows, at, kind, tight))
    assert not missed, (len(missed), missed[:8])
