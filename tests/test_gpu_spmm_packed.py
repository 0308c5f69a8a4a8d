"""SpMM on rows packed two of four (csrc/spmm_pack.hip): both tile shapes at the edges of units, steps, lists and rows, against float64;
patterns the packing has to notice; infinities; workspaces, streams and captures."""
import numpy as np
import pytest
import torch

from vectorsparse_amd import _lib, ops
from vectorsparse_amd import colvec_csr as cv

pytestmark = pytest.mark.gpu


def _packed(prob, rhs, shape, nonzeros=None, out=None):
    """The two launches through the C ABI, whatever the order of the columns, on a workspace of old bytes."""
    k, nnz = rhs.shape[1], prob.nnz_vec if nonzeros is None else nonzeros
    if out is None:
        out = torch.full((prob.m_vec * prob.vec_length, k), 7.0, dtype=torch.float16, device="cuda")
    with _lib.thread_options(spmm_packed=shape):
        need = ops.spmm_packed_workspace_bytes(prob.m_vec, prob.vec_length, k, prob.n, nnz, prob.longest_row_vec)
        assert need > 0
        workspace = torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda")
        status = _lib.lib().vs_spmm_f16_packed(
            0, prob.m_vec, prob.vec_length, k, prob.n, nnz, prob.longest_row_vec, prob.row_offsets.data_ptr(), prob.column_indices.data_ptr(),
            prob.values.data_ptr(), rhs.data_ptr(), out.data_ptr(), workspace.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    assert status == 0
    return out


def _check(got, pat, B, what):
    """Products of halves are exact in fp32; each of their sums and the result's rounding are not."""
    ro, ci, values, B = pat.row_offsets, pat.column_indices, pat.values.astype(np.float64), B.astype(np.float64)
    W = np.zeros((pat.m, pat.n))
    for i in range(pat.m_vec):
        for v in range(pat.vec_length):
            np.add.at(W[i * pat.vec_length + v], ci[ro[i]:ro[i + 1]], values[ro[i]:ro[i + 1], v])
    A = np.zeros_like(W)
    for i in range(pat.m_vec):
        for v in range(pat.vec_length):
            np.add.at(A[i * pat.vec_length + v], ci[ro[i]:ro[i + 1]], np.abs(values[ro[i]:ro[i + 1], v]))
    want, size = W @ B, A @ np.abs(B)
    longest = int(np.diff(ro).max(initial=1))
    got = got.double().cpu().numpy()
    assert (np.abs(got - want) <= longest * 2.0 ** -23 * size + 2.0 ** -11 * np.abs(want) + 2.0 ** -24).all(), what


def _pattern(kind, m_vec, n, V):
    rng = np.random.default_rng(m_vec + n + V)
    if kind == "dense and empty rows":       # half of every group is listed: lists longer than LDS holds, turns beyond the kept ones
        lengths = np.where(np.arange(m_vec) % 3 == 1, 0, n)
        return cv.ColVecCSR(m_vec, n, V, *cv._pattern_from_lengths(rng, m_vec, n, lengths))
    if kind == "a nonzero":
        ro = np.zeros(m_vec + 1, dtype=np.int32)
        ro[m_vec // 2 + 1:] = 1
        return cv.ColVecCSR(m_vec, n, V, ro, np.array([n - 1], dtype=np.int32))
    if kind == "groups of every kind":       # all sixteen ways to fill a group of four, one after the other
        keep = np.array([(g >> b) & 1 for g in np.tile(np.arange(16), n // 64 + 1) for b in range(4)], dtype=bool)
        rows = [np.flatnonzero(np.roll(keep, 4 * i)[:n]).astype(np.int32) for i in range(m_vec)]
        return cv.ColVecCSR(m_vec, n, V, np.cumsum([0] + [len(r) for r in rows]).astype(np.int32), np.concatenate(rows))
    pat = cv.binomial_pattern(m_vec, n, 0.8, seed=3, vec_length=V)
    if kind == "uniform":
        return pat
    cols = pat.column_indices.copy()
    for i in range(0, m_vec, 3 if kind == "a row in three shuffled" else 1):
        beg, end = pat.row_offsets[i], pat.row_offsets[i + 1]
        if kind == "repeated columns":       # (ascending, some twice)
            cols[beg:end] = np.sort(rng.integers(0, n, end - beg))
        else:
            rng.shuffle(cols[beg:end])
    return cv.ColVecCSR(m_vec, n, V, pat.row_offsets, cols)


@pytest.mark.parametrize("shape", [2, 3])
@pytest.mark.parametrize("V", [1, 2, 4, 8])
@pytest.mark.parametrize("kind,rows,n,N", [
    ("a nonzero", 8, 1, 8), ("uniform", 256, 256, 128), ("uniform", 264, 257, 136), ("uniform", 1000, 63, 72), ("uniform", 120, 4161, 264),
    ("uniform", 136, 9000, 24), ("dense and empty rows", 144, 1030, 72), ("a nonzero", 304, 500, 64), ("groups of every kind", 128, 700, 128),
    ("repeated columns", 136, 800, 64), ("a row in three shuffled", 272, 500, 200)])
def test_packed_rows_match_float64(gpu, kind, rows, n, N, V, shape):
    pat = cv.random_values(_pattern(kind, max(1, rows // V), n, V), 5)
    B = cv.dense_uniform(n, N, seed=6)
    prob = ops.DeviceProblem(pat)
    pad = torch.full((pat.m + 32, N), 7.0, dtype=torch.float16, device="cuda")
    _packed(prob, torch.from_numpy(B).cuda(), shape, out=pad[16:16 + pat.m])
    torch.cuda.synchronize()
    assert bool((pad[:16] == 7.0).all()) and bool((pad[16 + pat.m:] == 7.0).all())
    _check(pad[16:16 + pat.m], pat, B, kind)


@pytest.mark.parametrize("V", [1, 4])
def test_a_pattern_longer_than_it_was_said_to_be(gpu, V):
    """The workspace holds the lists of the nonzeros that were announced; units whose lists do not fit go nonzero by nonzero."""
    pat = cv.random_values(_pattern("dense and empty rows", 600 // V, 520, V), 5)
    B = cv.dense_uniform(520, 136, seed=6)
    _check(_packed(ops.DeviceProblem(pat), torch.from_numpy(B).cuda(), 2, nonzeros=1), pat, B, "announced: one nonzero")


@pytest.mark.parametrize("V", [1, 2, 4, 8])
def test_a_single_pair_out_of_order_is_noticed(gpu, V):
    """At the edges of what a wave looks at in one turn, of what stays in registers, and of rows."""
    rng = np.random.default_rng(V)
    n, turn, kept = 2600, 64, (8 if V <= 2 else 4) * V * 64
    B = cv.dense_uniform(n, 40, seed=6)
    rhs = torch.from_numpy(B).cuda()
    for length in (2, 3, turn, turn + 1, kept, kept + 1, kept + turn + 1):
        for at in sorted({1, length // 2, length - 1, min(turn, length - 1), min(kept, length - 1)}):
            if not 0 < at < length or length > n - 8:
                continue
            for kind in ("repeated", "misplaced"):
                rows = [np.sort(rng.choice(np.arange(4, n), size, replace=False)) for size in (3, length, 1)]
                rows[1][at] = rows[1][at - 1] if kind == "repeated" else 1
                ro = np.cumsum([0] + [len(r) for r in rows]).astype(np.int32)
                pat = cv.random_values(cv.ColVecCSR(3, n, V, ro, np.concatenate(rows).astype(np.int32)), 5)
                _check(_packed(ops.DeviceProblem(pat), rhs, 3), pat, B, (length, at, kind))


@pytest.mark.parametrize("shape", [2, 3])
def test_infinities_and_nans_stay_where_the_nonzeros_put_them(gpu, shape):
    """Rows of rhs that hold an infinity or a NaN meet the zeros of every other row of a tile and the list's padding."""
    V, m_vec, n, N = 4, 100, 700, 136
    pat = cv.random_values(cv.binomial_pattern(m_vec, n, 0.8, seed=7, vec_length=V), 8)
    B = cv.dense_uniform(n, N, seed=9)
    B[11, 5], B[13, 70], B[350, 131], B[0, 100], B[n - 1, 0] = np.inf, np.nan, -np.inf, np.inf, 65504.0
    prob, rhs = ops.DeviceProblem(pat), torch.from_numpy(B).cuda()
    with _lib.thread_options(spmm_tile=1, spmm_packed=1):
        want = prob.spmm(rhs).cpu().numpy()
    with _lib.thread_options(spmm_packed=shape):
        got = prob.spmm(rhs).cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    assert np.isnan(want).any() and np.isinf(want).any() and np.isfinite(want).mean() > 0.9


def test_the_automatic_route(gpu):
    """2048 x 4096 x 2048, V = 1, 95 %: packed by itself with fp16 outputs, the same bits on another stream and from both kernels; other
    routes for fp32 outputs, inside a capture (eager results there too) and where the option says so."""
    pat = cv.random_values(cv.binomial_pattern(2048, 4096, 0.95, seed=3, vec_length=1), 4)
    B = torch.from_numpy(cv.dense_uniform(4096, 2048, seed=5)).cuda()
    prob = ops.DeviceProblem(pat)
    assert ops.spmm_packed_workspace_bytes(2048, 1, 2048, 4096, prob.nnz_vec, prob.longest_row_vec) > 0
    packed = prob.spmm(B)
    assert torch.equal(prob.spmm(B, kernel="cuda"), packed) and torch.equal(_packed(prob, B, 2), packed)
    with _lib.thread_options(spmm_packed=1):
        other = prob.spmm(B)
        f32 = prob.spmm(B, out_dtype=torch.float32)
    assert not torch.equal(other, packed)
    assert torch.equal(prob.spmm(B, out_dtype=torch.float32), f32)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for current, stream in ((side, None), (torch.cuda.current_stream(), side.cuda_stream)):
        out = torch.empty_like(packed)
        torch.cuda.synchronize()
        with torch.cuda.stream(current):
            prob.spmm(B, out=out, stream=stream)
        torch.cuda.synchronize()
        assert torch.equal(out, packed)
    out = torch.empty_like(packed)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        prob.spmm(B, out=out)
    for _ in range(3):
        out.fill_(3.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, other)


def test_what_the_entry_point_refuses(gpu):
    pat = cv.random_values(cv.binomial_pattern(64, 512, 0.8, seed=3, vec_length=2), 4)
    prob, lib = ops.DeviceProblem(pat), _lib.lib()
    B = torch.zeros((512, 64), dtype=torch.float16, device="cuda")
    out, stream = torch.full((128, 64), 7.0, dtype=torch.float16, device="cuda"), torch.cuda.current_stream().cuda_stream

    def call(k, workspace, size):
        return lib.vs_spmm_f16_packed(0, 64, 2, k, 512, prob.nnz_vec, prob.longest_row_vec, prob.row_offsets.data_ptr(), prob.column_indices.data_ptr(),
                                      prob.values.data_ptr(), B.data_ptr(), out.data_ptr(), workspace, size, stream)

    assert call(64, out.data_ptr(), 1 << 40) == 801          # too small to gain anything
    with _lib.thread_options(spmm_packed=2):
        need = ops.spmm_packed_workspace_bytes(64, 2, 64, 512, prob.nnz_vec, prob.longest_row_vec)
        workspace = torch.empty(need + 16, dtype=torch.uint8, device="cuda")
        assert call(60, workspace.data_ptr(), need) == 801   # k % 8
        assert call(64, 0, need) == 1 and call(64, workspace.data_ptr(), need - 1) == 1 and call(64, workspace.data_ptr() + 8, need) == 1
    torch.cuda.synchronize()
    assert bool((out == 7.0).all())


@pytest.mark.parametrize("shape", [2, 3])
def test_lists_behind_two_gigabytes(gpu, shape):
    """2^25 rows: the operands of the last units' lists lie from step 2^21 on, 2^31 bytes into the lists."""
    V, m_vec, n, dense = 8, 1 << 22, 64, 64
    ro = np.zeros(m_vec + 1, dtype=np.int32)
    ro[m_vec - dense + 1:] = n * np.arange(1, dense + 1)
    pat = cv.random_values(cv.ColVecCSR(m_vec, n, V, ro, np.tile(np.arange(n, dtype=np.int32), dense)), 5)
    B = cv.dense_uniform(n, 8, seed=6)
    got = _packed(ops.DeviceProblem(pat), torch.from_numpy(B).cuda(), shape)
    assert not bool(got[:-dense * V].any())
    last = cv.ColVecCSR(dense, n, V, n * np.arange(dense + 1, dtype=np.int32), pat.column_indices, pat.values)
    _check(got[-dense * V:], last, B, "the last rows")


@pytest.mark.parametrize("shape", [2, 3])
def test_lists_that_do_not_fit_start_nowhere(gpu, shape):
    """One nonzero announced: the units behind a row of 2^18 nonzeros would have their lists half a megabyte behind the workspace."""
    n = 1 << 18
    lengths = [3] + [0] * 15 + [n] + [0] * 15 + [5] * 32
    ro = np.cumsum([0] + lengths).astype(np.int32)
    pat = cv.random_values(cv.ColVecCSR(64, n, 1, ro, np.concatenate([np.arange(size, dtype=np.int32) for size in lengths])), 5)
    B = cv.dense_uniform(n, 8, seed=6)
    _check(_packed(ops.DeviceProblem(pat), torch.from_numpy(B).cuda(), shape, nonzeros=1), pat, B, "announced: one nonzero")


def test_uneven_rows_are_not_packed(gpu):
    """4096 x 4096 x 1024, V = 2, 90 %: Pareto rows run as if packing were off, with both kernels and both schedules."""
    rng = np.random.default_rng(3)
    lengths = np.minimum((rng.pareto(1.5, 2048) + 0.3) * 4096 * 0.1 / 1.9, 4096).astype(np.int64)
    pat = cv.random_values(cv.ColVecCSR(2048, 4096, 2, *cv._pattern_from_lengths(rng, 2048, 4096, lengths)), 4)
    prob, B = ops.DeviceProblem(pat), torch.from_numpy(cv.dense_uniform(4096, 1024, seed=5)).cuda()
    for kernel in ("wmma", "cuda"):
        for hint in (False, True):
            got = prob.spmm(B, kernel=kernel, row_length_hint=hint)
            with _lib.thread_options(spmm_packed=1):
                assert torch.equal(prob.spmm(B, kernel=kernel, row_length_hint=hint), got)
            with _lib.thread_options(spmm_packed=2):
                assert not torch.equal(prob.spmm(B, kernel=kernel, row_length_hint=hint), got)


def test_two_streams_pack_at_the_same_time(gpu):
    """Every call packs into a workspace of its stream: two problems on two streams, without a wait between them, give the bits that
    each gives alone."""
    problems = []
    for seed in (3, 4):
        pat = cv.random_values(cv.binomial_pattern(2048, 4096, 0.95, seed=seed, vec_length=1), seed)
        problems.append((ops.DeviceProblem(pat), torch.from_numpy(cv.dense_uniform(4096, 2048, seed=seed)).cuda()))
    alone = [prob.spmm(B) for prob, B in problems]
    outs = [[torch.empty_like(x) for _ in range(4)] for x in alone]
    streams = [torch.cuda.Stream() for _ in problems]
    torch.cuda.synchronize()
    for turn in range(4):
        for (prob, B), mine, stream in zip(problems, outs, streams):
            with torch.cuda.stream(stream):
                prob.spmm(B, out=mine[turn])
    torch.cuda.synchronize()
    for want, got in zip(alone, outs):
        assert all(torch.equal(want, x) for x in got)
