"""SDDMM on dense tiles (csrc/sddmm_tile.hip): both tile sizes at the edges of tiles, rows, columns and contraction
steps, against the C oracle, and bit for bit against the gathering MFMA kernel (same products in the same order),
whatever the order of a row's columns."""
import numpy as np
import pytest
import torch

from oracle import c_oracle as co
from vectorsparse_amd import _lib, ops
from vectorsparse_amd import colvec_csr as cv
from util import assert_parity

pytestmark = pytest.mark.gpu


def _shuffled(pat, seed):
    rng = np.random.default_rng(seed)
    cols = pat.column_indices.copy()
    for i in range(pat.m_vec):
        rng.shuffle(cols[pat.row_offsets[i]:pat.row_offsets[i + 1]])
    return cv.ColVecCSR(pat.m_vec, pat.n, pat.vec_length, pat.row_offsets, cols)


def _pattern(kind, m_vec, n, V):
    rng = np.random.default_rng(m_vec + n + V)
    if kind == "shuffled columns":
        return _shuffled(cv.binomial_pattern(m_vec, n, 0.6, seed=3, vec_length=V), 4)
    if kind == "repeated columns":   # more nonzeros of one column than a tile has columns
        lengths = np.where(np.arange(m_vec) % 3 == 0, 300, 5)
        ro = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
        return cv.ColVecCSR(m_vec, n, V, ro, np.sort(rng.integers(0, 3, ro[-1])).astype(np.int32))
    if kind == "dense and empty rows":
        lengths = np.where(np.arange(m_vec) % 2 == 0, n, 0)
        ro, ci = cv._pattern_from_lengths(rng, m_vec, n, lengths)
        return cv.ColVecCSR(m_vec, n, V, ro, ci)
    if kind == "clustered columns":  # far from uniform: the search's first probes are all off; most tiles are empty
        rows = [np.sort(rng.choice(np.r_[0:17, n - 9:n], 20, replace=False)) for _ in range(m_vec)]
        ro = (np.arange(m_vec + 1) * 20).astype(np.int32)
        return cv.ColVecCSR(m_vec, n, V, ro, np.concatenate(rows).astype(np.int32))
    return cv.binomial_pattern(m_vec, n, 0.7, seed=5, vec_length=V)


@pytest.mark.parametrize("tile", [2, 3])
@pytest.mark.parametrize("V", [1, 2, 4, 8])
@pytest.mark.parametrize("kind,rows,n,K", [
    ("uniform", 1, 1, 8), ("uniform", 64, 64, 64), ("uniform", 128, 128, 128), ("uniform", 136, 129, 72),
    ("uniform", 56, 63, 320), ("uniform", 1048, 300, 40), ("clustered columns", 200, 900, 136),
    ("dense and empty rows", 72, 200, 264), ("shuffled columns", 96, 200, 96), ("shuffled columns", 136, 1500, 264),
    ("repeated columns", 48, 65, 64)])
def test_dense_tiles_match_the_oracle_and_the_gathering_kernel(gpu, kind, rows, n, K, V, tile):
    m_vec = max(1, rows // V)
    pat = _pattern(kind, m_vec, n, V)
    A, B = cv.dense_normal(pat.m, K, seed=6), cv.dense_normal(n, K, seed=7)
    prob = ops.DeviceProblem(pat)
    Ad, Bd = torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()
    ref = co.sddmm_host_ref_f32(pat.m_vec, K, V, pat.row_offsets, pat.column_indices, A, B)
    for dtype in (torch.float16, torch.float32):
        pad = torch.full((pat.nnz_vec + 32, V), 7.0, dtype=dtype, device="cuda")
        got = pad[16:16 + pat.nnz_vec]
        with _lib.thread_options(sddmm_tile=tile):
            prob.sddmm(Ad, Bd, out=got, algorithm=1)
        with _lib.thread_options(sddmm_tile=1):
            gathered = prob.sddmm(Ad, Bd, out_dtype=dtype, algorithm=1)
        torch.cuda.synchronize()
        assert bool((pad[:16] == 7.0).all()) and bool((pad[16 + pat.nnz_vec:] == 7.0).all())
        assert_parity(got.cpu().numpy().reshape(-1), ref, "%s %s" % (kind, dtype))
        # Shuffled columns: a nonzero is then written by several tiles (CPU model of the search over 40 rows of 820 of 4096
        # columns: two in three lie between the bounds of several tiles, 6 % of them of their own and of another one).
        assert torch.equal(got, gathered)


def test_dense_tiles_batched(gpu):
    V, heads, n, K = 2, 3, 190, 72
    mask = cv.binomial_pattern(75, n, 0.6, seed=8, vec_length=V)
    prob = ops.DeviceProblem(mask)
    g = torch.Generator(device="cuda").manual_seed(1)
    A = torch.randn((heads, mask.m, K), device="cuda", generator=g).half()
    B = torch.randn((heads, n, K), device="cuda", generator=g).half()
    out = torch.empty((heads, mask.nnz_vec, V), dtype=torch.float16, device="cuda")
    for tile in (2, 3):
        with _lib.thread_options(sddmm_tile=tile):
            ops.sddmm_batched(mask.m_vec, K, n, mask.nnz_vec, prob.row_indices, prob.row_offsets, prob.column_indices, A, B,
                              out, V)
        with _lib.thread_options(sddmm_tile=1):
            one = [prob.sddmm(A[h], B[h], algorithm=1) for h in range(heads)]
        torch.cuda.synchronize()
        for h in range(heads):
            assert torch.equal(out[h], one[h]), "head %d" % h


@pytest.mark.parametrize("kernel", ["wmma", "cuda"])
def test_the_automatic_route_takes_tiles_only_where_columns_ascend(gpu, kernel):
    """A mask dense enough for tiles (V = 1, 512 x 1024 at 50 %, K = 256; gathering it takes the fine-grained kernel, whose
    fp32 bits are not those of the matrix cores): ascending columns known to the caller run on tiles, the same columns
    without that word, or shuffled ones, are gathered, and a wrong word changes no bit.  At 98 % gathering is expected to be
    faster whatever the order."""
    mask = cv.binomial_pattern(512, 1024, 0.5, seed=9, vec_length=1)
    A = torch.from_numpy(cv.dense_normal(mask.m, 256, seed=10)).cuda()
    B = torch.from_numpy(cv.dense_normal(mask.n, 256, seed=11)).cuda()
    for pat in (mask, _shuffled(mask, 12)):
        prob = ops.DeviceProblem(pat)
        assert prob.columns_sorted == (pat is mask)
        with _lib.thread_options(sddmm_tile=1):
            gathered = prob.sddmm(A, B, kernel=kernel, out_dtype=torch.float32)
            matrix_cores = prob.sddmm(A, B, out_dtype=torch.float32, algorithm=1)
        assert not torch.equal(gathered, matrix_cores)
        assert torch.equal(prob.sddmm(A, B, kernel=kernel, out_dtype=torch.float32), matrix_cores if pat is mask else gathered)
        out = torch.empty_like(gathered)
        args = (prob.m_vec, 256, prob.n, prob.nnz_vec, prob.row_indices, prob.row_offsets, prob.column_indices, A, B, out, 1)
        call, extra = (ops.sddmm.wmmaSddmm, dict(algorithm=0)) if kernel == "wmma" else (ops.sddmm.cudaSddmm, {})
        assert torch.equal(call(*args, **extra), gathered)
        # (the compiled binding, then the checks of ops.py, which take the stream as an object)
        for stream in (None, torch.cuda.current_stream()):
            assert torch.equal(call(*args, stream=stream, columns_sorted=True, **extra), matrix_cores)
        one = torch.empty((1, prob.nnz_vec, 1), dtype=torch.float16, device="cuda")
        args = args[:7] + (A[None], B[None], one, 1)
        for stream in (None, torch.cuda.current_stream()):
            ops.sddmm_batched(*args, kernel=kernel, stream=stream, columns_sorted=True, **extra)
            assert torch.equal(one[0], matrix_cores.half())
        torch.cuda.synchronize()
    sparse = cv.binomial_pattern(512, 1024, 0.98, seed=9, vec_length=1)
    prob = ops.DeviceProblem(sparse)
    assert prob.columns_sorted
    with _lib.thread_options(sddmm_tile=1):
        gathered = prob.sddmm(A, B, kernel=kernel, out_dtype=torch.float32)
    with _lib.thread_options(sddmm_tile=2):
        tiles = prob.sddmm(A, B, kernel=kernel, out_dtype=torch.float32)
    assert torch.equal(prob.sddmm(A, B, kernel=kernel, out_dtype=torch.float32), gathered) and not torch.equal(gathered, tiles)
