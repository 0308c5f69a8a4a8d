// SDDMM on dense tiles (V = 1, 2, 4, 8): out[j*V + v] = sum_l lhs[(i*V + v)*K + l] * rhs[col_j*K + l].
//
// The gathering kernels (sddmm_mfma.hip, sddmm_valu.hip) fetch one row of rhs from the L2s for every nonzero vector:
// V multiply-adds per two bytes gathered.  Where a mask keeps a good share of a tile - short vectors, low sparsity -
// it is cheaper to multiply the whole tile of lhs * rhs^T on the matrix cores, both operands read once per tile, and to
// keep only the masked outputs.  A workgroup owns TM scalar rows x TN columns:
//   1. the nonzeros of its rows that fall in its columns: a search for both column bounds in every row (a quad of
//      lanes per bound, sixteen entries per probe, the first probe where uniform columns would put the bound); the
//      4 V lanes of a vector row then fetch the column indices of their nonzeros ahead of
//   2. the product: K in steps of 64 through LDS, v_mfma_f32_16x16x32_f16 in ascending k - the same products in the
//      same order as the gathering MFMA kernel, hence the same bits,
//   3. the tile, converted, to LDS; every lane picks its nonzeros' outputs there and writes them out.
// Columns need not be sorted: the bound of (row, column) depends on nothing else, the first bound of a row is its
// first nonzero and the last one its end, so every nonzero lies between the two bounds of at least one tile whatever
// the order - of several, where the bounds of the row do not ascend.  A nonzero found in a tile that does not hold its
// column is multiplied there by itself, to the same bits, so that it does not matter which of its tiles writes it last.
// (Slow: with shuffled columns two nonzeros in three lie in several tiles; 4096 x 4096, V = 1, K = 256, 80 %:
// 1130 us against 19 us sorted and 87 us gathered.)
//
// What bounds it (4096 x 4096, V = 1, K = 256, 80 %, tiles of 128: 18.9 us): nothing alone - vector ALU 8 us, LDS 6 us, matrix
// cores 3 us, 225 MB through the L2s 10 us, around a tile's chain of dependent loads (row extent, two probes, columns) of
// about 3 us that two workgroups of eight waves per CU hide from each other.  A flat list of the tile's nonzeros over all
// threads instead of 4 V lanes per vector row (a scan and an owner per nonzero in LDS) took 34 us, one step of operands in
// flight instead of two 22.5 us.
#include <cmath>
#include <type_traits>

#include "vs_common.hpp"

namespace vs {

namespace {

constexpr int kTileK = 64;  // contraction elements per step: 128 bytes of every row

// OR over the four lanes of a quad.
__device__ __forceinline__ uint32_t quad_or(uint32_t x)
{
    x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xF, 0xF, true);
    x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xF, 0xF, true);
    return x;
}

// The search for the first of columns[beg, end) that is not below x, sixteen entries at a time (four per lane of a
// quad): `window` places a probe, `narrow` reads it.
struct BoundSearch {
    int beg, end, lo, hi, x, w;
    bool done;

    __device__ __forceinline__ void start(int row_beg, int row_end, int column, bool first, bool last)
    {
        beg = lo = row_beg;
        end = hi = row_end;
        x = column;
        if (first) hi = lo;
        if (last) lo = hi;
        done = lo >= hi;
    }
    __device__ __forceinline__ void window(int guess)
    {
        guess = guess < lo ? lo : (guess > hi ? hi : guess);
        const int top = end - 16 > beg ? end - 16 : beg;
        w = guess - 8 < beg ? beg : (guess - 8 > top ? top : guess - 8);
    }
    __device__ __forceinline__ int4_t probe(const int *columns, int q) const
    {
        if (end - beg >= 16) return *reinterpret_cast<const int4_a4 *>(columns + w + 4 * q);
        int4_t e;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int at = w + 4 * q + i;
            e[i] = columns[at < end ? at : end - 1];
        }
        return e;
    }
    // Sets lo = hi = the bound when the probe holds it, else narrows [lo, hi] and returns the next guess.
    __device__ __forceinline__ int narrow(const int4_t &e, int q, float per_column, int round)
    {
        uint32_t bits = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int at = w + 4 * q + i;
            if (at >= lo && at < hi && e[i] >= x) bits |= 1u << (4 * q + i);
        }
        bits = quad_or(bits);
        const int first = __builtin_amdgcn_update_dpp(0, e[0], 0x00, 0xF, 0xF, true);  // quad_perm [0,0,0,0]
        const int last = __builtin_amdgcn_update_dpp(0, e[3], 0xFF, 0xF, 0xF, true);   // quad_perm [3,3,3,3]
        const int from = w > lo ? w : lo, to = w + 16 < hi ? w + 16 : hi;
        int guess;
        if (bits == 0) {
            lo = to;
            guess = lo + (int)fminf((float)(x - last) * per_column, (float)(hi - lo));
        } else {
            const int at = w + __builtin_ctz(bits);
            if (at > from || from == lo) {
                lo = hi = at;
                guess = at;
            } else {
                hi = from;
                guess = hi - (int)fminf((float)(first - x) * per_column, (float)(hi - lo));
            }
        }
        done = lo >= hi;
        return round < 2 ? guess : (lo + hi) >> 1;  // columns far from uniform: halves
    }
};

// 16-byte piece p of row r of an operand in LDS, in halves.  Rows are 128 bytes, half of the banks' width: sixteen lanes
// that read one piece of sixteen consecutive rows then touch every bank once.  (Rows sixteen apart: a constant apart.)
__device__ __forceinline__ int operand_place(int r, int p) { return r * kTileK + 8 * (p ^ ((r >> 1) & 7)); }

// DEEP: K > 64 - two steps of operands on their way in registers, two in LDS (one barrier per step); else one step.
template <int V, int TM, int TN, bool DEEP, typename OutT>
__global__ void __launch_bounds__(4 * TM, DEEP ? 4 : 6)
sddmm_tile_kernel(int m_vec, int K, int n, int row_blocks, int column_tiles, const int *__restrict__ row_offsets,
                  const int *__restrict__ col_indices, const half_t *__restrict__ lhs, const half_t *__restrict__ rhs,
                  OutT *__restrict__ out, long long stride_lhs, long long stride_rhs, long long stride_out)
{
    constexpr int THREADS = 4 * TM, WAVES = THREADS / 64;
    constexpr int ROWS = TM / V;                        // vector rows, 4 V lanes each
    constexpr int LPR = 4 * V;
    constexpr int PITCH = TN + (V == 1 ? 4 : 0);         // columns of the tile in LDS (V = 1: rows on shifted banks)
    constexpr int WN = WAVES / 2;                       // waves: two blocks of rows x WN blocks of columns
    constexpr int MI = TM / 32, NJ = TN / (16 * WN);     // 16 x 16 tiles of a wave
    constexpr int AR = TM * 8 / THREADS, BR = TN * 8 / THREADS;  // 16-byte pieces of a thread per k step
    constexpr int STEP = (TM + TN) * kTileK * 2, OPERANDS = (DEEP ? 2 : 1) * STEP, RESULT = ROWS * PITCH * V * (int)sizeof(OutT);
    constexpr int BOUNDS = V == 1 ? 2 : 1;              // bounds a quad looks for
    constexpr int EACH = V == 1 ? 4 : 1;                // consecutive nonzeros of a lane
    constexpr int AHEAD = V == 1 ? 3 : (V == 2 ? 4 : (V == 4 ? 3 : 2));  // (groups of) nonzeros a lane fetches ahead
    __shared__ __align__(32) unsigned char area[OPERANDS > RESULT ? OPERANDS : RESULT];
    __shared__ int any[WAVES];

    // Row blocks are dealt to the XCDs (consecutive workgroups go to consecutive XCDs), each of which takes a row
    // block's column tiles one after the other: its L2 sees its own rows of lhs and the output lines that
    // neighbouring tiles share, and rhs once.
    int rb, ct;
    if (row_blocks >= 8) {
        const int i = blockIdx.x >> 3;
        rb = (int)(blockIdx.x & 7) + 8 * (i / column_tiles);
        ct = i % column_tiles;
        if (rb >= row_blocks) return;
    } else {
        rb = blockIdx.x / column_tiles;
        ct = blockIdx.x % column_tiles;
    }
    if (blockIdx.y != 0) {
        lhs += blockIdx.y * stride_lhs;
        rhs += blockIdx.y * stride_rhs;
        out += blockIdx.y * stride_out;
    }
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c0 = ct * TN;
    const int m = m_vec * V;

    // this lane's vector row, and its place among the row's lanes
    const int row_here = tid / LPR, row = rb * ROWS + row_here, li = tid % LPR;
    int row_beg = 0, row_end = 0;
    if (row < m_vec) {
        row_beg = row_offsets[row];
        row_end = row_offsets[row + 1];
    }

    // the operands' pieces of the first step are on their way during the search
    const int piece = tid & 7, piece_row = tid >> 3;
    struct Pieces {
        uint4_t a[AR], b[BR];
    };
    Pieces ahead[DEEP ? 2 : 1];
    // a thread's rows as byte offsets from the tile's first row of each operand; rows past the end repeat the last one,
    // their results are dropped
    unsigned a_row[AR], b_row[BR];
#pragma unroll
    for (int i = 0; i < AR; ++i) {
        const int r = piece_row + THREADS / 8 * i, end = m - rb * TM;
        a_row[i] = (unsigned)(r < end ? r : end - 1) * (unsigned)K * 2;
    }
#pragma unroll
    for (int i = 0; i < BR; ++i) {
        const int r = piece_row + THREADS / 8 * i, end = n - c0;
        b_row[i] = (unsigned)(r < end ? r : end - 1) * (unsigned)K * 2;
    }
    const char *const a_base = reinterpret_cast<const char *>(lhs + (size_t)rb * TM * K);
    const char *const b_base = reinterpret_cast<const char *>(rhs + (size_t)c0 * K);
    // (K % 8 == 0: a piece is whole or absent; absent ones re-read the step's first and become zeros on their way to LDS)
    auto fetch = [&](Pieces &to, int k0) {
        const unsigned at = k0 + 8 * piece < K ? 16 * piece : 0;
        const size_t from = k0 < K ? 2 * (size_t)k0 : 0;
#pragma unroll
        for (int i = 0; i < AR; ++i) to.a[i] = *reinterpret_cast<const uint4_t *>(a_base + from + (a_row[i] + at));
#pragma unroll
        for (int i = 0; i < BR; ++i) to.b[i] = *reinterpret_cast<const uint4_t *>(b_base + from + (b_row[i] + at));
    };
    fetch(ahead[0], 0);
    if constexpr (DEEP) fetch(ahead[1], kTileK);

    // [beg, end): the row's nonzeros in this tile's columns
    int beg, end;
    {
        const int q = tid & 3;
        const float per_column = (float)(row_end - row_beg) / (float)n;
        BoundSearch search[BOUNDS];
        int4_t e[BOUNDS];
#pragma unroll
        for (int p = 0; p < BOUNDS; ++p) {
            const int x = c0 + (V == 1 ? p : (tid >> 2) & 1) * TN;   // V > 1: the row's quads take turns
            search[p].start(row_beg, row_end, x, x == 0, x >= n);
            search[p].window(row_beg + (int)((float)x * per_column));
            if (!search[p].done) e[p] = search[p].probe(col_indices, q);
        }
#pragma unroll
        for (int p = 0; p < BOUNDS; ++p)
            for (int round = 0; !search[p].done; ++round) {
                const int guess = search[p].narrow(e[p], q, per_column, round);
                if (search[p].done) break;
                search[p].window(guess);
                e[p] = search[p].probe(col_indices, q);
            }
        if constexpr (V == 1) {
            beg = search[0].lo;
            end = search[1].lo;
        } else {
            const int mine = search[0].lo;
            const int other = __builtin_amdgcn_update_dpp(0, mine, 0x141, 0xF, 0xF, true);  // row_half_mirror: the other quad of eight lanes
            beg = tid & 4 ? other : mine;
            end = tid & 4 ? mine : other;
        }
    }

    // columns of this lane's nonzeros, AHEAD x EACH at a time
    int col[AHEAD][EACH];
    auto fetch_columns = [&](int base) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int j = base + EACH * (li + LPR * u);
            if constexpr (V == 1) {
                if (j < end) {
                    if (j + 4 <= row_end) {
                        const int4_t x = *reinterpret_cast<const int4_a4 *>(col_indices + j);
#pragma unroll
                        for (int i = 0; i < EACH; ++i) col[u][i] = x[i];
                    } else {
#pragma unroll
                        for (int i = 0; i < EACH; ++i) col[u][i] = col_indices[j + i < row_end ? j + i : row_end - 1];
                    }
                }
            } else {
                if (j < end) col[u][0] = col_indices[j];
            }
        }
    };
    fetch_columns(beg);
    const uint64_t some = __builtin_amdgcn_ballot_w64(beg < end);
    if (lane == 0) any[wave] = some != 0;
    __syncthreads();
    {   // a tile without a nonzero (bands, blocks) is left here
        int total = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) total |= any[w];
        if (__builtin_amdgcn_readfirstlane(total) == 0) return;
    }

    const int c = lane & 15, g = lane >> 4;
    const int wm = (wave / WN) * (TM / 2), wn = (wave % WN) * (TN / WN);
    float4_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    const int put = operand_place(piece_row, piece), take[2] = {operand_place(c, g), operand_place(c, 4 + g)};
    // One step: its pieces to LDS, the pieces two steps on requested (MORE), the products.  Whether something is
    // requested is part of the code and not a branch: a wait after a branch would count for the path without requests.
    auto step = [&](auto more, Pieces &mine, int buffer, int k0) {
        constexpr bool MORE = decltype(more)::value;
        half_t *const la = reinterpret_cast<half_t *>(area + buffer * STEP);
        half_t *const lb = la + TM * kTileK;
        const bool whole = MORE || k0 + 8 * piece < K;
        const uint4_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < AR; ++i)
            *reinterpret_cast<uint4_t *>(la + put + THREADS / 8 * i * kTileK) = whole ? mine.a[i] : zero;
#pragma unroll
        for (int i = 0; i < BR; ++i)
            *reinterpret_cast<uint4_t *>(lb + put + THREADS / 8 * i * kTileK) = whole ? mine.b[i] : zero;
        if constexpr (MORE) fetch(mine, k0 + 2 * kTileK);
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            half8_t a[MI], b[NJ];
#pragma unroll
            for (int i = 0; i < MI; ++i) a[i] = *reinterpret_cast<const half8_t *>(la + take[kk] + (wm + 16 * i) * kTileK);
#pragma unroll
            for (int j = 0; j < NJ; ++j) b[j] = *reinterpret_cast<const half8_t *>(lb + take[kk] + (wn + 16 * j) * kTileK);
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    // V = 1: transposed, so that a lane holds four columns of one row (one LDS write below)
                    if constexpr (V == 1) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[j], a[i], acc[i][j], 0, 0, 0);
                    else acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b[j], acc[i][j], 0, 0, 0);
                }
        }
    };
    constexpr std::true_type more;
    constexpr std::false_type last;
    if constexpr (DEEP) {
        // two steps per turn (an odd number of steps ends in one of zeros)
        int k0 = 0;
        for (; k0 + 2 * kTileK < K; k0 += 2 * kTileK) {
            step(more, ahead[0], 0, k0);
            step(more, ahead[1], 1, k0 + kTileK);
        }
        step(last, ahead[0], 0, k0);
        step(last, ahead[1], 1, k0 + kTileK);
    } else {
        step(last, ahead[0], 0, 0);
    }
    __syncthreads();
    OutT *const tile = reinterpret_cast<OutT *>(area);  // [vector row][column][v]
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const float x[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
            if constexpr (V == 1) {
                store_converted<OutT, 4>(tile + (wm + 16 * i + c) * PITCH + wn + 16 * j + 4 * g, x);
            } else {
                const int r = wm + 16 * i + 4 * g, column = wn + 16 * j + c;
                if constexpr (V == 2) {
                    store_converted<OutT, 2>(tile + ((r / 2) * PITCH + column) * 2, x);
                    store_converted<OutT, 2>(tile + ((r / 2 + 1) * PITCH + column) * 2, x + 2);
                } else {
                    store_converted<OutT, 4>(tile + ((r / V) * PITCH + column) * V + r % V, x);
                }
            }
        }
    __syncthreads();

    struct __align__(sizeof(OutT) * V) Vec {
        OutT x[V];
    };
    const OutT *const tile_row = tile + row_here * PITCH * V;
    bool elsewhere = false;   // a nonzero between the bounds whose column the tile does not hold
    for (int base = beg; base < end;) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int j = base + EACH * (li + LPR * u);
            if constexpr (V == 1) {
                unsigned at[4];
                bool all = j + 4 <= end;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    at[i] = (unsigned)(col[u][i] - c0);
                    all = all && at[i] < (unsigned)TN;
                }
                if (all) {
                    OutT x[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[i] = tile_row[at[i]];
                    __builtin_memcpy(out + j, x, sizeof(x));   // (aligned as one output is)
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (j + i < end) {
                            if (at[i] < (unsigned)TN) out[j + i] = tile_row[at[i]];
                            else elsewhere = true;
                        }
                }
            } else if (j < end) {
                const unsigned at = (unsigned)(col[u][0] - c0);
                if (at < (unsigned)TN) *reinterpret_cast<Vec *>(out + (size_t)j * V) = *reinterpret_cast<const Vec *>(tile_row + at * V);
                else elsewhere = true;
            }
        }
        base += EACH * LPR * AHEAD;
        if (base < end) fetch_columns(base);
    }

    // Rows of unsorted columns: the wave multiplies such nonzeros 16 / V at a time, each with its own rows of both operands
    // (the results wanted are the product's diagonal), on the matrix cores and in the same steps of 32 as the tiles.  Such
    // a nonzero can lie between the bounds of several tiles, its own among them; whichever of them writes it last, it
    // writes the same bits.
    if (__builtin_amdgcn_ballot_w64(elsewhere) == 0) return;
    constexpr int AT_ONCE = 16 / V;
    for (int j = beg + li; __builtin_amdgcn_ballot_w64(j < end) != 0; j += LPR) {
        const int column = j < end ? col_indices[j] : c0;
        const bool mine = (unsigned)(column - c0) >= (unsigned)TN;
        const uint64_t some_lanes = __builtin_amdgcn_ballot_w64(mine);
        const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(some_lanes >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)some_lanes, 0));
        for (int first = 0, left = __builtin_popcountll(some_lanes); left > 0; first += AT_ONCE, left -= AT_ONCE) {
            // lane i < AT_ONCE gets nonzero `first + i` (the last lane takes what is not wanted)
            const int to = 4 * (mine && rank >= first && rank < first + AT_ONCE ? rank - first : 63);
            const int rows = __builtin_amdgcn_ds_permute(to, row), columns = __builtin_amdgcn_ds_permute(to, column);
            const int places = __builtin_amdgcn_ds_permute(to, j);
            const int its_row = __builtin_amdgcn_ds_bpermute(4 * (c / V), rows), its_column = __builtin_amdgcn_ds_bpermute(4 * c, columns);
            const int its_place = __builtin_amdgcn_ds_bpermute(4 * c, places);
            const half_t *const a = lhs + ((size_t)(c / V < left ? its_row : rb * ROWS) * V + c % V) * K;
            const half_t *const b = rhs + (size_t)(c < AT_ONCE && c < left ? its_column : c0) * K;
            float4_t sum = {0.f, 0.f, 0.f, 0.f};
            for (int k0 = 0; k0 < K; k0 += 32) {
                const bool there = k0 + 8 * g < K;
                const int at = there ? k0 + 8 * g : 0;
                const uint4_t x = *reinterpret_cast<const uint4_t *>(a + at), y = *reinterpret_cast<const uint4_t *>(b + at);
                const uint4_t zero = {0u, 0u, 0u, 0u};
                const uint4_t xs = there ? x : zero, ys = there ? y : zero;
                sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, xs), __builtin_bit_cast(half8_t, ys), sum, 0, 0, 0);
            }
            // (all four results land before a register of those that are not stored is used again)
            asm volatile("s_nop 15" : "+v"(sum));
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c < left && (4 * g + e) / V == c) out[(size_t)its_place * V + (4 * g + e) % V] = (OutT)sum[e];
        }
    }
}

template <int V, int TM, typename OutT>
int launch_tile(int m_vec, int k, int n, const int *row_offsets, const int *col_indices, const half_t *lhs,
                const half_t *rhs, OutT *out, hipStream_t stream, const Batch &batch)
{
    constexpr int TN = TM;
    const long long row_blocks = ((long long)m_vec * V + TM - 1) / TM, column_tiles = ((long long)n + TN - 1) / TN;
    const long long blocks = (row_blocks >= 8 ? (row_blocks + 7) / 8 * 8 : row_blocks) * column_tiles;
    if (blocks > 0x7fffffffLL) return hipErrorNotSupported;
    const auto kernel = k > kTileK ? sddmm_tile_kernel<V, TM, TN, true, OutT> : sddmm_tile_kernel<V, TM, TN, false, OutT>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks, (unsigned)batch.count), dim3(4 * TM), 0, stream, m_vec, k, n, (int)row_blocks, (int)column_tiles, row_offsets, col_indices, lhs, rhs, out,
                       batch.stride_a, batch.stride_b, batch.stride_out);
    return (int)hipGetLastError();
}

template <int V, typename OutT>
int launch_tile_shape(bool wide, int m_vec, int k, int n, const int *row_offsets, const int *col_indices, const half_t *lhs,
                      const half_t *rhs, OutT *out, hipStream_t stream, const Batch &batch)
{
    if (wide) return launch_tile<V, 128, OutT>(m_vec, k, n, row_offsets, col_indices, lhs, rhs, out, stream, batch);
    return launch_tile<V, 64, OutT>(m_vec, k, n, row_offsets, col_indices, lhs, rhs, out, stream, batch);
}

}  // namespace

// Both sides of the choice as microseconds per launch, fitted to 600 problems (64..4096 rows, 64..4608 columns, K = 32..512,
// 50..98 %, every V; device time).  Gathering: a launch and its chain of round trips, then V times fewer bytes through the
// L2s the longer the vectors (a MB of gathered rows in 0.064 us at V = 1, 0.1 us at V = 8, whose waves hold fewer of them).
// Tiles: up to 512 tiles of 64 x 64 all run at once and a launch costs one tile's chain (search, product, sampling); larger
// problems take tiles of 128 x 128 (half the operand traffic), a quarter of a thousand at a time, 0.7 us per 64 of K; the
// masked outputs come on top.  Over 1400 problems of the same ranges the rule is 0.6 % off always taking the faster side; it
// sends 213 of them to the tiles and is wrong by more than 3 % on eight (by 11 % at most: either side's estimate is
// good to about that).  A line that spares those eight (0.80 for 0.92) gathers others that tiles serve up to 1.6 times faster.
// 4096 x 4096, V = 1, K = 256: 190 / 80 / 43 / 11.4 us gathering at 50 / 80 / 90 / 98 %, 26.1 / 18.9 / 17.5 / 16.2 us on tiles;
// 2048 x 2304, V = 4, K = 512: 14.7 against 11.2 us at 90 %, 4.7 against 10.7 us at 98 %; 2048 x 2048, V = 8, K = 64: 2.5 against
// 3.8 us at 90 %, 5.0 against 4.6 us at 50 %; at the line, 2048 x 2048, V = 1, K = 64: 8.3 / 5.1 / 3.6 against 5.8 / 5.4 / 5.1 us
// at 80 / 90 / 95 % (tiles at 80 and 90 %).
// Only where the caller vouches for ascending columns: with shuffled ones most nonzeros are multiplied one by one, in
// several tiles each, which no row length or sparsity makes up for, and sizes do not tell the order.
int sddmm_tile_choice(int m_vec, int k, int n, long long nonzeros_vec, int vec_length, const Batch &problems)
{
    const int batch = problems.count;
    const Options &o = options();
    if (k <= 0 || k % 8 != 0 || n <= 0 || k > (1 << 20) || o.sddmm_tile == 1) return 0;
    if (o.sddmm_tile >= 2) return o.sddmm_tile - 1;
    if (!problems.sorted_columns) return 0;
    if (o.sddmm_slots || o.sddmm_group || o.sddmm_block_waves) return 0;  // a launch shape of the gathering kernels is asked for
    const double nonzeros = (double)nonzeros_vec * batch, steps = (k + kTileK - 1) / kTileK;
    const double per_mega = vec_length == 1 ? 0.128 : (vec_length == 2 ? 0.145 : (vec_length == 4 ? 0.175 : 0.21));
    const double gather = 2.75 + per_mega * 1e-6 * nonzeros * k;
    auto tiles = [&](double side) { return std::ceil((double)m_vec * vec_length / side) * std::ceil(n / side) * batch; };
    const bool narrow = tiles(64) <= 512;
    const double rounds = tiles(128) > 256 ? tiles(128) / 256 : 1;
    const double product = narrow ? 4.0 + 0.25 * steps : 3.9 + (0.1 + 0.7 * steps) * rounds;
    if (product + 1.15e-6 * nonzeros * vec_length > 0.92 * gather) return 0;
    return narrow ? 1 : 2;
}

template <typename OutT>
int launch_sddmm_tile(int shape, int m_vec, int k, int n, const int *row_offsets, const int *col_indices, const half_t *lhs,
                      const half_t *rhs, OutT *out, int vec_length, hipStream_t stream, const Batch &batch)
{
    const bool wide = shape == 2;
    switch (vec_length) {
    case 1: return launch_tile_shape<1, OutT>(wide, m_vec, k, n, row_offsets, col_indices, lhs, rhs, out, stream, batch);
    case 2: return launch_tile_shape<2, OutT>(wide, m_vec, k, n, row_offsets, col_indices, lhs, rhs, out, stream, batch);
    case 4: return launch_tile_shape<4, OutT>(wide, m_vec, k, n, row_offsets, col_indices, lhs, rhs, out, stream, batch);
    case 8: return launch_tile_shape<8, OutT>(wide, m_vec, k, n, row_offsets, col_indices, lhs, rhs, out, stream, batch);
    default: return hipErrorInvalidValue;
    }
}

template int launch_sddmm_tile<half_t>(int, int, int, int, const int *, const int *, const half_t *, const half_t *,
                                       half_t *, int, hipStream_t, const Batch &);
template int launch_sddmm_tile<float>(int, int, int, int, const int *, const int *, const half_t *, const half_t *, float *,
                                      int, hipStream_t, const Batch &);

}  // namespace vs
