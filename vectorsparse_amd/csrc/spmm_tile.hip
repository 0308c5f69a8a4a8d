// SpMM on dense tiles (V = 1, 2, 4, 8; fp16 outputs): C[i*V + v][c] = sum_j values[j*V + v] * rhs[col_j][c].
//
// The gathering kernels (spmm_mfma.hip, spmm_valu.hip) pull one row of rhs through the L2s for every nonzero vector, 2 N
// bytes for V N multiply-adds, and the L2s deliver 21 to 26 TB/s of that and no more.  Where the pattern keeps a good share
// of a block of rows it is cheaper to read every row of rhs once per block and to multiply the zeros as well: the bytes
// fall by (density x TM / V).  A workgroup owns TM scalar rows x TN columns and walks the contraction in chunks of KC, two
// workgroups per CU taking turns at the two halves of a chunk:
//   1. the nonzeros of the chunk are scattered into a zeroed operand in LDS ([k][row], so that a nonzero vector is one
//      write and a transposing read brings four k of a row; 32 bytes more than TM rows per k put the eight k of half a wave
//      on all banks).  The lanes of a vector row hold a window of its nonzeros, take what falls into the chunk, advance the
//      row's cursor by their number and request the next window, a chunk ahead of its use.  A wave zeroes and fills only
//      rows that it owns (LDS operations of a wave stay in order: no barrier between the two);
//   2. KW x NWC waves multiply: rows of rhs straight from global memory to registers, DEPTH steps ahead, eight rows of four
//      columns per lane, transposed with v_perm_b32 (as the gathering kernel does), every operand used for TM / 16
//      products; the KW waves of a column block share the chunk's steps of 32 and add up their fp32 tiles at the end.
//
// What a dense product cannot see is put right afterwards, per workgroup: a zero times an infinity or a NaN of rhs is a NaN
// in the tile, and a row whose columns do not ascend strictly would lose nonzeros - both are noticed (NaN outputs, a column
// that does not follow its predecessor or its chunk, a cursor that does not end with its row) and the workgroup then
// computes its tile again nonzero by nonzero, with the steps of the gathering kernel.
//
// What bounds it (4096 x 4096 x 2048, V = 4, 80 %, tiles of 128 x 128: 75 us, 130 us gathering): of a workgroup's 134 k
// cycles 48 k go into filling, 60 k into multiplying, 20 k into barriers.  By the counters the matrix cores are busy for 37 %
// of the launch at 2.4 GHz (44 % at the 2 GHz or so that their load leaves; the products alone take 44 us), LDS for 38 %, of
// which 42 % are bank conflicts.  Small launches wait for rhs: the
// vector memory path takes about 18 cycles per request of 512 bytes.  Measured and not kept, same problem: one operand
// ahead in LDS and the two waves of a SIMD filling and multiplying in opposite order 71 us (one workgroup per CU, 79 us for
// half the steps per barrier); waves that only fill beside waves that only multiply 70 us (accumulators in AGPRs, else
// spills) to 88 us (starts of the chunks scouted ahead); rhs copied to LDS without registers 73 to 83 us.  Where a workspace
// may be had, rows packed two of four (spmm_pack.hip) take 67 us there.
#include <cmath>
#include <type_traits>

#include "spmm_mfma_step.hpp"

namespace vs {

namespace {

// Sum over the LPR lanes of a vector row (an aligned block of lanes).
template <int LPR>
__device__ __forceinline__ int row_sum(int x)
{
    const auto add = [&](float y) { x += __builtin_bit_cast(int, y); };
    if constexpr (LPR > 1) add(partner<1>(__builtin_bit_cast(float, x)));
    if constexpr (LPR > 2) add(partner<2>(__builtin_bit_cast(float, x)));
    if constexpr (LPR > 4) add(partner<4>(__builtin_bit_cast(float, x)));
    if constexpr (LPR > 8) add(partner<8>(__builtin_bit_cast(float, x)));
    if constexpr (LPR > 16) add(partner<16>(__builtin_bit_cast(float, x)));
    if constexpr (LPR > 32) add(partner<32>(__builtin_bit_cast(float, x)));
    return x;
}

// Orders LDS only: requests of rhs rows and of nonzeros stay in flight across it.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

constexpr int smaller(int a, int b) { return a < b ? a : b; }
constexpr int larger(int a, int b) { return a > b ? a : b; }

template <int V, int MI, int NWC, int KW, int STEPS, int EACH_>
struct TileShape {
    static constexpr int TM = 16 * MI, TN = 64 * NWC, WAVES = NWC * KW, THREADS = 64 * WAVES;
    static constexpr int KC = 32 * KW * STEPS;               // contraction elements per chunk: STEPS steps of every wave
    static constexpr int ROWS = TM / V;                      // vector rows
    static constexpr int LPR = smaller(64, THREADS / ROWS);  // lanes per vector row
    static constexpr int EACH = EACH_;                       // consecutive nonzeros of a lane
    static constexpr int PITCH = TM * 2 + 32;                // bytes per k of a chunk's operand
    static constexpr int RPW = 64 / LPR;                     // vector rows of a wave
    static constexpr int UNIT = smaller(16, RPW * V * 2), PER_K = RPW * V * 2 / UNIT;  // pieces a wave zeroes, pieces per k
    static constexpr int DUMP = PITCH * KC;                  // a place for what is not taken
    static constexpr int UNITS = MI * 4;                     // a wave's outputs in units of a row x four columns per lane
    // LDS: the operand; at the end the sums, of a pair of waves the half that the other one finishes
    static constexpr int AREA = larger(DUMP + 64 * 16, KW > 1 ? WAVES * UNITS / (KW == 2 ? 2 : 1) * 1024 : 0);
    static_assert(THREADS >= ROWS && UNITS % KW == 0 && AREA >= WAVES * stage_bytes<V>() && AREA <= 79 * 1024 && RPW * V * 2 >= 8, "");
};

template <int V, int MI, int NWC, int KW, int STEPS, int DEPTH, int EACH>
__global__ void __launch_bounds__(64 * NWC * KW, NWC * KW * 2 / 4)
spmm_tile_kernel(int m_vec, int N, int n, int column_tiles, const int *__restrict__ row_offsets,
                 const int *__restrict__ col_indices, const half_t *__restrict__ values, const half_t *__restrict__ rhs,
                 half_t *__restrict__ out, long long stride_values, long long stride_rhs, long long stride_out)
{
    using S = TileShape<V, MI, NWC, KW, STEPS, EACH>;
    constexpr int TM = S::TM, KC = S::KC, ROWS = S::ROWS, LPR = S::LPR, RPW = S::RPW, PITCH = S::PITCH;
    static_assert(STEPS % DEPTH == 0, "the ring of requested steps closes with the chunk");
    extern __shared__ __align__(16) unsigned char area[];

    const int ct = blockIdx.x % column_tiles, rb = blockIdx.x / column_tiles;
    if (blockIdx.y != 0) {
        values += blockIdx.y * stride_values;
        rhs += blockIdx.y * stride_rhs;
        out += blockIdx.y * stride_out;
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int cw = wave % NWC, kw = wave / NWC;

    // this lane's vector row and its place among the row's lanes
    const int row_here = tid / LPR, row = rb * ROWS + row_here, li = tid % LPR;
    const int nonzeros = row_offsets[m_vec];
    int cursor = 0, row_end = 0;
    if (row_here < ROWS && row < m_vec) {
        cursor = row_offsets[row];
        row_end = row_offsets[row + 1];
    }

    // rhs: the lane's eight rows of a step are k 4g..4g+3 and 16+4g..16+4g+3 (both operands number the contraction that
    // way, for the transposing reads); columns past the width and rows past the end read as zeros (out of the buffer's range)
    const int col0 = ct * S::TN + 64 * cw + 4 * c;
    unsigned b_off[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) b_off[e] = col0 < N ? ((unsigned)(4 * g + (e < 4 ? e : 12 + e)) * (unsigned)N + (unsigned)col0) * 2u : 0x80000000u;
    RowChunk<4> b[DEPTH][8];
    auto request = [&](RowChunk<4> (&to)[8], int k0) __attribute__((always_inline)) {
        const long long left = (long long)(n - k0) * N * 2;
        const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<half_t *>(rhs + (size_t)(left > 0 ? k0 : 0) * N), 0, left > 0 ? (int)left : 0, 0x00020000);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            to[e].d = __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(rows, (int)b_off[e], 0, 0));
    };

    // two windows of a row's next LPR * EACH nonzeros each; the second one is looked at only where a row of the wave has
    // all of the first in the chunk
    struct Window {
        int at, from, col[EACH];   // positions of the lane's first nonzero and of the first fetched one
        PackedVector<V> val[EACH];
    };
    Window first_window, second_window;
    auto fetch = [&](Window &w, int start) __attribute__((always_inline)) {
        w.at = start + li * EACH;
        w.from = w.at < nonzeros - EACH ? w.at : nonzeros - EACH;
        __builtin_memcpy(w.col, col_indices + w.from, sizeof(w.col));
        __builtin_memcpy(w.val, values + (size_t)w.from * V, sizeof(w.val));
    };
    auto fetch_windows = [&]() __attribute__((always_inline)) {
        fetch(first_window, cursor);
        fetch(second_window, cursor + LPR * EACH);
    };
    // (a pattern of fewer nonzeros than a lane fetches at once goes nonzero by nonzero)
    const bool few = nonzeros < EACH;
    uint64_t disorder = 0;
    const int own_row = wave * RPW;                       // the wave's first vector row
    const unsigned zero_place = (unsigned)(lane / S::PER_K * PITCH + own_row * V * 2 + lane % S::PER_K * S::UNIT);
    const unsigned place_row = (unsigned)(row_here * V * 2), dump = (unsigned)(S::DUMP + 16 * lane);
    // Takes what the window holds of the chunk at k0.  `before`: the column ahead of the window's first one, k0 - 1 at a
    // chunk's first window (so that a column of an earlier chunk is out of order too).  Free of branches but for the ends of
    // rows: a nonzero that is not taken is written to a place that nothing reads.
    auto take_window = [&](Window &w, int k0, int before) __attribute__((always_inline)) {
        const int first = w.at - w.from, last = row_end - w.from;   // the lane's nonzeros: [first, last)
        int taken = 0, previous = __builtin_amdgcn_update_dpp(-1, w.col[EACH - 1], 0x138, 0xF, 0xF, false);  // wave_shr:1
        previous = li == 0 ? before : previous;
        if (__builtin_amdgcn_ballot_w64(first > 0 || last < EACH) != 0) {
            // entries ahead of the lane's own (a run moved back from the pattern's end) pass as very small ones and are not
            // counted; the first of its own still follows what its predecessor says
            if (__builtin_amdgcn_ballot_w64(first > 0) != 0) {
                int own = 0x7fffffff;
#pragma unroll
                for (int e = 1; e < EACH; ++e) own = e == first && e < last ? w.col[e] : own;
                disorder |= __builtin_amdgcn_ballot_w64(own < k0 + KC) & __builtin_amdgcn_ballot_w64(previous >= own);
                if (first > 0) previous = (int)0x80000000;
            }
#pragma unroll
            for (int e = 0; e < EACH; ++e) w.col[e] = e >= last ? 0x7fffffff : (e < first ? (int)0x80000001 + e : w.col[e]);
            taken = first < last ? first : last;
            taken = taken < 0 ? 0 : (taken > EACH ? -EACH : -taken);
        }
#pragma unroll
        for (int e = 0; e < EACH; ++e) {
            const uint64_t passed = __builtin_amdgcn_ballot_w64(w.col[e] < k0 + KC);
            disorder |= passed & __builtin_amdgcn_ballot_w64(previous >= w.col[e]);
            previous = w.col[e];
            taken += w.col[e] < k0 + KC ? 1 : 0;
            const unsigned rel = (unsigned)w.col[e] - (unsigned)k0, place = __umul24(rel, (unsigned)PITCH) + place_row;
            w.val[e].store(reinterpret_cast<half_t *>(area + (rel < (unsigned)KC ? place : dump)));
        }
        taken = row_sum<LPR>(taken);
        cursor += taken;
        return taken == LPR * EACH;
    };
    auto fill = [&](int k0) __attribute__((always_inline)) {
        if (own_row < ROWS) {
#pragma unroll
            for (int z = 0; z < KC * S::PER_K / 64; ++z) {
                unsigned char *const p = area + zero_place + z * (64 / S::PER_K) * PITCH;
                if constexpr (S::UNIT == 16) *reinterpret_cast<uint4_t *>(p) = uint4_t{0u, 0u, 0u, 0u};
                else *reinterpret_cast<uint2_t *>(p) = uint2_t{0u, 0u};
            }
        }
        wave_lds_fence();
        bool whole = take_window(first_window, k0, k0 - 1);
        if (__builtin_amdgcn_ballot_w64(whole) != 0) {
            int ahead = __builtin_amdgcn_ds_bpermute((lane | (LPR - 1)) * 4, first_window.col[EACH - 1]);
            whole = take_window(second_window, k0, whole ? ahead : k0 - 1);
            // rare: both windows taken
            while (__builtin_expect(__builtin_amdgcn_ballot_w64(whole) != 0, 0)) {
                fetch(second_window, cursor);
                ahead = li == 0 && whole ? col_indices[cursor - 1] : k0 - 1;
                whole = take_window(second_window, k0, ahead);
            }
        }
        fetch_windows();
    };

    float4_t acc[MI][4];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    // transposing reads: a block of 4 k x 16 rows per 16 lanes, lane c pointing at four rows of k c / 4
    const unsigned operand = (unsigned)((32 * kw + 4 * g + (c >> 2)) * PITCH + 8 * (c & 3));
    auto read = [&](int s, int i) __attribute__((always_inline)) {
        typedef short short4_v __attribute__((ext_vector_type(4)));
        typedef short short8_v __attribute__((ext_vector_type(8)));
        const unsigned char *const p = area + operand + (unsigned)(32 * s * KW * PITCH + 32 * i);
        const short4_v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_v *)p);
        const short4_v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_v *)(p + 16 * PITCH));
        return __builtin_bit_cast(half8_t, (short8_v){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
    };
    bool bad = few;
    if (!few) {
        fetch_windows();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < DEPTH; ++t) request(b[t], 32 * (t * KW + kw));
        __builtin_amdgcn_sched_barrier(0);
        for (int k0 = 0; k0 < n; k0 += KC) {
            fill(k0);
            lds_barrier();
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                if (s > 0 && k0 + 32 * s * KW >= n) break;   // (uniform: nothing left in the last chunk)
                half8_t a[MI], bt[4];
#pragma unroll
                for (int i = 0; i < (MI + 1) / 2; ++i) a[i] = read(s, i);
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    uint4_t even, odd;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        even[q] = pack_lo(b[s % DEPTH][2 * q].dword(p), b[s % DEPTH][2 * q + 1].dword(p));
                        odd[q] = pack_hi(b[s % DEPTH][2 * q].dword(p), b[s % DEPTH][2 * q + 1].dword(p));
                    }
                    bt[2 * p] = __builtin_bit_cast(half8_t, even);
                    bt[2 * p + 1] = __builtin_bit_cast(half8_t, odd);
                }
                const int t = s + DEPTH;
                request(b[s % DEPTH], t < STEPS ? k0 + 32 * (t * KW + kw) : k0 + KC + 32 * ((t - STEPS) * KW + kw));
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = (MI + 1) / 2; i < MI; ++i) a[i] = read(s, i);
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], bt[j], acc[i][j], 0, 0, 0);
            }
            lds_barrier();
        }
        bad = disorder != 0 || cursor != row_end;
    }

    // the KW tiles of a column added up; unit (i, e) of a wave: row 4g + e of block i, four columns per lane
    float4_t *const sums = reinterpret_cast<float4_t *>(area);
    auto mine = [&](int unit) __attribute__((always_inline)) {
        const int i = unit / 4, e = unit % 4;
        return float4_t{acc[i][0][e], acc[i][1][e], acc[i][2][e], acc[i][3][e]};
    };
    auto finish = [&](int unit, const float4_t &total) __attribute__((always_inline)) {
        const size_t r = (size_t)rb * TM + 16 * (unit / 4) + 4 * g + unit % 4;
        const float x[4] = {total[0], total[1], total[2], total[3]};
#pragma unroll
        for (int j = 0; j < 4; ++j) bad |= x[j] != x[j];
        if (r < (size_t)m_vec * V && col0 < N) store_converted<half_t, 4>(out + r * N + col0, x);
    };
    if constexpr (KW == 2) {
        // each wave hands the other's half over and finishes its own from its registers
        auto exchange = [&](auto which) __attribute__((always_inline)) {
            constexpr int HALF = S::UNITS / 2, KEPT = decltype(which)::value * HALF, GIVEN = HALF - KEPT;
#pragma unroll
            for (int u = 0; u < HALF; ++u) sums[(wave * HALF + u) * 64 + lane] = mine(GIVEN + u);
            lds_barrier();
#pragma unroll
            for (int u = 0; u < HALF; ++u) {
                const float4_t x = mine(KEPT + u), y = sums[((wave ^ NWC) * HALF + u) * 64 + lane];
                float4_t total;
#pragma unroll
                for (int j = 0; j < 4; ++j) total[j] = x[j] + y[j];
                finish(KEPT + u, total);
            }
        };
        if (kw == 0) exchange(std::integral_constant<int, 0>());
        else exchange(std::integral_constant<int, 1>());
    } else if constexpr (KW > 1) {
#pragma unroll
        for (int u = 0; u < S::UNITS; ++u) sums[(wave * S::UNITS + u) * 64 + lane] = mine(u);
        lds_barrier();
#pragma unroll
        for (int u = 0; u < S::UNITS / KW; ++u) {
            const int unit = kw * (S::UNITS / KW) + u;
            float4_t total = sums[(cw * S::UNITS + unit) * 64 + lane];
#pragma unroll
            for (int w = 1; w < KW; ++w) {
                const float4_t y = sums[((w * NWC + cw) * S::UNITS + unit) * 64 + lane];
#pragma unroll
                for (int j = 0; j < 4; ++j) total[j] += y[j];
            }
            finish(unit, total);
        }
    } else {
#pragma unroll
        for (int u = 0; u < S::UNITS; ++u) finish(u, mine(u));
    }
    if (__syncthreads_or(bad) == 0) return;

    // nonzero by nonzero: a wave per vector row and 64 columns, one step of 32 at a time
    int *const idx_s = reinterpret_cast<int *>(area + wave * stage_bytes<V>());
    half_t *const vec_s = reinterpret_cast<half_t *>(idx_s + kStep);
    for (int item = wave; item < ROWS * NWC; item += S::WAVES) {
        const int r = rb * ROWS + item / NWC, first_col = ct * S::TN + 64 * (item % NWC) + 4 * c;
        if (r >= m_vec) break;
        const int beg = row_offsets[r], end = row_offsets[r + 1];
        float4_t sum[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[j] = float4_t{0.f, 0.f, 0.f, 0.f};
        for (int base = beg; base < end; base += kStep) {
            if (lane < kStep) {
                const int j = base + lane, jc = j < end ? j : end - 1;
                half_t x[V];
                load_vector<V>(x, values + (size_t)jc * V);
                idx_s[lane] = col_indices[jc];
#pragma unroll
                for (int v = 0; v < V; ++v) vec_s[v * kStep + lane] = j < end ? x[v] : (half_t)0.f;
            }
            wave_lds_fence();
            spmm_mfma_step<V, 4, true>(idx_s, vec_s, rhs, N, first_col < N ? (uint32_t)first_col : 0u, c, g, sum, [] {});
            wave_lds_fence();
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (4 * g + e < V && first_col < N) {
                const float x[4] = {sum[0][e], sum[1][e], sum[2][e], sum[3][e]};
                store_converted<half_t, 4>(out + ((size_t)r * V + 4 * g + e) * N + first_col, x);
            }
    }
}

template <int V, int MI, int NWC, int KW, int STEPS, int DEPTH, int EACH>
int launch_shape(int m_vec, int k, int n, const int *row_offsets, const int *col_indices, const half_t *values,
                 const half_t *rhs, half_t *out, hipStream_t stream, const Batch &batch)
{
    using S = TileShape<V, MI, NWC, KW, STEPS, EACH>;
    const long long row_blocks = ((long long)m_vec + S::ROWS - 1) / S::ROWS, column_tiles = ((long long)k + S::TN - 1) / S::TN;
    if (row_blocks * column_tiles > 0x7fffffffLL) return hipErrorNotSupported;
    const auto kernel = spmm_tile_kernel<V, MI, NWC, KW, STEPS, DEPTH, EACH>;
    static std::atomic<unsigned long long> lds_allowed{0};
    const hipError_t attr = allow_large_lds(reinterpret_cast<const void *>(kernel), S::AREA, lds_allowed);
    if (attr != hipSuccess) return (int)attr;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(row_blocks * column_tiles), (unsigned)batch.count), dim3(S::THREADS), S::AREA,
                       stream, m_vec, k, n, (int)column_tiles, row_offsets, col_indices, values, rhs, out, batch.stride_a,
                       batch.stride_b, batch.stride_out);
    return (int)hipGetLastError();
}

// Consecutive nonzeros of a lane, by shape and vector length (a window is LPR times as many; two windows are on their way).
constexpr int each_of(int shape, int vec_length) { return shape < 3 ? (vec_length <= 2 ? 8 : 4) : (vec_length == 1 ? 8 : (vec_length <= 4 ? 4 : 2)); }

template <int V>
int launch_tile(int shape, int m_vec, int k, int n, const int *row_offsets, const int *col_indices, const half_t *values,
                const half_t *rhs, half_t *out, hipStream_t stream, const Batch &batch)
{
    switch (shape) {
    case 1: return launch_shape<V, 2, 1, 4, 6, 6, each_of(1, V)>(m_vec, k, n, row_offsets, col_indices, values, rhs, out, stream, batch);
    case 2: return launch_shape<V, 4, 2, 2, 6, 3, each_of(2, V)>(m_vec, k, n, row_offsets, col_indices, values, rhs, out, stream, batch);
    case 3: return launch_shape<V, 8, 2, 2, 4, 2, each_of(3, V)>(m_vec, k, n, row_offsets, col_indices, values, rhs, out, stream, batch);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

// Gathering, in the estimates of fastest_tile below.
double spmm_gather_us(bool fine_grained, int vec_length, double nonzeros_vec, int k)
{
    const int v = vec_length == 1 ? 0 : (vec_length == 2 ? 1 : (vec_length == 4 ? 2 : 3));
    static constexpr double kPerMega[2][4] = {{0.088, 0.089, 0.0925, 0.0995}, {0.076, 0.091, 0.134, 0.28}};
    return (fine_grained ? 4.7 : 4.0) + kPerMega[fine_grained][v] * 1e-6 * nonzeros_vec * k;
}

// Both sides of the choice as microseconds per launch, fitted to 2500 problems (64..4096 rows, 64..4608 columns, widths of
// 32..2048, 50..95 %, every V; device time).
// Gathering: a launch, then a time per nonzero vector and dense column (the fine-grained kernel's grows with V).  Tiles: a
// launch, then per workgroup and contraction element a share of walking, one of scattering the block's nonzeros and, where a
// row has more nonzeros in a chunk than two windows hold, one of fetching more; a CU runs one workgroup as fast as it can, a
// second one at a part of that.  Over those problems the rule (three shapes, a margin of a fifth) takes tiles for 452 of 2500
// on the MFMA path and for 624 on the fine-grained one: 1.12 and 1.17 times faster in the mean of all 2500, 1.13 and 1.20 being
// what always taking the faster side would give; six are slower by more than 3 % (9 % at most).  A margin of a tenth would
// gain half a percent more and make eighteen slower, by up to 17 %.
// How good the estimates are, over 370 problems drawn again from those ranges and both kernels
// (profiles/spmm_tile_rule_survey.txt): tiles 12 % high to 7 % low in the mean by shape and size, with spreads of 8 to 18 %.  Gathering: 40 % (MFMA) and
// 30 % (fine-grained) high below 1e7 nonzero vectors x columns, where tiles are far behind; above 1e8 20 % and 11 % low with a
// spread of 23 % and 20 %, which errs on the gathering side (the largest problems go either way: 4096 x 4096 x 2048, V = 4,
// 80 % is put at 163 us and takes 130).  One of the 740 choices is slower by more than 3 %: 12 %, 520 workgroups of 32 x 64 on the
// 512 places of the chip.  Above 1e8 the choice is 1.48 (MFMA) and 1.59 times faster in the mean, 1.60 and 1.68 with the faster side.
// 4096 x 4096 x 2048, V = 4, 80 %: 130 us gathering, 75 us on tiles of 128 x 128; 4096 x 4096 x 512, V = 1, 50 %: 317 against
// 79 us (64 x 128); 2048 x 2304 x 256, V = 2, 50 %: 31 against 18 us (32 x 64); 2048 x 2304 x 512, V = 4, 90 %: 9.1 against
// 18.5 us; at the line, 2048 x 2304 x 256, V = 1, 90 %: 13.4 (MFMA) and 12.6 us (fine-grained) against 12.9 us.
// Only where the caller vouches for strictly ascending columns: a row in another order makes its workgroup go nonzero by nonzero.
// The fastest tile shape where one is expected to be ahead of gathering (0: none), and the time of what is then run.
static int fastest_tile(bool fine_grained, int m_vec, int k, int n, int vec_length, double nonzeros_vec, int longest_vec, double &us)
{
    const double gather = spmm_gather_us(fine_grained, vec_length, nonzeros_vec, k);
    const double density = nonzeros_vec / ((double)m_vec * n), longest = (double)longest_vec / n;
    struct Shape {
        int rows, columns, chunk;
        double launch, per_block, walk, scatter, more, second;
    };
    static constexpr Shape kShapes[3] = {{32, 64, 768, 2.7, 2.94, 2.89, 0.19, 6.06, 0.76},
                                         {64, 128, 384, 0.0, 5.26, 6.31, 0.222, 5.58, 0.63},
                                         {128, 128, 256, 0.0, 6.0, 10.4, 0.28, 4.6, 0.25}};
    int best = 0;
    double least = 0.8 * gather;
    for (int shape = 1; shape <= 3; ++shape) {
        const Shape &s = kShapes[shape - 1];
        const int lanes = smaller(64, 256 * vec_length / s.rows);
        const double windows = longest * s.chunk / (2.0 * lanes * each_of(shape, vec_length));
        const double blocks = std::ceil((double)m_vec * vec_length / s.rows) * std::ceil((double)k / s.columns) / 256.0;
        const double load = 1 + s.second * (std::fmin(std::fmax(blocks, 1.0), 2.0) - 1) + std::fmax(blocks - 2, 0.0) * (1 + s.second) / 2;
        const double per_element = s.walk + s.scatter * density * s.rows / vec_length + s.more * std::fmax(0.0, windows - 1) * 100 / s.chunk;
        const double time = s.launch + (s.per_block + 1e-3 * n * per_element) * load;
        if (time < least) {
            least = time;
            best = shape;
        }
    }
    us = best ? least : gather;
    return best;
}

double spmm_expected_us(bool fine_grained, int m_vec, int k, int n, int vec_length, int nonzeros_vec, int longest_vec)
{
    double us = 0;
    fastest_tile(fine_grained, m_vec, k, n, vec_length, nonzeros_vec, longest_vec, us);
    return us;
}

int spmm_tile_choice(bool fine_grained, int m_vec, int k, int n, int vec_length, const Batch &batch)
{
    const Options &o = options();
    if (o.spmm_tile == 1 || (o.spmm_tile == 0 && !batch.sorted_columns)) return 0;
    // (the kernel's offsets into a step's rows of rhs, and into rhs, are 32-bit)
    if (m_vec <= 0 || k <= 0 || k % 4 != 0 || n <= 0 || (long long)n * k >= (1LL << 30) || k >= (1 << 24) || batch.count < 1 || batch.count > 65535) return 0;
    if (o.spmm_tile >= 2) return o.spmm_tile - 1;
    if (o.spmm_waves || o.spmm_cols_per_lane || o.spmm_steps || o.spmm_pipe || o.spmm_gather || o.spmm_teams || o.spmm_blocks_per_wave || o.spmm_guard_waves)
        return 0;  // a launch shape of the gathering kernels is asked for
    double us;
    return fastest_tile(fine_grained, m_vec, k, n, vec_length, batch.tile_nonzeros_vec, batch.tile_longest_vec, us);
}

int launch_spmm_tile(int shape, int m_vec, int vec_length, int k, int n, const int *row_offsets, const int *col_indices,
                     const half_t *values, const half_t *rhs, half_t *out, hipStream_t stream, const Batch &batch)
{
    switch (vec_length) {
    case 1: return launch_tile<1>(shape, m_vec, k, n, row_offsets, col_indices, values, rhs, out, stream, batch);
    case 2: return launch_tile<2>(shape, m_vec, k, n, row_offsets, col_indices, values, rhs, out, stream, batch);
    case 4: return launch_tile<4>(shape, m_vec, k, n, row_offsets, col_indices, values, rhs, out, stream, batch);
    case 8: return launch_tile<8>(shape, m_vec, k, n, row_offsets, col_indices, values, rhs, out, stream, batch);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace vs
