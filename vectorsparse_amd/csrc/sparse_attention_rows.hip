// A sparse attention layer in one launch, a workgroup per vector row (V = 1, 2, 4, 8; d_qk = d_v = 64 or 128):
// p[j] = softmax_row(scale * q[i] . k[col_j]), out[i] = sum_j p[j] v[col_j]; KEEP: the probabilities are written out too.
//
// The two launches it replaces (SDDMM, then softmax and SpMM) each walk from row extents to column indices to gathered rows,
// and hand the scores over through memory.  Here a wave takes up to 32 STEPS of the row's nonzeros, keeps their scores in the registers
// that the matrix cores leave them in, and gathers k and v by the same indices:
//   scores of sixteen nonzeros: sixteen rows of k (lane c of a group of sixteen: row c) times the vector row's V rows of q, so
//   that lane (c, g) has those of scalar row c and nonzeros 4 g .. 4 g + 3 - which is what the second product wants of its
//   first operand when a step of 32 numbers its nonzeros 4 g + e and 16 + 4 g + e (a contraction's order is free);
//   maximum and sum: over the wave's registers, the four groups, the waves; the probabilities are rounded to fp16 and it is
//   those that are multiplied, as the operators do.
//
// What bounds it (8 heads x 2048, V = 4, width 64, rows of 102, HIP-graph replays: 15.1 us with the probabilities, 14.8 us without; 18.6 and 17.8 us
// as two launches): the gathers - 107 MB, of which a request asks sixteen half lines (k) or four lines (v) - behind a chain of five dependent loads that
// four waves per SIMD hide from each other in part.  Registers hold both gathers of a wave's two steps; of three and four steps k comes in
// halves and v behind it (all of k at once spills: 8 heads x 648, width 128, rows of 65: 13.7 against 9.9 us).
#include <type_traits>

#include "spmm_mfma_step.hpp"

namespace vs {

namespace {

// The CPL columns of a gathered row of v that a lane multiplies (zeros for a nonzero that does not exist).
template <int CPL>
__device__ __forceinline__ void load_row_of_v(RowChunk<CPL> &to, const __amdgpu_buffer_rsrc_t &from, unsigned offset)
{
    if constexpr (CPL == 4) to.d = __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(from, (int)offset, 0, 0));
    else to.d = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(from, (int)offset, 0, 0));
}

template <int V, int CPL, int STEPS, int W, bool KEEP>
__global__ void __launch_bounds__(64 * W, 4)
attention_rows_kernel(int heads, int n, const int *__restrict__ row_indices, const int *__restrict__ row_offsets,
                      const int *__restrict__ col_indices, const half_t *q /* (out in its place is allowed) */, const half_t *__restrict__ k,
                      const half_t *__restrict__ v, half_t *out, half_t *__restrict__ kept, long long stride_q, long long stride_k,
                      long long stride_v, long long stride_out, long long stride_kept, float scale_log2e)
{
    constexpr int D = 16 * CPL, KK = D / 32;
    __shared__ float stat[2][W][16];
    __shared__ __align__(16) float sums[W > 1 ? W * V * D : 1];
    __shared__ __align__(16) half_t staged[KEEP ? W * STEPS * kStep * V : 1];
    // (heads change fastest: with a multiple of eight of them an XCD has the rows of k and v of its own heads only)
    const int head = blockIdx.x % heads, row = row_indices[blockIdx.x / heads];
    const int lane = threadIdx.x & 63, wave = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
    const int c = lane & 15, g = lane >> 4;
    const int beg = row_offsets[row], end = row_offsets[row + 1];
    q += head * stride_q + (size_t)row * V * D;
    k += head * stride_k;
    v += head * stride_v;
    out += head * stride_out + (size_t)row * V * D;
    if constexpr (KEEP) kept += head * stride_kept;
    if (beg >= end) {
        if (wave == 0)
            for (int i = lane; i < V * D / 8; i += 64) reinterpret_cast<uint4_t *>(out)[i] = uint4_t{0u, 0u, 0u, 0u};
        return;
    }
    const __amdgpu_buffer_rsrc_t v_rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t *>(v), 0, (int)((long long)n * D * 2), 0x00020000);
    half8_t query[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
        const uint4_t x = *reinterpret_cast<const uint4_t *>(q + (c < V ? c : 0) * D + 32 * kk + 8 * g);
        query[kk] = c < V ? __builtin_bit_cast(half8_t, x) : half8_t{0, 0, 0, 0, 0, 0, 0, 0};
    }

    // 2 NS groups of sixteen nonzeros from `base` on: their columns (lane c: that of nonzero c) and scaled scores
    auto columns_of = [&](auto count, int (&column)[2 * STEPS], int base) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 2 * decltype(count)::value; ++t) {
            const int j = base + 16 * t + c;
            column[t] = col_indices[j < end ? j : end - 1];
        }
    };
    auto scores_of = [&](auto count, const int (&column)[2 * STEPS], float4_t (&score)[2 * STEPS], int base) __attribute__((always_inline)) {
        constexpr int GROUPS = 2 * decltype(count)::value, AT_ONCE = GROUPS * KK <= 8 ? GROUPS : 8 / KK;
#pragma unroll
        for (int t0 = 0; t0 < GROUPS; t0 += AT_ONCE) {
            half8_t key[AT_ONCE][KK];
#pragma unroll
            for (int t = 0; t < AT_ONCE; ++t)
#pragma unroll
                for (int kk = 0; kk < KK; ++kk)
                    if (t0 + t < GROUPS) key[t][kk] = *reinterpret_cast<const half8_t *>(k + ((uint32_t)column[t0 + t] * (uint32_t)D + (uint32_t)(32 * kk + 8 * g)));
            if constexpr (AT_ONCE < GROUPS) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < AT_ONCE; ++t)
                if (t0 + t < GROUPS) {
                    float4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int kk = 0; kk < KK; ++kk) s = __builtin_amdgcn_mfma_f32_16x16x32_f16(key[t][kk], query[kk], s, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) score[t0 + t][e] = base + 16 * (t0 + t) + 4 * g + e < end ? s[e] * scale_log2e : -__builtin_inff();
                }
            if constexpr (AT_ONCE < GROUPS) __builtin_amdgcn_sched_barrier(0);
        }
    };
    // over the four groups of lanes
    auto most = [&](float x) { x = fmaxf(x, partner<16>(x)); return fmaxf(x, partner<32>(x)); };
    auto total = [&](float x) { x += partner<16>(x); return x + partner<32>(x); };
    // ... and over the waves; `what`: 0 maximum, 1 sum
    auto all_waves = [&](float x, int what) __attribute__((always_inline)) {
        if constexpr (W == 1) return x;
        if (lane < 16) stat[what][wave][lane] = x;
        __syncthreads();
        float y = stat[what][0][c];
#pragma unroll
        for (int w = 1; w < W; ++w) y = what == 0 ? fmaxf(y, stat[what][w][c]) : y + stat[what][w][c];
        return y;
    };
    float4_t acc[CPL];
#pragma unroll
    for (int j = 0; j < CPL; ++j) acc[j] = float4_t{0.f, 0.f, 0.f, 0.f};
    half_t *const mine = staged + (KEEP ? wave * STEPS * kStep * V : 0);
    // a step's probabilities (of groups t and t + 1, already divided by the sum) times its rows of v
    auto multiply = [&](const RowChunk<CPL> (&rows)[8], const half8_t &p) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < CPL / 2; ++x) {
            uint4_t even, odd;
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                even[y] = pack_lo(rows[2 * y].dword(x), rows[2 * y + 1].dword(x));
                odd[y] = pack_hi(rows[2 * y].dword(x), rows[2 * y + 1].dword(x));
            }
            acc[2 * x] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p, __builtin_bit_cast(half8_t, even), acc[2 * x], 0, 0, 0);
            acc[2 * x + 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(p, __builtin_bit_cast(half8_t, odd), acc[2 * x + 1], 0, 0, 0);
        }
    };
    auto gather_v = [&](RowChunk<CPL> (&rows)[8], const int (&column)[2 * STEPS], int s, int base) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int t = 2 * s + e / 4, from = 4 * g + e % 4;
            const int col = __builtin_amdgcn_ds_bpermute(4 * from, column[t]);
            load_row_of_v<CPL>(rows[e], v_rows, base + 16 * t + from < end ? ((unsigned)col * (unsigned)D + (unsigned)(CPL * c)) * 2u : 0x80000000u);
        }
    };
    auto keep = [&](int nonzeros, int base) __attribute__((always_inline)) {   // staged probabilities of the wave, written out in whole pieces
        wave_lds_fence();
        const int halves = nonzeros * V;
        half_t *const to = kept + (size_t)base * V;
        for (int i = 8 * lane; i < halves; i += 512) {
            if (i + 8 <= halves) {
                typedef uint32_t words_t __attribute__((ext_vector_type(4), aligned(2)));
                *reinterpret_cast<words_t *>(to + i) = __builtin_bit_cast(words_t, *reinterpret_cast<const uint4_t *>(mine + i));
            } else {
                for (int h = i; h < halves; ++h) to[h] = mine[h];
            }
        }
        wave_lds_fence();
    };
    auto probabilities = [&](const float4_t (&score)[2 * STEPS], int s, float inverse) __attribute__((always_inline)) {
        half8_t p;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int t = 2 * s + e / 4;
            p[e] = (half_t)(score[t][e % 4] * inverse);
            if (KEEP && c < V) mine[(16 * t + 4 * g + e % 4) * V + c] = p[e];
        }
        return p;
    };

    const int steps = (end - beg + kStep - 1) / kStep, per = (steps + W - 1) / W;
    if (per <= STEPS) {
        const int base = beg + wave * per * kStep, count = steps - wave * per < per ? steps - wave * per : per;
        auto run = [&](auto number) __attribute__((always_inline)) {
            constexpr int NS = decltype(number)::value;
            int column[2 * STEPS];
            float4_t score[2 * STEPS];
            float peak = -__builtin_inff();
            // (both gathers in flight at once where the registers hold them)
            constexpr bool EARLY = NS * CPL <= 8;
            RowChunk<CPL> rows[NS > 0 ? NS : 1][8];
            if constexpr (NS > 0) {
                columns_of(number, column, base);
                if constexpr (EARLY) {
#pragma unroll
                    for (int s = 0; s < NS; ++s) gather_v(rows[s], column, s, base);
                }
                scores_of(number, column, score, base);
            }
            if constexpr (!EARLY) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int s = 0; s < NS; ++s) gather_v(rows[s], column, s, base);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int t = 0; t < 2 * NS; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) peak = fmaxf(peak, score[t][e]);
            peak = all_waves(most(peak), 0);
            float sum = 0.f;
#pragma unroll
            for (int t = 0; t < 2 * NS; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    score[t][e] = __builtin_amdgcn_exp2f(score[t][e] - peak);
                    sum += score[t][e];
                }
            const float inverse = 1.f / all_waves(total(sum), 1);
#pragma unroll
            for (int s = 0; s < NS; ++s) multiply(rows[s], probabilities(score, s, inverse));
            if constexpr (KEEP && NS > 0) keep(end - base < NS * kStep ? end - base : NS * kStep, base);
        };
        if (count <= 0) run(std::integral_constant<int, 0>());
        else if (count == 1) run(std::integral_constant<int, 1>());
        else if (STEPS >= 2 && count == 2) run(std::integral_constant<int, 2>());
        else if constexpr (STEPS >= 4) {
            if (count == 3) run(std::integral_constant<int, 3>());
            else run(std::integral_constant<int, 4>());
        }
    } else {
        // a row longer than the launch was made for: its scores once for maximum and sum, once more for the product
        constexpr std::integral_constant<int, STEPS> whole;
        int column[2 * STEPS];
        float4_t score[2 * STEPS];
        float peak = -__builtin_inff(), sum = 0.f;
        for (int base = beg + wave * STEPS * kStep; base < end; base += W * STEPS * kStep) {
            columns_of(whole, column, base);
            scores_of(whole, column, score, base);
            float here = peak;
#pragma unroll
            for (int t = 0; t < 2 * STEPS; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) here = fmaxf(here, score[t][e]);
            if (here > -__builtin_inff()) {
                sum *= __builtin_amdgcn_exp2f(peak - here);
#pragma unroll
                for (int t = 0; t < 2 * STEPS; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum += __builtin_amdgcn_exp2f(score[t][e] - here);
            } else {   // (nothing, or NaN alone: the row's)
#pragma unroll
                for (int t = 0; t < 2 * STEPS; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum += score[t][e] == score[t][e] ? 0.f : score[t][e];
            }
            peak = here;
        }
        const float highest = all_waves(most(peak), 0);
        const float inverse = 1.f / all_waves(total(peak > -__builtin_inff() ? sum * __builtin_amdgcn_exp2f(peak - highest) : sum), 1);
        for (int base = beg + wave * STEPS * kStep; base < end; base += W * STEPS * kStep) {
            columns_of(whole, column, base);
            scores_of(whole, column, score, base);
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                RowChunk<CPL> rows[8];
                gather_v(rows, column, s, base);
#pragma unroll
                for (int t = 2 * s; t < 2 * s + 2; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) score[t][e] = __builtin_amdgcn_exp2f(score[t][e] - highest);
                multiply(rows, probabilities(score, s, inverse));
            }
            if constexpr (KEEP) keep(end - base < STEPS * kStep ? end - base : STEPS * kStep, base);
        }
    }

    // lane (c, g), element e of acc[j]: row 4 g + e, column CPL c + j
    if constexpr (W > 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (4 * g + e < V) {
#pragma unroll
                for (int j = 0; j < CPL; ++j) sums[(wave * V + 4 * g + e) * D + CPL * c + j] = acc[j][e];
            }
        __syncthreads();
        for (int i = 4 * threadIdx.x; i < V * D; i += 256 * W) {
            float4_t x = *reinterpret_cast<const float4_t *>(sums + i);
#pragma unroll
            for (int w = 1; w < W; ++w) {
                const float4_t y = *reinterpret_cast<const float4_t *>(sums + w * V * D + i);
#pragma unroll
                for (int j = 0; j < 4; ++j) x[j] += y[j];
            }
            const float xs[4] = {x[0], x[1], x[2], x[3]};
            store_converted<half_t, 4>(out + i, xs);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (4 * g + e < V) {
                float x[CPL];
#pragma unroll
                for (int j = 0; j < CPL; ++j) x[j] = acc[j][e];
                store_converted<half_t, CPL>(out + (4 * g + e) * D + CPL * c, x);
            }
    }
}

template <int V, int CPL, int STEPS, int W>
int launch_rows(bool keep, int m_vec, int n, const int *row_indices, const int *row_offsets, const int *col_indices, const half_t *q,
                const half_t *k, const half_t *v, half_t *out, half_t *kept, float scale, long long stride_q, long long stride_k,
                long long stride_v, long long stride_out, long long stride_kept, int heads, hipStream_t stream)
{
    const auto kernel = keep ? attention_rows_kernel<V, CPL, STEPS, W, true> : attention_rows_kernel<V, CPL, STEPS, W, false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((long long)m_vec * heads)), dim3(64 * W), 0, stream, heads, n, row_indices, row_offsets,
                       col_indices, q, k, v, out, kept, stride_q, stride_k, stride_v, stride_out, stride_kept, scale * kLog2e);
    return (int)hipGetLastError();
}

template <int V, int CPL, typename... Args>
int launch_rows_shape(int waves, Args... args)
{
    constexpr int STEPS = 16 / CPL;
    switch (waves) {
    case 1: return launch_rows<V, CPL, STEPS, 1>(args...);
    case 2: return launch_rows<V, CPL, STEPS, 2>(args...);
    case 4: return launch_rows<V, CPL, STEPS, 4>(args...);
    case 8: return launch_rows<V, CPL, STEPS, 8>(args...);
    default: return hipErrorInvalidValue;
    }
}

template <int V, typename... Args>
int launch_rows_width(int d, int waves, Args... args)
{
    return d == 64 ? launch_rows_shape<V, 4>(waves, args...) : launch_rows_shape<V, 8>(waves, args...);
}

}  // namespace

// One launch against the two it replaces as microseconds, fitted to 1920 masks (bands and random ones, 1..16 heads x 512..4096, head
// widths of 64 and 128, rows of 10 to 490 nonzero vectors, every V; profiles/attention_rows_rule_survey.txt), the two to within 7 %, the
// one to within 6 %: one launch costs 2 to 3 us less, and nothing per row beyond its gathers, which come by the same columns; the two gather
// in wider waves, so that many long rows are theirs.  Taken for 2569 of 3840 layers, 1.44 times faster in the median (16 heads x 788, V =
// 4, rows of 16: 11.2 against 6.7 us; 8 x 2048, V = 4, rows of 102: 17.9 against 14.8 us), slower for 32, by more than 3 % for 15 (8 x 2728, V
// = 2, width 128, a band of 36: 27.0 against 31.6 us); of the others 145 would gain more than 5 %.  Not taken for 16 x 3928, V = 8, rows of
// 393 (69 against 75 us) and 8 x 2048, V = 1, rows of 102 (43 against 47 us).
int attention_rows_waves(bool keep, int heads, int m_vec, int n, int vec_length, int d_qk, int d_v, int nonzeros_vec, int longest_row_vec)
{
    const Options &o = options();
    if (o.attention_rows == 1) return 0;
    if (d_qk != d_v || (d_v != 64 && d_v != 128) || n <= 0 || m_vec <= 0 || heads <= 0 || (long long)n * d_v >= (1LL << 30) ||
        (long long)m_vec * heads >= (1LL << 32) / 512)
        return 0;   // (a launch has fewer than 2^32 threads, eight waves for a row at most)
    if (o.attention_rows >= 2) return 1 << (o.attention_rows - 2);
    if (longest_row_vec < 0 || longest_row_vec > 512 || o.softmax_spmm || o.sddmm_slots || o.sddmm_block_waves || o.sddmm_group || o.sddmm_tile ||
        o.spmm_waves || o.spmm_cols_per_lane || o.spmm_steps)
        return 0;   // (a launch shape of the other kernels is asked for)
    const int wide = d_v == 128, v = vec_length == 1 ? 0 : (vec_length == 2 ? 1 : (vec_length == 4 ? 2 : 3));
    const double rows = 1e-3 * m_vec * heads, gathers = 1e-6 * (double)nonzeros_vec * heads, mean = 1e-2 * nonzeros_vec / m_vec;
    struct Cost {
        double launch, row, gather, mean;
    };
    static constexpr Cost kTwo[2][2][4] = {{{{5.5, 0.44, 13.02, 1.62}, {6.02, 0.49, 14.03, 1.09}, {6.42, 0.66, 16.21, 0.89}, {6.83, 0.92, 19.01, 1.06}},
                                            {{5.39, 0.88, 15.75, 2.25}, {5.75, 0.91, 20.36, 1.89}, {6.41, 1.11, 26.43, 1.06}, {6.84, 1.56, 31.24, 1.21}}},
                                           {{{5.95, 0.47, 13.31, 1.37}, {6.45, 0.56, 14.14, 0.85}, {6.6, 0.81, 16.72, 0.91}, {7.16, 1.17, 20.41, 1.11}},
                                            {{5.84, 0.96, 14.94, 1.93}, {6.04, 1.08, 20.0, 1.45}, {6.91, 1.19, 26.75, 0.98}, {7.86, 1.36, 32.77, 1.25}}}};
    static constexpr Cost kOne[2][2][4] = {{{{3.45, 0.12, 22.04, 0.74}, {3.72, 0.12, 22.46, 0.58}, {3.77, 0.13, 23.11, 0.61}, {3.98, 0.02, 24.86, 0.4}},
                                            {{3.52, 0.23, 38.51, 0.73}, {3.85, 0.33, 38.78, 0.65}, {4.0, 0.34, 41.06, 0.61}, {4.24, 0.31, 43.76, 0.54}}},
                                           {{{3.88, 0.17, 22.39, 0.3}, {4.07, 0.18, 22.48, 0.34}, {4.07, 0.19, 23.01, 0.42}, {4.17, 0.1, 25.62, 0.31}},
                                            {{3.85, 0.19, 40.09, 0.9}, {4.16, 0.04, 49.08, 0.81}, {4.2, 0.09, 45.64, 0.68}, {4.36, 0.03, 47.67, 0.66}}}};
    const auto us = [&](const Cost &c) { return c.launch + c.row * rows + c.gather * gathers + c.mean * mean; };
    if (us(kOne[keep][wide][v]) > 0.95 * us(kTwo[keep][wide][v])) return 0;
    // as few waves as hold the row; twice as many where the chip has room for them
    const int steps = (longest_row_vec + kStep - 1) / kStep, held = d_v == 64 ? 4 : 2;
    int waves = 1;
    while (waves < 8 && (waves * held < steps || ((long long)m_vec * heads * waves < 4096 && steps > 2 * waves))) waves *= 2;
    return waves;
}

int launch_attention_rows(int waves, bool keep, int m_vec, int vec_length, int n, int d, const int *row_indices, const int *row_offsets,
                          const int *col_indices, const half_t *q, const half_t *k, const half_t *v, half_t *out, half_t *kept, float scale,
                          long long stride_q, long long stride_k, long long stride_v, long long stride_out, long long stride_kept, int heads,
                          hipStream_t stream)
{
    switch (vec_length) {
    case 1: return launch_rows_width<1>(d, waves, keep, m_vec, n, row_indices, row_offsets, col_indices, q, k, v, out, kept, scale, stride_q, stride_k, stride_v, stride_out, stride_kept, heads, stream);
    case 2: return launch_rows_width<2>(d, waves, keep, m_vec, n, row_indices, row_offsets, col_indices, q, k, v, out, kept, scale, stride_q, stride_k, stride_v, stride_out, stride_kept, heads, stream);
    case 4: return launch_rows_width<4>(d, waves, keep, m_vec, n, row_indices, row_offsets, col_indices, q, k, v, out, kept, scale, stride_q, stride_k, stride_v, stride_out, stride_kept, heads, stream);
    case 8: return launch_rows_width<8>(d, waves, keep, m_vec, n, row_indices, row_offsets, col_indices, q, k, v, out, kept, scale, stride_q, stride_k, stride_v, stride_out, stride_kept, heads, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace vs
