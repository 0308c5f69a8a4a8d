// SpMM on rows packed two of four (V = 1, 2, 4, 8): C[i*V + v][c] = sum_j values[j*V + v] * rhs[col_j][c].
//
// The sparse matrix instructions multiply, in the time of a dense step of 32, sixteen rows that keep at most two of every four
// neighbouring k by 64 rows of rhs.  Patterns of 80 % and more mostly fit: a group of four of a row holds a third nonzero with
// probability 0.027 at 80 %, 0.004 at 90 %.  Two launches:
//   1. spmm_pack_kernel writes the rows as the operands of those instructions to a workspace: per 16 scalar rows (a unit)
//      and 64 columns (a step) eight halves and sixteen bits of positions per lane.  What does not fit, the third and fourth
//      nonzero of a group, goes to a list of the unit, 32 at a time as operands of dense steps and the 32 columns they meet;
//   2. spmm_packed_kernel is a matrix product without an irregularity: TM x TN outputs per workgroup of eight waves, both operands
//      copied to four buffers in LDS without registers, a barrier per step; a wave's fragments of a step are read while the one
//      before is multiplied.  Every unit's list follows, its rows of rhs gathered.
// A row of rhs is read once per TM rows, a packed operand once per TN columns.
//
// What bounds it (device time, 4096 x 4096 x 2048, 256 tiles of 256 x 128): packing 11 us at V = 4, 80 % (9 us at 98 %: 19 MB of
// writes behind a chain of dependent loads), the product 39 us whatever the pattern, the lists 14 us at 80 %, 5 us at 90 %.  A step of the
// product takes 0.5 us: the workgroup's 34 KB come in 0.34 us when nothing else is done, reading and multiplying alone take 0.33 us,
// the products 0.24 us; two thirds of a step's pipes overlap.  Measured and not kept: operands through registers into two
// buffers 43 us for 39; four waves of 128 x 64 outputs, a third less read from LDS, 43 us; two groups of four waves that take turns at
// the steps 40 us; lists sorted by column, so that workgroups gather the same rows at about the same time, as long.
// With what ran before (dense tiles, gathering): V = 4, 80 %: 75 to 67 us; V = 1, 90 %: 104 to 68 us; 1600 x 3556 x 1080, V = 1, 95 %:
// 61 to 35 us.
//
// What a dense product cannot see is put right afterwards, per workgroup, as in spmm_tile.hip: zeros times infinities
// (noticed as NaN outputs) and columns that do not ascend strictly (noticed while packing) make a workgroup compute its tile
// again nonzero by nonzero.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "spmm_mfma_step.hpp"

namespace vs {

namespace {

typedef half_t half16_t __attribute__((ext_vector_type(16)));

constexpr int kUnitRows = 16, kBlockRows = 128, kBlockUnits = kBlockRows / kUnitRows;
constexpr int kStepColumns = 64;                 // contraction elements of a step
constexpr int kUnitBytes = 1024;                 // a unit's packed values of a step: 16 bytes per lane
constexpr int kListed = 32, kListBytes = 1024, kListColumnBytes = kListed * 4;   // a step of a unit's list: operand, columns

// Where things lie in the workspace (bytes).
struct PackedLayout {
    long long blocks, steps, capacity;           // blocks of 128 rows, steps, steps of all lists
    long long positions, units, columns, lists, total;   // offsets; packed values lie at 0
    PackedLayout(long long m, int n, long long nonzeros_vec)
    {
        blocks = (m + 2 * kBlockRows - 1) / (2 * kBlockRows) * 2;
        steps = (n + 4LL * kStepColumns - 1) / (4 * kStepColumns) * 4;
        capacity = nonzeros_vec / 64 + blocks * kBlockUnits;
        positions = blocks * steps * kBlockUnits * kUnitBytes;
        units = positions + blocks * steps * 1024;
        columns = units + blocks * kBlockUnits * 16;
        lists = columns + (capacity + 4) * kListColumnBytes;   // (four steps' columns are fetched at a time)
        total = lists + capacity * kListBytes + 65536;   // (four steps are requested past the end)
    }
};

// What the second launch has to know of a unit.
struct __align__(16) UnitInfo {
    int first, count, bad, unused;               // its steps in the lists; 1: rows that have to go nonzero by nonzero
};

constexpr int kPackThreads = 1024, kPackSteps = 64;   // steps of a unit in LDS at once (64 KB)
template <int V>
constexpr int list_steps_in_lds() { return V == 1 ? 16 : 8; }
template <int V>
constexpr int pack_lds_bytes(int steps) { return steps * (kUnitBytes + kUnitRows / V * 8) + list_steps_in_lds<V>() * (kListBytes + kListColumnBytes); }

// A workgroup packs one unit, V waves per vector row; what a lane fetched stays in its registers from the count of what goes to
// the list to the scattering into LDS, where 64 steps at a time and the list are put together.
template <int V>
__global__ void __launch_bounds__(kPackThreads)
spmm_pack_kernel(int m_vec, int n, int blocks, int steps, int chunk_steps, int capacity, const int *__restrict__ row_offsets,
                 const int *__restrict__ col_indices, const half_t *__restrict__ values, unsigned char *__restrict__ packed,
                 unsigned char *__restrict__ positions, UnitInfo *__restrict__ units, int *__restrict__ list_columns,
                 unsigned char *__restrict__ lists)
{
    constexpr int ROWS = kUnitRows / V, WAVES = kPackThreads / 64, PER_ROW = WAVES / ROWS;
    constexpr int LIST_STEPS = list_steps_in_lds<V>(), KEPT = V <= 2 ? 8 : 4;
    static_assert(PER_ROW == V, "");
    extern __shared__ __align__(16) unsigned char area[];
    __shared__ int wave_count[WAVES], any_bad;
    // the eight units of a block share lines of the positions: one XCD (consecutive workgroups go to consecutive XCDs)
    const int i = blockIdx.x >> 3, block = (int)(blockIdx.x & 7) + 8 * (i >> 3), unit_here = i & 7;
    if (block >= blocks) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int unit = block * kBlockUnits + unit_here, row = wave / PER_ROW, row_at = unit * ROWS + row;
    const int row_beg = row_offsets[row_at < m_vec ? row_at : m_vec], row_end = row_offsets[row_at + 1 < m_vec ? row_at + 1 : m_vec];
    const int start = row_offsets[unit * ROWS < m_vec ? unit * ROWS : m_vec], stop = row_offsets[(unit + 1) * ROWS < m_vec ? (unit + 1) * ROWS : m_vec];
    if (tid == 0) any_bad = 0;

    // A turn: 64 nonzeros of the row, one per lane.
    bool bad = false;
    auto turn_at = [&](int turn) { return row_beg + (turn * PER_ROW + wave % PER_ROW) * 64; };
    auto fetch_column = [&](int turn) __attribute__((always_inline)) {
        const int j = turn_at(turn) + lane;
        return col_indices[j < row_end ? j : (row_end > 0 ? row_end - 1 : 0)];
    };
    auto fetch = [&](PackedVector<V> &to, int turn) __attribute__((always_inline)) {
        const int j = turn_at(turn) + lane;
        to.load(values + (size_t)(j < row_end ? j : (row_end > 0 ? row_end - 1 : 0)) * V);
    };
    // A nonzero's column and, in the upper two bits, its number among those of its group of four; absent (-1): past the row's end,
    // or out of order.
    auto look = [&](int column, int turn) __attribute__((always_inline)) {
        const int base = turn_at(turn), j = base + lane;
        // the three columns before (in front of the turn's first: uniform)
        const int one = __builtin_amdgcn_update_dpp(col_indices[base > row_beg ? base - 1 : base], column, 0x138, 0xF, 0xF, false);   // wave_shr:1
        const int two = __builtin_amdgcn_update_dpp(col_indices[base > row_beg ? base - 2 : base], one, 0x138, 0xF, 0xF, false);
        const int three = __builtin_amdgcn_update_dpp(col_indices[base > row_beg ? base - 3 : base], two, 0x138, 0xF, 0xF, false);
        const int group = column >> 2, place = j - row_beg;
        const int number = (place >= 1 && (one >> 2) == group) + (place >= 2 && (two >> 2) == group) + (place >= 3 && (three >> 2) == group);
        const bool there = j < row_end, in_order = column >= 0 && column < n && (place == 0 || column > one);
        bad |= there && !in_order;
        return there && in_order ? column | (number << 30) : -1;
    };
    int kept[KEPT], listed = 0;
    PackedVector<V> kept_value[KEPT];
    if (stop > start) {   // (all on their way before the first is looked at)
#pragma unroll
        for (int t = 0; t < KEPT; ++t) {
            kept[t] = fetch_column(t);
            fetch(kept_value[t], t);
        }
    }

    half_t *const operand = reinterpret_cast<half_t *>(area);
    uint32_t *const place_bits = reinterpret_cast<uint32_t *>(area + chunk_steps * kUnitBytes);   // [step][row][two quarters of a step each]
    half_t *const list = reinterpret_cast<half_t *>(area + chunk_steps * (kUnitBytes + ROWS * 8));
    int *const list_column = reinterpret_cast<int *>(list + LIST_STEPS * (kListBytes / 2));
    auto clear = [&](int here) __attribute__((always_inline)) {
        for (int p = tid; p < here * 64; p += kPackThreads) reinterpret_cast<uint4_t *>(area)[p] = uint4_t{0u, 0u, 0u, 0u};
        // (an absent nonzero: positions 0 and 3 of its group)
        for (int p = tid; p < here * ROWS * 2; p += kPackThreads) place_bits[p] = 0xCCCCCCCCu;
    };
    clear(steps < chunk_steps ? steps : chunk_steps);
    auto clear_list = [&]() __attribute__((always_inline)) {
        for (int p = tid; p < LIST_STEPS * 64; p += kPackThreads) reinterpret_cast<uint4_t *>(list)[p] = uint4_t{0u, 0u, 0u, 0u};
        for (int p = tid; p < LIST_STEPS * kListed; p += kPackThreads) list_column[p] = n;   // (row n of rhs reads as zeros)
    };
    clear_list();

    // the list: every wave's part of it lies behind those of the waves before (-1 is no third nonzero)
    auto goes_to_list = [](int code) { return code != -1 && (unsigned)code >= 0x80000000u; };
#pragma unroll
    for (int t = 0; t < KEPT; ++t)
        if (turn_at(t) < row_end) {
            kept[t] = look(kept[t], t);
            listed += __builtin_popcountll(__builtin_amdgcn_ballot_w64(goes_to_list(kept[t])));
        }
    for (int t = KEPT; turn_at(t) < row_end; ++t) listed += __builtin_popcountll(__builtin_amdgcn_ballot_w64(goes_to_list(look(fetch_column(t), t))));
    if (lane == 0) wave_count[wave] = listed;
    __syncthreads();
    if (bad) any_bad = 1;
    int count = 0, mine = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        mine += w < wave ? wave_count[w] : 0;
        count += wave_count[w];
    }
    // (of four nonzeros two are listed at most, so the lists of the units do not overlap; a pattern that is longer than it was
    // said to be does not fit)
    const int list_steps = (count + kListed - 1) / kListed, list_first = (start >> 6) + unit;
    const bool fits = list_first + list_steps <= capacity && list_steps <= ((stop - start) >> 6) + 1;
    auto list_place = [](int kk) { return 16 * ((kk >> 2) & 3) * 8 + (kk & 3) + (kk >= 16 ? 4 : 0); };   // a step's nonzero kk, row 0
    // rows of rhs are fetched by eight lanes each, four rows per lane: row 8 q + l by the lanes of eighth l
    auto column_place = [](int kk) { return (kk & 7) * 4 + (kk >> 3); };
    // what of a turn lies in [from, from + LIST_STEPS * 32) of the list, in LDS
    auto put_in_list = [&](int code, const PackedVector<V> &value, int &next, int from) __attribute__((always_inline)) {
        const bool to_list = goes_to_list(code);
        const uint64_t some = __builtin_amdgcn_ballot_w64(to_list);
        const int at = next - from + __builtin_amdgcn_mbcnt_hi((uint32_t)(some >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)some, 0));
        next += __builtin_popcountll(some);
        if (to_list && (unsigned)at < (unsigned)(LIST_STEPS * kListed)) {
            list_column[at / kListed * kListed + column_place(at % kListed)] = code & 0x3fffffff;
#pragma unroll
            for (int v = 0; v < V; ++v) list[at / kListed * (kListBytes / 2) + list_place(at % kListed) + (row * V + v) * 8] = value.at(v);
        }
    };
    auto write_list = [&](int from) __attribute__((always_inline)) {
        const int here = list_steps - from < LIST_STEPS ? list_steps - from : LIST_STEPS;
        const size_t at = (size_t)list_first + from;
        for (int p = tid; p < here * 64; p += kPackThreads)
            *reinterpret_cast<uint4_t *>(lists + at * kListBytes + p * 16) = reinterpret_cast<const uint4_t *>(list)[p];
        for (int p = tid; p < here * kListed; p += kPackThreads) list_columns[at * kListed + p] = list_column[p];
    };
    for (int first = 0; first < steps; first += chunk_steps) {
        const int here = steps - first < chunk_steps ? steps - first : chunk_steps;
        if (first > 0) {
            clear(here);
            __syncthreads();
        }
        int next = mine;
        auto put = [&](int code, const PackedVector<V> &value) __attribute__((always_inline)) {
            if (first == 0) put_in_list(code, value, next, 0);
            const int column = code & 0x3fffffff, step = (column >> 6) - first;
            if (code == -1 || goes_to_list(code) || (unsigned)step >= (unsigned)here) return;
            // groups of four: 8 h + 4 i + g of a step is number 8 h + 2 g + i to the instruction, which puts the rows of rhs
            // where the transposing reads of the second launch want them
            const int q = (column >> 2) & 15, group = (q & 8) | ((q & 3) << 1) | ((q >> 2) & 1), at = column & 3;
            const int slot = code >= (1 << 30) || at == 3 ? 1 : 0, quarter = group >> 2;
#pragma unroll
            for (int v = 0; v < V; ++v)
                operand[step * (kUnitBytes / 2) + (16 * quarter + row * V + v) * 8 + 2 * (group & 3) + slot] = value.at(v);
            const uint32_t bits = slot ? (uint32_t)(at ^ 3) << 2 : (uint32_t)at;
            if (bits) atomicXor(&place_bits[(step * ROWS + row) * 2 + (quarter >> 1)], bits << (16 * (quarter & 1) + 4 * (group & 3)));
        };
#pragma unroll
        for (int t = 0; t < KEPT; ++t)
            if (turn_at(t) < row_end) put(kept[t], kept_value[t]);
        for (int t = KEPT; turn_at(t) < row_end; ++t) {
            PackedVector<V> value;
            fetch(value, t);
            put(look(fetch_column(t), t), value);
        }
        __syncthreads();
        // (a list that does not fit starts nowhere: the second launch fetches four steps' columns from every list's start)
        if (first == 0 && tid == 0) units[unit] = UnitInfo{fits ? list_first : 0, fits ? list_steps : 0, any_bad || !fits, 0};
        for (int p = tid; p < here * 64; p += kPackThreads) {
            const long long at = (long long)block * steps + first + (p >> 6);
            *reinterpret_cast<uint4_t *>(packed + (at * kBlockUnits + unit_here) * kUnitBytes + lane * 16) = reinterpret_cast<const uint4_t *>(area)[p];
            const uint32_t word = place_bits[((p >> 6) * ROWS + (lane & 15) / V) * 2 + (lane >> 5)];
            reinterpret_cast<uint16_t *>(positions)[(at * kBlockUnits + unit_here) * 64 + lane] = (uint16_t)(word >> (lane & 16));
        }
        if (first + chunk_steps < steps) __syncthreads();
    }
    if (!fits) return;
    write_list(0);
    for (int from = LIST_STEPS; from < list_steps; from += LIST_STEPS) {
        __syncthreads();
        clear_list();
        __syncthreads();
        int next = mine;
        for (int t = 0; turn_at(t) < row_end; ++t) {
            PackedVector<V> value;
            fetch(value, t);
            put_in_list(look(fetch_column(t), t), value, next, from * kListed);
        }
        __syncthreads();
        write_list(from);
    }
}

// MI units x 64 columns per wave, WM x WN waves; operands of DEPTH steps in LDS.
template <int MI, int WM, int WN, int DEPTH>
struct PackedShape {
    static constexpr int WAVES = WM * WN, THREADS = 64 * WAVES, TM = kUnitRows * MI * WM, TN = 64 * WN;
    static constexpr int A_BYTES = TM * 64, P_BYTES = TM * 8, B_PITCH = TN * 2, B_BYTES = kStepColumns * B_PITCH;
    static constexpr int STEP = A_BYTES + P_BYTES + B_BYTES;
    static constexpr int A_LOADS = A_BYTES / 1024 / WAVES, B_LOADS = B_BYTES / 1024 / WAVES, LOADS = A_LOADS + B_LOADS + 1;   // of a wave and step
    // the lists: rows of rhs and operands of LIST_DEPTH steps of a wave, in the place of the steps; behind them a wave's columns
    // of four steps of every unit
    static constexpr int LIST_DEPTH = 3, LIST_STEP = kListed * 128 + kListBytes, LIST_AT_ONCE = 4;
    static constexpr int MAIN = DEPTH * STEP, AFTER = WAVES * LIST_DEPTH * LIST_STEP, COLUMNS = MAIN > AFTER ? MAIN : AFTER;
    static constexpr int AREA = COLUMNS + WAVES * MI * LIST_AT_ONCE * kListColumnBytes;
    static_assert(AREA <= 160 * 1024 - 512, "");
    static_assert(A_LOADS * 1024 * WAVES == A_BYTES && B_LOADS * 1024 * WAVES == B_BYTES && P_BYTES % 1024 == 0 && P_BYTES / 256 <= WAVES && TM % kBlockRows == 0, "");
    static_assert(TN == 128, "rows of rhs in LDS: eight pieces of 32 bytes");
};

template <int MI, int WM, int WN, int DEPTH>
__global__ void __launch_bounds__(64 * WM * WN, 2)
spmm_packed_kernel(int m, int V, int N, int n, int steps, int row_tiles, int column_tiles, const int *__restrict__ row_offsets,
                   const int *__restrict__ col_indices, const half_t *__restrict__ values, const half_t *__restrict__ rhs,
                   half_t *__restrict__ out, const unsigned char *__restrict__ packed, const unsigned char *__restrict__ positions,
                   const UnitInfo *__restrict__ units, const int *__restrict__ list_columns, const unsigned char *__restrict__ lists)
{
    using S = PackedShape<MI, WM, WN, DEPTH>;
    extern __shared__ __align__(16) unsigned char area[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int wm = wave / WN, wn = wave % WN;

    // An XCD takes a run of the tiles, sixteen columns of them wide: what its workgroups share meets in its L2.
    int rt, ct;
    {
        const int tiles = row_tiles * column_tiles, share = (tiles + 7) / 8;
        const int id = (int)(blockIdx.x & 7) * share + (int)(blockIdx.x >> 3);
        if ((int)(blockIdx.x >> 3) >= share || id >= tiles) return;
        const int wide = 16, band = id / (row_tiles * wide), first = band * wide;
        const int width = column_tiles - first < wide ? column_tiles - first : wide;
        const int in_band = id - band * row_tiles * wide;
        rt = in_band / width;
        ct = first + in_band % width;
    }
    const int block0 = rt * (S::TM / kBlockRows), unit0 = rt * (S::TM / kUnitRows) + wm * MI;   // the tile's first block, the wave's first unit

    // A step's operands: the wave's share of the packed values (16 KB of 8 KB per block), of their positions and of the rows
    // of rhs.  A row of rhs is eight pieces of 32 bytes, piece p at place p ^ (row % 8): transposing reads of eight rows then
    // touch every bank once.  Out of range (columns past the width, rows past the end) reads as zeros; steps past the end
    // are requested and not used (the workspace goes on for that long).
    constexpr unsigned A_STEP = kBlockUnits * kUnitBytes;
    const uint4_t a_from = buffer_of(packed + (size_t)block0 * steps * A_STEP, 0x7fffffffu);
    const uint4_t p_from = buffer_of(positions + (size_t)(block0 + wave / 4 % (S::TM / kBlockRows)) * steps * 1024 + wave % 4 * 256, 0x7fffffffu);
    const uint4_t b_from = buffer_of(rhs, (unsigned)((long long)n * N * 2));
    unsigned a_off[S::A_LOADS], b_off[S::B_LOADS];
#pragma unroll
    for (int p = 0; p < S::A_LOADS; ++p) {
        const int unit = wave * S::A_LOADS + p;
        a_off[p] = (unsigned)(unit / kBlockUnits) * (unsigned)steps * A_STEP + (unsigned)(unit % kBlockUnits * kUnitBytes + lane * 16);
    }
#pragma unroll
    for (int p = 0; p < S::B_LOADS; ++p) {
        const int row = (wave * S::B_LOADS + p) * 4 + (lane >> 4), piece = ((lane & 15) >> 1) ^ (row & 7);
        const int column = ct * S::TN + piece * 16 + (lane & 1) * 8;
        b_off[p] = column < N ? ((unsigned)row * (unsigned)N + (unsigned)column) * 2u : 0x80000000u;
    }
    const unsigned b_step = (unsigned)kStepColumns * (unsigned)N * 2u;
    const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void *)area;
    // (a quarter of a step's requests; PART < 0: all of them)
    auto request = [&](auto part, int s, int buffer) __attribute__((always_inline)) {
        constexpr int PART = decltype(part)::value;
        const unsigned to = lds + (unsigned)(buffer * S::STEP);
        if constexpr (PART <= 0)
            request_to_lds<4>(to + S::A_BYTES + wave % (S::P_BYTES / 256) * 256, p_from, (unsigned)(lane * 4), (unsigned)s * 1024u);
#pragma unroll
        for (int p = 0; p < S::A_LOADS; ++p)
            if (PART < 0 || PART == p) request_to_lds<16>(to + (wave * S::A_LOADS + p) * 1024, a_from, a_off[p], (unsigned)s * A_STEP);
#pragma unroll
        for (int p = 0; p < S::B_LOADS; ++p)
            if (PART < 0 || PART == 4 - S::B_LOADS + p) {
                request_to_lds<16>(to + S::A_BYTES + S::P_BYTES + (wave * S::B_LOADS + p) * 1024, b_from, b_off[p], 0u);
                b_off[p] += b_step;
            }
    };

    static_assert(MI == 4 || MI == 2, "");
    struct Fragments {
        half8_t a[MI];
        half16_t b[4];
        int places[MI];
    };
    Fragments fragments[2];
    typedef short short4_v __attribute__((ext_vector_type(4)));
    auto transposed = [&](const unsigned char *p) __attribute__((always_inline)) {   // four k of a column per lane
        return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_v *)p);
    };
    const unsigned a_take = (unsigned)(wm * MI * kUnitBytes + lane * 16);
    const unsigned p_take = (unsigned)(S::A_BYTES + wm * MI * 128 + lane * 2);
    unsigned b_take[4];
    {
        const int row = 4 * g + (c >> 2);
#pragma unroll
        for (int j = 0; j < 4; ++j) b_take[j] = (unsigned)(S::A_BYTES + S::P_BYTES + row * S::B_PITCH + ((4 * wn + j) ^ (row & 7)) * 32 + 8 * (c & 3));
    }
    // (a quarter of a step's fragments)
    auto take = [&](auto part, Fragments &to, int buffer) __attribute__((always_inline)) {
        constexpr int PART = decltype(part)::value;
        const unsigned char *const from = area + buffer * S::STEP;
        if constexpr (PART < MI) to.places[PART] = *reinterpret_cast<const uint16_t *>(from + p_take + PART * 128);
        if constexpr (PART < MI) to.a[PART] = *reinterpret_cast<const half8_t *>(from + a_take + PART * kUnitBytes);
        const unsigned char *const p = from + b_take[PART];
        typedef short short16_v __attribute__((ext_vector_type(16)));
        const short4_v w = transposed(p), x = transposed(p + 16 * S::B_PITCH), y = transposed(p + 32 * S::B_PITCH), z = transposed(p + 48 * S::B_PITCH);
        to.b[PART] = __builtin_bit_cast(half16_t, (short16_v){w[0], w[1], w[2], w[3], x[0], x[1], x[2], x[3],
                                                              y[0], y[1], y[2], y[3], z[0], z[1], z[2], z[3]});
    };
    float4_t acc[MI][4];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    // (a quarter of a step's products)
    auto multiply = [&](auto part, const Fragments &f) __attribute__((always_inline)) {
        constexpr int PART = decltype(part)::value, i = PART * MI / 4;
#pragma unroll
        for (int j = PART * MI % 4; j < PART * MI % 4 + MI; ++j) {
            acc[i][j] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(f.a[i], f.b[j], acc[i][j], f.places[i], 0, 0);
        }
    };
    // Before a step: the wave's own requests for the next one have arrived (LATER steps were requested since), its reads are
    // done; behind the barrier that holds for all.
    auto meet = [&](auto later) __attribute__((always_inline)) {
        constexpr int LEFT = decltype(later)::value * S::LOADS;
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LEFT) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // the lists of the wave's units: the first columns are on their way from here on
    int list_first[MI], list_left[MI], list_total = 0;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const UnitInfo info = units[unit0 + i];
        list_first[i] = __builtin_amdgcn_readfirstlane(info.first);
        list_left[i] = __builtin_amdgcn_readfirstlane(info.count);
        list_total += list_left[i];
        bad |= info.bad != 0;
    }
    const unsigned my_columns = (unsigned)(S::COLUMNS + wave * MI * S::LIST_AT_ONCE * kListColumnBytes);
    auto request_columns = [&]() __attribute__((always_inline)) {
        static_assert(S::LIST_AT_ONCE * kListColumnBytes == 512, "two requests per unit");
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const uint4_t from = buffer_of(list_columns + (size_t)list_first[i] * kListed, 0x7fffffffu);
            request_to_lds<4>(lds + my_columns + i * 512, from, (unsigned)(lane * 4), 0u);
            request_to_lds<4>(lds + my_columns + i * 512 + 256, from, (unsigned)(lane * 4), 256u);
        }
    };
    if (list_total > 0) request_columns();
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) request(std::integral_constant<int, -1>(), d, d);
    meet(std::integral_constant<int, DEPTH - 1>());
    take(std::integral_constant<int, 0>(), fragments[0], 0);
    take(std::integral_constant<int, 1>(), fragments[0], 0);
    take(std::integral_constant<int, 2>(), fragments[0], 0);
    take(std::integral_constant<int, 3>(), fragments[0], 0);
    // A quarter of a step: requests for step s + DEPTH, over step s, whose fragments every wave has; fragments of step s + 1 and
    // products of step s, reads in the shadow of products.  In quarters because a wave that makes all its requests at once
    // stands before the memory pipe, which takes sixteen cycles for each of the workgroup's forty, with its products undone.
    auto quarter = [&](auto number, auto part, int s) __attribute__((always_inline)) {
        constexpr int Q = decltype(number)::value;
        take(part, fragments[(Q + 1) % 2], (Q + 1) % DEPTH);
        multiply(part, fragments[Q % 2]);
#pragma unroll
        for (int q = 0; q < MI; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x100, (6 + MI - 1) / MI, 0);   // LDS reads
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                   // products
        }
        __builtin_amdgcn_sched_barrier(0);
        request(part, s + DEPTH, Q);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](auto number, int s) __attribute__((always_inline)) {
        meet(std::integral_constant<int, DEPTH - 2>());
        quarter(number, std::integral_constant<int, 0>(), s);
        quarter(number, std::integral_constant<int, 1>(), s);
        quarter(number, std::integral_constant<int, 2>(), s);
        quarter(number, std::integral_constant<int, 3>(), s);
    };
    static_assert(DEPTH == 4, "a turn of the loop goes once round the buffers, an even number of steps");
    for (int s = 0; s < steps; s += 4) {   // (a multiple of four)
        step(std::integral_constant<int, 0>(), s);
        step(std::integral_constant<int, 1>(), s + 1);
        step(std::integral_constant<int, 2>(), s + 2);
        step(std::integral_constant<int, 3>(), s + 3);
    }
    meet(std::integral_constant<int, 0>());   // (nothing is on its way to LDS any more)

    // The lists, up to four steps of every unit at a time: step t's operand and rows of rhs, gathered, go to LDS three steps
    // ahead.  (Every step has the same number of requests; past the end they are out of range, which fetches nothing.)
    const int col_wave = ct * S::TN + wn * 64;
    if (list_total > 0) {
        const unsigned mine = (unsigned)(wave * S::LIST_DEPTH * S::LIST_STEP);
        // (from the wave's first list on: those of its units lie within 2^20 + 4 steps, where all lists may take more than 4 GB)
        const int lists_at = list_first[0];
        const uint4_t operands_from = buffer_of(lists + (size_t)lists_at * kListBytes, 0x7fffffffu);
        for (bool first_time = true; list_total > 0; first_time = false) {
            if (!first_time) {
                request_columns();
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            }
            int end[MI], steps_now = 0;   // the units' steps one after the other: [end[i - 1], end[i])
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                steps_now += list_left[i] < S::LIST_AT_ONCE ? list_left[i] : S::LIST_AT_ONCE;
                end[i] = steps_now;
            }
            auto request_step = [&](int t, unsigned slot) __attribute__((always_inline)) {
                int unit = 0, begin = 0, first = list_first[0];
#pragma unroll
                for (int i = 1; i < MI; ++i)
                    if (t >= end[i - 1]) {
                        unit = i;
                        begin = end[i - 1];
                        first = list_first[i];
                    }
                const bool there = t < steps_now;
                const unsigned to = lds + mine + slot * S::LIST_STEP;
                const int4_t rows = *reinterpret_cast<const int4_t *>(area + my_columns + (unit * S::LIST_AT_ONCE + (there ? t - begin : 0)) * kListColumnBytes + (lane >> 3) * 16);
                request_to_lds<16>(to + kListed * 128, operands_from, there ? (unsigned)(first - lists_at + t - begin) * (unsigned)kListBytes + lane * 16 : 0x80000000u, 0u);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    // (pieces of 32 bytes: p of row r at place p ^ (r / 2 % 4))
                    const int row = 8 * q + (lane >> 3), column = col_wave + (((lane & 7) >> 1) ^ ((row >> 1) & 3)) * 16 + (lane & 1) * 8;
                    const unsigned off = there && column < N ? ((unsigned)rows[q] * (unsigned)N + (unsigned)column) * 2u : 0x80000000u;
                    request_to_lds<16>(to + q * 1024, b_from, off, 0u);
                }
            };
#pragma unroll
            for (int t = 0; t < S::LIST_DEPTH; ++t) request_step(t, t);
            unsigned slot = 0;
            for (int t = 0; t < steps_now; ++t) {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S::LIST_DEPTH - 1) * 5) : "memory");
                const unsigned char *const from = area + mine + slot * S::LIST_STEP;
                const half8_t a = *reinterpret_cast<const half8_t *>(from + kListed * 128 + lane * 16);
                half8_t b[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    typedef short short8_v __attribute__((ext_vector_type(8)));
                    const int row = 4 * g + (c >> 2);
                    const unsigned char *const p = from + row * 128 + (j ^ ((row >> 1) & 3)) * 32 + 8 * (c & 3);
                    const short4_v w = transposed(p), x = transposed(p + 16 * 128);
                    b[j] = __builtin_bit_cast(half8_t, (short8_v){w[0], w[1], w[2], w[3], x[0], x[1], x[2], x[3]});
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (read before it is written over)
                request_step(t + S::LIST_DEPTH, slot);
                slot = slot == S::LIST_DEPTH - 1 ? 0 : slot + 1;
                int unit = 0;
#pragma unroll
                for (int i = 1; i < MI; ++i) unit += t >= end[i - 1] ? 1 : 0;
#pragma unroll
                for (int i = 0; i < MI; ++i)
                    if (unit == i) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[j], acc[i][j], 0, 0, 0);
                    }
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            list_total = 0;
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int done = list_left[i] < S::LIST_AT_ONCE ? list_left[i] : S::LIST_AT_ONCE;
                list_first[i] += done;
                list_left[i] -= done;
                list_total += list_left[i];
            }
        }
    }

    // outputs: a unit at a time through LDS, whole segments of 64 columns per row
    {
        constexpr int PER_ROW = 64 * (int)sizeof(half_t) / 16, PITCH = 64 * (int)sizeof(half_t) + 16, ROUNDS = 16 * PER_ROW / 64;
        static_assert(16 * PITCH <= S::LIST_STEP, "");
        unsigned char *const mine = area + wave * S::LIST_DEPTH * S::LIST_STEP;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int unit_row = (unit0 + i) * kUnitRows;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x = acc[i][j][e];
                    bad |= x != x && unit_row + 4 * g + e < m && col_wave + 16 * j + c < N;
                    *reinterpret_cast<half_t *>(mine + (4 * g + e) * PITCH + (16 * j + c) * (int)sizeof(half_t)) = (half_t)x;
                }
            wave_lds_fence();
#pragma unroll
            for (int q = 0; q < ROUNDS; ++q) {
                const int at = q * 64 + lane, r = at / PER_ROW, column = at % PER_ROW * (16 / (int)sizeof(half_t));
                const uint4_t x = *reinterpret_cast<const uint4_t *>(mine + r * PITCH + at % PER_ROW * 16);
                if (unit_row + r < m && col_wave + column < N) *reinterpret_cast<uint4_t *>(out + (size_t)(unit_row + r) * N + col_wave + column) = x;
            }
            wave_lds_fence();
        }
    }
    if (__syncthreads_or(bad) == 0) return;

    // nonzero by nonzero: a wave per vector row and 64 columns, one step of 32 at a time
    int *const idx_s = reinterpret_cast<int *>(area + wave * stage_bytes<8>());
    half_t *const vec_s = reinterpret_cast<half_t *>(idx_s + kStep);
    const int tile_rows = S::TM / V, m_vec = m / V;
    for (int item = wave; item < tile_rows * WN; item += S::WAVES) {
        const int r = rt * tile_rows + item / WN, first_col = ct * S::TN + 64 * (item % WN) + 4 * c;
        if (r >= m_vec) break;
        const int beg = row_offsets[r], end = row_offsets[r + 1];
        float4_t sum[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[j] = float4_t{0.f, 0.f, 0.f, 0.f};
        for (int base = beg; base < end; base += kStep) {
            if (lane < kStep) {
                const int j = base + lane, jc = j < end ? j : end - 1;
                idx_s[lane] = col_indices[jc];
#pragma unroll
                for (int v = 0; v < 8; ++v) vec_s[v * kStep + lane] = v < V && j < end ? values[(size_t)jc * V + v] : (half_t)0.f;
            }
            wave_lds_fence();
            spmm_mfma_step<8, 4, true>(idx_s, vec_s, rhs, N, first_col < N ? (uint32_t)first_col : 0u, c, g, sum, [] {});
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

template <int V>
int launch_pack(int m_vec, int n, const PackedLayout &at, const int *row_offsets, const int *col_indices, const half_t *values,
                unsigned char *workspace, hipStream_t stream)
{
    const int chunks = (int)((at.steps + kPackSteps - 1) / kPackSteps), chunk_steps = (int)((at.steps + chunks - 1) / chunks);
    const int lds = pack_lds_bytes<V>(chunk_steps);
    const auto kernel = spmm_pack_kernel<V>;
    static std::atomic<unsigned long long> lds_allowed{0};
    const hipError_t attr = allow_large_lds(reinterpret_cast<const void *>(kernel), pack_lds_bytes<V>(kPackSteps), lds_allowed);
    if (attr != hipSuccess) return (int)attr;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((at.blocks + 7) / 8 * 64)), dim3(kPackThreads), lds, stream, m_vec, n, (int)at.blocks, (int)at.steps,
                       chunk_steps, (int)at.capacity, row_offsets, col_indices, values, workspace, workspace + at.positions,
                       reinterpret_cast<UnitInfo *>(workspace + at.units), reinterpret_cast<int *>(workspace + at.columns), workspace + at.lists);
    return (int)hipGetLastError();
}

template <int MI, int WM, int WN>
int launch_packed_shape(int m, int V, int k, int n, const PackedLayout &at, const int *row_offsets, const int *col_indices,
                        const half_t *values, const half_t *rhs, half_t *out, const unsigned char *workspace, hipStream_t stream)
{
    using S = PackedShape<MI, WM, WN, 4>;
    const long long row_tiles = ((long long)m + S::TM - 1) / S::TM, column_tiles = ((long long)k + S::TN - 1) / S::TN;
    const long long blocks = (row_tiles * column_tiles + 7) / 8 * 8;
    if (blocks > 0x7fffffffLL) return hipErrorNotSupported;
    const auto kernel = spmm_packed_kernel<MI, WM, WN, 4>;
    static std::atomic<unsigned long long> lds_allowed{0};
    const hipError_t attr = allow_large_lds(reinterpret_cast<const void *>(kernel), S::AREA, lds_allowed);
    if (attr != hipSuccess) return (int)attr;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(S::THREADS), S::AREA, stream, m, V, k, n, (int)at.steps, (int)row_tiles,
                       (int)column_tiles, row_offsets, col_indices, values, rhs, out, workspace, workspace + at.positions,
                       reinterpret_cast<const UnitInfo *>(workspace + at.units), reinterpret_cast<const int *>(workspace + at.columns),
                       workspace + at.lists);
    return (int)hipGetLastError();
}

}  // namespace

// Both launches as microseconds, fitted to 220 problems (256..4096 rows, 256..4608 columns, widths of 128..2048, 50..98 %, every V;
// profiles/spmm_packed_rule_survey.txt) to within 6 % (tiles of 256 rows) and 9 %: a step of a tile takes its time whatever
// else runs (LDS and the memory pipe of one CU), a listed nonzero of a unit a gather of its row for every tile.  The rule
// takes them for 20 of the survey's 440 choices: 18 are 1.14 to 2.3 times faster than what ran before, two level (3368 x 1801 x 992, V = 4,
// 80 %: 0.99 and 1.01); of the others 30 would gain more than 5 %, up to 1.86 times, mostly where rhs no longer fits an XCD's L2, which the
// others' estimate does not know.  The line lies 15 % on this side of that estimate: at the line, 2248 x 2742 x 1488, V = 1, 90 %: 44.3
// against 33.7 us.  Below 25 us the packing is
// too large a part of it: 1571 x 1116 x 1976, V = 1, 92 %: 20.8 against 22.5 us.
//
// The lists of uneven rows, or of columns in clusters, are many times those of even ones, and a wave goes through those of its units
// alone: 0.94 us per step of the fullest 64 rows (tiles of 256), 0.5 us of the fullest 32 (of 128), and packing a row beyond what a
// wave keeps 0.55 us per turn of 64 nonzeros and 0.27 us more for every further pass over it, which its unit's list asks for.  Fitted
// to 81 problems (4096 x 4096 x 2048 and less, even to Pareto rows; profiles/spmm_packed_uneven_survey.txt) within 4 % (tiles of 256) and 6 %.
// Of 320 choices drawn again 29 are packed, two of them slower (0.87 and 0.92 of the speed).  Gathering waits for its longest
// row too: 0.005 us per nonzero vector beyond two mean rows, 0.03 us on the fine-grained path where it fills the chip (a dense row
// among even ones, 4096 x 4096 x 2048, V = 4, 95 %: 187 us, 140 packed, 52 without it; 1148 x 4419 x 1808, V = 4, 90 %: 78 us, 125 packed).  4096 x 4096 x 2048, V = 4, 80 %:
// 67 us for even rows, 171 us (and 118 us as they run now) for log-normal rows of width 0.5, 364 us (124 us) for Pareto rows.
//
// The workspace grows with the matrix, whatever its sparsity, and those who call the operators did not ask for one: none beyond
// 1 GiB, which takes in what gains most (16384 x 16384 x 2048, V = 1, 95 %: 0.54 GB, 1.17 ms as gathered, 0.80 ms packed; 32768 x 16384 x
// 2048, V = 4, 90 %: 0.85 GB, 1.90 and 1.55 ms; refused: 32768 x 32768 x 1024, V = 8, 90 %: 1.45 GB, 1.82 and 1.59 ms).
constexpr long long kMostWorkspace = 1LL << 30;

int spmm_packed_choice(bool fine_grained, int m_vec, int k, int n, int vec_length, int nonzeros_vec, int longest_row_vec,
                       const PackedLists *lists)
{
    const Options &o = options();
    if (o.spmm_packed == 1) return 0;
    if (m_vec <= 0 || k <= 0 || k % 8 != 0 || n <= 0 || nonzeros_vec <= 0 || nonzeros_vec > (1 << 26) || ((long long)n + 1024) * k >= (1LL << 30) || k >= (1 << 24)) return 0;
    // (a tile's packed operands are addressed with 32-bit offsets; a launch has fewer than 2^32 threads: 64 per row for the packing, 512 per
    // tile of 128 x 128 for the product)
    if ((long long)m_vec * vec_length > (1 << 26) - 2048 || n > (1 << 22)) return 0;
    if (((long long)m_vec * vec_length / 128 + 2) * (k / 128 + 2) >= (1LL << 32) / 512) return 0;
    if (o.spmm_packed >= 2) return o.spmm_packed - 1;
    if (o.spmm_tile || o.spmm_waves || o.spmm_cols_per_lane || o.spmm_steps || o.spmm_pipe || o.spmm_gather || o.spmm_teams || o.spmm_blocks_per_wave || o.spmm_guard_waves)
        return 0;  // a launch shape of other kernels is asked for
    const double gather = spmm_gather_us(fine_grained, vec_length, nonzeros_vec, k);
    if (gather < 25 || spmm_packed_bytes(m_vec, vec_length, n, nonzeros_vec) > kMostWorkspace) return 0;
    double others = spmm_expected_us(fine_grained, m_vec, k, n, vec_length, nonzeros_vec, longest_row_vec);
    if (others < 25) return 0;
    const double m = (double)m_vec * vec_length, density = nonzeros_vec / ((double)m_vec * n), steps = 4 * std::ceil(n / 256.0);
    const double unit = (double)kUnitRows / vec_length * n * density;   // nonzero vectors, and those of them that are listed
    const double listed = (double)kUnitRows / vec_length * n / 4 * (4 * density * density * density * (1 - density) + 2 * density * density * density * density);
    const double wide = std::ceil(m / 256) * std::ceil(k / 128.0) / 256, narrow = std::ceil(m / 128) * std::ceil(k / 128.0) / 256;
    double wide_us = 11.8 + (0.498 * steps + 0.116 * listed) * std::ceil(wide) + 9.4 * wide + 0.19e-3 * unit;
    double narrow_us = 6.6 + (0.417 * steps + 0.043 * listed) * std::ceil(narrow) + 7.1 * narrow + 0.57e-3 * unit;
    const bool full = fine_grained && m_vec * std::ceil(k / 128.0) >= 16384;
    if (others >= gather) others += (full ? 0.03 : 0.005) * std::fmax(0.0, longest_row_vec - 2 * density * n);
    if (lists) {   // (nothing here makes packing look faster: the launch, which has no lists, takes what was found with them)
        // (what the fullest of 64 even rows takes: a fourth more than the mean, half a step of padding per unit)
        const double even = 1.25 * 4 * (listed / kListed + 0.5);
        const auto turns = [&](double row) { return std::fmax(0.0, std::ceil(row / (64 * vec_length)) - (vec_length <= 2 ? 8 : 4)); };
        const double more_turns = std::fmax(0.0, turns(longest_row_vec) - turns(1.25 * density * n));
        const double passes = std::fmax(0.0, std::ceil(lists->rows16 / (vec_length == 1 ? 16.0 : 8.0)) - 1);
        constexpr double kDoubt = 1.4;   // (the line below is drawn for even rows)
        const double packing = more_turns * (0.55 + 0.27 * passes);
        wide_us += kDoubt * (packing + 0.94 * std::fmax(0.0, lists->rows64 - even) * std::ceil(wide));
        narrow_us += kDoubt * (packing + 0.5 * std::fmax(0.0, lists->rows32 - even / 2) * std::ceil(narrow));
    }
    if (std::fmin(wide_us, narrow_us) > 1.15 * others) return 0;
    return wide_us <= narrow_us ? 1 : 2;
}

bool spmm_packed_lists(int m_vec, int vec_length, const int *row_offsets, const int *column_indices, PackedLists &most)
{
    const int unit_rows = kUnitRows / vec_length;
    most = {0, 0, 0};
    int two = 0, four = 0, falls = 0;
    for (int unit = 0; unit * (long long)unit_rows < m_vec; ++unit) {
        const int first = unit * unit_rows, behind = std::min(first + unit_rows, m_vec);
        int count = 0;
        for (int r = first; r < behind; ++r) {
            const int beg = row_offsets[r], end = row_offsets[r + 1];
            if (end - beg > 1) falls |= column_indices[beg + 1] <= column_indices[beg];
            for (int j = beg + 2; j < end; ++j) {
                falls |= column_indices[j] <= column_indices[j - 1];
                count += ((column_indices[j] ^ column_indices[j - 2]) & ~3) == 0;
            }
        }
        const int steps = (count + kListed - 1) / kListed;
        two = (unit & 1 ? two : 0) + steps;
        four = (unit & 3 ? four : 0) + steps;
        most = {std::max(most.rows16, steps), std::max(most.rows32, two), std::max(most.rows64, four)};
    }
    return !falls;
}

PackedLists spmm_packed_lists_bound(int m_vec, int n, int vec_length, int nonzeros_vec, int longest_row_vec)
{
    const double mean = nonzeros_vec / ((double)m_vec * n), longest = std::fmin(std::fmax((double)longest_row_vec / n, mean), 1.0);
    const double row = n / 4 * (4 * longest * longest * longest * (1 - longest) + 2 * longest * longest * longest * longest);
    const double others = row * (mean > 0 ? mean / longest : 0.0);
    const auto steps = [&](int rows) { return (int)((row + (rows / vec_length - 1) * others) / kListed + 0.5 * rows / kUnitRows); };
    return {steps(16), steps(32), steps(64)};
}

long long spmm_packed_bytes(int m_vec, int vec_length, int n, int nonzeros_vec)
{
    return PackedLayout((long long)m_vec * vec_length, n, nonzeros_vec).total;
}

int launch_spmm_packed(int shape, int m_vec, int vec_length, int k, int n, int nonzeros_vec, const int *row_offsets,
                       const int *col_indices, const half_t *values, const half_t *rhs, half_t *out, void *workspace, hipStream_t stream)
{
    const PackedLayout at((long long)m_vec * vec_length, n, nonzeros_vec);
    unsigned char *const ws = static_cast<unsigned char *>(workspace);
    int status;
    switch (vec_length) {
    case 1: status = launch_pack<1>(m_vec, n, at, row_offsets, col_indices, values, ws, stream); break;
    case 2: status = launch_pack<2>(m_vec, n, at, row_offsets, col_indices, values, ws, stream); break;
    case 4: status = launch_pack<4>(m_vec, n, at, row_offsets, col_indices, values, ws, stream); break;
    case 8: status = launch_pack<8>(m_vec, n, at, row_offsets, col_indices, values, ws, stream); break;
    default: return hipErrorInvalidValue;
    }
    if (status != hipSuccess) return status;
    const int m = m_vec * vec_length;
    switch (shape) {
    case 1: return launch_packed_shape<4, 4, 2>(m, vec_length, k, n, at, row_offsets, col_indices, values, rhs, out, ws, stream);
    case 2: return launch_packed_shape<2, 4, 2>(m, vec_length, k, n, at, row_offsets, col_indices, values, rhs, out, ws, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace vs
