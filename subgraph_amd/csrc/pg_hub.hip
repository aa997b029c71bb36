// Hub rows of the forward neighbour sum in the reference's order.
//
// The reference adds a vertex's neighbour rows one after another, in column
// order, starting from zero (CSCGraph::spmmSplit, CSCGraph.hpp:254-307).  To
// reproduce its FP32 rounding each Y value must be one running sum over the
// whole neighbour list, so a hub of degree 163k (R-MAT scale 22) is a chain of
// 163k dependent adds per value.
//
// What bounds the chain.  The adds themselves are some 4 cycles each; the
// loads that feed them (entry ids, row addresses, the rows) cost ten
// instructions per entry and a memory latency per batch.  One wavefront doing
// both took 2.6 us per batch of 56 entries: 1.86 ms for the 39,881 entries of
// R-MAT scale 20's largest hub, and as much for the launch, whatever else it
// held.  Here several wavefronts of a workgroup share a hub's list: wavefront
// w takes the batches w, w + W, ..., has all of a batch's rows in registers
// before its turn comes, and in its turn only adds them to the running sums,
// which go from wavefront to wavefront through LDS.  The order of the
// additions is that of one wavefront; the loads of W batches overlap.  The
// same launch takes 0.18 ms (0.25 us per turn, of which the adds are 0.08 and
// the hand-over the rest; batches of 32 entries: 0.30 ms, of 40: 0.26, of 48:
// 0.21, of 60: 0.18; without the raised issue priority in the turn: 0.20).
// Scale 22's largest hub, 162,718 entries, went from 8.9 ms to 1.6-1.7 ms in
// the steps of the 12-vertex tree whose rows one wavefront holds.
//
// Lanes.  A lane owns one Y value.  Rows of 64 values and more take one
// coloring per wavefront (the neighbour's colour is then a scalar); narrower
// rows of several colorings are packed, 64 values over as many colorings as
// they span, and each lane reads its coloring's neighbour colours from LDS.
// Such lanes read a row at permuted places, 20 cycles of a CU per load against
// 5 for a contiguous one: where most lanes are used the rows are instead loaded
// whole and the values brought to their lanes by a permute (HUB_ROW).
//
// The result is the hub's Y row, stored as its partial row (one per hub); the
// finishing launch of the gathering kernel combines it with the main table.
#include "pg_kernels.hpp"

#include <algorithm>

namespace pgbsc {

namespace {

constexpr int kHubWaves = 16;      // wavefronts of a workgroup
// wavefronts that share a hub outside the big prefix: 2, 4 and 8 are within 4%
// of each other on every measured case (the launch is then bound by its loads)
constexpr int kHubSmallWaves = 4;
constexpr int kHubTeams = kHubWaves / kHubSmallWaves;
constexpr int kHubRowLanes = 63;    // row values a wavefront loads at once (ROW); its last lane holds zero
constexpr int kHubPackColors = 32;  // colorings a packed wavefront spans at most, plus one
// LDS bytes per coloring of a packed batch's neighbour colours, a byte per
// entry: an odd number of words, so the colorings start in different banks
constexpr int kHubColorBytes = 68;
constexpr int kHubColorsBytes = (kHubPackColors + 1) * kHubColorBytes;  // of a wavefront
constexpr uint32_t kNoValue = 0x7ffffff8u;  // a row offset past every row: the bounds-checked load gives zero

__device__ __forceinline__ uint32_t hub_expand_bit(uint32_t m, uint32_t c)
{
    return (m & ((1u << c) - 1u)) | ((m >> c) << (c + 1u));
}

__device__ __forceinline__ uint32_t hub_squeeze_bit(uint32_t m, uint32_t c)
{
    return (m & ((1u << c) - 1u)) | ((m >> (c + 1u)) << c);
}

template <typename T>
__device__ __forceinline__ T lane_value(T x, int j);

template <>
__device__ __forceinline__ float lane_value<float>(float x, int j)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), j));
}

template <>
__device__ __forceinline__ double lane_value<double>(double x, int j)
{
    const long long bits = __double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)bits, j);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(bits >> 32), j);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// the value at byte `off` of a row of `bytes` bytes (a multiple of the value
// size), zero past its end: the buffer load's own bounds check
template <typename T>
__device__ __forceinline__ T row_value(const T* row, int bytes, uint32_t off);

template <>
__device__ __forceinline__ float row_value<float>(const float* row, int bytes, uint32_t off)
{
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(row), 0, bytes, 0x00027000);
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}

template <>
__device__ __forceinline__ double row_value<double>(const double* row, int bytes, uint32_t off)
{
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(row), 0, bytes, 0x00027000);
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0);
    return __longlong_as_double((long long)(((uint64_t)v.y << 32) | v.x));
}

// A lane's running sum and the batch that it is complete before, in LDS
// (volatile pointers of the LDS address space: every access stays an LDS
// instruction, in program order, in which a wavefront's are done).
template <typename T>
struct TurnSum;

// FP32: one 64-bit word, read and written whole
template <>
struct TurnSum<float> {
    unsigned long long word;
    typedef __attribute__((address_space(3))) volatile unsigned long long lds_word;
    __device__ __forceinline__ void put(float s, int t)
    {
        *(lds_word*)&word = ((unsigned long long)(unsigned)t << 32) | __float_as_uint(s);
    }
    __device__ __forceinline__ int get(float& s)
    {
        const unsigned long long x = *(lds_word*)&word;
        s = __uint_as_float((unsigned)x);
        return (int)(x >> 32);
    }
};

// FP64: the sum before the turn where it is written, after it where it is read
template <>
struct TurnSum<double> {
    double sum;
    int turn, pad;
    typedef __attribute__((address_space(3))) volatile double lds_sum;
    typedef __attribute__((address_space(3))) volatile int lds_turn;
    __device__ __forceinline__ void put(double s, int t)
    {
        *(lds_sum*)&sum = s;
        *(lds_turn*)&turn = t;
    }
    __device__ __forceinline__ int get(double& s)
    {
        const int t = *(lds_turn*)&turn;
        s = *(lds_sum*)&sum;
        return t;
    }
};

// How a launch's Y values are dealt to wavefronts.
enum HubMode : int {
    HUB_GATHER = 0,  // unit: 64 values of one coloring
    HUB_PACK = 1,    // unit: `slots` of the hub's B * Wy values
    HUB_ROW = 2,     // unit: all values of `colorings` colorings, rows loaded whole and permuted
};

struct HubGeom {
    int n_big;         // hubs [0, n_big) take a whole workgroup per unit, the others a quarter
    int64_t big;       // workgroups of the big hubs
    int units;         // units per hub
    int per_coloring;  // units per coloring (not packed)
    int slots;         // values per unit (packed)
    int colorings;     // colorings per unit (row)
    bool unit_major;   // a unit of all hubs before the next unit, else a hub's units together
};

// dynamic LDS per workgroup: the index tables of its teams, then (packed) each
// wavefront's staged neighbour colours
__host__ __device__ constexpr size_t hub_tab_bytes(int k) { return (size_t)(k + 1) * 64 * 4; }

template <typename T, int NB, int MODE>
__global__ __launch_bounds__(kHubWaves * 64) void k_hub_seq(const SubArgs<T> a, const HubGeom g)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    static_assert(NB <= 64, "a batch's entries sit one per lane");
    static_assert(NB % 4 == 0, "colours are read four entries at a time");
    constexpr bool ROW = MODE == HUB_ROW, PACK = MODE != HUB_GATHER;
    static_assert(!ROW || sizeof(T) == 4, "rows are permuted by 32-bit lanes");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool big = (int64_t)blockIdx.x < g.big;
    const int W = big ? kHubWaves : kHubSmallWaves;
    const int team = big ? 0 : wave / kHubSmallWaves;
    const int wv = big ? wave : wave - team * kHubSmallWaves;
    // hub h, unit q of it, among the big hubs or the others
    const int64_t at = big ? (int64_t)blockIdx.x : ((int64_t)blockIdx.x - g.big) * kHubTeams + team;
    const int h0 = big ? 0 : g.n_big, n = big ? g.n_big : a.n_items - g.n_big;
    const bool live = at < (int64_t)n * g.units;
    const int per = g.unit_major ? n : g.units;
    const int outer = live ? (int)(at / per) : 0, inner = live ? (int)(at - (int64_t)outer * per) : 0;
    const int h = h0 + (g.unit_major ? inner : outer);
    const int q = g.unit_major ? outer : inner;
    const int B = a.B, Wy = a.Wy;
    const int v = a.item_base + (live ? h : 0);
    // the lane's Y value i of coloring b
    int b, i, b0 = 0, nc = 1;
    bool mine;
    if (ROW) {
        b0 = q * g.colorings;
        nc = min(g.colorings, B - b0);
        const int c = lane / Wy;
        mine = c < nc;
        i = lane - c * Wy;
        b = mine ? b0 + c : b0;
    } else if (PACK) {
        const int s0 = q * g.slots, s1 = min(s0 + g.slots, B * Wy);
        mine = s0 + lane < s1;
        const int s = mine ? s0 + lane : s0;
        b = s / Wy;
        i = s - b * Wy;
        b0 = s0 / Wy;
        nc = (s1 - 1) / Wy - b0 + 1;
    } else {
        b = q / g.per_coloring;
        i = (q - b * g.per_coloring) * 64 + lane;
        mine = i < Wy;
    }
    // per team: for each neighbour colour cu, the byte offset in a neighbour's
    // row of the value the lane adds (kNoValue: none; row k: none for any
    // lane, the colour of an entry past the list's end), [cu][lane]; ROW: four
    // times the lane that loads the value (the last lane, which holds zero: none)
    uint32_t* s_tab = reinterpret_cast<uint32_t*>(smem_raw) + (size_t)team * (a.k + 1) * 64;
    __shared__ TurnSum<T> sums[kHubTeams][64];
    TurnSum<T>& s_turn = sums[team][lane];
    unsigned char* s_col = smem_raw + kHubTeams * hub_tab_bytes(a.k) + (size_t)wave * kHubColorsBytes;
    const uint32_t cv = a.colors[(int64_t)v * B + b];
    if (live) {
        const uint32_t set = mine ? hub_expand_bit(a.ymask[i], cv) : 0u;
        for (int cu = wv; cu <= a.k; cu += W) {
            uint32_t off = ROW ? (uint32_t)kHubRowLanes * 4u : kNoValue;
            if (cu < a.k && ((set >> cu) & 1u))
                off = (uint32_t)((ROW ? b - b0 : b) * a.Wa + a.rank_tab[hub_squeeze_bit(set & ~(1u << cu), (uint32_t)cu)]) *
                      (uint32_t)sizeof(T);
            s_tab[cu * 64 + lane] = off;
        }
        if (wv == 0) s_turn.put(T(0), 0);
    }
    __syncthreads();
    if (!live) return;
    const int e0 = a.rowptr[v], e1 = a.rowptr[v + 1];
    const int nbat = (e1 - e0 + NB - 1) / NB;
    const int rowbytes = a.lda * (int)sizeof(T);
    // ROW: the lane's place in the segment of the unit's colorings
    const uint32_t place = lane < nc * a.Wa ? (uint32_t)(b0 * a.Wa + lane) * (uint32_t)sizeof(T) : kNoValue;
    // lane j < NB holds entry j of the batch; one past the end reads the
    // list's first entry with colour k, which adds nothing
    int um = 0;
    uint32_t cm = 0;
    T wm = T(1);
    uint32_t pd[kHubPackColors / 4 + 1];
    uint32_t pt[3];
    auto meta = [&](int t) {
        const int e = e0 + t * NB + lane;
        const bool ok = lane < NB && e < e1;
        const int ec = ok ? e : e0;
        um = a.col[ec];
        wm = a.w && ok ? a.w[ec] : T(1);
        const uint8_t* ep = a.ecol + (int64_t)ec * B;
        if (PACK) {
            ep += b0;
            const uint32_t none = (uint32_t)a.k * 0x01010101u;
#pragma unroll
            for (int d = 0; d < kHubPackColors / 4 + 1; ++d)
                if (4 * d + 4 <= nc) {
                    uint32_t x;
                    __builtin_memcpy(&x, ep + 4 * d, 4);
                    pd[d] = ok ? x : none;
                }
#pragma unroll
            for (int r = 0; r < 3; ++r)
                if (r < (nc & 3)) pt[r] = ok ? (uint32_t)ep[(nc & ~3) + r] : (uint32_t)a.k;
        } else {
            cm = ok ? (uint32_t)ep[b] : (uint32_t)a.k;
        }
    };
    if (wv < nbat) meta(wv);
    for (int t = wv; t < nbat; t += W) {
        const int uc = um;
        const uint32_t cc = cm;
        const T wc = wm;
        if (PACK) {
            unsigned char* to = s_col + lane;
#pragma unroll
            for (int d = 0; d < kHubPackColors / 4 + 1; ++d)
                if (4 * d + 4 <= nc)
#pragma unroll
                    for (int r = 0; r < 4; ++r) to[(4 * d + r) * kHubColorBytes] = (unsigned char)(pd[d] >> (8 * r));
#pragma unroll
            for (int r = 0; r < 3; ++r)
                if (r < (nc & 3)) to[((nc & ~3) + r) * kHubColorBytes] = (unsigned char)pt[r];
            wave_sync();
        }
        if (t + W < nbat) meta(t + W);  // the next batch's ids, ahead of this one's rows
        // the table's entries of the batch's entries j .. j + 3
        const unsigned char* from = s_col + (b - b0) * kHubColorBytes;
        auto tab_at = [&](int j, uint32_t (&at)[4]) {
            const uint32_t four = PACK ? *reinterpret_cast<const uint32_t*>(from + j) : 0u;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t cu = PACK ? (four >> (8 * r)) & 255u
                                         : (uint32_t)__builtin_amdgcn_readlane((int)cc, j + r);
                at[r] = s_tab[cu * 64 + lane];
            }
        };
        uint32_t off[ROW ? 1 : NB];
        if constexpr (!ROW)
#pragma unroll
            for (int j = 0; j < NB; j += 4) {
                uint32_t at[4];
                tab_at(j, at);
#pragma unroll
                for (int r = 0; r < 4; ++r) off[ROW ? 0 : j + r] = at[r];
            }
        T x[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int u = __builtin_amdgcn_readlane(uc, j);
            x[j] = row_value<T>(a.aux + (int64_t)u * a.lda, rowbytes, ROW ? place : off[ROW ? 0 : j]);
        }
        if constexpr (ROW)
#pragma unroll
            for (int j = 0; j < NB; j += 4) {
                uint32_t at[4];
                tab_at(j, at);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    x[j + r] = __int_as_float(__builtin_amdgcn_ds_bpermute((int)at[r], __float_as_int(x[j + r])));
            }
        // every row has arrived before the turn: vmcnt(0)
        __builtin_amdgcn_s_waitcnt(0x0f70);
        // The wavefront before this one is of the same workgroup and ends its
        // turn without waiting for any later one.  The next in line polls
        // without a pause and at a higher issue priority, since its adds are
        // what the whole list waits for.
        T acc;
        for (;;) {
            const int now = s_turn.get(acc);
            if (__all(now == t)) break;
            if (t - __builtin_amdgcn_readfirstlane(now) > 1) __builtin_amdgcn_s_sleep(1);
            else __builtin_amdgcn_s_setprio(3);
        }
        if (a.w) {
#pragma unroll
            for (int j = 0; j < NB; ++j) acc = acc + lane_value<T>(wc, j) * x[j];
        } else {
#pragma unroll
            for (int j = 0; j < NB; ++j) acc = acc + x[j];
        }
        if (t + 1 < nbat) {
            s_turn.put(acc, t + 1);
            __builtin_amdgcn_s_setprio(0);
        } else if (mine) {
            a.out[(int64_t)h * a.ldo + (int64_t)b * Wy + i] = acc;
        }
    }
}

template <typename T, int NB, int MODE>
hipError_t launch_hub_seq_t(const SubArgs<T>& a, const HubGeom& g, hipStream_t st)
{
    const size_t lds = kHubTeams * hub_tab_bytes(a.k) + (MODE != HUB_GATHER ? (size_t)kHubWaves * kHubColorsBytes : 0);
    // a dispatch holds < 2^32 work-items: more hubs than that take another launch
    const int64_t per_launch = std::max<int64_t>(1, ((int64_t)1 << 21) / g.units);
    for (int64_t first = 0; first < a.n_items; first += per_launch) {
        SubArgs<T> s = a;
        s.item_base = a.item_base + (int)first;
        s.n_items = (int)std::min<int64_t>(per_launch, a.n_items - first);
        s.out = a.out + first * a.ldo;
        const int64_t n_big = std::min<int64_t>(std::max<int64_t>(g.n_big - first, 0), s.n_items);
        HubGeom sg = g;
        sg.n_big = (int)n_big;
        sg.big = n_big * g.units;
        const int64_t grid = sg.big + ((s.n_items - n_big) * g.units + kHubTeams - 1) / kHubTeams;
        hipLaunchKernelGGL((k_hub_seq<T, NB, MODE>), dim3((unsigned)grid), dim3(kHubWaves * 64), lds, st, s, sg);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

size_t hub_seq_lds_bytes(int k)
{
    const size_t fixed = kHubTeams * 64 * sizeof(TurnSum<double>);  // running sums and turns
    return fixed + kHubTeams * hub_tab_bytes(k) + (size_t)kHubWaves * kHubColorsBytes;
}

template <typename T>
hipError_t launch_hub_seq(const SubArgs<T>& a, int n_big, hipStream_t st)
{
    if (a.n_items <= 0) return hipSuccess;
    if (a.K < 1 || a.k > kMaxK || !a.ymask || !a.rank_tab || a.out_mode != OUT_PARTIAL || n_big < 0 ||
        n_big > a.n_items || (int64_t)a.lda * (int64_t)sizeof(T) >= (int64_t)kNoValue)
        return hipErrorInvalidValue;
    constexpr int NB = sizeof(T) == 4 ? 56 : 32;
    HubGeom g{};
    g.n_big = n_big;
    g.per_coloring = (a.Wy + 63) / 64;
    g.units = a.B * g.per_coloring;
    // Wide rows: the wavefronts at work read the same 64 values' part of the rows,
    // of which the L2 holds more rows (462 values, R-MAT scale 20, 4 colorings:
    // 15.7 -> 13.3 ms; scale 22, one: 20.4 -> 19.2).  Narrower rows gain nothing
    // (126 and 165 values: within 1% at scales 18 and 20, scale 22 5.1 -> 5.4 ms).
    g.unit_major = g.per_coloring > 4;
    // Rows loaded whole where a unit's lanes are mostly used and the rows no
    // wider than the sums: k_hub_seq's launches of 15 -> 20 and 6 -> 15 values,
    // 64 colorings, R-MAT scale 20: 5.98 -> 5.73 and 3.97 -> 2.67 ms; of 11 -> 55,
    // scale 20 and 22: 1.32 -> 1.14, 1.84 -> 1.62; of 4 -> 6, 16 colorings, scale
    // 18: 0.28 -> 0.22.  With 20 lanes of 64 (15 -> 20, one coloring) 0.18 -> 0.21,
    // with 36 (9 -> 36, 4 colorings in 4 units against 3 packed) 0.34 -> 0.38: a
    // gather of few lanes is the cheaper load.
    if constexpr (sizeof(T) == 4)
        if (a.Wa <= a.Wy && a.Wy <= 64 && a.Wa <= kHubRowLanes) {
            const int most = std::min({a.B, 64 / a.Wy, kHubRowLanes / a.Wa, kHubPackColors});
            const int units = (a.B + most - 1) / most;
            if (a.B * a.Wy >= 40 * units) {
                g.units = units;
                g.colorings = (a.B + units - 1) / units;
                return launch_hub_seq_t<T, NB, HUB_ROW>(a, g, st);
            }
        }
    // packed where that saves a quarter of the units: a packed lane looks its
    // neighbour colours up in LDS, an unpacked one takes them as scalars, which
    // costs more than it saves at a tenth (FP32 steps of 165-value rows, 4
    // colorings, 11 units against 12: 3.96 ms packed, 3.80 ms not)
    g.slots = a.Wy == 1 ? kHubPackColors : 64;
    const int packed = (a.B * a.Wy + g.slots - 1) / g.slots;
    const bool pack = 4 * packed <= 3 * g.units;
    if (pack) g.units = packed;
    return pack ? launch_hub_seq_t<T, NB, HUB_PACK>(a, g, st) : launch_hub_seq_t<T, NB, HUB_GATHER>(a, g, st);
}

template hipError_t launch_hub_seq<float>(const SubArgs<float>&, int, hipStream_t);
template hipError_t launch_hub_seq<double>(const SubArgs<double>&, int, hipStream_t);

}  // namespace pgbsc
