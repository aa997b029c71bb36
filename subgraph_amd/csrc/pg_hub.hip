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
// Scale 22's largest hub, 162,718 entries, went from 8.9 ms to 1.8 ms in the
// steps of the 12-vertex tree whose rows one wavefront holds.
//
// Lanes.  A lane owns one Y value.  Rows of 64 values and more take one
// coloring per wavefront (the neighbour's colour is then a scalar); narrower
// rows of several colorings are packed, 64 values over as many colorings as
// they span, and each lane reads its coloring's neighbour colours from LDS.
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
constexpr int kHubPackColors = 32;  // colorings a packed wavefront spans at most, plus one
// LDS bytes per entry of a packed batch's neighbour colours: an odd number of
// words, so the lanes' entries start in different banks
constexpr int kHubColorBytes = 36;
static_assert(kHubColorBytes > kHubPackColors, "a packed wavefront's colours fit");
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

// How a launch's Y values are dealt to wavefronts: unit q of a hub is 64
// values of one coloring, or (packed) `slots` of the hub's B * Wy values.
struct HubGeom {
    int n_big;         // hubs [0, n_big) take a whole workgroup per unit, the others a quarter
    int64_t big;       // workgroups of the big hubs
    int units;         // units per hub
    int per_coloring;  // units per coloring (not packed)
    int slots;         // values per unit (packed)
};

// dynamic LDS per workgroup: the index tables of its teams, then (packed) each
// wavefront's staged neighbour colours
__host__ __device__ constexpr size_t hub_tab_bytes(int k) { return (size_t)(k + 1) * 64 * 4; }

template <typename T, int NB, bool PACK>
__global__ __launch_bounds__(kHubWaves * 64) void k_hub_seq(const SubArgs<T> a, const HubGeom g)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    static_assert(NB <= 64, "a batch's entries sit one per lane");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool big = (int64_t)blockIdx.x < g.big;
    const int W = big ? kHubWaves : kHubSmallWaves;
    const int team = big ? 0 : wave / kHubSmallWaves;
    const int wv = big ? wave : wave - team * kHubSmallWaves;
    const int64_t unit =
        big ? (int64_t)blockIdx.x : g.big + ((int64_t)blockIdx.x - g.big) * kHubTeams + team;
    const int h = (int)(unit / g.units);
    const bool live = h < a.n_items;
    const int q = (int)(unit - (int64_t)h * g.units);
    const int B = a.B, Wy = a.Wy;
    const int v = a.item_base + (live ? h : 0);
    // the lane's Y value i of coloring b
    int b, i, b0 = 0, nc = 1;
    bool mine;
    if (PACK) {
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
    // lane, the colour of an entry past the list's end), [cu][lane]
    uint32_t* s_tab = reinterpret_cast<uint32_t*>(smem_raw) + (size_t)team * (a.k + 1) * 64;
    __shared__ TurnSum<T> sums[kHubTeams][64];
    TurnSum<T>& s_turn = sums[team][lane];
    unsigned char* s_col = smem_raw + kHubTeams * hub_tab_bytes(a.k) + (size_t)wave * 64 * kHubColorBytes;
    const uint32_t cv = a.colors[(int64_t)v * B + b];
    if (live) {
        const uint32_t set = mine ? hub_expand_bit(a.ymask[i], cv) : 0u;
        for (int cu = wv; cu <= a.k; cu += W) {
            uint32_t off = kNoValue;
            if (cu < a.k && ((set >> cu) & 1u))
                off = (uint32_t)(b * a.Wa + a.rank_tab[hub_squeeze_bit(set & ~(1u << cu), (uint32_t)cu)]) *
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
            unsigned char* to = s_col + lane * kHubColorBytes;
#pragma unroll
            for (int d = 0; d < kHubPackColors / 4 + 1; ++d)
                if (4 * d + 4 <= nc) *reinterpret_cast<uint32_t*>(to + 4 * d) = pd[d];
#pragma unroll
            for (int r = 0; r < 3; ++r)
                if (r < (nc & 3)) to[(nc & ~3) + r] = (unsigned char)pt[r];
            wave_sync();
        }
        if (t + W < nbat) meta(t + W);  // the next batch's ids, ahead of this one's rows
        uint32_t off[NB];
        if (PACK) {
            const unsigned char* from = s_col + (b - b0);
#pragma unroll
            for (int j = 0; j < NB; ++j) off[j] = s_tab[(uint32_t)from[j * kHubColorBytes] * 64 + lane];
        } else {
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                const uint32_t cu = (uint32_t)__builtin_amdgcn_readlane((int)cc, j);
                off[j] = s_tab[cu * 64 + lane];
            }
        }
        T x[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int u = __builtin_amdgcn_readlane(uc, j);
            x[j] = row_value<T>(a.aux + (int64_t)u * a.lda, rowbytes, off[j]);
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

template <typename T, int NB, bool PACK>
hipError_t launch_hub_seq_t(const SubArgs<T>& a, const HubGeom& g, hipStream_t st)
{
    const size_t lds = kHubTeams * hub_tab_bytes(a.k) + (PACK ? (size_t)kHubWaves * 64 * kHubColorBytes : 0);
    // a dispatch holds < 2^32 work-items: more hubs than that take another launch
    const int64_t per_launch = std::max<int64_t>(1, ((int64_t)1 << 21) / g.units);
    for (int64_t first = 0; first < a.n_items; first += per_launch) {
        SubArgs<T> s = a;
        s.item_base = a.item_base + (int)first;
        s.n_items = (int)std::min<int64_t>(per_launch, a.n_items - first);
        s.out = a.out + first * a.ldo;
        const int64_t n_big = std::min<int64_t>(std::max<int64_t>(g.n_big - first, 0), s.n_items);
        HubGeom sg = g;
        sg.big = n_big * g.units;
        const int64_t grid = sg.big + ((s.n_items - n_big) * g.units + kHubTeams - 1) / kHubTeams;
        hipLaunchKernelGGL((k_hub_seq<T, NB, PACK>), dim3((unsigned)grid), dim3(kHubWaves * 64), lds, st, s, sg);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

size_t hub_seq_lds_bytes(int k)
{
    const size_t fixed = kHubTeams * 64 * sizeof(TurnSum<double>);  // running sums and turns
    return fixed + kHubTeams * hub_tab_bytes(k) + (size_t)kHubWaves * 64 * kHubColorBytes;
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
    // packed where that saves a quarter of the units: a packed lane looks its
    // neighbour colours up in LDS, an unpacked one takes them as scalars, which
    // costs more than it saves at a tenth (FP32 steps of 165-value rows, 4
    // colorings, 11 units against 12: 3.96 ms packed, 3.80 ms not)
    g.slots = a.Wy == 1 ? kHubPackColors : 64;
    const int packed = (a.B * a.Wy + g.slots - 1) / g.slots;
    const bool pack = 4 * packed <= 3 * g.units;
    if (pack) g.units = packed;
    return pack ? launch_hub_seq_t<T, NB, true>(a, g, st) : launch_hub_seq_t<T, NB, false>(a, g, st);
}

template hipError_t launch_hub_seq<float>(const SubArgs<float>&, int, hipStream_t);
template hipError_t launch_hub_seq<double>(const SubArgs<double>&, int, hipStream_t);

}  // namespace pgbsc
