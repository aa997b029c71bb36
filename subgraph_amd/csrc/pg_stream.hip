// Narrow neighbour rows of several colorings, streamed in list order.
//
// What bounds the gathering kernel (k_sub) there.  Its lanes read a row's
// values at permuted places, and a 64-lane load whose lanes are permuted takes
// the address unit 20 cycles of a CU where a contiguous one takes 5 (measured
// on rows in the L2; with a lane permute after it, 8).  R-MAT scale 20, the
// 7-vertex tree's 20-value step, 64 colorings: 34 cycles per 64 values, 3.4
// TB/s of rows.
//
// Here a wavefront owns up to 64 values of the vertices' rows: the Y values of
// as many colorings as fit.  It walks the lists of a tile of consecutive
// vertices as one stream of entries, NB rows in flight whatever the vertices'
// degrees: an entry's row segment (those colorings' values, contiguous) is one
// contiguous load, and a lane permute brings each lane the value it adds, from
// a table of the places by (vertex colour, neighbour colour) in LDS.  Where a
// vertex's list ends the sums go out and start again from zero: the reference's
// order (CSCGraph.hpp:254-307), so FP32 sums keep its rounding.
//
// Measured (R-MAT; k_sub, then this kernel): scale 20, 12-vertex tree, 4
// colorings, rows of 11 into 55 values 3.1 and 1.88 ms; scale 18, 5-path, 16
// colorings, rows of 4 and 6 0.61 and 0.42 ms; the 7-vertex tree's step above
// 10.3 and 9.27 ms.  That step is now bound by the memory behind the L2: 6.9
// TB/s of 128-byte lines, of which the 180-byte segments use two thirds (23
// cycles of a CU per 64 values; with a tile's chunks over all XCDs 10.0 ms).
// The others wait on latency and lane work: batches of 32 entries, which give
// more wavefronts, take 1-12% longer, of 56 the same; the values of a vertex
// added one by one under a branch instead of eight at a time, 5-30% longer.
// FP64, batches of 32: 7-vertex tree, scale 20, 16 colorings 15.1 -> 13.3 ms a
// call; 10-vertex, scale 18, 4 colorings 10.4 -> 10.2.  Its transposed gather
// with gradients stays with k_sub: 158-190 VGPRs here, 5-path, scale 18, 16
// colorings 5.39 ms a call by k_sub, 5.67 by this kernel.
#include "pg_kernels.hpp"

#include <algorithm>
#include <map>

namespace pgbsc {

namespace {

constexpr int kStreamColors = 32;      // colorings of a wavefront at most
constexpr int kStreamColorBytes = 68;  // LDS bytes per coloring of a batch's colour pairs: an odd number of words
constexpr int kStreamRowLanes = 63;    // row values a wavefront loads at once; its last lane holds zero
constexpr int kXcds = 8;
// rows in flight
template <typename T>
constexpr int kStreamBatch = sizeof(T) == 4 ? 48 : 32;
constexpr uint32_t kStreamNoValue = 0xfffffff0u;  // a byte offset past every table: the load gives zero

__host__ __device__ constexpr size_t stream_tab_bytes(int k, int Wy) { return ((size_t)(k * k + 1) * Wy + 15) & ~(size_t)15; }

// 64-bit values by their two halves
__device__ __forceinline__ double join(uint32_t lo, uint32_t hi)
{
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
__device__ __forceinline__ uint32_t low(double x) { return (uint32_t)__double_as_longlong(x); }
__device__ __forceinline__ uint32_t high(double x) { return (uint32_t)((uint64_t)__double_as_longlong(x) >> 32); }

template <int CTRL>
__device__ __forceinline__ float dpp(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}

__device__ __forceinline__ float lane_value(float x, int j)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), j));
}

__device__ __forceinline__ double lane_value(double x, int j)
{
    return join((uint32_t)__builtin_amdgcn_readlane((int)low(x), j), (uint32_t)__builtin_amdgcn_readlane((int)high(x), j));
}

// the value of lane at / 4
__device__ __forceinline__ float permuted(int at, float x)
{
    return __int_as_float(__builtin_amdgcn_ds_bpermute(at, __float_as_int(x)));
}

__device__ __forceinline__ double permuted(int at, double x)
{
    return join((uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)low(x)),
                (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)high(x)));
}

// the value at byte off + row of the table, zero past its end
template <typename T>
__device__ __forceinline__ T table_value(__amdgpu_buffer_rsrc_t table, uint32_t off, int row)
{
    if constexpr (sizeof(T) == 4) {
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(table, (int)off, row, 0));
    } else {
        typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
        const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(table, (int)off, row, 0);
        return join(v.x, v.y);
    }
}

// a's sums over lanes l and l ^ BIT (32 or 16) in the lanes without that bit,
// b's in those with it
template <int BIT>
__device__ __forceinline__ float swap_add(float a, float b)
{
    const auto r = BIT == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false)
                             : __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The sums over all 64 lanes of 16 values at once: lane l's result is the sum of
// value l / 4.  Each step adds two lanes and halves the values a lane carries
// (row rotation by 8, mirror of 8 lanes), then the quad's lanes.
__device__ __forceinline__ float lane_sums(const float (&p)[16], int lane)
{
    float h[8], q[4], r[2];
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = swap_add<32>(p[i], p[i + 8]);
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = swap_add<16>(h[i], h[i + 4]);
    const bool b3 = lane & 8, b2 = lane & 4;
#pragma unroll
    for (int i = 0; i < 2; ++i) r[i] = (b3 ? q[i + 2] : q[i]) + dpp<0x128>(b3 ? q[i] : q[i + 2]);
    float x = (b2 ? r[1] : r[0]) + dpp<0x141>(b2 ? r[0] : r[1]);
    x = x + dpp<0x4e>(x);
    return x + dpp<0xb1>(x);
}

// TG: the adjoint's transposed gather, which also takes the gradient of each
// entry's transpose, the dot of what the entry adds with the vertex's own row:
// grad[e] += sum over lanes of dy[v] * x, in FP32 over the wavefront's colorings
// (up to 64 values; the gradient gather adds up to 256), for 16 entries at a
// time by adds that leave each entry's sum in four lanes (lane_sums; a reduction
// of its own per entry would take six).  HUB: tiles are {vertex, first entry,
// end entry, output row}, parts of one list each.
template <typename T, int NB, bool TG, bool HUB>
__global__ __launch_bounds__(kBlock) void k_stream(const SubArgs<T> a, const int4* tiles, int n_tiles,
                                                   const uint8_t* local, int CB, int nch, uint32_t table_bytes)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    constexpr int GR = TG ? 16 : 8;  // entries whose values are brought to their lanes together
    constexpr int SHARE = 64 / GR;   // lanes that hold the same entry's lane_sums
    static_assert(NB <= 64 && NB % GR == 0, "a batch's entries sit one per lane");
    static_assert(NB / GR <= SHARE, "a lane keeps one of its groups' sums");
    static_assert(!TG || sizeof(T) == 4, "lane_sums adds 32-bit lanes");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int B = a.B, Wy = a.Wy, k = a.k;
    // four times the place in a coloring's row of the value that Y value i of a
    // vertex of colour cv takes from a neighbour of colour cu, [cv * k + cu][i]
    // (255: none); row k * k is none, the colour of an entry past the tile
    uint8_t* s_tab = smem_raw;
    unsigned char* s_pair = smem_raw + stream_tab_bytes(k, Wy) + (size_t)wave * kStreamColors * kStreamColorBytes;
    for (int x = threadIdx.x; x < (k * k + 1) * Wy; x += kBlock) {
        const int p = x / Wy;
        const int r = p < k * k ? a.gidx[p * a.Wy4 + (x - p * Wy)] : -1;
        s_tab[x] = (uint8_t)(r < 0 ? 255 : 4 * r);
    }
    __syncthreads();
    const uint32_t rowbytes = (uint32_t)a.lda * (uint32_t)sizeof(T);
    const __amdgpu_buffer_rsrc_t table =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a.aux), 0, (int)table_bytes, 0x00027000);
    const int lane_coloring = lane / Wy;
    const uint8_t* tab = s_tab + (lane - lane_coloring * Wy);
    // a tile's chunks of colorings go to one XCD (workgroups are dealt to the 8
    // in turn), close in time: they share the lines of the neighbour colours
    // and those where two segments of a row meet
    // (TG: in one wavefront, one after another, so that an entry's gradient adds
    // its chunks in a fixed order)
    const int apart = TG ? 1 : nch;
    const int64_t n_work = (int64_t)((n_tiles + kXcds - 1) / kXcds) * apart;
    const int64_t step = (int64_t)(gridDim.x / kXcds) * (kBlock / 64);
    for (int64_t work = (int64_t)(blockIdx.x / kXcds) * (kBlock / 64) + wave; work < n_work; work += step) {
        const int tile = (int)(work / apart) * kXcds + (int)(blockIdx.x % kXcds);
        const int b_first = (int)(work % apart) * CB;
        if (tile >= n_tiles) continue;
        int b0 = b_first;
        do {
            const int nc = min(CB, B - b0);
            const int4 t4 = tiles[tile];  // first vertex, vertices, first entry, entries
            const int v0 = t4.x, e0 = HUB ? t4.y : t4.z, e1 = HUB ? t4.z : t4.z + t4.w;
            const int v_last = HUB ? v0 : v0 + t4.y - 1;
            const bool mine = lane < nc * Wy;
            const int c = min(lane_coloring, nc - 1);
            const int shift = TG && !mine ? kStreamRowLanes * 4 : c * a.Wa * 4;  // (past the values: none)
            const uint32_t place = lane < nc * a.Wa ? (uint32_t)(b0 * a.Wa + lane) * (uint32_t)sizeof(T) : kStreamNoValue;
            const int nbat = (e1 - e0 + NB - 1) / NB;
            // lane j < NB holds entry j of a batch; one past the tile reads its
            // first entry with colours that add nothing
            int um = 0, lv = 0, lv_next = 0;
            T wm = T(1);
            bool last = false;
            uint32_t pd[kStreamColors / 4];
            uint32_t pt[3];
            auto locate = [&](int t) {
                if (HUB) return;
                const int e = e0 + t * NB + lane;
                const int ec = e < e1 ? e : e0;
                lv = local[ec];
                lv_next = e + 1 < e1 ? (int)local[ec + 1] : -1;
            };
            auto meta = [&](int t) {  // after locate(t)
                const int e = e0 + t * NB + lane;
                const bool ok = lane < NB && e < e1;
                const int ec = ok ? e : e0;
                last = ok && (HUB ? e + 1 == e1 : lv_next != lv);
                um = (int)((uint32_t)a.col[ec] * rowbytes);
                wm = a.w && ok ? a.w[ec] : T(1);
                const uint8_t* ep = a.ecol + (int64_t)ec * B + b0;
                const uint8_t* vp = a.colors + (int64_t)(v0 + lv) * B + b0;
                const uint32_t none = (uint32_t)(k * k);
#pragma unroll
                for (int d = 0; d < kStreamColors / 4; ++d)
                    if (4 * d + 4 <= nc) {
                        uint32_t x, y;
                        __builtin_memcpy(&x, ep + 4 * d, 4);
                        __builtin_memcpy(&y, vp + 4 * d, 4);
                        // four colour pairs at once: cv * k + cu < 256 carries into no neighbour
                        pd[d] = ok ? y * (uint32_t)k + x : none * 0x01010101u;
                    }
#pragma unroll
                for (int r = 0; r < 3; ++r)
                    if (r < (nc & 3)) pt[r] = ok ? (uint32_t)vp[(nc & ~3) + r] * (uint32_t)k + ep[(nc & ~3) + r] : none;
            };
            locate(0);
            meta(0);
            if (nbat > 1) locate(1);
            T acc = T(0);
            int v = v0;
            // TG: the lane's values of the own rows of v and of the vertex after it
            auto own_row = [&](int u) {
                return mine ? a.dy[(int64_t)min(u, v_last) * a.ldd + b0 * Wy + lane] : T(0);
            };
            T own = T(0), own_next = T(0);
            if (TG) {
                own = own_row(v0);
                own_next = own_row(v0 + 1);
            }
            for (int t = 0; t < nbat; ++t) {
                const int uc = um;
                const T wc = wm;
                const uint64_t ends = __ballot(last);
                unsigned char* to = s_pair + lane;
#pragma unroll
                for (int d = 0; d < kStreamColors / 4; ++d)
                    if (4 * d + 4 <= nc)
#pragma unroll
                        for (int r = 0; r < 4; ++r) to[(4 * d + r) * kStreamColorBytes] = (unsigned char)(pd[d] >> (8 * r));
#pragma unroll
                for (int r = 0; r < 3; ++r)
                    if (r < (nc & 3)) to[((nc & ~3) + r) * kStreamColorBytes] = (unsigned char)pt[r];
                wave_sync();
                T x[NB];
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    x[j] = table_value<T>(table, place, __builtin_amdgcn_readlane(uc, j));
                if (t + 1 < nbat) {
                    meta(t + 1);  // the next batch's ids, behind this one's rows
                    if (t + 2 < nbat) locate(t + 2);
                }
                const unsigned char* from = s_pair + c * kStreamColorBytes;
                T sums = T(0);
                // the lanes' values first, a group at a time, without a branch
                // between them: their LDS reads and permutes overlap
#pragma unroll
                for (int g = 0; g < NB; g += GR) {
                    int at[GR];
#pragma unroll
                    for (int j = 0; j < GR; j += 4) {
                        const uint32_t p4 = *reinterpret_cast<const uint32_t*>(from + g + j);
#pragma unroll
                        for (int r = 0; r < 4; ++r) at[j + r] = (int)((p4 >> (8 * r)) & 255u);
                    }
#pragma unroll
                    for (int j = 0; j < GR; ++j)
                        at[j] = min((int)tab[__umul24((uint32_t)at[j], (uint32_t)Wy)] + shift, kStreamRowLanes * 4);
#pragma unroll
                    for (int j = 0; j < GR; ++j)
                        x[g + j] = permuted(at[j], x[g + j]);
                    T p[GR];  // TG: of the values without their weights
                    if (!TG && a.w)
#pragma unroll
                        for (int j = 0; j < GR; ++j)
                            x[g + j] = lane_value(wc, g + j) * x[g + j];
                    auto scaled = [&](int j) {
                        if (!TG || !a.w) return x[g + j];
                        return lane_value(wc, g + j) * x[g + j];
                    };
                    const uint32_t group_ends = (uint32_t)(ends >> g) & ((1u << GR) - 1u);
                    if (group_ends == 0) {
#pragma unroll
                        for (int j = 0; j < GR; ++j) acc = acc + scaled(j);
                        if (TG)
#pragma unroll
                            for (int j = 0; j < GR; ++j) p[j] = own * x[g + j];
                    } else {
#pragma unroll
                        for (int j = 0; j < GR; ++j) {
                            acc = acc + scaled(j);
                            if (TG) p[j] = own * x[g + j];
                            if ((group_ends >> j) & 1) {
                                if (mine) {
                                    T out = acc;
                                    if (!TG && a.out_mode == OUT_EMA_SCALED) out = (T)((double)acc * (double)a.scale);
                                    const int64_t row = HUB ? t4.w : v;
                                    a.out[row * a.ldo + b0 * Wy + lane] = out;
                                    if (!TG && a.ykeep) a.ykeep[(int64_t)v * a.ldy + b0 * Wy + lane] = acc;
                                }
                                acc = T(0);
                                ++v;
                                if (TG && !HUB) {
                                    own = own_next;
                                    own_next = own_row(v + 1);
                                }
                            }
                        }
                    }
                    if constexpr (TG) {
                        const T s = lane_sums(p, lane);
                        if (lane % SHARE == g / GR) sums = s;
                    }
                }
                if constexpr (TG) {
                    const int j = lane % SHARE * GR + lane / SHARE;
                    const int e = e0 + t * NB + j;
                    if (j < NB && e < e1) (void)unsafeAtomicAdd(&a.grad[e], (double)sums);  // (returns nothing: no wait)
                }
                wave_sync();  // the pairs are read before the next batch's are written
            }
            b0 += CB;
        } while (TG && b0 < B);
    }
}

template <typename T, bool TG, bool HUB>
hipError_t launch_stream_t(const SubArgs<T>& a, const int4* tiles, int n_tiles, const uint8_t* local,
                           uint32_t table_bytes, int num_cus, hipStream_t st)
{
    const int most = stream_colorings(a.B, a.Wy, a.Wa);
    const int nch = (a.B + most - 1) / most;
    const int CB = (a.B + nch - 1) / nch;
    constexpr int NB = kStreamBatch<T>;
    const size_t lds = stream_tab_bytes(a.k, a.Wy) + (size_t)(kBlock / 64) * kStreamColors * kStreamColorBytes;
    static thread_local std::map<size_t, int> per_cu_cache;
    auto it = per_cu_cache.find(lds);
    if (it == per_cu_cache.end()) {
        int per_cu = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_stream<T, NB, TG, HUB>, kBlock, lds);
        if (e != hipSuccess) return e;
        if (per_cu < 1) return hipErrorInvalidConfiguration;
        it = per_cu_cache.emplace(lds, per_cu).first;
    }
    const int64_t need = ((int64_t)n_tiles * (TG ? 1 : nch) + kBlock / 64 - 1) / (kBlock / 64);
    const int64_t most_blocks = std::min<int64_t>(need, (int64_t)it->second * num_cus);
    const int grid = (int)((most_blocks + kXcds - 1) / kXcds) * kXcds;
    hipLaunchKernelGGL((k_stream<T, NB, TG, HUB>), dim3(grid), dim3(kBlock), lds, st, a, tiles, n_tiles, local, CB, nch,
                       table_bytes);
    return hipGetLastError();
}

}  // namespace

int stream_colorings(int B, int Wy, int Wa)
{
    return std::min({B, 64 / Wy, kStreamRowLanes / Wa, kStreamColors});
}

bool stream_fits(int64_t n_rows, int64_t row_bytes, int Wy, int Wa)
{
    return Wy >= 1 && Wy <= 64 && Wa >= 1 && Wa <= kStreamRowLanes && n_rows * row_bytes <= (int64_t)kStreamNoValue;
}

template <typename T>
hipError_t launch_stream(StreamMode mode, const SubArgs<T>& a, const int4* tiles, int n_tiles, const uint8_t* local,
                         int64_t n_rows, int num_cus, hipStream_t st)
{
    if (n_tiles <= 0) return hipSuccess;
    const int64_t row_bytes = (int64_t)a.lda * (int64_t)sizeof(T);
    if (a.k > kMaxK || !a.gidx || !stream_fits(n_rows, row_bytes, a.Wy, a.Wa)) return hipErrorInvalidValue;
    const uint32_t bytes = (uint32_t)(n_rows * row_bytes);
    if (mode == STREAM_FORWARD) {
        if (a.out_mode != OUT_EMA && a.out_mode != OUT_EMA_SCALED) return hipErrorInvalidValue;
        return launch_stream_t<T, false, false>(a, tiles, n_tiles, local, bytes, num_cus, st);
    }
    if constexpr (sizeof(T) == 4)
        if (a.dy && a.grad && (a.out_mode == OUT_Y || a.out_mode == OUT_PARTIAL))
            return mode == STREAM_TG ? launch_stream_t<T, true, false>(a, tiles, n_tiles, local, bytes, num_cus, st)
                                     : launch_stream_t<T, true, true>(a, tiles, n_tiles, local, bytes, num_cus, st);
    return hipErrorInvalidValue;
}

template hipError_t launch_stream<float>(StreamMode, const SubArgs<float>&, const int4*, int, const uint8_t*, int64_t, int,
                                         hipStream_t);
template hipError_t launch_stream<double>(StreamMode, const SubArgs<double>&, const int4*, int, const uint8_t*, int64_t,
                                          int, hipStream_t);

__global__ void k_local_ids(uint8_t* local, const int4* tiles, int n_tiles, const int32_t* rowptr)
{
    for (int t = blockIdx.x; t < n_tiles; t += gridDim.x) {
        const int4 q = tiles[t];
        for (int j = threadIdx.x; j < q.y; j += blockDim.x)
            for (int e = rowptr[q.x + j]; e < rowptr[q.x + j + 1]; ++e) local[e] = (uint8_t)j;
    }
}

hipError_t launch_local_ids(uint8_t* local, const int4* tiles, int n_tiles, const int32_t* rowptr, hipStream_t st)
{
    if (n_tiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_local_ids, dim3(std::min(n_tiles, 1 << 16)), dim3(64), 0, st, local, tiles, n_tiles, rowptr);
    return hipGetLastError();
}

}  // namespace pgbsc
