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
#include "pg_kernels.hpp"

#include <algorithm>
#include <map>

namespace pgbsc {

namespace {

constexpr int kStreamColors = 32;      // colorings of a wavefront at most
constexpr int kStreamColorBytes = 68;  // LDS bytes per coloring of a batch's colour pairs: an odd number of words
constexpr int kStreamRowLanes = 63;    // row values a wavefront loads at once; its last lane holds zero
constexpr int kXcds = 8;
constexpr uint32_t kStreamNoValue = 0xfffffff0u;  // a byte offset past every table: the load gives zero

__host__ __device__ constexpr size_t stream_tab_bytes(int k, int Wy) { return ((size_t)(k * k + 1) * Wy + 15) & ~(size_t)15; }

template <int NB>
__global__ __launch_bounds__(kBlock) void k_stream(const SubArgs<float> a, const int4* tiles, int n_tiles,
                                                   const uint8_t* local, int CB, int nch, uint32_t table_bytes)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    static_assert(NB <= 64, "a batch's entries sit one per lane");
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
    const uint32_t rowbytes = (uint32_t)a.lda * 4u;
    const __amdgpu_buffer_rsrc_t table =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.aux), 0, (int)table_bytes, 0x00027000);
    const int lane_coloring = lane / Wy;
    const uint8_t* tab = s_tab + (lane - lane_coloring * Wy);
    // a tile's chunks of colorings go to one XCD (workgroups are dealt to the 8
    // in turn), close in time: they share the lines of the neighbour colours
    // and those where two segments of a row meet
    const int64_t n_work = (int64_t)((n_tiles + kXcds - 1) / kXcds) * nch;
    const int64_t step = (int64_t)(gridDim.x / kXcds) * (kBlock / 64);
    for (int64_t work = (int64_t)(blockIdx.x / kXcds) * (kBlock / 64) + wave; work < n_work; work += step) {
        const int tile = (int)(work / nch) * kXcds + (int)(blockIdx.x % kXcds);
        const int b0 = (int)(work % nch) * CB;
        if (tile >= n_tiles) continue;
        const int nc = min(CB, B - b0);
        const int4 t4 = tiles[tile];  // first vertex, vertices, first entry, entries
        const int v0 = t4.x, e0 = t4.z, e1 = t4.z + t4.w;
        const bool mine = lane < nc * Wy;
        const int c = min(lane_coloring, nc - 1);
        const int shift = c * a.Wa * 4;
        const uint32_t place = lane < nc * a.Wa ? (uint32_t)(b0 * a.Wa + lane) * 4u : kStreamNoValue;
        const int nbat = (t4.w + NB - 1) / NB;
        // lane j < NB holds entry j of a batch; one past the tile reads its
        // first entry with colours that add nothing
        int um = 0, lv = 0, lv_next = 0;
        float wm = 1.0f;
        bool last = false;
        uint32_t pd[kStreamColors / 4];
        uint32_t pt[3];
        auto locate = [&](int t) {
            const int e = e0 + t * NB + lane;
            const int ec = e < e1 ? e : e0;
            lv = local[ec];
            lv_next = e + 1 < e1 ? (int)local[ec + 1] : -1;
        };
        auto meta = [&](int t) {  // after locate(t)
            const int e = e0 + t * NB + lane;
            const bool ok = lane < NB && e < e1;
            const int ec = ok ? e : e0;
            last = ok && lv_next != lv;
            um = (int)((uint32_t)a.col[ec] * rowbytes);
            wm = a.w && ok ? a.w[ec] : 1.0f;
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
        float acc = 0.0f;
        int v = v0;
        for (int t = 0; t < nbat; ++t) {
            const int uc = um;
            const float wc = wm;
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
            float x[NB];
#pragma unroll
            for (int j = 0; j < NB; ++j)
                x[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                    table, (int)place, __builtin_amdgcn_readlane(uc, j), 0));
            if (t + 1 < nbat) {
                meta(t + 1);  // the next batch's ids, behind this one's rows
                if (t + 2 < nbat) locate(t + 2);
            }
            const unsigned char* from = s_pair + c * kStreamColorBytes;
            // the lanes' values first, a group at a time, without a branch
            // between them: their LDS reads and permutes overlap
            constexpr int GR = 8;
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
                for (int j = 0; j < GR; ++j) at[j] = min((int)tab[__umul24((uint32_t)at[j], (uint32_t)Wy)] + shift, kStreamRowLanes * 4);
#pragma unroll
                for (int j = 0; j < GR; ++j)
                    x[g + j] = __int_as_float(__builtin_amdgcn_ds_bpermute(at[j], __float_as_int(x[g + j])));
                if (a.w)
#pragma unroll
                    for (int j = 0; j < GR; ++j)
                        x[g + j] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wc), g + j)) * x[g + j];
                const uint32_t e8 = (uint32_t)(ends >> g) & ((1u << GR) - 1u);
                if (e8 == 0) {
#pragma unroll
                    for (int j = 0; j < GR; ++j) acc = acc + x[g + j];
                } else {
#pragma unroll
                    for (int j = 0; j < GR; ++j) {
                        acc = acc + x[g + j];
                        if ((e8 >> j) & 1) {
                            if (mine) {
                                const float out =
                                    a.out_mode == OUT_EMA_SCALED ? (float)((double)acc * (double)a.scale) : acc;
                                a.out[(int64_t)v * a.ldo + b0 * Wy + lane] = out;
                                if (a.ykeep) a.ykeep[(int64_t)v * a.ldy + b0 * Wy + lane] = acc;
                            }
                            acc = 0.0f;
                            ++v;
                        }
                    }
                }
            }
            wave_sync();  // the pairs are read before the next batch's are written
        }
    }
}

constexpr int kStreamBatch = 48;

}  // namespace

int stream_colorings(const SubArgs<float>& a)
{
    return std::min({a.B, 64 / a.Wy, kStreamRowLanes / a.Wa, kStreamColors});
}

hipError_t launch_stream(const SubArgs<float>& a, const int4* tiles, int n_tiles, const uint8_t* local, int64_t n_rows,
                         int num_cus, hipStream_t st)
{
    if (n_tiles <= 0) return hipSuccess;
    const int64_t table_bytes = n_rows * a.lda * 4;
    if (a.out_mode != OUT_EMA && a.out_mode != OUT_EMA_SCALED) return hipErrorInvalidValue;
    if (a.Wy > 64 || a.Wa > kStreamRowLanes || a.k > kMaxK || !a.gidx || table_bytes > (int64_t)kStreamNoValue)
        return hipErrorInvalidValue;
    const int most = stream_colorings(a);
    const int nch = (a.B + most - 1) / most;
    const int CB = (a.B + nch - 1) / nch;
    const size_t lds = stream_tab_bytes(a.k, a.Wy) + (size_t)(kBlock / 64) * kStreamColors * kStreamColorBytes;
    static thread_local std::map<size_t, int> per_cu_cache;
    auto it = per_cu_cache.find(lds);
    if (it == per_cu_cache.end()) {
        int per_cu = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_stream<kStreamBatch>, kBlock, lds);
        if (e != hipSuccess) return e;
        if (per_cu < 1) return hipErrorInvalidConfiguration;
        it = per_cu_cache.emplace(lds, per_cu).first;
    }
    const int64_t need = ((int64_t)n_tiles * nch + kBlock / 64 - 1) / (kBlock / 64);
    const int64_t most_blocks = std::min<int64_t>(need, (int64_t)it->second * num_cus);
    const int grid = (int)((most_blocks + kXcds - 1) / kXcds) * kXcds;
    hipLaunchKernelGGL((k_stream<kStreamBatch>), dim3(grid), dim3(kBlock), lds, st, a, tiles, n_tiles, local, CB, nch,
                       (uint32_t)table_bytes);
    return hipGetLastError();
}

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
