// The combine of a forward step whose Y rows are in memory:
// out[o] = sum over the P splits (y, m) of output o, in the reference's order
// (DataTableColMajor.cpp:402-500), of Y[y] * main[m].
//
// What bounds it.  A step with P * Wo products per (vertex, coloring) far above
// its row widths is bound by LDS: each product takes a value of Y and one of the
// main row at places that the split list gives.  With a lane per output, one
// vertex at a time (the gathering kernels' own combine), a wavefront's reads
// fall on LDS banks at random and a third read fetches the split: some 13
// cycles of a CU per 64 products, and the wavefront gathers nothing meanwhile.
// Here 16 rows lie side by side in LDS, [value][row], and a thread owns four
// rows of an output: a split is read once for 4 products, and the four threads
// of an output read 64 consecutive bytes, so a read's groups of lanes meet on
// a bank a quarter of the time.  The quarters of a value's 64 bytes are
// exchanged by its place (lds_place), so that staging, in which consecutive
// lanes hold consecutive values of a row, writes without conflicts.
// Measured (12-vertex tree, R-MAT scale 20, 4 colorings): the step of 84 splits,
// 55 outputs, main rows of 462 values: 7.5 ms in k_runs beside its gather, 2.56
// here; of 10 splits, 462 outputs, main rows of 165: 6 ms in k_sub, 2.35 here,
// both 4.7-5.0 TB/s of rows read and written: the copy rate of the card.
#include "pg_kernels.hpp"

#include <algorithm>
#include <map>

namespace pgbsc {

namespace {

constexpr int kRows = kCombineRows;  // rows of a workgroup: four threads of four
static_assert(kRows == 16, "four quarters of four rows");

typedef float f32x4 __attribute__((ext_vector_type(4)));

// byte offset of quarter 0 of value i's rows; quarter q is at lds_place(i) ^ 16 q
__device__ __forceinline__ uint32_t lds_place(uint32_t i) { return i * 64u + ((i >> 2) & 3u) * 16u; }

// rows [it, it + 16) of a dense table of width w into LDS, zeros past n: a
// wavefront takes four rows, of every WAVES / 4-th 64 values
template <int WAVES>
__device__ __forceinline__ void stage_rows(unsigned char* to, const float* from, int64_t it, int64_t n, int w)
{
    const int q = (threadIdx.x >> 6) & 3, lane = (threadIdx.x & 63) + (threadIdx.x >> 8) * 64;
    constexpr int STEP = WAVES / 4 * 64;
    const float* row = from + (it + 4 * q) * w;
    bool ok[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) ok[s] = it + 4 * q + s < n;
    constexpr int U = 4;
    for (int c0 = lane; c0 < w; c0 += STEP * U) {
        f32x4 x[U];
#pragma unroll
        for (int t = 0; t < U; ++t)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int c = c0 + STEP * t;
                x[t][s] = ok[s] && c < w ? row[(int64_t)s * w + c] : 0.0f;
            }
#pragma unroll
        for (int t = 0; t < U; ++t) {
            const int c = c0 + STEP * t;
            if (c < w) *reinterpret_cast<f32x4*>(to + (lds_place((uint32_t)c) ^ (16u * q))) = x[t];
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_combine_rows(const float* y, const float* m, float* out,
                                                         const uint32_t* split, int64_t n, int Wy, int Wm, int Wo,
                                                         int P)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    unsigned char* s_y = smem_raw;                  // [Wy][16] floats
    unsigned char* s_m = s_y + (size_t)Wy * 64;     // [Wm][16]
    uint32_t* s_split = reinterpret_cast<uint32_t*>(s_m + (size_t)Wm * 64);  // [P][Wo]: places of y, of m << 16
    for (int i = threadIdx.x; i < P * Wo; i += kBlock) {
        const int r = i / P;
        const uint32_t p = split[i];
        s_split[(i - r * P) * Wo + r] = lds_place(p & 0xffffu) | lds_place(p >> 16) << 16;
    }
    const uint32_t q = threadIdx.x & 3u, q16 = 16u * q;
    for (int64_t it = (int64_t)blockIdx.x * kRows; it < n; it += (int64_t)gridDim.x * kRows) {
        __syncthreads();  // the split table is complete, the last rows are read
        stage_rows<kBlock / 64>(s_y, y, it, n, Wy);
        stage_rows<kBlock / 64>(s_m, m, it, n, Wm);
        __syncthreads();
        const int rows = (int)min((int64_t)4, n - it - 4 * (int64_t)q);
        for (int o = threadIdx.x >> 2; o < Wo; o += kBlock / 4) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            const uint32_t* sp = s_split + o;
            constexpr int U = 4;
            int j = 0;
            for (; j + U <= P; j += U) {
                f32x4 yy[U], mm[U];
#pragma unroll
                for (int t = 0; t < U; ++t) {
                    const uint32_t p = sp[(j + t) * Wo];
                    yy[t] = *reinterpret_cast<const f32x4*>(s_y + ((p & 0xffffu) ^ q16));
                    mm[t] = *reinterpret_cast<const f32x4*>(s_m + ((p >> 16) ^ q16));
                }
#pragma unroll
                for (int t = 0; t < U; ++t) {
                    const f32x4 prod = yy[t] * mm[t];
                    acc = acc + prod;
                }
            }
            for (; j < P; ++j) {
                const uint32_t p = sp[j * Wo];
                const f32x4 prod = *reinterpret_cast<const f32x4*>(s_y + ((p & 0xffffu) ^ q16)) *
                                   *reinterpret_cast<const f32x4*>(s_m + ((p >> 16) ^ q16));
                acc = acc + prod;
            }
            float* dst = out + (it + 4 * (int64_t)q) * Wo + o;
#pragma unroll
            for (int s = 0; s < 4; ++s)
                if (s < rows) dst[(int64_t)s * Wo] = acc[s];
        }
    }
}

__device__ __forceinline__ float node_add(float acc, float g, float r) { return __builtin_fmaf(g, r, acc); }
__device__ __forceinline__ double node_add(double acc, float g, float r) { return acc + (double)g * (double)r; }

constexpr int kNodeBlock = 512;

// The adjoint of the combine, for 16 rows: dY[x] = sum over split list x of
// G[o] * main[i], G_main[x] = sum over its list of G[o] * Y[i], each in list
// order, in Acc.  As k_combine_rows; the three tables' rows and both lists
// take some 80 KB, so two workgroups of eight wavefronts share a CU.  A
// wavefront takes 16 outputs at a time from a counter, the long lists (dY's)
// first: 4 of 84 terms and 11 of 28 leave eight wavefronts uneven by turns.
// Measured (12-vertex tree, R-MAT scale 20, 4 colorings): the step of 462, 165
// and 55 values 9.1 ms with a lane per output of 8 rows, 3.6 here; of 55, 462
// and 165 8.1 and 3.8 (the rows alone at the copy rate: 1.9).
template <typename Acc>
__global__ __launch_bounds__(kNodeBlock) void k_bwd_node_rows16(const NodeArgs<float> a)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ int s_next;
    const bool do_dy = a.part != 2, do_gm = a.part != 1;
    const int wm = do_dy ? a.Wm : 0, wy = do_gm ? a.Wy : 0;
    unsigned char* s_g = smem_raw;               // [Wo][16] floats
    unsigned char* s_m = s_g + (size_t)a.Wo * 64;  // [wm][16]
    unsigned char* s_y = s_m + (size_t)wm * 64;  // [wy][16]
    uint32_t* s_la = reinterpret_cast<uint32_t*>(s_y + (size_t)wy * 64);  // [Pa][Wy]: places of main, of G << 16
    const int la = do_dy ? a.Pa * a.Wy : 0, lm = do_gm ? a.Pm * a.Wm : 0;
    uint32_t* s_lm = s_la + la;  // [Pm][Wm]: places of Y, of G << 16
    for (int i = threadIdx.x; i < la; i += kNodeBlock) {
        const uint32_t p = a.by_auxT[i];
        s_la[i] = lds_place(p & 0xffffu) | lds_place(p >> 16) << 16;
    }
    for (int i = threadIdx.x; i < lm; i += kNodeBlock) {
        const uint32_t p = a.by_mainT[i];
        s_lm[i] = lds_place(p & 0xffffu) | lds_place(p >> 16) << 16;
    }
    const int64_t n = (int64_t)a.n_act * a.B;
    const int t_dy = do_dy ? (a.Wy + 15) / 16 : 0, t_all = t_dy + (do_gm ? (a.Wm + 15) / 16 : 0);
    const uint32_t q = threadIdx.x & 3u, q16 = 16u * q;
    const Acc scale = (Acc)a.scale;
    for (int64_t it = (int64_t)blockIdx.x * kRows; it < n; it += (int64_t)gridDim.x * kRows) {
        __syncthreads();  // the lists are complete, the last rows are read
        if (threadIdx.x == 0) s_next = 0;
        stage_rows<kNodeBlock / 64>(s_g, a.G, it, n, a.Wo);
        if (do_dy) stage_rows<kNodeBlock / 64>(s_m, a.Tm, it, n, a.Wm);
        if (do_gm) stage_rows<kNodeBlock / 64>(s_y, a.Y, it, n, a.Wy);
        __syncthreads();
        const int rows = (int)min((int64_t)4, n - it - 4 * (int64_t)q);
        for (;;) {
            int task = 0;
            if ((threadIdx.x & 63u) == 0) task = atomicAdd(&s_next, 1);
            task = __builtin_amdgcn_readfirstlane(task);
            if (task >= t_all) break;
            const bool is_dy = task < t_dy;
            const int w = is_dy ? a.Wy : a.Wm, P = is_dy ? a.Pa : a.Pm;
            const int x = (is_dy ? task : task - t_dy) * 16 + ((threadIdx.x & 63) >> 2);
            if (x >= w) continue;
            const uint32_t* list = (is_dy ? s_la : s_lm) + x;
            const unsigned char* rows_of = is_dy ? s_m : s_y;
            Acc acc[4] = {Acc(0), Acc(0), Acc(0), Acc(0)};
            constexpr int U = 4;
            int j = 0;
            for (; j + U <= P; j += U) {
                f32x4 gg[U], rr[U];
#pragma unroll
                for (int t = 0; t < U; ++t) {
                    const uint32_t p = list[(j + t) * w];
                    rr[t] = *reinterpret_cast<const f32x4*>(rows_of + ((p & 0xffffu) ^ q16));
                    gg[t] = *reinterpret_cast<const f32x4*>(s_g + ((p >> 16) ^ q16));
                }
#pragma unroll
                for (int t = 0; t < U; ++t)
#pragma unroll
                    for (int s = 0; s < 4; ++s) acc[s] = node_add(acc[s], gg[t][s], rr[t][s]);
            }
            for (; j < P; ++j) {
                const uint32_t p = list[j * w];
                const f32x4 rr = *reinterpret_cast<const f32x4*>(rows_of + ((p & 0xffffu) ^ q16));
                const f32x4 gg = *reinterpret_cast<const f32x4*>(s_g + ((p >> 16) ^ q16));
#pragma unroll
                for (int s = 0; s < 4; ++s) acc[s] = node_add(acc[s], gg[s], rr[s]);
            }
            float* dst = (is_dy ? a.dY : a.Gm) + (it + 4 * (int64_t)q) * w + x;
#pragma unroll
            for (int s = 0; s < 4; ++s)
                if (s < rows) dst[(int64_t)s * w] = (float)(acc[s] * scale);
        }
    }
}

template <typename Acc>
hipError_t launch_node_rows16(const NodeArgs<float>& a, size_t lds, int num_cus, hipStream_t st)
{
    static thread_local std::map<size_t, int> per_cu_cache;
    auto it = per_cu_cache.find(lds);
    if (it == per_cu_cache.end()) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_bwd_node_rows16<Acc>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)kNodeRows16Lds);
        int per_cu = 0;
        if (e == hipSuccess)
            e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_bwd_node_rows16<Acc>, kNodeBlock, lds);
        if (e != hipSuccess) return e;
        if (per_cu < 1) return hipErrorInvalidConfiguration;
        it = per_cu_cache.emplace(lds, per_cu).first;
    }
    const int64_t need = ((int64_t)a.n_act * a.B + kRows - 1) / kRows;
    const int grid = (int)std::min<int64_t>(need, (int64_t)it->second * num_cus);
    hipLaunchKernelGGL(k_bwd_node_rows16<Acc>, dim3(grid), dim3(kNodeBlock), lds, st, a);
    return hipGetLastError();
}

}  // namespace

size_t node_rows16_lds_bytes(const NodeArgs<float>& a)
{
    const bool do_dy = a.part != 2, do_gm = a.part != 1;
    return (size_t)64 * (a.Wo + (do_dy ? a.Wm : 0) + (do_gm ? a.Wy : 0)) +
           (size_t)4 * ((do_dy ? (size_t)a.Pa * a.Wy : 0) + (do_gm ? (size_t)a.Pm * a.Wm : 0));
}

hipError_t launch_bwd_node_rows16(const NodeArgs<float>& a, int num_cus, hipStream_t st)
{
    const size_t lds = node_rows16_lds_bytes(a);
    if (!a.G || !a.Tm || a.y_from_h || lds > kNodeRows16Lds || a.Wo >= 1024 || a.Wm >= 1024 || a.Wy >= 1024)
        return hipErrorInvalidValue;
    if ((int64_t)a.n_act * a.B <= 0) return hipSuccess;
    return a.sums32 ? launch_node_rows16<float>(a, lds, num_cus, st) : launch_node_rows16<double>(a, lds, num_cus, st);
}

size_t combine_rows_lds_bytes(int Wy, int Wm, int Wo, int P)
{
    return (size_t)64 * (Wy + Wm) + (((size_t)4 * P * Wo + 15) & ~(size_t)15);
}

hipError_t launch_combine_rows(const float* y, const float* m, float* out, const uint32_t* split, int64_t n, int Wy,
                               int Wm, int Wo, int P, int num_cus, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    if (Wy < 1 || Wm < 1 || Wy >= 1024 || Wm >= 1024) return hipErrorInvalidValue;
    const size_t lds = combine_rows_lds_bytes(Wy, Wm, Wo, P);
    static thread_local std::map<size_t, int> per_cu_cache;
    auto it = per_cu_cache.find(lds);
    if (it == per_cu_cache.end()) {
        int per_cu = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_combine_rows, kBlock, lds);
        if (e != hipSuccess) return e;
        if (per_cu < 1) return hipErrorInvalidConfiguration;
        it = per_cu_cache.emplace(lds, per_cu).first;
    }
    const int64_t need = (n + kRows - 1) / kRows;
    const int grid = (int)std::min<int64_t>(need, (int64_t)it->second * num_cus);
    hipLaunchKernelGGL(k_combine_rows, dim3(grid), dim3(kBlock), lds, st, y, m, out, split, n, Wy, Wm, Wo, P);
    return hipGetLastError();
}

}  // namespace pgbsc
