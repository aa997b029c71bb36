// The root's neighbour sum in the reference's order, below the hubs.
//
// A root whose main child is a leaf has one Y value per vertex and coloring:
// each entry adds one value of the neighbour's row.  The gathering kernel
// (k_sub) gives a vertex a team of 8 lanes of which one works, four loads in
// flight: on R-MAT scale 16 its longest list below the hubs, 512 entries, took
// 56 us, the whole launch's time.  Here a workgroup takes a tile, consecutive
// vertices of up to 1,024 entries in all: a thread per entry loads the entry's
// value into LDS, then a thread per vertex adds its values one after another,
// in list order from zero (the reference's order, CSCGraph.hpp:254-307).  The
// loads of a tile wait for nothing but their ids, and bound the launch: one
// line per entry and coloring.
// Measured, one coloring: scale 16, 3-path, 56 -> 11 us; scale 20, 7-vertex
// tree, 136 -> 65 us; four colorings, scale 18, 10-vertex tree, 180 -> 63 us
// (FP64 205 -> 88).
#include "pg_kernels.hpp"

#include <algorithm>

namespace pgbsc {

namespace {

// C: colorings taken together (their values of one entry share its lines)
template <typename T, int C>
__global__ __launch_bounds__(kBlock) void k_root_seq(const SubArgs<T> a, const int4* tiles, int n_tiles)
{
    constexpr int R = 4;  // values a thread loads at a time
    __shared__ T s_x[kRootTileEntries * C];
    __shared__ int s_u[kRootTileEntries];
    __shared__ uint8_t s_lv[kRootTileEntries];
    __shared__ int s_rp[kRootTileVertices + 1];
    const int tid = threadIdx.x;
    const int B = a.B;
    for (int tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const int4 t = tiles[tile];  // first vertex, vertices, first entry, entries
        const int v0 = t.x, nv = t.y, e0 = t.z, ne = t.w;
        __syncthreads();  // the tile before is done
        for (int j = tid; j <= nv; j += kBlock) s_rp[j] = a.rowptr[v0 + j] - e0;
        T carry = T(0);  // a lone vertex may have more entries than a tile holds
        for (int b0 = 0; b0 < B; b0 += C) {
            const int nc = min(C, B - b0);
            // (once for a tile without entries: its vertices' sums are zero)
            int w0 = 0;
            do {
                const int nw = min(kRootTileEntries, ne - w0);
                __syncthreads();
                for (int e = tid; e < nw; e += kBlock) {
                    s_u[e] = a.col[e0 + w0 + e];
                    int lo = 0, hi = nv;  // the entry's vertex: the last whose list begins at or before it
                    while (hi - lo > 1) {
                        const int mid = (lo + hi) >> 1;
                        if (s_rp[mid] <= w0 + e) lo = mid;
                        else hi = mid;
                    }
                    s_lv[e] = (uint8_t)lo;
                }
                if (C > 1) __syncthreads();  // (one coloring: a thread reads back only its own entries)
                for (int p0 = tid; p0 < nw * C; p0 += R * kBlock) {
                    int idx[R];
                    T x[R];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const int p = min(p0 + r * kBlock, nw * C - 1 - (nw * C - 1 - tid) % kBlock);
                        const int e = p / C, b = b0 + min(p % C, nc - 1);
                        const int64_t eb = (int64_t)(e0 + w0 + e) * B + b;
                        const int cv = a.colors[(int64_t)(v0 + s_lv[e]) * B + b];
                        idx[r] = a.gidx[(cv * a.k + a.ecol[eb]) * a.Wy4];
                        x[r] = a.aux[(int64_t)s_u[e] * a.lda + (int64_t)b * a.Wa + (idx[r] < 0 ? 0 : idx[r])];
                    }
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const int p = p0 + r * kBlock;
                        const T val = idx[r] < 0 ? T(0) : x[r];
                        if (p < nw * C) s_x[p] = a.w ? a.w[e0 + w0 + p / C] * val : val;
                    }
                }
                __syncthreads();
                for (int p = tid; p < nv * C; p += kBlock) {
                    const int j = p / C, c = p % C;
                    if (c >= nc) continue;
                    T acc = w0 ? carry : T(0);
                    int e = nv > 1 ? s_rp[j] : 0;
                    const int e1 = nv > 1 ? s_rp[j + 1] : nw;
                    for (; e + 8 <= e1; e += 8) {
                        T y[8];
#pragma unroll
                        for (int r = 0; r < 8; ++r) y[r] = s_x[(e + r) * C + c];
#pragma unroll
                        for (int r = 0; r < 8; ++r) acc = acc + y[r];
                    }
                    for (; e < e1; ++e) acc = acc + s_x[e * C + c];
                    carry = acc;
                    // f32 product y * 1, widened (DataTableColMajor.cpp:396)
                    if (w0 + nw >= ne) a.root_vals[(int64_t)(b0 + c) * a.n_root + v0 + j] = (double)acc;
                }
                w0 += kRootTileEntries;
            } while (w0 < ne);
        }
    }
}

}  // namespace

template <typename T>
hipError_t launch_root_seq(const SubArgs<T>& a, const int4* tiles, int n_tiles, int num_cus, hipStream_t st)
{
    if (n_tiles <= 0) return hipSuccess;
    if (a.Wy != 1 || a.out_mode != OUT_ROOT || a.main || !a.gidx || a.ykeep) return hipErrorInvalidValue;
    const int grid = std::min(n_tiles, num_cus * 8);
    if (a.B == 1) hipLaunchKernelGGL((k_root_seq<T, 1>), dim3(grid), dim3(kBlock), 0, st, a, tiles, n_tiles);
    else hipLaunchKernelGGL((k_root_seq<T, 4>), dim3(grid), dim3(kBlock), 0, st, a, tiles, n_tiles);
    return hipGetLastError();
}

template hipError_t launch_root_seq<float>(const SubArgs<float>&, const int4*, int, int, hipStream_t);
template hipError_t launch_root_seq<double>(const SubArgs<double>&, const int4*, int, int, hipStream_t);

}  // namespace pgbsc
