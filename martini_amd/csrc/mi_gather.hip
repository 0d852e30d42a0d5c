// What stands around the gather: the reduction of split cells' partial tiles,
// the kernel weight tables, and the entry points that evaluate kernel
// integrals and spectra by themselves.
#include <hip/hip_runtime.h>

#include <mutex>

#include "mi_device.h"
#include "mi_internal.h"
#include "mi_tile.h"

namespace mi {

// Sums the partial tiles of each split cell in item order, in FP64 (their sum
// then costs one rounding: 1.3e-7 -> 0.8e-7 of error on 1e4 particles in 400
// items), and adds them to the cube.  Block (cell, part): 256 threads x 4 voxels cover four 1 KiB
// sub-tiles of the CELL_VOXELS = 16384-voxel tile, one per wave.  A wave reads
// the masks of 64 items at a time, one per lane, and then only the sub-tiles
// that their items wrote, RED_DEEP loads in flight (1e6 particles, MFMA: 28 us;
// 39 with the masks read item by item, 31 with four loads in flight);
// voxels no item wrote keep the cube's value.
constexpr int RED_PARTS = CELL_VOXELS / (NT * 4);
constexpr int RED_DEEP = 8;

__global__ __launch_bounds__(NT) void k_reduce(const uint32_t* __restrict__ item_off,
                                               const uint32_t* __restrict__ multi_off,
                                               const uint32_t* __restrict__ status, Grid g,
                                               const float* __restrict__ partials,
                                               const uint64_t* __restrict__ part_masks,
                                               float* __restrict__ cube) {
    if (status[ST_OVERFLOW]) return;
    const int cell = blockIdx.x / RED_PARTS;
    const int part = blockIdx.x - cell * RED_PARTS;
    const uint32_t ni = item_off[cell + 1] - item_off[cell];
    if (ni <= 1) return;
    const size_t tile = (size_t)CELL_VOXELS / 4;  // float4 per partial tile
    const float4* base = reinterpret_cast<const float4*>(partials) + (size_t)multi_off[cell] * tile;
    const uint64_t* mk = part_masks + multi_off[cell];
    const int v4 = part * NT + threadIdx.x;  // float4 index within the tile
    // v4 = (sub-tile * SUB_CH + channel) * 4 + float4 within the 16 pixels
    static_assert(TILE_Y == 16 && SUB_CH == 16 && NT % 64 == 0, "one sub-tile per wave");
    const int sub = v4 >> 6;  // row * blocks + block, the same in a wave
    const int nblk = (1 << g.cb_shift) / SUB_CH;
    const int prow = sub / nblk, jl = (v4 & 3) * 4;
    const int cl = (sub - prow * nblk) * SUB_CH + ((v4 >> 2) & 15);
    const int bit = sub_bit(g.tx_shift, prow, sub - prow * nblk);
    const float4* src = base + v4;
    const uint32_t lane = threadIdx.x & 63;
    double s0[4] = {0.0, 0.0, 0.0, 0.0};
    uint64_t seen = 0u;
    for (uint32_t q0 = 0; q0 < ni; q0 += 64) {
        uint64_t set = __ballot(q0 + lane < ni && ((mk[q0 + lane] >> bit) & 1u));
        seen |= set;
        const float4* p = src + q0 * tile;
        while (set) {
            float4 v[RED_DEEP];
            int n = 0;
#pragma unroll
            for (int k = 0; k < RED_DEEP; ++k) {
                if (!set) break;  // uniform
                v[k] = p[(size_t)__builtin_ctzll(set) * tile];
                set &= set - 1u;
                n = k + 1;
            }
#pragma unroll
            for (int k = 0; k < RED_DEEP; ++k) {
                if (k >= n) break;
                s0[0] += (double)v[k].x;
                s0[1] += (double)v[k].y;
                s0[2] += (double)v[k].z;
                s0[3] += (double)v[k].w;
            }
        }
    }
    if (!seen) return;
    const CellPos cp = cell_pos(cell, g);
    const int i = cp.x0 + prow, j = cp.y0 + jl, c = cp.c0 + cl;
    if (i >= g.nx || c >= g.nc) return;
    float* dst = cube + ((size_t)i * g.ny + j) * g.nc + c;
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (j + u < g.ny) {
            float& v = dst[(size_t)u * g.nc];
            v = (float)((double)v + s0[u]);
        }
}

// The weight tables are constant data (the FP64 closed forms of the four
// tabulated kernels), so each device holds one copy, filled on first use.
__device__ float4 g_wtab[WTAB_KERNELS * WTAB_N];

__global__ void k_fill_wtab(float4* __restrict__ tab) { fill_wtab(tab); }

hipError_t weight_table(hipStream_t s, const float4** out) {
    static std::mutex mu;
    static const float4* table[MAX_DEVICES] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mu);
    if (table[dev] == nullptr) {
        // First use on this device: fill on the caller's stream and wait for it,
        // so that work on any stream may read the table afterwards.
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(g_wtab));
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_fill_wtab, dim3((WTAB_KERNELS * WTAB_N + 255) / 256), dim3(256), 0, s,
                           static_cast<float4*>(p));
        e = hipGetLastError();
        if (e != hipSuccess) return e;
        e = hipStreamSynchronize(s);
        if (e != hipSuccess) return e;
        table[dev] = static_cast<const float4*>(p);
    }
    *out = table[dev];
    return hipSuccess;
}

__global__ void k_weights(int kind, float gt, float ginv, const float* __restrict__ dx,
                          const float* __restrict__ dy, const float* __restrict__ h,
                          const float4* __restrict__ wtab, float* __restrict__ out, int64_t n) {
    int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) out[k] = pixel_weight(kind, (double)dx[k], (double)dy[k], h[k], gt, ginv, wtab);
}

__global__ void k_spectra(const mi_particle* __restrict__ P, int64_t n, mi_cube_desc d,
                          float* __restrict__ out) {
    const int nc = d.nc;
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n * nc) return;
    int64_t p = e / nc;
    int c = (int)(e - p * nc);
    out[e] = channel_flux(P[p], c, d);
}

hipError_t reduce_partials(const Grid& g, char* ws, const Layout& L, float* d_cube,
                           hipStream_t s) {
    hipLaunchKernelGGL(k_reduce, dim3((unsigned)(g.ncells * RED_PARTS)), dim3(NT), 0, s,
                       (const uint32_t*)(ws + L.item_off), (const uint32_t*)(ws + L.multi_off),
                       (const uint32_t*)(ws + L.status), g, (const float*)(ws + L.partials),
                       (const uint64_t*)(ws + L.part_masks), d_cube);
    return hipGetLastError();
}

hipError_t launch_weights(int kind, float gt, float ginv, const float* dx, const float* dy,
                          const float* h, float* out, int64_t n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const float4* wtab = nullptr;
    hipError_t e = weight_table(s, &wtab);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_weights, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, kind, gt,
                       ginv, dx, dy, h, wtab, out, n);
    return hipGetLastError();
}

hipError_t launch_spectra(const mi_particle* d_p, int64_t n, const mi_cube_desc& d, float* out,
                          hipStream_t s) {
    int64_t tot = n * d.nc;
    if (tot <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_spectra, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, d_p, n, d,
                       out);
    return hipGetLastError();
}

}  // namespace mi
