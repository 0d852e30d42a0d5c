// What stands around the gather: the reduction of split cells' partial tiles,
// the kernel weight tables, and the entry points that evaluate kernel
// integrals and spectra by themselves.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "mi_device.h"
#include "mi_internal.h"
#include "mi_tile.h"

namespace mi {

// Sums the partial tiles of the split cells in FP64 (their sum then costs one
// rounding: 1.3e-7 -> 0.8e-7 of error on 1e4 particles in 400 items), and adds
// them to the cube.  A wave takes a 1 KiB sub-tile of a cell at a time: it reads
// the masks of 64 items, one per lane, and then only the sub-tiles that those items
// wrote, RED_DEEP loads in flight (1e6 particles, MFMA: 39 us with the masks read
// item by item, 31 with four loads in flight).
//
// Where cells are split RED_SHARED times or more on average, too few sub-tiles are
// left for the chip and each is a long chain of loads: the waves of a work group
// then share one, every fourth item each (1e6 particles, 72 cells in 32 items: 38
// -> 21 us; 1e4: 9.2 -> 6.8).  With fewer items the sharing's barrier costs more than
// the loads (3e5 particles, 11 a cell: 20 us, shared 26).  The sub-tiles of the listed
// split cells go round RED_GROUPS work groups: work groups for every cell of the
// cube were mostly for empty ones (1e7 particles: 95 -> 87 us; 3e5 on 512 x 512 x
// 256: 55 -> 38).
// Voxels no item wrote keep the cube's value; the order of a sum depends on the
// input alone.
constexpr int RED_DEEP = 8;
constexpr int RED_GROUPS = 8192;
constexpr int RED_SHARED = 16;
constexpr int RED_SUBS = CELL_VOXELS / (16 * SUB_CH);  // sub-tiles of a cell

__global__ __launch_bounds__(NT) void k_reduce(const uint32_t* __restrict__ item_off,
                                               const uint32_t* __restrict__ multi_off,
                                               const uint32_t* __restrict__ split_cells,
                                               const uint32_t* __restrict__ status, Grid g,
                                               const float* __restrict__ partials,
                                               const uint64_t* __restrict__ part_masks,
                                               float* __restrict__ cube) {
    if (status[ST_OVERFLOW]) return;
    constexpr int SHARES = NT / 64;
    // two, in turn: a wave may be one sub-tile ahead of the wave that sums
    __shared__ double sums[2][SHARES - 1][4][64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63;
    const size_t tile = (size_t)CELL_VOXELS / 4;  // float4 per partial tile
    const int nblk = (1 << g.cb_shift) / SUB_CH;
    const uint32_t n = status[ST_SPLIT] * RED_SUBS;
    const bool shared = status[ST_MULTI] >= RED_SHARED * status[ST_SPLIT];
    const uint64_t every = shared ? 0x1111111111111111ull << wave : ~0ull;
    const uint32_t stride = shared ? gridDim.x : gridDim.x * SHARES;
    int turn = 0;
    for (uint32_t e = shared ? blockIdx.x : blockIdx.x * SHARES + wave; e < n; e += stride) {
        const int cell = (int)split_cells[e / RED_SUBS];
        const int sub = (int)(e % RED_SUBS);  // row * blocks + block
        const uint32_t ni = item_off[cell + 1] - item_off[cell], first = multi_off[cell];
        // float4 `lane` of the sub-tile: channel lane / 4, four pixels from 4 (lane % 4) on
        static_assert(TILE_Y == 16 && SUB_CH == 16, "64 float4 a sub-tile");
        const float4* src =
            reinterpret_cast<const float4*>(partials) + (size_t)first * tile + sub * 64 + lane;
        const uint64_t* mk = part_masks + first;
        const int prow = sub / nblk, blk = sub - prow * nblk;
        const int bit = sub_bit(g.tx_shift, prow, blk);
        double s0[4] = {0.0, 0.0, 0.0, 0.0};
        uint64_t seen = 0u;
        for (uint32_t q0 = 0; q0 < ni; q0 += 64) {
            const uint64_t all = __ballot(q0 + lane < ni && ((mk[q0 + lane] >> bit) & 1u));
            seen |= all;
            uint64_t set = all & every;
            const float4* p = src + q0 * tile;
            while (set) {
                float4 v[RED_DEEP];
                int m = 0;
#pragma unroll
                for (int k = 0; k < RED_DEEP; ++k) {
                    if (!set) break;  // uniform
                    v[k] = p[(size_t)__builtin_ctzll(set) * tile];
                    set &= set - 1u;
                    m = k + 1;
                }
#pragma unroll
                for (int k = 0; k < RED_DEEP; ++k) {
                    if (k >= m) break;
                    s0[0] += (double)v[k].x;
                    s0[1] += (double)v[k].y;
                    s0[2] += (double)v[k].z;
                    s0[3] += (double)v[k].w;
                }
            }
        }
        if (!seen) continue;  // the same for the waves that share a sub-tile
        if (shared) {
            double(&buf)[SHARES - 1][4][64] = sums[turn];
            turn ^= 1;
            if (wave > 0) {
#pragma unroll
                for (int u = 0; u < 4; ++u) buf[wave - 1][u][lane] = s0[u];
            }
            __syncthreads();
            if (wave > 0) continue;
#pragma unroll
            for (int w = 0; w < SHARES - 1; ++w)
#pragma unroll
                for (int u = 0; u < 4; ++u) s0[u] += buf[w][u][lane];
        }
        const CellPos cp = cell_pos(cell, g);
        const int i = cp.x0 + prow, j = cp.y0 + (lane & 3) * 4, c = cp.c0 + blk * SUB_CH + (lane >> 2);
        float* dst = cube + ((size_t)i * g.ny + j) * g.nc + c;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i < g.nx && c < g.nc && j + u < g.ny) {
                float& v = dst[(size_t)u * g.nc];
                v = (float)((double)v + s0[u]);
            }
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
    if (L.split_max <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_reduce, dim3((unsigned)std::min<int64_t>(L.split_max * RED_SUBS, RED_GROUPS)),
                       dim3(NT), 0, s, (const uint32_t*)(ws + L.item_off),
                       (const uint32_t*)(ws + L.multi_off), (const uint32_t*)(ws + L.split_cells),
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
