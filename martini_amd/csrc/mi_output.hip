// The FITS data unit of a cube, made on the device: Martini.write_fits
// (martini/martini.py:939-1055) drops the pad, takes the array's transpose
// (:1049, so that FITS axis 1 -- x -- runs fastest, then y, then channel),
// casts it (:1050-1051) and has astropy write it big-endian.  Here one kernel
// reads the padded [nx + 2 padx][ny + 2 pady][nc] cube (FP32 as the gathers
// leave it, or FP64 as the host holds it), and writes the unpadded region in
// FITS order as big-endian float32 or float64, ready to follow the header in
// the file; the same pass finds DATAMIN and DATAMAX.
//
// A work group moves 64 (x) x 64 (channel) tiles of `rows` rows y through LDS:
// read along channels (the cube's contiguous axis), written along x (the
// file's), 16 bytes per lane on either side where the rows are aligned for it.
// Bound by HBM: the next row's loads are in flight while the current one is
// written, with stores that do not stay in the caches.  512 x 512 x 256 FP64 to
// FP64: 304 us with one value per load and no overlap, 244 us (4.4 TB/s; a
// copy runs at 5.2); FP32 to FP32 182 -> 126 us; 64 x 64 x 32 FP32 42 -> 17 us
// (the atomics' share below).  Min and max use order-preserving integer images of the values,
// reduced in the work group, so their atomics give the same result in any
// order; a group whose extremes do not pass the running ones sends none (all
// groups' atomics go to one cache line, about 11 ns each).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/martini_mi355x.h"
#include "mi_internal.h"

namespace mi {

constexpr int FT = 64;  // tile edge (x and channel)

// Unsigned image of a floating value whose integer order is the numeric order.
__device__ inline uint32_t order_of(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u >> 31) ? ~u : (u | 0x80000000u);
}
__device__ inline uint64_t order_of(double f) {
    const uint64_t u = (uint64_t)__double_as_longlong(f);
    return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}
__device__ inline float value_of(uint32_t u) {
    return __uint_as_float((u >> 31) ? (u & 0x7fffffffu) : ~u);
}
__device__ inline double value_of(uint64_t u) {
    return __longlong_as_double((long long)((u >> 63) ? (u & 0x7fffffffffffffffull) : ~u));
}

template <typename In>
struct OrderOf;
template <>
struct OrderOf<float> {
    using type = uint32_t;
};
template <>
struct OrderOf<double> {
    using type = uint64_t;
};

__device__ inline uint32_t big_endian(float v) { return __builtin_bswap32(__float_as_uint(v)); }
__device__ inline uint64_t big_endian(double v) {
    return __builtin_bswap64((uint64_t)__double_as_longlong(v));
}

__global__ void k_range_init(unsigned long long* __restrict__ range) {
    if (threadIdx.x == 0) {
        range[0] = ~0ull;  // running min
        range[1] = 0ull;   // running max
    }
}

__global__ void k_range_finish(unsigned long long* __restrict__ range) {
    if (threadIdx.x < 2) {
        const double f = value_of((uint64_t)range[threadIdx.x]);
        reinterpret_cast<double*>(range)[threadIdx.x] = f;
    }
}

template <typename T, int N>
using Pack = T __attribute__((ext_vector_type(N)));

// LN channels per load and SN pixels per store: 16 bytes each, or one value
// where the rows are not aligned for that.
template <typename In, typename Out, int LN, int SN>
__global__ __launch_bounds__(256) void k_cube_to_fits(const In* __restrict__ cube, int nx, int ny,
                                                      int nc, int padx, int pady, int rows,
                                                      void* __restrict__ out,
                                                      unsigned long long* __restrict__ range) {
    using Order = typename OrderOf<In>::type;
    using Word = decltype(big_endian(Out()));
    __shared__ In tile[FT][FT + 1];
    __shared__ Order wlo[4], whi[4];
    const int xt = (nx + FT - 1) / FT;
    const int x0 = (blockIdx.x % xt) * FT, c0 = (blockIdx.x / xt) * FT;
    const int t = threadIdx.x;
    const size_t NY = (size_t)ny + 2 * (size_t)pady;
    const size_t plane = (size_t)nx * ny;
    Order lo = (Order)~(Order)0, hi = 0;
    const int y0 = blockIdx.y * rows, y1 = min(ny, y0 + rows);
    // load j of a row: x row lx + j * LROWS, channels lc .. lc + LN - 1
    constexpr int LROWS = 256 / (FT / LN), LJ = FT / LROWS;
    const int lx = t / (FT / LN), lc = (t % (FT / LN)) * LN;
    // store j: channel sc + j * SROWS, pixels sx .. sx + SN - 1
    constexpr int SROWS = 256 / (FT / SN), SJ = FT / SROWS;
    const int sc = t / (FT / SN), sx = (t % (FT / SN)) * SN;
    const bool lok = c0 + lc < nc;  // nc is a multiple of LN, nx of SN
    const bool sok = x0 + sx < nx;
    Pack<In, LN> v[LJ];
    auto load = [&](int y) {
#pragma unroll
        for (int j = 0; j < LJ; ++j) {
            const int x = x0 + lx + j * LROWS;
            if (lok && x < nx)
                v[j] = *reinterpret_cast<const Pack<In, LN>*>(
                    cube + ((size_t)(x + padx) * NY + (size_t)(y + pady)) * nc + c0 + lc);
        }
    };
    load(y0);
    for (int y = y0; y < y1; ++y) {
#pragma unroll
        for (int j = 0; j < LJ; ++j) {
            if (!lok || x0 + lx + j * LROWS >= nx) continue;
#pragma unroll
            for (int k = 0; k < LN; ++k) {
                const In f = v[j][k];
                const Order o = order_of(f);
                lo = o < lo ? o : lo;
                hi = o > hi ? o : hi;
                tile[lx + j * LROWS][lc + k] = f;
            }
        }
        __syncthreads();
        if (y + 1 < y1) load(y + 1);
#pragma unroll
        for (int j = 0; j < SJ; ++j) {
            const int ci = sc + j * SROWS;
            if (!sok || c0 + ci >= nc) continue;
            Pack<Word, SN> w;
#pragma unroll
            for (int k = 0; k < SN; ++k) w[k] = big_endian((Out)tile[sx + k][ci]);
            __builtin_nontemporal_store(
                w, reinterpret_cast<Pack<Word, SN>*>(reinterpret_cast<Word*>(out) +
                                                     (size_t)(c0 + ci) * plane + (size_t)y * nx +
                                                     x0 + sx));
        }
        __syncthreads();  // the tile is rewritten for the next row
    }
    for (int d = 32; d > 0; d >>= 1) {
        const Order ol = __shfl_xor(lo, d, 64), oh = __shfl_xor(hi, d, 64);
        lo = ol < lo ? ol : lo;
        hi = oh > hi ? oh : hi;
    }
    if ((t & 63) == 0) {
        wlo[t >> 6] = lo;
        whi[t >> 6] = hi;
    }
    __syncthreads();
    if (t == 0) {
        for (int w = 1; w < 4; ++w) {
            lo = wlo[w] < lo ? wlo[w] : lo;
            hi = whi[w] > hi ? whi[w] : hi;
        }
        const unsigned long long l = order_of((double)value_of(lo));
        const unsigned long long h = order_of((double)value_of(hi));
        if (l < __hip_atomic_load(&range[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMin(&range[0], l);
        if (h > __hip_atomic_load(&range[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(&range[1], h);
    }
}

template <typename In, typename Out>
static void launch_to_fits(const In* cube, int nx, int ny, int nc, int padx, int pady, void* out,
                           unsigned long long* range, hipStream_t s) {
    const int64_t tiles = (int64_t)((nx + FT - 1) / FT) * ((nc + FT - 1) / FT);
    const int rows = fits_rows(tiles, ny);
    const dim3 grid((unsigned)tiles, (unsigned)((ny + rows - 1) / rows));
    constexpr int L = 16 / sizeof(In), S = 16 / sizeof(Out);
    const bool la = nc % L == 0 && (reinterpret_cast<uintptr_t>(cube) & 15) == 0;
    const bool sa = nx % S == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, cube, nx, ny, nc, padx, pady, rows,
                           out, range);
    };
    if (la && sa)
        launch(k_cube_to_fits<In, Out, L, S>);
    else if (la)
        launch(k_cube_to_fits<In, Out, L, 1>);
    else if (sa)
        launch(k_cube_to_fits<In, Out, 1, S>);
    else
        launch(k_cube_to_fits<In, Out, 1, 1>);
}

hipError_t cube_to_fits(const void* cube, bool cube_f64, int nx, int ny, int nc, int padx,
                        int pady, bool f64, void* out, double* range, hipStream_t s) {
    auto* r = reinterpret_cast<unsigned long long*>(range);
    hipLaunchKernelGGL(k_range_init, dim3(1), dim3(64), 0, s, r);
    auto go = [&](auto* c) {
        if (f64)
            launch_to_fits<std::remove_const_t<std::remove_pointer_t<decltype(c)>>, double>(
                c, nx, ny, nc, padx, pady, out, r, s);
        else
            launch_to_fits<std::remove_const_t<std::remove_pointer_t<decltype(c)>>, float>(
                c, nx, ny, nc, padx, pady, out, r, s);
    };
    if (cube_f64)
        go(static_cast<const double*>(cube));
    else
        go(static_cast<const float*>(cube));
    hipLaunchKernelGGL(k_range_finish, dim3(1), dim3(64), 0, s, r);
    return hipGetLastError();
}

}  // namespace mi
