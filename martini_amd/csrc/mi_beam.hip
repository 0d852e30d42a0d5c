// Beam convolution of the resident cube: every channel map convolved with the
// beam image (martini/martini.py:863-901, which runs
// scipy.signal.fftconvolve(spatial_slice, beam.kernel, mode="same") per
// channel).  'same' mode with zero boundary, for an odd kx x ky beam image K:
//
//   out[i, j, c] = sum_{a < kx, b < ky} K[a, b] * in[i + kx/2 - a, j + ky/2 - b, c]
//
// The cube is [nx][ny][nc], channels contiguous.  Three kernels:
//   k_convolve_line   one-dimensional images.  A separable beam (a circular or
//                     axis-aligned Gaussian's image is the outer product of two
//                     vectors) is convolved by the caller as two such passes, a
//                     kx x 1 and a 1 x ky image;
//   k_convolve_image  other images, where the cube fills the chip with its tiles;
//   k_convolve_beam   other images on small cubes: a 16 x 16 pixel x 4-channel
//                     output tile per work group, the beam image in blocks of H
//                     rows x W columns whose input halo ((16 + H - 1) x (16 + W - 1)
//                     pixels x 4 channels) and taps (H x W) fit in LDS.
// Any beam size runs with each.  Direct summation in a fixed order
// (deterministic): FP64, or FP32 along each row segment of a block and FP64
// across them.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/martini_mi355x.h"
#include "mi_internal.h"

namespace mi {

// Rotated (non-separable) images: k_convolve_image.  A wave computes one output
// row of a tile, 16 R pixels along y by 16 channels: lane = (pixel group of R,
// quad of channels), so a tap is the same for the whole wave (a scalar
// operand) and each 16-byte LDS read of an input pixel feeds R outputs from a
// window of registers.  The IMG_X waves of a work group share the input rows,
// which pass through LDS one at a time (two buffers, one barrier a row, the
// next row's loads in flight): input row m feeds output row i through image
// row i + kx/2 - m.  Each segment of an image row (up to IMG_MAX_W taps) is
// summed in FP32 and added to FP64 totals, image rows in order: the FP32
// rounding grows with the segment, not with kx * ky.
// Bound by FP32 multiply-adds and the LDS reads beside them (27 x 27 taps on
// 282 x 282 x 128: 0.19 ms of multiply-adds without packed FP32, 0.28 ms
// measured; 0.31 with four outputs per lane and its 64-column tiles, 0.34 with
// two, 0.36 with eight rows per group).  k_convolve_beam, with one LDS read of a
// pixel and one of a tap for four multiply-adds, takes 0.60 ms there.
constexpr int IMG_X = 4;          // output rows (waves) per work group
constexpr int IMG_T = 64 * IMG_X;
constexpr int IMG_C = 16;         // channels per work group
constexpr int IMG_MAX_W = 128;    // image columns per segment
constexpr int IMG_MIN = 1000;      // k_convolve_beam's work groups from which this kernel is taken

// LDS slots of 64 bytes (one pixel's 16 channels) in a row buffer of px pixels.
// The pixel groups of a wave lie R pixels apart: with an even R one spare slot
// after every fourth pixel lets them read from different banks.  Four pixels
// lie in front, which the register window may run into (and not use).
template <int R>
__host__ __device__ inline int img_slot(int px) { return R % 2 ? px : px + (px >> 2); }
template <int R>
__host__ __device__ inline int img_row_slots(int px) { return img_slot<R>(px + 4) + 1; }

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int R, bool VEC>
__global__ __launch_bounds__(IMG_T) void k_convolve_image(const float* __restrict__ in,
                                                          float* __restrict__ out, int nx, int ny,
                                                          int nc, const float* __restrict__ K,
                                                          int kx, int ky) {
    extern __shared__ float4 rows[];  // two row buffers
    constexpr int TY = 16 * R;
    const int tiles_y = (ny + TY - 1) / TY;
    const int x0 = (blockIdx.x / tiles_y) * IMG_X, y0 = (blockIdx.x % tiles_y) * TY;
    const int c0 = blockIdx.y * IMG_C;
    const int t = threadIdx.x, lane = t & 63;
    const int i = x0 + __builtin_amdgcn_readfirstlane(t >> 6);  // this wave's output row
    const int quad = lane & 3, yg = lane >> 2;
    const int hx = kx / 2, hy = ky / 2;
    const int wmax = ky < IMG_MAX_W ? ky : IMG_MAX_W;
    const int buf = img_row_slots<R>(TY - 1 + wmax) * 4;  // float4s per row buffer
    double tot[R][4];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) tot[r][c] = 0.0;

    // Input rows reaching the tile, from the last (image row 0 first) to the first.
    const int m_hi = min(nx - 1, x0 + IMG_X - 1 + hx), m_lo = max(0, x0 + hx - (kx - 1));
    constexpr int PF = ((TY - 1 + IMG_MAX_W) * 4 + IMG_T - 1) / IMG_T;  // float4s per thread and row
    for (int b0 = 0; b0 < ky; b0 += IMG_MAX_W) {
        const int W = min(IMG_MAX_W, ky - b0);
        const int ry0 = y0 + hy - b0 - (W - 1);  // input column of row pixel 0
        const int n4 = (TY - 1 + W) * 4;
        float4 pf[PF];
        auto load = [&](int m) {
#pragma unroll
            for (int q = 0; q < PF; ++q) {
                const int e = t + q * IMG_T, j = ry0 + (e >> 2), c = c0 + (e & 3) * 4;
                pf[q] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (e >= n4 || j < 0 || j >= ny) continue;
                const float* src = in + ((size_t)m * ny + j) * nc + c;
                if (VEC) {
                    if (c < nc) pf[q] = *reinterpret_cast<const float4*>(src);
                } else {
                    if (c < nc) pf[q].x = src[0];
                    if (c + 1 < nc) pf[q].y = src[1];
                    if (c + 2 < nc) pf[q].z = src[2];
                    if (c + 3 < nc) pf[q].w = src[3];
                }
            }
        };
        __syncthreads();  // the last segment's rows are no longer read
        int cur = 0;
        load(m_hi);
        for (int m = m_hi; m >= m_lo; --m) {
            float4* row = rows + cur * buf;
#pragma unroll
            for (int q = 0; q < PF; ++q) {
                const int e = t + q * IMG_T;
                if (e < n4) row[img_slot<R>((e >> 2) + 4) * 4 + (e & 3)] = pf[q];
            }
            __syncthreads();  // the other buffer's readers are past the barrier before this one
            if (m > m_lo) load(m - 1);
            cur ^= 1;
            const int a = i + hx - m;  // image row
            if (a < 0 || a >= kx) continue;  // the same for the wave
            const float* __restrict__ kr = K + (size_t)a * ky + b0;
            // Tap b of the segment reads pixel yg R + r + (W - 1 - b) for output r;
            // slot s of the window holds pixel p + s, p = yg R + W - 1 - b.
            auto at = [&](int p) { return row[img_slot<R>(p + 4) * 4 + quad]; };
            f32x4 acc[R], win[R];
            auto get = [&](int p) {
                const float4 v = at(p);
                return f32x4{v.x, v.y, v.z, v.w};
            };
            int p = yg * R + W - 1;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
                win[r] = get(p + r);
            }
            auto step = [&](float k, int s) {  // tap with the window turned by s
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const f32x4 v = win[(r + R - s) % R];
                    acc[r].x = fmaf(k, v.x, acc[r].x);
                    acc[r].y = fmaf(k, v.y, acc[r].y);
                    acc[r].z = fmaf(k, v.z, acc[r].z);
                    acc[r].w = fmaf(k, v.w, acc[r].w);
                }
            };
            int b = 0;
            for (; b + R < W; b += R, p -= R) {
                f32x4 next[R];
#pragma unroll
                for (int s = 0; s < R; ++s) next[s] = get(p - 1 - s);
#pragma unroll
                for (int s = 0; s < R; ++s) {
                    step(kr[b + s], s);
                    win[R - 1 - s] = next[s];
                }
            }
#pragma unroll
            for (int s = 0; s < R; ++s) {  // the last 1 .. R taps
                if (b + s >= W) break;
                step(kr[b + s], s);
                if (s + 1 < R) win[R - 1 - s] = get(p - 1 - s);
            }
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int c = 0; c < 4; ++c) tot[r][c] += (double)acc[r][c];
        }
    }
    const int c = c0 + quad * 4;
    if (i >= nx || c >= nc) return;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int j = y0 + yg * R + r;
        if (j >= ny) continue;
        float* dst = out + ((size_t)i * ny + j) * nc + c;
        if (VEC) {
            *reinterpret_cast<float4*>(dst) = make_float4((float)tot[r][0], (float)tot[r][1],
                                                          (float)tot[r][2], (float)tot[r][3]);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (c + q < nc) dst[q] = (float)tot[r][q];
        }
    }
}

template <int R>
static hipError_t convolve_image(const float* in, float* out, int nx, int ny, int nc,
                                 const float* K, int kx, int ky, hipStream_t s) {
    const dim3 grid((unsigned)(((nx + IMG_X - 1) / IMG_X) * ((ny + 16 * R - 1) / (16 * R))),
                    (unsigned)((nc + IMG_C - 1) / IMG_C));
    const size_t lds = 2 * 64 * (size_t)img_row_slots<R>(16 * R - 1 + (ky < IMG_MAX_W ? ky : IMG_MAX_W));
    const bool vec = nc % 4 == 0 &&
                     ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    if (vec)
        hipLaunchKernelGGL((k_convolve_image<R, true>), grid, dim3(IMG_T), lds, s, in, out, nx, ny,
                           nc, K, kx, ky);
    else
        hipLaunchKernelGGL((k_convolve_image<R, false>), grid, dim3(IMG_T), lds, s, in, out, nx,
                           ny, nc, K, kx, ky);
    return hipGetLastError();
}

constexpr int BT = 16;               // output tile edge (pixels)
constexpr int BEAM_LDS = 56 * 1024;  // bytes of LDS for one block's halo and taps
constexpr int BEAM_MAX_W = 128;      // beam columns per block

// Columns and rows of the beam image per block.
__host__ __device__ inline int beam_block_cols(int ky) { return ky < BEAM_MAX_W ? ky : BEAM_MAX_W; }

__host__ __device__ inline int beam_block_rows(int kx, int ky) {
    const int w = beam_block_cols(ky);
    int h = BEAM_LDS / (16 * (BT - 1 + w) + 4 * w) - (BT - 1);
    if (h > kx) h = kx;
    return h < 1 ? 1 : h;
}

__global__ __launch_bounds__(256) void k_convolve_beam(const float* __restrict__ in,
                                                       float* __restrict__ out, int nx, int ny,
                                                       int nc, const float* __restrict__ K,
                                                       int kx, int ky, int band_h, int band_w) {
    extern __shared__ float4 lds[];
    const int tiles_y = (ny + BT - 1) / BT;
    const int tile = blockIdx.x;
    const int x0 = (tile / tiles_y) * BT, y0 = (tile % tiles_y) * BT;
    const int c0 = blockIdx.y * 4;
    const int t = threadIdx.x;
    const int tx = t / BT, ty = t % BT;
    const int hx = kx / 2, hy = ky / 2;
    const int wy = BT - 1 + band_w;  // halo width along y
    float4* halo = lds;
    float* taps = reinterpret_cast<float*>(lds + (BT - 1 + band_h) * wy);

    // each row segment of a block is summed in FP32 and added to FP64 totals,
    // so the FP32 rounding grows with the block width, not with kx * ky
    double ax = 0.0, ay = 0.0, az = 0.0, aw = 0.0;
    for (int a0 = 0; a0 < kx; a0 += band_h) {
        const int H = min(band_h, kx - a0);
        for (int b0 = 0; b0 < ky; b0 += band_w) {
            const int W = min(band_w, ky - b0);
            // output (x0 + tx, y0 + ty) reads input (x0 + tx + hx - a, y0 + ty + hy - b)
            // for a in [a0, a0 + H), b in [b0, b0 + W)
            const int rx0 = x0 + hx - a0 - (H - 1);  // input row of halo row 0
            const int ry0 = y0 + hy - b0 - (W - 1);  // input column of halo column 0
            const int hrows = BT - 1 + H, hcols = BT - 1 + W;
            __syncthreads();  // the previous block's halo is no longer read
            for (int e = t; e < hrows * hcols; e += 256) {
                const int r = e / hcols, q = e - r * hcols;
                const int i = rx0 + r, j = ry0 + q;
                float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
                if (i >= 0 && i < nx && j >= 0 && j < ny) {
                    const float* src = in + ((size_t)i * ny + j) * nc + c0;
                    if (c0 + 3 < nc && (nc & 3) == 0) {
                        v = *reinterpret_cast<const float4*>(src);
                    } else {
                        v.x = src[0];
                        if (c0 + 1 < nc) v.y = src[1];
                        if (c0 + 2 < nc) v.z = src[2];
                        if (c0 + 3 < nc) v.w = src[3];
                    }
                }
                halo[r * wy + q] = v;
            }
            for (int e = t; e < H * W; e += 256) {
                const int da = e / W, db = e - da * W;
                taps[e] = K[(size_t)(a0 + da) * ky + b0 + db];
            }
            __syncthreads();
            // tap (a0 + da, b0 + db) reads halo row tx + H - 1 - da, column ty + W - 1 - db
            for (int da = 0; da < H; ++da) {
                const float4* hrow = halo + (tx + H - 1 - da) * wy + ty + W - 1;
                const float* krow = taps + da * W;
                float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
                for (int db = 0; db < W; ++db) {
                    const float k = krow[db];
                    const float4 v = hrow[-db];
                    acc.x = fmaf(k, v.x, acc.x);
                    acc.y = fmaf(k, v.y, acc.y);
                    acc.z = fmaf(k, v.z, acc.z);
                    acc.w = fmaf(k, v.w, acc.w);
                }
                ax += acc.x;
                ay += acc.y;
                az += acc.z;
                aw += acc.w;
            }
        }
    }
    const int i = x0 + tx, j = y0 + ty;
    if (i < nx && j < ny) {
        float* dst = out + ((size_t)i * ny + j) * nc + c0;
        dst[0] = (float)ax;
        if (c0 + 1 < nc) dst[1] = (float)ay;
        if (c0 + 2 < nc) dst[2] = (float)az;
        if (c0 + 3 < nc) dst[3] = (float)aw;
    }
}

// One-dimensional pass over a [O][L][E] view of the cube (E contiguous), along L:
//
//   out[o][l][e] = sum_{a < k} K[a] * in[o][l + k/2 - a][e],  zero outside [0, L).
//
// A kx x 1 image is the pass along x (O = 1, L = nx, E = ny * nc), a 1 x ky
// image the pass along y (O = nx, L = ny, E = nc).  It is a contraction with a
// banded matrix of taps, and runs on the FP64 matrix units: a wave takes
// LINE_R consecutive outputs along L, as LINE_R / 16 blocks of 16, for 64
// columns (the (o, e) pairs, flattened, so any number of channels fills it):
// four 16-column blocks, lane n of a block holding column 4 n + block, so that
// its row of each is one 16-byte load (`vec`: E a multiple of 4 and aligned
// buffers) or, without that, column 16 * block + n.  Each step multiplies four
// input rows into every block of outputs that they reach; the taps of a step
// come from a zero-padded FP64 copy in LDS, one read for eight products.
// Sums are FP64 in a fixed order (deterministic; FP32 rounding only at the
// output).
//
// Bound by HBM (8 bytes per voxel and pass) and the matrix units together:
// k + 15 rows, rounded up to fours, are multiplied for 16 outputs.  On
// 538 x 538 x 256 with 27 taps a pass takes 146 us (4.1 TB/s), about 110 of
// which the products would take alone; the previous vector form (eight outputs
// per lane, one tap test and one LDS tap read per four multiply-adds, each
// input row read (k + 7) / 8 times) took 200 us.  16 outputs per wave read more
// halo rows (168 us), 64 leave too few registers for four waves per SIMD;
// stores that stay in the caches 156 us.
// A row outside the band meets a zero tap, and zero times an infinity or a NaN
// would spread it to its neighbours along L, so a wave that ends with a
// non-finite sum forms its sums again tap by tap.
constexpr int LINE_R = 32;       // outputs per wave along the axis
constexpr int LINE_T = LINE_R / 16;
constexpr int LINE_WAVES = 2;    // waves per work group (consecutive strips along L)
constexpr int LINE_COLS = 64;    // columns per wave
constexpr int LINE_MAX_K = 4096; // taps held in LDS (33 KB); longer images take k_convolve_beam
constexpr int LINE_PAD = 20;     // zeros on either side of the taps
constexpr int LINE_G = 2;        // steps whose rows are loaded together

typedef double f64x4 __attribute__((ext_vector_type(4)));

// LONG leaves out the steps whose rows all lie outside the cube: for an image longer
// than the cube, most of them (4001 taps along 256 rows of 256 x 128: 1623 us with them,
// 131 without).  For a shorter one the loop's plain start costs less (27 taps, 538 x
// 538 x 256: two passes 281 us, 318 with LONG).
template <bool VEC, bool LONG>
__global__ __launch_bounds__(64 * LINE_WAVES) __attribute__((amdgpu_waves_per_eu(4))) void
k_convolve_line(
    const float* __restrict__ in, float* __restrict__ out, int L, int64_t E, int64_t cols,
    const float* __restrict__ K, int k) {
    extern __shared__ double taps[];  // taps[LINE_PAD + a]
    for (int a = threadIdx.x; a < k + 2 * LINE_PAD; a += 64 * LINE_WAVES)
        taps[a] = a >= LINE_PAD && a < k + LINE_PAD ? (double)K[a - LINE_PAD] : 0.0;
    __syncthreads();
    const int lane = threadIdx.x & 63, n = lane & 15, kk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l0 = (blockIdx.y * LINE_WAVES + wave) * LINE_R;
    if (l0 >= L) return;
    // This lane's columns: their offsets from row 0 (in floats), -1 past the end.
    int64_t at[VEC ? 1 : 4];
#pragma unroll
    for (int j = 0; j < (VEC ? 1 : 4); ++j) {
        const int64_t c = (int64_t)blockIdx.x * LINE_COLS + (VEC ? 4 * n : 16 * j + n);
        const int64_t o = c / E;
        at[j] = c < cols ? o * L * E + (c - o * E) : -1;
    }
    f64x4 acc[LINE_T][4];
#pragma unroll
    for (int q = 0; q < LINE_T; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[q][j] = f64x4{0.0, 0.0, 0.0, 0.0};
    // Step s takes input rows m0 + 4 s + kk; row m0 + r feeds output l0 + q
    // through tap q + k - 1 - r.  Block q of 16 outputs needs steps 4 q .. 4 q + S - 1.
    const int S = (k + 15 + 3) / 4;
    const LineSteps steps(l0, L, k, S + 4 * (LINE_T - 1));
    const int m0 = steps.m0, first = LONG ? steps.first : 0;
    const int last = LONG ? steps.last : S + 4 * (LINE_T - 1);
    auto load = [&](int s, float (&v)[4]) {
        const int m = m0 + 4 * s + kk;
        const bool ok = m >= 0 && m < L;
        if (VEC) {
            float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
            if (ok && at[0] >= 0) x = *reinterpret_cast<const float4*>(in + at[0] + (int64_t)m * E);
            v[0] = x.x;
            v[1] = x.y;
            v[2] = x.z;
            v[3] = x.w;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[j] = ok && at[VEC ? 0 : j] >= 0 ? in[at[VEC ? 0 : j] + (int64_t)m * E] : 0.0f;
        }
    };
    const double* tap = taps + LINE_PAD + n - kk + k - 1;  // the lane's tap of step s: tap[-4 s]
    float v[LINE_G][4];
#pragma unroll
    for (int g = 0; g < LINE_G; ++g) load(first + g, v[g]);
    for (int s0 = first; s0 < last; s0 += LINE_G) {
        float w[LINE_G][4];
#pragma unroll
        for (int g = 0; g < LINE_G; ++g)
            if (s0 + LINE_G < last) load(s0 + LINE_G + g, w[g]);
#pragma unroll
        for (int g = 0; g < LINE_G; ++g) {
            const int s = s0 + g;
#pragma unroll
            for (int q = 0; q < LINE_T; ++q) {
                const int sq = s - 4 * q;
                if (sq < 0 || sq >= S) continue;  // uniform
                const double a = tap[-4 * sq];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[q][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, (double)v[g][j], acc[q][j],
                                                                     0, 0, 0);
            }
        }
#pragma unroll
        for (int g = 0; g < LINE_G; ++g)
#pragma unroll
            for (int j = 0; j < 4; ++j) v[g][j] = w[g][j];
    }
    // Lane: outputs l0 + 16 q + 4 i + kk (i = 0..3) of its columns.
    bool finite = true;
#pragma unroll
    for (int q = 0; q < LINE_T; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) finite = finite && __builtin_isfinite(acc[q][j][i]);
    if (!__all(finite)) {
#pragma unroll 1
        for (int q = 0; q < LINE_T; ++q)
#pragma unroll 1
            for (int i = 0; i < 4; ++i) {
                const int l = l0 + 16 * q + 4 * i + kk;
                double sum[4] = {0.0, 0.0, 0.0, 0.0};
                for (int a = min(k - 1, l + k / 2); a >= 0; --a) {
                    const int m = l + k / 2 - a;
                    if (m >= L) break;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int64_t c = VEC ? at[0] : at[VEC ? 0 : j];
                        if (c >= 0)
                            sum[j] = fma(taps[LINE_PAD + a],
                                         (double)in[c + (VEC ? j : 0) + (int64_t)m * E], sum[j]);
                    }
                }
#pragma unroll
                for (int q2 = 0; q2 < LINE_T; ++q2)
#pragma unroll
                    for (int i2 = 0; i2 < 4; ++i2)
                        if (q2 == q && i2 == i)
#pragma unroll
                            for (int j = 0; j < 4; ++j) acc[q2][j][i2] = sum[j];
            }
    }
#pragma unroll
    for (int q = 0; q < LINE_T; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int l = l0 + 16 * q + 4 * i + kk;
            if (l >= L) continue;
            if (VEC) {
                if (at[0] >= 0)
                    __builtin_nontemporal_store(
                        f32x4{(float)acc[q][0][i], (float)acc[q][1][i], (float)acc[q][2][i],
                              (float)acc[q][3][i]},
                        reinterpret_cast<f32x4*>(out + at[0] + (int64_t)l * E));
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (at[VEC ? 0 : j] >= 0)
                        out[at[VEC ? 0 : j] + (int64_t)l * E] = (float)acc[q][j][i];
            }
        }
}

static hipError_t convolve_line(const float* in, float* out, int64_t O, int L, int64_t E,
                                const float* K, int k, hipStream_t s) {
    const int64_t cols = O * E;
    const dim3 grid((unsigned)((cols + LINE_COLS - 1) / LINE_COLS),
                    (unsigned)((L + LINE_R * LINE_WAVES - 1) / (LINE_R * LINE_WAVES)));
    const size_t lds = sizeof(double) * (size_t)(k + 2 * LINE_PAD);
    const bool vec = E % 4 == 0 &&
                     ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(64 * LINE_WAVES), lds, s, in, out, L, E, cols, K, k);
    };
    if (k > L)
        launch(vec ? k_convolve_line<true, true> : k_convolve_line<false, true>);
    else
        launch(vec ? k_convolve_line<true, false> : k_convolve_line<false, false>);
    return hipGetLastError();
}

size_t beam_lds_bytes(int kx, int ky) {
    const int h = beam_block_rows(kx, ky), w = beam_block_cols(ky);
    return sizeof(float4) * (size_t)(BT - 1 + h) * (BT - 1 + w) + sizeof(float) * (size_t)h * w;
}

hipError_t convolve_beam(const float* in, float* out, int nx, int ny, int nc, const float* K,
                         int kx, int ky, hipStream_t s) {
    if (ky == 1 && kx <= LINE_MAX_K)  // along x: [1][nx][ny * nc]
        return convolve_line(in, out, 1, nx, (int64_t)ny * nc, K, kx, s);
    if (kx == 1 && ky <= LINE_MAX_K)  // along y: [nx][ny][nc]
        return convolve_line(in, out, nx, ny, nc, K, ky, s);
    const int64_t tiles = (int64_t)((nx + BT - 1) / BT) * ((ny + BT - 1) / BT), cq = (nc + 3) / 4;
    // k_convolve_image where there is work for it: its rows, one after another, are a
    // chain of some 60 us (27 x 27 taps) however few its work groups are, while
    // k_convolve_beam's time goes with the number of its small tiles (720 of them, 256
    // x 70 x 36: 65 us against 49; 768, 256 x 87 x 30: 58 against 50; 960, 89 x
    // 65 x 128: 65 against 62; 1024, 128 x 128 x 64: 60 against 64.5; 2560, 256 x
    // 68 x 128: 87 against 130; 10368, 282 x 282 x 128: 283 against 596; images of 3 x 3
    // to 15 x 15 on nine shapes from 1000 tiles on: 0.33 to 1.01 of its time); and where
    // its tiles of 48 columns or more are not half empty (256 x 24 x 128: 66 against
    // 62).  Three outputs per lane against four by the columns they cover: three take
    // 1.09 times as long per column.
    const int64_t y3 = (ny + 47) / 48, y4 = (ny + 63) / 64;
    const bool three = y3 * 48 * 12 < y4 * 64 * 11;
    if (ny > 32 && tiles * cq >= IMG_MIN)
        return three ? convolve_image<3>(in, out, nx, ny, nc, K, kx, ky, s)
                     : convolve_image<4>(in, out, nx, ny, nc, K, kx, ky, s);
    const int h = beam_block_rows(kx, ky), w = beam_block_cols(ky);
    const size_t lds = beam_lds_bytes(kx, ky);
    hipLaunchKernelGGL(k_convolve_beam, dim3((unsigned)tiles, (unsigned)cq), dim3(256), lds, s, in, out, nx, ny, nc, K,
                       kx, ky, h, w);
    return hipGetLastError();
}

}  // namespace mi
