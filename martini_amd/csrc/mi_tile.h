// Chunk staging of the tile gather, shared by its two forms: the cell-sorted
// particle records of a work item are taken 32 at a time, their footprints
// clipped to the cell's tile, and W evaluated once per (particle, footprint
// pixel) pair.
//
// A wave stages two chunks at once, with DPP scans (no serial loop), while its
// work group waits; it loads the records of the next two while the current ones
// are processed, so the global-memory latency is hidden behind the
// W/S/accumulate work.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "mi_device.h"
#include "mi_internal.h"

namespace mi {

constexpr int KC = 32;    // particles per chunk
constexpr int NT = 256;   // threads per work group
// An item's kernel table in LDS: the WTAB_N intervals and one zero entry
// after them, which the branch-free walk reads for q >= 1.
constexpr int LTAB_N = WTAB_N + 1;

// What the W walk needs of a particle, read with two 16-byte loads by every
// thread that takes some of its pixels.  px, py hold
//   the particle's position ix + fx, iy + fy (exact in FP64) for the Gaussian kernel;
//   for the other closed forms its offsets from the footprint's first pixel in
//   FP32 (tile_offset), for the tabulated ones in table intervals (f a pixel), and
//   1/h^2 (inv_h2); their position is in the chunk's GaussRec slot;
//   as int64 bits (table_walk) the index of pixel (0, 0) in the caller's weight
//   table and the row stride of the particle's weights for MI_KERNEL_TABLE.
struct __attribute__((aligned(16))) WalkRec {
    double px, py;
    float f;         // Gaussian: WFactors::b; tabulated kernels: WTAB_N / h
    // the first of the threads that share its pixels; and, << 16, its spectral window
    // clipped to the cell and the cube: first channel | channels past it << 8,
    // NO_WINDOW when empty
    uint32_t first_win;
    // the footprint clipped to the tile: its corner (row | column << 4), width
    // (<< 8) and rows (<< 16)
    uint32_t box;
    // tile rows (bits 0..15) and 16-channel blocks (16..23) reached, zero without
    // a footprint in the cell; kernel kind << 24 | Gaussian table index << 28
    uint32_t cover;

    __device__ int first() const { return first_win & 255u; }
    __device__ int win_lo() const { return (first_win >> 16) & 255u; }
    __device__ uint32_t win_past() const { return first_win >> 24; }
    __device__ int row() const { return box & 15; }
    __device__ int col() const { return (box >> 4) & 15; }
    __device__ int width() const { return (box >> 8) & 31; }
    __device__ int rows() const { return box >> 16; }
    __device__ int kind() const { return (cover >> 24) & 15; }
    __device__ int gidx() const { return cover >> 28; }
};

__device__ inline double pack2(float lo, float hi) {
    return __hiloint2double(__float_as_int(hi), __float_as_int(lo));
}
__device__ inline float2 tile_offset(const WalkRec& w) {
    return make_float2(__int_as_float(__double2loint(w.px)), __int_as_float(__double2hiint(w.px)));
}
__device__ inline float inv_h2(const WalkRec& w) { return __int_as_float(__double2loint(w.py)); }

// Weight-table walk of an MI_KERNEL_TABLE particle: weights[base + i * stride + j]
// is its weight at pixel (i, j).
struct TableWalk {
    int64_t base, stride;
};

__device__ inline TableWalk table_walk(const WalkRec& w) {
    return TableWalk{__double_as_longlong(w.px), __double_as_longlong(w.py)};
}

// What the Gaussian walk needs beyond the WalkRec: WFactors::a and e.  For the
// other closed forms: the particle's position.
struct GaussRec {
    double a, e;
};

constexpr uint32_t NO_WINDOW = 255u;  // no channel of a cell lies there

// What the S fill needs of a particle beside its window: mi_particle's fields.
struct __attribute__((aligned(16))) SpecRec {
    int32_t k0;
    float fu, s, amp;
};

// One chunk's state, small enough that four chunks', with the 16 x 16 x 64 cells'
// operand tiles, leave room for three work groups on a CU (2096 bytes; 192 more
// in all would not).
struct ChunkState {
    WalkRec walk[KC];
    GaussRec gr[KC];    // Gaussian kernel factors
    SpecRec p[KC];
    // Bit t: thread t + 1 is the first of a particle; and, a byte per wave, how
    // many of the bits belong to the waves before.
    __attribute__((aligned(16))) uint32_t starts[NT / 32];
    uint32_t started;
    // tile rows (x offsets; bits 0..15) touched by any footprint of the chunk and
    // 16-channel blocks of the cell (16..23) touched by any window; pairs per
    // thread << 24; whether a line is left out (odd_line) << 31
    uint32_t cover_per;
    uint32_t gmask;     // particles of the Gaussian kernel with a footprint in the tile

    __device__ static uint32_t rowmask(uint32_t cover_per) { return cover_per & 0xffffu; }
    __device__ static uint32_t chanmask(uint32_t cover_per) { return (cover_per >> 16) & 255u; }
    __device__ static bool odd(uint32_t cover_per) { return cover_per >> 31; }
    __device__ int per() const { return (int)((cover_per >> 24) & 127u); }
};

// The separable factors of the Gaussian kernel's pixel weight for the chunk's
// Gaussian particles, per footprint row and column: ex[k][r] = erf span of row
// r of particle k's clipped footprint, ey[k][c] that of column c (weight_at's
// ex and ey).  Filled once per chunk, they leave one erf and the FP64
// truncation term per pixel.
struct GaussTables {
    float ex[KC][TILE_MAX];
    float ey[KC][TILE_MAX];
};

// Wave-wide inclusive scans with DPP (row shifts within 16-lane rows, then the
// row broadcasts of lanes 15 and 31): VALU moves only, no LDS round trip as
// with shuffles.  All 64 lanes must be active.
template <class Op>
__device__ inline uint32_t wave_scan(uint32_t x, Op op) {
    // dpp_ctrl: row_shr:n = 0x110 + n, row_bcast:15 = 0x142, row_bcast:31 = 0x143;
    // lanes whose source is out of range keep `old` (the identity 0 for + and |)
    x = op(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false));
    x = op(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false));
    x = op(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false));
    x = op(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false));
    x = op(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false));
    x = op(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false));
    return x;
}

// The same within each half of the wave: lanes 0..31 and 32..63.
template <class Op>
__device__ inline uint32_t half_scan(uint32_t x, Op op) {
    x = op(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false));
    x = op(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false));
    x = op(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false));
    x = op(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false));
    return op(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false));
}

__device__ inline int wave_scan_add(int x) {
    return (int)wave_scan((uint32_t)x, [](uint32_t a, uint32_t b) { return a + b; });
}

// A particle record held in registers between its prefetch and its staging,
// as three 16-byte pieces.  (A prefetched mi_particle copied as a whole struct
// can be given a per-thread LDS or scratch slot by the compiler, and the
// store into that slot then waits for the load: the prefetch would stall.)
struct RecRegs {
    uint4 a, b, c;
};

__device__ inline RecRegs load_record(const mi_particle* __restrict__ P, uint32_t i) {
    const uint4* q = reinterpret_cast<const uint4*>(P + i);
    return RecRegs{q[0], q[1], q[2]};
}

__device__ inline mi_particle unpack_record(const RecRegs& r) {
    mi_particle p;
    p.ix = (int32_t)r.a.x;
    p.iy = (int32_t)r.a.y;
    p.fx = __uint_as_float(r.a.z);
    p.fy = __uint_as_float(r.a.w);
    p.h = __uint_as_float(r.b.x);
    p.r_kind = (int32_t)r.b.y;
    p.c_lo = (int32_t)r.b.z;
    p.c_hi = (int32_t)r.b.w;
    p.k0 = (int32_t)r.c.x;
    p.fu = __uint_as_float(r.c.y);
    p.s = __uint_as_float(r.c.z);
    p.amp = __uint_as_float(r.c.w);
    return p;
}

// Entry i (0..3) of a 4-entry kernel-argument array for a lane-varying i, by
// selects over wave-uniform values: an indexed read of the kernel arguments
// would be a memory load on the staging path.
__device__ inline float pick4(const float (&v)[4], int i) {
    const float v0 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v[0])));
    const float v1 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v[1])));
    const float v2 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v[2])));
    const float v3 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v[3])));
    return i == 0 ? v0 : i == 1 ? v1 : i == 2 ? v2 : v3;
}

// Called by all 64 lanes of one wave, for two chunks at once: lane t holds
// particle t % KC of chunk t / KC in `r`.  Clips footprints to the tile, scans
// the pair counts, ORs the row and channel-block masks across each half of the
// wave and forms each particle's weight factors.  The staging is on every
// chunk's critical path (the other waves wait for it), and one wave's
// instructions for two chunks are those of one.  In the FP32 form lines that are not
// finite (odd_line) get no window and are only marked in cover_per.
template <bool FP32>
__device__ inline void stage_chunks(const RecRegs& r, bool valid, int x0, int y0, int c0,
                                    const Grid& g, const mi_cube_desc& d, ChunkState* both) {
    static_assert(KC == 32, "half a wave per chunk");
    const int half = (threadIdx.x >> 5) & 1, lane = threadIdx.x & (KC - 1);
    ChunkState& cs = both[half];
    const mi_particle p = unpack_record(r);
    // Straight-line code with selects: every lane forms the clipped footprint,
    // lanes without a particle or a footprint in the tile end with cnt = 0.
    int fi_lo = 0, fi_hi = -1, fj_lo = 0, fj_hi = -1;
    const bool fp = footprint(p, g.nx, g.ny, fi_lo, fi_hi, fj_lo, fj_hi);
    const int ci_lo = max(fi_lo, x0), ci_hi = min(fi_hi, x0 + (1 << g.tx_shift) - 1);
    const int cj_lo = max(fj_lo, y0), cj_hi = min(fj_hi, y0 + TILE_Y - 1);
    const bool ok = valid && fp && ci_lo <= ci_hi && cj_lo <= cj_hi;
    const int ilo = ok ? ci_lo : 1, ihi = ok ? ci_hi : 0;
    const int jlo = ok ? cj_lo : 1, jhi = ok ? cj_hi : 0;
    const int cnt = ok ? (ihi - ilo + 1) * (jhi - jlo + 1) : 0;
    const uint32_t rows = ok ? (2u << (ihi - x0)) - (1u << (ilo - x0)) : 0u;
    const int ca = max(p.c_lo, c0) - c0, cb = min(p.c_hi, c0 + (1 << g.cb_shift) - 1) - c0;
    const uint32_t chans = ok && ca <= cb ? (2u << (cb >> 4)) - (1u << (ca >> 4)) : 0u;
    const auto add = [](uint32_t a, uint32_t b) { return a + b; };
    const auto bit_or = [](uint32_t a, uint32_t b) { return a | b; };
    const int incl = (int)half_scan((uint32_t)cnt, add);
    static_assert(TILE_MAX <= 16 && GeoWide::CB / 16 <= 8, "rows and channel blocks share one word");
    const bool odd = FP32 && valid && d.spectrum != MI_SPECTRUM_TABLE && odd_line(p.s, p.fu, p.amp);
    const uint32_t masks = half_scan(rows | (chans << 16) | (uint32_t)odd << 31, bit_or);  // one reduction for all
    const uint64_t gauss = __ballot(cnt > 0 && kind_of(p.r_kind) == MI_KERNEL_GAUSS);
    // Each particle's pairs go to max(1, ceil(cnt / per)) threads of their own, per
    // = ceil(total / (NT - KC)): at most total / per + KC <= NT threads in all.  No
    // two particles share a first thread, so a thread finds its particle by counting
    // the first threads up to itself (one bit each).
    const int total0 = __builtin_amdgcn_readlane(incl, KC - 1);
    const int total1 = __builtin_amdgcn_readlane(incl, 2 * KC - 1);
    const int per0 = max(1, (total0 + (NT - KC) - 1) / (NT - KC));
    const int per1 = max(1, (total1 + (NT - KC) - 1) / (NT - KC));
    const int per = half ? per1 : per0;
    // ceil(cnt / per) = floor((cnt + per - 1 + 1/2) / per): the quotient lies at
    // least 1/74 from an integer (per <= 37), far beyond the reciprocal's error
    const float rper = __builtin_amdgcn_rcpf((float)per);
    const int threads = max((int)(((float)(cnt + per - 1) + 0.5f) * rper), 1);
    const int first = (int)half_scan((uint32_t)threads, add) - threads;
    if (lane < NT / 32) cs.starts[lane] = 0u;
    if (lane > 0)
        __hip_atomic_fetch_or(&cs.starts[(first - 1) >> 5], 1u << ((first - 1) & 31),
                              __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    uint32_t started = 0u;
    static_assert(NT / 64 == 4 && KC <= 255, "a byte per wave");
#pragma unroll
    for (int v = 1; v < NT / 64; ++v) {
        const uint64_t b = __ballot(lane > 0 && first <= 64 * v);
        started |= (uint32_t)__builtin_popcount((uint32_t)(b >> (half * KC))) << (8 * v);
    }
    const int cl = min(cb, g.nc - 1 - c0);
    const uint32_t window = valid && !odd && ca <= cl ? (uint32_t)ca | (uint32_t)(cl - ca) << 8 : NO_WINDOW;
    const int width = max(jhi - jlo + 1, 1);
    const int kind = kind_of(p.r_kind), gi = gidx_of(p.r_kind);
    cs.p[lane] = SpecRec{p.k0, p.fu, p.s, p.amp};
    WalkRec w;
    const double px = (double)p.ix + (double)p.fx, py = (double)p.iy + (double)p.fy;
    w.px = px;
    w.py = py;
    w.first_win = (uint32_t)first | window << 16;
    w.box = 0u;
    w.cover = 0u;
    WFactors f{0.0, 0.0, 0.0f, 0.0f, 0.0f};
    if (ok) {
        w.box = (uint32_t)(ilo - x0) | (uint32_t)(jlo - y0) << 4 | (uint32_t)width << 8 |
                (uint32_t)(ihi - ilo + 1) << 16;
        w.cover = rows | (chans << 16) | (uint32_t)kind << 24 | (uint32_t)gi << 28;
        if (kind == MI_KERNEL_GAUSS) {  // the truncation only for the Gaussian
            f = weight_factors(kind, p.h, pick4(d.gauss_t, gi), 0.0f);
            cs.gr[lane] = GaussRec{f.a, f.e};
        } else {
            cs.gr[lane] = GaussRec{px, py};
            f = weight_factors(kind, p.h, 0.0f, 0.0f);  // b = 1/h^2
            float scale = 1.0f;
            if (kind <= MI_KERNEL_QUARTIC) {  // WTAB_N / h, one Newton step past the hardware's 1/h
                const float rh = __builtin_amdgcn_rcpf(p.h);
                scale = (float)WTAB_N * fmaf(rh, fmaf(-p.h, rh, 1.0f), rh);
            }
            w.px = pack2((float)((px - (double)ilo) * scale), (float)((py - (double)jlo) * scale));
            w.py = pack2(f.b, 0.0f);
            f.b = scale;
        }
        if (kind == MI_KERNEL_TABLE) {
            // its weights are laid out over its cube-clipped footprint
            const int64_t stride = fj_hi - fj_lo + 1;
            w.px = __longlong_as_double((int64_t)table_offset(p) - (int64_t)fi_lo * stride - fj_lo);
            w.py = __longlong_as_double(stride);
        }
    }
    w.f = f.b;
    cs.walk[lane] = w;
    if (lane == KC - 1) {  // holds its half's reductions
        cs.started = started;
        cs.cover_per = masks | (uint32_t)per << 24;
        cs.gmask = (uint32_t)(gauss >> (half * KC));
    }
}

// The weight of a tabulated kernel as weight_at computes it but without
// branches: fb = 1/h^2, x2 = (q WTAB_N)^2 for q = dr / h, tab the
// kernel's table with its zero entry at LTAB_N - 1, CUBIC whether the seam term of
// the cubic spline applies.  The table position is clamped to that zero entry, so q >= 1 reads
// it (and the seam term is zero beyond q = 1/2): no mask, and the row is read
// for every pixel (no branch around the LDS load).
template <bool CUBIC>
__device__ inline float table_weight_select(const float4* __restrict__ tab, float x2, float fb) {
    const float x = fminf(__builtin_amdgcn_sqrtf(x2), (float)WTAB_N);
    const int i = (int)x;
    const float t = __builtin_amdgcn_fractf(x);
    const float4 c = tab[i];
    float w = fmaf(fmaf(fmaf(c.w, t, c.z), t, c.y), t, c.x);
    if (CUBIC) {  // R2 sqrt(1 - R2) / (8 * 1.5969), R2 = 4 q^2, zero for R2 >= 1
        constexpr double N2 = (double)WTAB_N * WTAB_N;
        w = fmaf(x2 * (float)(4.0 / (8.0 * 1.59689476201133 * N2)),
                 __builtin_amdgcn_sqrtf(fmaxf(fmaf((float)(-4.0 / N2), x2, 1.0f), 0.0f)), w);
    }
    return w * fb;
}

// Fills gt for the chunk's Gaussian particles (cs.gmask): thread t takes
// particle t % KC and rows (then columns) t / KC, t / KC + NT / KC, ... of its
// clipped footprint.  Loops end once no lane of the wave has a row (column)
// left.  The values are weight_at's: the same offsets and spans.
__device__ inline void fill_gauss_tables(const ChunkState& cs, int x0, int y0, GaussTables& gt) {
    const int k = threadIdx.x & (KC - 1), slot = threadIdx.x / KC;
    const bool gk = (cs.gmask >> k) & 1u;
    const WalkRec w = cs.walk[k];
    const int i0 = x0 + w.row(), j0 = y0 + w.col();
    const int rows = gk ? w.rows() : 0, cols = gk ? w.width() : 0;
    for (int r = slot; __any(r < rows); r += NT / KC)
        if (r < rows) gt.ex[k][r] = erf_span((float)(w.px - (double)(i0 + r)) * w.f, w.f);
    for (int c = slot; __any(c < cols); c += NT / KC)
        if (c < cols) gt.ey[k][c] = erf_span((float)(w.py - (double)(j0 + c)) * w.f, w.f);
}

// The Gaussian kernel's weight as weight_at computes it, its separable
// factors ex, ey read from the tables: zero beyond the truncation edge, and
// the truncation term zmax = sqrt(t^2 - u^2) formed in FP64.
__device__ inline float gauss_weight(double dx, double dy, double fa, double fe, float t,
                                     float n, float ex, float ey) {
    const double dr2 = dx * dx + dy * dy;
    if (dr2 > fe) return 0.0f;
    const double z2 = (double)t * (double)t - dr2 * fa;
    const float zmax = z2 > 0.0 ? __builtin_amdgcn_sqrtf((float)z2) : 0.0f;
    return 0.25f * erff(zmax * 0.70710678118654752f) * ex * ey * n;
}

// Evaluates W for every (particle, pixel) pair of the chunk and hands each
// value to store(k, PXS * pixel-in-tile, w), or two of them to
// store2(k, PXS * pixel1, w1, PXS * pixel2, w2).  Particle k's pairs (pixel row l / width,
// column l % width of its clipped footprint, l < cnt) are split over the threads
// from its first one on, `per` consecutive pairs each, so a thread stays on one
// particle.  It finds the particle by counting start bits: a search of the
// threads' scan (three dependent LDS reads and 30 instructions, for 3 or 4 pixels)
// cost 1 to 2% of an insertion (1e7 particles, split BF16: 5.04 -> 4.97 ms; 1e6,
// FP32: 556 -> 547 us).  When every
// particle of the wave's pairs uses the item's LDS table, the walk is
// branch-free and takes two pixels per step, whose evaluations overlap.
template <int PXS, class Store, class Store2>
__device__ inline void fill_weights(const ChunkState& cs, int x0, int y0,
                                    const float4* __restrict__ wtab, int tab_kind,
                                    const float4* __restrict__ tab, const GaussTables& gt,
                                    const mi_cube_desc& d, Store store, Store2 store2) {
    const int t = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint2 starts = *reinterpret_cast<const uint2*>(cs.starts + 2 * wave);
    const uint32_t before = (cs.started >> (8 * wave)) & 255u;
    const int k = (int)__builtin_amdgcn_mbcnt_hi(starts.y, __builtin_amdgcn_mbcnt_lo(starts.x, before));
    const int per = cs.per();
    const WalkRec w = cs.walk[k];
    const int width = max(w.width(), 1), kind = w.kind();
    const int l0 = (t - w.first()) * per;
    const int l1 = min(l0 + per, w.rows() * w.width());
    const bool active = l0 < l1;
    const int ti = w.row(), tj = w.col();  // footprint corner in the tile

    if (tab_kind >= 0 && __all(!active || kind == tab_kind)) {
        // x^2 in FP32 from the offset in table intervals, a few ulps from the FP64
        // form, far below the table's own error.  (Offsets in pixels cost two more
        // products a pixel: 3e6 heterogeneous particles, FP32, 3.45 -> 3.41 ms with
        // the shorter addresses of put and put2.)
        const float gx = tile_offset(w).x, gy = tile_offset(w).y;
        const float f = w.f, fb = inv_h2(w);
        // Pixel l of the footprint lies in row floor((l + 1/2) / width) (exact, as
        // for a above) and column l - row * width, all small integers formed in
        // FP32: no wrap tests, and the offsets from the particle need no
        // conversion.  Its index in the tile is row * TILE_Y + column + corner.
        const float rw = __builtin_amdgcn_rcpf((float)width), wf = (float)width;
        const float hrw = 0.5f * rw, corner = (float)(PXS * (ti * TILE_Y + tj));
        auto at = [&](float lf, float& af, float& bf) {
            af = floorf(fmaf(lf, rw, hrw));  // (l + 1/2) / width, one rounding
            bf = fmaf(-af, wf, lf);
        };
        auto px_of = [&](float af, float bf) {
            return (int)fmaf(af, (float)(PXS * TILE_Y), fmaf(bf, (float)PXS, corner));
        };
        auto walk = [&](auto cubic) {
            auto eval = [&](float af, float bf) {
                const float dx = fmaf(-af, f, gx), dy = fmaf(-bf, f, gy);
                return table_weight_select<decltype(cubic)::value>(tab, fmaf(dx, dx, dy * dy), fb);
            };
            float lf = (float)l0;
            const float lend = (float)l1;
            for (; lf + 1.0f < lend; lf += 2.0f) {
                float a1, b1, a2, b2;
                at(lf, a1, b1);
                at(lf + 1.0f, a2, b2);
                const float v1 = eval(a1, b1), v2 = eval(a2, b2);
                store2(k, px_of(a1, b1), v1, px_of(a2, b2), v2);
            }
            if (lf < lend) {
                float a1, b1;
                at(lf, a1, b1);
                store(k, px_of(a1, b1), eval(a1, b1));
            }
        };
        if (tab_kind == MI_KERNEL_CUBIC)  // uniform
            walk(std::true_type{});
        else
            walk(std::false_type{});
        return;
    }

    // l0 / width: (l0 + 1/2) / width lies at least 1/32 from an integer (l0 <
    // 256 pixels, width <= 16), far beyond the reciprocal's error
    int a = (int)(((float)l0 + 0.5f) * __builtin_amdgcn_rcpf((float)width));
    int b = l0 - a * width;
    if (kind == MI_KERNEL_TABLE) {
        // the caller's weights (binning checked that they lie inside the table)
        const TableWalk tw = table_walk(w);
        for (int l = l0; l < l1; ++l) {
            const int i = x0 + ti + a, j = y0 + tj + b;
            store(k, PXS * ((ti + a) * TILE_Y + tj + b), d.weights[tw.base + (int64_t)i * tw.stride + j]);
            if (++b == width) {
                b = 0;
                ++a;
            }
        }
        return;
    }
    if (kind == MI_KERNEL_GAUSS || !active) {
        // Gaussian particles: the separable factors come from the chunk's tables
        const GaussRec gg = cs.gr[k];
        const int gi = w.gidx();
        const float gt_t = pick4(d.gauss_t, gi), gt_n = pick4(d.gauss_inv_norm, gi);
        for (int l = l0; l < l1; ++l) {
            const int i = x0 + ti + a, j = y0 + tj + b;
            store(k, PXS * ((ti + a) * TILE_Y + tj + b),
                  gauss_weight(w.px - (double)i, w.py - (double)j, gg.a, gg.e, gt_t, gt_n,
                               gt.ex[k][a], gt.ey[k][b]));
            if (++b == width) {
                b = 0;
                ++a;
            }
        }
        return;
    }
    const float fb = inv_h2(w);
    const WFactors f{(double)fb, 0.0, fb, 0.0f, 0.0f};
    const GaussRec at = cs.gr[k];
    for (int l = l0; l < l1; ++l) {
        const int i = x0 + ti + a, j = y0 + tj + b;
        store(k, PXS * ((ti + a) * TILE_Y + tj + b),
              weight_at(kind, at.a - (double)i, at.e - (double)j, f, wtab, tab_kind, tab));
        if (++b == width) {
            b = 0;
            ++a;
        }
    }
}

constexpr double LOG2E = 1.4426950408889634074;
constexpr float SQRT_LOG2E = 1.20112240878645110f;

// The flux of a Gaussian line of unit width in a channel of span D about m,
//   amp / 2 (erf(m + D/2) - erf(m - D/2))
//     = amp D / sqrt(pi) sum_k D^2k / (4^k (2k + 1)!) d^2k/dm^2k exp(-m^2)
//     = exp(-m^2) sum_j e_j m^2j,
// the sum over k to K (span_series' terms for K = 3); the e_j are formed once per
// particle.  SCALED: as exp2(-n^2) times a polynomial in n^2 of n = m sqrt(log2 e),
// a product less per channel and n's factor rounded once for all channels.  The first
// term left out is D^(2K+2) / (4^(K+1) (K+1)! (2K+3)) of the peak at most: 7e-8 for
// K = 3, D = 1/2 (1.2e-9 at 0.3) and 8e-10 for K = 8, D = 3/2.  In the line's last
// channels, at 1e-7 of the peak and less, it is 2.3e-4 and 1.3e-6 of the value.
template <int K, bool SCALED, bool EXACT>
struct LineSeries {
    float e[K + 1];

    // 1 / sqrt(pi) in FP32 is 5e-8 too large, for every line alike.  EXACT: the
    // coefficients take that back (1 - 5e-8 is within 1e-8 of an FP32 number).  The split
    // form's narrow lines keep it, as they had it before the series: its chains over all
    // of an item's chunks come out low by as much or more on the longest (error against
    // FP64 of 1e7 particles, 512 x 512 x 256: 1.3e-7, 1.5e-7 without it; 1.5e6: 2.67e-7,
    // 2.75e-7; 1.6e5, sparse: 4.43e-7 either way; 1e6, 256 x 256 x 128: 1.43e-7, 1.31e-7).
    static constexpr float ROOT = 0.564189583547756287f;
    // c[k][j]: of D^2k m^2j (the Hermite polynomials' coefficients)
    struct Table {
        float c[K + 1][K + 1];
    };
    static constexpr Table table() {
        Table t{};
        // 1 / (2 j)!, its scale included, and (-1)^i / (4^i i!)
        double inv_2j[K + 1] = {}, inv_i[K + 1] = {};
        double a = EXACT ? 0.564189583547756287 / (double)ROOT : 1.0, b = 1.0;
        for (int j = 0; j <= K; ++j) {
            inv_2j[j] = a;
            inv_i[j] = b;
            a /= (2 * j + 1) * (2 * j + 2) * (SCALED ? LOG2E : 1.0);
            b /= -4.0 * (j + 1);
        }
        for (int k = 0; k <= K; ++k)
            for (int j = 0; j <= k; ++j) t.c[k][j] = (float)(inv_i[k - j] * inv_2j[j] / (2 * k + 1));
        return t;
    }
    __device__ LineSeries(float s, float amp) {
        constexpr Table T = table();
        const float D2 = s * s;
        float f = amp * ROOT * s;
#pragma unroll
        for (int j = 0; j <= K; ++j) {
            float c = T.c[K][j];
#pragma unroll
            for (int k = K - 1; k >= j; --k) c = fmaf(c, D2, T.c[k][j]);
            e[j] = f * c;
            f *= D2;
        }
    }
    __device__ float polynomial(float x) const {
        float p = e[K];
#pragma unroll
        for (int j = K - 1; j >= 0; --j) p = fmaf(p, x, e[j]);
        return p;
    }
    // at n (SCALED)
    __device__ float operator()(float n) const {
        const float n2 = n * n;
        return __builtin_amdgcn_exp2f(-n2) * polynomial(n2);
    }
    // at m = s d (not SCALED), m^2 and its logarithm to base 2 carried to twice FP32's
    // precision: they reach 22 there, and a rounding of 2^-24 of that is 1.3e-6 of the value.
    __device__ float at(float s, float d) const {
        const float m = s * d, ml = fmaf(s, d, -m);
        const float m2 = m * m, m2l = fmaf(m + m, ml, fmaf(m, m, -m2));
        const float y = m2 * (float)LOG2E, yl = fmaf(m2, (float)LOG2E, -y);
        const float g = __builtin_amdgcn_exp2f(-y);
        // g is zero long before the polynomial overflows: its argument ends there
        return fmaf(-g, fmaf(yl, 0.693147181f, m2l), g) * polynomial(fminf(m2, 256.0f));
    }
};

// Evaluates S for the chunk's KC particles x CB channels of the cell and
// hands the values to store2(k, block, r, s1, s2), the channels r and r + 8 of
// the 16-channel block of one particle at a time; channels outside its window give 0.  Thread t takes particle t % KC and the channels t / KC + 8 i, so its
// record fields are read once.  Only the 16-channel blocks set in `blocks`
// (wave-uniform) are evaluated; the others are left untouched.  In the FP32 form,
// returns whether the thread left out a value of the caller's table that is not finite.  The values
// are line_flux's to FP32 rounding (channels up to half a line width by the same series
// with its polynomial expanded, up to 3/2 by a longer one in place of an erf difference),
// computed as straight-line code (the window test is one unsigned compare and a
// select) so that the evaluations of a thread overlap.
template <int CB, bool FP32, class Store2>
__device__ inline bool fill_spectra(const ChunkState& cs, int c0, const mi_cube_desc& d,
                                    Store2 store2,
                                    uint32_t blocks = (1u << (CB / 16)) - 1u) {
    constexpr int PER_BLOCK = 16 / (NT / KC);  // a thread's channels in one 16-channel block
    static_assert(PER_BLOCK == 2, "a thread stores its two channels of a block together");
    const int k = threadIdx.x & (KC - 1);
    const int cl0 = threadIdx.x / KC;
    const SpecRec p = cs.p[k];
    const int k0 = p.k0;
    const float fu = p.fu, s = p.s, amp = p.amp;
    const int spectrum = d.spectrum;
    // Channel cl0 + o of the cell lies in the window when (unsigned)(o - w0) <= wl.
    const int w0 = cs.walk[k].win_lo() - cl0;
    const uint32_t wl = cs.walk[k].win_past();
    auto inside = [&](int o) { return (uint32_t)(o - w0) <= wl; };
    auto put = [&](int b, float v0, float v1) {
        const int o0 = 16 * b, o1 = o0 + NT / KC;
        store2(k, b, cl0, inside(o0) ? v0 : 0.0f, inside(o1) ? v1 : 0.0f);
    };
    if (spectrum == MI_SPECTRUM_TABLE) {  // uniform: the caller's spectra
        bool odd = false;
#pragma unroll
        for (int b = 0; b < CB / 16; ++b) {
            if (!((blocks >> b) & 1u)) continue;
            // the row of the caller's table from the thread's first channel on
            // (channel c0 + cl0 + o is inside the window when inside(o))
            const float* row = d.spectra + ((int64_t)k0 * d.spectra_ld + c0 + cl0);
            const int o0 = (NT / KC) * (b * PER_BLOCK), o1 = o0 + NT / KC;
            const float v0 = inside(o0) ? amp * row[o0] : 0.0f, v1 = inside(o1) ? amp * row[o1] : 0.0f;
            const bool odd0 = FP32 && not_finite(v0), odd1 = FP32 && not_finite(v1);
            odd = odd || odd0 || odd1;
            store2(k, b, cl0, odd0 ? 0.0f : v0, odd1 ? 0.0f : v1);
        }
        return odd;
    }
    if (spectrum == MI_SPECTRUM_DIRAC) {  // uniform: the whole amplitude in the window
#pragma unroll
        for (int b = 0; b < CB / 16; ++b)
            if ((blocks >> b) & 1u) put(b, amp, amp);
        return false;
    }
    // Channel c = c0 + cl0 + o of this thread sits at k0 - c + fu - 1/2 = (kf - o) + fh
    // from the line centre (in channels): the first difference is exact, so that each
    // offset is rounded to its own precision (formed from the cell's first channel
    // it was off by up to 4e-6 channels: 1.2e4 particles, 256 x 256 x 128, FP32,
    // relative to FP64: 1.7e-7, 0.7e-7 so).
    const int kc = k0 - c0 - cl0;
    const float kf = (float)kc, fh = fu - 0.5f;
    // exp(-m^2) as exp2(-n^2) with n = m sqrt(log2 e).
    const float sn = s * SQRT_LOG2E;
    using Narrow = LineSeries<3, true, FP32>;
    auto narrow = [&](const Narrow& line, int o) { return line(sn * ((kf - (float)o) + fh)); };
    if (!__any(s > 0.5f)) {
        const Narrow line(s, amp);
#pragma unroll
        for (int b = 0; b < CB / 16; ++b)
            if ((blocks >> b) & 1u)  // uniform
                put(b, narrow(line, 16 * b), narrow(line, 16 * b + NT / KC));
        return false;
    }
    if (!__any(s > 1.5f)) {
        // A longer series, a third of the erf difference's work per channel (1e6 particles,
        // s = 0.62, split BF16: 382 -> 341 us per insertion; 3e5, s = 0.81: 216 -> 206).  With
        // seven terms and a plain exponent it took 325 and 203 us, and the last channels
        // at s = 3/2 were off by up to 1e-5 of their value (erf differences: 2.5e-6, now 3e-6).
        // The amplitude last: in the coefficients, which grow with s^16 and are far larger
        // than the flux beside the line, it left FP32's range from 1e36 on.
        const LineSeries<8, false, true> line(s, 1.0f);
#pragma unroll 1
        for (uint32_t left = blocks; left != 0u; left &= left - 1u) {
            const int b = __builtin_ctz(left);
            const float j = kf - (float)(16 * b);
            put(b, amp * line.at(s, j + fh), amp * line.at(s, j - (float)(NT / KC) + fh));
        }
        return false;
    }
    // Wider channels: the line spans a few channels, and the erfc differences are
    // taken only inside its window.  A loop of its own: unrolled into the narrow lines'
    // code it made the kernel too long for the instruction cache (1e7 particles,
    // narrow lines: 4.78 -> 4.67 ms; 3e6 with wide ones 3.05 -> 3.06).
    const Narrow line(s, amp);
#pragma unroll 1
    for (uint32_t left = blocks; left != 0u; left &= left - 1u) {
        const int b = __builtin_ctz(left);
        float v[PER_BLOCK];
#pragma unroll
        for (int i = 0; i < PER_BLOCK; ++i) {
            const int o = 16 * b + i * (NT / KC);
            v[i] = narrow(line, o);
            if (s > 0.5f && inside(o)) {
                const float j = (float)(kc - o);  // k0 - channel; each edge to its own precision
                v[i] = 0.5f * amp * erf_diff(s * ((j - 1.0f) + fu), s * (j + fu));
            }
        }
        put(b, v[0], v[1]);
    }
    return false;
}

// Copies the table of the kernel kind of the item's first particle (when it
// is a tabulated kind) into LDS, with a zero entry after it; returns that
// kind, or -1.  Particles of one
// cell are sorted with the tabulated kinds first, so this is the table the
// item uses (a second tabulated kind in the same cell reads the global copy).
// The copy is complete after the next __syncthreads().
__device__ inline int stage_table(const mi_particle* __restrict__ P,
                                  const uint32_t* __restrict__ order, int begin,
                                  const float4* __restrict__ wtab, float4* local) {
    const int kind = kind_of(P[order[begin]].r_kind);
    if (kind > MI_KERNEL_QUARTIC) return -1;
    for (int e = threadIdx.x; e < WTAB_N; e += NT) local[e] = wtab[kind * WTAB_N + e];
    if (threadIdx.x == 0) local[WTAB_N] = make_float4(0.f, 0.f, 0.f, 0.f);
    return kind;
}

// Cell coordinates of a work item.
struct CellPos {
    int x0, y0, c0;
};

__device__ inline CellPos cell_pos(int cell, const Grid& g) {
    const int cb = cell % g.ncb;
    const int txy = cell / g.ncb;
    return CellPos{(txy / g.nty) << g.tx_shift, (txy % g.nty) << g.ty_shift, cb << g.cb_shift};
}

}  // namespace mi
