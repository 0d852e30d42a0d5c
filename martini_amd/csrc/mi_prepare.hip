// FP64 setup on the device: raw particle arrays (positions, velocities,
// masses, smoothing lengths, temperatures) -> mi_particle records, pruned and
// compacted in input order.  The same sequence the host runs in
// martini_amd (sources.py / datacube.py / sph_kernels.py / martini.py /
// _pack.py), restating:
//   SPHSource.rotate and the observed frame     sph_source.py:276-296, :442-526
//   sky coordinates                              sph_source.py:265-326
//   TAN + linear spectral WCS                    datacube.py:426-486, sph_source.py:328-362
//   smoothing lengths, adaptive choice, ranges   sph_kernels.py:235-262, :1241-1274
//   pruning                                      martini.py:168-241
//   thermal line width                           spectral_models.py:465-485
// Everything is FP64; the records carry the same integer/fraction splits as
// the host packer.
//
// One pass over the particles: every work group sets up PREP_SPAN of them,
// packs the records it keeps in LDS, finds its place in the output by a
// decoupled look-back over the groups before it, and copies its records there.
#include <hip/hip_runtime.h>

#include <cmath>

#include "../../include/martini_mi355x.h"
#include "mi_device.h"
#include "mi_internal.h"
#include "mi_lookback.h"

namespace mi {

constexpr double PI = 3.14159265358979323846;
constexpr double DEG_PER_RAD = 180.0 / PI;
constexpr double RAD_PER_DEG = PI / 180.0;
constexpr double ARCSEC_PER_RAD = 180.0 / PI * 3600.0;
constexpr double K_B = 1.380649e-23;       // J/K
constexpr double M_P = 1.67262192369e-27;  // kg
constexpr double HI_FREQ = 1.420405751e9;  // Hz
constexpr double C_LIGHT = 299792458.0;    // m/s
constexpr double MHI_TO_JY = 2.36e5;
constexpr double WINDOW_ARG = 4.0;         // erf argument of the spectral window edge
constexpr double MAX_INDEX = 2097152.0;    // 2^21: |pixel coordinate| bound
constexpr double MAX_RANGE = 4194304.0;    // 2^22: r bound (r_kind has 24 bits for it)

struct Setup {
    bool keep;
    uint32_t flags;
    uint64_t mask_px;  // pixels of the reference's square mask inside the padded cube
    mi_particle rec;
};

__device__ inline void matvec(const double* m, const double* v, double* out) {
    out[0] = m[0] * v[0] + m[1] * v[1] + m[2] * v[2];
    out[1] = m[3] * v[0] + m[4] * v[1] + m[5] * v[2];
    out[2] = m[6] * v[0] + m[7] * v[1] + m[8] * v[2];
}

// The cube centre's sines and cosines, formed once on the host.
struct Centre {
    double sin_a0, cos_a0, sin_d0, cos_d0;
};

__device__ Setup setup_particle(int64_t i, const double* __restrict__ xyz,
                                const double* __restrict__ vxyz, const double* __restrict__ mHI,
                                const double* __restrict__ hsm, const double* __restrict__ T,
                                const double* __restrict__ edges, const mi_observation& o,
                                const Centre& c) {
    Setup S;
    S.flags = 0;
    // source frame: the source's rotation, then the observed frame
    double x0[3] = {xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2]};
    double v0[3] = {vxyz[3 * i], vxyz[3 * i + 1], vxyz[3 * i + 2]};
    double xr[3], vr[3];
    matvec(o.rotation, x0, xr);
    matvec(o.rotation, v0, vr);
    const double xk[3] = {xr[0] / 1000.0, xr[1] / 1000.0, xr[2] / 1000.0};
    double pos[3], vel[3];
    matvec(o.sky_rotation, xk, pos);
    matvec(o.sky_rotation, vr, vel);
    const double hub = o.hubble_h * 100.0;
    for (int a = 0; a < 3; ++a) {
        pos[a] += o.distance_mpc * o.pointing[a];
        vel[a] += hub * pos[a] + o.vpeculiar_kms * o.pointing[a];
    }
    const double dist = sqrt(pos[0] * pos[0] + pos[1] * pos[1] + pos[2] * pos[2]);
    const double vlos = (pos[0] * vel[0] + pos[1] * vel[1] + pos[2] * vel[2]) / dist;

    // TAN projection about the cube centre, RA to the left.  With the position
    // (X, Y, Z) = dist (cos dec cos ra, cos dec sin ra, sin dec), the angles'
    // products are ratios of linear forms in it: no inverse trigonometry, and
    // no rounding of a right ascension near 360 degrees.
    double X = pos[0], Y = pos[1], Z = pos[2];
    if (!(dist < INFINITY) || dist < 0x1p-500) {
        if (isinf(X) || isinf(Y) || isinf(Z)) {  // the direction that atan2 gives them
            X = isinf(X) ? copysign(1.0, X) : X - X;
            Y = isinf(Y) ? copysign(1.0, Y) : Y - Y;
            const double across = sqrt(X * X + Y * Y);
            Z = isinf(Z) ? copysign(across > 0.0 ? across : 1.0, Z) : Z - Z;
        } else {  // components whose squares leave the range still have one
            const double k = dist < 1.0 ? 0x1p600 : 0x1p-600;
            X *= k;
            Y *= k;
            Z *= k;
        }
        if (X == 0.0 && Y == 0.0 && Z == 0.0) X = 1.0;  // the observer: both angles zero
    }
    const double across = Y * c.cos_a0 - X * c.sin_a0;  // cos dec sin(ra - a0)
    const double along = X * c.cos_a0 + Y * c.sin_a0;   // cos dec cos(ra - a0)
    const double den = Z * c.sin_d0 + along * c.cos_d0;
    const double nan = __builtin_nan("");
    double x = nan, y = nan;
    if (den > 0.0) {
        const double xi = across / den * DEG_PER_RAD;
        const double eta = (Z * c.cos_d0 - along * c.sin_d0) / den * DEG_PER_RAD;
        x = o.crpix[0] - 1.0 + xi / o.cdelt[0];
        y = o.crpix[1] - 1.0 + eta / o.cdelt[1];
    }
    const double v_ms = vlos * 1e3;
    const double spec = o.freq_channels ? HI_FREQ * (1.0 - v_ms / C_LIGHT) : v_ms;
    const double z = o.crpix[2] - 1.0 + (spec - o.crval2) / o.cdelt[2];

    // smoothing length in pixels and the kernel tier
    const double h_px = atan(hsm[i] / (dist * 1000.0)) * ARCSEC_PER_RAD / o.px_size_arcsec;
    int use = 0;
    if (o.n_tiers > 1) {
        int idx = -1;
        for (int k = 0; k < o.n_tiers && idx < 0; ++k) {
            const double he = h_px * o.tier_rescale[k];
            if (he >= o.tier_min[k] && he <= o.tier_max[k]) idx = k;
        }
        if (idx < 0) S.flags |= MI_PREP_INVALID_KERNEL;
        use = idx < 0 ? 0 : idx;
    } else if (!(h_px >= o.tier_min[0] && h_px <= o.tier_max[0])) {
        S.flags |= MI_PREP_INVALID_KERNEL;  // a fixed kernel validates the raw h_px
    }
    const double r = ceil(h_px * o.tier_size[use]);
    const double h_eff = h_px * o.tier_rescale[use];
    const int kind = o.tier_kind[use];

    // line width (km/s) and pruning
    const double m = mHI[i];
    double sigma = 0.0;
    if (o.spectrum == MI_SPECTRUM_GAUSS)
        sigma = o.sigma_kms >= 0.0 ? o.sigma_kms : sqrt(K_B * T[i] / M_P) / 1000.0;
    bool reject = false;
    if (o.prune) {
        const double hw = sigma / o.dv_max_kms;
        const int nxp = o.nx + 2 * o.padx, nyp = o.ny + 2 * o.pady;
        reject = (x + r < 0.0) || (y + r < 0.0) || (x - r > (double)nxp) || (y - r > (double)nyp) ||
                 isnan(x) || isnan(y) || (z + 4.0 * hw < 0.0) || (z - 4.0 * hw > (double)o.nc) ||
                 m == 0.0;
    }
    S.keep = !reject;
    S.mask_px = 0;
    if (!S.keep) {
        S.flags = 0;
        return S;
    }

    // record: footprint fields (_pack.kernel_fields), padded extent
    const int nx = o.nx + 2 * o.padx, ny = o.ny + 2 * o.pady;
    const bool alive = isfinite(x) && isfinite(y) && r >= 0.0 && x + r >= 0.0 && y + r >= 0.0 &&
                       x - r <= (double)(nx - 1) && y - r <= (double)(ny - 1);
    if (alive) {  // |i - x| <= r, |j - y| <= r (martini.py:271-274) within the padded cube
        const double mx = fmin((double)(nx - 1), floor(x + r)) - fmax(0.0, ceil(x - r)) + 1.0;
        const double my = fmin((double)(ny - 1), floor(y + r)) - fmax(0.0, ceil(y - r)) + 1.0;
        if (mx > 0.0 && my > 0.0) S.mask_px = (uint64_t)mx * (uint64_t)my;
    }
    const double xs = alive ? x : 0.0, ys = alive ? y : 0.0;
    if (fabs(xs) >= MAX_INDEX || fabs(ys) >= MAX_INDEX) S.flags |= MI_PREP_COORD_LIMIT;
    double ix = floor(xs), iy = floor(ys);
    double fx = xs - ix, fy = ys - iy;
    double rr = alive ? fmin(r, MAX_RANGE) : -1.0;
    if (kind == MI_KERNEL_DIRAC) {
        const double pi_ = floor(xs + 0.5), pj = floor(ys + 0.5);
        const bool ok = fabs(xs - pi_) < 0.5 && fabs(ys - pj) < 0.5 && fabs(xs - pi_) <= rr &&
                        fabs(ys - pj) <= rr && pi_ >= 0.0 && pi_ <= (double)(nx - 1) && pj >= 0.0 &&
                        pj <= (double)(ny - 1) && alive;
        ix = pi_;
        iy = pj;
        fx = 0.0;
        fy = 0.0;
        rr = ok ? 0.0 : -1.0;
    }
    mi_particle& p = S.rec;
    p.ix = (int32_t)ix;
    p.iy = (int32_t)iy;
    p.fx = (float)fx;
    p.fy = (float)fy;
    p.h = (float)h_eff;
    p.r_kind = (int32_t)((int64_t)rr * 256 + (int64_t)o.tier_gidx[use] * 16 + kind);

    // spectral fields (_pack.spectral_fields)
    const int nc = o.nc;
    const double u = (v_ms - o.e0_ms) / o.de_ms;
    const bool finite = isfinite(u);
    const double uu = finite ? u : 0.0;
    const double k0 = floor(uu);
    const double fu = uu - k0;
    const double ade = fabs(o.de_ms);
    const double amp = m * (1.0 / (dist * dist)) / (ade / 1e3) / MHI_TO_JY * o.out_scale;
    double c_lo, c_hi, s = 0.0;
    if (o.spectrum == MI_SPECTRUM_GAUSS) {
        s = ade / (1.4142135623730951 * sigma * 1e3);
        const double half = WINDOW_ARG / s;
        c_lo = floor(uu - 1.0 - half) + 1.0;
        c_hi = ceil(uu + half) - 1.0;
    } else {
        c_lo = INFINITY;
        c_hi = -INFINITY;
        for (int dd = -1; dd <= 1; ++dd) {
            const double cf = k0 + dd;
            const int c = (int)fmin(fmax(cf, 0.0), (double)(nc - 1));
            const double lo_e = fmin(edges[c], edges[c + 1]), hi_e = fmax(edges[c], edges[c + 1]);
            if (v_ms >= lo_e && v_ms <= hi_e && finite && cf >= 0.0 && cf <= (double)(nc - 1)) {
                c_lo = fmin(c_lo, (double)c);
                c_hi = fmax(c_hi, (double)c);
            }
        }
    }
    c_lo = fmin(fmax(finite ? c_lo : (double)nc, 0.0), (double)nc);
    c_hi = fmin(fmax(finite ? c_hi : -1.0, -1.0), (double)(nc - 1));
    if (c_lo > c_hi) {
        c_lo = 1.0;
        c_hi = 0.0;
    }
    // a shared cube addresses this source's channels from channel_offset on
    const bool empty = c_lo > c_hi;
    p.c_lo = (int32_t)c_lo + (empty ? 0 : o.channel_offset);
    p.c_hi = (int32_t)c_hi + (empty ? 0 : o.channel_offset);
    p.k0 = (int32_t)fmin(fmax(k0, -1073741824.0), 1073741824.0) + o.channel_offset;
    p.fu = (float)fu;
    p.s = (float)s;
    p.amp = (float)amp;
    return S;
}

// A work group takes PREP_R rounds of PREP_T particles: 512 of them share one
// look-back word and one ticket (requests to one cache line from all eight XCDs
// are served one after another, about 11 ns each), and their records take
// 24 KB of LDS, so six groups fit a CU.
constexpr int PREP_T = 256;
constexpr int PREP_R = 2;
constexpr int PREP_SPAN = PREP_T * PREP_R;

__host__ __device__ inline int64_t prep_groups(int64_t n) { return (n + PREP_SPAN - 1) / PREP_SPAN; }

// What a group adds to the totals (besides its records).
struct PrepSums {
    unsigned long long pairs, px, flags;
};

__global__ void k_prep_init(unsigned long long* __restrict__ counts,
                            unsigned long long* __restrict__ look, uint32_t* __restrict__ ticket,
                            int64_t groups) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < groups) look[i] = 0ull;
    if (i < 4) counts[i] = 0ull;
    if (i == 0 && ticket) *ticket = 0u;
}

__device__ inline unsigned long long wave_sum(unsigned long long v) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

// Bound by the FP64 setup of a particle and by HBM (72 bytes read, 48 written).
// Two passes (flags, scan, then the setup again with the records written at
// their offsets and up to four atomics per wave on one cache line) took 387 +
// 38 us for 1e6 particles, most of it in those atomics; this one takes 63 us
// (1.9 TB/s), and the whole call with its counters read back 482 -> 117 us.
// Groups of 256 particles make it 127 us, of 1024 117 us; held to 128 registers
// (four waves per SIMD instead of three) it spills and takes 130 us.
__global__ __launch_bounds__(PREP_T) void k_prepare(
    const double* __restrict__ xyz, const double* __restrict__ vxyz,
    const double* __restrict__ mHI, const double* __restrict__ hsm, const double* __restrict__ T,
    const double* __restrict__ edges, int64_t n, mi_observation o, Centre ctr,
    Grid g, mi_particle* __restrict__ out, unsigned long long* __restrict__ counts,
    unsigned long long* __restrict__ look, uint32_t* __restrict__ ticket,
    PrepSums* __restrict__ sums) {
    __shared__ uint4 recs[PREP_SPAN * 3];  // the kept records, packed
    __shared__ uint32_t s_group, s_base, wcnt[PREP_R][PREP_T / 64];
    __shared__ PrepSums wsum[PREP_T / 64];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (t == 0)
        s_group = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int64_t group = s_group;
    unsigned long long pairs = 0, px = 0;
    uint32_t flags = 0, kept = 0;
#pragma unroll 1
    for (int r = 0; r < PREP_R; ++r) {
        const int64_t i = group * PREP_SPAN + r * PREP_T + t;
        Setup S;
        S.keep = false;
        if (i < n) S = setup_particle(i, xyz, vxyz, mHI, hsm, T, edges, o, ctr);
        const uint64_t mask = __ballot(S.keep);
        if (lane == 0) wcnt[r][wave] = (uint32_t)__builtin_popcountll(mask);
        __syncthreads();
        uint32_t at = kept + (uint32_t)__builtin_popcountll(mask & ((1ull << lane) - 1ull));
#pragma unroll
        for (int w = 0; w < PREP_T / 64; ++w) {
            at += w < wave ? wcnt[r][w] : 0u;
            kept += wcnt[r][w];
        }
        if (S.keep) {
            int a, b, c, d, e, f;
            pairs += cells_of(S.rec, g, a, b, c, d, e, f);
            flags |= S.flags;
            px += S.mask_px;
            uint4 words[3];
            __builtin_memcpy(words, &S.rec, sizeof(words));
#pragma unroll
            for (int q = 0; q < 3; ++q) recs[at * 3 + q] = words[q];
        }
    }
    if (t == 0) look_store(&look[group], (group == 0 ? LB_ALL : LB_GROUP) | kept);
    pairs = wave_sum(pairs);
    px = wave_sum(px);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) flags |= __shfl_xor(flags, d, 64);
    if (lane == 0) wsum[wave] = PrepSums{pairs, px, flags};
    if (wave == 0) {
        const uint32_t base = (uint32_t)look_back(look, group);  // records kept before this group's
        if (lane == 0) {
            s_base = base;
            if (group > 0) look_store(&look[group], LB_ALL | (base + kept));
            if (group == prep_groups(n) - 1) counts[0] = (unsigned long long)base + kept;
        }
    }
    __syncthreads();
    if (t == 0) {
        PrepSums s = wsum[0];
#pragma unroll
        for (int w = 1; w < PREP_T / 64; ++w) {
            s.pairs += wsum[w].pairs;
            s.px += wsum[w].px;
            s.flags |= wsum[w].flags;
        }
        sums[group] = s;
    }
    uint4* dst = reinterpret_cast<uint4*>(out + s_base);
    for (uint32_t e = t; e < kept * 3u; e += PREP_T) dst[e] = recs[e];
}

// The groups' sums into counts[1..3] (integers: any order gives the same).
constexpr int PREP_SUM_T = 1024;

__global__ __launch_bounds__(PREP_SUM_T) void k_prep_totals(const PrepSums* __restrict__ sums,
                                                            int64_t groups,
                                                            unsigned long long* __restrict__ counts) {
    __shared__ PrepSums w[PREP_SUM_T / 64];
    PrepSums s{0, 0, 0};
    for (int64_t i = threadIdx.x; i < groups; i += PREP_SUM_T) {
        s.pairs += sums[i].pairs;
        s.px += sums[i].px;
        s.flags |= sums[i].flags;
    }
    s.pairs = wave_sum(s.pairs);
    s.px = wave_sum(s.px);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) s.flags |= __shfl_xor(s.flags, d, 64);
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < PREP_SUM_T / 64; ++k) {
            s.pairs += w[k].pairs;
            s.px += w[k].px;
            s.flags |= w[k].flags;
        }
        counts[1] = s.pairs;
        counts[2] = s.flags;
        counts[3] = s.px;
    }
}

// Workspace: the groups' look-back words, the ticket, the groups' sums.
static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

hipError_t prep_layout(int64_t n, PrepLayout* L) {
    const size_t groups = (size_t)(n > 0 ? prep_groups(n) : 1);
    size_t o = 0;
    L->look = o;
    o += align256(sizeof(unsigned long long) * groups);
    L->ticket = o;
    o += align256(sizeof(uint32_t));
    L->sums = o;
    o += align256(sizeof(PrepSums) * groups);
    L->total = o;
    return hipSuccess;
}

hipError_t prepare_particles(const double* xyz, const double* vxyz, const double* mHI,
                             const double* hsm, const double* T, const double* edges, int64_t n,
                             const mi_observation& o, const Grid& g, mi_particle* out,
                             unsigned long long* counts, char* ws, const PrepLayout& L,
                             hipStream_t s) {
    const int64_t groups = n > 0 ? prep_groups(n) : 0;
    auto* look = (unsigned long long*)(ws + L.look);
    auto* ticket = (uint32_t*)(ws + L.ticket);
    auto* sums = (PrepSums*)(ws + L.sums);
    if (groups == 0) {  // no workspace needed
        hipLaunchKernelGGL(k_prep_init, dim3(1), dim3(256), 0, s, counts, look, nullptr, groups);
        return hipGetLastError();
    }
    const double a0 = o.cube_ra_deg * RAD_PER_DEG, d0 = o.cube_dec_deg * RAD_PER_DEG;
    const Centre ctr{sin(a0), cos(a0), sin(d0), cos(d0)};
    hipLaunchKernelGGL(k_prep_init, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, s, counts,
                       look, ticket, groups);
    hipLaunchKernelGGL(k_prepare, dim3((unsigned)groups), dim3(PREP_T), 0, s, xyz, vxyz, mHI, hsm,
                       T, edges, n, o, ctr, g, out, counts, look, ticket, sums);
    hipLaunchKernelGGL(k_prep_totals, dim3(1), dim3(PREP_SUM_T), 0, s, sums, groups, counts);
    return hipGetLastError();
}

}  // namespace mi
