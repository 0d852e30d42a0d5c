// On-GPU binning of particles into (pixel tile x channel block) cells.
//
// Replaces the reference's per-pixel O(N) square mask
// (martini/martini.py:271-274): every particle is listed once in each cell
// its footprint and channel window touch, and the list is sorted by
// (cell, kernel group, tile row) with a stable radix sort, so that each cell's
// particles form one contiguous, deterministic segment, spatially compact.
// Long segments are cut into work items of at most item_length() particles;
// such cells get one partial tile per item.
//
// Launches: k_bin_init, k_emit (pairs, in particle order), one k_radix per
// digit, k_cell_bounds, k_items (and k_build_items for many cells).  The kernels
// that place data by a running total (k_emit, k_radix) take it from a decoupled
// look-back (mi_lookback.h); the radix passes are those of Adinets and Merrill,
// "Onesweep: A Faster Least Significant Digit Radix Sort for GPUs", 2022.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <utility>

#include "mi_device.h"
#include "mi_internal.h"
#include "mi_lookback.h"
#include "mi_tile.h"

namespace mi {

Grid make_grid(const mi_cube_desc& d) {
    Grid g;
    g.nx = d.nx;
    g.ny = d.ny;
    g.nc = d.nc;
    g.wide = wide_cells(d.nc);
    g.tx_shift = g.wide ? 3 : 4;
    g.ty_shift = 4;
    g.cb_shift = g.wide ? 7 : 6;
    static_assert(GeoWide::TX == 8 && GeoSquare::TX == 16 && GeoWide::TY == 16 &&
                      GeoSquare::TY == 16 && GeoWide::CB == 128 && GeoSquare::CB == 64,
                  "the shifts above");
    g.ntx = (d.nx + (1 << g.tx_shift) - 1) >> g.tx_shift;
    g.nty = (d.ny + (1 << g.ty_shift) - 1) >> g.ty_shift;
    g.ncb = (d.nc + (1 << g.cb_shift) - 1) >> g.cb_shift;
    g.ncells = (int64_t)g.ntx * g.nty * g.ncb;
    int b = 1;
    while (((int64_t)1 << b) < g.ncells) ++b;
    g.cell_bits = b;
    return g;
}

// Work group shapes of the emit and radix passes.
struct GroupShape {
    int threads, items;  // items per thread
};
constexpr bool same(const GroupShape& a, const GroupShape& b) {
    return a.threads == b.threads && a.items == b.items;
}

// Emit pass: `threads` threads per group, `items` particles per thread.  Large
// groups on large inputs: a group's look-back waits for those before it, and
// the waiting groups' reads delay each other (1e7 particles: 320 us with 1024
// particles per group, 248 with 4096); small groups on small ones, so that they
// spread over the CUs.
constexpr GroupShape EMIT_SMALL{256, 1}, EMIT_MID{1024, 1}, EMIT_LARGE{1024, 4};

static GroupShape emit_shape(int64_t n) {
    return n >= 524288 ? EMIT_LARGE : n >= 65536 ? EMIT_MID : EMIT_SMALL;
}
static int64_t emit_groups(int64_t n) {
    const GroupShape e = emit_shape(n);
    const int64_t span = (int64_t)e.threads * e.items;
    return n > 0 ? (n + span - 1) / span : 0;
}

// Radix passes: tiles of `threads` x `items` pairs.  Large tiles write longer
// runs of equal digits and look back less (2.9e7 pairs, a pass: 240 us with tiles
// of 2048, 196 with 4096, 180 with 8192; rocPRIM's took 212); small inputs take
// small ones, so that they spread over the CUs.
constexpr GroupShape RADIX_TILE_SMALL{256, 4}, RADIX_TILE_MID{1024, 4}, RADIX_TILE_LARGE{1024, 8};
constexpr int64_t RADIX_MID = 131072, RADIX_LARGE = 1 << 20;
constexpr int RADIX_BITS = 8;  // at most, per pass
constexpr int RADIX_PASSES = (32 + RADIX_BITS - 1) / RADIX_BITS;
constexpr int LOCAL_ROW_BITS = 4;  // of the local order, enough for a 16-row tile's row

static GroupShape radix_shape(int64_t n_pairs) {
    return n_pairs >= RADIX_LARGE ? RADIX_TILE_LARGE
           : n_pairs >= RADIX_MID ? RADIX_TILE_MID : RADIX_TILE_SMALL;
}
static int64_t radix_tiles(int64_t n_pairs) {
    const GroupShape r = radix_shape(n_pairs);
    const int64_t tile = (int64_t)r.threads * r.items;
    return (n_pairs + tile - 1) / tile;
}

// The passes over the sorted bits, which are the cell and the kernel group and,
// as far as the passes that these take have bits left, the top of the local
// order; the stable sort keeps the record order in the rest.
struct RadixPlan {
    int begin, passes, bits;
};
static RadixPlan radix_plan(const Grid& g) {
    RadixPlan r;
    const int need = g.cell_bits + KEY_LOCAL_BITS - 8;
    r.passes = (need + RADIX_BITS - 1) / RADIX_BITS;
    const int width = std::min(r.passes * RADIX_BITS, need + LOCAL_ROW_BITS);
    r.begin = g.cell_bits + KEY_LOCAL_BITS - width;
    r.bits = (width + r.passes - 1) / r.passes;
    return r;
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

hipError_t layout_for(const Grid& g, int64_t n, int64_t n_pairs, Layout* L) {
    size_t off = 0;
    auto take = [&](size_t bytes) {
        size_t at = off;
        off = align256(off + bytes);
        return at;
    };
    const size_t np = (size_t)(n_pairs > 0 ? n_pairs : 1);
    const size_t nc = (size_t)g.ncells, nc1 = nc + 1;
    L->item_len = item_length(n_pairs);
    L->items_max = g.ncells + n_pairs / L->item_len + 1;
    L->split_max = split_cells_max(n_pairs, L->item_len, g.ncells);
    L->multi_max = partial_tiles_max(n_pairs, L->item_len, g.ncells);
    // cleared by k_bin_init, from status on
    L->status = take(sizeof(uint32_t) * ST_WORDS);
    L->hist = take(sizeof(uint32_t) * RADIX_PASSES << RADIX_BITS);
    L->cell_start = take(4 * nc);
    L->cell_end = take(4 * nc);
    L->emit_look = take(sizeof(unsigned long long) * (size_t)emit_groups(n));
    const RadixPlan r = radix_plan(g);
    L->radix_look = take(sizeof(unsigned long long) *
                         (((size_t)r.passes * (size_t)radix_tiles(n_pairs)) << r.bits));
    L->cleared = off;
    L->keys = take(4 * np);
    L->vals = take(4 * np);
    L->keys2 = take(4 * np);
    L->vals2 = take(4 * np);
    L->item_off = take(4 * nc1);
    L->multi_off = take(4 * nc1);
    L->item_pos = take(4 * nc);
    L->split_cells = take(4 * (size_t)L->split_max);
    L->items = take(sizeof(Item) * (size_t)L->items_max);
    L->partials = take(sizeof(float) * (size_t)L->multi_max * CELL_VOXELS);
    L->part_masks = take(sizeof(uint64_t) * (size_t)L->multi_max);
    L->total = off;
    return hipSuccess;
}

// Kernel families in a cell's sort order: tabulated closed forms first (the
// item stages the first one's table in LDS), then Gaussian, Dirac, and the
// caller's weight tables.
__device__ inline uint32_t kernel_group(int kind) {
    return kind == MI_KERNEL_GAUSS ? 1u
           : kind == MI_KERNEL_DIRAC ? 2u
           : kind == MI_KERNEL_TABLE ? 3u : 0u;
}

// Whether a record with a footprint can be inserted: a known kernel kind, and
// for MI_KERNEL_TABLE weights that lie inside the descriptor's table.
__device__ inline bool record_ok(const mi_particle& p, const Grid& g, const float* uw,
                                 int64_t uw_n) {
    const int kind = kind_of(p.r_kind);
    if (kind < MI_KERNEL_TABLE) return true;
    if (kind > MI_KERNEL_TABLE || uw == nullptr) return false;
    int i_lo, i_hi, j_lo, j_hi;
    if (!footprint(p, g.nx, g.ny, i_lo, i_hi, j_lo, j_hi)) return true;
    const int64_t end = (int64_t)table_offset(p) + (int64_t)(i_hi - i_lo + 1) * (j_hi - j_lo + 1);
    return end <= uw_n;
}

// Writes the (key, particle) pairs of each particle, in particle order: group b
// takes particles b * ROUNDS * T + i * T + t (rounds i, thread t), so the record
// loads of a round are contiguous.  The records are read once: a
// group holds its particles' cell ranges in registers, scans their counts and
// takes its base from the look-back.  A particle of more than EMIT_WIDE cells is
// written by its whole wave.  The digits of every radix pass are counted too
// (hist), in EMIT_COPIES copies in LDS, a lane in eight to each: neighbouring
// records share their cells, and adds to one address wait for each other.
// The low 8 key bits are the particle's tile row (LOCAL_ROW_BITS) and column in
// the cell, clamped to the tile: particles of one row side by side make the
// gather's 32-particle chunks compact, and its products are skipped by tile row.
// A total above the capacity raises the
// overflow flag; nothing is written past the capacity, and the passes that
// follow do nothing.
constexpr uint32_t EMIT_WIDE = 8;
constexpr int EMIT_COPIES = 8;

template <int T, int ROUNDS>
__global__ __launch_bounds__(T) void k_emit(
    const mi_particle* __restrict__ P, int64_t n, int64_t cap, Grid g,
    const float* __restrict__ uw, int64_t uw_n, unsigned long long* __restrict__ look,
    uint32_t* __restrict__ keys, uint32_t* __restrict__ vals, uint32_t* __restrict__ hist,
    uint32_t* __restrict__ status, int begin, int passes, int bits) {
    __shared__ uint32_t wsum[ROUNDS][T / 64];
    extern __shared__ uint32_t lhist[];  // EMIT_COPIES x ((passes << bits) + 1)
    __shared__ uint32_t s_group;
    __shared__ unsigned long long s_base;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (t == 0)
        s_group = __hip_atomic_fetch_add(&status[ST_TICKET], 1u, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t mask = (1u << bits) - 1u;
    const int digits = passes << bits, copy = digits + 1;
    for (int e = t; e < EMIT_COPIES * copy; e += T) lhist[e] = 0u;
    __syncthreads();
    const int64_t group = s_group;
    const int64_t base_k = group * (T * ROUNDS) + t;
    // tile and block ranges of the thread's particles, and their pair counts
    uint32_t tx[ROUNDS], ty[ROUNDS], kg[ROUNDS], cnt[ROUNDS], at[ROUNDS];
    int cb0[ROUNDS], cb1[ROUNDS], px[ROUNDS], py[ROUNDS];
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
        const int64_t k = base_k + (int64_t)i * T;
        cnt[i] = 0u;
        tx[i] = ty[i] = kg[i] = 0u;
        cb0[i] = cb1[i] = px[i] = py[i] = 0;
        if (k < n) {
            const mi_particle p = P[k];
            int tx0, tx1, ty0, ty1;
            cnt[i] = cells_of(p, g, tx0, tx1, ty0, ty1, cb0[i], cb1[i]);
            if (cnt[i] > 0u) {  // tile indices below 2^15
                if (!record_ok(p, g, uw, uw_n)) status[ST_BADREC] = 1u;  // same value from all
                tx[i] = (uint32_t)tx0 | (uint32_t)tx1 << 16;
                ty[i] = (uint32_t)ty0 | (uint32_t)ty1 << 16;
                kg[i] = kernel_group(kind_of(p.r_kind));
                px[i] = p.ix;
                py[i] = p.iy;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
        const uint32_t incl = (uint32_t)wave_scan_add((int)cnt[i]);
        at[i] = incl - cnt[i];
        if (lane == 63) wsum[i][wave] = incl;
    }
    __syncthreads();
    uint32_t total = 0;
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i)
#pragma unroll
        for (int w = 0; w < T / 64; ++w) {
            if (w == wave) at[i] += total;
            total += wsum[i][w];
        }
    if (wave == 0) {
        // The total again without wrapping: 4096 particles of up to 2^21 cells make up
        // to 2^33 pairs.  (In 64 bits by every thread, above, 1e7 particles took 160 us
        // more.)
        static_assert(ROUNDS * (T / 64) <= 64, "a lane per sum");
        PairSum sum(lane < ROUNDS * (T / 64) ? (&wsum[0][0])[lane] : 0u);
        sum.upper = __builtin_amdgcn_readlane(wave_scan_add((int)sum.upper), 63);
        sum.lower = __builtin_amdgcn_readlane(wave_scan_add((int)sum.lower), 63);
        const unsigned long long all = sum.total();
        if (lane == 0) look_store(&look[group], (group == 0 ? LB_ALL : LB_GROUP) | all);
        const unsigned long long b = look_back(look, group);
        if (lane == 0) {
            s_base = b + (all - total);  // past any capacity where `total` has wrapped
            if (group > 0) look_store(&look[group], LB_ALL | (b + all));
            if ((group + 1) * (T * ROUNDS) >= n) {
                status[ST_PAIRS] = (uint32_t)(b + all);
                status[ST_OVERFLOW] = b + all > (uint64_t)cap ? 1u : 0u;
            }
        }
    }
    __syncthreads();
    const unsigned long long base = s_base;
    if (base + total > (uint64_t)cap) return;  // uniform
    uint32_t* mine = lhist + (lane & (EMIT_COPIES - 1)) * copy;
    auto put = [&](uint32_t x, uint32_t y, uint32_t cb, uint32_t kind, int ix, int iy, uint32_t k,
                   size_t q) {
        const uint32_t cell = (x * (uint32_t)g.nty + y) * (uint32_t)g.ncb + cb;
        const int row = min(max(ix - (int)(x << g.tx_shift), 0), (1 << g.tx_shift) - 1);
        const int col = min(max(iy - (int)(y << g.ty_shift), 0), TILE_Y - 1);
        const uint32_t key = (cell << KEY_LOCAL_BITS) | (kind << 8) |
                             ((uint32_t)row << (8 - g.tx_shift)) |
                             ((uint32_t)col << (4 - g.tx_shift));
        keys[q] = key;
        vals[q] = k;
        for (int p = 0; p < passes; ++p)
            atomicAdd(&mine[(p << bits) + ((key >> (begin + p * bits)) & mask)], 1u);
    };
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
        const uint32_t k = (uint32_t)(base_k + (int64_t)i * T);
        if (cnt[i] > 0u && cnt[i] <= EMIT_WIDE) {
            size_t q = (size_t)base + at[i];
            for (uint32_t x = tx[i] & 0xffffu; x <= tx[i] >> 16; ++x)
                for (uint32_t y = ty[i] & 0xffffu; y <= ty[i] >> 16; ++y)
                    for (int cb = cb0[i]; cb <= cb1[i]; ++cb) 
                        put(x, y, (uint32_t)cb, kg[i], px[i], py[i], k, q++);
        }
        uint64_t wide = __ballot(cnt[i] > EMIT_WIDE);
        while (wide) {
            const int l = __builtin_ctzll(wide);
            wide &= wide - 1ull;
            auto of = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, l); };
            const uint32_t x0 = of(tx[i]) & 0xffffu, yy = of(ty[i]), y0 = yy & 0xffffu;
            const uint32_t ny = (yy >> 16) - y0 + 1u, b0 = of((uint32_t)cb0[i]);
            const uint32_t nb = of((uint32_t)cb1[i]) - b0 + 1u, n_cells = of(cnt[i]);
            const uint32_t lk = of(k), lg = of(kg[i]);
            const int lx = (int)of((uint32_t)px[i]), ly = (int)of((uint32_t)py[i]);
            const size_t q = (size_t)base + of(at[i]);
            for (uint32_t e = lane; e < n_cells; e += 64) {
                const uint32_t xy = e / nb, x = xy / ny;
                put(x0 + x, y0 + (xy - x * ny), b0 + (e - xy * nb), lg, lx, ly, lk, q + e);
            }
        }
    }
    __syncthreads();
    for (int e = t; e < digits; e += T) {
        uint32_t sum = 0;
#pragma unroll
        for (int c = 0; c < EMIT_COPIES; ++c) sum += lhist[c * copy + e];
        if (sum) atomicAdd(&hist[e], sum);
    }
}

// Pairs the emit pass produced, zero after an overflow.
__device__ inline int64_t device_pairs(const uint32_t* __restrict__ status) {
    return status[ST_OVERFLOW] ? 0 : (int64_t)status[ST_PAIRS];
}

// One stable radix pass over `bits` key bits from `shift` on.  A tile of
// T * ITEMS pairs is ranked wave by wave (each wave a contiguous run, 64
// pairs at a time, lanes of equal digit found by ballots), its digit counts are
// published, digit d's place in the output is the look-back sum of the earlier
// tiles' counts of d after all smaller digits (hist), and the tile goes out
// through LDS in sorted order, so that equal digits are written side by side.
template <int T, int ITEMS>
__global__ __launch_bounds__(T) void k_radix(
    const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals,
    uint32_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out,
    const uint32_t* __restrict__ hist, unsigned long long* __restrict__ look,
    uint32_t* __restrict__ ticket, const uint32_t* __restrict__ status, int shift, int bits) {
    constexpr int WAVES = T / 64, TILE = T * ITEMS, RADIX = 1 << RADIX_BITS;
    static_assert(T >= RADIX, "a thread per digit");
    __shared__ uint32_t whist[WAVES][RADIX];
    __shared__ uint32_t tbase[RADIX], gbase[RADIX];
    __shared__ uint32_t wtot[2][WAVES];
    __shared__ uint32_t skey[TILE], sval[TILE];
    __shared__ uint32_t s_tile;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (t == 0)
        s_tile = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int e = t; e < WAVES * RADIX; e += T) (&whist[0][0])[e] = 0u;
    __syncthreads();
    const int64_t tile = s_tile, np = device_pairs(status);
    const int64_t begin = tile * TILE;
    if (begin >= np) return;  // uniform
    const int count = (int)min((int64_t)TILE, np - begin);
    const uint32_t mask = (1u << bits) - 1u;

    uint32_t key[ITEMS], val[ITEMS], rank[ITEMS];
    const int first = wave * 64 * ITEMS + lane;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const int e = first + i * 64;
        key[i] = e < count ? keys[begin + e] : 0xffffffffu;
        val[i] = e < count ? vals[begin + e] : 0u;
    }
    volatile uint32_t* mine = whist[wave];  // read and written by this wave only, in order
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t d = (key[i] >> shift) & mask;
        uint64_t peers = __ballot(first + i * 64 < count);
        for (int b = 0; b < bits; ++b) {  // uniform
            const bool one = (d >> b) & 1u;
            const uint64_t m = __ballot(one);
            peers &= one ? m : ~m;
        }
        const uint32_t before = (uint32_t)__builtin_popcountll(peers & ((1ull << lane) - 1ull));
        const uint32_t old = mine[d];
        rank[i] = old + before;
        if (first + i * 64 < count && before == 0u)
            mine[d] = old + (uint32_t)__builtin_popcountll(peers);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // thread d: this tile's count of digit d; the waves' offsets within it
    uint32_t mycount = 0;
    if (t < RADIX) {
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const uint32_t c = whist[w][t];
            whist[w][t] = mycount;
            mycount += c;
        }
    }
    const int radix = 1 << bits;
    unsigned long long* word = look + (tile << bits) + t;
    if (t < radix) look_store(word, (tile == 0 ? LB_ALL : LB_GROUP) | mycount);
    // exclusive scans over the digits: of the tile's counts and of all counts
    const uint32_t all = t < radix ? hist[t] : 0u;
    const uint32_t i0 = (uint32_t)wave_scan_add((int)mycount), i1 = (uint32_t)wave_scan_add((int)all);
    if (lane == 63) {
        wtot[0][wave] = i0;
        wtot[1][wave] = i1;
    }
    __syncthreads();
    uint32_t tb = i0 - mycount, gb = i1 - all;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
        if (w < wave) {
            tb += wtot[0][w];
            gb += wtot[1][w];
        }
    if (t < radix) {
        // four earlier tiles at a time, nearest first
        unsigned long long before = 0;
        int64_t j = 1;
        for (bool done = tile == 0; !done;) {
            unsigned long long v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                v[i] = j + i <= tile ? look_load(word - ((j + i) << bits)) : LB_ALL;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (done || (v[i] & LB_STATE) == 0ull) break;  // not published yet: read again
                before += v[i] & ~LB_STATE;
                done = (v[i] & LB_STATE) == LB_ALL;
                ++j;
            }
        }
        if (tile > 0) look_store(word, LB_ALL | (before + mycount));
        tbase[t] = tb;
        gbase[t] = gb + (uint32_t)before - tb;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if (first + i * 64 >= count) continue;
        const uint32_t d = (key[i] >> shift) & mask;
        const uint32_t at = tbase[d] + whist[wave][d] + rank[i];
        skey[at] = key[i];
        sval[at] = val[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const int e = t + i * T;
        if (e >= count) continue;
        const uint32_t k = skey[e];
        const size_t o = (size_t)(uint32_t)(gbase[(k >> shift) & mask] + (uint32_t)e);
        keys_out[o] = k;
        vals_out[o] = sval[e];
    }
}

// Clears the status words, histograms, cell bounds (cells without particles
// keep start = end = 0) and look-back words: `words` 16-byte words.
__global__ void k_bin_init(uint4* __restrict__ at, int64_t words) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < words; k += stride)
        at[k] = make_uint4(0u, 0u, 0u, 0u);
}

// Cell bounds from the sorted keys: thread t takes keys 4t .. 4t + 3 (one
// 16-byte load when the run lies inside the array, the workspace keys being
// 256-byte aligned) and the key on either side.
__global__ void k_cell_bounds(const uint32_t* __restrict__ keys,
                              const uint32_t* __restrict__ status, int64_t ncells,
                              uint32_t* __restrict__ start, uint32_t* __restrict__ end) {
    const int64_t np = device_pairs(status);
    const int64_t q0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (q0 >= np) return;
    uint32_t c[6];  // cells of keys q0 - 1 .. q0 + 4 (0xffffffff outside the array)
    if (q0 + 4 <= np) {
        const uint4 v = *reinterpret_cast<const uint4*>(keys + q0);
        c[1] = v.x >> KEY_LOCAL_BITS;
        c[2] = v.y >> KEY_LOCAL_BITS;
        c[3] = v.z >> KEY_LOCAL_BITS;
        c[4] = v.w >> KEY_LOCAL_BITS;
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i + 1] = q0 + i < np ? keys[q0 + i] >> KEY_LOCAL_BITS : 0xffffffffu;
    }
    c[0] = q0 > 0 ? keys[q0 - 1] >> KEY_LOCAL_BITS : 0xffffffffu;
    c[5] = q0 + 4 < np ? keys[q0 + 4] >> KEY_LOCAL_BITS : 0xffffffffu;
#pragma unroll
    for (int i = 1; i <= 4; ++i) {
        if ((int64_t)c[i] >= ncells) continue;  // past the end
        if (c[i] != c[i - 1]) start[c[i]] = (uint32_t)(q0 + i - 1);
        if (c[i] != c[i + 1]) end[c[i]] = (uint32_t)(q0 + i);
    }
}

// Work items per cell (ceil(len / item_len), none after an overflow), in one
// work group: thread t takes a contiguous run of cells, the run totals are
// scanned, and the offsets written.  item_off[ncells] and multi_off[ncells]
// hold the totals (also status words).  A cell's items share its chunks evenly,
// item q of ni taking chunks q, q + ni, ...: each sums a sample of the whole
// cell, not one side of it, so that a voxel's sum is spread over the items'
// FP32 accumulators (relative error against FP64 of heterogeneous 3e6 particles,
// FP32: 3.5e-7 with contiguous runs, 1.8e-7 so), and the items are equally long
// (1e6 particles, split BF16: 490 -> 453 us an insertion).
//
// The items are stored in their launch order, longest first (in buckets of one
// chunk): the gathers' work groups, dispatched in order, then take the long
// items early and the short ones fill the tail.  item_pos: the first of each
// cell.  Only the schedule depends on it: every cell sums its items in item
// order (their partial-tile slots), so the cube is bitwise the same in any launch
// order, and the order within a bucket may be left to the LDS atomics.
constexpr int SCAN_T = 1024;
constexpr int ITEM_BUCKETS = ITEM_MAX / KC;
constexpr int64_t ITEMS_IN_PLACE = 128;  // cells up to which k_items writes the items itself

struct CellItems {
    uint32_t items, bucket;
};

__device__ inline CellItems cell_items(uint32_t len, uint32_t L) {
    CellItems c;
    c.items = (len + L - 1) / L;
    // the longest item's chunks, at most ITEM_BUCKETS (L <= ITEM_MAX)
    const uint32_t chunks = (len + KC - 1) / KC;
    c.bucket = c.items ? ITEM_BUCKETS - (chunks + c.items - 1) / c.items : 0u;
    return c;
}

// Writes cell c's items with the lanes of one wave.
__device__ inline void write_items(uint32_t c, uint32_t n, uint32_t slot, uint32_t at,
                                   Item* __restrict__ items) {
    for (uint32_t q = threadIdx.x & 63; q < n; q += 64)
        items[at + q] = Item{(int32_t)c, (int32_t)q, (int32_t)n, n > 1u ? (int32_t)(slot + q) : -1};
}

__global__ __launch_bounds__(SCAN_T) void k_items(
    const uint32_t* __restrict__ start, const uint32_t* __restrict__ end, int64_t ncells,
    int item_len, uint32_t* __restrict__ status, uint32_t* __restrict__ item_off,
    uint32_t* __restrict__ multi_off, uint32_t* __restrict__ item_pos,
    uint32_t* __restrict__ split_cells, Item* __restrict__ items) {
    constexpr int WAVES = SCAN_T / 64;
    __shared__ uint32_t wtot[3][WAVES];
    __shared__ uint32_t bucket[ITEM_BUCKETS];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t per = (ncells + SCAN_T - 1) / SCAN_T;
    const int64_t c0 = min((int64_t)t * per, ncells), c1 = min(c0 + per, ncells);
    const bool none = status[ST_OVERFLOW] != 0u || status[ST_BADREC] != 0u;
    const uint32_t L = (uint32_t)item_len;
    if (t < ITEM_BUCKETS) bucket[t] = 0u;
    __syncthreads();
    auto of = [&](int64_t c) { return cell_items(none ? 0u : end[c] - start[c], L); };
    uint32_t sum[3] = {0u, 0u, 0u};  // items, partial tiles, split cells
    for (int64_t c = c0; c < c1; ++c) {
        const CellItems n = of(c);
        sum[0] += n.items;
        sum[1] += n.items > 1u ? n.items : 0u;
        sum[2] += n.items > 1u;
        if (n.items) atomicAdd(&bucket[n.bucket], n.items);
    }
    uint32_t at[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const uint32_t incl = (uint32_t)wave_scan_add((int)sum[k]);
        at[k] = incl - sum[k];
        if (lane == 63) wtot[k][wave] = incl;
    }
    __syncthreads();
    uint32_t total[3] = {0u, 0u, 0u};
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            if (w == wave) at[k] += total[k];
            total[k] += wtot[k][w];
        }
    if (wave == 0) {  // the buckets' first positions
        uint32_t run = 0u;
#pragma unroll
        for (int b = 0; b < ITEM_BUCKETS; b += 64) {
            const uint32_t v = bucket[b + lane], incl = (uint32_t)wave_scan_add((int)v);
            bucket[b + lane] = run + incl - v;
            run += __builtin_amdgcn_readlane(incl, 63);
        }
    }
    if (t == 0) {
        item_off[ncells] = total[0];
        multi_off[ncells] = total[1];
        status[ST_ITEMS] = total[0];
        status[ST_MULTI] = total[1];
        status[ST_SPLIT] = total[2];
    }
    __syncthreads();
    for (int64_t c = c0; c < c1; ++c) {
        const CellItems n = of(c);
        item_off[c] = at[0];
        multi_off[c] = at[1];
        item_pos[c] = n.items ? atomicAdd(&bucket[n.bucket], n.items) : 0u;
        at[0] += n.items;
        at[1] += n.items > 1u ? n.items : 0u;
        if (n.items > 1u) split_cells[at[2]++] = (uint32_t)c;
    }
    if (ncells > ITEMS_IN_PLACE) return;  // uniform
    __syncthreads();  // the positions above, read back from this work group's own writes
    for (int64_t c = wave; c < ncells; c += WAVES)
        write_items((uint32_t)c, item_off[c + 1] - item_off[c], multi_off[c], item_pos[c], items);
}

// One wave per cell writes the cell's items (cubes of more cells than k_items
// handles by itself).
__global__ __launch_bounds__(64) void k_build_items(const uint32_t* __restrict__ item_off,
                                                    const uint32_t* __restrict__ multi_off,
                                                    const uint32_t* __restrict__ item_pos,
                                                    Item* __restrict__ items) {
    const uint32_t c = blockIdx.x;
    write_items(c, item_off[c + 1] - item_off[c], multi_off[c], item_pos[c], items);
}

static inline unsigned blocks_for(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

hipError_t bin_particles(const mi_particle* d_p, int64_t n, int64_t n_pairs, const Grid& g,
                         const mi_cube_desc& d, char* ws, const Layout& L, hipStream_t s) {
    auto words = [&](size_t at) { return (uint32_t*)(ws + at); };
    uint32_t* status = words(L.status);
    uint32_t* hist = words(L.hist);
    auto* emit_look = (unsigned long long*)(ws + L.emit_look);
    auto* radix_look = (unsigned long long*)(ws + L.radix_look);
    const int T = 256;

    const int64_t clear = (int64_t)(L.cleared - L.status) / 16;
    hipLaunchKernelGGL(k_bin_init, dim3((unsigned)std::min<int64_t>((clear + T - 1) / T, 2048)),
                       dim3(T), 0, s, (uint4*)(ws + L.status), clear);
    const RadixPlan r = radix_plan(g);
    // the last pass ends in keys2 / vals2
    uint32_t *k0 = words(L.keys), *v0 = words(L.vals), *k1 = words(L.keys2), *v1 = words(L.vals2);
    if (r.passes % 2 == 0) {
        std::swap(k0, k1);
        std::swap(v0, v1);
    }
    const int64_t groups = emit_groups(n);
    const GroupShape shape = emit_shape(n);
    if (groups > 0) {
        auto emit = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)groups), dim3((unsigned)shape.threads),
                               sizeof(uint32_t) * EMIT_COPIES * ((r.passes << r.bits) + 1), s, d_p, n, n_pairs,
                               g, d.weights, d.weights_n, emit_look, k0, v0, hist, status, r.begin, r.passes,
                               r.bits);
        };
        if (same(shape, EMIT_SMALL))
            emit(k_emit<EMIT_SMALL.threads, EMIT_SMALL.items>);
        else if (same(shape, EMIT_MID))
            emit(k_emit<EMIT_MID.threads, EMIT_MID.items>);
        else
            emit(k_emit<EMIT_LARGE.threads, EMIT_LARGE.items>);
    }
    const int64_t tiles = radix_tiles(n_pairs);
    const GroupShape rs = radix_shape(n_pairs);
    for (int p = 0; p < r.passes && tiles > 0; ++p) {
        auto pass = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3((unsigned)rs.threads), 0, s, k0, v0, k1, v1,
                               hist + (p << r.bits), radix_look + ((p * tiles) << r.bits),
                               status + ST_TICKET + 1 + p, status, r.begin + p * r.bits, r.bits);
        };
        if (same(rs, RADIX_TILE_SMALL))
            pass(k_radix<RADIX_TILE_SMALL.threads, RADIX_TILE_SMALL.items>);
        else if (same(rs, RADIX_TILE_MID))
            pass(k_radix<RADIX_TILE_MID.threads, RADIX_TILE_MID.items>);
        else
            pass(k_radix<RADIX_TILE_LARGE.threads, RADIX_TILE_LARGE.items>);
        std::swap(k0, k1);
        std::swap(v0, v1);
    }
    if (n_pairs > 0)
        hipLaunchKernelGGL(k_cell_bounds, dim3(blocks_for((n_pairs + 3) / 4, T)), dim3(T), 0, s,
                           words(L.keys2), status, g.ncells, words(L.cell_start), words(L.cell_end));
    hipLaunchKernelGGL(k_items, dim3(1), dim3(SCAN_T), 0, s, words(L.cell_start), words(L.cell_end),
                       g.ncells, L.item_len, status, words(L.item_off), words(L.multi_off),
                       words(L.item_pos), words(L.split_cells), (Item*)(ws + L.items));
    if (g.ncells > ITEMS_IN_PLACE)
        hipLaunchKernelGGL(k_build_items, dim3((unsigned)g.ncells), dim3(64), 0, s,
                           words(L.item_off), words(L.multi_off), words(L.item_pos),
                           (Item*)(ws + L.items));
    return hipGetLastError();
}

}  // namespace mi
