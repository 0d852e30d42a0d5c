// The insertion contraction on the matrix cores:
//
//   cube[(i, j), c] += sum_p W[(i, j), p] * S[p, c]
//
// per cell (16 x 16 pixels x 64 channels, or 8 x 16 x 128 for cubes of 128
// channels or more) as a block-sparse product of a pixels x 32 W tile and a
// 32 x channels S tile per chunk of 32 particles, replacing the reference's
// per-pixel loop (martini/martini.py:243-283, :327-362).  Two forms of the
// products, the rest alike:
//
//   Float32    v_mfma_f32_16x16x4_f32: FP32 operands, products and sums.  A
//              16 x 16 x 4 step is skipped when none of its four particles
//              reaches the tile row or the channel block, so the cost follows the
//              footprints also where a chunk is not compact;
//   SplitBf16  both operands split into BF16 pairs x = hi + lo (|x - hi - lo| <=
//              2^-16 |x|) when they are written to LDS, and three
//              v_mfma_f32_16x16x32_bf16 products per 16 x 16 x 32 block -- hi*hi,
//              hi*lo, lo*hi -- accumulated in FP32 (the dropped lo*lo term is below
//              2^-16 of the product).
//
// Both are bound by the evaluation of W and S on the vector units (70% busy on 1e7
// particles, 512 x 512 x 256, split BF16: gather 3.89 ms; without the W fill 1.1 ms
// less, without the S fill 0.7, without the products 0.6); the FP32 products take
// about a quarter of the matrix units' time beside it (26% on 3e6 of heterogeneous
// size, 1024 x 1024 x 64: 2.77 ms).  On the vector units the
// FP32 products (64 multiply-adds per particle, thread and tile row, all
// channels) took most of that form's time: gather 643 us on 1e6 particles
// (WendlandC2, 256 x 256 x 128), 4.42 ms on 3e6 of heterogeneous size
// (1024 x 1024 x 64); on the matrix units 597 us and 3.59 ms at first, 367 us and
// 2.75 ms with what is described below.
//
// Wave w owns four tile rows (M = the 16 pixels of a row) and four 16-channel
// blocks (N): with 16 x 16-pixel x 64-channel cells the rows w, w + 4, .. and
// all four blocks; with 8 x 16 x 128 cells every other row and block, from row
// w % 2 and block w / 2 on, each pair of waves sharing its rows, which the second
// of the two to finish reading them clears (an LDS counter per row group
// decides).  A compact chunk reaches a few adjacent rows and blocks (4.2 and 3.3
// on average on the 1e6 particles below): dealt out one by one they are shared by
// the waves, where four adjacent ones were one wave's work that the others
// waited for (1e6 particles, FP32: insertion 627 -> 559 us; the split form,
// whose products are cheap, stays as it was).  The waves that stage the next
// chunks run ahead of the others on their SIMD (1e7 particles, split BF16: 5.07 ->
// 5.05 ms; 3e6 heterogeneous ones, FP32: 3.56 -> 3.54 ms).
// A (row, channel-block) product is skipped when no footprint of the chunk
// touches the row or no spectral window touches the block; the masks are
// wave-uniform, so the skips are scalar branches.
//
// Chunks are staged one per half of a wave, four at a time by two waves: the
// staging is on every chunk's critical path, and half its lanes were idle with one
// at a time (1e7 particles, 512 x 512 x 256, split BF16: gather 4.47 -> 4.32 ms;
// four at a time: see STAGED).
// Per chunk there are two barriers: (staging) -> W, S fill -> products, and one more
// (two with the square cells) in chunks with Gaussian-kernel particles, whose row
// and column factors are tabulated before the W fill.  Each wave clears the W rows it used right
// after reading them, so the next fill finds them zero; every fill rewrites
// the S blocks that the products will read.
// At the end of an item, accumulator blocks that are all zero are not
// written: a whole cell skips their read-modify-write of the cube, and a split
// cell's partial tile receives only the 1 KiB sub-tiles written, with a mask
// (16 bits per wave) that tells the reduction which to read.
// Accumulation order is fixed: deterministic, no atomics.
//
// FP32 sums: a chunk's 32 terms are a chain of multiply-adds of its own, the chunks'
// sums a chain of additions.  In one chain over all terms the many tails of far
// channels and pixels were lost against the bright voxels one by one, each sum 5e-8
// to 2e-7 low on sparse cubes (1.6e5 particles, 512 x 512 x 256, error against FP64:
// 1.4e-7 so, 5.2e-8 now; 1.5e6: 2.0e-7, 5.5e-8; heterogeneous 1e6, 512 x 512 x 64:
// 5.6e-8, 4.3e-8), for 1 to 5% of the form's time (1e7 particles, 512 x 512 x 256:
// insertion 6.66 -> 6.97 ms; 1e6, 256 x 256 x 128: 475 -> 480 us).  The tile rows are
// taken one by one for it: with a row's operands and one sum held instead of four
// rows' nothing spills.  The split form keeps one chain (the additions took 5% of
// 1e7 particles there).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mi_device.h"
#include "mi_internal.h"
#include "mi_tile.h"

namespace mi {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

// Operand tiles in LDS: OPK bytes per pixel (W) or channel (S) and chunk in
// either form.
constexpr int OPK = KC * 4;
constexpr unsigned AND_XOR = 0x6a;  // v_bitop3_b32: (a & b) ^ c

// BF16x3: a hi and a lo tile of 64 bytes per row, k contiguous, the four 16-byte
// k-groups of a row permuted by bits 2..3 of the row index: the 16 rows a
// 16-lane group reads for one k-group then fall in 16 distinct 16-byte bank slots.
template <int ROWS>
struct SplitTile {
    static constexpr int KROW = KC * 2;
    __attribute__((aligned(16))) char hi[ROWS * KROW];
    __attribute__((aligned(16))) char lo[ROWS * KROW];

    // Byte offset of element (row, k):
    //   row * KROW + (((k >> 3) ^ (row >> 2)) & 3) * 16 + (k & 7) * 2,
    // written with the k terms folded into one constant per thread (k_bits(k)).
    __device__ static int k_bits(int k) { return (((k >> 3) & 3) << 4) | ((k & 7) << 1); }
    __device__ static int at(int row, int kb) { return row * KROW + (((row << 2) & 48) ^ kb); }

    // at(row, kb) from q = SCALE * row: two instructions.
    static constexpr int SCALE = 4;
    __device__ static int at_scaled(int q, int kb) {
        return (q << 4) | (int)__builtin_amdgcn_bitop3_b32((unsigned)q, 48u, (unsigned)kb, AND_XOR);
    }

    // Writes x as a BF16 pair (round to nearest even) at row q / SCALE.
    __device__ void put(int q, int k, float x) {
        const __bf16 h = (__bf16)x;
        const __bf16 l = (__bf16)(x - (float)h);
        const int o = at_scaled(q, k_bits(k));
        *reinterpret_cast<__bf16*>(hi + o) = h;
        *reinterpret_cast<__bf16*>(lo + o) = l;
    }
    // Two values of column k, converted together (one packed conversion each for
    // the hi and the lo parts) at rows q1 / SCALE and q2 / SCALE.
    __device__ void put2(int k, int q1, float x1, int q2, float x2) {
        const floatx2 x = {x1, x2};
        const bf16x2 h = __builtin_convertvector(x, bf16x2);
        const floatx2 hf = __builtin_convertvector(h, floatx2);
        const bf16x2 l = __builtin_convertvector(floatx2{x1 - hf.x, x2 - hf.y}, bf16x2);
        const int kb = k_bits(k);
        const int o1 = at_scaled(q1, kb), o2 = at_scaled(q2, kb);
        *reinterpret_cast<__bf16*>(hi + o1) = h.x;
        *reinterpret_cast<__bf16*>(lo + o1) = l.x;
        *reinterpret_cast<__bf16*>(hi + o2) = h.y;
        *reinterpret_cast<__bf16*>(lo + o2) = l.y;
    }
    // put2 for the S fill, whose lanes l and l ^ 1 hold the rows r and r + 8 of a
    // block of 16 of particles k and k ^ 1 (a block is 1 KiB, an offset in the
    // store: eight addresses kept in registers made the FP32 form spill, 1e6 particles
    // 526 -> 504 us).  After one lane swap (DPP quad_perm [1, 0, 3, 2]) the even lane
    // writes row r and the odd lane row r + 8, each as the pair (k even, k odd) --
    // adjacent BF16 slots of one 4-byte word -- in both tiles: one paired 4-byte
    // store per lane (the hi and lo tiles lie a fixed distance apart) instead of
    // four 2-byte ones.  Every lane of the wave must call it.
    __device__ void put_pairs(int k, int block, int r, float x1, float x2) {
        constexpr int SWAP = 0xB1;  // quad_perm [1, 0, 3, 2]: lanes l and l ^ 1
        const float y1 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x1), SWAP, 0xF, 0xF, false));
        const float y2 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x2), SWAP, 0xF, 0xF, false));
        const bool even = (k & 1) == 0;
        const floatx2 x = even ? floatx2{x1, y1} : floatx2{y2, x2};  // particles k & ~1, k | 1
        const bf16x2 h = __builtin_convertvector(x, bf16x2);
        const floatx2 hf = __builtin_convertvector(h, floatx2);
        const bf16x2 l = __builtin_convertvector(floatx2{x.x - hf.x, x.y - hf.y}, bf16x2);
        char* to = hi + at(even ? r : r + 8, k_bits(k & ~1)) + block * (16 * KROW);
        *reinterpret_cast<bf16x2*>(to) = h;
        *reinterpret_cast<bf16x2*>(to + ROWS * KROW) = l;
    }
    // The 8 values of k-group kg of `row`, hi and lo.
    struct Op {
        bf16x8 h, l;
    };
    __device__ Op get(int row, int kg) const {
        const int o = row * KROW + (((kg ^ (row >> 2)) & 3) << 4);
        return Op{*reinterpret_cast<const bf16x8*>(hi + o), *reinterpret_cast<const bf16x8*>(lo + o)};
    }
    // Clears 16 rows from `row` on with one wave.
    __device__ void clear16(int row, int lane) {
        const int o = row * KROW + lane * 16;
        *reinterpret_cast<uint4*>(hi + o) = make_uint4(0u, 0u, 0u, 0u);
        *reinterpret_cast<uint4*>(lo + o) = make_uint4(0u, 0u, 0u, 0u);
    }
};

// FP32: 128 bytes per row.  A 16 x 16 x 4 product takes one value per lane and
// operand, lane group kg (of 16) the k-th of its four, so particle k is kept in
// slot 8 (k % 4) + k / 4: lane group kg then reads its eight values of the chunk
// with two 16-byte loads, and step s of the eight multiplies particles 4 s ..
// 4 s + 3.  The eight 16-byte groups of a row are permuted by bits 1..3 of the
// row index: the 16 rows that a 16-lane group reads together fall in distinct
// bank slots (even and odd rows lie in different halves of the banks).
template <int ROWS>
struct FloatTile {
    __attribute__((aligned(16))) char v[ROWS * OPK];

    __device__ static int k_bits(int k) { return ((k & 3) << 5) | ((k >> 2) << 2); }
    __device__ static int at(int row, int kb) { return row * OPK + (((row << 3) & 0x70) ^ kb); }
    static constexpr int SCALE = 8;
    __device__ static int at_scaled(int q, int kb) {
        return (q << 4) | (int)__builtin_amdgcn_bitop3_b32((unsigned)q, 0x70u, (unsigned)kb, AND_XOR);
    }
    __device__ void put(int q, int k, float x) {
        *reinterpret_cast<float*>(v + at_scaled(q, k_bits(k))) = x;
    }
    __device__ void put2(int k, int q1, float x1, int q2, float x2) {
        const int kb = k_bits(k);
        *reinterpret_cast<float*>(v + at_scaled(q1, kb)) = x1;
        *reinterpret_cast<float*>(v + at_scaled(q2, kb)) = x2;
    }
    __device__ void put_pairs(int k, int block, int r, float x1, float x2) {
        const int kb = k_bits(k);
        *reinterpret_cast<float*>(v + at(r, kb) + block * (16 * OPK)) = x1;
        *reinterpret_cast<float*>(v + at(r + 8, kb) + block * (16 * OPK)) = x2;
    }
    struct Op {
        floatx4 a, b;  // steps 0..3 and 4..7
        __device__ float step(int s) const { return s < 4 ? a[s] : b[s - 4]; }
    };
    __device__ Op get(int row, int kg) const {
        const int o = at(row, kg << 5);
        return Op{*reinterpret_cast<const floatx4*>(v + o),
                  *reinterpret_cast<const floatx4*>(v + (o ^ 16))};
    }
    __device__ void clear16(int row, int lane) {
        const int o = row * OPK + lane * 16;
        *reinterpret_cast<uint4*>(v + o) = make_uint4(0u, 0u, 0u, 0u);
        *reinterpret_cast<uint4*>(v + o + 1024) = make_uint4(0u, 0u, 0u, 0u);
    }
};

struct SplitBf16 {
    template <int ROWS>
    using Tile = SplitTile<ROWS>;
};
struct Float32 {
    template <int ROWS>
    using Tile = FloatTile<ROWS>;
};

// Chunks staged at a time, two by each of STAGED / 2 waves at once: the other waves
// wait for the staging, and with two chunks by one wave they did so twice as
// often (1e7 particles, 512 x 512 x 256, split BF16: 4.99 -> 4.83 ms; 3e6
// heterogeneous ones, FP32: 3.53 -> 3.47).  Eight by all four would leave LDS for
// two work groups on a CU only.
constexpr int STAGED = 4;
static_assert(STAGED % 2 == 0 && STAGED <= NT / 32 && (STAGED & (STAGED - 1)) == 0,
              "whole waves, and a power of two");

// What an item's chunks left out of the products because it is not finite
// (odd_line, values of the caller's table), each over its own footprint and
// channels: one particle after another, for the lane's voxels at rows i0 + RG r,
// columns j0 + q and channels ch0 + 16 CGN nb.  Rare, and kept short rather than fast.
template <int RG, int CGN, class Add>
__device__ inline void add_not_finite(const mi_particle* __restrict__ P,
                                      const uint32_t* __restrict__ order, ItemWalk chunks,
                                      const Grid& g, const mi_cube_desc& d,
                                      const float4* __restrict__ wtab, int i0, int j0, int ch0,
                                      Add add) {
    const bool table = d.spectrum == MI_SPECTRUM_TABLE;
#pragma unroll 1
    for (; chunks.more(); chunks.next())
#pragma unroll 1
        for (int k = 0; k < min(KC, chunks.left); ++k) {
            const mi_particle p = P[order[chunks.at() + k]];
            if (!table && !odd_line(p.s, p.fu, p.amp)) continue;
            const int kind = kind_of(p.r_kind), gi = gidx_of(p.r_kind);
            int i_lo, i_hi, j_lo, j_hi;
            if (!footprint(p, g.nx, g.ny, i_lo, i_hi, j_lo, j_hi)) continue;
#pragma unroll 1
            for (int e = 0; e < 64; ++e) {
                const int r = e >> 4, nb = (e >> 2) & 3, q = e & 3;
                const int i = i0 + RG * r, j = j0 + q, c = ch0 + 16 * CGN * nb;
                if (i < i_lo || i > i_hi || j < j_lo || j > j_hi || c < p.c_lo || c > p.c_hi || c >= g.nc)
                    continue;
                const float s = channel_flux(p, c, d);
                if (table && !not_finite(s)) continue;
                const float w = kind == MI_KERNEL_TABLE
                                    ? d.weights[table_offset(p) + (int64_t)(i - i_lo) * (j_hi - j_lo + 1) + j - j_lo]
                                    : pixel_weight(kind, (double)(p.ix - i) + (double)p.fx,
                                                   (double)(p.iy - j) + (double)p.fy, p.h, d.gauss_t[gi],
                                                   d.gauss_inv_norm[gi], wtab);
                add(r, nb, q, w * s);
            }
        }
}

// Bits 0, n, 2 n and 3 n.
constexpr uint32_t every(int n) { return 1u | 1u << n | 1u << 2 * n | 1u << 3 * n; }

// Three waves per SIMD: the 64 accumulators then live in VGPRs and three work
// groups share a CU (LDS 49 and 53 KB each).
template <class G, class F>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(3))) void k_gather(
    const mi_particle* __restrict__ P, const uint32_t* __restrict__ order,
    const Item* __restrict__ items, const uint32_t* __restrict__ cell_start,
    const uint32_t* __restrict__ cell_end, const uint32_t* __restrict__ status,
    const float4* __restrict__ wtab, Grid g, mi_cube_desc d, float* __restrict__ cube,
    float* __restrict__ partials, uint64_t* __restrict__ part_masks) {
    if (status[ST_OVERFLOW]) return;
    if (blockIdx.x >= status[ST_ITEMS]) return;
    const Item it = items[blockIdx.x];  // longest items first
    ItemWalk chunks(cell_start[it.cell], cell_end[it.cell], it, KC);
    const int begin = chunks.at(), step = chunks.step;
    const CellPos cp = cell_pos(it.cell, g);
    const int x0 = cp.x0, y0 = cp.y0, c0 = cp.c0;

    constexpr bool FP32 = std::is_same_v<F, Float32>;
    using WTile = typename F::template Tile<G::PX>;
    using STile = typename F::template Tile<G::CB>;
    __shared__ WTile W;            // [pixel][k]
    __shared__ STile S;            // [channel][k]
    __shared__ ChunkState staged[STAGED];  // chunks staged together
    __shared__ float4 Tk[LTAB_N];  // the item's kernel table
    // The chunk's Gaussian-kernel factors.  The square cells' lie in the S tile, for
    // which such a chunk waits once more: three work groups share the LDS then.
    constexpr bool GT_IN_S = G::PX > G::CB;
    __shared__ __attribute__((aligned(16))) char gt_own[GT_IN_S ? 16 : sizeof(GaussTables)];
    static_assert(sizeof(GaussTables) <= sizeof(STile), "the factors fit the S tile");
    GaussTables& gt = *reinterpret_cast<GaussTables*>(GT_IN_S ? reinterpret_cast<char*>(&S) : gt_own);
    // Waves: RG groups of four tile rows x CGN groups of four 16-channel blocks,
    // rows rh, rh + RG, ... and blocks ch, ch + CGN, ...
    constexpr int RG = G::TX / 4, CGN = G::CB / 64;
    constexpr uint32_t ROW_BITS = every(RG), BLK_BITS = every(CGN);  // of group 0
    static_assert(RG * CGN == NT / 64, "one (row group, channel group) per wave");
    static_assert(SUB_CH == 16, "a sub-tile is one 16 x 16 product block");
    __shared__ uint32_t done_rows[RG];  // waves done reading each row group this chunk

    const int t = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);  // wave-uniform
    const int lane = t & 63;
    const int m = lane & 15;   // A row / B column / D column of this lane
    const int kg = lane >> 4;  // K group (A, B); D row group of 4

    static_assert(sizeof(WTile) == G::PX * OPK && TILE_Y == 16, "16 pixels per tile row");
    for (int e = wave; e < G::TX; e += NT / 64) W.clear16(e * TILE_Y, lane);
    if (t < RG) done_rows[t] = 0u;
    const int rh = wave % RG, ch = wave / RG;  // this wave's row group and channel group

    floatx4 acc[4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) acc[r][nb] = floatx4{0.f, 0.f, 0.f, 0.f};

    // STAGED chunks are staged at a time, two by each of two waves, which hold the
    // records of their two of the next STAGED and the sort indices of those after.
    const int tkind = stage_table(P, order, begin, wtab, Tk);
    // Odd work groups stage with their last waves: every SIMD has its share.
    const int pair = (wave + (int)blockIdx.x * 2) & (NT / 64 - 1);
    const int at = (2 * pair + lane / KC) * step + (lane & (KC - 1));  // the lane's particle
    const bool stages = 2 * pair < STAGED;
    RecRegs next{};
    uint32_t next_idx = 0;
    if (stages && at < chunks.left) next = load_record(P, order[begin + at]);
    if (stages && at + STAGED * step < chunks.left) next_idx = order[begin + STAGED * step + at];

    // What is not finite is left out and added at the end.  The split form takes it like
    // any value: it reaches all columns of the tile rows and blocks that its chunk
    // reaches.  (Left out there too, more scalar registers spilled: 1e7 particles 4590 ->
    // 4675 us.)
    bool odd = false;        // a line was left out (the same for every thread)
    bool odd_value = false;  // this thread left out a value of the caller's table
    for (int slot = 0; chunks.more(); chunks.next(), slot = (slot + 1) & (STAGED - 1)) {
        const int left = chunks.left;
        if (slot == 0 && stages && 2 * pair * step < left) {
            __builtin_amdgcn_s_setprio(3);  // the other waves wait for it: first on its SIMD
            stage_chunks<FP32>(next, at < left, x0, y0, c0, g, d, staged + 2 * pair);
            __builtin_amdgcn_s_setprio(0);
            if (at + STAGED * step < left) next = load_record(P, next_idx);
            if (at + 2 * STAGED * step < left) next_idx = order[chunks.at() + 2 * STAGED * step + at];
        }
        const ChunkState& cs = staged[slot];
        __syncthreads();
        const uint32_t cover = __builtin_amdgcn_readfirstlane(cs.cover_per);
        const uint32_t chanmask = ChunkState::chanmask(cover);
        odd = odd || (FP32 && ChunkState::odd(cover));
        const uint32_t rows = (ChunkState::rowmask(cover) >> rh) & ROW_BITS;
        const uint32_t chans = (chanmask >> ch) & BLK_BITS;
        if (cs.gmask != 0u) {  // the same for every thread
            fill_gauss_tables(cs, x0, y0, gt);
            __syncthreads();
        }
        fill_weights<WTile::SCALE>(cs, x0, y0, wtab, tkind, Tk, gt, d,
                     [&](int k, int q, float w) { W.put(q, k, w); },
                     [&](int k, int q1, float w1, int q2, float w2) { W.put2(k, q1, w1, q2, w2); });
        if (GT_IN_S && cs.gmask != 0u) __syncthreads();
        odd_value |= fill_spectra<G::CB, FP32>(cs, c0, d,
                     [&](int k, int b, int r, float s1, float s2) { S.put_pairs(k, b, r, s1, s2); },
                     chanmask);
        // FP32: the particles (bits) that reach each of this wave's rows and blocks
        uint32_t prow[4] = {}, pblk[4] = {};
        if constexpr (FP32) {
            const uint32_t mine = lane < KC ? cs.walk[lane].cover : 0u;
#pragma unroll
            for (int r = 0; r < 4; ++r) prow[r] = (uint32_t)__ballot((mine >> (rh + RG * r)) & 1u);
#pragma unroll
            for (int nb = 0; nb < 4; ++nb)
                pblk[nb] = (uint32_t)__ballot((mine >> (16 + ch + CGN * nb)) & 1u);
        }
        __syncthreads();
        if (rows != 0u) {
            if constexpr (FP32) {
                // The chunk's sum by itself, then added: terms far below a voxel's value
                // (a chunk's tails) would be rounded away one by one against it, all in one
                // direction (see FP32 sums above).
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (!(rows & (1u << (RG * r))) || chans == 0u) continue;
                    const typename WTile::Op a = W.get((rh + RG * r) * TILE_Y + m, kg);
#pragma unroll
                    for (int nb = 0; nb < 4; ++nb) {
                        uint32_t q = prow[r] & pblk[nb];
                        if (q == 0u) continue;
                        const typename STile::Op b = S.get((ch + CGN * nb) * 16 + m, kg);
                        // bit 4 s: one of the particles 4 s .. 4 s + 3 reaches this row and block
                        q |= q >> 1;
                        const uint32_t need = q | (q >> 2);
                        floatx4 sum{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int s = 0; s < KC / 4; ++s)
                            if (need & (1u << (4 * s)))
                                sum = __builtin_amdgcn_mfma_f32_16x16x4f32(a.step(s), b.step(s), sum, 0, 0, 0);
                        acc[r][nb] += sum;
                    }
                }
            } else {
                // The wave's four tile rows held together: each S operand read serves all.
                typename WTile::Op a[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    a[r] = typename WTile::Op{};
                    if (!(rows & (1u << (RG * r))) || chans == 0u) continue;
                    a[r] = W.get((rh + RG * r) * TILE_Y + m, kg);
                }
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) {
                    if (!(chans & (1u << (CGN * nb)))) continue;
                    const typename STile::Op b = S.get((ch + CGN * nb) * 16 + m, kg);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if (!(rows & (1u << (RG * r)))) continue;
                        floatx4 c = acc[r][nb];
                        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r].h, b.h, c, 0, 0, 0);
                        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r].h, b.l, c, 0, 0, 0);
                        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r].l, b.h, c, 0, 0, 0);
                        acc[r][nb] = c;
                    }
                }
            }
            // The last of the CGN waves sharing these rows to get here clears
            // the rows' 2 KiB (two 16-byte stores per lane each): the counter's
            // update orders it after every such wave's reads of them (LDS requests
            // of a wave are served in order; the release keeps the reads before the
            // update).
            uint32_t before = 0u;
            if (CGN > 1 && lane == 0)
                before = __hip_atomic_fetch_add(&done_rows[rh], 1u, __ATOMIC_ACQ_REL,
                                                __HIP_MEMORY_SCOPE_WORKGROUP);
            if (CGN == 1 || __builtin_amdgcn_readlane(before, 0) == CGN - 1) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (rows & (1u << (RG * r))) W.clear16((rh + RG * r) * TILE_Y, lane);
                if (CGN > 1 && lane == 0) done_rows[rh] = 0u;
            }
        }
    }

    // D layout of a 16x16 block: lane holds rows 4*kg..4*kg+3 (pixels j) of column m
    // (channel).  Blocks that are all zero (no product reached them) are not
    // written; a partial tile's mask records the blocks that were.
    auto any = [](const floatx4& v) {
        return __ballot(v[0] != 0.f || v[1] != 0.f || v[2] != 0.f || v[3] != 0.f) != 0u;
    };
    if (FP32 && d.spectrum == MI_SPECTRUM_TABLE) {  // uniform
        __syncthreads();  // S is no longer read
        uint32_t* seen = reinterpret_cast<uint32_t*>(&S);
        const bool some = __any(odd_value);
        if (lane == 0) seen[wave] = some;
        __syncthreads();
        odd = (seen[0] | seen[1] | seen[2] | seen[3]) != 0u;
    }
    constexpr int BLOCKS = G::CB / SUB_CH;
    float* part = partials + (size_t)it.slot * CELL_VOXELS + sub_offset(BLOCKS, rh, ch);
    // Adds to this lane's voxel (row rh + RG r, column 4 kg + q; channel m of block
    // ch + CGN nb) in the cube or the partial tile.
    auto add = [&](int r, int nb, int q, float v) {
        if (it.slot >= 0)
            part[sub_offset(BLOCKS, RG * r, CGN * nb) + m * 16 + kg * 4 + q] += v;
        else
            cube[((size_t)(x0 + rh + RG * r) * g.ny + y0 + kg * 4 + q) * g.nc + c0 + (ch + CGN * nb) * 16 + m] += v;
    };
    auto add_odd = [&]() {
        ItemWalk again(cell_start[it.cell], cell_end[it.cell], it, KC);
        add_not_finite<RG, CGN>(P, order, again, g, d, wtab, x0 + rh, y0 + kg * 4, c0 + ch * 16 + m, add);
    };
    if (it.slot >= 0) {
        // a lane's four pixels are next to one another in a partial tile: one store each
        floatx4* tile = reinterpret_cast<floatx4*>(part) + m * 4 + kg;
        uint32_t mine = 0u;  // bit 4 r + nb: block (r, nb) written
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int nb = 0; nb < 4; ++nb)
                if ((FP32 && odd) || any(acc[r][nb])) {
                    mine |= 1u << (4 * r + nb);
                    tile[sub_offset(BLOCKS, RG * r, CGN * nb) / 4] = acc[r][nb];
                }
        static_assert(NT / 64 == 4, "four 16-bit parts per mask");
        if (lane == 0)  // this wave's part: bits 16 * wave + 4 r + nb
            reinterpret_cast<uint16_t*>(part_masks + it.slot)[wave] = (uint16_t)mine;
        if (FP32 && odd) add_odd();
        return;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = x0 + rh + RG * r;
        if (i >= g.nx) break;
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            if (!any(acc[r][nb])) continue;
            const int c = c0 + (ch + CGN * nb) * 16 + m;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j = y0 + kg * 4 + q;
                if (j < g.ny && c < g.nc) cube[((size_t)i * g.ny + j) * g.nc + c] += acc[r][nb][q];
            }
        }
    }
    if (FP32 && odd) add_odd();
}

hipError_t gather(const mi_particle* d_p, const Grid& g, const mi_cube_desc& d, char* ws,
                  const Layout& L, bool split_bf16, float* d_cube, hipStream_t s) {
    if (L.items_max <= 0) return hipSuccess;
    const float4* wtab = nullptr;
    hipError_t e = weight_table(s, &wtab);
    if (e != hipSuccess) return e;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)L.items_max), dim3(NT), 0, s, d_p,
                           (const uint32_t*)(ws + L.vals2), (const Item*)(ws + L.items),
                           (const uint32_t*)(ws + L.cell_start),
                           (const uint32_t*)(ws + L.cell_end), (const uint32_t*)(ws + L.status), wtab, g, d, d_cube,
                           (float*)(ws + L.partials), (uint64_t*)(ws + L.part_masks));
    };
    if (split_bf16) {
        if (g.wide)
            launch(k_gather<GeoWide, SplitBf16>);
        else
            launch(k_gather<GeoSquare, SplitBf16>);
    } else {
        if (g.wide)
            launch(k_gather<GeoWide, Float32>);
        else
            launch(k_gather<GeoSquare, Float32>);
    }
    return hipGetLastError();
}

}  // namespace mi
