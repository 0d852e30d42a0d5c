// Internal interfaces between the library's translation units: workspace
// layout and the host-side launchers of each stage.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/martini_mi355x.h"
#include "mi_device.h"

namespace mi {

struct Grid {
    int nx, ny, nc;      // padded cube extent
    bool wide;           // cell shape: GeoWide, else GeoSquare (wide_cells)
    int tx_shift, ty_shift, cb_shift;  // log2 of the tile sides and the block
    int ntx, nty, ncb;   // tiles along x, y; channel blocks
    int64_t ncells;
    int cell_bits;       // bits needed for a cell id
};

Grid make_grid(const mi_cube_desc& d);

// Number of cells particle p lands in (0 if its footprint or window is empty).
__host__ __device__ inline uint32_t cells_of(const mi_particle& p, const Grid& g, int& tx0, int& tx1,
                                    int& ty0, int& ty1, int& cb0, int& cb1) {
    int i_lo, i_hi, j_lo, j_hi;
    if (!footprint(p, g.nx, g.ny, i_lo, i_hi, j_lo, j_hi)) return 0;
    int c_lo = p.c_lo < 0 ? 0 : p.c_lo;
    int c_hi = p.c_hi > g.nc - 1 ? g.nc - 1 : p.c_hi;
    if (c_lo > c_hi) return 0;
    tx0 = i_lo >> g.tx_shift;  // footprints and windows are clipped: non-negative
    tx1 = i_hi >> g.tx_shift;
    ty0 = j_lo >> g.ty_shift;
    ty1 = j_hi >> g.ty_shift;
    cb0 = c_lo >> g.cb_shift;
    cb1 = c_hi >> g.cb_shift;
    return (uint32_t)((tx1 - tx0 + 1) * (ty1 - ty0 + 1) * (cb1 - cb0 + 1));
}

// A sum of pair counts in two 32-bit parts, of the counts' upper and lower 16 bits
// (64 counts of up to 2^27 each do not fit 32 bits together).
struct PairSum {
    uint32_t upper, lower;
    __host__ __device__ explicit PairSum(uint32_t count = 0u) : upper(count >> 16), lower(count & 0xffffu) {}
    __host__ __device__ unsigned long long total() const {
        return ((unsigned long long)upper << 16) + lower;
    }
};

// Byte offsets of the workspace regions (each 256-byte aligned).
struct Layout {
    // cleared at the start of every binning (status .. cleared)
    size_t status;                     // uint32[ST_WORDS]
    size_t hist;                       // uint32: digit counts of every radix pass
    size_t cell_start, cell_end;       // uint32[ncells] each
    size_t emit_look, radix_look;      // uint64: look-back words of the emit groups and radix tiles
    size_t cleared;                    // end of the region
    size_t keys, vals, keys2, vals2;   // uint32[n_pairs] each; vals2: particle index in cell order
    size_t item_off, multi_off;        // uint32[ncells + 1] each: exclusive scans of the
                                       // items and the partial-tile slots per cell
    size_t item_pos;                   // uint32[ncells]: launch position of a cell's first item
    size_t split_cells;                // uint32[split_max]: the cells of more than one item
    size_t items;                      // int4[items_max], in launch order
    size_t partials;                   // float[multi_max * CELL_VOXELS]
    size_t part_masks;                 // uint64[multi_max]: the sub-tiles each partial holds
    size_t total;
    int64_t items_max, multi_max, split_max;
    int item_len;                      // particles per work item
};

// At most so many cells hold more than item_len of n_pairs pairs; and their items,
// ceil(length / item_len) = 1 + (length - 1) / item_len each, are at most so many.
inline int64_t split_cells_max(int64_t n_pairs, int item_len, int64_t ncells) {
    const int64_t most = n_pairs / (item_len + 1);
    return ncells < most ? ncells : most;
}
inline int64_t partial_tiles_max(int64_t n_pairs, int item_len, int64_t ncells) {
    const int64_t cells = split_cells_max(n_pairs, item_len, ncells);
    return cells + (n_pairs - cells) / item_len;
}

// status[0]: number of pairs the device produced; status[1]: overflow flag.
// status[4]: a record with a footprint has an unknown kernel kind or table
// weights beyond the descriptor's table (no work items are then made).
// ST_SPLIT: number of cells with more than one item.
// ST_TICKET on: group tickets of the emit pass and of each radix pass.
enum { ST_PAIRS = 0, ST_OVERFLOW = 1, ST_ITEMS = 2, ST_MULTI = 3, ST_BADREC = 4, ST_SPLIT = 5, ST_TICKET = 8,
       ST_WORDS = 16 };

hipError_t layout_for(const Grid& g, int64_t n, int64_t n_pairs, Layout* L);

// Binning: emit, sort, cell bounds, items.  Asynchronous.
hipError_t bin_particles(const mi_particle* d_p, int64_t n, int64_t n_pairs, const Grid& g,
                         const mi_cube_desc& d, char* ws, const Layout& L, hipStream_t s);

// Gather over work items (products in FP32, or in split BF16), then the
// partial-tile reduction.
hipError_t gather(const mi_particle* d_p, const Grid& g, const mi_cube_desc& d, char* ws,
                  const Layout& L, bool split_bf16, float* d_cube, hipStream_t s);
hipError_t reduce_partials(const Grid& g, char* ws, const Layout& L, float* d_cube,
                           hipStream_t s);

// Devices the library keeps per-device state for (tables, scratch pointers).
constexpr int MAX_DEVICES = 64;

// The per-device weight tables (WTAB_KERNELS x WTAB_N), filled by fill_wtab on
// the device's first use: launched on stream s, which is then synchronised.
hipError_t weight_table(hipStream_t s, const float4** out);
hipError_t launch_weights(int kind, float gt, float ginv, const float* dx, const float* dy,
                          const float* h, float* out, int64_t n, hipStream_t s);
hipError_t launch_spectra(const mi_particle* d_p, int64_t n, const mi_cube_desc& d, float* out,
                          hipStream_t s);

// Device FP64 setup (mi_prepare.hip): workspace layout and launcher.
struct PrepLayout {
    size_t look, ticket, sums, total;
};
hipError_t prep_layout(int64_t n, PrepLayout* L);
hipError_t prepare_particles(const double* xyz, const double* vxyz, const double* mHI,
                             const double* hsm, const double* T, const double* edges, int64_t n,
                             const mi_observation& o, const Grid& g, mi_particle* out,
                             unsigned long long* counts, char* ws, const PrepLayout& L,
                             hipStream_t s);

// Beam convolution of a cube (mi_beam.hip).
size_t beam_lds_bytes(int kx, int ky);
// Rows y of a tile per work group.  Work groups aimed at, at most while a group can
// take more rows: four 33 KB tiles on each of the 256 CUs, so that a small cube still
// fills them and a large one leaves a group rows to overlap (301 x 257 x 131 FP32: 54
// us with 8 rows per group, 34 with the 4 of this rule; 512 x 512 x 256 FP64 253 us with
// 8 rows, 246 with 16).  Rounded down, narrow tiles made twice as many groups, each
// for a row (3 x 2000 x 5 FP32: 28 to 31 us, 25 with 8 rows per group, 22 so; 64 x 1025
// x 64 FP64: 41, 64, 21).
constexpr int64_t FITS_GROUPS = 1024;
constexpr int FITS_MAX_ROWS = 16;
inline int fits_rows(int64_t tiles, int ny) {
    const int64_t rows = (tiles * ny + FITS_GROUPS - 1) / FITS_GROUPS;
    return (int)(rows < FITS_MAX_ROWS ? rows : FITS_MAX_ROWS);
}
hipError_t cube_to_fits(const void* cube, bool cube_f64, int nx, int ny, int nc, int padx,
                        int pady, bool f64, void* out, double* range, hipStream_t s);
hipError_t convolve_beam(const float* in, float* out, int nx, int ny, int nc, const float* K,
                         int kx, int ky, hipStream_t s);

// A one-dimensional beam pass over L rows takes its input rows four a step, from
// m0 on (row m feeds output l through tap l + k/2 - m): the steps of the outputs from
// l0 on, `steps` without a border, of which those from `first` up to `last` meet a row of
// the cube.
struct LineSteps {
    int m0, first, last;
    __host__ __device__ LineSteps(int l0, int L, int k, int steps) : m0(l0 + k / 2 - (k - 1)) {
        first = m0 < 0 ? -m0 / 4 : 0;
        last = L > m0 ? (L - m0 + 3) / 4 : 0;
        if (last > steps) last = steps;
    }
};

// One work item: the q-th of a cell's n, which takes the cell's chunks q, q + n,
// ... of the sorted pair list; slot >= 0 names its partial tile, -1 means it
// writes the cube.
struct Item {
    int32_t cell, q, n, slot;
};

// A work item's chunks of `chunk` pairs: a walk over the sorted pair list from
// `begin`, the item's first chunk, to `end`, its cell's end, a step being the
// chunks of the cell's other items.  It counts the pairs left, not the
// position: a step is up to a 128th of the cell's pairs, and a position past the
// end of a cell that ends within a step of 2^31 would not be an int any more.
struct ItemWalk {
    int end, step, left;
    __host__ __device__ ItemWalk(uint32_t cell_start, uint32_t cell_end, const Item& it, int chunk)
        : end((int)cell_end), step(it.n * chunk), left((int)(cell_end - cell_start) - it.q * chunk) {}
    __host__ __device__ bool more() const { return left > 0; }
    __host__ __device__ int at() const { return end - left; }  // while more()
    __host__ __device__ void next() { left -= step; }
};

}  // namespace mi
