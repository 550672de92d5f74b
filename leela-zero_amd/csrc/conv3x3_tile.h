// Geometry of the direct 3x3 convolutions (conv3x3.hip, conv3x3_f32.hip): points, patches and how the
// tiles of a layer lie on the dies.
#pragma once
#include "kernel_util.h"

namespace lzhip {

typedef int int2v __attribute__((ext_vector_type(2)));
typedef unsigned uint2v __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------------------
// Geometry.  Row m of the implicit GEMM is point (b, y, x) of the batch.  The planes stand with a zero
// border, in memory (kernels.h: padded planes) as in LDS: point (b, y, x) is cell 400 (b + 1) + 20 (y + 1) + x,
// with one zero column between board rows (right border of one row and left border of the next) and
// one zero row between boards.  A tap (r, s) is then the constant offset 20 (r - 1) + (s - 1), without
// bounds logic, and the patch of a tile is one run of consecutive cells: every piece that a
// thread fetches lies a constant distance from its first.  (With dense planes in memory and the border
// made on the way to LDS an address took some 25 instructions, and up to 13 of them per thread came
// before the first load: 10x128 fp16 batch 5, 86.8 -> 82.8 us a forward, 15x192 batch 8, 218 -> 209,
// 20x256 batch 32, 676 -> 664; fp32, with more pieces, 6x128 batch 1, 83 -> 75.)
constexpr int kCellsPerBoard = kPadCells;
constexpr int kRowCells = 20;
// Cells that a tile of mt consecutive rows can reach: its own span (a cell more per board
// row ended, 20 more per board ended) and 21 on either side.
constexpr int conv_cells(int mt) {
    return mt - 1 + (mt - 1 + 18) / 19 + kRowCells * ((mt - 1 + 360) / 361) + 2 * (kRowCells + 1) + 1;
}

// The patch of a tile: the cells that its points reach.
struct PatchStart {
    unsigned q0;       // first cell: the upper left tap of the tile's first row
    unsigned mb, mp;   // board and point of the tile's first row
};
__device__ __forceinline__ PatchStart patch_start(unsigned m0) {
    PatchStart s;
    s.mb = m0 / kPts;
    s.mp = m0 - s.mb * kPts;
    s.q0 = (s.mb + 1) * kCellsPerBoard + s.mp + s.mp / kBoard - 1;
    return s;
}
// Cell of the patch in which the upper left tap of the tile's row `local` lies; the point itself is
// kPointCell further on.
constexpr unsigned kPointCell = kRowCells + 1;
__device__ __forceinline__ unsigned patch_cell(const PatchStart& s, unsigned local) {
    unsigned p = s.mp + local;
    const unsigned next = p >= kPts ? 1u : 0u;
    p -= next * kPts;
    const unsigned y = __umul24(p, 3450u) >> 16;   // p / 19
    return (s.mb + 1 + next) * kCellsPerBoard + p + y - 1 - s.q0;
}

// LDS is what a work-group shares: its writes are waited for, loads from memory stay in flight
// across the barrier.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// How the tiles of a layer lie on the 8 dies: 2^split dies side by side over the channel tiles
// (`cols` of them each), 8 / 2^split over the row tiles: a column of dies deals its tiles, row by
// row, in equal shares of `share`, which may end within a row (in whole rows, 44 boards of 384
// filters gave some dies 33 tiles for their 32 units: 52 us per layer, now
// 36; 44 boards of 192 filters 21.2, now 14.2).  Every die
// has an L2 of its own and starts a layer with it empty, so it fetches its share of the filters
// (all of them / 2^split) and of the planes (all of them / (8 / 2^split)): of the ways that load
// the dies equally the one that fetches least is taken.
struct ConvGrid {
    int split, cols, share, tiles_m;
    unsigned inv;   // ceil(2^31 / cols)
};
struct ConvTile {
    int m, n;
};
// Work-group x runs on die x % 8.
__device__ __forceinline__ ConvTile conv_tile(const ConvGrid& g) {
    const int die = blockIdx.x & 7;
    const unsigned i = (die >> g.split) * g.share + (blockIdx.x >> 3);
    const int m = (int)__umulhi(i * 2u, g.inv);
    return {m, (die & ((1 << g.split) - 1)) * g.cols + (int)i - m * g.cols};
}

constexpr int kUnits = 256;   // compute units

// filters, planes: bytes of a layer's filters and of its input planes
static inline ConvGrid conv_grid(int tiles_m, int tiles_n, size_t filters, size_t planes) {
    ConvGrid best{};
    size_t best_cost = ~(size_t)0;
    for (int split = 0; split < 4 && tiles_n % (1 << split) == 0; split++) {
        const int over_rows = 8 >> split;
        const int cols = tiles_n >> split;
        const ConvGrid g{split, cols, (tiles_m * cols + over_rows - 1) / over_rows, tiles_m,
                         ((1u << 31) + cols - 1) / cols};
        const size_t bytes = (filters >> split) + planes / over_rows;
        // (32 units a die; rounds of tiles first)
        const size_t rounds = ((size_t)g.share + 31) / 32;
        const size_t cost = rounds << 40 | bytes;
        if (cost < best_cost) {
            best_cost = cost;
            best = g;
        }
    }
    return best;
}

}  // namespace lzhip
