// Geometry of the direct 3x3 convolutions (conv3x3.hip, conv3x3_f32.hip): points, patches and how the
// tiles of a layer lie on the dies.
#pragma once
#include "kernel_util.h"

namespace lzhip {

typedef int int2v __attribute__((ext_vector_type(2)));
typedef unsigned uint2v __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------------------
// Geometry.  Row m of the implicit GEMM is point (b, y, x) of the batch.  In LDS the planes
// stand with a zero border: cell q(m) = 400 b + 20 (y + 1) + x, one zero column between board
// rows (right border of one row and left border of the next) and one zero row between
// boards.  A tap (r, s) is then the constant offset 20 (r - 1) + (s - 1), without bounds logic.
constexpr int kCellsPerBoard = 400;
// Cells that a tile of mt consecutive rows can reach: its own span (a cell more per board
// row ended, 20 more per board ended) and 21 on either side.
constexpr int conv_cells(int mt) {
    return mt - 1 + (mt - 1 + 18) / 19 + 20 * ((mt - 1 + 360) / 361) + 43;
}
__device__ __forceinline__ unsigned conv_cell(unsigned m) {
    const unsigned b = m / kPts, p = m - b * kPts, y = p / kBoard, x = p - y * kBoard;
    return b * kCellsPerBoard + (y + 1) * 20 + x;
}

// The patch of a tile (the cells that its points reach) and what lies where in it.  Where it
// begins is worked out once, in scalar registers; from there on every cell is less than 400 away
// and every division is a 24-bit multiplication and a shift.  (With full divisions by 400, 20,
// 361 and 19 and a branch for every kind of border a work-group spent 1400 to 4200 cycles, up to
// a third of its life, before its first load; so 1000 to 1900.)
struct PatchStart {
    unsigned q0, b0, y0, x0;   // first cell, one board on (stays positive), and its parts
    unsigned mb, mp;           // board and point of the tile's first row
};
__device__ __forceinline__ PatchStart patch_start(unsigned m0) {
    PatchStart s;
    s.q0 = conv_cell(m0) + kCellsPerBoard - 21;
    s.b0 = s.q0 / kCellsPerBoard;
    s.y0 = (s.q0 - s.b0 * kCellsPerBoard) / 20;
    s.x0 = s.q0 - s.b0 * kCellsPerBoard - s.y0 * 20;
    s.mb = m0 / kPts;
    s.mp = m0 - s.mb * kPts;
    return s;
}
// Cell of the patch in which the upper left tap of the tile's row `local` lies.
__device__ __forceinline__ unsigned patch_cell(const PatchStart& s, unsigned local) {
    unsigned p = s.mp + local;
    const unsigned next = p >= kPts ? 1u : 0u;
    p -= next * kPts;
    const unsigned y = __umul24(p, 3450u) >> 16;   // p / 19
    return (s.mb + next) * kCellsPerBoard + 20 + p + y + kCellsPerBoard - 21 - s.q0;
}
// Byte offset in X (row_bytes a point) of a thread's 16-byte piece i (PPC to a cell); cells off the board and boards
// outside the batch get an offset outside the buffer and read as zero.
template <int CELLS, int PPC, int NT>
__device__ __forceinline__ unsigned patch_offset(int i, const PatchStart& s, unsigned tid,
                                                 unsigned row_bytes) {
    static_assert(CELLS <= 380 && (PPC != 24 || CELLS * PPC + NT < 8200), "small divisions");
    const unsigned piece = tid + i * NT;
    const unsigned cell = PPC == 24 ? __umul24(piece, 2731u) >> 16 : piece / PPC;
    const unsigned part = piece - cell * PPC;
    const unsigned t = s.x0 + cell, dy = __umul24(t, 3277u) >> 16;   // t / 20
    const unsigned x = t - dy * 20, y = s.y0 + dy;                   // y >= 20: the next board
    // t - dy = 19 dy + x, in points of the board's rows; row y1 = 0 of the board before is kept
    // positive by `lead`
    const unsigned lead = (kPts + kBoard) * row_bytes;
    const unsigned pt = s.b0 * kPts + s.y0 * kBoard + t - dy - (y >= 20 ? 19u : 0u);
    unsigned off = __umul24(pt, row_bytes) + part * 16u - lead;
    asm volatile("" : "+v"(off));   // keeps the compiler from branching around it
    const unsigned bad = (unsigned)(cell >= (unsigned)CELLS) | (unsigned)(x == 19) |
                         (unsigned)(y == 0) | (unsigned)(y == 20);
    return off | (0u - bad);
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
