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
// before the first load: 15x192 fp16 batch 8, 217 -> 210 us a forward, 20x256 batch 32, 644 -> 627; 6x128
// fp32 batch 1, 76 -> 75; nothing where the host's launches are the bound, 10x128 fp16 batch 5, 77 to 87
// and 83 to 85.)
constexpr int kCellsPerBoard = kPadCells;
constexpr int kRowCells = 20;
// Cells that a tile of mt consecutive rows can reach: its own span (a cell more per board
// row ended, 20 more per board ended) and 21 on either side.
constexpr int conv_cells(int mt) {
    return mt - 1 + (mt - 1 + 18) / 19 + kRowCells * ((mt - 1 + 360) / 361) + 2 * (kRowCells + 1) + 1;
}

// The patch of a tile: the cells that its points reach.
struct PatchStart {
    unsigned q0, x0;   // first cell: the upper left tap of the tile's first row; its place in a row of LDS
    unsigned mb, mp;   // board and point of the tile's first row
};
__device__ __forceinline__ PatchStart patch_start(unsigned m0) {
    PatchStart s;
    s.mb = m0 / kPts;
    s.mp = m0 - s.mb * kPts;
    s.q0 = (s.mb + 1) * kCellsPerBoard + s.mp + s.mp / kBoard - 1;
    s.x0 = (s.q0 + 1) % kRowCells;
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

// Where the cells of conv3x3_k's patch lie in LDS, and who reads them.  A fragment read (16 bytes a lane) is
// served 16 lanes at a time, 256 bytes a cycle: lanes 0-3, 12-15 and 20-27 first, that is eight points of
// one quarter of the k-step (lane / 16) and the eight other points of the next quarter.  Three
// things make these 16 meet all 16 slots of 16 bytes, with addresses that are constants from one
// read to the next:
//   - a cell takes an odd number of slots (STR bytes), and the pieces of quarters 2 i and 2 i + 1 stand 4
//     slots apart: conv_slot;
//   - lanes 4-11 have the even points of a block of 16, the others the odd ones: conv_point;
//   - a row of 20 cells, left border first, is as long, modulo 256 bytes, as one of 19: the end of a
//     board row, where the cells of 16 points skip one, does not show.  What lies between two rows
//     is read as the right border of the first: zeros, which clear_gaps writes.
// Counted in a loop of reads: 4 cycles each; 8 with the pieces and points in their natural order, 12
// where 16 points end a board row.  It shows where 192x64 tiles load the LDS most: 20x256 batch 32 640 ->
// 614 us a forward, two side by side 979 -> 924; 16 boards 830 -> 820 of 40 blocks, the others within 1 %.
// The fp32 kernels, and conv3x3_split_k from 192 filters on, have the order of points and quarters (quarter_slot)
// without the longer rows, which cost them addresses (10x128 fp16 batch 5 84 -> 93, 10x256 fp32 batch 64 1280 -> 1292).
template <int STR>
struct CellPitch {
    static_assert(STR % 32 == 16, "an odd number of slots");
    static constexpr int kAdd = (256 - STR % 256) % 256;   // bytes more per row
    static constexpr int kRow = kRowCells * STR + kAdd;
};
// Bytes of a patch, with one more cell that takes the pieces past the end.
template <int STR>
constexpr int patch_bytes(int cells) {
    return (cells + 1) * STR + (cells + kRowCells - 1) / kRowCells * CellPitch<STR>::kAdd;
}
template <int STR>
__device__ __forceinline__ unsigned patch_at(const PatchStart& s, unsigned cell) {
    return cell * STR + (__umul24(s.x0 + cell, 3277u) >> 16) * CellPitch<STR>::kAdd;   // (/ 20)
}
// Threads 0 .. NT - 1 clear what lies between the rows of COPIES patches.
template <int STR, int CELLS, int NT, int COPIES>
__device__ __forceinline__ void clear_gaps(unsigned char* patches, const PatchStart& s, unsigned tid) {
    constexpr int GAPS = (CELLS + kRowCells - 1) / kRowCells, PIECES = CellPitch<STR>::kAdd / 16;
#pragma unroll
    for (int p = 0; p < (COPIES * GAPS * PIECES + NT - 1) / NT; p++) {
        const unsigned i = tid + p * NT, gap = i / PIECES % GAPS, copy = i / (PIECES * GAPS);
        const unsigned end = (gap + 1) * kRowCells - s.x0;   // cells before it
        if (copy < COPIES && end <= (unsigned)CELLS)
            *reinterpret_cast<int4v*>(patches + copy * patch_bytes<STR>(CELLS) + end * STR +
                                      gap * CellPitch<STR>::kAdd + i % PIECES * 16) = int4v{0, 0, 0, 0};
    }
}
// Slot of quarter q of half h of a cell.
__device__ __forceinline__ unsigned conv_slot(unsigned q, unsigned h) {
    return 4 * (q & 1) + 2 * (q >> 1) + h;
}
// Slot of quarter q of 32 channels where a cell has no room between them.
__device__ __forceinline__ unsigned quarter_slot(unsigned q) { return 2 * (q & 1) + (q >> 1); }
// The point of a block of 16 that a lane owns.
__device__ __forceinline__ int conv_point(unsigned lane) {
    const unsigned t = (lane + 4) & 15;
    return (int)(2 * (t & 7) + 1 - (t >> 3));
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

// Tiles of 128 channels, 16 rb points high, of a layer of `rows` points and `cols` such columns: the
// lowest from `lowest` to 10 blocks that makes no more than one work-group per unit (0: none does), and the
// one that takes the least rounds times tile (12 is the tile of 192x128, which wins where several take the same).
// A tile costs as much as two blocks of points more than it has: by its blocks alone three rounds of 80x128 would
// beat two of 128x128, and five of 112x128 three of 192x128, and do not (4 blocks, us: 256 filters, 81 boards 252.7 on 80x128,
// 245.6 on 128x128, 137: 413.3, 395.4 on 144x128; 384, 53: 340.0, 332.3 on 128x128, fp32 953, 909; 122: 768 on 112x128, 735 on
// 192x128).  Over 80 batches of 128 to 384 filters, the tile so chosen is 0.3 % from the best one, by the blocks alone 0.6.
static inline int one_round_blocks(int rows, int cols, int lowest) {
    for (int rb = lowest; rb <= 10; rb++)
        if ((rows + rb * 16 - 1) / (rb * 16) * cols <= kUnits) return rb;
    return 0;
}
static inline int least_rounds_blocks(int rows, int cols) {
    int best = 12, least = 0;
    for (int rb = 12; rb >= 5; rb--) {
        const int rounds = ((rows + rb * 16 - 1) / (rb * 16) * cols + kUnits - 1) / kUnits, work = rounds * (rb + 2);
        if (rb != 11 && (least == 0 || work < least)) {
            best = rb;
            least = work;
        }
    }
    return best;
}

// What a transformed filter may be off by however small it is: a few sums of numbers that were rounded
// to zero below 2^-126.
constexpr float kFilterFloor = 0x1p-123f;

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
