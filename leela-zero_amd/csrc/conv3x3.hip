// Direct 3x3 convolution for fp16 towers on the matrix cores (gfx950): one kernel per layer,
// convolution + batch norm + skip connection + ReLU, channels-last activations in and out.
//
// Why direct and not Winograd in fp16: F(4x4,3x3) needs 3.6 times fewer products, but as
// separate kernels it moves V and M (2 x 36/16 of a layer's planes) through memory in both
// directions, and at 256 filters that traffic, not the matrix pipe, is what a layer takes.
// As an implicit GEMM a layer reads its planes once and its filters once per die, and the
// fp16 matrix rate is high enough (v_mfma_f32_16x16x32_f16, fp32 accumulate) to do the
// whole sum.  Measured per layer, a forward of 40 blocks of 256 filters divided by its 81 layers,
// Winograd GEMM + fused transform -> this file: 64 boards 28.6 -> 22.4 us one forward at a time,
// 24.5 -> 19.8 with two side by side; 200 boards 83 -> 63 (1.36 PFLOP/s; torch.mm of 8192 x 8192 fp16
// matrices 1.19 to 1.33 on such cards); 16 boards 13.2 -> 9.8; 1 board, on conv3x3_split_k, 9.1 -> 4.2.
// What bounds it: with full tiles the matrix pipe, busy 56 % of a launch of 64 boards at the clock that
// the card's power allows (2.1 GHz); with one round of small tiles a chain of latencies, the first
// planes and filters, the tail, and the hand-over to the next layer.
// It also rounds less: planes and 3x3 filters are the only values kept in half precision.
#include <cmath>
#include <stdexcept>
#include <type_traits>

#include "conv3x3_tile.h"

namespace lzhip {

// Filters: [k-step][Kp / 16][64 lanes][8], k-step = (chunk of 64 input channels, tap, half of
// the chunk), i.e. the matrix instruction's row operand in the order it is used; every load of
// a wavefront is one contiguous KiB.  Lane l of block kb holds output channel
// conv_channel(kb, l % 16), input channels 32 (half) + 8 (l / 16) + 0..7 of the chunk.
// Register r of lane l of the result is row 4 (l / 16) + r of the row operand; with this order of
// the channels the registers of two neighbouring blocks are 8 consecutive channels, and a
// store instruction of a wavefront writes 64 contiguous bytes per point.
__host__ __device__ constexpr int conv_channel(int kb, int i) {
    return 32 * (kb >> 1) + 8 * (i >> 2) + 4 * (kb & 1) + (i & 3);
}
constexpr int kStepsPerChunk = 18;   // 9 taps x two k-steps of 32 channels
constexpr int kFilterLookahead = 18; // most k-steps requested ahead

__host__ __device__ static inline size_t conv3x3_index(int k, int c, int tap, int Kp) {
    const int kb = 2 * (k >> 5) + ((k >> 2) & 1), i = 4 * ((k >> 3) & 3) + (k & 3);
    const int step = ((c >> 6) * 9 + tap) * 2 + ((c >> 5) & 1);
    const int lane = ((c >> 3) & 3) * 16 + i;
    return (((size_t)step * (Kp / 16) + kb) * 64 + lane) * 8 + (c & 7);
}

size_t conv3x3_filter_count(int Cp, int Kp) {
    // the look-ahead reads past the last k-step (values that no instruction uses)
    return (size_t)(9 * Cp / 32 + kFilterLookahead) * Kp * 32;
}

// One work-group computes WR * RB * 16 points x WN * NB * 16 output channels; a wavefront owns
// RB x NB accumulator tiles of 16 x 16.
//
// Operands.  The filters are read once per work-group row of wavefronts straight from the
// die's L2 into registers (a ring of D k-steps, so that D - 1 steps of matrix instructions
// cover the latency).  Per k-step a wavefront has RB KiB of planes from LDS and NB KiB of filters from
// the L1 for RB * NB instructions of 16 cycles: 256 / NB of the LDS pipe's 256 bytes per cycle and 256 /
// RB of the 64 that the L1 delivers.  RB = 6, NB = 4 (25 % of one, 67 % of the other) is the
// tile for full batches.  The planes pass through LDS because every value is used nine times: the cells a
// tile reaches are staged once per chunk of input channels, in an order that the fragment reads
// take without bank conflicts (CellPitch), and the nine taps and two halves are immediate offsets of
// one address per 16 points.
//
// CC == 0: chunks of 64 input channels in two LDS buffers; the next chunk's pieces are loaded
// and stored in small groups between the matrix instructions (SGRP at a time: kept whole they
// would take the registers that let two work-groups share a compute unit), one barrier per
// chunk.  CC > 0 (64 CC channels, small tiles): everything is staged at once, one barrier in
// all, since a chunk's arithmetic would be over long before the next chunk has come.
//
// The sum over taps and channels runs in the same order in every variant, with the same
// instruction, so a position's result does not depend on the batch it is evaluated in.
template <int RB, int NB, int WR, int WN, int D, int DA, int CC, int OCC>
__global__ __launch_bounds__(64 * WR * WN, OCC) void conv3x3_k(
    const half_t* __restrict__ X, const half_t* __restrict__ Wf, const half_t* __restrict__ res,
    half_t* __restrict__ Y, const float* __restrict__ bn_scale, const float* __restrict__ bn_mean,
    float rfac, int n, int Cp, int Kp, ConvGrid g) {
    constexpr bool DB = CC == 0;
    constexpr int CH = DB ? 1 : CC;              // chunks of 64 channels staged together
    constexpr int NT = 64 * WR * WN;
    constexpr int MT = WR * RB * 16, CW = WN * NB * 16;
    constexpr int CELLS = conv_cells(MT);
    constexpr int STR = CH * 128 + 16;           // bytes per cell
    constexpr int ROW = CellPitch<STR>::kRow;
    constexpr int BUF = patch_bytes<STR>(CELLS);
    constexpr int PPC = 8;                       // 16-byte pieces per cell and chunk
    constexpr int NP = (CELLS * PPC + NT - 1) / NT;   // a thread's, per chunk
    constexpr int KS = kStepsPerChunk;
    constexpr int SGRP = 3;
    constexpr int NG = (NP + SGRP - 1) / SGRP;   // groups of pieces per chunk (CC == 0)
    constexpr int GS = KS / NG > 0 ? KS / NG : 1;
    constexpr int PR = NB >= 2 ? NB / 2 : 1;     // stores per point: two blocks give 16 bytes
    constexpr int E = NB >= 2 ? 8 : 4;           // channels per store
    // The skip connection is requested with the planes where its registers (4 RB PR) can wait
    // through the arithmetic (8 boards of 256 filters: the work-group's last phase 1500 -> 640
    // cycles).
    constexpr bool EARLY = RB * PR <= 6;
    static_assert(KS % D == 0 && KS % DA == 0, "rings turn a whole number of times per chunk");
    static_assert(D <= kFilterLookahead, "filter padding");
    static_assert(!DB || NG <= KS, "one group of pieces per k-step at most");
    static_assert(NB == 1 || NB % 2 == 0, "blocks are stored in pairs");
    __shared__ __attribute__((aligned(16))) unsigned char lds[DB ? 2 * BUF : BUF];
    __shared__ __attribute__((aligned(16))) float bn[2][CW];

    const ConvTile tile = conv_tile(g);
    const int tn = tile.n, tm = tile.m;
    if (tm >= g.tiles_m) return;
    const int rows = n * kPts, m0 = tm * MT;
    const unsigned tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const int wr = wave / WN, wn = wave % WN;

    // First of all what depends on nothing that has to be worked out: batch norm (waited for with
    // the planes; its loads come first, since loads are waited for in order) and filters.
    static_assert(CW <= NT, "one thread per channel");
    const unsigned bnoff = tid < (unsigned)CW ? (tn * CW + tid) * 4u : 0xfffffff0u;
    const float scale = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                      make_rsrc(bn_scale, Kp * 4), bnoff, 0, 0));
    const float mean = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                     make_rsrc(bn_mean, Kp * 4), bnoff, 0, 0));
    const int kb = (tn * WN + wn) * NB;          // first block of 16 output channels
    unsigned ws = (unsigned)kb * 1024u;
    const unsigned wstep = (unsigned)Kp * 64u;   // bytes per k-step
    const unsigned wv = lane * 16u;
    const __amdgpu_buffer_rsrc_t rW = make_rsrc(Wf, ((size_t)9 * Cp + 32 * kFilterLookahead) * Kp * 2);
    int4v w[D][NB];
    auto wload = [&](int slot, int j, unsigned st) {
        w[slot][j] = __builtin_amdgcn_raw_buffer_load_b128(rW, wv + j * 1024, ws + st * wstep, 0);
    };
#pragma unroll
    for (int d = 0; d < D - 1; d++)
#pragma unroll
        for (int j = 0; j < NB; j++) wload(d, j, d);
    __builtin_amdgcn_sched_barrier(0);

    const PatchStart ps = patch_start(m0);
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(X, (size_t)(n + 2) * kCellsPerBoard * Cp * 2);
    const unsigned xrow = (unsigned)Cp * 2u;     // bytes of a cell in memory
    const unsigned xoff = (ps.q0 + tid / PPC) * xrow + (tid % PPC) * 16u;
    // piece i, `at` bytes into the cells' channels
    auto xload = [&](int i, unsigned at) {
        return __builtin_amdgcn_raw_buffer_load_b128(rX, xoff, i * (NT / PPC) * xrow + at, 0);
    };
    unsigned laddr[NP];                          // LDS address of piece i
#pragma unroll
    for (int i = 0; i < NP; i++)
        laddr[i] = patch_at<STR>(ps, min(tid / PPC + i * (NT / PPC), (unsigned)CELLS)) +
                   conv_slot(tid & 3, tid >> 2 & 1) * 16u;

    const int chunks = Cp / 64;
    const int ch0 = (kb >> 1) * 32 + 8 * (int)(lane >> 4) + 4 * (kb & 1);   // first channel
    unsigned arow[RB];   // LDS address of this lane's point of each row block, tap (0, 0)
    unsigned ro[RB];     // byte offset of this lane's point and channel
    int4v rr[RB][PR];
    static_assert(MT <= kPts, "a tile touches two boards at most");
#pragma unroll
    for (int i = 0; i < RB; i++) {
        const int local = (wr * RB + i) * 16 + conv_point(lane);
        const unsigned cell = patch_cell(ps, min(local, rows - 1 - m0));
        arow[i] = patch_at<STR>(ps, cell) + conv_slot(lane >> 4, 0) * 16;
        ro[i] = m0 + local < rows ? ((ps.q0 + kPointCell + cell) * Kp + ch0) * 2u : 0xfffff000u;
    }
    const size_t ybytes = (size_t)(n + 2) * kCellsPerBoard * Kp * 2;
    const __amdgpu_buffer_rsrc_t rY = make_rsrc(Y, ybytes);
    const __amdgpu_buffer_rsrc_t rR = make_rsrc(res != nullptr ? res : Y, ybytes);
    auto load_res = [&](int from, int to) {
        if (res != nullptr) {
#pragma unroll
            for (int i = from; i < to; i++)
#pragma unroll
                for (int j = 0; j < PR; j++) {
                    if constexpr (NB >= 2) {
                        rr[i][j] = __builtin_amdgcn_raw_buffer_load_b128(rR, ro[i] + j * 64, 0, 0);
                    } else {
                        const int2v t = __builtin_bit_cast(
                            int2v, __builtin_amdgcn_raw_buffer_load_b64(rR, ro[i], 0, 0));
                        rr[i][j] = int4v{t.x, t.y, 0, 0};
                    }
                }
        } else {
#pragma unroll
            for (int i = from; i < to; i++)
#pragma unroll
                for (int j = 0; j < PR; j++) rr[i][j] = int4v{0, 0, 0, 0};
        }
    };

    clear_gaps<STR, CELLS, NT, DB ? 2 : 1>(lds, ps, tid);
    {
        int4v stg[CH][NP];
#pragma unroll
        for (int c = 0; c < CH; c++)
#pragma unroll
            for (int i = 0; i < NP; i++) stg[c][i] = xload(i, c * 128);
        if constexpr (EARLY) load_res(0, RB);
#pragma unroll
        for (int c = 0; c < CH; c++)
#pragma unroll
            for (int i = 0; i < NP; i++)
                *reinterpret_cast<int4v*>(lds + laddr[i] + c * 128) = stg[c][i];
        if (tid < (unsigned)CW) {
            bn[0][tid] = scale;
            bn[1][tid] = -scale * mean;
        }
    }
    float4v acc[RB][NB];
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    lds_barrier();

    int4v a[DA][RB];
    auto aread = [&](int i, int st) {
        const int sub = st / KS, tap = (st % KS) / 2, half = st & 1;
        return *reinterpret_cast<const int4v*>(lds + arow[i] + tap / 3 * ROW + tap % 3 * STR +
                                               sub * 128 + half * 16);
    };
    if constexpr (!DB) {
#pragma unroll
        for (int d = 0; d < DA; d++)
#pragma unroll
            for (int i = 0; i < RB; i++) a[d][i] = aread(i, d);
    }
    unsigned other = BUF;   // byte offset of the buffer being filled (CC == 0)
    // Chunk c; the last one stages nothing and fetches no filters past its end, and the skip connection
    // comes into the registers that this leaves.
    auto chunk = [&](int c, auto is_last) {
        constexpr bool LAST = decltype(is_last)::value;
        if constexpr (DB) {
#pragma unroll
            for (int d = 0; d < DA; d++)
#pragma unroll
                for (int i = 0; i < RB; i++) a[d][i] = aread(i, d);
        }
        const unsigned next = (unsigned)(c + 1) * 128u;
        int4v sg[SGRP];
#pragma unroll
        for (int st = 0; st < KS; st++) {
            if constexpr (LAST && !EARLY) {
                if (st == KS - 2) load_res(0, RB / 3);
                if (st == KS - 1) load_res(RB / 3, RB);
            }
            if constexpr (DB && !LAST) {
#pragma unroll
                for (int g = 0; g < NG; g++) {
                    if (st == g * GS) {
#pragma unroll
                        for (int i = 0; i < SGRP; i++)
                            if (g * SGRP + i < NP)
                                sg[i] = xload(g * SGRP + i, next);
                    }
                    if (st == (g + 1) * GS - 1) {
#pragma unroll
                        for (int i = 0; i < SGRP; i++)
                            if (g * SGRP + i < NP)
                                *reinterpret_cast<int4v*>(lds + laddr[g * SGRP + i] + other) = sg[i];
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            // The filters of step st + D - 1 go into the slot that step st - 1 has left, and each
            // row block's next fragment is read behind the instructions that used the last one;
            // the barriers keep this order.
#pragma unroll
            for (int i = 0; i < RB; i++) {
#pragma unroll
                for (int j = 0; j < NB; j++)
                    if (i == (RB >= NB ? j : 0) && (!LAST || st + D - 1 < KS))
                        wload((st + D - 1) % D, j, st + D - 1);
#pragma unroll
                for (int j = 0; j < NB; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        __builtin_bit_cast(half8v, w[st % D][j]),
                        __builtin_bit_cast(half8v, a[st % DA][i]), acc[i][j], 0, 0, 0);
                if (st + DA < KS || (!DB && !LAST)) a[st % DA][i] = aread(i, st + DA);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (LAST) return;
        ws += KS * wstep;
        if constexpr (DB) {
            lds_barrier();
            const unsigned flip = (c & 1) ? (unsigned)-BUF : (unsigned)BUF;
#pragma unroll
            for (int i = 0; i < RB; i++) arow[i] += flip;
            other -= flip;
        } else {
#pragma unroll
            for (int i = 0; i < RB; i++) arow[i] += 128;
        }
    };
#pragma unroll 1
    for (int c = 0; c < chunks - 1; c++) chunk(c, std::false_type{});
    chunk(chunks - 1, std::true_type{});

    // max(0, scale * (y - mean) + rfac * res), clamped to the stored range
#pragma unroll
    for (int j = 0; j < PR; j++) {
        const int cl = ch0 - tn * CW + j * 32;
        float sc[E], nb[E];
#pragma unroll
        for (int e = 0; e < E; e++) {
            sc[e] = bn[0][cl + e];
            nb[e] = bn[1][cl + e];
        }
#pragma unroll
        for (int i = 0; i < RB; i++) {
            const half8v rh = __builtin_bit_cast(half8v, rr[i][j]);
            half8v o;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if (e >= E) { o[e] = (half_t)0.0f; continue; }
                const float v = acc[i][NB >= 2 ? 2 * j + e / 4 : 0][e % 4];
                o[e] = (half_t)fminf(
                    fmaxf(0.0f, fmaf((float)rh[e], rfac, fmaf(v, sc[e % E], nb[e % E]))),
                    kActStoreMax);
            }
            const int4v bits = __builtin_bit_cast(int4v, o);
            if constexpr (NB >= 2)
                __builtin_amdgcn_raw_buffer_store_b128(bits, rY, ro[i] + j * 64, 0, kStoreThrough);
            else
                __builtin_amdgcn_raw_buffer_store_b64(uint2v{(unsigned)bits.x, (unsigned)bits.y},
                                                      rY, ro[i], 0, kStoreThrough);
        }
    }
}

template <int RB, int NB, int WR, int WN, int D, int DA, int CC, int OCC>
static void launch_conv_as(const half_t* X, const half_t* Wf, const half_t* res, half_t* Y,
                           const float* bn_scale, const float* bn_mean, float rfac, int n, int Cp,
                           int Kp, hipStream_t s, LaunchTimer* t) {
    constexpr int MT = WR * RB * 16, CW = WN * NB * 16;
    const int tiles_m = (n * kPts + MT - 1) / MT, tiles_n = Kp / CW;
    const ConvGrid best = conv_grid(tiles_m, tiles_n, (size_t)18 * Cp * Kp, (size_t)n * kPts * Cp * 2);
    launch(conv3x3_k<RB, NB, WR, WN, D, DA, CC, OCC>, dim3(8 * best.share),
           dim3(64 * WR * WN), s, t, X, Wf, res, Y, bn_scale, bn_mean, rfac, n, Cp, Kp, best);
}

// Which handles compute by direct convolution.  Its arithmetic grows with the square of the
// width, what the Winograd kernels move with the width itself: up to 384 filters the matrix pipe
// is through with the one before the memory is with the other; above, only where a layer is a
// chain of latencies, that is where tiles of 96x64 make no more than one work-group per unit.
// Measured per forward of 5 blocks, Winograd kernels -> this, us (one forward at a time | two | three
// side by side):
//   320 filters,  1 board 133 -> 52, 16: 250 -> 126 | 290 -> 202 | 366 -> 289, 64: 495 -> 406 | 856 -> 669
//   384 filters,  8 boards 200 -> 126 | 237 -> 177 | 289 -> 257, 44: 459 -> 333 | 730 -> 604 | 1087 -> 905,
//                 100: 842 -> 821 | 1716 -> 1365, 200: 1703 -> 1505 | 3379 -> 2833
//   448 filters,  8 boards 215 -> 141, 12: 277 -> 225 | 327 -> 362 | 457 -> 565, 64: 716 -> 806 | 1341 -> 1427
//   512 filters,  8 boards 238 -> 165, 10: 254 -> 240 | 324 -> 373 | 428 -> 545, 64: 784 -> 820 | 1486 -> 1519
//   640 filters,  6 boards 289 -> 189 | 435 -> 322 | 595 -> 515, 8: 301 -> 293 | 441 -> 471 | 613 -> 743
//   768 filters,  5 boards 278 -> 217 | 433 -> 373 | 591 -> 597, 16: 514 -> 534 | 857 -> 936
//  1024 filters,  4 boards 396 -> 294 | 598 -> 516 | 822 -> 810, 64: 2229 -> 2972
// Left out: 512 filters at 16 to 40 boards gain too (32: 572 -> 446 | 874 -> 780) and lose again
// beyond.  (The batches beyond each line were measured when the line was drawn.)  Taken in: what gains
// one and two at a time and loses three side by side, 448 filters at 9 boards (214 -> 146 | 258 -> 242 |
// 336 -> 388).
// The batch is the handle's largest, so that a network keeps its filters in one order and a
// position's result does not depend on what it is evaluated with.
bool conv3x3_serves(int Kp, int max_batch, int elem_bytes) {
    if (elem_bytes != 2 || Kp % 64 != 0) return false;
    return Kp <= 384 || (max_batch * kPts + 95) / 96 * (Kp / 64) <= kUnits;
}

// The tile.  A layer of few boards is a chain of latencies, so its points and channels are
// spread over the 256 compute units in the smallest tiles that still make no more than one
// work-group per unit; larger ones reuse each operand more.  Measured at 256 filters, us per
// layer of a dependent chain with tiles of points x channels, * where a tile makes more than 256
// work-groups, that is two or more on some unit:
//               48x64   96x64  128x64  192x64 128x128 192x128
//    8 boards    8.2     8.9     9.6    12.3    17.2    19.2
//   16 boards   11.7*    9.9    10.5    13.1    17.3    19.4
//   20 boards   13.7*   14.4*   11.0    13.5    17.6    20.0
//   24 boards   14.3*   14.9*   16.2*   14.1    17.8    20.1
//   32 boards   17.3*   15.5*   16.6*   14.4    18.2    20.1
//   40 boards   22.8*   21.5*   17.7*   21.5*   19.1    21.2
//   64 boards   32.0*   29.2*   26.4*   25.1*   28.5*   24.1
//   80 boards   40.1*   35.6*   32.2*   33.1*   30.2*   37.6*
//  128 boards   61.0*   54.2*   47.6*   45.6*   44.9*   42.9*
// (128x128 with its wavefronts two by two, a kernel that is gone; side by side, as they are now, 40 boards take
// 16.7.)  Two chains side by side want larger tiles (us per layer and chain): 20 boards 128x64 8.5, 192x64 8.9, 96x64
// 9.6; 40 boards 192x64 13.3, 128x64 14.3, 192x128 14.8; 64 boards 192x128 19.1, 192x64 20.2; 80 boards 192x128
// 23.7.  At other widths the order is the same: 128 filters, 44
// boards 48x64 7.9, 128x64 6.7 (two chains 5.9 | 4.9);
// 384 filters, 13 boards 192x64 16.8, 128x64 13.7 (13.4 | 12.0).  64 and 192 filters have no tile of 128
// channels; there 128x64 is taken up to two work-groups
// per unit (192 filters, 52 boards 128x192 15.9, 128x64 13.6, two chains 12.7 | 12.0; 64 filters, 150 boards
// 192x64 8.7, 128x64 7.1), and beyond, 128x192 takes the place of 192x128 (192 filters, 70 boards 192x64
// 17.9, 128x192 16.5).  64 filters, whose one chunk is over soon, keep 48x64 up to three work-groups
// (96 boards 5.8 against 6.4 with 192x64).
void launch_conv3x3(const half_t* X, const half_t* Wf, const half_t* res, half_t* Y,
                    const float* bn_scale, const float* bn_mean, float rfac, int n, int Cp, int Kp,
                    int lanes, hipStream_t s, LaunchTimer* t) {
    if (Kp % 64 != 0 || Cp % 64 != 0)
        throw std::invalid_argument("no direct convolution for this width");
    const int rows = n * kPts;
    auto groups = [&](int mt, int cw) { return ((rows + mt - 1) / mt) * (Kp / cw); };
#define LZ_CONV(RB, NB, WR, WN, D, DA, CC, OCC)                                                   \
    launch_conv_as<RB, NB, WR, WN, D, DA, CC, OCC>(X, Wf, res, Y, bn_scale, bn_mean, rfac, n, Cp, \
                                                   Kp, s, t)
    // whole patches in LDS: the input layer and towers of up to 256 filters
    const int cc = Cp / 64;
    if (cc <= 4 && groups(32, 32) <= kUnits) {
        switch (cc) {
            case 1: LZ_CONV(2, 1, 1, 2, 18, 6, 1, 1); return;
            case 2: LZ_CONV(2, 1, 1, 2, 18, 6, 2, 1); return;
            case 3: LZ_CONV(2, 1, 1, 2, 18, 6, 3, 1); return;
            default: LZ_CONV(2, 1, 1, 2, 18, 6, 4, 1); return;
        }
    }
    if (cc <= 4 && groups(32, 64) <= kUnits) {
        switch (cc) {
            case 1: LZ_CONV(2, 1, 1, 4, 18, 3, 1, 1); return;
            case 2: LZ_CONV(2, 1, 1, 4, 18, 3, 2, 1); return;
            case 3: LZ_CONV(2, 1, 1, 4, 18, 3, 3, 1); return;
            default: LZ_CONV(2, 1, 1, 4, 18, 3, 4, 1); return;
        }
    }
    // One small tile to a unit: four wavefronts of 16 channels, so that every SIMD has one (with two of
    // 32 the tile waited for its 54 steps of 96 cycles; the planes are now read from LDS twice as
    // often, which the pipe has room for).  Against 48x64 on two wavefronts and 96x64 on four, a
    // layer of 256 filters, 7 boards 7.8 -> 6.7 us, 9 boards 8.8 -> 7.4; 192 filters, 8 boards 6.4 ->
    // 5.8, 13 boards 7.4 -> 6.4; two forwards side by side 0 to 7 % faster, three 1 to 8 % slower.  Not
    // beyond: 96x64 on eight wavefronts, or with 16 channels to a wavefront, is 10 to 14 % slower than as below (16 boards of
    // 256 filters), and 80x64 no faster.
    if (groups(48, 64) <= kUnits) {
        if (lanes <= 2) LZ_CONV(3, 1, 1, 4, 9, 3, 0, 2);
        else LZ_CONV(3, 2, 1, 2, 6, 3, 0, 2);
        return;
    }
    if (groups(64, 64) <= kUnits && lanes <= 2) {
        LZ_CONV(4, 1, 1, 4, 9, 3, 0, 2);
        return;
    }
    if (groups(96, 64) <= kUnits) {
        LZ_CONV(3, 2, 2, 2, 6, 3, 0, 2);
        return;
    }
    if (groups(128, 64) <= kUnits) {
        LZ_CONV(4, 2, 2, 2, 6, 1, 0, 2);
        return;
    }
    if (Kp == 64 && groups(48, 64) <= 3 * kUnits) {
        LZ_CONV(3, 2, 1, 2, 6, 3, 0, 2);
        return;
    }
    // Larger tiles, the lowest that makes one round.  Of 128 channels where the width has them: the four
    // wavefronts stand side by side, every filter is fetched once and not by two rows of them, and
    // heights go in steps of 16 points.  Layers of 256 filters, 192x64 and 128x128 (wavefronts two by two) -> this, us:
    // 24 boards 13.4 -> 12.2 (80x128), 32: 13.6 -> 13.3 (96x128), 40: 18.1 -> 16.7 (128x128), 50: 20.1 -> 18.6
    // (144x128), 56: 21.5 -> 20.9; of 384, 16 boards 17.0 -> 15.3, 26: 23.6 -> 21.3; of 128, 50 boards 8.6 -> 7.7.
    // Two or three forwards side by side gain as much from 112x128 on (256 filters, 50 boards, two: 16.4 -> 15.3) and
    // nothing below (32 boards, two: 10.3 -> 10.6), so there 192x64 stays.
#define LZ_WIDE(RB)                         \
    case RB:                                \
        LZ_CONV(RB, 2, 1, 4, 6, 1, 0, 2);   \
        return
    auto wide = [&](int rb) {
        switch (rb) {
            LZ_WIDE(5);
            LZ_WIDE(6);
            LZ_WIDE(7);
            LZ_WIDE(8);
            LZ_WIDE(9);
            LZ_WIDE(10);
            default: LZ_CONV(6, 4, 2, 2, 3, 1, 0, 2); return;
        }
    };
#undef LZ_WIDE
    const bool wide_columns = Kp % 128 == 0;
    if (wide_columns && lanes == 1) {
        if (const int rb = one_round_blocks(rows, Kp / 128, 5)) return wide(rb);
    }
    // 192 filters, 33 boards 192x64 11.2, 160x64 10.1 us (two side by side 7.6 | 7.1).  Three side by side have nothing
    // from it and lose some (8 blocks of 320 filters, 20 boards 517 -> 527 us a forward of each, of 192, 33 boards 343 -> 346).
    if (!wide_columns && Kp != 64 && lanes <= 2 && groups(160, 64) <= kUnits) {
        LZ_CONV(5, 2, 2, 2, 6, 1, 0, 2);
        return;
    }
    if (groups(192, 64) <= kUnits) {
        LZ_CONV(6, 2, 2, 2, 6, 1, 0, 2);
        return;
    }
    if (wide_columns) {
        if (const int rb = one_round_blocks(rows, Kp / 128, 7)) return wide(rb);
    }
    if ((Kp == 64 || Kp == 192) && groups(128, 64) <= 2 * kUnits) {
        LZ_CONV(4, 2, 2, 2, 6, 1, 0, 2);
        return;
    }
    // More than a round of every tile.  What a forward with the device to itself takes is rounds times
    // tile, whether the last round is full or nearly empty: a layer of 256 filters, 70 boards 36 us on 192x128
    // and 26 on 112x128, 100 boards 38 and 34 (144x128); 10 blocks of 192 filters, 91 to 120 boards
    // 637 - 659 us on 128x192, 527 - 566 on 128x64, 135 boards
    // 678 and 590 on 192x64.  Side by side with another forward, which fills the gaps, the tile
    // that reads least is the best one.
    if (wide_columns) return wide(lanes == 1 ? least_rounds_blocks(rows, Kp / 128) : 12);
    auto rounds = [&](int mt, int cw) { return (groups(mt, cw) + kUnits - 1) / kUnits * mt * cw; };
    if (lanes == 1 && rounds(128, 64) < rounds(192, 64) &&
        (Kp != 192 || rounds(128, 64) < rounds(128, 192))) {
        LZ_CONV(4, 2, 2, 2, 6, 1, 0, 2);
        return;
    }
    if (Kp == 192 && (lanes > 1 || rounds(128, 192) <= rounds(192, 64)))
        LZ_CONV(4, 6, 2, 2, 3, 1, 0, 2);
    else
        LZ_CONV(6, 2, 2, 2, 6, 1, 0, 2);
#undef LZ_CONV
}

// ---------------------------------------------------------------------------
// The same layer with the sum over input channels dealt to the wavefronts of a work-group.
//
// With few boards a unit has one small tile, and what a layer takes is one chain of latencies.  In
// conv3x3_k the wavefronts of such a tile each own so narrow a part of it that every operand is
// fetched twice or four times, and all wait for the whole patch.  Here every wavefront owns the
// whole tile and KW-th of the k-steps (HPW halves of a chunk of 64 channels, all nine taps): each
// operand is fetched once, a wavefront stages its own input channels and waits for nobody, its
// filters are in flight all at once (D = 9 HPW; less where that would take the registers of another
// wavefront on the SIMD), and the partial sums meet in LDS at the end, in the order of the wavefronts.
// Measured per forward of 10 blocks, conv3x3_k -> this with tiles of 32 channels, us: 128 filters, 1 board 99 -> 82, 8 boards
// 110 -> 92; 192 filters, 1 board 120 -> 98, 5 boards 134 -> 114; 256 filters, 1 board 132 -> 104, 5
// boards 150 -> 138; of 5 blocks, 1 board: 320 filters 105 -> 60, 384 116 -> 63, 448 131 -> 70, 512
// 136 -> 76.
// 96x32 points x channels for larger batches is slower than conv3x3_k (192 filters, 11 boards 244 -> 259 us a
// forward of 20 blocks, two side by side 162 -> 210), 96x64 and 192x64 gave nothing either way.
// The order of the sum differs from conv3x3_k's, so a network uses one or the other whatever the
// batch (conv3x3_splits).
//
// From 192 filters on a wavefront has the filters of 12 of its 18 steps ahead: with all of them a unit holds one
// work-group of 192 or 256 filters, and a forward alone waits longer for its first ones too (8 blocks, us, one at a time |
// two side by side, 18 -> 12: 192 filters, 1 board 58.8 -> 57.3, 7: 91.9 -> 87.3 | 138 -> 112; 256, 1: 66.0 -> 63.2, 5:
// 101.4 -> 96.7; three side by side, 192 filters, 7 boards 203 -> 140).
// Left out: a wavefront for each half of a chunk at 192 and 256 filters, the halves summed apart, which gives other bits
// and is slower (192 filters, 7 boards 87.9 | 115.1; 256, 1: 64.9 | 81.5, 5: 102.5 | 125.0; at 320 and 384 too, 1 board
// 75.8 -> 79.0 and 93.3 -> 98.7); and tiles of 80x32 for the handles of 12 to 14 boards of 128 filters, 8 and 9 of 192, 6
// and 7 of 256, which are conv3x3_k's and would get other bits (0 to 7 % faster).
template <int RB, int NB, int KW, int HPW, int D>
__global__ __launch_bounds__(64 * KW, 1) void conv3x3_split_k(
    const half_t* __restrict__ X, const half_t* __restrict__ Wf, const half_t* __restrict__ res,
    half_t* __restrict__ Y, const float* __restrict__ bn_scale, const float* __restrict__ bn_mean,
    float rfac, int n, int Kp, ConvGrid g) {
    constexpr int DA = 3;                                  // planes read ahead
    constexpr int E = 4 * NB;                              // channels that a lane finishes
    typedef std::conditional_t<NB == 2, int4v, int2v> Piece;
    typedef half_t HalfE __attribute__((ext_vector_type(E)));
    constexpr int CH = KW * HPW / 2, Cp = 64 * CH, NT = 64 * KW;
    constexpr int MT = RB * 16, CW = NB * 16, CELLS = conv_cells(MT);
    constexpr int STR = HPW * 64 + 16, SLICE = (CELLS + 1) * STR;   // bytes per cell, wavefront
    constexpr int PPC = HPW * 4, NP = (CELLS * PPC + 63) / 64;   // 16-byte pieces: a cell's, a lane's
    constexpr int STEPS = 9 * HPW;
    constexpr int QP = (RB + KW - 1) / KW;   // blocks of 16 points that a wavefront finishes
    constexpr int BYTES = KW * (SLICE > RB * NB * 1024 ? SLICE : RB * NB * 1024);
    static_assert(D <= STEPS && CW <= NT, "tile");
    static_assert(HPW == 2 || (HPW == 1 && KW % 2 == 0), "whole chunks");
    __shared__ __attribute__((aligned(16))) unsigned char lds[BYTES];
    __shared__ __attribute__((aligned(16))) float bn[2][CW];

    const ConvTile tile = conv_tile(g);
    const int tn = tile.n, tm = tile.m;
    if (tm >= g.tiles_m) return;
    const int rows = n * kPts, m0 = tm * MT;
    const unsigned tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(tid >> 6));

    // channels in the order of the lanes that finish them
    auto channel = [&](int c) { return NB == 2 ? tn * CW + c : conv_channel(tn, c); };
    const unsigned bnoff = tid < (unsigned)CW ? channel(tid) * 4u : 0xfffffff0u;
    const float scale = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                      make_rsrc(bn_scale, Kp * 4), bnoff, 0, 0));
    const float mean = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                     make_rsrc(bn_mean, Kp * 4), bnoff, 0, 0));
    // this wavefront's k-steps, nine taps of one half after the other: their places in Wf
    const unsigned first = HPW == 2 ? wave * kStepsPerChunk
                                    : (wave >> 1) * kStepsPerChunk + (wave & 1);
    const unsigned wstep = (unsigned)Kp * 64u;
    const unsigned ws = first * wstep + (unsigned)(tn * NB) * 1024u;
    const __amdgpu_buffer_rsrc_t rW = make_rsrc(Wf, ((size_t)9 * Cp + 32 * kFilterLookahead) * Kp * 2);
    int4v w[D][NB];
    auto wload = [&](int slot, int j, unsigned st) {
        w[slot][j] = __builtin_amdgcn_raw_buffer_load_b128(rW, lane * 16u + j * 1024,
                                                           ws + (st % 9 * 2 + st / 9) * wstep, 0);
    };
    // A wavefront reads only its own input channels, so it stages them itself and waits for
    // nobody.  A few filters, the planes, the other filters: what the L1 delivers is what a tile
    // waits for at first, so the planes do not stand behind filters that are needed after them,
    // and each piece is requested as soon as its address is known.
    constexpr int F0 = D - 1 < 4 ? D - 1 : 4;
    auto filters = [&](int from, int to) {
#pragma unroll
        for (int d = 0; d < D - 1; d++)
#pragma unroll
            for (int j = 0; j < NB; j++)
                if (d >= from && d < to) wload(d, j, d);
        __builtin_amdgcn_sched_barrier(0);
    };
    filters(0, F0);
    const PatchStart ps = patch_start(m0);
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(X, (size_t)(n + 2) * kCellsPerBoard * Cp * 2);
    constexpr unsigned xrow = Cp * 2;   // bytes of a cell in memory
    const unsigned xoff = (ps.q0 + lane / PPC) * xrow + (lane % PPC) * 16u;
    int4v stg[NP];
#pragma unroll
    for (int i = 0; i < NP; i++)
        stg[i] = __builtin_amdgcn_raw_buffer_load_b128(
            rX, xoff, i * (64 / PPC) * xrow + wave * (HPW * 64), 0);
    __builtin_amdgcn_sched_barrier(0);
    filters(F0, D - 1);

    // the blocks of 16 points that this wavefront finishes: where they lie, and the skip connection
    unsigned ro[QP];
    Piece rr[QP];
    const size_t ybytes = (size_t)(n + 2) * kCellsPerBoard * Kp * 2;
    const __amdgpu_buffer_rsrc_t rY = make_rsrc(Y, ybytes);
    const __amdgpu_buffer_rsrc_t rR = make_rsrc(res != nullptr ? res : Y, ybytes);
    // The order of points and quarters in LDS (CellPitch) where more than four wavefronts' worth of channels is read (8
    // blocks, us: 320 filters, 1 board 78.5 -> 73.9, 384, 3: 119.5 -> 116.2; two side by side: 192 filters, 7 boards 115.4 ->
    // 111.5; 256, 1: 81.9 -> 80.1, 5: 124.2 -> 120.5). 64 filters, 1 board, lost by it (20 blocks 110.4 -> 111.5), 128 gained
    // nothing for one.
    constexpr bool SPREAD = KW * HPW > 4;
    const int point = SPREAD ? conv_point(lane) : (int)(lane & 15);   // this lane's, of a block of 16
    auto slot = [](unsigned q) { return SPREAD ? quarter_slot(q) : q; };
    const int cl = E * (int)(lane >> 4);   // first of this lane's channels
#pragma unroll
    for (int q = 0; q < QP; q++) {
        const int i = q * KW + wave, local = i * 16 + point;
        ro[q] = i < RB && m0 + local < rows
                    ? ((ps.q0 + kPointCell + patch_cell(ps, local)) * Kp + channel(cl)) * 2u
                    : 0xfffffff0u;
        rr[q] = Piece{};
    }
    if (res != nullptr) {
#pragma unroll
        for (int q = 0; q < QP; q++)
            if constexpr (NB == 2) rr[q] = __builtin_amdgcn_raw_buffer_load_b128(rR, ro[q], 0, 0);
            else rr[q] = __builtin_amdgcn_raw_buffer_load_b64(rR, ro[q], 0, 0);
    }
    unsigned char* const own = lds + wave * SLICE;
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const unsigned piece = lane + i * 64, cell = piece / PPC;
        *reinterpret_cast<int4v*>(own + (cell < (unsigned)CELLS ? cell : (unsigned)CELLS) * STR +
                                  (piece % PPC / 4 * 4 + slot(piece % 4)) * 16u) = stg[i];
    }
    if (tid < (unsigned)CW) {
        bn[0][tid] = scale;
        bn[1][tid] = -scale * mean;
    }
    unsigned arow[RB];
#pragma unroll
    for (int i = 0; i < RB; i++)
        arow[i] = patch_cell(ps, min(i * 16 + point, rows - 1 - m0)) * STR + slot(lane >> 4) * 16;
    float4v acc[RB][NB];
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

    int4v a[DA][RB];
    auto aread = [&](int i, int st) {
        const int half = st / 9, tap = st % 9;
        return *reinterpret_cast<const int4v*>(own + arow[i] + ((tap / 3) * 20 + tap % 3) * STR +
                                               half * 64);
    };
#pragma unroll
    for (int d = 0; d < DA; d++)
#pragma unroll
        for (int i = 0; i < RB; i++) a[d][i] = aread(i, d);
#pragma unroll
    for (int st = 0; st < STEPS; st++) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < RB; i++) {
#pragma unroll
            for (int j = 0; j < NB; j++)
                if (i == (RB >= NB ? j : 0) && st + D - 1 < STEPS)
                    wload((st + D - 1) % D, j, st + D - 1);
#pragma unroll
            for (int j = 0; j < NB; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    __builtin_bit_cast(half8v, w[st % D][j]),
                    __builtin_bit_cast(half8v, a[st % DA][i]), acc[i][j], 0, 0, 0);
            if (st + DA < STEPS) a[st % DA][i] = aread(i, st + DA);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // partial sums through LDS: [wavefront][row block][channel block][64 lanes][4]
    lds_barrier();
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++)
            *reinterpret_cast<float4v*>(lds + ((wave * RB + i) * NB + j) * 1024 + lane * 16) =
                acc[i][j];
    lds_barrier();
#pragma unroll
    for (int q = 0; q < QP; q++) {
        const int i = q * KW + wave;
        if (i >= RB) continue;
        float4v part[KW][NB];
#pragma unroll
        for (int k = 0; k < KW; k++)
#pragma unroll
            for (int j = 0; j < NB; j++)
                part[k][j] = *reinterpret_cast<const float4v*>(
                    lds + ((k * RB + i) * NB + j) * 1024 + lane * 16);
        const HalfE rh = __builtin_bit_cast(HalfE, rr[q]);
        HalfE o;
#pragma unroll
        for (int e = 0; e < E; e++) {
            float v = part[0][e / 4][e % 4];
#pragma unroll
            for (int k = 1; k < KW; k++) v += part[k][e / 4][e % 4];
            o[e] = (half_t)fminf(
                fmaxf(0.0f, fmaf((float)rh[e], rfac, fmaf(v, bn[0][cl + e], bn[1][cl + e]))),
                kActStoreMax);
        }
        if constexpr (NB == 2)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(int4v, o), rY, ro[q], 0,
                                                   kStoreThrough);
        else
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(int2v, o), rY, ro[q], 0,
                                                  kStoreThrough);
    }
}

// The tile, in blocks of 16 points by 16 channels: the smallest whose work-groups are no more
// than the compute units; {0, 0}: none is.  One block of channels halves the filters that the L1
// has to deliver to a work-group, which is what a layer of one board waits for: against 32 x 32
// tiles 128 filters 3.8 -> 3.3 us, 192 4.4 -> 3.8, 256 4.9 -> 4.3, 320 5.3 -> 4.7.  48 x 16 is worth
// 2 to 4 % up to 256 filters (192 filters, 2 boards 4.4 -> 4.3 us) and no longer beyond (384
// filters, 1 board 5.5 -> 5.7).
struct SplitTile {
    int rb, nb;
};
static SplitTile split_tile(int n, int Kp) {
    constexpr SplitTile kTiles[] = {{2, 1}, {3, 1}, {2, 2}, {3, 2}, {4, 2}};
    for (const SplitTile& t : kTiles)
        if ((t.rb * t.nb != 3 || Kp <= 256) &&
            (n * kPts + t.rb * 16 - 1) / (t.rb * 16) * (Kp / (16 * t.nb)) <= kUnits) return t;
    return {0, 0};
}

// A wavefront takes 64 input channels (32 of up to 128): eight wavefronts' planes are what the LDS
// holds, so 512 filters are the widest.
bool conv3x3_splits(int Kp, int max_batch) {
    return Kp % 64 == 0 && Kp <= 512 && split_tile(max_batch, Kp).rb > 0;
}

void launch_conv3x3_split(const half_t* X, const half_t* Wf, const half_t* res, half_t* Y,
                          const float* bn_scale, const float* bn_mean, float rfac, int n, int Cp,
                          int Kp, hipStream_t s, LaunchTimer* t) {
    const SplitTile tile = split_tile(n, Kp);
    if (!conv3x3_splits(Kp, n) || Cp != Kp)
        throw std::invalid_argument("no split convolution for this width or batch");
    const ConvGrid g = conv_grid((n * kPts + tile.rb * 16 - 1) / (tile.rb * 16), Kp / (16 * tile.nb),
                                 (size_t)18 * Cp * Kp, (size_t)n * kPts * Cp * 2);
    auto go = [&](auto kernel, int waves) {
        launch(kernel, dim3(8 * g.share), dim3(64 * waves), s, t, X, Wf, res, Y, bn_scale,
               bn_mean, rfac, n, Kp, g);
    };
    // KW wavefronts x HPW halves of a chunk
#define LZ_SPLIT(KW, HPW, D)                                               \
    if (tile.nb == 1) {                                                    \
        if (tile.rb == 2) go(conv3x3_split_k<2, 1, KW, HPW, D>, KW);       \
        else if constexpr (KW < 5) go(conv3x3_split_k<3, 1, KW, HPW, D>, KW); \
    } else if (tile.rb == 2) go(conv3x3_split_k<2, 2, KW, HPW, D>, KW);    \
    else if (tile.rb == 3) go(conv3x3_split_k<3, 2, KW, HPW, D>, KW);      \
    else if constexpr (KW < 8) go(conv3x3_split_k<4, 2, KW, HPW, D>, KW)
    switch (Kp) {
        case 64: LZ_SPLIT(2, 1, 9); break;
        case 128: LZ_SPLIT(4, 1, 9); break;
        // (from here on two thirds of the filters ahead)
        case 192: LZ_SPLIT(3, 2, 12); break;
        case 256: LZ_SPLIT(4, 2, 12); break;
        case 320: LZ_SPLIT(5, 2, 12); break;
        case 384: LZ_SPLIT(6, 2, 12); break;
        case 448: LZ_SPLIT(7, 2, 12); break;
        default: LZ_SPLIT(8, 2, 12); break;   // (the largest is for 3 boards, which no longer fit)
    }
#undef LZ_SPLIT
}

// ---------------------------------------------------------------------------
// 3x3 filters from their Winograd form U = G f G^T ([36][C][F], what a pipe is handed): the
// rows 0 and 5 of G are the unit vectors of f's outer taps and half the difference of rows 2
// and 1 is sqrt(2)/3 times the middle one, so f = L U L^T with the L below.  Every filter is
// checked by transforming it forward again: *bad is set if some u is further from G f G^T
// than rounding explains (such a U is no transform of a 3x3 filter, and only the Winograd
// kernels can compute with it).
__device__ constexpr float kG[6][3] = {{1.0f, 0.0f, 0.0f},
                                       {-2.0f / 3.0f, -0.47140452f, -1.0f / 3.0f},
                                       {-2.0f / 3.0f, 0.47140452f, -1.0f / 3.0f},
                                       {1.0f / 6.0f, 0.23570226f, 1.0f / 3.0f},
                                       {1.0f / 6.0f, -0.23570226f, 1.0f / 3.0f},
                                       {0.0f, 0.0f, 1.0f}};

__global__ __launch_bounds__(256) void filters_3x3_k(const float* __restrict__ U,
                                                     half_t* __restrict__ Wf, int C, int F, int Kp,
                                                     int* __restrict__ bad) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= C * F) return;
    const int c = i / F, k = i - c * F;
    float u[6][6], peak = 0.0f;
#pragma unroll
    for (int p = 0; p < 36; p++) {
        u[p / 6][p % 6] = U[((size_t)p * C + c) * F + k];
        peak = fmaxf(peak, fabsf(u[p / 6][p % 6]));
    }
    constexpr float kMid = 1.0606602f;   // 3 / (2 sqrt 2)
    float t[3][6], f[3][3];
#pragma unroll
    for (int x = 0; x < 6; x++) {
        t[0][x] = u[0][x];
        t[1][x] = (u[2][x] - u[1][x]) * kMid;
        t[2][x] = u[5][x];
    }
#pragma unroll
    for (int y = 0; y < 3; y++) {
        f[y][0] = t[y][0];
        f[y][1] = (t[y][2] - t[y][1]) * kMid;
        f[y][2] = t[y][5];
    }
    bool ok = true;
#pragma unroll
    for (int y = 0; y < 6; y++) {
        float g[3];
#pragma unroll
        for (int x = 0; x < 3; x++) g[x] = kG[y][0] * f[0][x] + kG[y][1] * f[1][x] + kG[y][2] * f[2][x];
#pragma unroll
        for (int x = 0; x < 6; x++) {
            const float v = g[0] * kG[x][0] + g[1] * kG[x][1] + g[2] * kG[x][2];
            ok = ok && fabsf(v - u[y][x]) <= 1e-4f * peak + kFilterFloor;
        }
    }
    if (!ok) *bad = 1;
#pragma unroll
    for (int tap = 0; tap < 9; tap++)
        Wf[conv3x3_index(k, c, tap, Kp)] =
            (half_t)fminf(fmaxf(f[tap / 3][tap % 3], -65504.0f), 65504.0f);
}

void conv3x3_filters(const float* U, half_t* Wf, int C, int F, int Kp, int* bad, hipStream_t s) {
    hipLaunchKernelGGL(filters_3x3_k, dim3((unsigned)((C * F + 255) / 256)), dim3(256), 0, s, U, Wf,
                       C, F, Kp, bad);
}

void conv3x3_winograd_filters(const half_t* Wf, int C, int Cp, int F, int Kp, half_t* U) {
    const double s2 = std::sqrt(2.0);
    const double G[6][3] = {{1, 0, 0},
                            {-2.0 / 3, -s2 / 3, -1.0 / 3},
                            {-2.0 / 3, s2 / 3, -1.0 / 3},
                            {1.0 / 6, s2 / 6, 1.0 / 3},
                            {1.0 / 6, -s2 / 6, 1.0 / 3},
                            {0, 0, 1}};
    for (int k = 0; k < F; k++)
        for (int c = 0; c < C; c++)
            for (int p = 0; p < kPos; p++) {
                double v = 0.0;
                for (int tap = 0; tap < 9; tap++)
                    v += G[p / 6][tap / 3] * G[p % 6][tap % 3] *
                         (double)Wf[conv3x3_index(k, c, tap, Kp)];
                U[((size_t)p * Kp + k) * Cp + c] = (half_t)v;
            }
}

}  // namespace lzhip
