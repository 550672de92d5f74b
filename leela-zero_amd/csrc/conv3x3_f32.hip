// Direct 3x3 convolution for fp32 towers on the fp16 matrix cores (gfx950): one kernel per layer,
// convolution + batch norm + skip connection + ReLU, channels-last fp32 activations in and out.
//
// The fp32 matrix instructions have a sixteenth of the fp16 rate.  Here every operand is the sum of
// two half-precision numbers, x = (hi + lo) / 2^e with hi = half(x 2^e), lo = half(x 2^e - hi): 22 bits
// of significand and the sign, one bit less than fp32 holds.  A product is hi hi' + hi lo' + lo hi' (the
// fourth term is below 2^-22 of it), three instructions at sixteen times the rate, accumulated in
// fp32.  2^e brings the operand to the top of half's range, so that lo is a normal number
// down to 2^-17 of the largest and exact to 2^-39 of it below: for planes from the largest
// activation of the board (each layer leaves it for the next), for filters from the largest weight of
// the output channel.  Channels of different magnitude are brought together beforehand, by powers of two
// in the filters and in the batch norm that leave every product as it is (balance_channels in
// hip_pipe.hip); a network that this does not help runs the Winograd kernels.  Error against float64 is smaller than the Winograd kernels' (F(4x4,3x3)
// amplifies fp32 rounding): figures at conv3x3_f32_serves.
//
// The matrix instruction drops bits of its products below the largest term's, downwards (measured: sums
// of 32 random products and an addend come out low by a third of an ulp where they are positive and by
// nothing where they are negative).  Over a tower's layers that adds up, so the filters of the second
// half of a layer's input channels are stored negated and the sum changes its sign in between: what
// the one half loses the other gains.
#include <algorithm>
#include <cmath>
#include <stdexcept>
#include <type_traits>

#include "conv3x3_tile.h"

namespace lzhip {

typedef _Float16 half4v __attribute__((ext_vector_type(4)));

constexpr int kF32Chunk = 32;         // input channels per 128 bytes of a cell
constexpr int kF32Steps = 18;         // k-steps per chunk: 9 taps x {hi, lo} of 32 channels
constexpr int kF32Lookahead = 18;     // most k-steps of filters requested ahead
constexpr int kPlaneTop = 14;         // planes are scaled to a maximum in [2^14, 2^15)
constexpr int kFilterTop = 11;        // filters of an output channel to [2^11, 2^12)

// Filters: [k-step][Kp / 16][64 lanes][8] half, k-step = (chunk of 32 input channels, tap, hi or lo): the
// matrix instruction's row operand.  Lane l of block kb holds output channel 16 kb + l % 16, input channels
// 8 (l / 16) + 0..7 of the chunk; register r of lane l of the result is channel 16 kb + 4 (l / 16) + r.
// Channels from Cp / 2 on are negated.
__host__ __device__ static inline bool conv3x3_f32_negated(int c, int Cp) { return c >= Cp / 2; }
__host__ __device__ static inline size_t conv3x3_f32_index(int k, int c, int tap, int part, int Kp) {
    const int step = ((c >> 5) * 9 + tap) * 2 + part;
    const int lane = ((c >> 3) & 3) * 16 + (k & 15);
    return (((size_t)step * (Kp / 16) + (k >> 4)) * 64 + lane) * 8 + (c & 7);
}

size_t conv3x3_f32_filter_count(int Cp, int Kp) {
    return (size_t)(18 * Cp / 32 + kF32Lookahead) * Kp * 32;
}

// Power of two that brings a board whose largest magnitude has these bits to the top of half's
// range, and its reciprocal.  (Exponents are kept where both are normal numbers; the largest
// magnitude recorded is finite.)
__device__ __forceinline__ unsigned peak_exponent(unsigned bits) {
    const unsigned e = bits >> 23;
    return min(max(e, (unsigned)kPlaneTop + 1u), 254u);
}
__device__ __forceinline__ float plane_scale(unsigned bits) {
    return __builtin_bit_cast(float, (254u + kPlaneTop - peak_exponent(bits)) << 23);
}
__device__ __forceinline__ float plane_unscale(unsigned bits) {
    return __builtin_bit_cast(float, (peak_exponent(bits) - kPlaneTop) << 23);
}

// Four values of a plane, split, to the hi and the lo half of a cell.
__device__ __forceinline__ void store_split(unsigned char* at, int4v bits, float scale) {
    const float4v v = __builtin_bit_cast(float4v, bits) * scale;
    half4v hi, lo;
#pragma unroll
    for (int e = 0; e < 4; e++) hi[e] = (half_t)v[e];
#pragma unroll
    for (int e = 0; e < 4; e++) lo[e] = (half_t)(v[e] - (float)hi[e]);
    *reinterpret_cast<half4v*>(at) = hi;
    *reinterpret_cast<half4v*>(at + 64) = lo;
}

__device__ __forceinline__ float4v mfma(int4v w, int4v x, float4v acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8v, w),
                                                  __builtin_bit_cast(half8v, x), acc, 0, 0, 0);
}

// Of conv3x3_k's order in LDS (CellPitch) these kernels take what costs no address: a lane's point is conv_point's,
// and quarters 2 i and 2 i + 1 of a cell's 32 channels stand an even number of 16 bytes apart, so that of the 16
// lanes served together eight meet odd and eight even slots, but in blocks that a board row ends in. (Its longer rows
// cost more than they gave.) With quarters and points in their natural order nearly every read took two turns, 17 %
// of a launch of 15x192, 8 boards, now 9; 40x256, 64 boards: 20, now 10. A forward, us: 15x192, 1 board 198 -> 191, 2
// boards 238 -> 223, 8: 319 -> 316; 20x256, 1 board 286 -> 272; 10x512, 1 board 256 -> 235; conv3x3_f32_k, 6 blocks:
// 256 filters, 1 board 151 -> 141, 8: 198 -> 191, 64: 740 -> 737; 128, 1 board 100 -> 93; 192, 8 boards 160 -> 153;
// 384, 24 boards 657 -> 650.
// Byte of piece x of a cell: channels 4 x to 4 x + 3.
__device__ __forceinline__ unsigned f32_piece(unsigned x) { return quarter_slot(x >> 1) * 16 + (x & 1) * 8; }

// Largest value of a wavefront, in every lane.
__device__ __forceinline__ unsigned wave_max(unsigned v) {
    auto step = [&](auto ctrl, auto rows) {
        v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value,
                                                         decltype(rows)::value, 0xf, false));
    };
    using std::integral_constant;
    step(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});   // row_shr:1, 2, 4, 8
    step(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});
    step(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});
    step(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});
    step(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});   // row_bcast:15, 31
    step(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// Peaks.  Every work-group leaves the largest finite results of its tile (bits of a float), first
// board and second board apart, in slots of its own: slots[tile row][2][tile column].  A work-group
// of the next layer takes the maximum over the tiles that meet its boards.  (One word per board
// that all work-groups update by atomics was measured too: atomics on a line take some 30 cycles
// each, 2.5 to 10 us at the end of a layer.)
struct PeakIn {
    const unsigned* slots;
    unsigned mt, tiles_n;   // points per tile, tile columns
    unsigned inv_m, inv_n;  // ceil(2^32 / mt), ceil(2^31 / tiles_n)
};
static PeakIn peak_in(const PeakMap& p) {
    return {p.slots, (unsigned)p.mt, (unsigned)p.tiles_n,
            (unsigned)((((uint64_t)1 << 32) + p.mt - 1) / p.mt),
            (unsigned)((((uint64_t)1 << 31) + p.tiles_n - 1) / p.tiles_n)};
}
// The most slots a board may have: it meets 360 / mt + 2 rows of tiles at most.
static constexpr int peak_slots(int mt, int tiles_n) { return (360 / mt + 2) * tiles_n; }
// Whether a layer's peaks, two a tile, lie within what conv3x3_f32_slots keeps for them.
static void slots_fit(int tiles_m, int tiles_n, int Kp, int n) {
    if (2 * (size_t)tiles_m * tiles_n > conv3x3_f32_slots(Kp, n)) throw std::logic_error("more peaks than slots");
}
static void peaks_fit(const PeakMap& p, int loads) {
    if (peak_slots(p.mt, p.tiles_n) > 64 * loads) throw std::logic_error("a board of more peaks than are read");
}
// Requests up to MAX x 64 slots of a board, the first ALL x 64 without a look at how many there are, and takes
// their maximum.  Behind a branch that is taken a request is waited for at the branch's end, with everything
// requested before it: small batches, whose tiles are small, had two to five of those before their planes.
// Without them a forward of 15 layers of 192 filters takes 198 us instead of 215 for 1 board, 20 of 256 283
// instead of 307 (2 boards 344, 359), 20 of 128 216 instead of 227, 10 of 512 255 instead of 272.
template <int ALL, int MAX>
struct BoardPeak {
    unsigned v[MAX];
    __device__ __forceinline__ void load(const PeakIn& p, unsigned board, unsigned lane) {
        const unsigned first = board * kPts, t0 = __umulhi(first, p.inv_m);
        const unsigned tiles = __umulhi(first + kPts - 1, p.inv_m) - t0 + 1, count = tiles * p.tiles_n;
        const unsigned late = t0 * p.mt < first ? 1u : 0u;   // the first tile's second board
        const __amdgpu_buffer_rsrc_t r =
            make_rsrc(p.slots + (size_t)t0 * 2 * p.tiles_n, (size_t)tiles * 2 * p.tiles_n * 4);
#pragma unroll
        for (int k = 0; k < MAX; k++) {
            if (k >= ALL) v[k] = 0;
            if (k < ALL || k * 64 < (int)count) {
                const unsigned i = lane + k * 64, t = __umulhi(i * 2u, p.inv_n);
                const unsigned at = (t * 2 + (t == 0 ? late : 0u)) * p.tiles_n + i - t * p.tiles_n;
                // (beyond the last row of tiles this lies outside the buffer: 0)
                v[k] = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, at * 4u, 0, 0);
            }
        }
    }
    __device__ __forceinline__ unsigned get() const {
        unsigned top = v[0];
#pragma unroll
        for (int k = 1; k < MAX; k++) top = max(top, v[k]);
        return wave_max(top);
    }
};
// Scales of a tile's first board and of the next one, and their reciprocals.
struct TileScales {
    float s0, s1, u0, u1;
};
// First cell of the patch that lies on the tile's second board (or past the patch).
__device__ __forceinline__ unsigned second_board(const PatchStart& s) {
    return (s.mb + 2) * kCellsPerBoard - s.q0;
}
template <int ALL, int MAX>
struct TilePeaks {
    BoardPeak<ALL, MAX> a, b;
    bool two;   // the tile reaches a second board
    __device__ __forceinline__ void load(const PeakIn& p, const PatchStart& s, int m0, int mt, int rows,
                                         unsigned lane) {
        const int m1 = ((int)s.mb + 1) * kPts;
        two = m0 + mt > m1 && m1 < rows;
        a.load(p, s.mb, lane);
        if (two) b.load(p, s.mb + 1, lane);
    }
    __device__ __forceinline__ TileScales scales() const {
        const unsigned p0 = a.get(), p1 = two ? b.get() : p0;
        return {plane_scale(p0), plane_scale(p1), plane_unscale(p0), plane_unscale(p1)};
    }
};
// What a wavefront leaves in red[wavefront] and, after a barrier, the work-group in its slots.
__device__ __forceinline__ float finite(float v) { return v < __builtin_inff() ? v : 0.0f; }
template <int WAVES>
__device__ __forceinline__ void leave_peaks(unsigned (*red)[2], unsigned* slots, int tm, int tn,
                                            int tiles_n, int wave, float top0, float top1) {
    const unsigned p0 = wave_max(__builtin_bit_cast(unsigned, top0));
    const unsigned p1 = wave_max(__builtin_bit_cast(unsigned, top1));
    if ((threadIdx.x & 63) < 2) red[wave][threadIdx.x & 63] = (threadIdx.x & 63) == 0 ? p0 : p1;
    lds_barrier();
    if (threadIdx.x < 2) {
        unsigned top = 0;
#pragma unroll
        for (int k = 0; k < WAVES; k++) top = max(top, red[k][threadIdx.x]);
        slots[(size_t)(tm * 2 + (int)threadIdx.x) * tiles_n + tn] = top;
    }
}

// One work-group computes WR * RB * 16 points x WN * NB * 16 output channels as conv3x3_k does (its
// comment has the reasons for the staging, the rings and the tiles).  A chunk is 32 input channels: a
// cell holds their hi parts in its first 64 bytes and their lo parts in the next 64, a k-step is one tap
// with the filters' hi or lo parts.  The fragments of both parts of a tap are read once and used
// three times, and so are two thirds of the filters, which halves what LDS and L1 deliver per
// instruction beside the fp16 kernel.
//
// CC == 0: chunks in two LDS buffers.  CC > 0: all CC chunks staged before the first product.
template <int RB, int NB, int WR, int WN, int D, int CC, int OCC>
__global__ __launch_bounds__(64 * WR * WN, OCC) void conv3x3_f32_k(
    const float* __restrict__ X, const half_t* __restrict__ Wf, const float* __restrict__ res,
    float* __restrict__ Y, const float* __restrict__ bn_scale, const float* __restrict__ bn_mean,
    float rfac, PeakIn peaks, unsigned* __restrict__ slots, int n, int Cp, int Kp, ConvGrid g) {
    constexpr bool DB = CC == 0;
    constexpr int NT = 64 * WR * WN;
    constexpr int MT = WR * RB * 16, CW = WN * NB * 16;
    constexpr int CELLS = conv_cells(MT);
    constexpr int STR = 144, BUF = (CELLS + 1) * STR;   // bytes per cell; per chunk
    constexpr int PPC = 8, NP = (CELLS * PPC + NT - 1) / NT;
    constexpr int KS = kF32Steps;
    constexpr bool BIG = RB * NB >= 24;                 // accumulators are most of the registers
    constexpr int SGRP = BIG ? 1 : 3, NG = (NP + SGRP - 1) / SGRP, GS = KS / NG > 0 ? KS / NG : 1;
    constexpr bool EARLY = RB * NB <= 6;
    constexpr int LO = BIG ? RB / 2 : RB;               // lo fragments held
    constexpr int RQ = EARLY ? RB : RB / 2;             // row blocks of the skip connection held
    static_assert(KS % D == 0 && D <= kF32Lookahead, "rings turn a whole number of times per chunk");
    static_assert(!DB || NG <= KS, "one group of pieces per k-step at most");
    static_assert(NT % PPC == 0 && CW <= NT && MT <= kPts, "tile");
    __shared__ __attribute__((aligned(16))) unsigned char lds[(DB ? 2 : CC) * BUF];
    __shared__ __attribute__((aligned(16))) float bn[2][CW];
    __shared__ unsigned red[NT / 64][2];

    const ConvTile tile = conv_tile(g);
    const int tn = tile.n, tm = tile.m;
    if (tm >= g.tiles_m) return;
    const int rows = n * kPts, m0 = tm * MT;
    const unsigned tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const int wr = wave / WN, wn = wave % WN;

    const unsigned bnoff = tid < (unsigned)CW ? (tn * CW + tid) * 4u : 0xfffffff0u;
    const float scale = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                      make_rsrc(bn_scale, Kp * 4), bnoff, 0, 0));
    const float mean = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                     make_rsrc(bn_mean, Kp * 4), bnoff, 0, 0));
    const int kb = (tn * WN + wn) * NB;
    unsigned ws = (unsigned)kb * 1024u;
    const unsigned wstep = (unsigned)Kp * 64u;
    const unsigned wv = lane * 16u;
    const __amdgpu_buffer_rsrc_t rW =
        make_rsrc(Wf, ((size_t)18 * Cp / 32 + kF32Lookahead) * Kp * 64);
    int4v w[D][NB];
    auto wload = [&](int slot, int j, unsigned st) {
        w[slot][j] = __builtin_amdgcn_raw_buffer_load_b128(rW, wv + j * 1024, ws + st * wstep, 0);
    };
    // The filters of two k-steps go before the planes, the others behind them (CC == 0): 6 blocks of 256 filters, 12
    // boards 248 -> 243 us, of 128, 32 boards 165 -> 162, of 192, 30 boards 276 -> 269, of 384, 8 boards 331 ->
    // 326; 20 boards of 256 filters and more within 1 %.
    constexpr int F0 = DB && D - 1 > 2 ? 2 : D - 1;
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
    TilePeaks<0, 2> tp;
    tp.load(peaks, ps, m0, MT, rows, lane);
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(X, (size_t)(n + 2) * kCellsPerBoard * Cp * 4);
    const unsigned xrow = (unsigned)Cp * 4u;     // bytes of a cell in memory
    const unsigned xoff = (ps.q0 + tid / PPC) * xrow + (tid % PPC) * 16u;
    // piece i, `at` bytes into the cells' channels
    auto xload = [&](int i, unsigned at) {
        return __builtin_amdgcn_raw_buffer_load_b128(rX, xoff, i * (NT / PPC) * xrow + at, 0);
    };
    // LDS address of piece i: a constant distance from piece 0 (the last may lie past the end)
    const unsigned lst = (tid / PPC) * STR + f32_piece(tid % PPC);
    TileScales ts;
    unsigned tv = tid;   // (opaque in every chunk: the scales of the pieces are not held)
    auto put = [&](int i, unsigned buffer, int4v bits) {
        const unsigned cell = tv / PPC + i * (NT / PPC);
        const unsigned at = i < NP - 1 || (CELLS * PPC) % NT == 0
                                ? lst + i * (NT / PPC) * STR
                                : min(cell, (unsigned)CELLS) * STR + f32_piece(tid % PPC);
        store_split(lds + buffer + at, bits, cell < second_board(ps) ? ts.s0 : ts.s1);
    };

    const int chunks = Cp / kF32Chunk;
    const int ch0 = kb * 16 + 4 * (int)(lane >> 4);   // first channel
    unsigned arow[RB];   // LDS address of this lane's point of each row block, tap (0, 0)
    unsigned ro[RB];     // byte offset of this lane's point and channel
    int4v rr[RQ][NB];
#pragma unroll
    for (int i = 0; i < RB; i++) {
        const int local = (wr * RB + i) * 16 + conv_point(lane);
        const unsigned cell = patch_cell(ps, min(local, rows - 1 - m0));
        arow[i] = cell * STR + quarter_slot(lane >> 4) * 16;
        ro[i] = m0 + local < rows ? ((ps.q0 + kPointCell + cell) * Kp + ch0) * 4u : 0xfffff000u;
    }
    const size_t ybytes = (size_t)(n + 2) * kCellsPerBoard * Kp * 4;
    const __amdgpu_buffer_rsrc_t rY = make_rsrc(Y, ybytes);
    const __amdgpu_buffer_rsrc_t rR = make_rsrc(res != nullptr ? res : Y, ybytes);
    auto load_res = [&](int i) {
#pragma unroll
        for (int j = 0; j < NB; j++)
            rr[i % RQ][j] = res != nullptr
                                ? __builtin_amdgcn_raw_buffer_load_b128(rR, ro[i] + j * 64, 0, 0)
                                : int4v{0, 0, 0, 0};
    };
    auto first_res = [&]() {
#pragma unroll
        for (int i = 0; i < RQ; i++) load_res(i);
    };

    if constexpr (DB) {
        int4v stg[NP];
#pragma unroll
        for (int i = 0; i < NP; i++) stg[i] = xload(i, 0);
        __builtin_amdgcn_sched_barrier(0);
        filters(F0, D - 1);
        if constexpr (EARLY) first_res();
        ts = tp.scales();
#pragma unroll
        for (int i = 0; i < NP; i++) put(i, 0, stg[i]);
    } else {
        constexpr int ALL = CC * NP, FLY = ALL < 24 ? ALL : 24;   // pieces in flight
        int4v stg[FLY];
#pragma unroll
        for (int p = 0; p < ALL + FLY; p++) {
            if (p == FLY) ts = tp.scales();
            if (p >= FLY) put((p - FLY) % NP, (p - FLY) / NP * BUF, stg[p % FLY]);
            if (p < ALL) stg[p % FLY] = xload(p % NP, p / NP * 128);
        }
        if constexpr (EARLY) first_res();
    }
    if (tid < (unsigned)CW) {
        bn[0][tid] = scale;
        bn[1][tid] = -scale * mean;
    }
    float4v acc[RB][NB];
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    lds_barrier();

    int4v hi[RB], lo[LO];   // fragments of the tap at hand
    auto aread = [&](int i, int part, int tap) {
        return *reinterpret_cast<const int4v*>(lds + arow[i] + ((tap / 3) * 20 + tap % 3) * STR +
                                               part * 64);
    };
    unsigned other = BUF;   // byte offset of the buffer being filled (CC == 0)
    // Chunk c; the last one stages nothing and fetches no filters past its end, and the skip connection
    // comes into the registers that this leaves.
    auto chunk = [&](int c, auto is_last) {
        constexpr bool LAST = decltype(is_last)::value;
        asm volatile("" : "+v"(tv));
        if (2 * c == chunks) {
#pragma unroll
            for (int i = 0; i < RB; i++)
#pragma unroll
                for (int j = 0; j < NB; j++) acc[i][j] = -acc[i][j];
        }
#pragma unroll
        for (int i = 0; i < RB; i++) {
            hi[i] = aread(i, 0, 0);
            if (i < LO) lo[i] = aread(i, 1, 0);
        }
        const unsigned next = (unsigned)(c + 1) * 128u;
        int4v sg[SGRP];
#pragma unroll
        for (int st = 0; st < KS; st++) {
            if constexpr (LAST && !EARLY) {
                if (st == KS - 1) first_res();
            }
            if constexpr (DB && !LAST) {
#pragma unroll
                for (int gr = 0; gr < NG; gr++) {
                    if (st == gr * GS) {
#pragma unroll
                        for (int i = 0; i < SGRP; i++)
                            if (gr * SGRP + i < NP)
                                sg[i] = xload(gr * SGRP + i, next);
                    }
                    if (st == (gr + 1) * GS - 1) {
#pragma unroll
                        for (int i = 0; i < SGRP; i++)
                            if (gr * SGRP + i < NP) put(gr * SGRP + i, other, sg[i]);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            const int part = st & 1, tap = st / 2;
#pragma unroll
            for (int i = 0; i < RB; i++) {
#pragma unroll
                for (int j = 0; j < NB; j++)
                    if (i == (RB >= NB ? j : 0) && (!LAST || st + D - 1 < KS))
                        wload((st + D - 1) % D, j, st + D - 1);
#pragma unroll
                for (int j = 0; j < NB; j++) acc[i][j] = mfma(w[st % D][j], hi[i], acc[i][j]);
                // (fragments are read behind the instructions that used their registers last)
                if (part == 0) {
#pragma unroll
                    for (int j = 0; j < NB; j++)
                        acc[i][j] = mfma(w[st % D][j], lo[i % LO], acc[i][j]);
                    if (i + LO < RB)
                        lo[i % LO] = aread(i + LO, 1, tap);
                    else if (tap < 8)
                        lo[i % LO] = aread(i + LO - RB, 1, tap + 1);
                } else if (tap < 8) {
                    hi[i] = aread(i, 0, tap + 1);
                }
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
            for (int i = 0; i < RB; i++) arow[i] += BUF;
        }
    };
#pragma unroll 1
    for (int c = 0; c < chunks - 1; c++) chunk(c, std::false_type{});
    chunk(chunks - 1, std::true_type{});

    // max(0, scale * (y - mean) + rfac * res)
    float top0 = 0.0f, top1 = 0.0f;
    const int m1 = ((int)ps.mb + 1) * kPts;   // first row of the tile's second board
#pragma unroll
    for (int i = 0; i < RB; i++) {
        const int m = m0 + (wr * RB + i) * 16 + conv_point(lane);
        const float unscale = m < m1 ? -ts.u0 : -ts.u1;   // (the sum ends negated)
        float top = 0.0f;
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const int cl = ch0 - tn * CW + j * 16;
            const float4v r = __builtin_bit_cast(float4v, rr[i % RQ][j]);
            float4v o;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                o[e] = fmaxf(0.0f, fmaf(r[e], rfac, fmaf(acc[i][j][e] * unscale, bn[0][cl + e],
                                                         bn[1][cl + e])));
                top = fmaxf(top, finite(o[e]));
            }
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(int4v, o), rY,
                                                   ro[i] + j * 64, 0, kStoreThrough);
        }
        if (i + RQ < RB) load_res(i + RQ);
        top0 = fmaxf(top0, m < m1 ? top : 0.0f);
        top1 = fmaxf(top1, m >= m1 && m < rows ? top : 0.0f);
    }
    leave_peaks<NT / 64>(red, slots, tm, tn, Kp / CW, wave, top0, top1);
}

template <int RB, int NB, int WR, int WN, int D, int CC, int OCC>
static PeakMap launch_f32_as(const float* X, const half_t* Wf, const float* res, float* Y,
                             const float* bn_scale, const float* bn_mean, float rfac,
                             const PeakMap& peaks, unsigned* slots, int n, int Cp, int Kp,
                             hipStream_t s, LaunchTimer* t) {
    constexpr int MT = WR * RB * 16, CW = WN * NB * 16;
    const ConvGrid g = conv_grid((n * kPts + MT - 1) / MT, Kp / CW, (size_t)36 * Cp * Kp,
                                 (size_t)n * kPts * Cp * 4);
    peaks_fit(peaks, 2);
    slots_fit(g.tiles_m, Kp / CW, Kp, n);
    launch(conv3x3_f32_k<RB, NB, WR, WN, D, CC, OCC>, dim3(8 * g.share), dim3(64 * WR * WN), s, t, X,
           Wf, res, Y, bn_scale, bn_mean, rfac, peak_in(peaks), slots, n, Cp, Kp, g);
    return {slots, MT, Kp / CW};
}

// The tiles and their order are conv3x3_k's (launch_conv3x3).  Measured, us per layer of a chain (two chains
// side by side, per chain): 256 filters, 20 boards 192x64 31.8, 128x64 24.5 (21.9 | 20.2); 192 filters, 28 boards
// 192x64 25.1, 128x64 19.7 (30 boards 19.5 | 17.3), 46 boards 128x192 40.0, 128x64 32.4 (28.1 | 25.3); 384 filters, 13
// boards 192x64 44.7, 128x64 33.5 (32.1 | 29.1).
PeakMap launch_conv3x3_f32(const float* X, const half_t* Wf, const float* res, float* Y,
                           const float* bn_scale, const float* bn_mean, float rfac,
                           const PeakMap& peaks, uint32_t* slots, int n, int Cp, int Kp,
                           int lanes, hipStream_t s, LaunchTimer* t) {
    if (Kp % 64 != 0 || Cp % 64 != 0)
        throw std::invalid_argument("no direct convolution for this width");
    const int rows = n * kPts;
    auto groups = [&](int mt, int cw) { return ((rows + mt - 1) / mt) * (Kp / cw); };
#define LZ_F32(RB, NB, WR, WN, D, CC, OCC)                                                        \
    launch_f32_as<RB, NB, WR, WN, D, CC, OCC>(X, Wf, res, Y, bn_scale, bn_mean, rfac, peaks,      \
                                              slots, n, Cp, Kp, s, t)
    const int cc = Cp / kF32Chunk;
    if (cc <= 8 && groups(32, 64) <= kUnits) {
        switch (cc) {
            case 2: return LZ_F32(2, 1, 1, 4, 9, 2, 1);
            case 4: return LZ_F32(2, 1, 1, 4, 9, 4, 1);
            case 6: return LZ_F32(2, 1, 1, 4, 9, 6, 1);
            default: return LZ_F32(2, 1, 1, 4, 9, 8, 1);
        }
    }
    // Four wavefronts of 16 channels for up to two forwards side by side: a layer of 256 filters, 8
    // boards 19.0 -> 15.5 us, 192 filters, 11 boards 15.0 -> 12.4 against two wavefronts of 32
    // channels, and three forwards side by side 4 to 7 % slower.  64x64 gains 2 to 5 % on 96x64 for a
    // forward with the device to itself and loses 14 % with three.
    if (groups(48, 64) <= kUnits) {
        if (lanes <= 2) return LZ_F32(3, 1, 1, 4, 6, 0, 2);
        return LZ_F32(3, 2, 1, 2, 6, 0, 2);
    }
    if (lanes == 1 && groups(64, 64) <= kUnits) {
        return LZ_F32(4, 1, 1, 4, 6, 0, 2);
    }
    if (groups(96, 64) <= kUnits) {
        return LZ_F32(3, 2, 2, 2, 6, 0, 2);
    }
    if (groups(128, 64) <= kUnits) {
        return LZ_F32(4, 2, 2, 2, 6, 0, 2);
    }
    // launch_conv3x3's tiles of 128 channels and 160x64.  256 filters, 24 boards 192x64 32.2, 80x128 27.8 us (two side by
    // side 23.9 | 22.3), 50 boards 192x128 50.4, 144x128 47.9 (42.8 | 41.0); 384 filters, 16 boards 44.6 -> 38.5, 26: 56.4
    // -> 53.3; 128 filters, 50 boards 19.5 -> 17.4; 192 filters, 33 boards 192x64 26.3, 160x64 23.5 (19.5 | 18.2).
#define LZ_WIDE(RB) \
    case RB:        \
        return LZ_F32(RB, 2, 1, 4, (RB < 9 ? 6 : 3), 0, 2)
    auto wide = [&](int rb) {
        switch (rb) {
            LZ_WIDE(5);
            LZ_WIDE(6);
            LZ_WIDE(7);
            LZ_WIDE(8);
            LZ_WIDE(9);
            LZ_WIDE(10);
            default: return LZ_F32(6, 4, 2, 2, 3, 0, 2);
        }
    };
#undef LZ_WIDE
    const bool wide_columns = Kp % 128 == 0;
    if (wide_columns && lanes <= 2) {
        const int rb = one_round_blocks(rows, Kp / 128, 5);
        if (rb > 0 && (lanes == 1 || rb != 6)) return wide(rb);
    }
    if (!wide_columns && Kp != 64 && groups(160, 64) <= kUnits) {
        return LZ_F32(5, 2, 2, 2, 6, 0, 2);
    }
    if (groups(192, 64) <= kUnits) {
        return LZ_F32(6, 2, 2, 2, 6, 0, 2);
    }
    if (wide_columns) {
        if (const int rb = one_round_blocks(rows, Kp / 128, 7)) return wide(rb);
    }
    if ((Kp == 64 || Kp == 192) && groups(128, 64) <= 2 * kUnits) {
        return LZ_F32(4, 2, 2, 2, 6, 0, 2);
    }
    // (launch_conv3x3's rule for more than a round)
    if (wide_columns) return wide(lanes == 1 ? least_rounds_blocks(rows, Kp / 128) : 12);
    auto rounds = [&](int mt, int cw) { return (groups(mt, cw) + kUnits - 1) / kUnits * mt * cw; };
    if (lanes == 1 && rounds(128, 64) < rounds(192, 64) &&
        (Kp != 192 || rounds(128, 64) < rounds(128, 192)))
        return LZ_F32(4, 2, 2, 2, 6, 0, 2);
    if (Kp == 192 && (lanes > 1 || rounds(128, 192) <= rounds(192, 64)))
        return LZ_F32(4, 6, 2, 2, 3, 0, 2);
    return LZ_F32(6, 2, 2, 2, 6, 0, 2);
#undef LZ_F32
}

// ---------------------------------------------------------------------------
// The same layer with the sum over input channels dealt to the wavefronts of a work-group, for handles
// whose batches leave a compute unit one tile (the reasons are conv3x3_split_k's): a wavefront
// computes the whole tile of RB * 16 points x NB * 16 output channels over HPW chunks of 32 input
// channels, which it stages itself, one after the other in the same place; the partial sums meet
// in LDS, in the order of the wavefronts.
//
// A tile is 16 channels wide where that makes no more than one work-group per unit: with hi
// and lo parts the filters are twice as many bytes as in fp16, and what the L1 delivers to a unit
// (filters of NB * 16 channels, planes of conv_cells(RB * 16) cells) is what a tile waits for.
//
// A unit has four SIMDs: two wavefronts leave two of them idle, five and six leave two or three with half the
// work of the others.  There WR x WN wavefronts share the channels, and each has its rows or columns of
// blocks; they stage the planes together.  Measured per forward of 10 blocks, us, WR * WN = 1 -> here (one at a
// time | two side by side): 64 filters, 1 board 96 -> 93 | 52 -> 50, 6: 111 -> 104 | 66 -> 64, 11: 115 -> 104 |
// 71 -> 71, 22: 152 -> 118 | 88 -> 73, 34: 179 -> 137 | 102 -> 88; 192 filters, 8 boards 227 -> 217 | 164 ->
// 158, 15: 302 -> 288 | 255 -> 241; 320, 6: 375 -> 356 | 325 -> 313; 384, 5: 386 -> 372 | 341 -> 332.  Tiles of 32
// channels and less of 192 filters and more stay: halves of their blocks fetch more from LDS per instruction
// (192 filters, 5 boards 187 -> 212), and so does 64 filters' 64x64 in quarters (45 boards 162 -> 174).  Four
// and eight wavefronts fill the SIMDs as they are (128 filters, 8 boards 155 -> 168, 256, 8: 277 -> 295).
//
// The peaks come from a layer of the same tiles, or from conv3x3_f32_k's 32x64 of the first layer.
static constexpr int split_peak_loads(int rb, int nb, int filters) {
    const int own = peak_slots(rb * 16, filters / (nb * 16)), first = peak_slots(32, filters / 64);
    return ((own > first ? own : first) + 63) / 64;
}
template <int RB, int NB, int KW, int HPW, int D, int WR, int WN>
__global__ __launch_bounds__(64 * KW * WR * WN, 1) void conv3x3_f32_split_k(
    const float* __restrict__ X, const half_t* __restrict__ Wf, const float* __restrict__ res,
    float* __restrict__ Y, const float* __restrict__ bn_scale, const float* __restrict__ bn_mean,
    float rfac, PeakIn peaks, unsigned* __restrict__ slots, int n, int Kp, ConvGrid g) {
    constexpr int Cp = kF32Chunk * HPW * KW, WS = WR * WN, NT = 64 * KW * WS;
    constexpr int RBW = RB / WR, NBW = NB / WN;   // a wavefront's blocks
    constexpr int MT = RB * 16, CW = NB * 16, CELLS = conv_cells(MT);
    constexpr int STR = 144, SLICE = (CELLS + 1) * STR;
    constexpr int PPC = 8, NP = (CELLS * PPC + 64 * WS - 1) / (64 * WS);
    constexpr int STEPS = kF32Steps * HPW;
    constexpr int BLOCKS = RB * NB, QB = (BLOCKS + KW * WS - 1) / (KW * WS);   // a wavefront finishes QB blocks
    constexpr int BYTES = KW * (SLICE > BLOCKS * 1024 ? SLICE : BLOCKS * 1024);
    static_assert(D <= STEPS && D <= kF32Lookahead && CW <= NT && MT <= kPts && RB % WR == 0 && NB % WN == 0, "tile");
    __shared__ __attribute__((aligned(16))) unsigned char lds[BYTES];
    __shared__ __attribute__((aligned(16))) float bn[2][CW];
    __shared__ unsigned red[NT / 64][2];

    const ConvTile tile = conv_tile(g);
    const int tn = tile.n, tm = tile.m;
    if (tm >= g.tiles_m) return;
    const int rows = n * kPts, m0 = tm * MT;
    const unsigned tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const int kw = WS == 1 ? wave : wave % KW, ww = WS == 1 ? 0 : wave / KW;   // its channels; its part of the tile
    const int wr = ww / WN, wn = ww % WN;

    const unsigned bnoff = tid < (unsigned)CW ? (tn * CW + tid) * 4u : 0xfffffff0u;
    const float scale = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                      make_rsrc(bn_scale, Kp * 4), bnoff, 0, 0));
    const float mean = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                     make_rsrc(bn_mean, Kp * 4), bnoff, 0, 0));
    const unsigned wstep = (unsigned)Kp * 64u;
    const unsigned ws = (unsigned)(kw * STEPS) * wstep + (unsigned)(tn * NB + wn * NBW) * 1024u;
    const __amdgpu_buffer_rsrc_t rW =
        make_rsrc(Wf, ((size_t)18 * Cp / 32 + kF32Lookahead) * Kp * 64);
    int4v w[D][NBW];
    auto wload = [&](int slot, int j, unsigned st) {
        w[slot][j] = __builtin_amdgcn_raw_buffer_load_b128(rW, lane * 16u + j * 1024, ws + st * wstep, 0);
    };
    // A few filters, the planes, the other filters (conv3x3_split_k).
    constexpr int F0 = D - 1 < 4 ? D - 1 : 4;
    auto filters = [&](int from, int to) {
#pragma unroll
        for (int d = 0; d < D - 1; d++)
#pragma unroll
            for (int j = 0; j < NBW; j++)
                if (d >= from && d < to) wload(d, j, d);
        __builtin_amdgcn_sched_barrier(0);
    };
    filters(0, F0);
    const PatchStart ps = patch_start(m0);
    constexpr int PEAKS = split_peak_loads(RB, NB, Cp);
    TilePeaks<PEAKS, PEAKS> tp;
    tp.load(peaks, ps, m0, MT, rows, lane);
    const __amdgpu_buffer_rsrc_t rX = make_rsrc(X, (size_t)(n + 2) * kCellsPerBoard * Cp * 4);
    constexpr unsigned xrow = Cp * 4;   // bytes of a cell in memory
    const unsigned xoff = (ps.q0 + ww * (64 / PPC) + lane / PPC) * xrow + (lane % PPC) * 16u;
    auto xload = [&](int i, int h) {   // piece i of the wavefront's chunk h
        return __builtin_amdgcn_raw_buffer_load_b128(
            rX, xoff, i * WS * (64 / PPC) * xrow + (kw * HPW + h) * 128, 0);
    };
    int4v stg[NP];
#pragma unroll
    for (int i = 0; i < NP; i++) stg[i] = xload(i, 0);
    __builtin_amdgcn_sched_barrier(0);
    filters(F0, D - 1);
    const TileScales ts = tp.scales();

    // the blocks that this wavefront finishes: where they lie, and the skip connection
    unsigned ro[QB];
    int4v rr[QB];
    const size_t ybytes = (size_t)(n + 2) * kCellsPerBoard * Kp * 4;
    const __amdgpu_buffer_rsrc_t rY = make_rsrc(Y, ybytes);
    const __amdgpu_buffer_rsrc_t rR = make_rsrc(res != nullptr ? res : Y, ybytes);
    const int cl = 4 * (int)(lane >> 4);   // first of this lane's 4 channels of a block
#pragma unroll
    for (int q = 0; q < QB; q++) {
        const int id = q * KW * WS + wave, local = id / NB * 16 + conv_point(lane);
        ro[q] = id < BLOCKS && m0 + local < rows
                    ? ((ps.q0 + kPointCell + patch_cell(ps, local)) * Kp + tn * CW + id % NB * 16 + cl) * 4u
                    : 0xfffffff0u;
        rr[q] = int4v{0, 0, 0, 0};
    }
    if (res != nullptr) {
#pragma unroll
        for (int q = 0; q < QB; q++)
            rr[q] = __builtin_amdgcn_raw_buffer_load_b128(rR, ro[q], 0, 0);
    }
    unsigned char* const own = lds + kw * SLICE;
    auto stage = [&]() {
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const unsigned cell = lane / PPC + (i * WS + ww) * (64 / PPC);
            store_split(own + (i < NP - 1 ? cell : min(cell, (unsigned)CELLS)) * STR + f32_piece(lane % PPC),
                        stg[i], cell < second_board(ps) ? ts.s0 : ts.s1);
        }
    };
    stage();
    if constexpr (HPW > 1) {
#pragma unroll
        for (int i = 0; i < NP; i++) stg[i] = xload(i, 1);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (tid < (unsigned)CW) {
        bn[0][tid] = scale;
        bn[1][tid] = -scale * mean;
    }
    unsigned arow[RBW];
#pragma unroll
    for (int i = 0; i < RBW; i++)
        arow[i] = patch_cell(ps, min((wr * RBW + i) * 16 + conv_point(lane), rows - 1 - m0)) * STR +
                  quarter_slot(lane >> 4) * 16;
    float4v acc[RBW][NBW];
#pragma unroll
    for (int i = 0; i < RBW; i++)
#pragma unroll
        for (int j = 0; j < NBW; j++) acc[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

    constexpr int AT = RBW * NBW >= 6 ? 1 : 2;   // taps read ahead
    int4v a[AT][2][RBW];   // [tap][hi, lo]
    auto aread = [&](int i, int part, int tap) {
        return *reinterpret_cast<const int4v*>(own + arow[i] + ((tap / 3) * 20 + tap % 3) * STR +
                                               part * 64);
    };
    static_assert(HPW <= 2, "chunks of a wavefront");
#pragma unroll
    for (int h = 0; h < HPW; h++) {
        if (h > 0) {
            if constexpr (WS > 1) lds_barrier();
            stage();
        }
        if constexpr (WS > 1) lds_barrier();
        if (h > 0 && (kw * HPW + h) * 2 == KW * HPW) {   // KW is odd: the middle one
#pragma unroll
            for (int i = 0; i < RBW; i++)
#pragma unroll
                for (int j = 0; j < NBW; j++) acc[i][j] = -acc[i][j];
        }
#pragma unroll
        for (int p = 0; p < 2 * AT; p++)
#pragma unroll
            for (int i = 0; i < RBW; i++) a[p / 2][p & 1][i] = aread(i, p & 1, p / 2);
#pragma unroll
        for (int sc = 0; sc < kF32Steps; sc++) {
            const int st = h * kF32Steps + sc, part = sc & 1, tap = sc / 2;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < RBW; i++) {
#pragma unroll
                for (int j = 0; j < NBW; j++)
                    if (i == (RBW >= NBW ? j : 0) && st + D - 1 < STEPS)
                        wload((st + D - 1) % D, j, st + D - 1);
#pragma unroll
                for (int j = 0; j < NBW; j++)
                    acc[i][j] = mfma(w[st % D][j], a[tap % AT][0][i], acc[i][j]);
                if (part == 0) {
#pragma unroll
                    for (int j = 0; j < NBW; j++)
                        acc[i][j] = mfma(w[st % D][j], a[tap % AT][1][i], acc[i][j]);
                }
                if (tap + AT < 9) a[tap % AT][1 - part][i] = aread(i, 1 - part, tap + AT);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }

    // partial sums through LDS: [wavefront][block][64 lanes][4]
    lds_barrier();
#pragma unroll
    for (int i = 0; i < RBW; i++)
#pragma unroll
        for (int j = 0; j < NBW; j++)
            *reinterpret_cast<float4v*>(lds + (kw * BLOCKS + (wr * RBW + i) * NB + wn * NBW + j) * 1024 + lane * 16) =
                acc[i][j];
    lds_barrier();
    float top0 = 0.0f, top1 = 0.0f;
    const int m1 = ((int)ps.mb + 1) * kPts;   // first row of the tile's second board
#pragma unroll
    for (int q = 0; q < QB; q++) {
        const int id = q * KW * WS + wave;
        if (id >= BLOCKS) continue;
        float4v part[KW];
#pragma unroll
        for (int k = 0; k < KW; k++)
            part[k] = *reinterpret_cast<const float4v*>(lds + (k * BLOCKS + id) * 1024 + lane * 16);
        const float4v r = __builtin_bit_cast(float4v, rr[q]);
        const int m = m0 + id / NB * 16 + conv_point(lane), c = id % NB * 16 + cl;
        const float unscale = m < m1 ? ts.u0 : ts.u1;
        float top = 0.0f;
        float4v o;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float v = part[0][e];
#pragma unroll
            for (int k = 1; k < KW; k++)
                v = ((k + 1) * HPW - 1) * 2 >= KW * HPW ? v - part[k][e] : v + part[k][e];
            o[e] = fmaxf(0.0f, fmaf(r[e], rfac, fmaf(v * unscale, bn[0][c + e], bn[1][c + e])));
            top = fmaxf(top, finite(o[e]));
        }
        // (Through the cache, unlike the other convolutions: tiles of 16 channels, half a cache line each, are slower
        // written through, 8 blocks of 128 filters, 1 board 92.2 -> 95.0 us, of 256 115.7 -> 117.4; those of 64 channels
        // would be 1 to 2 % faster, 22 boards of 128 filters 165.3 -> 162.2, 11 of 256 243.6 -> 240.8.)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(int4v, o), rY, ro[q], 0, 0);
        top0 = fmaxf(top0, m < m1 ? top : 0.0f);
        top1 = fmaxf(top1, m >= m1 && m < rows ? top : 0.0f);
    }
    leave_peaks<KW * WS>(red, slots, tm, tn, Kp / CW, wave, top0, top1);
}

// The tile, in blocks of 16 points and of 16 channels: the smallest that makes at most one work-group per
// unit; points 0 if none does.  The tiles of 64 channels are where conv3x3_f32_k's of the same size are
// bound by the L1 (each of its wavefronts fetches every other one's filters or planes too).  Measured
// per forward of 4 blocks, conv3x3_f32_k -> 48x64 or 64x64 here, us (one forward at a time | two side by
// side): 128 filters, 12 boards 116 -> 86 | 134 -> 105, 22: 116 -> 93 | 148 -> 126; 192 filters, 8: 140 -> 103 |
// 169 -> 147, 15: 143 -> 128 | 194 -> 199; 256 filters, 6: 175 -> 114 | 210 -> 160, 11: 176 -> 132 | 235 -> 227;
// 320 filters, 6: 201 -> 152 | 254 -> 252; 384 filters, 4: 231 -> 150 | 293 -> 222; 512 filters, 4: 293 -> 179 |
// 385 -> 320.  Left out: 64x64 above 256 filters, where the registers do not hold it (320 filters, 8
// boards 199 -> 245); 96x64 (256 filters, 16 boards 191 -> 193 | 299 -> 324).  64 filters take 32x64 for 48x32
// and 64x32: two thirds of the bytes per instruction (per forward of 10 blocks with the wavefronts below, 16
// boards 121 -> 112, 22 boards 129 -> 118).
struct SplitTile {
    int rb, nb;
};
static SplitTile f32_split_tile(int n, int Kp) {
    constexpr SplitTile kTiles[] = {{2, 1}, {3, 1}, {2, 2}, {2, 4}, {3, 2}, {4, 2}, {3, 4}, {4, 4}};
    for (const SplitTile& t : kTiles) {
        if (t.rb == 2 && t.nb == 4 ? Kp != 64 : t.rb * t.nb == 16 && Kp > 256) continue;
        if ((n * kPts + t.rb * 16 - 1) / (t.rb * 16) * (Kp / (16 * t.nb)) <= kUnits) return t;
    }
    return {0, 0};
}

bool conv3x3_f32_splits(int Kp, int max_batch) {
    return Kp % 64 == 0 && Kp <= 512 && f32_split_tile(max_batch, Kp).rb > 0;
}

PeakMap launch_conv3x3_f32_split(const float* X, const half_t* Wf, const float* res, float* Y,
                                 const float* bn_scale, const float* bn_mean, float rfac,
                                 const PeakMap& peaks, uint32_t* slots, int n, int Cp, int Kp,
                                 int lanes, hipStream_t s, LaunchTimer* t) {
    SplitTile tile = f32_split_tile(n, Kp);
    // Three forwards of 64 filters side by side have wavefronts enough: 64x64 gives way to 48x64, which a unit holds
    // four of (per forward of 8 blocks, 36 boards 67.7 -> 65.7 us, 42: 75.4 -> 72.4, 45: 79.1 -> 77.1; conv3x3_f32_k's
    // 96x64 took 66.7, 70.4 and 74.1 there), and 48x16 is not dealt (6: 38.8 -> 37.6, 8: 41.3 -> 36.4).
    if (lanes > 2 && Kp == 64 && tile.rb == 4 && tile.nb == 4) tile = {3, 4};
    if (!conv3x3_f32_splits(Kp, n) || Cp != Kp)
        throw std::invalid_argument("no split convolution for this width or batch");
    const ConvGrid g = conv_grid((n * kPts + tile.rb * 16 - 1) / (tile.rb * 16), Kp / (16 * tile.nb),
                                 (size_t)36 * Cp * Kp, (size_t)n * kPts * Cp * 4);
    peaks_fit(peaks, split_peak_loads(tile.rb, tile.nb, Kp));
    slots_fit(g.tiles_m, Kp / (16 * tile.nb), Kp, n);
    auto go = [&](auto kernel, int waves) {
        launch(kernel, dim3(8 * g.share), dim3(64 * waves), s, t, X, Wf, res, Y, bn_scale, bn_mean,
               rfac, peak_in(peaks), slots, n, Kp, g);
    };
    // KW x WR x WN wavefronts, HPW chunks each
#define LZ_TILE(RB, NB, KW, HPW, D, WR, WN) go(conv3x3_f32_split_k<RB, NB, KW, HPW, D, WR, WN>, KW * WR * WN)
#define LZ_SPLIT(KW, HPW, D)                                                                  \
    if (tile.nb == 4) {                                                                       \
        constexpr int WN = KW == 5 || KW == 6 ? 2 : 1;                                        \
        if (tile.rb == 3) LZ_TILE(3, 4, KW, HPW, (HPW == 2 ? 3 : 5), 1, WN);                  \
        else if constexpr (HPW == 1) LZ_TILE(4, 4, KW, HPW, 4, 1, WN);                        \
    } else if (tile.nb == 1) {                                                                \
        if (tile.rb == 2) LZ_TILE(2, 1, KW, HPW, D, 1, 1);                                    \
        else LZ_TILE(3, 1, KW, HPW, D, 1, 1);                                                 \
    } else if (tile.rb == 2) LZ_TILE(2, 2, KW, HPW, D, 1, 1);                                 \
    else if (tile.rb == 3) LZ_TILE(3, 2, KW, HPW, D, 1, 1);                                   \
    else LZ_TILE(4, 2, KW, HPW, (D < 18 ? 9 : D), 1, 1)
    switch (Kp) {
        case 64:
            if (tile.nb == 4) {
                if (tile.rb == 2) LZ_TILE(2, 4, 2, 1, 9, 1, 2);
                else if (tile.rb == 3) LZ_TILE(3, 4, 2, 1, 5, 1, 2);
                else LZ_TILE(4, 4, 2, 1, 4, 2, 1);
            } else if (tile.nb == 2) LZ_TILE(2, 2, 2, 1, 18, 2, 1);
            else if (tile.rb == 2) LZ_TILE(2, 1, 2, 1, 18, 2, 1);
            else if (lanes <= 2) LZ_TILE(3, 1, 2, 1, 18, 3, 1);
            else LZ_TILE(3, 1, 2, 1, 18, 1, 1);
            break;
        case 128: LZ_SPLIT(4, 1, 18); break;
        case 192: LZ_SPLIT(6, 1, 18); break;
        case 256: LZ_SPLIT(8, 1, 18); break;
        case 320: LZ_SPLIT(5, 2, 12); break;
        case 384: LZ_SPLIT(6, 2, 12); break;
        case 448: LZ_SPLIT(7, 2, 12); break;
        default: LZ_SPLIT(8, 2, 12); break;
    }
#undef LZ_SPLIT
#undef LZ_TILE
    return {slots, tile.rb * 16, Kp / (16 * tile.nb)};
}

// Two peaks a tile.  Tiles of less than 96x64 points by channels come in grids of at most three work-groups per unit; larger
// ones are fewer than those of 96x64 would be, by their area (the smallest are 128x64 and 80x128).  Every launch
// looks that its own fit (slots_fit).
size_t conv3x3_f32_slots(int Kp, int max_batch) {
    const size_t large = (size_t)(max_batch * kPts / 96 + 1) * (Kp / 64);
    return 2 * (large > 3 * kUnits ? large : 3 * kUnits);
}

// Which fp32 handles compute directly: all widths an fp32 network may have.  Measured per forward of
// 4 blocks, Winograd kernels -> this, us (one forward at a time | two side by side):
//    64 filters, 1 board 108 -> 43 | 130 -> 80, 8: 119 -> 52, 32: 173 -> 80, 64: 251 -> 83
//   128 filters, 1 board 106 -> 53 | 131 -> 85, 8: 123 -> 69, 12: 142 -> 83, 32: 198 -> 113, 64: 351 -> 184
//   192 filters, 1 board 140 -> 66, 8: 166 -> 98 | 236 -> 130, 32: 379 -> 222 | 543 -> 328, 64: 577 -> 363
//   256 filters, 1 board 164 -> 70, 8: 203 -> 116 | 312 -> 186, 32: 479 -> 300 | 783 -> 498, 64: 818 -> 503
//   384 filters, 1 board 211 -> 99, 4: 229 -> 150, 8: 353 -> 226, 32: 868 -> 625, 64: 1667 -> 1204
//   512 filters, 1 board 392 -> 116, 8: 555 -> 313, 32: 2370 -> 939, 64: 2744 -> 1749
// Relative error of the raw policy | value planes against a float64 network, 8 boards: 6x128 8.7e-7 -> 4.2e-7 |
// 6.6e-7 -> 3.2e-7 (handles of up to 11 positions 3.2e-7 | 2.4e-7), 15x192 4.4e-7 -> 2.7e-7 | 9.5e-7 ->
// 6.0e-7, 40x256 5.5e-7 -> 5.2e-7 | 2.6e-6 -> 2.2e-6, 40x64 6.5e-7 -> 4.7e-7 | 6.9e-7 -> 5.0e-7, 30x384
// 9.4e-7 -> 7.4e-7 | 1.2e-6 -> 9.7e-7, 20x512 1.9e-6 -> 1.4e-6 | 1.4e-6 -> 1.0e-6; without the change of sign
// the policy of 40x256 had 5.6e-7.
bool conv3x3_f32_serves(int Kp) { return Kp % 64 == 0 && Kp <= 512; }

// ---------------------------------------------------------------------------
// 3x3 filters from their Winograd form U = G f G^T ([36][C][F], what a pipe is handed), in double:
// f = P U P^T with P = (G^T G)^-1 G^T, the least-squares solution, so that the rounding of U is
// averaged.  Every filter is checked by transforming it forward again: *bad is set if some u is
// further from G f G^T than the rounding of a transform in single precision explains (such a U
// is no transform of a 3x3 filter, and only the Winograd kernels can compute with it); below the smallest
// normal number, 2^-126, rounding is no longer relative, and may be down to zero.
__device__ constexpr double kS2 = 1.4142135623730951;
__device__ constexpr double kGd[6][3] = {{1.0, 0.0, 0.0},
                                         {-2.0 / 3, -kS2 / 3, -1.0 / 3},
                                         {-2.0 / 3, kS2 / 3, -1.0 / 3},
                                         {1.0 / 6, kS2 / 6, 1.0 / 3},
                                         {1.0 / 6, -kS2 / 6, 1.0 / 3},
                                         {0.0, 0.0, 1.0}};
// G^T G = [[a, 0, b], [0, c, 0], [b, 0, d]]: its inverse by hand
__device__ constexpr double kGa = 1.0 + 2 * (4.0 / 9) + 2 * (1.0 / 36);
__device__ constexpr double kGb = 2 * (2.0 / 9) + 2 * (1.0 / 18);
__device__ constexpr double kGc = 2 * (2.0 / 9) + 2 * (2.0 / 36);
__device__ constexpr double kGdd = 1.0 + 2 * (1.0 / 9) + 2 * (1.0 / 9);
__device__ constexpr double kGdet = kGa * kGdd - kGb * kGb;

__device__ __forceinline__ void least_squares(const double (&u)[6], double (&f)[3]) {
    double t[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < 6; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) t[j] += kGd[i][j] * u[i];
    f[0] = (kGdd * t[0] - kGb * t[2]) / kGdet;
    f[1] = t[1] / kGc;
    f[2] = (kGa * t[2] - kGb * t[0]) / kGdet;
}
// The filter of (c, k); whether U is its transform.
__device__ __forceinline__ bool filter_3x3(const float* U, int C, int F, int c, int k,
                                           double (&f)[3][3]) {
    double half[6][3], peak = 0.0;
#pragma unroll
    for (int y = 0; y < 6; y++) {
        double u[6];
#pragma unroll
        for (int x = 0; x < 6; x++) {
            u[x] = U[((size_t)(y * 6 + x) * C + c) * F + k];
            peak = fmax(peak, fabs(u[x]));
        }
        least_squares(u, half[y]);
    }
#pragma unroll
    for (int x = 0; x < 3; x++) {
        double u[6], v[3];
#pragma unroll
        for (int y = 0; y < 6; y++) u[y] = half[y][x];
        least_squares(u, v);
#pragma unroll
        for (int y = 0; y < 3; y++) f[y][x] = v[y];
    }
    bool ok = true;
#pragma unroll
    for (int y = 0; y < 6; y++) {
        double g[3];
#pragma unroll
        for (int x = 0; x < 3; x++) g[x] = kGd[y][0] * f[0][x] + kGd[y][1] * f[1][x] + kGd[y][2] * f[2][x];
#pragma unroll
        for (int x = 0; x < 6; x++) {
            const double v = g[0] * kGd[x][0] + g[1] * kGd[x][1] + g[2] * kGd[x][2];
            ok = ok && fabs(v - U[((size_t)(y * 6 + x) * C + c) * F + k]) <= 4e-6 * peak + kFilterFloor;
        }
    }
    return ok;
}

// Binary exponents of an output channel's largest filter (times 2^-in_exp of its input channel) and of
// its largest product with an input channel of magnitude 2^mag; both kNoExp before.  (Maxima of
// integers: the same whatever the order.)
__global__ __launch_bounds__(256) void filters_f32_peak_k(const float* __restrict__ U,
                                                          const int* __restrict__ in_exp,
                                                          const int* __restrict__ mag, int C, int F,
                                                          int* __restrict__ peak,
                                                          int* __restrict__ reach,
                                                          int* __restrict__ bad) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= C * F) return;
    const int c = i / F, k = i - c * F;
    double f[3][3];
    if (!filter_3x3(U, C, F, c, k, f)) *bad = 1;
    double top = 0.0;
#pragma unroll
    for (int tap = 0; tap < 9; tap++) top = fmax(top, fabs(f[tap / 3][tap % 3]));
    if (!((float)top < __builtin_inff())) {
        *bad = 1;
        return;
    }
    if (!(top > 0.0)) return;
    const int e = ilogb(top);
    atomicMax(peak + k, e - in_exp[c]);
    if (mag[c] != kNoExp) atomicMax(reach + k, e + mag[c]);
}

__global__ __launch_bounds__(256) void filters_f32_k(const float* __restrict__ U,
                                                     const int* __restrict__ in_exp,
                                                     const int* __restrict__ exp,
                                                     half_t* __restrict__ Wf, int C, int Cp, int F,
                                                     int Kp) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= C * F) return;
    const int c = i / F, k = i - c * F;
    double f[3][3];
    filter_3x3(U, C, F, c, k, f);
    const double scale = ldexp(conv3x3_f32_negated(c, Cp) ? -1.0 : 1.0, exp[k] - in_exp[c]);
#pragma unroll
    for (int tap = 0; tap < 9; tap++) {
        const double v = f[tap / 3][tap % 3] * scale;
        const half_t hi = (half_t)(float)v;
        Wf[conv3x3_f32_index(k, c, tap, 0, Kp)] = hi;
        Wf[conv3x3_f32_index(k, c, tap, 1, Kp)] = (half_t)(float)(v - (double)(float)hi);
    }
}

void conv3x3_f32_peaks(const float* U, const int* in_exp, const int* mag, int C, int F, int* peak,
                       int* reach, int* bad, hipStream_t s) {
    hipLaunchKernelGGL(filters_f32_peak_k, dim3((unsigned)((C * F + 255) / 256)), dim3(256), 0, s, U,
                       in_exp, mag, C, F, peak, reach, bad);
}

void conv3x3_f32_filters(const float* U, const int* in_exp, const int* exp, half_t* Wf, int C, int Cp,
                         int F, int Kp, hipStream_t s) {
    hipLaunchKernelGGL(filters_f32_k, dim3((unsigned)((C * F + 255) / 256)), dim3(256), 0, s, U, in_exp,
                       exp, Wf, C, Cp, F, Kp);
}

// Where the halves lose what fp32 holds.  The lo half of a plane is exact to 2^-40 of the board's largest
// value, that of a filter to 2^-36 of its output channel's largest.  If the largest product of an
// output channel is at least 2^-14 of its largest filter times the largest input channel, either
// error stays below 2^-22 of that product, as it is with operands of the full 22 bits.
bool conv3x3_f32_holds(int peak, int reach, int top, int most) {
    return peak == kNoExp || top == kNoExp || reach >= peak + top - most;
}

// The exponent of an output channel's filters: their largest comes to kFilterTop, or as far towards it as
// the batch norm's numbers can take in (scale * 2^(out_exp - e), mean * 2^e).  They are the limit where
// filters have decayed to nothing: by then the convolution is less than 2^-100 of the mean, or of
// what channels of the same exponent hold.  False: no exponent does.
bool conv3x3_f32_exponent(int peak, float scale, float mean, int out_exp, int& e) {
    e = peak == kNoExp ? 0 : kFilterTop - peak;
    if (std::isfinite(mean) && mean != 0.0f) e = std::min(e, 126 - std::ilogb(mean));
    if (!std::isfinite(scale) || scale == 0.0f) return true;
    const int s = std::ilogb(scale) + out_exp;
    e = std::min(e, s + 126);
    return s - e <= 126;
}

void conv3x3_f32_winograd_filters(const half_t* Wf, const int* in_exp, const int* exp, int C, int Cp,
                                  int F, int Kp, float* U) {
    const double s2 = std::sqrt(2.0);
    const double G[6][3] = {{1, 0, 0},
                            {-2.0 / 3, -s2 / 3, -1.0 / 3},
                            {-2.0 / 3, s2 / 3, -1.0 / 3},
                            {1.0 / 6, s2 / 6, 1.0 / 3},
                            {1.0 / 6, -s2 / 6, 1.0 / 3},
                            {0, 0, 1}};
    for (int k = 0; k < F; k++) {
        for (int c = 0; c < C; c++) {
            const double unscale =
                std::ldexp(conv3x3_f32_negated(c, Cp) ? -1.0 : 1.0, in_exp[c] - exp[k]);
            double f[9];
            for (int tap = 0; tap < 9; tap++)
                f[tap] = unscale * ((double)Wf[conv3x3_f32_index(k, c, tap, 0, Kp)] +
                                    (double)Wf[conv3x3_f32_index(k, c, tap, 1, Kp)]);
            for (int p = 0; p < kPos; p++) {
                double v = 0.0;
                for (int tap = 0; tap < 9; tap++) v += G[p / 6][tap / 3] * G[p % 6][tap % 3] * f[tap];
                U[((size_t)p * Kp + k) * Cp + c] = (float)v;
            }
        }
    }
}

}  // namespace lzhip
