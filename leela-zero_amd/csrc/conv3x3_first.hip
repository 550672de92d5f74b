// The first layer of a direct fp16 tower from planes as floats, for small batches: what launch_pack_input and
// launch_conv3x3 do in two launches, in one.
#include <stdexcept>

#include "conv3x3_tile.h"
#include "kernel_util.h"

namespace lzhip {

namespace {

constexpr int kMt = 32, kCells = conv_cells(kMt);   // points of a tile, cells of its patch
constexpr int kThreads = 256, kCols = 64;           // output channels of a tile
constexpr int kPitch = 80;                          // bytes of a cell in LDS: 32 channels, 16 more
constexpr int kQuads = (kInPlanes + 3) / 4;
constexpr int kPieces = (kCells * kQuads + kThreads - 1) / kThreads;   // of four channels of a cell, a thread's

// One work-group computes 32 points x 64 channels, each wavefront 16 of them, over the nine taps of 32 input
// channels; the filters' second chunk of 32 meets nothing but zeros and is left out.  Its sums, and so
// its bits, are conv3x3_k's.
//
// What bounds it is a round trip for the planes and one for the filters, requested together, and for small
// batches the launch: without the planes in between one of 23 launches of 10 blocks is gone, and a pass over
// the planes.  All channels in one work-group, which fetches the planes once, took 1 us more at 256 filters: a
// unit waits for 147 KB of filters.  Packed bits in host memory stay with pack_input_bits_k: fetched over
// the bus by every tile they took as long as the launch that this saves (6x128 fp32, 1 board 90 -> 92
// us; 15x192 fp16, 8 boards 206 -> 208), and so do fp32 planes, whose peaks have to be known first.
__global__ __launch_bounds__(kThreads) void conv3x3_first_k(
    const float* __restrict__ planes, const half_t* __restrict__ Wf, half_t* __restrict__ Y,
    const float* __restrict__ bn_scale, const float* __restrict__ bn_mean, int n, int Cp, int Kp,
    PlaneBorders borders, unsigned pieces) {
    typedef half_t half4v __attribute__((ext_vector_type(4)));
    __shared__ __attribute__((aligned(16))) unsigned char lds[kCells * kPitch];

    if (blockIdx.y * kCols >= (unsigned)Kp) {   // (behind the tiles: borders)
        for (unsigned i = blockIdx.x * kThreads + threadIdx.x; i < pieces; i += gridDim.x * kThreads)
            clear_border(borders, i);
        return;
    }
    const int rows = n * kPts, m0 = blockIdx.x * kMt;
    const unsigned tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const PatchStart ps = patch_start(m0);

    // piece i: channels 4 (i / kCells) to + 3 of cell i % kCells; zero where the cell is a border
    const __amdgpu_buffer_rsrc_t rP = make_rsrc(planes, (size_t)n * kInPlanes * kPts * 4);
    float x[kPieces][4];
#pragma unroll
    for (int p = 0; p < kPieces; p++) {
        const unsigned i = tid + p * kThreads, c0 = i / kCells * 4, q = ps.q0 + i % kCells;
        const unsigned b = q / kCellsPerBoard, r = q - b * kCellsPerBoard, y = r / kRowCells, c = r - y * kRowCells;
        const bool point = b >= 1 && (int)b <= n && y >= 1 && c < kBoard;
        const unsigned at = (((b - 1) * kInPlanes + c0) * kPts + (y - 1) * kBoard + c) * 4u;
#pragma unroll
        for (int e = 0; e < 4; e++)
            x[p][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                rP, point && c0 + e < kInPlanes ? at + e * kPts * 4u : 0xfffffff0u, 0, 0));
    }
    const int kb = (int)blockIdx.y * (kCols / 16) + wave;   // block of 16 output channels
    const __amdgpu_buffer_rsrc_t rW = make_rsrc(Wf, (size_t)9 * Cp * Kp * 2);
    int4v w[9];   // (k-steps of channels 0 to 31; those of 32 to 63 lie between)
#pragma unroll
    for (int tap = 0; tap < 9; tap++)
        w[tap] = __builtin_amdgcn_raw_buffer_load_b128(rW, lane * 16u + kb * 1024u,
                                                       2 * tap * (unsigned)Kp * 64u, 0);
    const int ch0 = (kb >> 1) * 32 + 8 * (int)(lane >> 4) + 4 * (kb & 1);   // this lane's four channels
    const float4v scale = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(
                                                          make_rsrc(bn_scale, Kp * 4), ch0 * 4u, 0, 0));
    const float4v mean = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(
                                                         make_rsrc(bn_mean, Kp * 4), ch0 * 4u, 0, 0));
    __builtin_amdgcn_sched_barrier(0);

    for (unsigned i = tid; i < kCells * 3; i += kThreads)   // channels 20 to 31
        *reinterpret_cast<half4v*>(lds + i / 3 * kPitch + 40 + i % 3 * 8) = half4v{};
#pragma unroll
    for (int p = 0; p < kPieces; p++) {
        const unsigned i = tid + p * kThreads;
        half4v v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = (half_t)fminf(fmaxf(x[p][e], -65504.0f), 65504.0f);
        if (i < kCells * kQuads)
            *reinterpret_cast<half4v*>(lds + i % kCells * kPitch + i / kCells * 8) = v;
    }
    unsigned arow[2], ro[2];   // LDS address of this lane's point, tap (0, 0); byte offset of its result
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int local = i * 16 + (int)(lane & 15);
        const unsigned cell = patch_cell(ps, min(local, rows - 1 - m0));
        arow[i] = cell * kPitch + (lane >> 4) * 16;
        ro[i] = m0 + local < rows ? ((ps.q0 + kPointCell + cell) * Kp + ch0) * 2u : 0xfffff000u;
    }
    float4v acc[2] = {};
    lds_barrier();
#pragma unroll
    for (int tap = 0; tap < 9; tap++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int4v a = *reinterpret_cast<const int4v*>(lds + arow[i] +
                                                            (tap / 3 * kRowCells + tap % 3) * kPitch);
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8v, w[tap]),
                                                            __builtin_bit_cast(half8v, a), acc[i], 0, 0, 0);
        }

    const __amdgpu_buffer_rsrc_t rY = make_rsrc(Y, (size_t)(n + 2) * kCellsPerBoard * Kp * 2);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        half4v o;
#pragma unroll
        for (int e = 0; e < 4; e++)
            o[e] = (half_t)fminf(fmaxf(0.0f, fmaf(acc[i][e], scale[e], -scale[e] * mean[e])), kActStoreMax);
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2v, o), rY, ro[i], 0, kStoreThrough);
    }
}

}  // namespace

// Measured per forward of 10 blocks, us, two launches -> this one: 64 filters, 1 board 79 -> 76, 16: 80.3 -> 77.6; 128
// filters, 1: 73 -> 70, 5: 78.4 -> 75.9, 8: 96.4 -> 94.0, 16: 108.2 -> 105.8; 192 filters, 1: 100.5 -> 97.6, 8: 124.8 ->
// 122.4, 16: 158.5 -> 156.4; 256 filters, 4: 127.6 -> 123.0, 8: 144.5 -> 141.6, 16: 198.0 -> 195.7 (two versions one after
// the other; timed in turn, 128 filters at 5 boards is 82.0 -> 81.3, within the spread).
// What is saved is a launch, and what it costs grows with the batch: a tile of 32 points fetches the planes and the filters
// that launch_conv3x3's share among up to 192 points.  So 256 filters lose from 64 boards on (8 blocks, 367.7 -> 371.3;
// 128: 672.9 -> 680.4).  The line lies where every width was still measured to gain; between it and that loss a
// forward alone would gain 2 to 4 us more (64 filters, 64 boards 89.6 -> 86.6; 128, 64: 143.6 -> 141.3; 192, 64: 276.0 ->
// 273.0; 256, 32: 213.9 -> 211.4) or nothing (384, 17: 248.9 -> 248.3, 44: 516.0 -> 517.8).
bool conv3x3_first_serves(int Kp, int n) { return Kp % kCols == 0 && n <= 16; }

void launch_conv3x3_first(const float* planes, const half_t* Wf, half_t* Y, const float* bn_scale,
                          const float* bn_mean, int n, int Cp, int Kp, hipStream_t s,
                          const PlaneBorders* borders) {
    if (!conv3x3_first_serves(Kp, n) || Cp != 64) throw std::invalid_argument("no first layer for this width or batch");
    hipLaunchKernelGGL(conv3x3_first_k, dim3((n * kPts + kMt - 1) / kMt, Kp / kCols + (borders ? 1 : 0)),
                       dim3(kThreads), 0, s, planes, Wf, Y, bn_scale, bn_mean, n, Cp, Kp,
                       borders ? *borders : PlaneBorders(), border_pieces(borders));
}

}  // namespace lzhip
