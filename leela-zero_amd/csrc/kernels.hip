// gfx950 (CDNA4) kernels of the Winograd F(4x4,3x3) residual tower.
//
// Arithmetic follows the reference CPU pipe (reference src/CPUPipe.cpp:63-284,
// :352-377) and its OpenCL twins (src/kernels/convolve3.opencl:47-79); the
// decomposition, layouts and launch shapes are this library's own.
#include <cstdlib>
#include <stdexcept>
#include <type_traits>

#include "kernel_util.h"

namespace lzhip {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float8v __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));

#define SQ2 1.4142135623730951f
// ---------------------------------------------------------------------------
// Per-lane channel vector: how many consecutive channels one lane owns in the
// bandwidth-bound kernels (4 bytes per lane and access for both types).
template <typename P> struct ChanVec;
template <> struct ChanVec<float> {
    static constexpr int N = 1;
    static __device__ __forceinline__ void load(const float* p, float* o) { o[0] = *p; }
    static __device__ __forceinline__ void store(float* p, const float* v) { *p = v[0]; }
};
template <> struct ChanVec<half_t> {
    static constexpr int N = 2;
    static __device__ __forceinline__ void load(const half_t* p, float* o) {
        const half2v h = *reinterpret_cast<const half2v*>(p);
        o[0] = (float)h.x;
        o[1] = (float)h.y;
    }
    // Saturating: a value beyond the fp16 range is stored as +-65504, not inf.
    static __device__ __forceinline__ void store(half_t* p, const float* v) {
        half2v h;
        h.x = (half_t)fminf(fmaxf(v[0], -65504.0f), 65504.0f);
        h.y = (half_t)fminf(fmaxf(v[1], -65504.0f), 65504.0f);
        *reinterpret_cast<half2v*>(p) = h;
    }
};

template <typename P> __device__ __forceinline__ P to_storage(float v);
// Four consecutive storage elements as one LDS/global access.
template <typename P> struct Quad;
template <> struct Quad<float> { typedef float type __attribute__((ext_vector_type(4))); };
template <> struct Quad<_Float16> { typedef _Float16 type __attribute__((ext_vector_type(4))); };

template <> __device__ __forceinline__ float to_storage<float>(float v) { return v; }
template <> __device__ __forceinline__ half_t to_storage<half_t>(float v) {
    return (half_t)fminf(fmaxf(v, -65504.0f), 65504.0f);
}

// Stored activations are kept at or below kActStoreMax = 2040 < 65504 / 30.6 (30.6 = largest
// absolute row sum of B^T (x) B^T), so the input transform of a stored activation cannot
// leave the half-precision range and V needs no clamp of its own.  Every kernel that
// stores an activation (fused and unfused output transform) goes through this one clamp,
// and the activation-scale calibration measures through it.
template <typename P> __device__ __forceinline__ float act_clamp(float v);
template <> __device__ __forceinline__ float act_clamp<float>(float v) { return v; }
template <> __device__ __forceinline__ float act_clamp<half_t>(float v) {
    return fminf(v, kActStoreMax);
}
template <typename P> __device__ __forceinline__ P act_to_storage(float v) {
    return (P)act_clamp<P>(v);
}

// o = B^T i for one 6-vector (reference src/CPUPipe.cpp:88-106).
__device__ __forceinline__ void bt6(const float i0, const float i1, const float i2,
                                    const float i3, const float i4, const float i5, float& o0,
                                    float& o1, float& o2, float& o3, float& o4, float& o5) {
    const float a = i1 * -SQ2 + i3 * (SQ2 / 2.0f);
    const float b = i2 * -2.0f + i4;
    o0 = i0 + i2 * (-5.0f / 2.0f) + i4;
    o1 = a + b;
    o2 = -a + b;
    const float c = i3 * SQ2 + i1 * (-SQ2 / 2.0f);
    const float d = i2 * (-1.0f / 2.0f) + i4;
    o3 = c + d;
    o4 = -c + d;
    o5 = i1 + i3 * (-5.0f / 2.0f) + i5;
}

// o = A^T i for one 6-vector (reference src/CPUPipe.cpp:225-238; the same sums,
// associated so that they take twelve operations).
__device__ __forceinline__ void at6(const float i0, const float i1, const float i2,
                                    const float i3, const float i4, const float i5, float& o0,
                                    float& o1, float& o2, float& o3) {
    const float s12 = i1 + i2, d12 = i1 - i2;
    const float s34 = i3 + i4, d34 = i3 - i4;
    o0 = (i0 + s12) + s34;
    o1 = fmaf(d34, SQ2, d12 * (SQ2 / 2.0f));
    o2 = fmaf(s34, 2.0f, s12 * 0.5f);
    o3 = fmaf(d34, 2.0f * SQ2, fmaf(d12, SQ2 / 4.0f, i5));
}

// ---------------------------------------------------------------------------
// ---------------------------------------------------------------------------
// Planes NCHW fp32 [n][C][361] -> channels-last storage type [n][361][Cp],
// channels C..Cp-1 zero.  A thread takes one point and every fourth group of eight channels of
// it: the reads of sixteen points are 64 bytes of a plane, the writes of four threads 64 or 128
// bytes of a point.  (With a value per thread, channels first, 64 lanes read 64 planes: 200 boards
// took 13 us, now 6, and from packed planes in host memory, each word fetched by many, 28, now 9;
// 37 boards 8.2 and 5.3; one board takes the 4 us of a trip across the bus either way.)
constexpr int kPackThreads = 4 * kPts;   // of a board
template <typename P, typename Value>
__device__ __forceinline__ void pack_point(P* __restrict__ cell, int g, int C, int Cp,
                                           Value value) {
    typedef P P8 __attribute__((ext_vector_type(8)));
    for (int c0 = g * 8; c0 < Cp; c0 += 32) {
        P8 v = {};
        if (c0 < C) {   // (read past C without a branch to each, so that all eight are in flight)
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = value(min(c0 + e, C - 1));
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = c0 + e < C ? to_storage<P>(x[e]) : (P)0.0f;
        }
        *reinterpret_cast<P8*>(cell + c0) = v;
    }
}

// (work-groups from pack_groups on clear borders)
template <typename P>
__global__ __launch_bounds__(256) void pack_input_k(const float* __restrict__ in,
                                                    P* __restrict__ act, bool padded, int n, int C,
                                                    int Cp, unsigned pack_groups,
                                                    PlaneBorders borders) {
    if (blockIdx.x >= pack_groups) {
        clear_border(borders, (blockIdx.x - pack_groups) * 256 + threadIdx.x);
        return;
    }
    const size_t gid = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (gid >= (size_t)n * kPackThreads) return;
    const int b = (int)(gid / kPackThreads), i = (int)(gid % kPackThreads), pt = i >> 2;
    const float* planes = in + (size_t)b * C * kPts + pt;
    pack_point(act + plane_index(padded, b, pt) * Cp, i & 3, C, Cp,
               [&](int c) { return planes[(size_t)c * kPts]; });
}

template <typename P>
void launch_pack_input(const float* in, P* act, bool padded, int n, int C, int Cp, hipStream_t s,
                       LaunchTimer* t, const PlaneBorders* borders) {
    const unsigned groups = (unsigned)(((size_t)n * kPackThreads + 255) / 256);
    launch(pack_input_k<P>, dim3(groups + (border_pieces(borders) + 255) / 256), dim3(256), s, t, in,
           act, padded, n, C, Cp, groups, borders ? *borders : PlaneBorders());
}

// The same from bit-packed planes: bit (c*361 + pt) of a board's kInputWords words is
// plane c at point pt (planes that hold only 0 and 1, which is what the engine feeds).  The
// words may lie in host memory, across the bus: a work-group fetches its board's once, in one
// load, and there are three of them to a board.
template <typename P, bool SCALED>
__global__ __launch_bounds__(512) void pack_input_bits_k(const uint32_t* __restrict__ bits,
                                                         P* __restrict__ act, bool padded, int C,
                                                         int Cp, uint32_t* __restrict__ peaks,
                                                         const float* __restrict__ scale) {
    __shared__ uint32_t words[kInputWords];
    const int b = blockIdx.x, i = blockIdx.y * 512 + threadIdx.x, pt = i >> 2;
    if (threadIdx.x < kInputWords)
        words[threadIdx.x] = bits[(size_t)b * kInputWords + threadIdx.x];
    if (!SCALED && peaks && i < 2) peaks[2 * (size_t)b + i] = 0x3f800000u;
    __syncthreads();
    if (SCALED && peaks && blockIdx.y == 0 && threadIdx.x < 64) {
        // the largest factor of a plane that is not empty, as the float planes' peak would be
        const int c = threadIdx.x, from = c * kPts, to = from + kPts;
        float top = 0.0f;
        for (int w = from >> 5; c < C && w <= (to - 1) >> 5; w++) {
            const int lo = max(from - w * 32, 0), hi = min(to - w * 32, 32);   // bits [lo, hi) are c's
            if (words[w] >> lo & (hi - lo == 32 ? ~0u : (1u << (hi - lo)) - 1u)) top = scale[c];
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) top = fmaxf(top, __shfl_xor(top, off));
        if (c < 2) peaks[2 * (size_t)b + c] = __builtin_bit_cast(uint32_t, top);
    }
    if (pt >= kPts) return;
    pack_point(act + plane_index(padded, b, pt) * Cp, i & 3, C, Cp, [&](int c) {
        const int bit = c * kPts + pt;
        const float v = (float)((words[bit >> 5] >> (bit & 31)) & 1u);
        return SCALED ? v * scale[c] : v;
    });
}

// (A kernel of its own for planes with factors: the test of the pointer at every value cost 37 boards
// of 128 filters 4 us a call.)
template <typename P>
void launch_pack_input_bits(const uint32_t* bits, P* act, bool padded, int n, int C, int Cp,
                            uint32_t* peaks, const float* scale, hipStream_t s, LaunchTimer* t) {
    launch(scale ? pack_input_bits_k<P, true> : pack_input_bits_k<P, false>,
           dim3(n, (kPackThreads + 511) / 512), dim3(512), s, t, bits, act, padded, C, Cp, peaks, scale);
}

// Planes and peaks from float planes: the first work-group of a board packs nothing and reads all
// of it (26 KB); three pack; those beyond clear borders.
constexpr int kPeakGroups = 1 + (kPackThreads + 511) / 512;   // of a board
template <bool SCALED>
__global__ __launch_bounds__(512) void pack_input_peaks_k(const float* __restrict__ in,
                                                          float* __restrict__ act, int C, int Cp,
                                                          uint32_t* __restrict__ peaks,
                                                          const float* __restrict__ scale,
                                                          PlaneBorders borders) {
    const int b = blockIdx.x, tid = threadIdx.x;
    if (blockIdx.y >= kPeakGroups) {
        clear_border(borders, ((blockIdx.y - kPeakGroups) * gridDim.x + b) * 512 + tid);
        return;
    }
    const float* planes = in + (size_t)b * C * kPts;
    if (blockIdx.y > 0) {
        const int i = (blockIdx.y - 1) * 512 + tid, pt = i >> 2;
        if (pt < kPts)
            pack_point(act + plane_index(true, b, pt) * Cp, i & 3, C, Cp,
                       [&](int c) {
                           const float v = planes[(size_t)c * kPts + pt];
                           return SCALED ? v * scale[c] : v;
                       });
        return;
    }
    float top = 0.0f;
#pragma unroll 13
    for (int i = tid; i < C * kPts; i += 512) {
        const float v = fabsf(SCALED ? planes[i] * scale[i / kPts] : planes[i]);
        top = fmaxf(top, v < __builtin_inff() ? v : 0.0f);
    }
    __shared__ float tops[8];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) top = fmaxf(top, __shfl_xor(top, off));
    if ((tid & 63) == 0) tops[tid >> 6] = top;
    __syncthreads();
    if (tid == 0) {
        for (int i = 1; i < 8; i++) top = fmaxf(top, tops[i]);
        peaks[2 * b] = __builtin_bit_cast(uint32_t, top);
    }
}

void launch_pack_input_peaks(const float* in, float* act, int n, int C, int Cp, uint32_t* peaks,
                             const float* scale, hipStream_t s, LaunchTimer* t,
                             const PlaneBorders* borders) {
    launch(scale ? pack_input_peaks_k<true> : pack_input_peaks_k<false>,
           dim3(n, kPeakGroups + (border_pieces(borders) + 512 * n - 1) / (512 * n)),
           dim3(512), s, t, in, act, C, Cp, peaks, scale, borders ? *borders : PlaneBorders());
}

// ---------------------------------------------------------------------------
// Winograd input transform V = B^T d B (reference src/CPUPipe.cpp:63-183).
// One lane owns one tile and ChanVec<P>::N consecutive channels; consecutive
// lanes own consecutive channels, so every load and store of a wave covers a
// contiguous run of the channels-last arrays.  The 6x6 patch starts one point
// above/left of board point (4by, 4bx); points off the board read as zero.
// (At most four wavefronts per SIMD are asked for: aiming at eight, the compiler keeps the
// kernel within 64 registers by waiting for each of the 36 loads before it issues the next.)
template <typename P>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 4))) void in_transform_k(const P* __restrict__ act,
                                                      P* __restrict__ V, int T, int Cp,
                                                      int Tp) {
    constexpr int VN = ChanVec<P>::N;
    const int lpt = Cp / VN;  // lanes per tile
    const int gid = blockIdx.x * 256 + threadIdx.x;
    const int t = gid / lpt;
    if (t >= T) return;
    const int c = (gid - t * lpt) * VN;
    const int b = t / kTilesPerBoard;
    const int j = t - b * kTilesPerBoard;
    const int by = j / 5, bx = j - by * 5;
    const int y0 = 4 * by - 1, x0 = 4 * bx - 1;
    const P* base = act + (size_t)b * kPts * Cp + c;

    float d[VN][36];
#pragma unroll
    for (int yy = 0; yy < 6; yy++) {
#pragma unroll
        for (int xx = 0; xx < 6; xx++) {
            const int y = y0 + yy, x = x0 + xx;
            // clamped address + select instead of a branch: all 36 loads stay in flight
            const bool inb = (unsigned)y < (unsigned)kBoard && (unsigned)x < (unsigned)kBoard;
            const int pt = inb ? y * kBoard + x : 0;
            float tmp[VN];
            ChanVec<P>::load(base + (size_t)pt * Cp, tmp);
#pragma unroll
            for (int v = 0; v < VN; v++) d[v][yy * 6 + xx] = inb ? tmp[v] : 0.0f;
        }
    }
#pragma unroll
    for (int v = 0; v < VN; v++) {
        float t1[36];
#pragma unroll
        for (int xx = 0; xx < 6; xx++)  // columns: along y
            bt6(d[v][0 + xx], d[v][6 + xx], d[v][12 + xx], d[v][18 + xx], d[v][24 + xx],
                d[v][30 + xx], t1[0 + xx], t1[6 + xx], t1[12 + xx], t1[18 + xx], t1[24 + xx],
                t1[30 + xx]);
#pragma unroll
        for (int yy = 0; yy < 6; yy++)  // rows: along x
            bt6(t1[yy * 6 + 0], t1[yy * 6 + 1], t1[yy * 6 + 2], t1[yy * 6 + 3], t1[yy * 6 + 4],
                t1[yy * 6 + 5], d[v][yy * 6 + 0], d[v][yy * 6 + 1], d[v][yy * 6 + 2],
                d[v][yy * 6 + 3], d[v][yy * 6 + 4], d[v][yy * 6 + 5]);
    }
    P* vout = V + (size_t)t * Cp + c;
    const size_t pstride = (size_t)Tp * Cp;
#pragma unroll
    for (int p = 0; p < 36; p++) {
        float tmp[VN];
#pragma unroll
        for (int v = 0; v < VN; v++) tmp[v] = d[v][p];
        ChanVec<P>::store(vout + p * pstride, tmp);
    }
}

template <typename P>
void launch_in_transform(const P* act, P* V, int n, int Cp, int Tp, hipStream_t s,
                         LaunchTimer* t) {
    const int T = n * kTilesPerBoard;
    const int lanes = T * (Cp / ChanVec<P>::N);
    launch(in_transform_k<P>, dim3((lanes + 255) / 256), dim3(256), s, t, act, V, T, Cp, Tp);
}

// ---------------------------------------------------------------------------
// Output transform Y = A^T m A fused with batch-norm scale/shift, residual add
// and ReLU (reference src/CPUPipe.cpp:212-284 + :352-377; the reference GPU
// path fuses the same way, src/kernels/convolve3.opencl:218-318).
// out = max(0, scale*(y - mean) + rfac*res); rfac carries the ratio of the
// activation scales of the skip connection and of this layer (1 in fp32).
template <typename P>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 3))) void out_transform_k(
    const P* __restrict__ M, const P* __restrict__ res, P* __restrict__ out,
    const float* __restrict__ bn_scale, const float* __restrict__ bn_mean, float rfac, int T,
    int Kp, int Tp) {
    constexpr int VN = ChanVec<P>::N;
    const int lpt = Kp / VN;
    const int gid = blockIdx.x * 256 + threadIdx.x;
    const int t = gid / lpt;
    if (t >= T) return;
    const int c = (gid - t * lpt) * VN;
    const int b = t / kTilesPerBoard;
    const int j = t - b * kTilesPerBoard;
    const int by = j / 5, bx = j - by * 5;

    float m[VN][36];
    const P* msrc = M + (size_t)t * Kp + c;
    const size_t pstride = (size_t)Tp * Kp;
#pragma unroll
    for (int p = 0; p < 36; p++) {
        float tmp[VN];
        ChanVec<P>::load(msrc + p * pstride, tmp);
#pragma unroll
        for (int v = 0; v < VN; v++) m[v][p] = tmp[v];
    }
    float o[VN][16];
#pragma unroll
    for (int v = 0; v < VN; v++) {
        float t1[24];  // [4][6]
#pragma unroll
        for (int xx = 0; xx < 6; xx++)
            at6(m[v][0 + xx], m[v][6 + xx], m[v][12 + xx], m[v][18 + xx], m[v][24 + xx],
                m[v][30 + xx], t1[0 + xx], t1[6 + xx], t1[12 + xx], t1[18 + xx]);
#pragma unroll
        for (int i = 0; i < 4; i++)
            at6(t1[i * 6 + 0], t1[i * 6 + 1], t1[i * 6 + 2], t1[i * 6 + 3], t1[i * 6 + 4],
                t1[i * 6 + 5], o[v][i * 4 + 0], o[v][i * 4 + 1], o[v][i * 4 + 2],
                o[v][i * 4 + 3]);
    }
    float sc[VN], mn[VN];
#pragma unroll
    for (int v = 0; v < VN; v++) {
        sc[v] = bn_scale[c + v];
        mn[v] = bn_mean[c + v];
    }
    const size_t bbase = (size_t)b * kPts * Kp + c;
    const __amdgpu_buffer_rsrc_t rO =
        make_rsrc(out, (size_t)((T + kTilesPerBoard - 1) / kTilesPerBoard) * kPts * Kp * sizeof(P));
    float r[VN][16];
    if (res != nullptr) {  // uniform; clamped addresses keep the 16 loads free of branches
#pragma unroll
        for (int i = 0; i < 4; i++) {
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
                const int y = min(4 * by + i, kBoard - 1), x = min(4 * bx + jj, kBoard - 1);
                float tmp[VN];
                ChanVec<P>::load(res + bbase + (size_t)(y * kBoard + x) * Kp, tmp);
#pragma unroll
                for (int v = 0; v < VN; v++) r[v][i * 4 + jj] = tmp[v];
            }
        }
    } else {
#pragma unroll
        for (int v = 0; v < VN; v++)
#pragma unroll
            for (int q = 0; q < 16; q++) r[v][q] = 0.0f;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
            const int y = 4 * by + i, x = 4 * bx + jj;
            float val[VN];
#pragma unroll
            for (int v = 0; v < VN; v++)
                val[v] = act_clamp<P>(
                    fmaxf(0.0f, sc[v] * (o[v][i * 4 + jj] - mn[v]) + rfac * r[v][i * 4 + jj]));
            // Unconditional store through a buffer descriptor: points off the board get an
            // offset outside it and are dropped by the hardware (a branch around each store
            // makes the compiler wait for the store before it).
            const unsigned off = (y < kBoard && x < kBoard)
                                     ? (unsigned)((bbase + (size_t)(y * kBoard + x) * Kp) * sizeof(P))
                                     : 0xfffffff0u;
            if constexpr (sizeof(P) == 4) {
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, val[0]), rO, off,
                                                      0, 0);
            } else {
                half2v h;
                h.x = (half_t)fminf(fmaxf(val[0], -65504.0f), 65504.0f);
                h.y = (half_t)fminf(fmaxf(val[1], -65504.0f), 65504.0f);
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, h), rO, off, 0,
                                                      0);
            }
        }
    }
}

template <typename P>
void launch_out_transform(const P* M, const P* res, P* out, const float* bn_scale,
                          const float* bn_mean, float rfac, int n, int Kp, int Tp,
                          hipStream_t s, LaunchTimer* t) {
    const int T = n * kTilesPerBoard;
    const int lanes = T * (Kp / ChanVec<P>::N);
    launch(out_transform_k<P>, dim3((lanes + 255) / 256), dim3(256), s, t, M, res, out,
           bn_scale, bn_mean, rfac, T, Kp, Tp);
}

// ---------------------------------------------------------------------------
// Output transform of layer l fused with the input transform of layer l+1
// (the reference fuses the same pair for batch 1 only,
// src/kernels/convolve3.opencl:320-452).  Phase 1 turns the 25 M tiles of a
// board into the 19x19 activation plane (BN, residual, ReLU, rounded to the
// storage type exactly as the unfused kernel stores it) and keeps it in LDS;
// phase 2 reads the 6x6 patches back from LDS and writes the next layer's V.
// The activation itself goes to memory only when a later layer needs it as a
// skip connection.
//
// Raw buffer access: address = buffer base + scalar byte offset + per-lane byte
// offset.  Everything that selects a board, a tile pair or a Winograd position
// is wavefront-uniform and lives in the scalar offset, stepped with scalar
// adds; the per-lane offset never changes, so the global accesses need no
// vector address arithmetic, and accesses past the end of a buffer are benign.
template <typename P> struct BufIO;
template <> struct BufIO<float> {
    static __device__ __forceinline__ float load(__amdgpu_buffer_rsrc_t r, unsigned voff,
                                                 unsigned soff) {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
    }
    static __device__ __forceinline__ void store(float v, __amdgpu_buffer_rsrc_t r, unsigned voff,
                                                 unsigned soff) {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, voff, soff, 0);
    }
};
template <> struct BufIO<half_t> {
    static __device__ __forceinline__ half_t load(__amdgpu_buffer_rsrc_t r, unsigned voff,
                                                  unsigned soff) {
        return __builtin_bit_cast(half_t, __builtin_amdgcn_raw_buffer_load_b16(r, voff, soff, 0));
    }
    static __device__ __forceinline__ void store(half_t v, __amdgpu_buffer_rsrc_t r, unsigned voff,
                                                 unsigned soff) {
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), r, voff, soff,
                                              0);
    }
};
// Two consecutive channels per access (4 bytes in fp16, 8 in fp32).
template <typename P> struct BufIO2;
template <> struct BufIO2<float> {
    typedef float pair_t __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, unsigned voff,
                                                unsigned soff, float& a, float& b) {
        // two 4-byte loads: this compiler lowers the 8-byte raw buffer load builtin
        // to a single dword load
        a = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
        b = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff + 4, soff, 0));
    }
    template <int AUX = 0>
    static __device__ __forceinline__ void store(pair_t v, __amdgpu_buffer_rsrc_t r, unsigned voff,
                                                 unsigned soff) {
        typedef unsigned u2 __attribute__((ext_vector_type(2)));
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, voff, soff, AUX);
    }
    // the pair as stored, no conversion (so that nothing has to wait for the data yet)
    static __device__ __forceinline__ pair_t load_raw(__amdgpu_buffer_rsrc_t r, unsigned voff,
                                                      unsigned soff) {
        float a, b;
        load(r, voff, soff, a, b);
        pair_t v;
        v.x = a;
        v.y = b;
        return v;
    }
};
template <> struct BufIO2<half_t> {
    typedef half2v pair_t;
    static __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, unsigned voff,
                                                unsigned soff, float& a, float& b) {
        const half2v h =
            __builtin_bit_cast(half2v, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
        a = (float)h.x;
        b = (float)h.y;
    }
    template <int AUX = 0>
    static __device__ __forceinline__ void store(pair_t v, __amdgpu_buffer_rsrc_t r, unsigned voff,
                                                 unsigned soff) {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, voff, soff, AUX);
    }
    static __device__ __forceinline__ pair_t load_raw(__amdgpu_buffer_rsrc_t r, unsigned voff,
                                                      unsigned soff) {
        return __builtin_bit_cast(pair_t, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
    }
};

// One workgroup owns one board and 64 channels.  A lane owns two consecutive
// channels (one 4- or 8-byte access instead of two), a half-wave owns a tile,
// so a wavefront handles two neighbouring tiles at once and the 13 wavefronts
// cover the 25 tiles in a single pass: every wavefront issues its 36 M loads
// once, up front, instead of walking through several tiles with a full memory
// latency each, and the number of memory instructions (which bounded the
// one-channel-per-lane version) is halved.  The two tiles of a wavefront are
// adjacent rows of M and V, so the half-wave only adds a constant to the lane
// offset.  The LDS plane carries a zero halo: the 6x6 patch reads need no
// bounds handling.  Loads that fall outside the board (clipped tiles) read
// neighbouring memory or, past the end of the buffer, zero (raw buffer
// semantics); their results are never stored.
//
// CG = channels per workgroup.  64 (a half-wave per tile, 13 wavefronts) moves
// whole 128-byte runs and is the choice when there are enough boards to give
// every compute unit a workgroup; with few boards the kernel is bound by the
// arithmetic of the one compute unit a workgroup runs on, and 32 or 16 channels
// per workgroup (4 or 8 tiles per wavefront, 7 or 4 wavefronts) spread a board
// over more compute units.
// Cache policy of the fused transform's stores.  With 64 channels per work-group every
// store instruction writes whole 128-byte lines (64 channels of one tile row or board
// point), and nothing in the kernel reads them again: written through (sc0 sc1) they leave
// for memory while the kernel runs instead of staying behind as dirty lines that the end
// of the kernel has to flush (measured in fp16 at 64 boards, 256 filters: 15.2 -> 14.0 us per
// launch).  The narrower work-groups write half and quarter lines, which written through
// cost twice the time (32 channels at 64 boards: 16.4 us against 12.9): they stay write-back.
template <int CG> constexpr int xform_store_policy() { return CG == 64 ? kStoreThrough : 0; }
constexpr int kPlane = 22;       // LDS plane: 19 points + 1 zero halo before + 2 after
// Strides of the plane in channel pairs.  A store or load instruction of the transform
// touches the same cell of every tile in the wavefront, CG / 2 consecutive pairs each, and
// tiles lie 4 cells (and 4 rows) apart: with cells of exactly CG / 2 pairs the narrow shapes
// put all their tiles on the same banks (16 channels: 8 tiles on 8 of 32 banks, measured
// 237 k conflict cycles in 351 k active ones per launch).  Padded so that four cells and
// four rows both advance the bank by CG / 2, consecutive tiles take consecutive groups of
// banks (7.7 k conflict cycles left, the halo; the launch takes as long as before: LDS was
// not what it waited for).  The 64-channel shape (one tile per 32 lanes) needs no padding.
constexpr int plane_cell_pairs(int cg) { return cg == 16 ? 10 : cg == 32 ? 20 : cg / 2; }
constexpr int plane_row_pairs(int cg) {
    return cg == 16 ? kPlane * 10 + 6 : cg == 32 ? kPlane * 20 + 4 : kPlane * (cg / 2);
}
constexpr int plane_pairs(int cg) { return kPlane * plane_row_pairs(cg); }
constexpr int fuse_waves(int cg) { return (kTilesPerBoard + 128 / cg - 1) / (128 / cg); }

// M and Vn may be one array (every value of M is in a register before the same lane writes
// the value of V that takes its place), so neither is declared free of aliases.
template <typename P, int CG>
__global__ __launch_bounds__(fuse_waves(CG) * 64) void out_in_transform_k(
    const P* M, const P* __restrict__ res, P* __restrict__ act_out, P* Vn,
    const float* __restrict__ bn_scale, const float* __restrict__ bn_mean, float rfac, int n,
    int Kp, int Tp) {
    __shared__ typename BufIO2<P>::pair_t ybuf[plane_pairs(CG)];
    typedef typename BufIO2<P>::pair_t pair_t;
    constexpr int CP = CG / 2;        // channel pairs per plane cell = lanes per tile
    constexpr int CS = plane_cell_pairs(CG), RS = plane_row_pairs(CG);   // plane strides
    constexpr int TPW = 64 / CP;      // tiles per wavefront
    constexpr int WAVES = fuse_waves(CG);
    // Work-group w runs on die w % 8, each die with its own L2.  The narrow shapes share
    // 128-byte lines between the work-groups of neighbouring channel groups, so the items
    // (board, channel group) are cut into 8 contiguous segments and work-group w takes item
    // w / 8 of segment w % 8: the sharers then sit on one die and a line comes from memory
    // once, instead of once for each die that holds a piece of it.
    const int ncg = Kp / CG;
    const int per_die = (n * ncg + 7) >> 3;
    const int item = (int)(blockIdx.x & 7) * per_die + (int)(blockIdx.x >> 3);
    if (item >= n * ncg) return;
    const int b = item / ncg;
    const int cg = item - b * ncg;

    const unsigned lane = threadIdx.x & 63;
    const unsigned cl = lane % CP, sub = lane / CP;    // channel pair, tile within the wavefront
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned esz = (unsigned)sizeof(P);
    const int j = TPW * wave + (int)sub;               // this lane's tile
    const bool valid = j < kTilesPerBoard;
    const int jc = valid ? j : kTilesPerBoard - 1;
    const int by = jc / 5, bx = jc - by * 5;
    const int ny = min(4, kBoard - 4 * by), nx = min(4, kBoard - 4 * bx);

    const unsigned pstride = (unsigned)Tp * (unsigned)Kp * esz;   // bytes between positions
    const size_t tile_bytes = (size_t)kPos * Tp * Kp * esz;
    const size_t act_bytes = (size_t)n * kPts * Kp * esz;
    const __amdgpu_buffer_rsrc_t rM = make_rsrc(M, tile_bytes);
    const __amdgpu_buffer_rsrc_t rV = make_rsrc(Vn, tile_bytes);
    const __amdgpu_buffer_rsrc_t rR = make_rsrc(res != nullptr ? res : M, act_bytes);
    const __amdgpu_buffer_rsrc_t rA = make_rsrc(act_out != nullptr ? act_out : Vn, act_bytes);
    // per-lane byte offsets: channel pair (+ the tile's row within the wavefront) / tile origin
    unsigned voff_t = cl * 2 * esz + (valid ? sub : 0u) * (unsigned)Kp * esz;
    unsigned voff_a = cl * 2 * esz + (unsigned)((4 * by) * kBoard + 4 * bx) * (unsigned)Kp * esz;
    // Pin both offsets into registers here: computed later, between the two groups of
    // loads, their arithmetic waits for the first group's data (a register-reuse hazard).
    asm volatile("" : "+v"(voff_t), "+v"(voff_a));
    // uniform byte offsets of the wavefront's first tile / of the board
    const unsigned soff_t =
        ((unsigned)(b * kTilesPerBoard + TPW * wave) * (unsigned)Kp + cg * CG) * esz;
    const unsigned soff_a = ((unsigned)(b * kPts) * (unsigned)Kp + cg * CG) * esz;
    float sc[2], nb[2];   // scale * (y - mean) = y * scale + nb
#pragma unroll
    for (int v = 0; v < 2; v++) {
        sc[v] = bn_scale[cg * CG + cl * 2 + v];
        nb[v] = -sc[v] * bn_mean[cg * CG + cl * 2 + v];
    }

    // All loads of the pass go out before any arithmetic.  M's go first, column by
    // column of the 6x6 position grid: loads return in issue order at the rate the
    // memory system delivers them, and the first transform pass works on columns, so it
    // can start on the first six while the rest are still arriving.  The skip
    // connection (needed last) follows, left as stored: converting it here would wait
    // for it.  The scheduling barrier keeps the compiler from sinking those loads behind
    // the first arithmetic on M.
    pair_t m[36];   // as stored; converted where used
#pragma unroll
    for (int xx = 0; xx < 6; xx++) {
        unsigned so = soff_t + (unsigned)xx * pstride;
#pragma unroll
        for (int row = 0; row < 6; row++) {
            m[row * 6 + xx] = BufIO2<P>::load_raw(rM, voff_t, so);
            so += 6u * pstride;
        }
        __builtin_amdgcn_sched_barrier(0);   // keep the columns in this order
    }
    pair_t r[16];
    if (res != nullptr) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int jj = 0; jj < 4; jj++)
                r[i * 4 + jj] = BufIO2<P>::load_raw(
                    rR, voff_a, soff_a + (unsigned)(i * kBoard + jj) * (unsigned)Kp * esz);
    } else {
#pragma unroll
        for (int q = 0; q < 16; q++) {
            r[q].x = (P)0.0f;
            r[q].y = (P)0.0f;
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // zero the halo cells of the plane (rows and columns 0, 20, 21): 3 full rows
    // and 3 cells in each of the 19 rows between them; one cell per tile slot
    {
        pair_t zero;
        zero.x = (P)0.0f;
        zero.y = (P)0.0f;
        for (int q = TPW * wave + (int)sub; q < 3 * kPlane + 3 * kBoard; q += TPW * WAVES) {
            int cell;
            if (q < 3 * kPlane) {
                const int row = q < kPlane ? 0 : (q < 2 * kPlane ? kBoard + 1 : kBoard + 2);
                cell = row * RS + (q % kPlane) * CS;
            } else {
                const int e = q - 3 * kPlane, y = 1 + e / 3, c3 = e % 3;
                cell = y * RS + (c3 == 0 ? 0 : kBoard + c3) * CS;
            }
            ybuf[cell + cl] = zero;
        }
    }

    // ---- phase 1: A^T m A, BN (+ residual), ReLU -> LDS plane (+ memory)
    // plane cell of the tile's patch origin (board row 4by-1, column 4bx-1)
    pair_t* const origin = ybuf + (4 * by) * RS + (4 * bx) * CS + cl;
    pair_t keep[16];   // this tile's activations, written to memory after the barrier
    {
        float o[2][16];
        float t1[2][24];
        // column pass in the order the columns arrive (the barrier pins that order)
#pragma unroll
        for (int xx = 0; xx < 6; xx++) {
#pragma unroll
            for (int v = 0; v < 2; v++) {
                float c[6];
#pragma unroll
                for (int row = 0; row < 6; row++)
                    c[row] = (float)(v == 0 ? m[row * 6 + xx].x : m[row * 6 + xx].y);
                at6(c[0], c[1], c[2], c[3], c[4], c[5], t1[v][0 + xx], t1[v][6 + xx],
                    t1[v][12 + xx], t1[v][18 + xx]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int v = 0; v < 2; v++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                at6(t1[v][i * 6 + 0], t1[v][i * 6 + 1], t1[v][i * 6 + 2], t1[v][i * 6 + 3],
                    t1[v][i * 6 + 4], t1[v][i * 6 + 5], o[v][i * 4 + 0], o[v][i * 4 + 1],
                    o[v][i * 4 + 2], o[v][i * 4 + 3]);
#pragma unroll
        for (int i = 0; i < 4; i++) {
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
                pair_t sv;
                sv.x = act_to_storage<P>(fmaxf(
                    0.0f, fmaf((float)r[i * 4 + jj].x, rfac, fmaf(o[0][i * 4 + jj], sc[0], nb[0]))));
                sv.y = act_to_storage<P>(fmaxf(
                    0.0f, fmaf((float)r[i * 4 + jj].y, rfac, fmaf(o[1][i * 4 + jj], sc[1], nb[1]))));
                keep[i * 4 + jj] = sv;
                if (valid && i < ny && jj < nx) origin[(i + 1) * RS + (jj + 1) * CS] = sv;
            }
        }
    }
    __syncthreads();
    // The activation leaves only now: stores issued before the barrier would have to be
    // acknowledged before any wavefront may pass it; here they drain under phase 2.
    if (act_out != nullptr) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int jj = 0; jj < 4; jj++)
                if (valid && i < ny && jj < nx)
                    BufIO2<P>::template store<xform_store_policy<CG>()>(keep[i * 4 + jj], rA, voff_a,
                                     soff_a + (unsigned)(i * kBoard + jj) * (unsigned)Kp * esz);
    }

    // ---- phase 2: B^T d B of the next layer from the plane in LDS
    {
        pair_t raw[36];
#pragma unroll
        for (int yy = 0; yy < 6; yy++)
#pragma unroll
            for (int xx = 0; xx < 6; xx++) raw[yy * 6 + xx] = origin[yy * RS + xx * CS];
        pair_t outp[36];
#pragma unroll
        for (int v = 0; v < 2; v++) {
            float d[36], t1[36];
#pragma unroll
            for (int q = 0; q < 36; q++) d[q] = (float)(v == 0 ? raw[q].x : raw[q].y);
#pragma unroll
            for (int xx = 0; xx < 6; xx++)
                bt6(d[0 + xx], d[6 + xx], d[12 + xx], d[18 + xx], d[24 + xx], d[30 + xx],
                    t1[0 + xx], t1[6 + xx], t1[12 + xx], t1[18 + xx], t1[24 + xx], t1[30 + xx]);
#pragma unroll
            for (int yy = 0; yy < 6; yy++)
                bt6(t1[yy * 6 + 0], t1[yy * 6 + 1], t1[yy * 6 + 2], t1[yy * 6 + 3],
                    t1[yy * 6 + 4], t1[yy * 6 + 5], d[yy * 6 + 0], d[yy * 6 + 1], d[yy * 6 + 2],
                    d[yy * 6 + 3], d[yy * 6 + 4], d[yy * 6 + 5]);
#pragma unroll
            for (int q = 0; q < 36; q++) {
                if (v == 0) outp[q].x = (P)d[q];
                else outp[q].y = (P)d[q];
            }
        }
        if (valid) {
            unsigned so = soff_t;
#pragma unroll
            for (int p = 0; p < 36; p++) {
                BufIO2<P>::template store<xform_store_policy<CG>()>(outp[p], rV, voff_t, so);
                so += pstride;
            }
        }
    }
}

template <typename P>
void launch_out_in_transform(const P* M, const P* res, P* act_out, P* Vn, const float* bn_scale,
                             const float* bn_mean, float rfac, int n, int Kp, int Tp,
                             hipStream_t s, LaunchTimer* t) {
    // With few boards a narrow shape spreads a board's arithmetic over more compute units;
    // the 64-channel shape moves whole lines.  Measured per forward of 10 blocks of 256 filters,
    // us, with 16 / 32 / 64 channels per work-group.  fp16 (filters that are no 3x3 ones): 8
    // boards 307 / 324 / 356, 16 boards 415 / 425 / 443, 20 boards 478 / 468 / 478, 24 boards 507 / 494 /
    // 504, 32 boards 487 / 469 / 489, 64 boards 709 / 680 / 645.  fp32: 8 boards 477 / 504 / 586, 17
    // boards 692 / 667 / 802, 24 boards 908 / 878 / 990, 32 boards 1094 / 1079 / 1169, 40 boards 1354 /
    // 1384 / 1371, 64 boards 1954 / 1972 / 1974: there the 64-channel shape is no better at any batch,
    // and the line below, drawn in fp16, gives away up to a tenth from 21 to 32 boards.
    // The narrow shapes only pay with the die-aware item order of the kernel: dealt round-robin
    // over the dies, their work-groups fetch every line of M once per die that holds a piece
    // of it (16 channels at batch 16: 11.2 us per launch against 7.7).
    const int items64 = n * (Kp / 64);
    auto grid = [](int items) { return dim3((unsigned)(8 * ((items + 7) / 8))); };
    if (items64 > 80)
        launch(out_in_transform_k<P, 64>, grid(items64), dim3(fuse_waves(64) * 64), s, t, M, res,
               act_out, Vn, bn_scale, bn_mean, rfac, n, Kp, Tp);
    else if (items64 > 64)
        launch(out_in_transform_k<P, 32>, grid(items64 * 2), dim3(fuse_waves(32) * 64), s, t, M,
               res, act_out, Vn, bn_scale, bn_mean, rfac, n, Kp, Tp);
    else
        launch(out_in_transform_k<P, 16>, grid(items64 * 4), dim3(fuse_waves(16) * 64), s, t, M,
               res, act_out, Vn, bn_scale, bn_mean, rfac, n, Kp, Tp);
}

// ---------------------------------------------------------------------------
// The 36 independent GEMMs M_p[t][k] = sum_c V_p[t][c] * U_p[k][c]
// (reference src/CPUPipe.cpp:185-210; GPU twin XgemmBatched).
//
// One workgroup = 4 wavefronts (2x2) computes a BM x BN tile of one position.
// Both operands are staged through LDS in 128-byte-per-row slices (64 halves
// or 32 floats of the contraction index), double buffered, rows padded by 16
// bytes so that the 16-byte-per-lane fragment reads are conflict free.
// Each lane feeds the matrix cores with 16 contiguous bytes of its row:
//   fp16: one v_mfma_f32_32x32x16_f16 per fragment pair (8 halves per lane)
//   fp32: four v_mfma_f32_32x32x2_f32 per fragment pair (one float each)
// Lane l supplies row (l & 31) of its 32-row block of either operand, and the
// upper half-wave supplies the other half of the k-slice; the assignment of k
// values to MFMA k-slots is the same for both operands, which is all the
// contraction needs.  Accumulation is fp32 for both storage types.
// Workgroups of different Winograd positions start their walk over the k-slices at
// different slices (the sum over k may run in any order): at any moment the
// 128-byte pieces being fetched then spread over whole 512-byte rows instead of
// all workgroups hitting the same quarter of every row, which would leave most
// memory channels idle.  The rotation depends on the position only, so a given
// board sees the same summation order whatever else is in the batch.
__device__ __forceinline__ int rotated_slice(int k, int rot, int nk) {
    const int kk = k + rot;
    return kk >= nk ? kk - nk : kk;
}

template <typename P> struct Mma;
template <> struct Mma<half_t> {
    static __device__ __forceinline__ float16v run(int4v a, int4v b, float16v c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8v, a),
                                                      __builtin_bit_cast(half8v, b), c, 0, 0, 0);
    }
};
template <> struct Mma<float> {
    static __device__ __forceinline__ float16v run(int4v a, int4v b, float16v c) {
        const float4v fa = __builtin_bit_cast(float4v, a);
        const float4v fb = __builtin_bit_cast(float4v, b);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(fa.x, fb.x, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(fa.y, fb.y, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(fa.z, fb.z, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(fa.w, fb.w, c, 0, 0, 0);
        return c;
    }
};

// Work items are (position, row tile, column tile) triples, column tile fastest.
// The device hands workgroup b to accelerator die (XCD) b % 8, each die with its
// own L2, so the item list is cut into 8 contiguous segments and workgroup b
// takes item (b / 8) of segment (b % 8): all tiles of one position, and the
// column tiles that share a V row tile, then run on the same die, U_p and the
// V tile are fetched from memory once and the repeats hit that die's L2.
template <typename P, int BM, int BN, int NK>
__global__ __launch_bounds__(256) void wino_gemm_k(const P* __restrict__ V,
                                                   const P* __restrict__ U, P* __restrict__ M,
                                                   int Tp, int Cp, int Kp, int tiles_m,
                                                   int tiles_n, int seg) {
    constexpr int EPC = 16 / sizeof(P);   // elements per 16-byte chunk
    constexpr int BK = 128 / sizeof(P);   // contraction extent of one LDS stage
    // LDS rows: padded to 144 bytes, or (the 64-column tile) bare 128-byte rows whose
    // 16-byte chunks are permuted by the row number, which is just as conflict free for
    // the fragment reads (16 lanes = 16 rows: 8 chunk slots x 2 row parities = all 64
    // banks) and brings a stage pair under a third of the LDS, so that three
    // work-groups share a compute unit instead of two.
    constexpr bool SWZ = BN == 64 && sizeof(P) == 2;   // fp32 is bound by the matrix pipe: no gain
    constexpr int ROW = SWZ ? BK : BK + EPC;
    constexpr int WM = BM / 2, WN = BN / 2;
    constexpr int MB = WM / 32, NB = WN / 32;
    constexpr int A_CH = BM * 8 / 256, B_CH = BN * 8 / 256;  // chunks per thread and stage
    auto slot = [](int row, int chunk) { return SWZ ? (chunk ^ ((row >> 1) & 7)) : chunk; };
    constexpr int CROW = BN + EPC;        // padded row of the staged output tile
    constexpr int STAGE = (BM + BN) * ROW;
    constexpr int SMEM = (2 * STAGE > BM * CROW) ? 2 * STAGE : BM * CROW;
    static_assert(MB >= 1 && NB >= 1, "tile too small for a 2x2 wave grid");

    __shared__ __attribute__((aligned(16))) P smem[SMEM];

    const int n_items = kPos * tiles_m * tiles_n;
    const int xcd = blockIdx.x & 7;
    const int item = xcd * seg + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= seg || item >= n_items) return;
    const int tn = item % tiles_n;
    const int rest = item / tiles_n;
    const int tm = rest % tiles_m;
    const int p = rest / tiles_m;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wy = wave >> 1, wx = wave & 1;
    const P* Ag = V + ((size_t)p * Tp + (size_t)tm * BM) * Cp;
    const P* Bg = U + ((size_t)p * Kp + (size_t)tn * BN) * Cp;

    float16v acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    // Two register stages: the slice for step kt+2 is requested while step kt is
    // being multiplied, so two slices per workgroup are in flight.
    int4v ra[2][A_CH], rb[2][B_CH];
    (void)Cp;
    const int lrow = tid >> 3, lch = tid & 7;  // row / chunk of this thread's first chunk

    auto gload = [&](int st, int k0) {
#pragma unroll
        for (int i = 0; i < A_CH; i++)
            ra[st][i] = *reinterpret_cast<const int4v*>(Ag + (size_t)(lrow + i * 32) * Cp + k0 +
                                                        lch * EPC);
#pragma unroll
        for (int i = 0; i < B_CH; i++)
            rb[st][i] = *reinterpret_cast<const int4v*>(Bg + (size_t)(lrow + i * 32) * Cp + k0 +
                                                        lch * EPC);
    };
    auto lstore = [&](int st, int buf) {
        P* As = smem + buf * STAGE;
        P* Bs = As + BM * ROW;
#pragma unroll
        for (int i = 0; i < A_CH; i++)
            *reinterpret_cast<int4v*>(&As[(lrow + i * 32) * ROW + slot(lrow, lch) * EPC]) = ra[st][i];
#pragma unroll
        for (int i = 0; i < B_CH; i++)
            *reinterpret_cast<int4v*>(&Bs[(lrow + i * 32) * ROW + slot(lrow, lch) * EPC]) = rb[st][i];
    };

    // NK = Cp / BK is a template argument: the pipeline below is straight-line
    // code, so the compiler knows exactly which loads are outstanding at each
    // wait and the slice for step k+2 really stays in flight across step k.
    const int rot = p % NK;
    gload(0, rotated_slice(0, rot, NK) * BK);
    if (NK > 1) gload(1, rotated_slice(1, rot, NK) * BK);
    lstore(0, 0);
    __syncthreads();

    const int frow = lane & 31, fk = lane >> 5;   // tile offsets are multiples of 32 rows
#pragma unroll
    for (int k = 0; k < NK; k++) {
        const int h = k & 1;
        if (k + 2 < NK) {
            gload(h, rotated_slice(k + 2, rot, NK) * BK);
            __builtin_amdgcn_sched_barrier(0);  // request the slice before the math starts
        }
        const P* As = smem + h * STAGE;
        const P* Bs = As + BM * ROW;
#pragma unroll
        for (int kc = 0; kc < 4; kc++) {
            int4v fa[MB], fb[NB];
#pragma unroll
            for (int i = 0; i < MB; i++)
                fa[i] = *reinterpret_cast<const int4v*>(
                    &As[(wy * WM + i * 32 + frow) * ROW + slot(frow, kc * 2 + fk) * EPC]);
#pragma unroll
            for (int j = 0; j < NB; j++)
                fb[j] = *reinterpret_cast<const int4v*>(
                    &Bs[(wx * WN + j * 32 + frow) * ROW + slot(frow, kc * 2 + fk) * EPC]);
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int j = 0; j < NB; j++) acc[i][j] = Mma<P>::run(fb[j], fa[i], acc[i][j]);
        }
        if (k + 1 < NK) lstore(h ^ 1, h ^ 1);
        __syncthreads();
    }

    // The U block is the MFMA's row operand and the V block its column operand,
    // so register r of lane l holds output channel 8*(r/4) + 4*(l/32) + r%4 of
    // tile row l%32: four consecutive channels per lane, which go to the LDS
    // staging tile (all slices have been consumed) as one 8- or 16-byte write.
    // From there whole rows leave in 16-byte pieces.
    const int ccol = 4 * (lane >> 5), crow = lane & 31;
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                typename Quad<P>::type v;
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = to_storage<P>(acc[i][j][q * 4 + e]);
                *reinterpret_cast<typename Quad<P>::type*>(
                    &smem[(wy * WM + i * 32 + crow) * CROW + wx * WN + j * 32 + 8 * q + ccol]) = v;
            }
    __syncthreads();
    constexpr int CPR = BN / EPC;  // 16-byte chunks per output row
    P* Mg = M + ((size_t)p * Tp + (size_t)tm * BM) * Kp + (size_t)tn * BN;
#pragma unroll 4
    for (int q = tid; q < BM * CPR; q += 256) {
        const int row = q / CPR, ch = q - row * CPR;
        *reinterpret_cast<int4v*>(Mg + (size_t)row * Kp + ch * EPC) =
            *reinterpret_cast<const int4v*>(&smem[row * CROW + ch * EPC]);
    }
}

// Persistent variant for an even number of k-slices.  A workgroup walks
// through several work items of its die's segment; the global loads of the
// next item's first two slices are issued while the current item's last two
// slices are being multiplied, so every workgroup keeps two slices (64 KB at
// the 128x128 tile) in flight from its first to its last item instead of
// starting each tile with an empty pipeline.  The finished tile leaves through
// the LDS stage that the last slice has just vacated.
template <typename P, int BM, int BN, int NK>
__global__ __launch_bounds__(256, 2) void wino_gemm_persistent_k(
    const P* __restrict__ V, const P* __restrict__ U, P* __restrict__ M, int Tp, int Cp, int Kp,
    int tiles_m, int tiles_n, int seg, int wg_per_xcd) {
    static_assert(NK >= 2 && (NK % 2) == 0, "needs an even slice count");
    constexpr int EPC = 16 / sizeof(P);
    constexpr int BK = 128 / sizeof(P);
    constexpr int ROW = BK + EPC;
    constexpr int WM = BM / 2, WN = BN / 2;
    constexpr int MB = WM / 32, NB = WN / 32;
    constexpr int A_CH = BM * 8 / 256, B_CH = BN * 8 / 256;
    constexpr int CROW = BN + EPC;
    constexpr int STAGE = (BM + BN) * ROW;
    // output staging fits one vacated stage either whole or in two row halves
    constexpr int EP_PARTS = (BM * CROW > STAGE) ? 2 : 1;
    static_assert((BM / EP_PARTS) * CROW <= STAGE, "output staging does not fit a stage");
    static_assert(EP_PARTS == 1 || WM * 2 == BM, "row halves must coincide with the wave rows");

    __shared__ __attribute__((aligned(16))) P smem[2 * STAGE];

    const int n_items = kPos * tiles_m * tiles_n;
    const int xcd = blockIdx.x & 7, w = blockIdx.x >> 3;
    int item = xcd * seg + w;
    const int last = min(n_items, (xcd + 1) * seg);
    if (w >= wg_per_xcd || item >= last) return;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wy = wave >> 1, wx = wave & 1;
    const int lrow = tid >> 3, lch = tid & 7;
    const int frow = lane & 31, fk = (lane >> 5) * EPC;
    const int ccol = 4 * (lane >> 5), crow = lane & 31;
    (void)Cp;

    // rs = row stride of the operand loads; the look-ahead past a workgroup's last
    // item uses rs = 0 and one shared address, so that the loads stay
    // unconditional (the compiler can then count outstanding loads exactly)
    // without fetching anything real.
    struct Ptrs { const P* a; const P* b; P* m; size_t rs; int rot; };
    auto locate = [&](int it) {
        const int tn = it % tiles_n;
        const int rest = it / tiles_n;
        const int tm = rest % tiles_m;
        const int p = rest / tiles_m;
        Ptrs r;
        r.a = V + ((size_t)p * Tp + (size_t)tm * BM) * Cp + (size_t)lrow * Cp + lch * EPC;
        r.b = U + ((size_t)p * Kp + (size_t)tn * BN) * Cp + (size_t)lrow * Cp + lch * EPC;
        r.m = M + ((size_t)p * Tp + (size_t)tm * BM) * Kp + (size_t)tn * BN;
        r.rs = (size_t)Cp;
        r.rot = p % NK;
        return r;
    };

    int4v ra[2][A_CH], rb[2][B_CH];
    auto gload = [&](int st, const Ptrs& q, int k0) {
#pragma unroll
        for (int i = 0; i < A_CH; i++)
            ra[st][i] = *reinterpret_cast<const int4v*>(q.a + (size_t)(i * 32) * q.rs + k0);
#pragma unroll
        for (int i = 0; i < B_CH; i++)
            rb[st][i] = *reinterpret_cast<const int4v*>(q.b + (size_t)(i * 32) * q.rs + k0);
    };
    auto lstore = [&](int st, int buf) {
        P* As = smem + buf * STAGE;
        P* Bs = As + BM * ROW;
#pragma unroll
        for (int i = 0; i < A_CH; i++)
            *reinterpret_cast<int4v*>(&As[(lrow + i * 32) * ROW + lch * EPC]) = ra[st][i];
#pragma unroll
        for (int i = 0; i < B_CH; i++)
            *reinterpret_cast<int4v*>(&Bs[(lrow + i * 32) * ROW + lch * EPC]) = rb[st][i];
    };

    Ptrs cur = locate(item);
    gload(0, cur, rotated_slice(0, cur.rot, NK) * BK);
    gload(1, cur, rotated_slice(1, cur.rot, NK) * BK);
    lstore(0, 0);
    __syncthreads();

    for (;;) {
        const int nitem = item + wg_per_xcd;
        const bool has_next = nitem < last;  // uniform
        Ptrs nxt = locate(has_next ? nitem : item);
        if (!has_next) {
            nxt.a = V;
            nxt.b = U;
            nxt.rs = 0;
        }

        float16v acc[MB][NB];
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

#pragma unroll
        for (int k = 0; k < NK; k++) {
            const int h = k & 1;
            if (k + 2 < NK) {
                gload(h, cur, rotated_slice(k + 2, cur.rot, NK) * BK);
            } else {
                gload(h, nxt, rotated_slice(k + 2 - NK, nxt.rot, NK) * BK);
            }
            __builtin_amdgcn_sched_barrier(0);
            const P* As = smem + h * STAGE;
            const P* Bs = As + BM * ROW;
#pragma unroll
            for (int kc = 0; kc < 4; kc++) {
                int4v fa[MB], fb[NB];
#pragma unroll
                for (int i = 0; i < MB; i++)
                    fa[i] = *reinterpret_cast<const int4v*>(
                        &As[(wy * WM + i * 32 + frow) * ROW + kc * 2 * EPC + fk]);
#pragma unroll
                for (int j = 0; j < NB; j++)
                    fb[j] = *reinterpret_cast<const int4v*>(
                        &Bs[(wx * WN + j * 32 + frow) * ROW + kc * 2 * EPC + fk]);
#pragma unroll
                for (int i = 0; i < MB; i++)
#pragma unroll
                    for (int j = 0; j < NB; j++)
                        acc[i][j] = Mma<P>::run(fb[j], fa[i], acc[i][j]);
            }
            lstore(h ^ 1, h ^ 1);
            __syncthreads();
        }

        // The last slice sat in stage 1, which is free now (stage 0 already holds
        // the next item's first slice).
        P* stage = smem + STAGE;
        constexpr int CPR = BN / EPC;
        constexpr int PROWS = BM / EP_PARTS;
#pragma unroll
        for (int part = 0; part < EP_PARTS; part++) {
            if (EP_PARTS == 1 || wy == part) {
#pragma unroll
                for (int i = 0; i < MB; i++)
#pragma unroll
                    for (int j = 0; j < NB; j++)
#pragma unroll
                        for (int q = 0; q < 4; q++) {
                            typename Quad<P>::type v;
#pragma unroll
                            for (int e = 0; e < 4; e++) v[e] = to_storage<P>(acc[i][j][q * 4 + e]);
                            const int row = (EP_PARTS == 1 ? wy * WM : 0) + i * 32 + crow;
                            *reinterpret_cast<typename Quad<P>::type*>(
                                &stage[row * CROW + wx * WN + j * 32 + 8 * q + ccol]) = v;
                        }
            }
            __syncthreads();
#pragma unroll 4
            for (int q = tid; q < PROWS * CPR; q += 256) {
                const int row = q / CPR, ch = q - row * CPR;
                *reinterpret_cast<int4v*>(cur.m + (size_t)(part * PROWS + row) * Kp + ch * EPC) =
                    *reinterpret_cast<const int4v*>(&stage[row * CROW + ch * EPC]);
            }
            __syncthreads();
        }
        if (!has_next) break;
        item = nitem;
        cur = nxt;
    }
}

// Large-tile variant: one workgroup of 8 wavefronts (2 x 4) owns a 256 x 256
// tile, i.e. all output channels of 256 tiles when the network has 256
// filters.  Per multiply-add it moves half as many operand bytes from L2 to
// the compute unit as the 128 x 128 tile, which is what bounds this GEMM (its
// contraction is only 256 deep); at 64 boards the 7 x 36 tiles fill the 256
// compute units in a single round.
template <typename P, int NK>
__global__ __launch_bounds__(512) void wino_gemm_big_k(const P* __restrict__ V,
                                                       const P* __restrict__ U,
                                                       P* __restrict__ M, int T, int Tp, int Cp,
                                                       int Kp, int tiles_m, int tiles_n, int seg) {
    constexpr int BM = 256, BN = 256, NT = 512;
    constexpr int EPC = 16 / sizeof(P);
    constexpr int BK = 128 / sizeof(P);
    constexpr int ROW = BK + EPC;
    constexpr int WM = 128, WN = 64;       // per-wave tile, waves laid out 2 (rows) x 4 (columns)
    constexpr int MB = WM / 32, NB = WN / 32;
    constexpr int A_CH = BM * 8 / NT, B_CH = BN * 8 / NT;
    constexpr int CROW = BN + EPC;
    constexpr int STAGE = (BM + BN) * ROW;
    constexpr int EP_PARTS = sizeof(P) == 2 ? 2 : 4;   // output staged through one vacated stage
    constexpr int PROWS = BM / EP_PARTS;
    static_assert(PROWS * CROW <= STAGE, "output staging does not fit a stage");

    __shared__ __attribute__((aligned(16))) P smem[2 * STAGE];

    const int n_items = kPos * tiles_m * tiles_n;
    const int xcd = blockIdx.x & 7;
    const int item = xcd * seg + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= seg || item >= n_items) return;
    const int tn = item % tiles_n;
    const int rest = item / tiles_n;
    const int tm = rest % tiles_m;
    const int p = rest / tiles_m;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wy = wave >> 2, wx = wave & 3;
    const int lrow = tid >> 3, lch = tid & 7;   // 64 rows per pass of the workgroup
    // Rows past the last real tile re-read row T-1 (their products are never stored).
    const P* Ag[A_CH];
#pragma unroll
    for (int i = 0; i < A_CH; i++) {
        const int row = min(tm * BM + lrow + i * 64, T - 1);
        Ag[i] = V + ((size_t)p * Tp + row) * Cp + lch * EPC;
    }
    const P* Bg = U + ((size_t)p * Kp + (size_t)tn * BN + lrow) * Cp + lch * EPC;

    float16v acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    int4v ra[2][A_CH], rb[2][B_CH];
    auto gload = [&](int st, int k0) {
#pragma unroll
        for (int i = 0; i < A_CH; i++)
            ra[st][i] = *reinterpret_cast<const int4v*>(Ag[i] + k0);
#pragma unroll
        for (int i = 0; i < B_CH; i++)
            rb[st][i] = *reinterpret_cast<const int4v*>(Bg + (size_t)(i * 64) * Cp + k0);
    };
    auto lstore = [&](int st, int buf) {
        P* As = smem + buf * STAGE;
        P* Bs = As + BM * ROW;
#pragma unroll
        for (int i = 0; i < A_CH; i++)
            *reinterpret_cast<int4v*>(&As[(lrow + i * 64) * ROW + lch * EPC]) = ra[st][i];
#pragma unroll
        for (int i = 0; i < B_CH; i++)
            *reinterpret_cast<int4v*>(&Bs[(lrow + i * 64) * ROW + lch * EPC]) = rb[st][i];
    };

    const int rot = p % NK;
    gload(0, rotated_slice(0, rot, NK) * BK);
    if (NK > 1) gload(1, rotated_slice(1, rot, NK) * BK);
    lstore(0, 0);
    __syncthreads();

    const int frow = lane & 31, fk = (lane >> 5) * EPC;
#pragma unroll
    for (int k = 0; k < NK; k++) {
        const int h = k & 1;
        if (k + 2 < NK) {
            gload(h, rotated_slice(k + 2, rot, NK) * BK);
            __builtin_amdgcn_sched_barrier(0);
        }
        const P* As = smem + h * STAGE;
        const P* Bs = As + BM * ROW;
#pragma unroll
        for (int kc = 0; kc < 4; kc++) {
            int4v fa[MB], fb[NB];
#pragma unroll
            for (int i = 0; i < MB; i++)
                fa[i] = *reinterpret_cast<const int4v*>(
                    &As[(wy * WM + i * 32 + frow) * ROW + kc * 2 * EPC + fk]);
#pragma unroll
            for (int j = 0; j < NB; j++)
                fb[j] = *reinterpret_cast<const int4v*>(
                    &Bs[(wx * WN + j * 32 + frow) * ROW + kc * 2 * EPC + fk]);
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int j = 0; j < NB; j++) acc[i][j] = Mma<P>::run(fb[j], fa[i], acc[i][j]);
        }
        if (k + 1 < NK) lstore(h ^ 1, h ^ 1);
        __syncthreads();
    }

    // Output: PROWS rows at a time through LDS, then out in 16-byte pieces.
    const int ccol = 4 * (lane >> 5), crow = lane & 31;
    constexpr int CPR = BN / EPC;
    P* Mg = M + ((size_t)p * Tp + (size_t)tm * BM) * Kp + (size_t)tn * BN;
    const int real_rows = T - tm * BM;   // rows of this tile that hold tiles of a board
#pragma unroll
    for (int part = 0; part < EP_PARTS; part++) {
#pragma unroll
        for (int i = 0; i < MB; i++) {
            const int row0 = wy * WM + i * 32;      // first tile row of this MFMA block
            if (row0 / PROWS == part) {             // uniform per wave
#pragma unroll
                for (int j = 0; j < NB; j++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        typename Quad<P>::type v;
#pragma unroll
                        for (int e = 0; e < 4; e++) v[e] = to_storage<P>(acc[i][j][q * 4 + e]);
                        *reinterpret_cast<typename Quad<P>::type*>(
                            &smem[(row0 - part * PROWS + crow) * CROW + wx * WN + j * 32 + 8 * q +
                                  ccol]) = v;
                    }
            }
        }
        __syncthreads();
#pragma unroll 4
        for (int q = tid; q < PROWS * CPR; q += NT) {
            const int row = q / CPR, ch = q - row * CPR;
            if (part * PROWS + row < real_rows)   // padding rows are never read back
                *reinterpret_cast<int4v*>(Mg + (size_t)(part * PROWS + row) * Kp + ch * EPC) =
                    *reinterpret_cast<const int4v*>(&smem[row * CROW + ch * EPC]);
        }
        __syncthreads();
    }
}

template <typename P, int BN, int NK>
static void launch_gemm_nk(const P* V, const P* U, P* M, int tiles_m, int Tp, int Cp, int Kp,
                           hipStream_t s, LaunchTimer* t) {
    const int tiles_n = Kp / BN;
    const int n_items = kPos * tiles_m * tiles_n;
    int seg = (n_items + 7) / 8;
    seg = (seg + tiles_n - 1) / tiles_n * tiles_n;  // keep the column tiles of a row tile together
    if constexpr (NK >= 2 && (NK % 2) == 0 && BN == 128) {
        // two resident workgroups on each of a die's 32 compute units
        const int wg_per_xcd = seg < 64 ? seg : 64;
        launch(wino_gemm_persistent_k<P, kGemmBM, BN, NK>, dim3(8 * wg_per_xcd), dim3(256), s, t,
               V, U, M, Tp, Cp, Kp, tiles_m, tiles_n, seg, wg_per_xcd);
    } else {
        launch(wino_gemm_k<P, kGemmBM, BN, NK>, dim3(8 * seg), dim3(256), s, t, V, U, M, Tp, Cp,
               Kp, tiles_m, tiles_n, seg);
    }
}

// Channel counts are multiples of 64, so the number of 128-byte k-slices is
// Cp/64 for fp16 and Cp/32 for fp32; 1..8, 10, 12, 14 and 16 slices are instantiated
// (every width up to 512 channels in both types, 640..1024 by 128 in fp16).
template <typename P, int BN>
static void launch_gemm_bn(const P* V, const P* U, P* M, int tiles_m, int Tp, int Cp, int Kp,
                           hipStream_t s, LaunchTimer* t) {
    constexpr int BK = 128 / (int)sizeof(P);
    switch (Cp / BK) {
#define LZ_NK(N) case N: launch_gemm_nk<P, BN, N>(V, U, M, tiles_m, Tp, Cp, Kp, s, t); return;
        LZ_NK(1) LZ_NK(2) LZ_NK(3) LZ_NK(4) LZ_NK(5) LZ_NK(6) LZ_NK(7) LZ_NK(8)
        LZ_NK(10) LZ_NK(12) LZ_NK(14) LZ_NK(16)
#undef LZ_NK
        default: break;
    }
    // the pipe refuses such widths at creation (gemm_supports_channels)
    throw std::invalid_argument("no GEMM instantiated for this channel count");
}

// The 256 x 256 tile computed as two 128-row passes.  The stores of the first
// pass drain while the second pass streams its operands, so only half of the
// output is written with nothing else in flight; the price is that the U tile
// is read twice (the second time from L2).  The operand loads of the second
// pass are issued before the first pass's output leaves, and a second pass
// that holds only padding rows is skipped.
template <typename P, int NK, int HM>
__global__ __launch_bounds__(512) void wino_gemm_split_k(const P* __restrict__ V,
                                                         const P* __restrict__ U,
                                                         P* __restrict__ M, int T, int Tp, int Cp,
                                                         int Kp, int tiles_m, int tiles_n, int seg) {
    constexpr int BM = 256, BN = 256, NT = 512;
    constexpr int PASSES = BM / HM;
    constexpr int EPC = 16 / sizeof(P);
    constexpr int BK = 128 / sizeof(P);
    constexpr int ROW = BK + EPC;
    constexpr int WM = HM / 2, WN = 64;    // per-wave tile, waves laid out 2 (rows) x 4 (columns)
    constexpr int MB = WM / 32, NB = WN / 32;
    constexpr int A_CH = HM * 8 / NT, B_CH = BN * 8 / NT;
    constexpr int CROW = BN + EPC;
    constexpr int STAGE = (HM + BN) * ROW;
    constexpr int PROWS = sizeof(P) == 2 ? 64 : 32;
    constexpr int EP_PARTS = HM / PROWS;
    static_assert(PROWS * CROW <= STAGE, "output staging does not fit a stage");
    static_assert(HM % 64 == 0 && EP_PARTS >= 1, "pass height");

    __shared__ __attribute__((aligned(16))) P smem[2 * STAGE];

    const int n_items = kPos * tiles_m * tiles_n;
    const int xcd = blockIdx.x & 7;
    const int item = xcd * seg + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= seg || item >= n_items) return;
    const int tn = item % tiles_n;
    const int rest = item / tiles_n;
    const int tm = rest % tiles_m;
    const int p = rest / tiles_m;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wy = wave >> 2, wx = wave & 3;
    const int lrow = tid >> 3, lch = tid & 7;   // 64 rows per pass of the workgroup
    const P* Bg = U + ((size_t)p * Kp + (size_t)tn * BN + lrow) * Cp + lch * EPC;
    const int rot = p % NK;
    const int frow = lane & 31, fk = (lane >> 5) * EPC;
    const int ccol = 4 * (lane >> 5), crow = lane & 31;
    constexpr int CPR = BN / EPC;

    int4v ra[2][A_CH], rb[2][B_CH];
    const P* Ag[A_CH];
    auto set_rows = [&](int half) {
#pragma unroll
        for (int i = 0; i < A_CH; i++) {
            const int row = min(tm * BM + half * HM + lrow + i * 64, T - 1);
            Ag[i] = V + ((size_t)p * Tp + row) * Cp + lch * EPC;
        }
    };
    auto gload = [&](int st, int k0) {
#pragma unroll
        for (int i = 0; i < A_CH; i++)
            ra[st][i] = *reinterpret_cast<const int4v*>(Ag[i] + k0);
#pragma unroll
        for (int i = 0; i < B_CH; i++)
            rb[st][i] = *reinterpret_cast<const int4v*>(Bg + (size_t)(i * 64) * Cp + k0);
    };
    auto lstore = [&](int st, int buf) {
        P* As = smem + buf * STAGE;
        P* Bs = As + HM * ROW;
#pragma unroll
        for (int i = 0; i < A_CH; i++)
            *reinterpret_cast<int4v*>(&As[(lrow + i * 64) * ROW + lch * EPC]) = ra[st][i];
#pragma unroll
        for (int i = 0; i < B_CH; i++)
            *reinterpret_cast<int4v*>(&Bs[(lrow + i * 64) * ROW + lch * EPC]) = rb[st][i];
    };

    const int real_rows = T - tm * BM;          // rows of the tile that belong to boards
    const int halves = min(PASSES, (real_rows + HM - 1) / HM);  // uniform over the workgroup

    set_rows(0);
    gload(0, rotated_slice(0, rot, NK) * BK);
    if (NK > 1) gload(1, rotated_slice(1, rot, NK) * BK);

#pragma unroll
    for (int half = 0; half < PASSES; half++) {
        if (half < halves) {
            float16v acc[MB][NB];
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int j = 0; j < NB; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

            lstore(0, 0);
            __syncthreads();
#pragma unroll
            for (int k = 0; k < NK; k++) {
                const int h = k & 1;
                if (k + 2 < NK) {
                    gload(h, rotated_slice(k + 2, rot, NK) * BK);
                    __builtin_amdgcn_sched_barrier(0);
                } else if (half + 1 < halves) {
                    // the first slices of the next pass take the free register stages
                    if (k + 2 == NK) set_rows(half + 1);
                    gload(h, rotated_slice(k + 2 - NK, rot, NK) * BK);
                    __builtin_amdgcn_sched_barrier(0);
                }
                const P* As = smem + h * STAGE;
                const P* Bs = As + HM * ROW;
#pragma unroll
                for (int kc = 0; kc < 4; kc++) {
                    int4v fa[MB], fb[NB];
#pragma unroll
                    for (int i = 0; i < MB; i++)
                        fa[i] = *reinterpret_cast<const int4v*>(
                            &As[(wy * WM + i * 32 + frow) * ROW + kc * 2 * EPC + fk]);
#pragma unroll
                    for (int j = 0; j < NB; j++)
                        fb[j] = *reinterpret_cast<const int4v*>(
                            &Bs[(wx * WN + j * 32 + frow) * ROW + kc * 2 * EPC + fk]);
#pragma unroll
                    for (int i = 0; i < MB; i++)
#pragma unroll
                        for (int j = 0; j < NB; j++)
                            acc[i][j] = Mma<P>::run(fb[j], fa[i], acc[i][j]);
                }
                if (k + 1 < NK) lstore(h ^ 1, h ^ 1);
                __syncthreads();
            }

            // Output of this pass: PROWS rows at a time through LDS, out in 16-byte pieces.
            P* Mg = M + ((size_t)p * Tp + (size_t)tm * BM + half * HM) * Kp + (size_t)tn * BN;
            const int rows_here = real_rows - half * HM;
#pragma unroll
            for (int part = 0; part < EP_PARTS; part++) {
#pragma unroll
                for (int i = 0; i < MB; i++) {
                    const int row0 = wy * WM + i * 32;
                    if (row0 / PROWS == part) {     // uniform per wave
#pragma unroll
                        for (int j = 0; j < NB; j++)
#pragma unroll
                            for (int q = 0; q < 4; q++) {
                                typename Quad<P>::type v;
#pragma unroll
                                for (int e = 0; e < 4; e++)
                                    v[e] = to_storage<P>(acc[i][j][q * 4 + e]);
                                *reinterpret_cast<typename Quad<P>::type*>(
                                    &smem[(row0 - part * PROWS + crow) * CROW + wx * WN + j * 32 +
                                          8 * q + ccol]) = v;
                            }
                    }
                }
                __syncthreads();
#pragma unroll 4
                for (int q = tid; q < PROWS * CPR; q += NT) {
                    const int row = q / CPR, ch = q - row * CPR;
                    if (part * PROWS + row < rows_here)
                        *reinterpret_cast<int4v*>(Mg + (size_t)(part * PROWS + row) * Kp +
                                                  ch * EPC) =
                            *reinterpret_cast<const int4v*>(&smem[row * CROW + ch * EPC]);
                }
                __syncthreads();
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Filter-stationary streaming GEMM in fp32 (v_mfma_f32_32x32x2_f32, a sixteenth of the fp16
// matrix rate: this kernel is bound by the matrix pipe, not by the stream).  One work-group of
// NW wavefronts (8 at 256 filters, 6 / 4 at 192 / 128) owns one Winograd position and a run of
// consecutive 32-row blocks of V; wavefront w owns output channels 32w..32w+31 and keeps its
// share of U_p -- 32 channels x Cp input channels -- in Cp/2 registers per lane for the whole
// kernel, already in the order the matrix instruction wants it.  V streams through: a 32-row
// block (all Cp input channels, so the contraction of those rows completes in one step) is
// requested kStreamAhead steps ahead into registers and passes through a three-stage LDS ring,
// where all wavefronts read it as their column operand, 4 matrix instructions per 16-byte
// fragment read.  The contraction index is dealt so that one 16-byte read serves four
// instructions: in instruction 4j + i, lanes 0..31 hold input channel 8j + i and lanes 32..63
// channel 8j + 4 + i, of U (rows) and of V (columns) alike.
//
// Output: register r of lane l of a 32x32 accumulator holds row 8(r/4) + 4(l/32) + r%4
// of the row operand.  The row operand is U, and the host stores U's channels permuted
// (gemm_stream_channel) so that this lane's sixteen registers are the channels
// 16(r/8) + 8(l/32) + r%8 of the wavefront's 32, i.e. two runs of eight.  The block's result
// goes through a single LDS copy (two barriers per step are little beside 128 matrix
// instructions) and leaves as whole rows, 1 KiB per store instruction, write-through (sc0 sc1):
// whole lines leave for memory while the kernel runs, instead of collecting as dirty lines in
// the L2 that the end of the kernel has to flush with nothing else in flight.  (Stored straight
// from the accumulators instead, 64 bytes per lane with write-back stores and one barrier per
// step, the kernel is slower: 87 against 83 us per launch at 64 boards and 256 filters, 28
// against 24 at 128 filters.)
//
// Uf layout: [36][Kp/32][Cp/8][64 lanes][4 floats]; lane l of fragment (p, wb, j) holds
// U_p[32 wb + gemm_stream_channel(l % 32)][8 j + 4 (l / 32) + 0..3], so every operand load of a
// wavefront is one contiguous KiB.
constexpr int kStreamBlocks = 16;  // most 32-row blocks per work-group (steps of the pipeline)
constexpr int kStreamAhead = 2;    // blocks requested ahead of the one being multiplied

__host__ __device__ constexpr int gemm_stream_channel(int i) {
    // i = 8q + 4h + e  ->  16 (q / 2) + 8 h + 4 (q % 2) + e
    return 16 * (i >> 4) + 8 * ((i >> 2) & 1) + 4 * ((i >> 3) & 1) + (i & 3);
}

template <int NK8, int NBLK, int NW>
__global__ __launch_bounds__(64 * NW) void wino_gemm_stream32_k(const float* V,   // may be M
                                                                const float* __restrict__ Uf,
                                                                float* M, int T,
                                                                int Tp, int Kp, int chunks,
                                                                int nblk_total, int seg) {
    constexpr int D = kStreamAhead;
    constexpr int NT = 64 * NW;
    constexpr int CW = 32 * NW;
    constexpr int Cp = NK8 * 8;
    constexpr int CPRW = Cp / 4;                 // 16-byte chunks per row
    constexpr int NCH = 32 * CPRW;               // chunks per block
    constexpr int CH = (NCH + NT - 1) / NT;
    constexpr bool FULL = NCH % NT == 0;
    constexpr int ROWE = Cp + 4;                 // padded LDS row (floats)
    constexpr int STAGE = 32 * ROWE;
    constexpr int OROW = CW + 4;
    static_assert(D == 2, "pipeline shape");

    __shared__ __attribute__((aligned(16))) float smem[3 * STAGE + 32 * OROW];
    float* const obuf = smem + 3 * STAGE;

    const int n_items = kPos * chunks;
    const int xcd = blockIdx.x & 7;
    const int item = xcd * seg + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= seg || item >= n_items) return;
    const int ch = item % chunks;
    const int p = item / chunks;
    const int blk0 = (ch * nblk_total) / chunks;
    const int blk1 = ((ch + 1) * nblk_total) / chunks;
    const int nreal = blk1 - blk0;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hh = lane >> 5, jrow = lane & 31;

    int lrow[CH], lcc[CH];
    bool lval[CH];
#pragma unroll
    for (int i = 0; i < CH; i++) {
        const int idx = tid + i * NT;
        lval[i] = FULL || idx < NCH;
        lrow[i] = (idx / CPRW) & 31;
        lcc[i] = idx % CPRW;
    }
    const float* Vp = V + (size_t)p * Tp * Cp;

    int4v st[D][CH];
    auto gload = [&](int slot, int s) {
        // requests past the last real block re-read that block (cache hits, never used)
        const int blk = blk0 + (s < nreal ? s : nreal - 1);
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const int row = min(blk * 32 + lrow[i], T - 1);
            if (lval[i])
                st[slot][i] =
                    *reinterpret_cast<const int4v*>(Vp + (size_t)row * Cp + lcc[i] * 4);
        }
    };
    auto lstore = [&](int slot, int buf) {
        float* S = smem + buf * STAGE;
#pragma unroll
        for (int i = 0; i < CH; i++)
            if (lval[i]) *reinterpret_cast<int4v*>(&S[lrow[i] * ROWE + lcc[i] * 4]) = st[slot][i];
    };

    gload(0, 0);
    if (NBLK > 1) gload(1, 1);
    float4v u[NK8];
    {
        const float* Up = Uf + ((((size_t)p * (Kp / 32) + wave) * NK8) * 64 + lane) * 4;
#pragma unroll
        for (int j = 0; j < NK8; j++)
            u[j] = *reinterpret_cast<const float4v*>(Up + (size_t)j * 64 * 4);
    }
    lstore(0, 0);
    if (NBLK > 1) lstore(1, 1);
    __syncthreads();

    // rows past the last tile get an offset outside the buffer and are dropped
    const size_t m_bytes = (size_t)T * Kp * sizeof(float);
    const __amdgpu_buffer_rsrc_t rM = make_rsrc(M + (size_t)p * Tp * Kp, m_bytes);
    const unsigned m_rowb = (unsigned)Kp * 4u;
    constexpr int PPR = CW / 4;                  // 16-byte pieces per row
    auto send_rows = [&](int s) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int piece = tid + i * NT;
            const int r = piece / PPR;
            const int cc = piece - r * PPR;
            const int4v v = *reinterpret_cast<const int4v*>(obuf + r * OROW + cc * 4);
            const unsigned row = (unsigned)((blk0 + s) * 32 + r);
            __builtin_amdgcn_raw_buffer_store_b128(v, rM, row * m_rowb + (unsigned)cc * 16u, 0,
                                                   kStoreThrough);
        }
    };

    const int frag = jrow * ROWE + hh * 4;
    // NBLK bounds the steps; a work-group leaves after its own nreal (the same for all its
    // threads): a step costs 128 matrix instructions here, so the blocks of a position are
    // split evenly over the work-groups (gemm_stream_split) and none runs an idle step.
    int last = 0;
#pragma unroll
    for (int s = 0; s < NBLK; s++) {
        if (s >= nreal) break;
        last = s;
        if (s + D < NBLK) gload(s % D, s + D);
        if (s > 0) send_rows(s - 1);
        // the requests above stay above: left to itself the scheduler moves them down to the
        // LDS stores that consume them, and a step then ends in a wait for memory
        __builtin_amdgcn_sched_barrier(0);
        const float* S = smem + (s % 3) * STAGE + frag;
        float16v acc;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = 0.0f;
        // two fragment registers in turn: the read that refills one is issued behind the
        // four instructions that used it and has the other's four to arrive in
        static_assert(NK8 % 2 == 0, "fragments are read in pairs");
        float4v fa = *reinterpret_cast<const float4v*>(S);
        float4v fb = *reinterpret_cast<const float4v*>(S + 8);
#pragma unroll
        for (int j = 0; j < NK8; j += 2) {
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(u[j].x, fa.x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(u[j].y, fa.y, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(u[j].z, fa.z, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(u[j].w, fa.w, acc, 0, 0, 0);
            if (j + 2 < NK8) fa = *reinterpret_cast<const float4v*>(S + (j + 2) * 8);
            __builtin_amdgcn_sched_barrier(0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(u[j + 1].x, fb.x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(u[j + 1].y, fb.y, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(u[j + 1].z, fb.z, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(u[j + 1].w, fb.w, acc, 0, 0, 0);
            if (j + 3 < NK8) fb = *reinterpret_cast<const float4v*>(S + (j + 3) * 8);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (s + 2 < NBLK) lstore((s + 2) % D, (s + 2) % 3);
        __syncthreads();   // every wavefront has sent the rows of the block before
        float* O = obuf + jrow * OROW + wave * 32 + hh * 8;
        *reinterpret_cast<float4v*>(O) = float4v{acc[0], acc[1], acc[2], acc[3]};
        *reinterpret_cast<float4v*>(O + 4) = float4v{acc[4], acc[5], acc[6], acc[7]};
        *reinterpret_cast<float4v*>(O + 16) = float4v{acc[8], acc[9], acc[10], acc[11]};
        *reinterpret_cast<float4v*>(O + 20) = float4v{acc[12], acc[13], acc[14], acc[15]};
        __syncthreads();
    }
    send_rows(last);
}

// Fragment-order copy of one layer's filters for the streaming kernel: src is the reference
// layout [36][C][F] (F fastest), dst [36][Kp/32][Cp/8][64][4], zero padded.
void build_stream_filters(const float* src, int C, int F, int Cp, int Kp, float* dst) {
    constexpr int G = 4;                       // values per lane and fragment
    const int nfr = Cp / (2 * G), nwb = Kp / 32;
    for (int p = 0; p < kPos; p++)
        for (int wb = 0; wb < nwb; wb++)
            for (int fr = 0; fr < nfr; fr++)
                for (int l = 0; l < 64; l++) {
                    const int k = 32 * wb + gemm_stream_channel(l & 31);
                    for (int e = 0; e < G; e++) {
                        const int c = 2 * G * fr + G * (l >> 5) + e;
                        float v = 0.0f;
                        if (c < C && k < F) v = src[((size_t)p * C + c) * F + k];
                        dst[((((size_t)p * nwb + wb) * nfr + fr) * 64 + l) * G + e] = v;
                    }
                }
}

// fp32 -> storage type on the device (round to nearest even, as a host cast would): the
// filters of an fp16 net are laid out on the host in fp32 and converted here, which takes
// the conversion of 2 x 191 M values out of push_weights' host time for a 40 x 256 net.
__global__ __launch_bounds__(256) void convert_filters_k(const float* __restrict__ src,
                                                         half_t* __restrict__ dst, size_t n) {
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride)
        dst[i] = (half_t)src[i];
}

void convert_filters(const float* src, half_t* dst, size_t n, hipStream_t s) {
    const size_t blocks = (n + 255) / 256;
    hipLaunchKernelGGL(convert_filters_k, dim3((unsigned)(blocks < 2048 ? blocks : 2048)),
                       dim3(256), 0, s, src, dst, n);
}

// The split of a position's 32-row blocks over work-groups: as many work-groups per
// position as one round over the 256 compute units allows (7 at one column tile: 252
// work-groups), fewer when there are fewer blocks, more when a work-group would otherwise
// get more than kStreamBlocks.  A work-group takes floor or ceil of blocks / chunks and
// leaves after its own; the kernel is instantiated for the next power of two.
struct StreamSplit { int chunks, nb; };
static StreamSplit gemm_stream_split(int T, int Kp) {
    const int nblk = (T + 31) / 32;
    const int per_pos = 256 / (kPos * ((Kp + 255) / 256));
    int chunks = nblk < per_pos ? nblk : per_pos;
    const int least = (nblk + kStreamBlocks - 1) / kStreamBlocks;
    if (chunks < least) chunks = least;
    const int most = (nblk + chunks - 1) / chunks;   // blocks of the largest share
    int nb = 1;
    while (nb < most) nb *= 2;
    return {chunks, nb};
}

// Whether launch_gemm takes the streaming kernel for this shape when it is handed the
// fragment-order filters: input layer (64 padded planes) and tower layers, any batch, of fp32
// nets of 128, 192 and 256 filters (one column tile of Kp / 32 wavefronts).  Tiled -> streaming:
// 256 filters 88 -> 79-83 us per launch at 64 boards, 78 -> 58 at 48, 22 -> 13 at 8; 128 filters
// 27 -> 23 at 64 boards.  At 192 filters six wavefronts sit unevenly on four SIMDs: the
// streaming kernel is ahead up to 24 boards on one lane (15x192 forwards +6 % at 1 board, +11 %
// at 8, +20 % at 16, +10 % at 24; all lanes +4 % at 8, +2 % at 16, -15 % at 24) and behind beyond
// (-4 % at 32, -8 % at 64): gemm_stream_prefers says which kernel family a handle of a given
// batch limit holds the filters for.  One family per handle keeps a position's result
// independent of the batch it is evaluated in.
bool gemm_stream_shape(int T, int Cp, int Kp, int elem_bytes) {
    if (elem_bytes != 4 || T < 1 || !(Cp == 64 || Cp == Kp)) return false;
    return Kp == 128 || Kp == 256 || Kp == 192;
}
bool gemm_stream_prefers(int Kp, int max_batch) { return !(Kp == 192 && max_batch > 16); }

template <int NK8, int NW>
static void launch_gemm_stream32_nk(const float* V, const float* Uf, float* M, int T, int Tp,
                                    int Kp, hipStream_t s, LaunchTimer* t) {
    const int nblk = (T + 31) / 32;
    const StreamSplit sp = gemm_stream_split(T, Kp);
    const int nb = sp.nb, chunks = sp.chunks;
    const int seg = (kPos * chunks + 7) / 8;
    const dim3 grid(8 * seg), block(64 * NW);
    switch (nb) {
        case 1: launch(wino_gemm_stream32_k<NK8, 1, NW>, grid, block, s, t, V, Uf, M, T, Tp, Kp, chunks, nblk, seg); break;
        case 2: launch(wino_gemm_stream32_k<NK8, 2, NW>, grid, block, s, t, V, Uf, M, T, Tp, Kp, chunks, nblk, seg); break;
        case 4: launch(wino_gemm_stream32_k<NK8, 4, NW>, grid, block, s, t, V, Uf, M, T, Tp, Kp, chunks, nblk, seg); break;
        case 8: launch(wino_gemm_stream32_k<NK8, 8, NW>, grid, block, s, t, V, Uf, M, T, Tp, Kp, chunks, nblk, seg); break;
        default: launch(wino_gemm_stream32_k<NK8, 16, NW>, grid, block, s, t, V, Uf, M, T, Tp, Kp, chunks, nblk, seg); break;
    }
}

template <int NW>
static void launch_gemm_stream32_nw(const float* V, const float* Uf, float* M, int T, int Tp,
                                    int Cp, int Kp, hipStream_t s, LaunchTimer* t) {
    if (Cp == 64)
        launch_gemm_stream32_nk<8, NW>(V, Uf, M, T, Tp, Kp, s, t);
    else
        launch_gemm_stream32_nk<4 * NW, NW>(V, Uf, M, T, Tp, Kp, s, t);
}

static void launch_gemm_stream(const float* V, const float* Uf, float* M, int T, int Tp, int Cp,
                               int Kp, hipStream_t s, LaunchTimer* t) {
    if (Kp == 256)
        launch_gemm_stream32_nw<8>(V, Uf, M, T, Tp, Cp, Kp, s, t);
    else if (Kp == 192)
        launch_gemm_stream32_nw<6>(V, Uf, M, T, Tp, Cp, Kp, s, t);
    else
        launch_gemm_stream32_nw<4>(V, Uf, M, T, Tp, Cp, Kp, s, t);
}

template <typename P, int NK>
static void launch_gemm_big(const P* V, const P* U, P* M, int T, int tiles_m, int Tp, int Cp,
                            int Kp, hipStream_t s, LaunchTimer* t) {
    const int tiles_n = Kp / 256;
    const int n_items = kPos * tiles_m * tiles_n;
    int seg = (n_items + 7) / 8;
    seg = (seg + tiles_n - 1) / tiles_n * tiles_n;
    // Two 128-row passes wherever the k-pipeline has at least two slices to keep
    // the register stages busy across the pass boundary (measured 3 % faster than
    // one 256-row pass at 256 filters); the single-slice input layer keeps one pass,
    // and so do fp16 nets from 512 filters, where the GEMM is bound by the matrix and
    // LDS pipes and the 128 x 64 wave tile of the single pass reads less LDS per
    // instruction (measured 3 % faster at 512 filters, 6 % at 1024).
    if (NK >= 2 && !(sizeof(P) == 2 && NK >= 8))
        launch(wino_gemm_split_k<P, NK, 128>, dim3(8 * seg), dim3(512), s, t, V, U, M, T, Tp, Cp,
               Kp, tiles_m, tiles_n, seg);
    else
        launch(wino_gemm_big_k<P, NK>, dim3(8 * seg), dim3(512), s, t, V, U, M, T, Tp, Cp, Kp,
               tiles_m, tiles_n, seg);
}

// Channel counts (multiples of 64) for which a k-slice pipeline is instantiated:
// 1..8, 10, 12, 14 and 16 slices of 128 bytes.
template <typename P> bool gemm_supports_channels(int Cp) {
    constexpr int BK = 128 / (int)sizeof(P);
    if (Cp < 64 || Cp % 64 != 0) return false;
    const int nk = Cp / BK;
    return (nk >= 1 && nk <= 8) || nk == 10 || nk == 12 || nk == 14 || nk == 16;
}
template bool gemm_supports_channels<float>(int);
template bool gemm_supports_channels<half_t>(int);

// T = number of real tile rows (25 per board); Tp (the row count of V and M)
// must be a multiple of 256.
template <typename P>
void launch_gemm(const P* V, const P* U, const P* Uf, P* M, int T, int Tp, int Cp, int Kp,
                 hipStream_t s, LaunchTimer* t) {
    constexpr int BK = 128 / (int)sizeof(P);
    const int nk = Cp / BK;
    if constexpr (sizeof(P) == 4) {
        if (Uf != nullptr && gemm_stream_shape(T, Cp, Kp, (int)sizeof(P))) {
            launch_gemm_stream(V, Uf, M, T, Tp, Cp, Kp, s, t);
            return;
        }
    }
    // The 256 x 256 tile pays off once its tiles can occupy most of the 256 compute units
    // (measured at 256 filters: from 6 row tiles = 216 work-groups, batch 52; with 5 = 180 the
    // 128 x 128 tiles are 2 % ahead; fp32 keeps the earlier hand-over at 160).
    const int big_rows = (T + 255) / 256;
    if (Kp % 256 == 0 && big_rows * (Kp / 256) * kPos >= (sizeof(P) == 2 ? 200 : 160)) {
        switch (nk) {
#define LZ_BIG(N) case N: launch_gemm_big<P, N>(V, U, M, T, big_rows, Tp, Cp, Kp, s, t); return;
            LZ_BIG(1) LZ_BIG(2) LZ_BIG(4) LZ_BIG(8) LZ_BIG(16)
#undef LZ_BIG
            default: break;
        }
    }
    const int tiles_m = (T + kGemmBM - 1) / kGemmBM;
    // Below the 256 x 256 tile, fp16: the 128 x 64 tile, three work-groups to a compute unit,
    // gives the chip the most independent pieces (measured at 256 filters: ahead of 128 x 128
    // tiles, two to a unit, at every batch up to 40, by 4 % at 21 and 1 % at 40); 128 x 128
    // tiles take over where that would be more than two rounds of the narrow ones.  fp32 (two
    // narrow work-groups to a unit): 128 x 128 once there are more than 320 of them.
    if (Kp % 128 == 0 && kPos * tiles_m * (Kp / 128) > (sizeof(P) == 2 ? 600 : 320))
        launch_gemm_bn<P, 128>(V, U, M, tiles_m, Tp, Cp, Kp, s, t);
    else
        launch_gemm_bn<P, 64>(V, U, M, tiles_m, Tp, Cp, Kp, s, t);
}

// ---------------------------------------------------------------------------
// 1x1 policy (2 planes) and value (1 plane) convolutions in one pass over the
// last activation (reference src/CPUPipe.cpp:424-427).  Sixteen lanes to a
// board point up to 128 channels and 32 beyond, eight channels a lane and load, then a butterfly
// reduction.  (With a wavefront to a point and a channel a lane the number of wavefronts was the
// bound: 256 filters, 200 boards 25 us, now 13; 128 filters, 37 boards 5.4 and 3.5.)
template <typename P, int LP>
__global__ __launch_bounds__(256) void head_conv_k(const P* __restrict__ act, bool padded,
                                                   const float* __restrict__ w3,
                                                   float out_scale, float* __restrict__ pol,
                                                   float* __restrict__ val, int n, int Cp) {
    typedef P P8 __attribute__((ext_vector_type(8)));
    const int gp = (blockIdx.x * 256 + threadIdx.x) / LP;
    const int lane = threadIdx.x % LP;
    if (gp >= n * kPts) return;
    const int b = gp / kPts, pt = gp - b * kPts;
    const P* a = act + plane_index(padded, b, pt) * Cp;
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f;
    for (int c = lane * 8; c < Cp; c += LP * 8) {
        const P8 x = *reinterpret_cast<const P8*>(a + c);
        const float8v w0 = *reinterpret_cast<const float8v*>(w3 + c);
        const float8v w1 = *reinterpret_cast<const float8v*>(w3 + Cp + c);
        const float8v w2 = *reinterpret_cast<const float8v*>(w3 + 2 * Cp + c);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            s0 += (float)x[e] * w0[e];
            s1 += (float)x[e] * w1[e];
            s2 += (float)x[e] * w2[e];
        }
    }
#pragma unroll
    for (int off = LP / 2; off > 0; off >>= 1) {
        s0 += __shfl_xor(s0, off);
        s1 += __shfl_xor(s1, off);
        s2 += __shfl_xor(s2, off);
    }
    if (lane == 0) {
        pol[(size_t)b * 2 * kPts + pt] = s0 * out_scale;
        pol[(size_t)b * 2 * kPts + kPts + pt] = s1 * out_scale;
        val[(size_t)b * kPts + pt] = s2 * out_scale;
    }
}

template <typename P>
void launch_head_conv(const P* act, bool padded, const float* w3, float out_scale, float* pol,
                      float* val, int n, int Cp, hipStream_t s, LaunchTimer* t) {
    const int points = n * kPts;
    if (Cp > 128)
        launch(head_conv_k<P, 32>, dim3((points + 7) / 8), dim3(256), s, t, act, padded, w3,
               out_scale, pol, val, n, Cp);
    else
        launch(head_conv_k<P, 16>, dim3((points + 15) / 16), dim3(256), s, t, act, padded, w3,
               out_scale, pol, val, n, Cp);
}

// ---------------------------------------------------------------------------
template <typename P>
__global__ __launch_bounds__(256) void absmax_k(const P* __restrict__ x, size_t count,
                                                float* out) {
    float m = 0.0f;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < count;
         i += (size_t)gridDim.x * 256) {
        const float v = fabsf((float)x[i]);
        // NaN-propagating max so that a poisoned buffer is visible to the host.
        m = (v != v) ? INFINITY : fmaxf(m, v);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if ((threadIdx.x & 63) == 0) atomicMax(reinterpret_cast<int*>(out), __float_as_int(m));
}

template <typename P>
void launch_absmax(const P* x, size_t count, float* out, hipStream_t s) {
    size_t blocks = (count + 255) / 256;
    if (blocks > 2048) blocks = 2048;
    if (blocks == 0) blocks = 1;
    hipLaunchKernelGGL(absmax_k<P>, dim3((unsigned)blocks), dim3(256), 0, s, x, count, out);
}

// ---------------------------------------------------------------------------
// Head arithmetic above the pipe boundary (reference src/Network.cpp:833-851):
// policy: BN+ReLU on 2 planes -> FC 722->362 -> softmax(./temperature)
// value : BN+ReLU on 1 plane  -> FC 361->256 + ReLU -> FC 256->1 -> tanh
// One workgroup of 256 threads per position; FC rows are read by whole
// wavefronts (coalesced) and reduced with a butterfly.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
    return v;
}

// The two large fully connected layers -- policy 722 -> 362 and value 361 -> 256 -- are
// matrix products over the batch, [n x K] . [K x N], and run on the matrix cores in fp32
// (v_mfma_f32_32x32x2_f32: fp32 operands, fp32 accumulate).  One work-group computes a
// 32-position x 32-output tile over a quarter of the contraction index: its share of the 32
// input rows (batch norm and ReLU applied on the way) is staged in LDS once, the four
// wavefronts split the quarter four ways, and their partial tiles meet in LDS.  The quarters
// meet in the second kernel, which adds them and finishes: softmax over the 362 logits, and FC
// 256 -> 1 + tanh.  What bounds it is latency, not work: one round trip for the operands, then
// 24 dependent matrix instructions of 64 cycles.  With the whole index in one work-group these
// were 92, behind 92 values of the planes per thread with a division each; a call of up to 37
// positions took 13.2 us for this kernel, now 4.2 to 4.7, and one of 200 now takes 6.4.
// The weights are held in the operand order of the instruction (head_fc_fragments): lane l of
// k-step s supplies W^T[2s + l/32][32 cb + l%32], four consecutive steps per 16-byte load, so a
// wavefront's load is one contiguous KiB.
constexpr int kHeadQuarters = 4;    // work-groups that share a tile's contraction index
constexpr int kHeadStepsPol = 24;   // k-steps (of 2) per wavefront: 16 * 24 * 2 = 768 >= 722
constexpr int kHeadStepsVal = 12;   // 16 * 12 * 2 = 384 >= 361
constexpr int kHeadColsPol = 12;    // 32-wide output blocks: 384 >= 362
constexpr int kHeadColsVal = 8;     // 256

size_t head_work_count(int n) { return (size_t)kHeadQuarters * n * (362 + 256); }

size_t head_fc_fragment_count(bool policy) {
    return (size_t)(policy ? kHeadColsPol * kHeadStepsPol : kHeadColsVal * kHeadStepsVal) * 4 *
           kHeadQuarters * 64;
}

// W [N][K] row-major (as the network facade holds it) -> fragment order
// [col block][quarter][wavefront 4][steps/4][lane 64][4 consecutive steps], zero padded.
void head_fc_fragments(const float* W, bool policy, float* dst) {
    const int K = policy ? 2 * kPts : kPts, N = policy ? 362 : 256;
    const int steps = policy ? kHeadStepsPol : kHeadStepsVal;
    const int cols = policy ? kHeadColsPol : kHeadColsVal;
    for (int cb = 0; cb < cols; cb++)
        for (int q = 0; q < 4 * kHeadQuarters; q++)
            for (int g = 0; g < steps / 4; g++)
                for (int l = 0; l < 64; l++)
                    for (int e = 0; e < 4; e++) {
                        const int step = q * steps + g * 4 + e;
                        const int k = 2 * step + (l >> 5), j = cb * 32 + (l & 31);
                        const float v = (k < K && j < N) ? W[(size_t)j * K + k] : 0.0f;
                        const size_t share = (size_t)cb * 4 * kHeadQuarters + q;
                        dst[((share * (steps / 4) + g) * 64 + l) * 4 + e] = v;
                    }
}

// One layer's share of heads_fc_k.  Everything a work-group reads has been out of the caches
// since the last call (a tower of 81 layers ran in between) and the planes have just been
// written on other dies, so a round trip to memory takes ~2 us here: the wavefront's whole
// share of the weights and, per thread, its 24 or 16 values of the planes are requested before the
// first is used.  out: [kHeadQuarters][n][N] partial sums.
template <bool POL>
__device__ __forceinline__ void heads_fc_body(float* xs, const float* __restrict__ src,
                                              const HeadParams& hp, float* __restrict__ out,
                                              int cb, int quarter, int r0, int n) {
    constexpr int STEPS = POL ? kHeadStepsPol : kHeadStepsVal;
    constexpr int G = STEPS / 4;             // 16-byte weight loads per lane
    constexpr int KQ = 4 * STEPS * 2;        // contraction length of a quarter
    constexpr int KK = POL ? 2 * kPts : kPts;
    constexpr int N = POL ? 362 : 256;
    constexpr int ROW = KQ + 1;              // odd row length: conflict-free column reads
    constexpr int J = (KQ + 63) / 64, R = 8; // a lane's values per row, a wavefront's rows
    const int tid = threadIdx.x, lane = tid & 63;
    const int q = __builtin_amdgcn_readfirstlane(tid >> 6);

    const float4v* wf = reinterpret_cast<const float4v*>(POL ? hp.ip_pol_wf : hp.ip1_val_wf) +
                        ((((size_t)cb * kHeadQuarters + quarter) * 4 + q) * G) * 64 + lane;
    float4v w[G];
#pragma unroll
    for (int g = 0; g < G; g++) w[g] = wf[(size_t)g * 64];

    // 32 rows of the layer's input: batch norm + ReLU of the raw head planes, zero padded
    const float s0 = POL ? hp.bn_pol_scale[0] : hp.bn_val_scale[0];
    const float m0 = POL ? hp.bn_pol_mean[0] : hp.bn_val_mean[0];
    const float s1 = POL ? hp.bn_pol_scale[1] : s0;
    const float m1 = POL ? hp.bn_pol_mean[1] : m0;
    float x[R][J];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int j = 0; j < J; j++) {
            const int row = r0 + q * R + r, c = lane + 64 * j, k = quarter * KQ + c;
            x[r][j] = row < n && c < KQ && k < KK ? src[(size_t)row * KK + k] : 0.0f;
        }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int j = 0; j < J; j++) {
            const int row = r0 + q * R + r, c = lane + 64 * j, k = quarter * KQ + c;
            const bool second = POL && k >= kPts;
            float y = 0.0f;
            if (row < n && k < KK)
                y = fmaxf(0.0f, (second ? s1 : s0) * (x[r][j] - (second ? m1 : m0)));
            if (c < KQ) xs[(q * R + r) * ROW + c] = y;
        }
    __syncthreads();

    float16v acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    const float* xa = xs + (lane & 31) * ROW + q * STEPS * 2 + (lane >> 5);
#pragma unroll
    for (int g = 0; g < G; g++) {
        const float* x = xa + g * 8;
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[0], w[g].x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[2], w[g].y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[4], w[g].z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[6], w[g].w, acc, 0, 0, 0);
    }
    __syncthreads();   // everyone is done with the staged rows: reuse them for the partial tiles

    // register r of lane l holds row 8(r/4) + 4(l/32) + r%4, column l%32
    float* red = xs + q * (32 * 33);
#pragma unroll
    for (int r = 0; r < 16; r++)
        red[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * 33 + (lane & 31)] = acc[r];
    __syncthreads();
    out += (size_t)quarter * n * N;
    for (int i = tid; i < 32 * 32; i += 256) {
        const int r = i >> 5, j = i & 31;
        const int col = cb * 32 + j;
        if (r0 + r < n && col < N)
            out[(size_t)(r0 + r) * N + col] =
                xs[r * 33 + j] + xs[32 * 33 + r * 33 + j] + xs[2 * 32 * 33 + r * 33 + j] +
                xs[3 * 32 * 33 + r * 33 + j];
    }
}

__global__ __launch_bounds__(256) void heads_fc_k(const float* __restrict__ pol,
                                                  const float* __restrict__ val, HeadParams hp,
                                                  float* __restrict__ logits,
                                                  float* __restrict__ hidden, int n) {
    constexpr int STAGE = 32 * (8 * kHeadStepsPol + 1), MEET = 4 * 32 * 33;
    __shared__ float xs[STAGE > MEET ? STAGE : MEET];
    const int tasks = kHeadColsPol + kHeadColsVal;
    const int tile = blockIdx.x / kHeadQuarters, quarter = blockIdx.x % kHeadQuarters;
    const int rb = tile / tasks, task = tile - rb * tasks;
    if (task < kHeadColsPol)
        heads_fc_body<true>(xs, pol, hp, logits, task, quarter, rb * 32, n);
    else
        heads_fc_body<false>(xs, val, hp, hidden, task - kHeadColsPol, quarter, rb * 32, n);
}

// One wavefront per position: softmax over the logits at `temperature`, and the value
// head's second layer + tanh (reference src/Network.cpp:693-712, :846-851).
__global__ __launch_bounds__(256) void heads_finish_k(const float* __restrict__ logits_in,
                                                      const float* __restrict__ hidden,
                                                      HeadParams hp, float temperature,
                                                      float* __restrict__ policy,
                                                      float* __restrict__ logits_out,
                                                      float* __restrict__ value, int n) {
    const int pos = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (pos >= n) return;
    float l[6], m = -INFINITY;
#pragma unroll
    for (int qq = 0; qq < 6; qq++) {
        const int i = lane + 64 * qq;
        l[qq] = -INFINITY;
        if (i < 362) {
            float v = 0.0f;
#pragma unroll
            for (int k = 0; k < kHeadQuarters; k++) v += logits_in[((size_t)k * n + pos) * 362 + i];
            l[qq] = v + hp.ip_pol_b[i];
        }
        m = fmaxf(m, l[qq]);
    }
    m = wave_max(m);
    float e[6], s = 0.0f;
#pragma unroll
    for (int qq = 0; qq < 6; qq++) {
        e[qq] = lane + 64 * qq < 362 ? expf((l[qq] - m) / temperature) : 0.0f;
        s += e[qq];
    }
    s = wave_sum(s);
#pragma unroll
    for (int qq = 0; qq < 6; qq++) {
        const int i = lane + 64 * qq;
        if (i < 362) {
            policy[(size_t)pos * 362 + i] = e[qq] / s;
            if (logits_out != nullptr) logits_out[(size_t)pos * 362 + i] = l[qq];
        }
    }
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int i = lane + 64 * j;
        float v = 0.0f;
#pragma unroll
        for (int k = 0; k < kHeadQuarters; k++) v += hidden[((size_t)k * n + pos) * 256 + i];
        acc += fmaxf(0.0f, v + hp.ip1_val_b[i]) * hp.ip2_val_w[i];
    }
    acc = wave_sum(acc);
    if (lane == 0) value[pos] = tanhf(hp.ip2_val_b[0] + acc);
}

void launch_heads(const float* pol, const float* val, HeadParams hp, float temperature,
                  float* policy, float* logits, float* value, float* work, int n,
                  hipStream_t s) {
    // work: [kHeadQuarters][n][362] of the logits followed by [kHeadQuarters][n][256] of the
    // hidden units
    float* wl = work;
    float* wh = work + (size_t)kHeadQuarters * n * 362;
    const int rbs = (n + 31) / 32;
    hipLaunchKernelGGL(heads_fc_k, dim3(rbs * (kHeadColsPol + kHeadColsVal) * kHeadQuarters),
                       dim3(256), 0, s, pol, val, hp, wl, wh, n);
    hipLaunchKernelGGL(heads_finish_k, dim3((n + 3) / 4), dim3(256), 0, s, wl, wh, hp, temperature,
                       policy, logits, value, n);
}

// ---------------------------------------------------------------------------
#define INSTANTIATE(P)                                                                         \
    template void launch_pack_input<P>(const float*, P*, bool, int, int, int, hipStream_t,     \
                                       LaunchTimer*, const PlaneBorders*);                     \
    template void launch_pack_input_bits<P>(const uint32_t*, P*, bool, int, int, int,          \
                                            uint32_t*, const float*, hipStream_t,              \
                                            LaunchTimer*);                                     \
    template void launch_in_transform<P>(const P*, P*, int, int, int, hipStream_t,             \
                                         LaunchTimer*);                                        \
    template void launch_gemm<P>(const P*, const P*, const P*, P*, int, int, int, int,         \
                                 hipStream_t, LaunchTimer*);                                   \
    template void launch_out_transform<P>(const P*, const P*, P*, const float*, const float*,  \
                                          float, int, int, int, hipStream_t, LaunchTimer*);    \
    template void launch_out_in_transform<P>(const P*, const P*, P*, P*, const float*,         \
                                             const float*, float, int, int, int, hipStream_t,  \
                                             LaunchTimer*);                                    \
    template void launch_head_conv<P>(const P*, bool, const float*, float, float*, float*,     \
                                      int, int, hipStream_t, LaunchTimer*);                    \
    template void launch_absmax<P>(const P*, size_t, float*, hipStream_t);
INSTANTIATE(float)
INSTANTIATE(half_t)

}  // namespace lzhip
