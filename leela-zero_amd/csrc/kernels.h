// Launch interface of the gfx950 kernels of the residual tower.
//
// Device data layouts (P = storage type: float or _Float16):
//   act  [n][361][Cp]        activations, channels fastest ("channels-last"); for direct
//                            convolutions padded: [n + 2][400][Cp], point (y, x) of board b at
//                            cell 400 (b + 1) + 20 (y + 1) + x, every other cell zero
//   V    [36][Tp][Cp]        Winograd-domain input tiles, t = board*25 + by*5 + bx
//   U    [36][Kp][Cp]        Winograd-domain filters, input channel fastest
//   M    [36][Tp][Kp]        per-position GEMM results, output channel fastest
// Cp, Kp are the channel counts padded to a multiple of 64, Tp the tile count
// padded to a multiple of 256.  The contraction index (input channel) is the
// fastest-moving one of both GEMM operands, which is what the MFMA operand
// registers want: each lane fetches 16 contiguous bytes of one row.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace lzhip {

constexpr int kBoard = 19;
constexpr int kPts = 361;
constexpr int kPadCells = 400;   // cells of a board in padded planes
constexpr int kTilesPerBoard = 25;
constexpr int kPos = 36;       // 6x6 Winograd positions
constexpr int kInPlanes = 18;
constexpr int kGemmBM = 128;   // row extent of the standard GEMM tile
constexpr int kTileRowPad = 256;  // V and M row counts (Tp) are multiples of this
// Largest magnitude an activation is stored with in half precision (see act_clamp in
// kernels.hip); the calibration treats a measured maximum at this value as saturated.
constexpr float kActStoreMax = 2040.0f;

// Timing hook: when non-null every launch is bracketed by this event pair
// (device begin/end timestamps of that launch alone).
struct LaunchTimer {
    hipEvent_t start = nullptr, stop = nullptr;
};

// Index of point pt of board b: cell of padded planes, or point of dense ones.
__host__ __device__ static inline size_t plane_index(bool padded, int b, int pt) {
    return padded ? (size_t)(b + 1) * kPadCells + pt + pt / kBoard + 20 : (size_t)b * kPts + pt;
}
static inline size_t padded_cells(int n) { return (size_t)(n + 2) * kPadCells; }
// The padded planes of a forward of n boards, one of w0 and then three of w pieces of 16 bytes to a cell
// one after the other, whose borders the kernel that reads the input is to clear on the way.
struct PlaneBorders {
    int __attribute__((ext_vector_type(4)))* planes = nullptr;
    unsigned n = 0, w0 = 0, w = 0;
};

// NCHW fp32 planes [n][C][361] -> act [n][361][Cp] (channels >= C zero).
// 32-bit words of one position's 18 x 361 input planes packed one bit per value.
constexpr int kInputWords = (18 * 361 + 31) / 32;

// Largest magnitudes (bits of a float) of a layer's planes on every board, what the direct fp32
// convolution scales its operands by: slots[row][2][column] of the tiles of mt points that wrote
// them, for the first and the second board that a tile meets.
struct PeakMap {
    uint32_t* slots = nullptr;
    int mt = 0, tiles_n = 0;
};
// (peaks: null, or 2 n slots of input planes, one tile a board; scale: null, or a factor per plane)
template <typename P>
void launch_pack_input_bits(const uint32_t* bits, P* act, bool padded, int n, int C, int Cp,
                            uint32_t* peaks, const float* scale, hipStream_t s, LaunchTimer* t);
template <typename P>
void launch_pack_input(const float* in, P* act, bool padded, int n, int C, int Cp, hipStream_t s,
                       LaunchTimer* t, const PlaneBorders* borders = nullptr);
// The same with the peaks; padded.
void launch_pack_input_peaks(const float* in, float* act, int n, int C, int Cp, uint32_t* peaks,
                             const float* scale, hipStream_t s, LaunchTimer* t,
                             const PlaneBorders* borders = nullptr);

// act [n][361][Cp] -> V [36][Tp][Cp]
template <typename P>
void launch_in_transform(const P* act, P* V, int n, int Cp, int Tp, hipStream_t s,
                         LaunchTimer* t);

// Whether a GEMM pipeline exists for Cp channels (padded count, multiple of 64).
template <typename P> bool gemm_supports_channels(int Cp);

// M[p][t][k] = sum_c V[p][t][c] * U[p][k][c]
// T = real tile rows (25 per board); Tp = allocated rows, a multiple of kTileRowPad.
// Uf: the same filters in the fragment order of the streaming kernel (see
// build_stream_filters), or null; taken when gemm_stream_shape(T, Cp, Kp, sizeof(P)).
template <typename P>
void launch_gemm(const P* V, const P* U, const P* Uf, P* M, int T, int Tp, int Cp, int Kp,
                 hipStream_t s, LaunchTimer* t);
bool gemm_stream_shape(int T, int Cp, int Kp, int elem_bytes);
// Whether a handle for batches up to max_batch should hold the streaming kernel's filters
// where gemm_stream_shape allows them (measured; see there).
bool gemm_stream_prefers(int Kp, int max_batch);
// src [36][C][F] fp32 (F fastest) -> dst in the operand order of the streaming kernel
// ([36][Kp/32][Cp/8][64][4]), zero padded.
void build_stream_filters(const float* src, int C, int F, int Cp, int Kp, float* dst);
// fp32 -> fp16 on the device.
void convert_filters(const float* src, _Float16* dst, size_t n, hipStream_t s);

// M [36][Tp][Kp] -> out [n][361][Kp]:
// max(0, scale*(A^T m A - mean) + rfac*res)
template <typename P>
void launch_out_transform(const P* M, const P* res, P* out, const float* bn_scale,
                          const float* bn_mean, float rfac, int n, int Kp, int Tp,
                          hipStream_t s, LaunchTimer* t);

// Output transform of one layer fused with the input transform of the next:
// M [36][Tp][Kp] -> V_next [36][Tp][Kp]; the activation [n][361][Kp] is also
// written to act_out unless that is null.  Needs Kp to be a multiple of 64.
template <typename P>
void launch_out_in_transform(const P* M, const P* res, P* act_out, P* Vn, const float* bn_scale,
                             const float* bn_mean, float rfac, int n, int Kp, int Tp,
                             hipStream_t s, LaunchTimer* t);

// Direct 3x3 convolution in fp16 (conv3x3.hip), one launch per layer:
// X [Cp] -> Y [Kp] = min(max(0, scale*(conv - mean) + rfac*res), kActStoreMax), padded planes all three;
// res may be null and is not Y.  Wf: conv3x3_filter_count elements, zero but for what
// conv3x3_filters writes.  lanes: how many forwards may be running side by side.
// Whether a handle for batches of up to max_batch computes by it (measured; see there).
bool conv3x3_serves(int Kp, int max_batch, int elem_bytes);
size_t conv3x3_filter_count(int Cp, int Kp);
void launch_conv3x3(const _Float16* X, const _Float16* Wf, const _Float16* res, _Float16* Y,
                    const float* bn_scale, const float* bn_mean, float rfac, int n, int Cp, int Kp,
                    int lanes, hipStream_t s, LaunchTimer* t);
// The same layer with its sum dealt to the wavefronts of a work-group: for batches that leave a
// compute unit one tile.  It sums in another order, so a network takes one or the other for
// all its batches: this one where conv3x3_splits(Kp, largest batch).  Cp == Kp.
bool conv3x3_splits(int Kp, int max_batch);
void launch_conv3x3_split(const _Float16* X, const _Float16* Wf, const _Float16* res, _Float16* Y,
                          const float* bn_scale, const float* bn_mean, float rfac, int n, int Cp,
                          int Kp, hipStream_t s, LaunchTimer* t);
// Filters of one layer from U [36][C][F] fp32 on the device; *bad (device) is set if U is not
// the Winograd transform of 3x3 filters.
void conv3x3_filters(const float* U, _Float16* Wf, int C, int F, int Kp, int* bad, hipStream_t s);
// The way back, on the host: Winograd filters [36][Kp][Cp] of the filters as stored (padding of
// U is left as it is).
void conv3x3_winograd_filters(const _Float16* Wf, int C, int Cp, int F, int Kp, _Float16* U);

// The first layer of a direct fp16 tower from planes as floats [n][18][361] (conv3x3_first.hip): the results of
// launch_pack_input and launch_conv3x3, for batches that it serves (measured; see there).  Cp = 64.
bool conv3x3_first_serves(int Kp, int n);
void launch_conv3x3_first(const float* planes, const _Float16* Wf, _Float16* Y, const float* bn_scale,
                          const float* bn_mean, int n, int Cp, int Kp, hipStream_t s, const PlaneBorders* borders);

// Direct 3x3 convolution of fp32 towers (conv3x3_f32.hip), one launch per layer:
// X [Cp] -> Y [Kp] = max(0, scale*(conv - mean) + rfac*res) in fp32, padded planes, every operand split in
// two half-precision numbers.  Wf holds the filters of output channel k and input channel c times
// 2^(exp[k] - in_exp[c]): X holds channel c times 2^in_exp[c], scale is the caller's times 2^(out_exp[k]
// - exp[k]), mean times 2^exp[k], and Y comes out times 2^out_exp[k].  peaks: of X; those of Y
// go to `slots` (conv3x3_f32_slots words) and are returned.
bool conv3x3_f32_serves(int Kp);
size_t conv3x3_f32_filter_count(int Cp, int Kp);
size_t conv3x3_f32_slots(int Kp, int max_batch);
PeakMap launch_conv3x3_f32(const float* X, const _Float16* Wf, const float* res, float* Y,
                           const float* bn_scale, const float* bn_mean, float rfac,
                           const PeakMap& peaks, uint32_t* slots, int n, int Cp, int Kp,
                           int lanes, hipStream_t s, LaunchTimer* t);
// The same layer with its sum dealt to the wavefronts of a work-group (conv3x3_splits).
bool conv3x3_f32_splits(int Kp, int max_batch);
PeakMap launch_conv3x3_f32_split(const float* X, const _Float16* Wf, const float* res, float* Y,
                                 const float* bn_scale, const float* bn_mean, float rfac,
                                 const PeakMap& peaks, uint32_t* slots, int n, int Cp, int Kp,
                                 int lanes, hipStream_t s, LaunchTimer* t);
// Of every output channel of U [36][C][F]: the exponents of its largest filter times 2^-in_exp and of its
// largest product with inputs of magnitude 2^mag (kNoExp before; kNoExp: none); *bad as above.
constexpr int kNoExp = -(1 << 28);
void conv3x3_f32_peaks(const float* U, const int* in_exp, const int* mag, int C, int F, int* peak,
                       int* reach, int* bad, hipStream_t s);
// Whether an output channel's largest product is at least 2^-most of its largest filter times the largest
// input (exponents as above, of inputs of magnitude up to 2^top): with most = 14 halves hold what fp32 does.
bool conv3x3_f32_holds(int peak, int reach, int top, int most);
bool conv3x3_f32_exponent(int peak, float scale, float mean, int out_exp, int& e);
// Filters of one layer from U (device), exponents per channel (device).
void conv3x3_f32_filters(const float* U, const int* in_exp, const int* exp, _Float16* Wf, int C, int Cp,
                         int F, int Kp, hipStream_t s);
void conv3x3_f32_winograd_filters(const _Float16* Wf, const int* in_exp, const int* exp, int C, int Cp,
                                  int F, int Kp, float* U);

// 1x1 head convolutions: act [n][361][Cp] x w[3][Cp] -> pol [n][2][361], val [n][361],
// both multiplied by out_scale.
template <typename P>
void launch_head_conv(const P* act, bool padded, const float* w3, float out_scale, float* pol,
                      float* val, int n, int Cp, hipStream_t s, LaunchTimer* t);

// max |x| over count elements -> *out (float, must be zeroed before).
template <typename P>
void launch_absmax(const P* x, size_t count, float* out, hipStream_t s);

// Head arithmetic above the pipe boundary: BN + ReLU, the two large fully connected layers
// on the matrix cores, softmax / FC + tanh.  Device pointers; the two large FC matrices are
// held in the operand order of the matrix instruction (head_fc_fragments).
struct HeadParams {
    const float *bn_pol_mean, *bn_pol_scale, *ip_pol_wf, *ip_pol_b;
    const float *bn_val_mean, *bn_val_scale, *ip1_val_wf, *ip1_val_b, *ip2_val_w, *ip2_val_b;
};
// Element count of the fragment-order copy of the policy (true) / value (false) matrix, and
// its construction from W [outputs][inputs] row-major.
size_t head_fc_fragment_count(bool policy);
void head_fc_fragments(const float* W, bool policy, float* dst);
// work: device scratch of head_work_count(n) floats (partial sums of the logits and of the hidden
// units between the two kernels).  logits may be null.
size_t head_work_count(int n);
void launch_heads(const float* pol, const float* val, HeadParams hp, float temperature,
                  float* policy, float* logits, float* value, float* work, int n,
                  hipStream_t s);

}  // namespace lzhip
