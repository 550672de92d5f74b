// HIPPipe implementation: buffer management, weight upload, the layer loop
// (the role of OpenCL_Network::forward, reference src/OpenCL.cpp:142-329)
// and the fp16 activation-scale calibration.
#include "hip_pipe.h"

#include <hip/hip_runtime.h>

#include <atomic>
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <map>
#include <tuple>
#include <stdexcept>

#include "kernels.h"
#include "layer_graphs.h"
#include "plane_bits.h"

namespace lzhip {

typedef _Float16 half_t;

#define HIP_CHECK(expr)                                                                     \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess) {                                                             \
            throw std::runtime_error(std::string("HIP error: ") + hipGetErrorString(e_) +   \
                                     " at " + __FILE__ + ":" + std::to_string(__LINE__) +   \
                                     " (" #expr ")");                                       \
        }                                                                                   \
    } while (0)


// Working memory of the entry point that allocates nothing (forward_device_static):
// the buffers a lane otherwise gets from hipMalloc -- packed input planes, three
// activation planes, V and M -- for up to kStaticMaxBatch positions of a net with up
// to kStaticMaxFp filters (padded count) in the wider storage type (fp32):
//   V, M   2 x 36 x 256 x 256 x 4 B = 18 874 368
//   act0   8 x 361 x 64 x 4 B       =    739 328
//   act[3] 3 x 8 x 361 x 256 x 4 B  =  8 871 936      total 28 485 632 B (27.2 MiB)
// (a direct tower lays its padded planes and the peaks there instead, 13.5 MB at most).
// Every GPU the library runs on holds its own copy from module load to process end.
// In host code `scratch` is only a handle for hipGetSymbolAddress: the address kernels
// may use is the one resolved per device in static_scratch().
constexpr int kStaticMaxBatch = 8;
constexpr int kStaticMaxFp = 256;
constexpr int kStaticTp = 256;   // 8 x 25 tiles rounded up to kTileRowPad
constexpr size_t kStaticTileBytes = (size_t)kPos * kStaticTp * kStaticMaxFp * 4;
constexpr size_t kStaticAct0Bytes = (size_t)kStaticMaxBatch * kPts * 64 * 4;
constexpr size_t kStaticActBytes = (size_t)kStaticMaxBatch * kPts * kStaticMaxFp * 4;
constexpr size_t kStaticBytes = 2 * kStaticTileBytes + kStaticAct0Bytes + 3 * kStaticActBytes;
static_assert(kStaticTileBytes % 256 == 0 && kStaticAct0Bytes % 256 == 0 &&
              kStaticActBytes % 256 == 0, "sub-buffers keep the 256-byte alignment");
static __device__ __align__(256) unsigned char scratch[kStaticBytes];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static unsigned char* g_scratch_ptr[kMaxDevices] = {};
// One event per device, recorded behind every forward that uses the device's array and
// waited for by the next one, whichever handle and stream it comes from: forwards of
// different handles on one GPU then follow one another on the device instead of
// overwriting each other's tiles.  g_scratch_order_mu makes "wait, enqueue, record" one
// step, so the order of the records is the order of the waits.
static hipEvent_t g_scratch_event[kMaxDevices] = {};
static std::mutex g_scratch_order_mu;

// Device address of this device's copy of `scratch`; resolved once per device, with
// that device current (called from the pipe's constructor, i.e. from lzhip_create).
static unsigned char* static_scratch(int device) {
    if (device < 0 || device >= kMaxDevices) throw std::invalid_argument("device ordinal out of range");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        HIP_CHECK(hipSetDevice(device));
        unsigned char* ptr = nullptr;
        HIP_CHECK(hipGetSymbolAddress(reinterpret_cast<void**>(&ptr), HIP_SYMBOL(scratch)));
        if (!ptr) throw std::runtime_error("hipGetSymbolAddress returned a null address");
        HIP_CHECK(hipEventCreateWithFlags(&g_scratch_event[device], hipEventDisableTiming));
        g_scratch_ptr[device] = ptr;
    }
    return g_scratch_ptr[device];
}

template <typename T> struct DevBuf {
    T* p = nullptr;
    size_t count = 0;
    void alloc(size_t n) {
        release();
        if (n == 0) return;
        HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&p), n * sizeof(T)));
        HIP_CHECK(hipMemset(p, 0, n * sizeof(T)));
        count = n;
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        count = 0;
    }
    ~DevBuf() { release(); }
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    DevBuf(DevBuf&& o) noexcept : p(o.p), count(o.count) { o.p = nullptr; o.count = 0; }
};

template <typename T> struct PinnedBuf {
    T* p = nullptr;
    void alloc(size_t n) {
        release();
        HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&p), n * sizeof(T), hipHostMallocDefault));
    }
    void release() {
        if (p) (void)hipHostFree(p);
        p = nullptr;
    }
    ~PinnedBuf() { release(); }
};

template <typename P> constexpr int precision_of();
template <> constexpr int precision_of<float>() { return LZHIP_FP32; }
template <> constexpr int precision_of<half_t>() { return LZHIP_FP16; }

template <typename P>
class HIPPipeImpl final : public HIPPipe {
public:
    HIPPipeImpl(int device, int max_batch, int filters)
        : m_device(device), m_max_batch(max_batch), m_filters(filters) {
        if (max_batch < 1 || max_batch > 4096) throw std::invalid_argument("max_batch out of range");
        if (filters < 1 || filters > 4096) throw std::invalid_argument("filters out of range");
        int count = 0;
        HIP_CHECK(hipGetDeviceCount(&count));
        if (device < 0 || device >= count) throw std::runtime_error("no such HIP device");
        HIP_CHECK(hipSetDevice(device));
        hipDeviceProp_t prop;
        HIP_CHECK(hipGetDeviceProperties(&prop, device));
        if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
            throw std::runtime_error(std::string("device is ") + prop.gcnArchName +
                                     ", this library contains gfx950 code only");
        // Small batches leave more of the device idle at every kernel boundary.  Evaluations of
        // all lanes, a third lane against two: 20x64 fp16, batch 8 +34 %; 20x128 fp16, batch 32 +1 %;
        // 20x256 fp16, batch 16 +4 %, 32 +1 %, 40 +4 %; 20x192 fp32, batch 8 +1 %, 32 +10 %; 20x256 fp32,
        // batch 8 -5 %, 48 +8 %.  The line lies where it did for fp16 Winograd kernels.
        m_n_lanes = max_batch <= 48 ? 3 : 2;
        if (const char* e = std::getenv("LZHIP_LANES")) {   // measurement knob: 1..3 lanes
            const int v = std::atoi(e);
            if (v >= 1 && v <= kLanes) m_n_lanes = v;
        }
        // Every refusal comes before the first stream, event or allocation is made: a
        // constructor that throws runs no destructor.
        m_Fp = (int)ceil_multiple((size_t)filters, 64);
        if (!gemm_supports_channels<P>(m_Fp))
            throw std::invalid_argument(
                "unsupported filter count: after rounding up to a multiple of 64, fp16 takes up "
                "to 512 and 640, 768, 896, 1024; fp32 takes up to 512");
        m_C0p = 64;
        m_Tp = (int)ceil_multiple((size_t)max_batch * kTilesPerBoard, kTileRowPad);
        // The transform kernels address V and M through 32-bit buffer offsets.
        if ((size_t)kPos * m_Tp * m_Fp * sizeof(P) >= ((size_t)1 << 31))
            throw std::invalid_argument(
                "max_batch x filters too large: the Winograd tile buffers would exceed 2 GiB");
        m_static = static_scratch(device);
        struct Unwind {   // releases what the body below has created if it throws
            HIPPipeImpl* self;
            bool armed = true;
            ~Unwind() { if (armed) self->release_device_objects(); }
        } unwind{this};
        for (int i = 0; i < m_n_lanes; i++) {
            HIP_CHECK(hipStreamCreate(&m_lane[i].stream));
        }
        const size_t B = (size_t)max_batch;
        m_din.alloc(B * kInPlanes * kPts);
        m_dpol.alloc(B * 2 * kPts);
        m_dval.alloc(B * kPts);
        for (int i = 0; i < m_n_lanes; i++) {
            IoSlot& sl = m_slot[i];
            sl.hin.alloc(B * kInPlanes * kPts);
            sl.hpol.alloc(B * 2 * kPts);
            sl.hval.alloc(B * kPts);
            sl.din.alloc(B * kInPlanes * kPts);
            sl.dpol.alloc(B * 2 * kPts);
            sl.dval.alloc(B * kPts);
            sl.hbits.alloc(B * kInputWords);
            HIP_CHECK(hipEventCreateWithFlags(&sl.done, hipEventDisableTiming));
        }
        for (int i = 0; i < m_n_lanes; i++) {
            Lane& ln = m_lane[i];
            // (padded planes of a direct tower; the dense ones of another take less)
            ln.act0.alloc(padded_cells(max_batch) * m_C0p);
            for (auto& a : ln.act) a.alloc(padded_cells(max_batch) * m_Fp);
        }
        if (const char* e = std::getenv("LZHIP_INPLACE"))   // measurement knob
            m_in_place = std::atoi(e) != 0;
        m_scalar.alloc(4);
        for (int i = 0; i < kTimerPool; i++) {
            HIP_CHECK(hipEventCreate(&m_ev_start[i]));
            HIP_CHECK(hipEventCreate(&m_ev_stop[i]));
        }
        unwind.armed = false;
    }

    ~HIPPipeImpl() override { release_device_objects(); }

    // Streams and events (the buffers free themselves).  Also run by the constructor
    // when it fails half way.
    void release_device_objects() {
        (void)hipSetDevice(m_device);
        for (auto& ln : m_lane)
            if (ln.stream) (void)hipStreamSynchronize(ln.stream);
        clear_graphs();
        for (int i = 0; i < kTimerPool; i++) {
            if (m_ev_start[i]) (void)hipEventDestroy(m_ev_start[i]);
            if (m_ev_stop[i]) (void)hipEventDestroy(m_ev_stop[i]);
            m_ev_start[i] = m_ev_stop[i] = nullptr;
        }
        for (auto& sl : m_slot) {
            if (sl.done) (void)hipEventDestroy(sl.done);
            sl.done = nullptr;
        }
        for (auto& ln : m_lane) {
            if (ln.stream) (void)hipStreamDestroy(ln.stream);
            ln.stream = nullptr;
        }
    }

    int max_batch() const override { return m_max_batch; }
    int max_concurrency() const override { return m_n_lanes; }
    bool has_heads() const override { return m_heads_ready; }
    int filters() const override { return m_filters; }
    int precision() const override { return precision_of<P>(); }
    void* stream() override { return m_lane[0].stream; }
    int lanes() const override { return m_n_lanes; }
    std::vector<float> act_scales() const override { return m_s; }

    // -------------------------------------------------------------------
    // All or nothing: a failure anywhere below (an allocation, a copy, the calibration)
    // leaves the handle as it was before the call -- no layers, forwards refused, and a
    // later push_weights accepted.
    void push_weights(int n_layers, const float* const* U, const float* const* bn_mean,
                      const float* const* bn_scale, const float* pol_w,
                      const float* val_w) override {
        Lane& ln = m_lane[0];
        std::lock_guard<std::mutex> lk(ln.mu);
        if (n_layers < 1 || (n_layers % 2) != 1)
            throw std::invalid_argument("n_layers must be 1 + 2*blocks");
        if (m_ready || !m_layers.empty()) throw std::invalid_argument("push_weights called twice");
        HIP_CHECK(hipSetDevice(m_device));
        try {
            build_layers(n_layers, U, bn_mean, bn_scale, pol_w, val_w);
        } catch (...) {
            (void)hipStreamSynchronize(ln.stream);
            m_layers.clear();
            m_direct = false;
            m_chan.clear();
            m_in_scale.release();
            for (auto& l : m_lane) l.peaks.release();
            m_w3.release();
            m_s.clear();
            release_tiles();
            throw;
        }
        m_ready = true;
    }

    void build_layers(int n_layers, const float* const* U, const float* const* bn_mean,
                      const float* const* bn_scale, const float* pol_w, const float* val_w) {
        auto& ln = m_lane[0];
        const int F = m_filters;
        m_layers.resize(n_layers);
        // fp32 towers, and fp16 towers that conv3x3_serves names, are computed by direct convolution,
        // provided that what was handed over are transforms of 3x3 filters; all else goes
        // through the Winograd kernels and needs their tile arrays.
        m_direct = (sizeof(P) == 2 ? conv3x3_serves(m_Fp, m_max_batch, (int)sizeof(P))
                                   : conv3x3_f32_serves(m_Fp)) &&
                   build_direct_filters(n_layers, U, bn_mean, bn_scale);
        if (!m_direct) alloc_tiles();
        // Filters are laid out on the host in fp32; an fp16 net converts them on the device.
        std::vector<float> tmp;
        DevBuf<float> stage;
        auto upload = [&](DevBuf<P>& d) {
            d.alloc(tmp.size());
            if constexpr (sizeof(P) == 4) {
                HIP_CHECK(hipMemcpy(d.p, tmp.data(), tmp.size() * sizeof(float),
                                    hipMemcpyHostToDevice));
            } else {
                if (stage.count < tmp.size()) stage.alloc(tmp.size());
                HIP_CHECK(hipMemcpy(stage.p, tmp.data(), tmp.size() * sizeof(float),
                                    hipMemcpyHostToDevice));
                convert_filters(stage.p, d.p, tmp.size(), ln.stream);
                HIP_CHECK(hipGetLastError());
                HIP_CHECK(hipStreamSynchronize(ln.stream));
            }
        };
        for (int l = 0; l < n_layers; l++) {
            Layer& L = m_layers[l];
            L.C = l == 0 ? kInPlanes : F;
            L.Cp = l == 0 ? m_C0p : m_Fp;
            if (!m_direct) tmp.assign((size_t)kPos * m_Fp * L.Cp, 0.0f);
            // One copy of the filters, in the order the kernel of this width and precision
            // reads them.  Which kernel that is does not depend on the batch of a forward
            // (only on the handle's limit), so a network holds one order, never two.
            if (m_direct) {
            } else if (gemm_stream_shape(kTilesPerBoard, L.Cp, m_Fp, (int)sizeof(P)) &&
                       gemm_stream_prefers(m_Fp, m_max_batch)) {
                build_stream_filters(U[l], L.C, F, L.Cp, m_Fp, tmp.data());
                upload(L.Uf);
            } else {
                // reference layout [36][C][F] (F fastest)  ->  [36][Fp][Cp] (C fastest),
                // zero padded (the role of zeropad_U, reference src/OpenCLScheduler.cpp:60-82)
                for (int p = 0; p < kPos; p++)
                    for (int c = 0; c < L.C; c++) {
                        const float* src = U[l] + ((size_t)p * L.C + c) * F;
                        for (int k = 0; k < F; k++)
                            tmp[((size_t)p * m_Fp + k) * L.Cp + c] = src[k];
                    }
                upload(L.U);
            }
            L.mean.assign(bn_mean[l], bn_mean[l] + F);
            L.scale.assign(bn_scale[l], bn_scale[l] + F);
            L.d_mean.alloc(m_Fp);
            L.d_scale.alloc(m_Fp);
        }
        std::vector<float> w3((size_t)3 * m_Fp, 0.0f);
        for (int c = 0; c < F; c++) {
            const int e = chan(n_layers, c);
            w3[c] = std::ldexp(pol_w[c], -e);
            w3[m_Fp + c] = std::ldexp(pol_w[F + c], -e);
            w3[2 * m_Fp + c] = std::ldexp(val_w[c], -e);
        }
        m_w3.alloc(w3.size());
        HIP_CHECK(hipMemcpy(m_w3.p, w3.data(), w3.size() * sizeof(float), hipMemcpyHostToDevice));

        m_s.assign(n_layers + 1, 1.0f);
        for (int l = 0; l < n_layers; l++) upload_bn(l);
        if (precision_of<P>() == LZHIP_FP16) calibrate();
        HIP_CHECK(hipStreamSynchronize(ln.stream));
    }

    // Filters of the direct convolution for every layer; false (and nothing kept) if some layer's
    // U is not the transform of 3x3 filters, or fp32 operands do not fit into two halves.
    bool build_direct_filters(int n_layers, const float* const* U, const float* const* bn_mean,
                              const float* const* bn_scale) {
        DevBuf<float> stage;
        stage.alloc((size_t)kPos * m_filters * (m_filters > kInPlanes ? m_filters : kInPlanes));
        bool good = true;
        if constexpr (sizeof(P) == 2) {
            hipStream_t s = m_lane[0].stream;
            DevBuf<int> bad;
            bad.alloc(1);
            for (int l = 0; l < n_layers; l++) {
                Layer& L = m_layers[l];
                const int Cp = l == 0 ? m_C0p : m_Fp;
                L.W3.alloc(conv3x3_filter_count(Cp, m_Fp));
                conv3x3_filters(upload_filters(stage, U, l), L.W3.p, channels(l), m_filters, m_Fp, bad.p, s);
                HIP_CHECK(hipGetLastError());
                HIP_CHECK(hipStreamSynchronize(s));
            }
            int is_bad = 0;
            HIP_CHECK(hipMemcpy(&is_bad, bad.p, sizeof(int), hipMemcpyDeviceToHost));
            good = !is_bad;
        } else {
            good = build_split_filters(n_layers, U, bn_mean, bn_scale, stage);
        }
        if (!good) {
            for (auto& L : m_layers) {
                L.W3.release();
                L.exp.clear();
            }
            m_chan.clear();
            m_in_scale.release();
        } else {
            // the planes' borders are zero, whatever a push that failed has left there
            for (int i = 0; i < m_n_lanes; i++) {
                Lane& ln = m_lane[i];
                HIP_CHECK(hipMemset(ln.act0.p, 0, ln.act0.count * sizeof(P)));
                for (auto& a : ln.act) HIP_CHECK(hipMemset(a.p, 0, a.count * sizeof(P)));
            }
        }
        if (good && sizeof(P) == 4)
            for (int i = 0; i < m_n_lanes; i++)
                m_lane[i].peaks.alloc(2 * conv3x3_f32_slots(m_Fp, m_max_batch) + 2 * (size_t)m_max_batch);
        return good;
    }
    int channels(int l) const { return l == 0 ? kInPlanes : m_filters; }
    const float* upload_filters(DevBuf<float>& stage, const float* const* U, int l) {
        HIP_CHECK(hipMemcpy(stage.p, U[l], sizeof(float) * (size_t)kPos * channels(l) * m_filters,
                            hipMemcpyHostToDevice));
        return stage.p;
    }

    // fp32.  A direct tower holds its operands as two halves, relative to the largest of a board and of an
    // output channel, so channels whose activations lie far below others' would lose bits that fp32
    // keeps.  What a channel's magnitude is, is estimated from the filters and the batch norm, layer by
    // layer, as a binary exponent.  Where some output channel's largest product lies 2^8 or more below
    // its largest filter times the largest input, that layer's input planes hold the smaller channels
    // times a power of two (m_chan), which the producer's batch norm puts in and the next layer's
    // filters and the heads take out.  Batch norm and ReLU commute with it, so every product is the
    // one that it would be.  Any other layer is left as it is: an estimate may be far too high, for a
    // channel that never fires, and others raised to it would lose bits of their filters.
    bool build_split_filters(int n_layers, const float* const* U, const float* const* bn_mean,
                             const float* const* bn_scale, DevBuf<float>& stage) {
        hipStream_t s = m_lane[0].stream;
        const int F = m_filters;
        const size_t wide = F > kInPlanes ? F : kInPlanes;
        DevBuf<int> in_exp, mag, out;   // out: peak, reach, bad; then the filters' exponents
        in_exp.alloc(wide);
        mag.alloc(wide);
        out.alloc(2 * (size_t)F + 1);
        auto put = [](DevBuf<int>& d, const std::vector<int>& v) {
            HIP_CHECK(hipMemcpy(d.p, v.data(), v.size() * sizeof(int), hipMemcpyHostToDevice));
        };
        // magnitudes of layer l's input channels: m[0] of the planes, m[l] of layer l - 1's output
        std::vector<std::vector<int>> m(n_layers + 1, std::vector<int>(F, kNoExp));
        m[0].assign(kInPlanes, 0);
        m_chan.assign(n_layers + 1, std::vector<int>(F, 0));
        m_chan[0] = plane_exponents(U[0]);
        std::vector<char> move(n_layers + 1, 0);   // layers whose inputs are to be brought together
        for (int pass = 0; pass < 2; pass++) {
            bool holds = true;
            for (int l = 0; l < n_layers; l++) {
                Layer& L = m_layers[l];
                const int C = channels(l), Cp = l == 0 ? m_C0p : m_Fp;
                upload_filters(stage, U, l);
                put(in_exp, m_chan[l]);
                put(mag, m[l]);
                std::vector<int> ends(2 * (size_t)F + 1, kNoExp);
                ends[2 * F] = 0;
                put(out, ends);
                conv3x3_f32_peaks(stage.p, in_exp.p, mag.p, C, F, out.p, out.p + F, out.p + 2 * F,
                                  s);
                HIP_CHECK(hipGetLastError());
                HIP_CHECK(hipStreamSynchronize(s));
                HIP_CHECK(hipMemcpy(ends.data(), out.p, ends.size() * sizeof(int), hipMemcpyDeviceToHost));
                if (ends[2 * F]) return false;
                int top = kNoExp;
                for (int c = 0; c < C; c++)
                    if (m[l][c] != kNoExp) top = std::max(top, m[l][c] + m_chan[l][c]);
                L.exp.resize(F);
                for (int k = 0; k < F; k++) {
                    holds = holds && (l == 0 || conv3x3_f32_holds(ends[k], ends[F + k], top, 14)) &&
                            conv3x3_f32_exponent(ends[k], bn_scale[l][k], bn_mean[l][k],
                                                 m_chan[l + 1][k], L.exp[k]);
                    if (pass == 0) {
                        if (l > 0 && !conv3x3_f32_holds(ends[k], ends[F + k], top, 8)) move[l] = 1;
                        const bool second = l >= 2 && l % 2 == 0;
                        m[l + 1][k] = std::max(second ? m[l - 1][k] : kNoExp,
                                               magnitude(ends[F + k], bn_scale[l][k], bn_mean[l][k]));
                    }
                }
                put(out, L.exp);
                if (pass == 0) L.W3.alloc(conv3x3_f32_filter_count(Cp, m_Fp));
                conv3x3_f32_filters(stage.p, in_exp.p, out.p, L.W3.p, C, Cp, F, m_Fp, s);
                HIP_CHECK(hipGetLastError());
                HIP_CHECK(hipStreamSynchronize(s));
            }
            if (pass == 1 || !balance_channels(m, move)) {
                if (!holds) return false;
                break;
            }
        }
        std::vector<float> f(kInPlanes);
        for (int c = 0; c < kInPlanes; c++) f[c] = std::ldexp(1.0f, m_chan[0][c]);
        if (*std::min_element(f.begin(), f.end()) < 1.0f) {
            m_in_scale.alloc(kInPlanes);
            HIP_CHECK(hipMemcpy(m_in_scale.p, f.data(), f.size() * sizeof(float), hipMemcpyHostToDevice));
        }
        return true;
    }
    // Exponents of the input planes, at most 0: the engine's are 0 and 1, but a caller's may be of any
    // magnitude, which the first layer's filters then make up for.  A plane whose filters are
    // small in every output channel, beside that channel's largest, is taken down by as much.
    std::vector<int> plane_exponents(const float* U) const {
        const int F = m_filters;
        std::vector<float> most(F, 0.0f), of((size_t)kInPlanes * F, 0.0f);
        for (int p = 0; p < kPos; p++)
            for (int c = 0; c < kInPlanes; c++)
                for (int k = 0; k < F; k++) {
                    const float v = std::fabs(U[((size_t)p * kInPlanes + c) * F + k]);
                    most[k] = std::max(most[k], v);
                    of[(size_t)c * F + k] = std::max(of[(size_t)c * F + k], v);
                }
        std::vector<int> e(kInPlanes, 0);
        for (int c = 0; c < kInPlanes; c++) {
            int best = kNoExp;
            for (int k = 0; k < F; k++)
                if (of[(size_t)c * F + k] > 0.0f)
                    best = std::max(best, std::ilogb(of[(size_t)c * F + k]) - std::ilogb(most[k]));
            if (best != kNoExp) e[c] = -std::min(-best / 8 * 8, 96);
        }
        return e;
    }
    // Exponent of what a channel puts out: its largest product, times what 9 F of them come to (a sum of
    // F = 64 to 512 random ones is 4 to 12 times the largest), or its batch norm's constant where
    // that adds to it.
    static int magnitude(int reach, float scale, float mean) {
        if (!std::isfinite(scale) || scale == 0.0f) return kNoExp;
        const int s = std::ilogb(scale);
        const int conv = reach == kNoExp ? kNoExp : s + reach + 3;
        const bool adds = std::isfinite(mean) && (scale > 0.0f ? mean < 0.0f : mean > 0.0f);
        return adds ? std::max(conv, s + std::ilogb(mean)) : conv;
    }
    // m_chan from the magnitudes, for the inputs of the layers that `move` names: in whole 2^8, and by at
    // most 2^64; the channels of the residual stream have one exponent throughout, by which none comes
    // above the largest of its layer anywhere.  False: nothing to move.
    bool balance_channels(const std::vector<std::vector<int>>& m, const std::vector<char>& move) {
        const int n_layers = (int)m.size() - 1, F = m_filters;
        auto below = [&](int l, int k, int top) { return m[l][k] == kNoExp ? 64 : top - m[l][k]; };
        std::vector<int> stream(F, 64);
        bool moved = false, move_stream = false;
        for (int l = 1; l < n_layers; l += 2) move_stream = move_stream || move[l];
        for (int l = 1; l <= n_layers; l++) {
            const int top = *std::max_element(m[l].begin(), m[l].end());
            if (top == kNoExp) continue;
            for (int k = 0; k < F; k++) {
                if (l % 2) stream[k] = std::min(stream[k], below(l, k, top));
                else if (move[l] && m[l][k] != kNoExp) m_chan[l][k] = std::min(below(l, k, top), 64) / 8 * 8;
            }
        }
        for (int l = 1; l <= n_layers; l++)
            for (int k = 0; k < F; k++) {
                if (l % 2) m_chan[l][k] = !move_stream || m[n_layers][k] == kNoExp ? 0 : stream[k] / 8 * 8;
                moved = moved || m_chan[l][k] != 0;
            }
        return moved;
    }

    void alloc_tiles() {
        for (int i = 0; i < m_n_lanes; i++) {
            m_lane[i].V.alloc((size_t)kPos * m_Tp * m_Fp);
            m_lane[i].M.alloc((size_t)kPos * m_Tp * m_Fp);
        }
    }
    void release_tiles() {
        for (int i = 0; i < m_n_lanes; i++) {
            m_lane[i].V.release();
            m_lane[i].M.release();
        }
    }

    // -------------------------------------------------------------------
    void forward_device(int lane, int n, const float* d_in, float* d_pol, float* d_val) override {
        if (lane < 0 || lane >= m_n_lanes) throw std::invalid_argument("no such lane");
        Lane& ln = m_lane[lane];
        std::lock_guard<std::mutex> lk(ln.mu);
        check_ready(n);
        HIP_CHECK(hipSetDevice(m_device));
        run_forward(ln, n, d_in, nullptr, d_pol, d_val);
        HIP_CHECK(hipGetLastError());
    }

    // The same forward with every working buffer taken from the device's static
    // `scratch` array instead of the lane's allocations: kernel launches only, no
    // allocation of any kind.  Enqueued on lane 0's stream.  All calls on one GPU share
    // the array (whatever the handle): each waits on the device for the one enqueued
    // before it (one event per device, see g_scratch_event), so calls from different
    // handles or threads of this process run one after the other on the device.  While
    // the stream is being captured into a graph no event is recorded or waited for (the
    // captured launches are then ordered by the graph's own dependencies, and replays
    // that overlap with other users of the array race).  The borders of a direct tower's planes are
    // cleared by each call (another handle's may lie elsewhere), by the kernel that packs its input: a
    // launch of its own for all of the planes cost a call of 1 to 6 blocks 1 to 9 us in fp16 (6x128, 8
    // positions, with the device to itself: 83, now 71 to 75).  Nothing else has to start at
    // zero: every element a kernel reads for a real tile is written earlier in the same call (rows
    // of V past the last tile feed only rows of M that no kernel reads).
    // Calls wait for one another, so each takes the kernels of a forward alone.
    void forward_device_static(int n, const float* d_in, float* d_pol, float* d_val) override {
        Lane& ln = m_lane[0];
        std::lock_guard<std::mutex> lk(ln.mu);
        if (!m_ready) throw std::invalid_argument("push_weights has not been called");
        if (n < 1 || n > kStaticMaxBatch || n > m_max_batch)
            throw std::invalid_argument(
                "the no-allocation forward takes 1..8 positions (and at most max_batch): its "
                "static working memory is sized for 8");
        if (m_Fp > kStaticMaxFp)
            throw std::invalid_argument(
                "the no-allocation forward takes networks of up to 256 filters: its static "
                "working memory is sized for that");
        HIP_CHECK(hipSetDevice(m_device));
        unsigned char* base = m_static;
        Work w;
        w.stream = ln.stream;
        w.Tp = kStaticTp;
        PlaneBorders borders;
        if (m_direct) {
            // a direct tower has no tiles: its planes, padded and one after the other, are all
            // there is, and in fp32 the peaks behind them
            const size_t cells = padded_cells(n) * sizeof(P);
            w.act0 = reinterpret_cast<P*>(base);
            for (int i = 0; i < 3; i++)
                w.act[i] = reinterpret_cast<P*>(base + cells * (m_C0p + i * m_Fp));
            size_t need = cells * (m_C0p + 3 * m_Fp);
            if (sizeof(P) == 4) {
                w.peaks = reinterpret_cast<uint32_t*>(base + need);
                need += peak_words(n) * sizeof(uint32_t);
            }
            if (need > kStaticBytes)
                throw std::invalid_argument("no room in the static working memory");
            constexpr int piece = 16 / sizeof(P);
            borders.planes = reinterpret_cast<decltype(borders.planes)>(base);
            borders.n = n;
            borders.w0 = m_C0p / piece;
            borders.w = m_Fp / piece;
            w.borders = &borders;
        } else {
            w.V = reinterpret_cast<P*>(base);
            w.M = reinterpret_cast<P*>(base + kStaticTileBytes);
            w.act0 = reinterpret_cast<P*>(base + 2 * kStaticTileBytes);
            for (int i = 0; i < 3; i++)
                w.act[i] = reinterpret_cast<P*>(base + 2 * kStaticTileBytes + kStaticAct0Bytes +
                                                (size_t)i * kStaticActBytes);
        }
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        HIP_CHECK(hipStreamIsCapturing(ln.stream, &cap));
        const bool ordered = cap == hipStreamCaptureStatusNone;
        std::lock_guard<std::mutex> order(g_scratch_order_mu);
        hipEvent_t ev = g_scratch_event[m_device];
        if (ordered) HIP_CHECK(hipStreamWaitEvent(ln.stream, ev, 0));
        enqueue_forward(w, n, d_in, nullptr, d_pol, d_val, false);
        HIP_CHECK(hipGetLastError());
        if (ordered) HIP_CHECK(hipEventRecord(ev, ln.stream));
    }

    void sync() override {
        HIP_CHECK(hipSetDevice(m_device));
        for (int i = 0; i < m_n_lanes; i++) HIP_CHECK(hipStreamSynchronize(m_lane[i].stream));
    }

    // Host-buffer forward.  Up to kIoSlots callers may be inside at once: each packs its planes
    // into its own pinned staging, enqueues the forward on the lane of that slot under the
    // lane's lock, and waits for its own event outside the lock, so that packing and copies on the
    // host overlap the other callers' device work (see run_host_batch).
    void forward_batch(int n, const float* in, float* pol, float* val) override {
        HostCall c;
        c.in = in;
        c.pol = pol;
        c.val = val;
        run_host_batch(n, c);
    }

    // Bit-packed planes: 816 bytes per position travel instead of 26 KB; the first kernel
    // expands them.  Results are those of the float path on the same 0/1 planes.
    bool accepts_bits() const override { return true; }
    void run_bits(int n, const uint32_t* bits, bool heads, float temperature, float* out_a,
                  float* out_b) override {
        HostCall c;
        c.bits = bits;
        c.heads = heads;
        c.temperature = temperature;
        (heads ? c.policy : c.pol) = out_a;
        (heads ? c.value : c.val) = out_b;
        run_host_batch(n, c);
    }

    // The same path with the heads computed on the device: policy [n][362] and the
    // tanh value [n] come back instead of the raw planes.
    void evaluate_heads_batch(int n, const float* in, float temperature, float* policy,
                              float* value) override {
        evaluate_batch(n, in, temperature, policy, value, nullptr, nullptr, nullptr);
    }

    void evaluate_batch(int n, const float* in, float temperature, float* policy, float* value,
                        float* logits, float* pol, float* val) override {
        HostCall c;
        c.in = in;
        c.heads = true;
        c.temperature = temperature;
        c.policy = policy;
        c.value = value;
        c.logits = logits;
        c.pol = pol;
        c.val = val;
        run_host_batch(n, c);
    }

    // One batch with its planes and results in the caller's host memory: the planes as floats
    // or as bits; the heads or the raw planes; results that are null are not wanted.
    struct HostCall {
        const float* in = nullptr;
        const uint32_t* bits = nullptr;
        bool heads = false;
        float temperature = 1.0f;
        float *policy = nullptr, *value = nullptr, *logits = nullptr;
        float *pol = nullptr, *val = nullptr;
    };

    // Pinned host memory is mapped into the device's address space: the first kernel reads the
    // packed planes and the last ones write the results straight through it, so that no copy
    // command sits between this batch's kernels and the next batch's (each one is a bubble of
    // tens of microseconds on the stream, and copies to and from the caller's pageable
    // memory also wait for one another: they were two thirds of a 37-position call on a
    // 10x128 network).  Planes that hold only 0 and 1 -- the engine's -- are packed on the way
    // into pinned memory; other values, 32 times larger, go by copy.
    void run_host_batch(int n, const HostCall& c) {
        check_ready(n);
        if (c.heads && !m_heads_ready)
            throw std::invalid_argument("push_heads has not been called");
        if (c.heads && !(c.temperature > 0.0f))
            throw std::invalid_argument("temperature must be positive");
        HIP_CHECK(hipSetDevice(m_device));
        IoSlot* sl = nullptr;
        {
            std::unique_lock<std::mutex> lk(m_slot_mu);
            m_slot_cv.wait(lk, [&] {
                for (int i = 0; i < m_n_lanes; i++)
                    if (!m_slot[i].busy) return true;
                return false;
            });
            for (int i = 0; i < m_n_lanes && !sl; i++)
                if (!m_slot[i].busy) sl = &m_slot[i];
            sl->busy = true;
        }
        struct Release {
            HIPPipeImpl* self;
            IoSlot* sl;
            ~Release() {
                {
                    std::lock_guard<std::mutex> lk(self->m_slot_mu);
                    sl->busy = false;
                }
                self->m_slot_cv.notify_all();
            }
        } release{this, sl};
        const size_t in_size = (size_t)kInPlanes * kPts;
        bool packed = true;
        if (c.bits)
            std::memcpy(sl->hbits.p, c.bits, sizeof(uint32_t) * (size_t)n * kInputWords);
        else
            for (int i = 0; i < n && packed; i++)
                packed = pack_planes(c.in + (size_t)i * in_size,
                                     sl->hbits.p + (size_t)i * kInputWords);
        if (!packed) std::memcpy(sl->hin.p, c.in, sizeof(float) * (size_t)n * in_size);
        {
            // each staging slot has a lane of its own: two batches run side by side
            Lane& ln = m_lane[sl - m_slot];
            std::lock_guard<std::mutex> lk(ln.mu);
            float* pol_dev = c.heads ? sl->dpol.p : sl->hpol.p;   // raw planes: straight to host
            float* val_dev = c.heads ? sl->dval.p : sl->hval.p;
            if (!packed)
                HIP_CHECK(hipMemcpyAsync(sl->din.p, sl->hin.p, sizeof(float) * (size_t)n * in_size,
                                         hipMemcpyHostToDevice, ln.stream));
            run_forward(ln, n, packed ? nullptr : sl->din.p, packed ? sl->hbits.p : nullptr,
                        pol_dev, val_dev);
            if (c.heads) {
                launch_heads(pol_dev, val_dev, head_params(), c.temperature, sl->hpol.p,
                             c.logits ? sl->hlogits.p : nullptr, sl->hval.p, sl->dwork.p, n,
                             ln.stream);
                // (rarely asked for)
                if (c.pol)
                    HIP_CHECK(hipMemcpyAsync(c.pol, pol_dev, sizeof(float) * (size_t)n * 2 * kPts,
                                             hipMemcpyDeviceToHost, ln.stream));
                if (c.val)
                    HIP_CHECK(hipMemcpyAsync(c.val, val_dev, sizeof(float) * (size_t)n * kPts,
                                             hipMemcpyDeviceToHost, ln.stream));
            }
            HIP_CHECK(hipGetLastError());
            HIP_CHECK(hipEventRecord(sl->done, ln.stream));
        }
        HIP_CHECK(hipEventSynchronize(sl->done));
        auto fetch = [n](float* dst, const float* src, size_t each) {
            if (dst) std::memcpy(dst, src, sizeof(float) * (size_t)n * each);
        };
        if (c.heads) {
            fetch(c.policy, sl->hpol.p, 362);
            fetch(c.value, sl->hval.p, 1);
            fetch(c.logits, sl->hlogits.p, 362);
        } else {
            fetch(c.pol, sl->hpol.p, 2 * kPts);
            fetch(c.val, sl->hval.p, kPts);
        }
    }

    HeadParams head_params() const {
        return HeadParams{m_h[0].p, m_h[1].p, m_h[2].p, m_h[3].p, m_h[4].p,
                          m_h[5].p, m_h[6].p, m_h[7].p, m_h[8].p, m_h[9].p};
    }

    // -------------------------------------------------------------------
    void push_heads(const HeadWeightsHost& hw) override {
        Lane& ln = m_lane[0];
        std::lock_guard<std::mutex> lk(ln.mu);
        HIP_CHECK(hipSetDevice(m_device));
        auto up = [&](DevBuf<float>& d, const float* src, size_t n) {
            d.alloc(n);
            HIP_CHECK(hipMemcpy(d.p, src, n * sizeof(float), hipMemcpyHostToDevice));
        };
        up(m_h[0], hw.bn_pol_mean, 2);
        up(m_h[1], hw.bn_pol_scale, 2);
        {   // FC matrices go up in the operand order of the matrix instruction
            std::vector<float> t(head_fc_fragment_count(true));
            head_fc_fragments(hw.ip_pol_w, true, t.data());
            up(m_h[2], t.data(), t.size());
            t.assign(head_fc_fragment_count(false), 0.0f);
            head_fc_fragments(hw.ip1_val_w, false, t.data());
            up(m_h[6], t.data(), t.size());
        }
        up(m_h[3], hw.ip_pol_b, 362);
        up(m_h[4], hw.bn_val_mean, 1);
        up(m_h[5], hw.bn_val_scale, 1);
        up(m_h[7], hw.ip1_val_b, 256);
        up(m_h[8], hw.ip2_val_w, 256);
        up(m_h[9], hw.ip2_val_b, 1);
        const size_t B = (size_t)m_max_batch;
        m_dpolicy.alloc(B * 362);
        m_dvalue.alloc(B);
        m_dwork.alloc(head_work_count(m_max_batch));
        for (int i = 0; i < m_n_lanes; i++) {
            m_slot[i].dwork.alloc(head_work_count(m_max_batch));
            m_slot[i].hlogits.alloc(B * 362);
        }
        m_heads_ready = true;
    }

    float timed_evaluations(int n, int reps, const float* in, float temperature, float* policy,
                            float* value) override {
        Lane& ln = m_lane[0];
        std::lock_guard<std::mutex> lk(ln.mu);
        check_ready(n);
        if (!m_heads_ready) throw std::invalid_argument("push_heads has not been called");
        if (!(temperature > 0.0f)) throw std::invalid_argument("temperature must be positive");
        if (reps < 1 || reps > 100000) throw std::invalid_argument("reps out of range");
        HIP_CHECK(hipSetDevice(m_device));
        const size_t in_count = (size_t)n * kInPlanes * kPts;
        PinnedBuf<float> hin, hpolicy, hvalue;
        hin.alloc(in_count);
        hpolicy.alloc((size_t)n * 362);
        hvalue.alloc((size_t)n);
        std::memcpy(hin.p, in, in_count * sizeof(float));
        const HeadParams hp = head_params();
        HIP_CHECK(hipStreamSynchronize(ln.stream));
        HIP_CHECK(hipEventRecord(m_ev_start[0], ln.stream));
        for (int r = 0; r < reps; r++) {
            HIP_CHECK(hipMemcpyAsync(m_din.p, hin.p, in_count * sizeof(float),
                                     hipMemcpyHostToDevice, ln.stream));
            run_forward(ln, n, m_din.p, nullptr, m_dpol.p, m_dval.p);
            launch_heads(m_dpol.p, m_dval.p, hp, temperature, m_dpolicy.p, nullptr, m_dvalue.p,
                         m_dwork.p, n, ln.stream);
            HIP_CHECK(hipMemcpyAsync(hpolicy.p, m_dpolicy.p, sizeof(float) * (size_t)n * 362,
                                     hipMemcpyDeviceToHost, ln.stream));
            HIP_CHECK(hipMemcpyAsync(hvalue.p, m_dvalue.p, sizeof(float) * (size_t)n,
                                     hipMemcpyDeviceToHost, ln.stream));
        }
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipEventRecord(m_ev_stop[0], ln.stream));
        HIP_CHECK(hipEventSynchronize(m_ev_stop[0]));
        float ms = 0.0f;
        HIP_CHECK(hipEventElapsedTime(&ms, m_ev_start[0], m_ev_stop[0]));
        std::memcpy(policy, hpolicy.p, sizeof(float) * (size_t)n * 362);
        std::memcpy(value, hvalue.p, sizeof(float) * (size_t)n);
        return ms;
    }

    // -------------------------------------------------------------------
    void debug_layer(int layer, int n, const float* act_in, const float* res, float* Vout,
                     float* Mout, float* Yout) override {
        Lane& ln = m_lane[0];
        std::lock_guard<std::mutex> lk(ln.mu);
        check_ready(n);
        if (layer < 0 || layer >= (int)m_layers.size()) throw std::invalid_argument("bad layer");
        HIP_CHECK(hipSetDevice(m_device));
        Layer& L = m_layers[layer];
        const int F = m_filters, C = L.C, Cp = L.Cp;
        const int Tu = n * kTilesPerBoard;
        DevBuf<float> d_planes, d_res, d_sc, d_mn;
        d_planes.alloc((size_t)n * C * kPts);
        HIP_CHECK(hipMemcpy(d_planes.p, act_in, sizeof(float) * (size_t)n * C * kPts, hipMemcpyHostToDevice));
        P* a_in = (layer == 0) ? ln.act0.p : ln.act[0].p;
        PeakMap peaks{ln.peaks.p, kPts, 1};
        DevBuf<float> d_own;   // the planes as a forward holds them (m_chan)
        if constexpr (sizeof(P) == 4) {
            if (m_direct) {
                upload_planes(d_own, act_in, n, C, layer);
                launch_pack_input_peaks(d_own.p, a_in, n, C, Cp, peaks.slots, nullptr, ln.stream, nullptr);
            }
        }
        if (sizeof(P) == 2 || !m_direct)
            launch_pack_input<P>(d_planes.p, a_in, m_direct, n, C, Cp, ln.stream, nullptr);
        const P* r = nullptr;
        if (res) {
            upload_planes(d_res, res, n, F, layer + 1);
            launch_pack_input<P>(d_res.p, ln.act[1].p, m_direct, n, F, m_Fp, ln.stream, nullptr);
            r = ln.act[1].p;
        }
        std::vector<float> sc(m_Fp, 0.0f), mn(m_Fp, 0.0f);
        for (int k = 0; k < F; k++) {
            const int e = L.exp.empty() ? 0 : L.exp[k];
            sc[k] = std::ldexp(L.scale[k], chan(layer + 1, k) - e);
            mn[k] = std::ldexp(L.mean[k], e);
        }
        d_sc.alloc(m_Fp); d_mn.alloc(m_Fp);
        HIP_CHECK(hipMemcpy(d_sc.p, sc.data(), sizeof(float) * m_Fp, hipMemcpyHostToDevice));
        HIP_CHECK(hipMemcpy(d_mn.p, mn.data(), sizeof(float) * m_Fp, hipMemcpyHostToDevice));
        // A direct tower has no Winograd stages of its own: V and M are computed from the
        // filters it holds by the tiled kernels, Y by the kernel a forward runs.
        DevBuf<P> d_V, d_M, d_U;
        P *V = ln.V.p, *M = ln.M.p;
        const P *U = L.U.p, *Uf = L.Uf.p;
        if (m_direct) {
            std::vector<half_t> w3(L.W3.count);
            std::vector<P> u((size_t)kPos * m_Fp * Cp, (P)0.0f);
            HIP_CHECK(hipMemcpy(w3.data(), L.W3.p, w3.size() * sizeof(half_t), hipMemcpyDeviceToHost));
            if constexpr (sizeof(P) == 2)
                conv3x3_winograd_filters(w3.data(), C, Cp, F, m_Fp, u.data());
            else
                conv3x3_f32_winograd_filters(w3.data(), m_chan[layer].data(), L.exp.data(), C, Cp, F, m_Fp,
                                             u.data());
            d_U.alloc(u.size());
            HIP_CHECK(hipMemcpy(d_U.p, u.data(), u.size() * sizeof(P), hipMemcpyHostToDevice));
            d_V.alloc((size_t)kPos * m_Tp * m_Fp);
            d_M.alloc((size_t)kPos * m_Tp * m_Fp);
            V = d_V.p; M = d_M.p; U = d_U.p; Uf = nullptr;
        }
        const P* dense = a_in;   // (V is computed from dense planes)
        DevBuf<P> d_dense;
        if (m_direct) {
            d_dense.alloc((size_t)n * kPts * Cp);
            launch_pack_input<P>(d_planes.p, d_dense.p, false, n, C, Cp, ln.stream, nullptr);
            dense = d_dense.p;
        }
        launch_in_transform<P>(dense, V, n, Cp, m_Tp, ln.stream, nullptr);
        launch_gemm<P>(V, U, Uf, M, Tu, m_Tp, Cp, m_Fp, ln.stream, nullptr);
        if (m_direct)
            conv_direct(L, a_in, r, ln.act[2].p, d_sc.p, d_mn.p, 1.0f, peaks,
                        peak_slots(peaks.slots, n, 0), n, 1, ln.stream, nullptr);
        else
            launch_out_transform<P>(M, r, ln.act[2].p, d_sc.p, d_mn.p, 1.0f, n, m_Fp, m_Tp,
                                    ln.stream, nullptr);
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipStreamSynchronize(ln.stream));
        const int T = n * kTilesPerBoard;
        if (Vout) {
            std::vector<P> h((size_t)kPos * m_Tp * Cp);
            HIP_CHECK(hipMemcpy(h.data(), V, h.size() * sizeof(P), hipMemcpyDeviceToHost));
            for (int t = 0; t < T; t++)
                for (int p = 0; p < kPos; p++)
                    for (int c = 0; c < C; c++)
                        Vout[(((size_t)(t / 25) * kPos + p) * C + c) * 25 + t % 25] =
                            (float)h[((size_t)p * m_Tp + t) * Cp + c];
        }
        if (Mout) {
            std::vector<P> h((size_t)kPos * m_Tp * m_Fp);
            HIP_CHECK(hipMemcpy(h.data(), M, h.size() * sizeof(P), hipMemcpyDeviceToHost));
            for (int t = 0; t < T; t++)
                for (int p = 0; p < kPos; p++)
                    for (int k = 0; k < F; k++)
                        Mout[(((size_t)(t / 25) * kPos + p) * F + k) * 25 + t % 25] =
                            (float)h[((size_t)p * m_Tp + t) * m_Fp + k];
        }
        if (Yout) {
            std::vector<P> h((m_direct ? padded_cells(n) : (size_t)n * kPts) * m_Fp);
            HIP_CHECK(hipMemcpy(h.data(), ln.act[2].p, h.size() * sizeof(P), hipMemcpyDeviceToHost));
            for (int b = 0; b < n; b++)
                for (int pt = 0; pt < kPts; pt++)
                    for (int k = 0; k < F; k++)
                        Yout[((size_t)b * F + k) * kPts + pt] =
                            std::ldexp((float)h[plane_index(m_direct, b, pt) * m_Fp + k], -chan(layer + 1, k));
        }
    }
    // Planes [n][C][361], of layer l's input channels, times 2^m_chan, to the device.
    void upload_planes(DevBuf<float>& d, const float* planes, int n, int C, int l) {
        std::vector<float> h(planes, planes + (size_t)n * C * kPts);
        for (size_t i = 0; i < h.size(); i++) h[i] = std::ldexp(h[i], chan(l, (int)(i / kPts % C)));
        d.alloc(h.size());
        HIP_CHECK(hipMemcpy(d.p, h.data(), sizeof(float) * h.size(), hipMemcpyHostToDevice));
    }

    // -------------------------------------------------------------------
    void profile_forward(int n, const float* d_in, float* d_pol, float* d_val, float* ms,
                         int* launches) override {
        Lane& ln = m_lane[0];
        std::lock_guard<std::mutex> lk(ln.mu);
        check_ready(n);
        HIP_CHECK(hipSetDevice(m_device));
        if ((int)m_layers.size() * 3 + 2 > kTimerPool)
            throw std::invalid_argument("network too deep for the timer pool");
        m_timer_used = 0;
        enqueue_forward(ln, n, d_in, nullptr, d_pol, d_val, 1, true);
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipStreamSynchronize(ln.stream));
        for (int k = 0; k < LZHIP_K_COUNT; k++) { ms[k] = 0.0f; launches[k] = 0; }
        for (int i = 0; i < m_timer_used; i++) {
            float t = 0.0f;
            HIP_CHECK(hipEventElapsedTime(&t, m_ev_start[i], m_ev_stop[i]));
            ms[m_timer_class[i]] += t;
            launches[m_timer_class[i]]++;
        }
    }

private:
    typedef std::tuple<int, int, const void*, float*, float*> GraphKey;   // (n, lanes in use, buffers)
    // A lane is a stream with the working buffers of one forward.  Two batches on two
    // lanes run side by side on the device: each kernel's start-up and tail overlap with
    // the other lane's work, which a single chain of dependent kernels cannot do.
    // Lane 0 also serves calibration, profiling and the single-batch entry points.
    struct Lane {
        hipStream_t stream = nullptr;
        std::mutex mu;  // serialises enqueues on this lane
        DevBuf<P> act0, act[3], V, M;
        DevBuf<uint32_t> peaks;   // direct fp32 towers: peak_words
        std::map<GraphKey, hipGraphExec_t> graphs;
        LayerGraphs<hipGraphExec_t> layers;  // by 4 n + lanes in use
    };
    static constexpr int kLanes = 3;   // upper bound; m_n_lanes are in use

    // The working buffers of one forward as plain pointers: a lane's own allocations
    // or the static array.  Tp = rows of V and M per Winograd position.
    struct Work {
        hipStream_t stream = nullptr;
        P *act0 = nullptr, *act[3] = {nullptr, nullptr, nullptr}, *V = nullptr, *M = nullptr;
        int Tp = 0;
        uint32_t* peaks = nullptr;   // (direct fp32 towers)
        int lanes = 1;               // forwards that may be running side by side (lanes_in_use)
        LayerGraphs<hipGraphExec_t>* layers = nullptr;  // the lane's (none: plain launches)
        const PlaneBorders* borders = nullptr;          // to be cleared with the packing
    };
    // Slots of the input planes, then two sets that the layers write in turn.
    size_t peak_words(int n) const { return 2 * (size_t)n + 2 * conv3x3_f32_slots(m_Fp, n); }
    // Where layer l, of n boards, leaves its peaks; -1: the input planes.
    uint32_t* peak_slots(uint32_t* peaks, int n, int l) const {
        return l < 0 || !peaks ? peaks : peaks + 2 * n + (l & 1) * conv3x3_f32_slots(m_Fp, n);
    }
    Work work_of(Lane& ln) const {
        Work w;
        w.stream = ln.stream;
        w.act0 = ln.act0.p;
        for (int i = 0; i < 3; i++) w.act[i] = ln.act[i].p;
        w.V = ln.V.p;
        w.M = ln.M.p;
        w.Tp = m_Tp;
        w.peaks = m_direct ? ln.peaks.p : nullptr;
        return w;
    }

    struct Layer {
        int C = 0, Cp = 0;
        // the filters in one of three orders, the other two empty:
        DevBuf<P> U;                          // [36][Fp][Cp] (tiled GEMMs)
        DevBuf<P> Uf;                         // fragment order of the streaming GEMM
        DevBuf<half_t> W3;                    // 3x3, fragment order of the direct convolution
        std::vector<int> exp;                 // (fp32) exponent of each output channel's W3
        std::vector<float> mean, scale;       // as pushed (unscaled)
        DevBuf<float> d_mean, d_scale;        // with activation scales folded in
        float rfac = 1.0f;
    };

    void check_ready(int n) const {
        if (!m_ready) throw std::invalid_argument("push_weights has not been called");
        if (n < 1 || n > m_max_batch) throw std::invalid_argument("batch size out of range");
    }

    // BN parameters of layer l for stored activations x/s:
    //   out/s_out = relu(scale*s_in/s_out * (conv(x/s_in) - mean/s_in) + (s_res/s_out) * res/s_res)
    void upload_bn(int l) {
        Layer& L = m_layers[l];
        const float s_in = m_s[l], s_out = m_s[l + 1];
        std::vector<float> sc(m_Fp, 0.0f), mn(m_Fp, 0.0f);
        for (int k = 0; k < m_filters; k++) {
            const int e = L.exp.empty() ? 0 : L.exp[k];
            sc[k] = std::ldexp(L.scale[k] * (s_in / s_out), chan(l + 1, k) - e);
            mn[k] = std::ldexp(L.mean[k] / s_in, e);
        }
        const bool second = l >= 2 && (l % 2) == 0;
        L.rfac = second ? m_s[l - 1] / s_out : 1.0f;
        HIP_CHECK(hipMemcpy(L.d_scale.p, sc.data(), sizeof(float) * m_Fp, hipMemcpyHostToDevice));
        HIP_CHECK(hipMemcpy(L.d_mean.p, mn.data(), sizeof(float) * m_Fp, hipMemcpyHostToDevice));
    }

    LaunchTimer* timer(bool timed, int cls) {
        if (!timed) return nullptr;
        const int i = m_timer_used++;
        m_timer_class[i] = cls;
        m_timer.start = m_ev_start[i];
        m_timer.stop = m_ev_stop[i];
        return &m_timer;
    }

    // Activation buffer roles rotate: cur = block input, mid, nxt = block output.
    void run_conv(Lane& ln, int l, int n, const P* in, const P* res, P* out, bool timed) {
        Layer& L = m_layers[l];
        if (m_direct) {
            PeakMap none;
            conv_direct(L, in, res, out, L.d_scale.p, L.d_mean.p, L.rfac, none, nullptr, n, 1, ln.stream,
                        timer(timed, LZHIP_K_GEMM));
            return;
        }
        const int Tu = n * kTilesPerBoard;
        launch_in_transform<P>(in, ln.V.p, n, L.Cp, m_Tp, ln.stream, timer(timed, LZHIP_K_IN));
        launch_gemm<P>(ln.V.p, L.U.p, L.Uf.p, ln.M.p, Tu, m_Tp, L.Cp, m_Fp, ln.stream,
                       timer(timed, LZHIP_K_GEMM));
        launch_out_transform<P>(ln.M.p, res, out, L.d_scale.p, L.d_mean.p, L.rfac, n, m_Fp, m_Tp,
                                ln.stream, timer(timed, LZHIP_K_OUT));
    }

    // With LZHIP_GRAPH=1 the launches of a forward (2 + one per layer of a direct tower; 2 + two
    // per layer with Winograd kernels) are captured once per (batch size, lanes in use, buffers) into a HIP
    // graph and replayed, which takes the launch work off the host thread.  Only kernel
    // nodes are captured (no memsets or copies).  On one lane the replay measured no faster
    // than stream launches (40x256 fp16 at batch 16: 0.84 against 0.83 ms; the gaps between
    // these kernels are drain and cache write-back, not launch latency), so plain stream
    // launches are the default, but for small direct towers on several lanes
    // (launch_layers_graph).
    void clear_graphs(Lane& ln) {
        for (auto& kv : ln.graphs) (void)hipGraphExecDestroy(kv.second);
        ln.graphs.clear();
        ln.layers.clear([](hipGraphExec_t g) { (void)hipGraphExecDestroy(g); });
    }
    void clear_graphs() {
        for (auto& ln : m_lane) clear_graphs(ln);
    }
    // On how many lanes this forward and the two before it were put: how much of the device it
    // can expect for itself, which the direct convolutions' tiles depend on (the results do not).
    int lanes_in_use(const Lane& ln) {
        const uint32_t id = (uint32_t)(&ln - m_lane);
        const uint32_t h = (m_recent.load(std::memory_order_relaxed) << 8 | id) & 0xffffffu;
        m_recent.store(h, std::memory_order_relaxed);
        const uint32_t b = h >> 8 & 255, c = h >> 16;
        return 1 + (b != 255 && b != id) + (c != 255 && c != id && c != b);
    }
    // d_in: fp32 planes, or, when null, d_bits: the planes one bit per value
    void run_forward(Lane& ln, int n, const float* d_in, const uint32_t* d_bits, float* d_pol,
                     float* d_val) {
        const int lanes = lanes_in_use(ln);
        if (!m_use_graph) {
            enqueue_forward(ln, n, d_in, d_bits, d_pol, d_val, lanes, false);
            return;
        }
        const GraphKey key(n, lanes, d_in ? (const void*)d_in : (const void*)d_bits, d_pol, d_val);
        auto it = ln.graphs.find(key);
        if (it == ln.graphs.end()) {
            if (ln.graphs.size() >= 64) {
                HIP_CHECK(hipStreamSynchronize(ln.stream));
                clear_graphs(ln);
            }
            hipGraph_t g = nullptr;
            hipGraphExec_t ge = nullptr;
            HIP_CHECK(hipStreamBeginCapture(ln.stream, hipStreamCaptureModeThreadLocal));
            enqueue_forward(ln, n, d_in, d_bits, d_pol, d_val, lanes, false);
            HIP_CHECK(hipStreamEndCapture(ln.stream, &g));
            const hipError_t e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
            (void)hipGraphDestroy(g);
            HIP_CHECK(e);
            it = ln.graphs.emplace(key, ge).first;
        }
        HIP_CHECK(hipGraphLaunch(it->second, ln.stream));
    }

    // Layer loop; a direct tower has its own (enqueue_direct).  With the Winograd kernels every
    // layer but the last ends in the fused kernel that turns M_l straight into V_{l+1}; the
    // spatial activation is written only where a
    // later layer adds it back as a skip connection (layer 0 and every block
    // output), and by the last layer for the 1x1 heads.
    void enqueue_forward(Lane& ln, int n, const float* d_in, const uint32_t* d_bits,
                         float* d_pol, float* d_val, int lanes, bool timed) {
        Work w = work_of(ln);
        w.lanes = lanes;
        if (!m_use_graph) w.layers = &ln.layers;
        enqueue_forward(w, n, d_in, d_bits, d_pol, d_val, timed);
    }
    void enqueue_forward(const Work& w, int n, const float* d_in, const uint32_t* d_bits,
                         float* d_pol, float* d_val, bool timed) {
        const int nl = (int)m_layers.size();
        const int Tu = n * kTilesPerBoard;
        if constexpr (sizeof(P) == 2) {
            // (Forwards side by side replay their layers as one launch, from the lane's own planes.  A timed pass
            // reports packing and every convolution as launches of their own, whatever the batch.)
            if (m_direct && d_in && !timed && w.lanes == 1 && conv3x3_first_serves(m_Fp, n)) {
                const Layer& L = m_layers[0];
                launch_conv3x3_first(d_in, L.W3.p, w.act[0], L.d_scale.p, L.d_mean.p, n, m_C0p, m_Fp, w.stream,
                                     w.borders);
                enqueue_direct(w, n, d_pol, d_val, timed, 1);
                return;
            }
        }
        LaunchTimer* pack = timer(timed, LZHIP_K_PACK);
        if (!d_in)
            launch_pack_input_bits<P>(d_bits, w.act0, m_direct, n, kInPlanes, m_C0p, w.peaks, m_in_scale.p,
                                      w.stream, pack);
        else if (!pack_with_peaks(w, d_in, n, pack))
            launch_pack_input<P>(d_in, w.act0, m_direct, n, kInPlanes, m_C0p, w.stream, pack, w.borders);
        if (m_direct) {
            enqueue_direct(w, n, d_pol, d_val, timed, 0);
            return;
        }
        launch_in_transform<P>(w.act0, w.V, n, m_C0p, w.Tp, w.stream, timer(timed, LZHIP_K_IN));
        // With the streaming GEMM (fp32 networks whose filters are no 3x3 ones) the tower's layers
        // work in place: M_l is written over V_l and V_{l+1} over M_l (see the kernels), so a
        // lane's tiles are one array instead of two (59 MB less per lane at 64 boards of 256
        // filters), of which more stays in the 256 MB memory-side cache.  Layer 0 reads 64
        // padded planes and keeps its own output.
        P* tiles = w.M;
        const bool in_place = m_in_place && m_layers.size() > 1 &&
                              gemm_stream_shape(Tu, m_Fp, m_Fp, (int)sizeof(P)) &&
                              m_layers[1].Uf.p != nullptr;
        int cur = 0, nxt = 1;  // block input (skip) / block output
        launch_gemm<P>(w.V, m_layers[0].U.p, m_layers[0].Uf.p, w.M, Tu, w.Tp, m_layers[0].Cp, m_Fp,
                       w.stream, timer(timed, LZHIP_K_GEMM));
        for (int l = 0; l < nl; l++) {
            Layer& L = m_layers[l];
            const bool block_end = (l % 2) == 0;      // layer 0 and second convs
            const P* res = (block_end && l >= 2) ? w.act[cur] : nullptr;
            P* out = l == 0 ? w.act[cur] : w.act[nxt];
            if (l == nl - 1) {
                launch_out_transform<P>(tiles, res, out, L.d_scale.p, L.d_mean.p, L.rfac, n, m_Fp,
                                        w.Tp, w.stream, timer(timed, LZHIP_K_OUT));
                launch_head_conv<P>(out, false, m_w3.p, m_s[nl], d_pol, d_val, n, m_Fp, w.stream,
                                    timer(timed, LZHIP_K_HEAD));
            } else {
                Layer& N = m_layers[l + 1];
                launch_out_in_transform<P>(tiles, res, block_end ? out : nullptr, w.V, L.d_scale.p,
                                           L.d_mean.p, L.rfac, n, m_Fp, w.Tp, w.stream,
                                           timer(timed, LZHIP_K_OUTIN));
                if (in_place) tiles = w.V;
                launch_gemm<P>(w.V, N.U.p, N.Uf.p, tiles, Tu, w.Tp, N.Cp, m_Fp, w.stream,
                               timer(timed, LZHIP_K_GEMM));
            }
            if (block_end && l >= 2) { const int o = cur; cur = nxt; nxt = o; }
        }
    }

    bool pack_with_peaks(const Work& w, const float* d_in, int n, LaunchTimer* t) {
        if constexpr (sizeof(P) == 4) {
            if (w.peaks) {
                launch_pack_input_peaks(d_in, w.act0, n, kInPlanes, m_C0p, w.peaks, m_in_scale.p, w.stream,
                                        t, w.borders);
                return true;
            }
        }
        return false;
    }

    // One layer of a direct tower; which of the two kernels depends on the handle, not on n.
    // fp32: peaks are those of `in` and become those of `out`, which go to `slots`.
    void conv_direct(const Layer& L, const P* in, const P* res, P* out, const float* scale,
                     const float* mean, float rfac, PeakMap& peaks, uint32_t* slots, int n,
                     int lanes, hipStream_t s, LaunchTimer* t) {
        if constexpr (sizeof(P) == 2) {
            const bool split = L.Cp == m_Fp && conv3x3_splits(m_Fp, m_max_batch);
            if (split)
                launch_conv3x3_split(in, L.W3.p, res, out, scale, mean, rfac, n, L.Cp, m_Fp, s, t);
            else
                launch_conv3x3(in, L.W3.p, res, out, scale, mean, rfac, n, L.Cp, m_Fp, lanes, s, t);
        } else {
            const bool split = L.Cp == m_Fp && conv3x3_f32_splits(m_Fp, m_max_batch);
            peaks = split ? launch_conv3x3_f32_split(in, L.W3.p, res, out, scale, mean, rfac, peaks,
                                                     slots, n, L.Cp, m_Fp, lanes, s, t)
                          : launch_conv3x3_f32(in, L.W3.p, res, out, scale, mean, rfac, peaks, slots,
                                               n, L.Cp, m_Fp, lanes, s, t);
        }
    }

    // The layer loop of a direct tower: one launch per layer.
    // The layers of a direct tower from `first` on, 0 (from the packed planes) or 1, to the last activation, which
    // is returned.
    const P* enqueue_layers(const Work& w, int n, bool timed, int first) {
        const int nl = (int)m_layers.size();
        const P* last = w.act[0];
        PeakMap peaks{w.peaks, kPts, 1};
        int cur = 0, nxt = 2;   // block input (skip) / block output; 1 lies between
        for (int l = first; l < nl; l++) {
            Layer& L = m_layers[l];
            const bool second = l >= 2 && (l % 2) == 0;
            const P* in = l == 0 ? w.act0 : second ? w.act[1] : w.act[cur];
            P* out = l == 0 ? w.act[cur] : second ? w.act[nxt] : w.act[1];
            conv_direct(L, in, second ? w.act[cur] : nullptr, out, L.d_scale.p, L.d_mean.p, L.rfac,
                        peaks, peak_slots(w.peaks, n, l), n, w.lanes, w.stream,
                        timer(timed, LZHIP_K_GEMM));
            last = out;
            if (second) { const int o = cur; cur = nxt; nxt = o; }
        }
        return last;
    }
    const P* last_activation(const Work& w) const {
        return w.act[((int)m_layers.size() / 2) % 2 ? 2 : 0];
    }
    // The layers as one launch, of a graph that holds them for this lane and batch size: nothing but
    // kernels, and between the lane's own buffers only, so that it is good for any caller's planes
    // and results.  It takes the host thread off the layers' 3.5 us a launch, which is what bounds small
    // networks on several lanes; on one lane, where the kernels are as long as their launches, plain
    // launches are 3 to 8 % faster.  A lane has graphs of the sixteen most frequent pairs of batch size and
    // lanes in use at most (LayerGraphs).
    bool launch_layers_graph(const Work& w, int n) {
        if (!w.layers || w.lanes < 2 || !launch_bound(n)) return false;
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(w.stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone)
            return false;
        const hipGraphExec_t g = w.layers->use(
            4 * n + w.lanes, [&] { return layers_graph(w, n); },
            [&](hipGraphExec_t old) {
                (void)hipStreamSynchronize(w.stream);   // (its last launch may still be running)
                (void)hipGraphExecDestroy(old);
            });
        if (!g) return false;
        HIP_CHECK(hipGraphLaunch(g, w.stream));
        return true;
    }
    // Recorded on a stream of its own that no other work is ordered against, so that a call of
    // another thread on the default stream cannot meet the recording; null if the runtime declines.
    hipGraphExec_t layers_graph(Work w, int n) {
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;
        hipStream_t s = nullptr;
        HIP_CHECK(hipGetLastError());   // (the caller's own, before any of this)
        if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        w.stream = s;
        if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) == hipSuccess) {
            std::exception_ptr failed;
            try {
                enqueue_layers(w, n, false, 0);
            } catch (...) {
                failed = std::current_exception();
            }
            if (hipStreamEndCapture(s, &graph) != hipSuccess) graph = nullptr;
            if (failed) {
                if (graph) (void)hipGraphDestroy(graph);
                (void)hipStreamDestroy(s);
                std::rethrow_exception(failed);
            }
        }
        if (graph && hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) != hipSuccess)
            exec = nullptr;
        if (graph) (void)hipGraphDestroy(graph);
        (void)hipStreamDestroy(s);
        if (!exec) (void)hipGetLastError();   // (what was declined is not the caller's error)
        return exec;
    }
    // Whether the layers of two lanes take the device no longer than their launches take the host.
    // 20 blocks on two lanes, plain launches -> graph, us for both forwards: fp16 64 filters 1 board 302 ->
    // 114, 34: 314 -> 200, 90: 316 -> 268; 128 filters 1 board 296 -> 146, 12: 322 -> 249, 25: 318 -> 305, 35:
    // 338 -> 343; 192 filters 8 boards 315 -> 287, 14: 351 -> 356; 256 filters 1 board 314 -> 190, 5: 326 ->
    // 292, 8: 376 -> 373; 384 filters 1 board 324 -> 272, 3: 412 -> 415.  fp32 64 filters 1 board 312 -> 188, 16:
    // 313 -> 299; 128 filters 1 board 236 to 301 -> 246, 8: 326 -> 333; 192 filters 1 board 325 -> 336.
    bool launch_bound(int n) const {
        return (size_t)n * m_Fp * m_Fp <= (sizeof(P) == 2 ? 5u * 256 * 256 : 8u * 64 * 64);
    }
    void enqueue_direct(const Work& w, int n, float* d_pol, float* d_val, bool timed, int first) {
        const int nl = (int)m_layers.size();
        const P* last = last_activation(w);
        if (first > 0 || timed || !launch_layers_graph(w, n)) last = enqueue_layers(w, n, timed, first);
        launch_head_conv<P>(last, true, m_w3.p, m_s[nl], d_pol, d_val, n, m_Fp, w.stream,
                            timer(timed, LZHIP_K_HEAD));
    }

    float absmax(const P* x, size_t count) {
        Lane& ln = m_lane[0];
        HIP_CHECK(hipMemsetAsync(m_scalar.p, 0, sizeof(float), ln.stream));
        launch_absmax<P>(x, count, m_scalar.p, ln.stream);
        float v = 0.0f;
        HIP_CHECK(hipMemcpyAsync(&v, m_scalar.p, sizeof(float), hipMemcpyDeviceToHost, ln.stream));
        HIP_CHECK(hipStreamSynchronize(ln.stream));
        return v;
    }

    // fp16 storage needs every stored activation to sit well inside the
    // half-precision range, also after the up-to-20x growth of the input
    // transform.  Convolution, ReLU and the residual add commute with positive
    // scaling, so layer l stores x_l / s_l with s_l a power of two chosen here
    // from a forward pass over synthetic positions; the scales are folded
    // into the batch-norm parameters and undone in the 1x1 heads, which is
    // exact in real arithmetic.  Trained networks keep |x| small and get
    // s_l = 1 (plain fp16 storage, as the reference's half pipeline).
    void calibrate() {
        Lane& ln = m_lane[0];
        const int n = m_max_batch < 8 ? m_max_batch : 8;
        std::vector<float> in((size_t)n * kInPlanes * kPts, 0.0f);
        uint64_t st = 0x9E3779B97F4A7C15ull;
        auto rnd = [&]() {
            st = st * 6364136223846793005ull + 1442695040888963407ull;
            return (double)(st >> 11) * (1.0 / 9007199254740992.0);
        };
        for (int b = 0; b < n; b++) {
            float* x = in.data() + (size_t)b * kInPlanes * kPts;
            for (int h = 0; h < 8; h++)
                for (int pt = 0; pt < kPts; pt++) {
                    const double u = rnd();
                    if (u < 0.2) x[h * kPts + pt] = 1.0f;
                    else if (u < 0.4) x[(8 + h) * kPts + pt] = 1.0f;
                }
            for (int pt = 0; pt < kPts; pt++) x[16 * kPts + pt] = 1.0f;
        }
        HIP_CHECK(hipMemcpy(m_din.p, in.data(), in.size() * sizeof(float), hipMemcpyHostToDevice));
        launch_pack_input<P>(m_din.p, ln.act0.p, m_direct, n, kInPlanes, m_C0p, ln.stream, nullptr);

        const float target = 16.0f;
        const int nl = (int)m_layers.size();
        const size_t cnt = (m_direct ? padded_cells(n) : (size_t)n * kPts) * m_Fp;
        int cur = 0, mid = 1, nxt = 2;
        auto settle = [&](int l, const P* src, const P* res, P* dst) {
            // provisional: keep the incoming scale, then correct from the measured range
            m_s[l + 1] = m_s[l];
            bool adjusted = false;
            for (int attempt = 0; attempt < 8; attempt++) {
                upload_bn(l);
                if (attempt == 0 || m_direct) {
                    run_conv(ln, l, n, src, res, dst, false);
                } else {
                    Layer& L = m_layers[l];
                    launch_out_transform<P>(ln.M.p, res, dst, L.d_scale.p, L.d_mean.p, L.rfac, n,
                                            m_Fp, m_Tp, ln.stream, nullptr);
                }
                const float mx = absmax(dst, cnt);
                if (!(mx < kActStoreMax)) {  // at the storage clamp (or NaN): coarser scale, try again
                    m_s[l + 1] *= 256.0f;
                    adjusted = false;
                    continue;
                }
                if (adjusted) return;  // re-run with the corrected scale is in range
                const float true_max = mx * m_s[l + 1];
                float want = 1.0f;
                if (true_max > target) want = std::exp2(std::ceil(std::log2(true_max / target)));
                if (want == m_s[l + 1]) return;
                m_s[l + 1] = want;
                adjusted = true;
            }
            throw std::runtime_error("activation-scale calibration did not converge");
        };
        settle(0, ln.act0.p, nullptr, ln.act[cur].p);
        for (int l = 1; l + 1 < nl; l += 2) {
            settle(l, ln.act[cur].p, nullptr, ln.act[mid].p);
            settle(l + 1, ln.act[mid].p, ln.act[cur].p, ln.act[nxt].p);
            const int o = cur; cur = nxt; nxt = o;
        }
    }

    static constexpr int kTimerPool = 512;
    int m_device, m_max_batch, m_filters;
    int m_Fp = 0, m_C0p = 0, m_Tp = 0;
    unsigned char* m_static = nullptr;   // this device's copy of the static working memory
    Lane m_lane[kLanes];
    int m_n_lanes = 2;
    DevBuf<float> m_din, m_dpol, m_dval, m_w3, m_scalar;  // evaluate_batch / calibration
    // Staging of forward_batch: kIoSlots batches may be between "copied in" and
    // "copied out" at once, slot i on lane i.
    struct IoSlot {
        PinnedBuf<float> hin, hpol, hval, hlogits;
        PinnedBuf<uint32_t> hbits;
        DevBuf<float> din, dpol, dval;
        DevBuf<float> dwork;   // heads: logits and hidden units between the two kernels
        hipEvent_t done = nullptr;
        bool busy = false;
    };
    static constexpr int kIoSlots = kLanes;
    IoSlot m_slot[kIoSlots];
    std::mutex m_slot_mu;
    std::condition_variable m_slot_cv;
    std::vector<Layer> m_layers;
    std::atomic<bool> m_ready{false};   // set by a push_weights that ran to its end
    std::vector<float> m_s;  // activation scales, m_s[0] = input
    DevBuf<float> m_h[10], m_dpolicy, m_dvalue, m_dwork;
    bool m_heads_ready = false;
    hipEvent_t m_ev_start[kTimerPool] = {}, m_ev_stop[kTimerPool] = {};
    int m_timer_class[kTimerPool] = {};
    int m_timer_used = 0;
    LaunchTimer m_timer;
    // LZHIP_GRAPH=1 (any value but 0): forwards replay a captured graph
    bool m_use_graph = [] {
        const char* e = std::getenv("LZHIP_GRAPH");
        return e != nullptr && std::atoi(e) != 0;
    }();
    bool m_direct = false;               // direct convolutions (set by push_weights)
    // (direct fp32) planes of layer l's input channel c are held times 2^m_chan[l][c]; the last: the heads'
    std::vector<std::vector<int>> m_chan;
    DevBuf<float> m_in_scale;            // 2^m_chan[0], or none where all of it is 0
    int chan(int l, int c) const { return m_chan.empty() ? 0 : m_chan[l][c]; }
    std::atomic<uint32_t> m_recent{0xffffffu};   // lanes of the last three forwards, a byte each
    bool m_in_place = true;              // tower layers keep V and M in one array (see enqueue_forward)
};

std::unique_ptr<HIPPipe> create_hip_pipe(int device, int precision, int max_batch, int filters) {
    if (precision == LZHIP_FP32)
        return std::unique_ptr<HIPPipe>(new HIPPipeImpl<float>(device, max_batch, filters));
    if (precision == LZHIP_FP16)
        return std::unique_ptr<HIPPipe>(new HIPPipeImpl<half_t>(device, max_batch, filters));
    throw std::invalid_argument("precision must be LZHIP_FP32 or LZHIP_FP16");
}

std::unique_ptr<BatchExecutor> make_hip_pipe(int device, int precision, int max_batch,
                                             int filters) {
    return create_hip_pipe(device, precision, max_batch, filters);
}

}  // namespace lzhip
