// Packs the planes of a position one bit per value.
#pragma once
#include <cstdint>
#include <cstring>

#include "lzhip.h"

#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
#define LZHIP_X86_PACK 1
#include <immintrin.h>
#endif

namespace lzhip {

// One version per vector width, chosen by what the processor has: value by value the loop is
// bound by its own arithmetic (about 5 us a position), 16 at a time by reading the planes
// (26 KB, about 0.6 us from the caches).
namespace plane_bits {

constexpr int kWords = LZHIP_INPUT_SIZE / 32, kTail = LZHIP_INPUT_SIZE % 32;
constexpr uint32_t kOne = 0x3f800000u;

inline bool scalar(const float* in, uint32_t* bits, int words, int tail) {
    static_assert(sizeof(float) == sizeof(uint32_t), "float size");
    uint32_t other = 0;
    for (int w = 0; w < words + (tail != 0); w++) {
        uint32_t word = 0;
        const int n = w < words ? 32 : tail;
        for (int i = 0; i < n; i++) {
            uint32_t v;
            std::memcpy(&v, in + 32 * w + i, sizeof(v));
            other |= (v != 0u && v != kOne) ? 1u : 0u;
            word |= (uint32_t)(v == kOne) << i;
        }
        bits[w] = word;
    }
    return other == 0;
}

#ifdef LZHIP_X86_PACK
__attribute__((target("avx512f"))) inline bool avx512(const float* in, uint32_t* bits) {
    const __m512i one = _mm512_set1_epi32((int)kOne), zero = _mm512_setzero_si512();
    unsigned other = 0;
    for (int w = 0; w < kWords; w++) {
        const __m512i a = _mm512_loadu_si512(in + 32 * w), b = _mm512_loadu_si512(in + 32 * w + 16);
        const __mmask16 ma = _mm512_cmpeq_epi32_mask(a, one), mb = _mm512_cmpeq_epi32_mask(b, one);
        other |= _mm512_mask_cmpneq_epi32_mask((__mmask16)~ma, a, zero);
        other |= _mm512_mask_cmpneq_epi32_mask((__mmask16)~mb, b, zero);
        bits[w] = (uint32_t)ma | (uint32_t)mb << 16;
    }
    return other == 0 && scalar(in + 32 * kWords, bits + kWords, 0, kTail);
}

__attribute__((target("avx2"))) inline bool avx2(const float* in, uint32_t* bits) {
    const __m256i one = _mm256_set1_epi32((int)kOne), zero = _mm256_setzero_si256();
    __m256i fine = _mm256_set1_epi32(-1);
    for (int w = 0; w < kWords; w++) {
        uint32_t word = 0;
        for (int q = 0; q < 4; q++) {
            const __m256i v = _mm256_loadu_si256(
                reinterpret_cast<const __m256i*>(in + 32 * w + 8 * q));
            const __m256i eq = _mm256_cmpeq_epi32(v, one);
            fine = _mm256_and_si256(fine, _mm256_or_si256(eq, _mm256_cmpeq_epi32(v, zero)));
            word |= (uint32_t)_mm256_movemask_ps(_mm256_castsi256_ps(eq)) << (8 * q);
        }
        bits[w] = word;
    }
    return _mm256_movemask_ps(_mm256_castsi256_ps(fine)) == 0xff &&
           scalar(in + 32 * kWords, bits + kWords, 0, kTail);
}
#endif

}  // namespace plane_bits

// Packs planes that hold only +0.0f and 1.0f; false (and `bits` unspecified) if any other
// value shows up.
inline bool pack_planes(const float* in, uint32_t* bits) {
#ifdef LZHIP_X86_PACK
    if (__builtin_cpu_supports("avx512f")) return plane_bits::avx512(in, bits);
    if (__builtin_cpu_supports("avx2")) return plane_bits::avx2(in, bits);
#endif
    return plane_bits::scalar(in, bits, plane_bits::kWords, plane_bits::kTail);
}

}  // namespace lzhip
