// Pieces shared by the files that hold device code.
#pragma once
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace lzhip {

typedef _Float16 half_t;
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef int int4v __attribute__((ext_vector_type(4)));

constexpr int kStoreThrough = 17;  // cache policy of a raw buffer store: sc0 | sc1 (write-through)

template <typename K, typename... Args>
static inline void launch(K kernel, dim3 grid, dim3 block, hipStream_t s, LaunchTimer* t,
                          Args... args) {
    if (t && t->start) {
        hipExtLaunchKernelGGL(kernel, grid, block, 0, s, t->start, t->stop, 0, args...);
    } else {
        hipLaunchKernelGGL(kernel, grid, block, 0, s, args...);
    }
}

template <typename P>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const P* base, size_t bytes) {
    // untyped 32-bit-element descriptor for gfx9-family raw buffer instructions
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<P*>(base), 0, (int)bytes, 0x00020000);
}

}  // namespace lzhip
