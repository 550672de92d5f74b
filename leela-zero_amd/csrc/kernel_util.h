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

// The border of padded planes, as far as a tap of some point reads it: the last cell before the first
// board, and of every board the row above it and the cell that ends each row, and the row below the
// last.  Thread i clears a piece of one cell; 39 n + 21 cells of 400 (n + 2).
__device__ __forceinline__ void clear_border(const PlaneBorders& p, unsigned i) {
    const unsigned per = p.w0 + 3 * p.w, j = i / per, q = i - j * per;
    if (j >= 39u * p.n + 21u) return;
    const unsigned b = (j + 38) / 39, r = j + 38 - b * 39;   // (from the cell before the first board)
    const unsigned cell = b * kPadCells + (r < 20 ? r : (r - 19) * 20 + 19);
    const unsigned cells = (p.n + 2) * kPadCells;
    const unsigned plane = q < p.w0 ? 0u : (q - p.w0) / p.w;
    const size_t at = q < p.w0 ? (size_t)cell * p.w0 + q
                               : (size_t)cells * (p.w0 + plane * p.w) + (size_t)cell * p.w +
                                     (q - p.w0 - plane * p.w);
    p.planes[at] = int4v{0, 0, 0, 0};
}
static inline unsigned border_pieces(const PlaneBorders* p) {
    return p ? (39u * p->n + 21u) * (p->w0 + 3 * p->w) : 0u;
}

}  // namespace lzhip
