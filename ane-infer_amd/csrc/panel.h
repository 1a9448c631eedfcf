// panel.h — the panel layout of quantised weights (see gemv.hip) and the
// vector types its kernels share.
#pragma once

#include "common.h"

namespace anehip {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWave = 64;
// word 3 of a raw buffer resource on gfx9-family parts (data format 32 bit)
constexpr int kBufferWord3 = 0x00020000;

// A panel: 64 rows x 256 columns.  kChunks 16-byte quant vectors per row
// ([chunk][64 rows][16 B]), then each row's 8 fp16 block scales ([64 rows][16 B]).
template <uint32_t T> struct Panel;
template <> struct Panel<ANEHIP_GGML_Q8_0> {
    static constexpr int kChunks = 16;
    static constexpr int kBytes = 17 * 1024;
};
template <> struct Panel<ANEHIP_GGML_Q4_0> {
    static constexpr int kChunks = 8;
    static constexpr int kBytes = 9 * 1024;
};

// Barrier for LDS traffic only: the fences order LDS accesses, so waves do
// not wait for their outstanding global loads (the prefetched units) here.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

}  // namespace anehip
