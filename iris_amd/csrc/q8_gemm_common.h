// What the multi-token products share: the activations' signed byte digits
// and the digit counts their preparation leaves (q8_gemm.hip).
#pragma once

#include "q8_internal.h"

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int PL_MAX = 5;             // digit planes of an i32
constexpr uint32_t FRAG = 1024;       // bytes of one 32 x 32 operand
constexpr uint32_t PLANE_KB = GEMM_PLANE_KB;

__device__ __forceinline__ uint64_t digits5(int32_t v) {
    return (uint64_t)((int64_t)v + 0x8080808080LL) ^ 0x8080808080ULL;
}

__device__ __forceinline__ int limbs_needed(uint64_t d) {
    return (d >> 32) ? 5 : (d >> 24) ? 4 : (d >> 16) ? 3 : (d >> 8) ? 2 : 1;
}

__device__ __forceinline__ uint32_t plane_byte4(uint64_t d0, uint64_t d1, uint64_t d2, uint64_t d3, int l) {
    const int sh = 8 * l;
    return (uint32_t)((d0 >> sh) & 0xff) | ((uint32_t)((d1 >> sh) & 0xff) << 8) | ((uint32_t)((d2 >> sh) & 0xff) << 16) |
           ((uint32_t)((d3 >> sh) & 0xff) << 24);
}

// The digits a workgroup's token tiles tt0 .. tt0 + tg - 1 need: the most
// any k chunk of them needs, from digit_planes_kernel's counts.
__device__ __forceinline__ int tiles_limbs(const GemvArgs& a, uint32_t tt0, uint32_t tg, int& s_limbs) {
    const uint32_t tid = threadIdx.x, TT = (a.tokens + 31) / 32;
    const uint32_t chunks = (a.w.cols / 32 + PLANE_KB - 1) / PLANE_KB;
    const int32_t* need = a.token_limbs + a.tokens;
    if (tid == 0) s_limbs = 1;
    __syncthreads();
    for (uint32_t i = tid; i < tg * chunks; i += blockDim.x) {
        const uint32_t t = tt0 + i % tg;
        if (t < TT) atomicMax(&s_limbs, need[(i / tg) * TT + t]);
    }
    __syncthreads();
    const int limbs = s_limbs;
    __syncthreads();
    return limbs;
}

// Products of few tokens (q8_skinny.hip), their digit planes already made.
bool iris_skinny_applies(const GemvArgs& a);
int iris_skinny_launch(const GemvArgs& a, hipStream_t stream);
