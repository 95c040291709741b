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

// The digits a workgroup's TG token tiles from tt0 (uniform) need: the most
// any k chunk of them needs, from digit_planes_kernel's counts. Every wave
// reads them itself through scalar loads (written by an earlier launch, only
// read here): no LDS, no barrier, and no wait on the vector loads in flight.
template <uint32_t TG>
__device__ __forceinline__ int tiles_limbs(const GemvArgs& a, uint32_t tt0) {
    const uint32_t TT = (a.tokens + 31) / 32, chunks = (a.w.cols / 32 + PLANE_KB - 1) / PLANE_KB;
    const auto* need = (const __attribute__((address_space(4))) int32_t*)(uintptr_t)(a.token_limbs + a.tokens);
    int limbs = 1;
#pragma unroll 4
    for (uint32_t c = 0; c < chunks; c++)
#pragma unroll
        for (uint32_t t = 0; t < TG; t++) limbs = max(limbs, need[c * TT + min(tt0 + t, TT - 1)]);
    return limbs;
}

// Products of few tokens (q8_skinny.hip), their digit planes already made.
bool iris_skinny_applies(const GemvArgs& a);
int iris_skinny_launch(const GemvArgs& a, hipStream_t stream);
void iris_skinny_route(const GemvArgs& a, char* name, size_t size);
