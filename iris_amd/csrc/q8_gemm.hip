// Multi-token Q8_0 products on gfx950's int8 matrix cores, exact.
//
// When every block of a row shares one scale (the row-scale layout),
// det_num::q8::dot_row (crates/det-num/src/q8.rs:56-72) of a token is the
// single ties-to-even rounding of scale[row] * sum_b blocksum_b, and the
// block sums add up to the full-row integer dot product sum_k q[row][k] *
// x[k] (|.| < K * 2^38). So the product is an integer GEMM followed by the
// GEMV's rounding and epilogue. The activations are split into signed byte
// digits, x = sum_l 256^l d_l with d_l in [-128, 127] (the bytes of
// x + 0x8080808080, each xor 0x80; five digits only for x >= 0x7F7F7F80),
// and every digit plane is an int8 GEMM with exact int32 accumulation
// (|sum| <= K * 2^14 < 2^31 for K < 2^17) on v_mfma_i32_32x32x32_i8.
//
// Operand layout. One v_mfma_i32_32x32x32_i8 takes, in lane l, 16 bytes of
// row (A) or column (B) l % 32 at reduction offset 16 * (l / 32), and
// leaves output i of lane l at row 8 * (i / 4) + 4 * (l / 32) + i % 4,
// column l % 32. (On gfx950 this instruction runs at about twice the rate
// of the 16x16x64 one.) A weight operand, 32 rows by 32 k, is four 256-byte
// runs of the Q8_0 tile layout (two 16-row tiles, two 16-byte halves of a
// 32-wide block); the digit planes are written directly in operand shape:
// plane l, 32-token tile tt and 32-wide k block kb form one 1 KB block at
// ((l * TT + tt) * KB + kb) * 1024. Every operand is copied from global
// memory straight into LDS (global_load_lds_dwordx4: each lane fetches its
// own 16 bytes, the wave writes one contiguous kilobyte, no registers in
// between) through a ring of 64-wide k steps, and read back by each lane as
// one conflict-free 16-byte LDS load.
//
// This file: the activations' preparation and the dispatch. The tiled
// products are in q8_gemm_row.hip and q8_gemm_fold.hip, those of few tokens
// in q8_skinny.hip.
#include "detnum_dev.h"
#include "q8_gemm_common.h"
#include "q8_gemm_row.h"
#include "q8_internal.h"

namespace {

// Per token, one workgroup each, under the rms_norm prologue only: the
// token's scale (ops.rs:98-114, rms_norm_scale of the order-free saturating
// sum of squares) at token_limbs[t]. A launch of few tokens lasts as long as
// one token's chain, so its row is spread over four waves with four loads in
// flight per lane (K = 4096: one round; one wave with one load at a time
// took 9.2 us for 45 tokens and 9.6 for 512, now 4.7 and 5.3).
__global__ __launch_bounds__(256) void token_prep_kernel(const GemvArgs a) {
    __shared__ int64_t s_sum[4];
    const uint32_t t = blockIdx.x, tid = threadIdx.x, K4 = a.w.cols / 4;
    const int4* x = (const int4*)(a.x + (size_t)t * a.x_stride);
    int64_t s = 0;
    for (uint32_t k = tid; k < K4; k += 1024) {
        int4 v[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) v[u] = x[min(k + 256 * u, K4 - 1)];
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) {
            if (k + 256 * u >= K4) continue;
            s = dn::acc_add_sat(s, (int64_t)v[u].x * v[u].x);
            s = dn::acc_add_sat(s, (int64_t)v[u].y * v[u].y);
            s = dn::acc_add_sat(s, (int64_t)v[u].z * v[u].z);
            s = dn::acc_add_sat(s, (int64_t)v[u].w * v[u].w);
        }
    }
    for (int off = 32; off >= 1; off >>= 1) s = dn::acc_add_sat(s, __shfl_xor(s, off));
    if (tid % 64 == 0) s_sum[tid / 64] = s;
    __syncthreads();
    if (tid) return;
    for (int i = 1; i < 4; i++) s = dn::acc_add_sat(s, s_sum[i]);
    a.token_limbs[t] = dn::rms_scale_from_sum(s, a.w.cols, a.norm_eps);
}

// The digit planes of one 32-token tile over PLANE_KB k blocks (one k
// chunk) per workgroup, after the optional rms_norm (mul_sat(mul_sat(v,
// scale), w)), in the operand layout above, and the digits the chunk's
// values need, stored for the (chunk, tile) at token_limbs[M + chunk * TT +
// tile]: every launch writes each of its counts, so none needs a reset.
// Tokens past the end of the last tile get zero digits. A launch of few
// workgroups takes one wave per k block, so that it lasts one load's latency
// instead of two (K = 4096, us: 45 tokens 8.2 -> 6.4); with many, four waves
// of two blocks each are faster (2048 tokens, normed: 21.5 against 26.5).
// The gated rows' counts, which the product's workgroups raise, start at 1:
// set here (ones of them) for the product that follows.
constexpr uint32_t DP_THREADS = 64 * PLANE_KB;
__global__ __launch_bounds__(DP_THREADS) void digit_planes_kernel(const GemvArgs a, uint32_t ones) {
    __shared__ int s_need;
    const uint32_t tt = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t K = a.w.cols, M = a.tokens, TT = (M + 31) / 32, KB = K / 32;
    const uint32_t kb0 = blockIdx.y * PLANE_KB, kb1 = min(kb0 + PLANE_KB, KB);
    const bool norm = a.prologue == PRO_RMSNORM;
    for (uint32_t i = (blockIdx.y * gridDim.x + blockIdx.x) * blockDim.x + tid; i < ones;
         i += gridDim.x * gridDim.y * blockDim.x)
        a.out_gemm_limbs[M + i] = 1;
    if (tid == 0) s_need = 1;
    __syncthreads();
    // Lane l writes the 16 bytes of token l % 32 at k-offset 16 * (l / 32)
    // of each 32-wide block the wave takes.
    const uint32_t tl = lane & 31, q = lane >> 5, t = tt * 32 + tl;
    const bool valid = t < M;
    const int32_t scale = norm && valid ? a.token_limbs[t] : 0;
    const int32_t* x = a.x + (size_t)(valid ? t : 0) * a.x_stride;
    const size_t lstride = (size_t)TT * KB * FRAG;
    int need = 1;
    for (uint32_t kb = kb0 + wave; kb < kb1; kb += blockDim.x / 64) {
        const uint32_t k0 = kb * 32 + q * 16;
        uint32_t out[PL_MAX][4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            int4 v = *(const int4*)(x + k0 + 4 * c);  // not behind a branch: all are in flight together
            if (!valid) v = make_int4(0, 0, 0, 0);
            if (norm) {
                const int4 nw = *(const int4*)(a.norm_w + k0 + 4 * c);
                v.x = dn::mul_sat(dn::mul_sat(v.x, scale), nw.x);
                v.y = dn::mul_sat(dn::mul_sat(v.y, scale), nw.y);
                v.z = dn::mul_sat(dn::mul_sat(v.z, scale), nw.z);
                v.w = dn::mul_sat(dn::mul_sat(v.w, scale), nw.w);
            }
            const uint64_t d0 = digits5(v.x), d1 = digits5(v.y), d2 = digits5(v.z), d3 = digits5(v.w);
            need = max(need, max(max(limbs_needed(d0), limbs_needed(d1)), max(limbs_needed(d2), limbs_needed(d3))));
#pragma unroll
            for (int l = 0; l < PL_MAX; l++) out[l][c] = plane_byte4(d0, d1, d2, d3, l);
        }
        int8_t* dst = a.planes + ((size_t)tt * KB + kb) * FRAG + lane * 16;
#pragma unroll
        for (int l = 0; l < PL_MAX; l++)
            *(uint4*)(dst + l * lstride) = make_uint4(out[l][0], out[l][1], out[l][2], out[l][3]);
    }
    for (int off = 32; off >= 1; off >>= 1) need = max(need, __shfl_xor(need, off));
    if (lane == 0) atomicMax(&s_need, need);  // the largest of the waves: any order
    __syncthreads();
    if (tid == 0) a.token_limbs[M + blockIdx.y * TT + tt] = s_need;
}

}  // namespace

bool iris_gemm_applies(const GemvArgs& a) {
    if (iris_skinny_applies(a)) return true;
    if (!a.planes || !a.token_limbs || a.tokens < 2 || a.w.cols % 64 || a.epilogue == EPI_HEAD_SELECT ||
        a.prologue == PRO_NORM_RES_NORM)
        return false;
    if (a.w.scale_mode == Q8_SCALE_ROW) return a.w.cols < (1u << 17);
    // Folded per-block scales: shared-shift sums stay below 2^31.
    return a.w.scale_mode == Q8_SCALE_F16 && a.w.fold_planes && a.w.fold_nplanes >= 1 &&
           a.w.fold_nplanes <= Q8_FOLD_MAX_PLANES && a.w.cols <= 16384;
}

int iris_gemm_launch(const GemvArgs& a, hipStream_t stream) {
    if (!iris_gemm_applies(a) || a.x_stride % 4 || ((uintptr_t)a.x & 15) || ((uintptr_t)a.planes & 255))
        return IRIS_E_INVALID;
    if (a.prologue == PRO_RMSNORM && ((uintptr_t)a.norm_w & 15)) return IRIS_E_INVALID;
    // (Ready planes are the down product's: what sets the gated rows' counts
    // is the launch that makes the planes.)
    if (a.planes_ready && (a.prologue != PRO_NONE || a.out_gemm_planes)) return IRIS_E_INVALID;
    const bool gated = a.epilogue == EPI_SWIGLU || a.epilogue == EPI_GEGLU;
    if (a.out_gemm_planes && (!gated || !a.out_gemm_limbs || (a.w.rows / 2) % 32 || ((uintptr_t)a.out_gemm_planes & 255) ||
                              a.out_gemm_planes == a.planes || a.out_gemm_limbs == a.token_limbs))
        return IRIS_E_INVALID;
    if (!a.out && !a.out_gemm_planes) return IRIS_E_INVALID;
    const uint32_t TT = (a.tokens + 31) / 32, KB = a.w.cols / 32;
    // The gated rows' counts start at 1 (every workgroup raises its own).
    const uint32_t ones = a.out_gemm_planes ? (uint32_t)(gemm_limb_ints(a.w.rows / 2, a.tokens) - a.tokens) : 0;
    if (!a.planes_ready) {
        if (a.prologue == PRO_RMSNORM)
            hipLaunchKernelGGL(token_prep_kernel, dim3(a.tokens), dim3(256), 0, stream, a);
        const dim3 grid(TT, (KB + PLANE_KB - 1) / PLANE_KB);
        const bool few = grid.x * grid.y <= 2 * (uint32_t)iris_device_cus();
        hipLaunchKernelGGL(digit_planes_kernel, grid, dim3(few ? DP_THREADS : 256), 0, stream, a, ones);
    }
    hipError_t st = hipGetLastError();
    if (st != hipSuccess) return (int)st;
    if (iris_skinny_applies(a)) return iris_skinny_launch(a, stream);
    return a.w.scale_mode == Q8_SCALE_F16 ? iris_gemm_fold_launch(a, stream) : iris_gemm_row_launch(a, stream);
}

void iris_gemm_route(const GemvArgs& a, char* name, size_t size) {
    if (iris_skinny_applies(a)) iris_skinny_route(a, name, size);
    else if (a.w.scale_mode == Q8_SCALE_F16) iris_gemm_fold_route(a, name, size);
    else iris_gemm_row_route(a, name, size);
}
