// Multi-token Q8_0 products of few tokens, exact, on gfx950's int8 matrix
// cores, the weights read once as they were uploaded.
//
// The tiled GEMM (q8_gemm.hip) gives a workgroup 128 rows x 64 tokens, so a
// product of a handful of tokens leaves most of the chip idle (4096 rows: 32
// workgroups on 256 CUs), and a per-block scale matrix is read as its folded
// digit planes, three bytes a weight. Such a product is bound by the
// weights' bytes, so here a workgroup takes one tile of rows and all its
// waves walk interleaved k steps of it: operands go straight from
// memory into registers, a ring of steps deep enough to keep the CU's share
// of HBM busy, and the waves' integer sums meet in LDS at the end (exact:
// the whole row's sum fits int32, see q8_gemm.hip). With per-block scales
// each lane holds 16 weights of one row and one block, so it forms their
// digits itself: w' = q * f, f = the block's scale over the row's least
// power of two (under 2^16), three signed byte digits, about 70 VALU
// instructions per 16 weights beside nine matrix instructions.
//
// Measured against the tiled GEMM (us per product, preparation included):
// 4096 x 14336 per-block scales, 13 tokens 225 -> 23.4 (2.7 TB/s of weights);
// 6144 x 4096 row scales, 77 tokens 39.6 -> 26.5; 4096 x 4096 per-block, 24
// tokens 81 -> 22; and where an unfolded per-block matrix went through the
// one-token kernel once per token, 24 tokens of 4096 x 4096 93 -> 22.
//
// Q16.16 matrices (the per-layer-embedding projections of gemma-dense) come
// as two digit planes made once, a step of both read as they are.
//
// Two shapes: SH = 16 (16 rows x 16 tokens, v_mfma_i32_16x16x64_i8, twice
// the workgroups) for up to 16 tokens, SH = 32 (32 x 32,
// v_mfma_i32_32x32x32_i8) for more, one 32-token tile per workgroup; the
// workgroups of one row tile are dealt to the same XCD one after the other,
// so that its L2 fetches the weights once. Launches of at most one tile per
// CU split a tile over eight waves; larger ones over four, so that a CU
// holds two to four workgroups and one's start and end overlap another's
// stream (28672 x 4096, 16 tokens: 58 -> 42 us with eight waves -> four).
// Four k steps in flight per wave: six hold the 16-row shape at 139
// registers and one workgroup per CU, five spill its per-block form.
#include <cstdio>
#include <type_traits>

#include "detnum_dev.h"
#include "q8_epilogue.h"
#include "q8_gemm_common.h"

namespace {

template <int SH>
struct Shape;
template <>
struct Shape<16> {
    using Acc = v4i;
    static constexpr int EL = 4;         // outputs per lane
    static constexpr uint32_t NB = 2;    // 32-wide blocks per k step
    static __device__ __forceinline__ Acc mfma(v4i a, v4i b, Acc c) {
        return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
    }
    // Output i of a lane: its row and token within the tile.
    static __device__ __forceinline__ uint32_t row(uint32_t lane, uint32_t i) { return 4 * (lane / 16) + i; }
};
template <>
struct Shape<32> {
    using Acc = v16i;
    static constexpr int EL = 16;
    static constexpr uint32_t NB = 1;
    static __device__ __forceinline__ Acc mfma(v4i a, v4i b, Acc c) {
        return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t row(uint32_t lane, uint32_t i) {
        return 8 * (i / 4) + 4 * (lane / 32) + i % 4;
    }
};

// Four weights (the bytes of q) times f, as three signed byte digits: byte
// l of w + 0x808080, xor 0x80, l = 0..2, packed low to high per digit.
// |q * f| < 2^23 (the launch's rule), so each product and sum is a 24-bit
// multiply-add.
__device__ __forceinline__ void weight_digits(uint32_t q, int32_t f, int (&d)[3], int bias) {
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; k++) w[k] = (uint32_t)(__mul24((int32_t)(int8_t)(q >> (8 * k)), f) + bias);
    const uint32_t a = __builtin_amdgcn_perm(w[1], w[0], 0x05010400), b = __builtin_amdgcn_perm(w[3], w[2], 0x05010400);
    const uint32_t hi = __builtin_amdgcn_perm(w[1], w[0], 0x0c0c0602) | __builtin_amdgcn_perm(w[3], w[2], 0x06020c0c);
    d[0] = (int)(__builtin_amdgcn_perm(b, a, 0x05040100) ^ 0x80808080u);
    d[1] = (int)(__builtin_amdgcn_perm(b, a, 0x07060302) ^ 0x80808080u);
    d[2] = (int)(hi ^ 0x80808080u);
}

// One tile of rows against one tile of tokens, LG activation digits, MODE's
// scales. DEPTH k steps of each wave are in flight.
template <int SH, int MODE, int LG, int DEPTH, uint32_t SK_WAVES>
__device__ __forceinline__ void skinny_tile(const GemvArgs& a, int32_t* smem, uint32_t rt, uint32_t tt) {
    using S = Shape<SH>;
    using Acc = typename S::Acc;
    constexpr int WP = MODE == Q8_SCALE_ROW ? 1 : MODE == Q16_PLANES ? 2 : 3, NS = WP + LG - 1;
    constexpr int QP = MODE == Q16_PLANES ? 2 : 1;  // weight planes read
    constexpr uint32_t SK_THREADS = 64 * SK_WAVES;
    const Q8View& w = a.w;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t KB = w.nb, TT = (a.tokens + 31) / 32, steps = KB / S::NB;
    const size_t lstride = (size_t)TT * KB * FRAG;
    // This lane's row, its 16 bytes of a step's weights and its scale.
    const uint32_t r = lane % SH, tile16 = SH == 16 ? rt : min(2 * rt + r / 16, w.tiles - 1);
    const uint32_t row = tile16 * 16 + r % 16;
    const uint8_t* qp = (MODE == Q16_PLANES ? (const uint8_t*)w.fold_planes : w.qs) + (size_t)tile16 * KB * Q8_TILE_BLOCK_BYTES +
                        (SH == 16 ? lane * 16 : (lane / 32) * 256 + (r % 16) * 16);
    const size_t qstride = (size_t)w.tiles * KB * Q8_TILE_BLOCK_BYTES;
    const uint16_t* sp = MODE == Q8_SCALE_F16 ? w.sc16 + ((size_t)tile16 * KB + (SH == 16 ? lane / 32 : 0)) * 16 + r % 16
                                              : nullptr;
    const int32_t least = MODE == Q8_SCALE_F16 ? w.fold_shift[row] : 0;
    // ... and its 16 bytes of a step's digits (token tile tt; the 16-token
    // shape takes the tile's first half).
    const int8_t* bp = a.planes + (size_t)tt * KB * FRAG +
                       (SH == 16 ? (lane / 32) * FRAG + ((lane / 16 % 2) * 32 + lane % 16) * 16 : lane * 16);

    Acc acc[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) acc[s] = Acc{};
    v4i q[DEPTH][QP], b[DEPTH][LG];
    uint32_t sc[DEPTH];
    auto load = [&](int u, uint32_t step) __attribute__((always_inline)) {
        // Past the end: the last step again (never used), so no branch
        // separates the loads from their waits.
        const uint32_t kb = min(step, steps - 1) * S::NB;
#pragma unroll
        for (int p = 0; p < QP; p++) q[u][p] = *(const v4i*)(qp + p * qstride + (size_t)kb * Q8_TILE_BLOCK_BYTES);
        if (MODE == Q8_SCALE_F16) sc[u] = sp[(size_t)kb * 16];
#pragma unroll
        for (int l = 0; l < LG; l++) b[u][l] = *(const v4i*)(bp + l * lstride + (size_t)kb * FRAG);
    };
    auto compute = [&](int u) __attribute__((always_inline)) {
        if (MODE != Q8_SCALE_F16) {
#pragma unroll
            for (int l = 0; l < LG; l++)
#pragma unroll
                for (int p = 0; p < QP; p++) acc[p + l] = S::mfma(q[u][p], b[u][l], acc[p + l]);
        } else {
            const uint32_t e = (sc[u] >> 10) & 0x1f, mant = sc[u] & 0x3ff;
            const int32_t m = (int32_t)(e ? 1024 + mant : mant);
            const int32_t up = m << (m ? max((int32_t)e - 1, 0) - least : 0), f = sc[u] & 0x8000 ? -up : up;
            v4i wd[WP];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                int d[3];
                weight_digits((uint32_t)q[u][0][c], f, d, 0x808080);
#pragma unroll
                for (int p = 0; p < WP; p++) wd[p][c] = d[p];
            }
#pragma unroll
            for (int l = 0; l < LG; l++)
#pragma unroll
                for (int p = 0; p < WP; p++) acc[p + l] = S::mfma(wd[p], b[u][l], acc[p + l]);
        }
    };
    // The wave's steps wave, wave + 8, ...: neighbouring waves read
    // neighbouring runs of the weights.
#pragma unroll
    for (int u = 0; u < DEPTH; u++) load(u, wave + u * SK_WAVES);
    uint32_t step = wave;
    for (; step + (DEPTH - 1) * SK_WAVES < steps; step += DEPTH * SK_WAVES) {
#pragma unroll
        for (int u = 0; u < DEPTH; u++) {
            compute(u);
            load(u, step + (DEPTH + u) * SK_WAVES);
        }
    }
#pragma unroll
    for (int u = 0; u < DEPTH - 1; u++)
        if (step + u * SK_WAVES < steps) compute(u);

    // The waves' sums, one shared-shift accumulator at a time through LDS
    // (two buffers, so one barrier each): thread (wave, lane) keeps outputs
    // wave, wave + 8, ... of its lane.
    constexpr int MINE = (S::EL + SK_WAVES - 1) / SK_WAVES;
    using Tot = typename std::conditional<(LG <= 3), int64_t, dn::i128>::type;  // |total| < 2^61 at three digits each
    Tot tot[MINE];
#pragma unroll
    for (int m = 0; m < MINE; m++) tot[m] = 0;
#pragma unroll
    for (int s = 0; s < NS; s++) {
        int32_t* buf = smem + (s & 1) * (SK_WAVES * S::EL * 64);
#pragma unroll
        for (int e = 0; e < S::EL; e++) buf[(wave * S::EL + e) * 64 + lane] = acc[s][e];
        lds_barrier();
#pragma unroll
        for (int m = 0; m < MINE; m++) {
            const uint32_t e = wave + m * SK_WAVES;
            if (e < (uint32_t)S::EL) {
                int32_t sum = 0;  // the whole row's plane sum: fits int32
#pragma unroll
                for (uint32_t v = 0; v < SK_WAVES; v++) sum += buf[(v * S::EL + e) * 64 + lane];
                tot[m] += (Tot)sum * ((Tot)1 << (8 * s));
            }
        }
    }
    lds_barrier();
    // Rounded once (q8.rs:94-104), parked as [row][token].
    constexpr uint32_t STRIDE = SH + 1;
#pragma unroll
    for (int m = 0; m < MINE; m++) {
        const uint32_t e = wave + m * SK_WAVES;
        if (e < (uint32_t)S::EL) {
            const uint32_t rl = S::row(lane, e), orow = rt * SH + rl;
            int32_t v = 0;
            if (orow < w.rows)
                v = MODE == Q8_SCALE_ROW ? dn::round_to_i32((dn::i128)tot[m] * (dn::i128)w.row_scale[orow], 24)
                                         : dn::round_to_i32((dn::i128)((dn::u128)(dn::i128)tot[m] << w.fold_shift[orow]), 24);
            smem[rl * STRIDE + lane % SH] = v;
        }
    }
    __syncthreads();
    const uint32_t row0 = rt * SH, tok0 = tt * 32;
    if (a.epilogue != EPI_SWIGLU && a.epilogue != EPI_GEGLU) {
        for (uint32_t c = tid; c < SH * SH; c += SK_THREADS) {
            const uint32_t rl = c % SH, tl = c / SH;
            if (row0 + rl >= w.rows || tok0 + tl >= a.tokens) continue;
            if (MODE == Q16_PLANES && a.epilogue == EPI_GELU_MUL)
                a.out[(size_t)(tok0 + tl) * a.out_stride + row0 + rl] = dn::mul_sat(
                    dn::gelu(smem[rl * STRIDE + tl]), a.residual[(size_t)(tok0 + tl) * a.residual_stride + row0 + rl]);
            else
                store_output(a, row0 + rl, tok0 + tl, smem[rl * STRIDE + tl], smem[(rl ^ 1) * STRIDE + tl]);
        }
        return;
    }
    // Gate and up rows alternate: one activation per pair, left in the
    // gate's slot for the digit planes of the next product.
    constexpr uint32_t PAIRS = SH / 2;
    for (uint32_t c = tid; c < PAIRS * SH; c += SK_THREADS) {
        const uint32_t pl = c % PAIRS, tl = c / PAIRS, pair = row0 / 2 + pl, token = tok0 + tl;
        if (2 * pair >= w.rows || token >= a.tokens) continue;
        const int32_t gate = smem[2 * pl * STRIDE + tl], up = smem[(2 * pl + 1) * STRIDE + tl];
        const int32_t act = a.epilogue == EPI_GEGLU ? dn::gelu(gate) : dn::silu_quick(gate, a.silu_tab);
        const int32_t o = dn::mul_sat(act, up);
        if (a.out) a.out[(size_t)token * a.out_stride + pair] = o;
        smem[2 * pl * STRIDE + tl] = o;
    }
    if (!a.out_gemm_planes) return;
    // PAIRS consecutive gated values of one token are PAIRS bytes of one
    // operand lane per plane (digit_planes_kernel's layout); the digits they
    // need raise the (k chunk, token tile)'s count.
    int* s_need = smem + SH * STRIDE;
    if (tid == 0) *s_need = 1;
    __syncthreads();
    if (tid < SH) {
        const uint32_t tl = tid, token = tok0 + tl, pair0 = row0 / 2, K = w.rows / 2;
        if (pair0 < K) {
            int8_t* dst = a.out_gemm_planes + ((size_t)tt * (K / 32) + pair0 / 32) * FRAG +
                          (tl + 32 * ((pair0 % 32) / 16)) * 16 + pair0 % 16;
            int need = 1;
            uint32_t out[PL_MAX][PAIRS / 4];
#pragma unroll
            for (uint32_t c = 0; c < PAIRS / 4; c++) {
                uint64_t d[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    d[k] = digits5(token < a.tokens ? smem[2 * (4 * c + k) * STRIDE + tl] : 0);
                    need = max(need, limbs_needed(d[k]));
                }
#pragma unroll
                for (int l = 0; l < PL_MAX; l++) out[l][c] = plane_byte4(d[0], d[1], d[2], d[3], l);
            }
#pragma unroll
            for (int l = 0; l < PL_MAX; l++)
#pragma unroll
                for (uint32_t c = 0; c < PAIRS / 4; c += 2)
                    *(uint2*)(dst + l * ((size_t)TT * K) * 32 + 4 * c) = make_uint2(out[l][c], out[l][c + 1]);
            atomicMax(s_need, need);
        }
    }
    __syncthreads();
    if (tid == 0 && row0 / 2 < w.rows / 2)
        atomicMax(&a.out_gemm_limbs[a.tokens + row0 / 2 / (32 * PLANE_KB) * TT + tt], *s_need);
}

template <int SH, int MODE, uint32_t W>
__global__ __launch_bounds__(64 * W, SH == 16 ? 4 : 2) void q8_skinny_kernel(const GemvArgs a, uint32_t row_tiles,
                                                                            uint32_t tok_tiles) {
    __shared__ __attribute__((aligned(16))) int32_t smem[2 * W * Shape<SH>::EL * 64];
    // Groups of 8 row tiles, one per XCD, each with its token tiles in turn.
    const uint32_t g = blockIdx.x / (8 * tok_tiles), in = blockIdx.x % (8 * tok_tiles);
    const uint32_t rt = g * 8 + in % 8, tt = in / 8;
    if (rt >= row_tiles) return;
    if (tiles_limbs<1>(a, tt) <= 3) skinny_tile<SH, MODE, 3, 4, W>(a, smem, rt, tt);
    else skinny_tile<SH, MODE, 5, 3, W>(a, smem, rt, tt);
}

}  // namespace

// Whether a product the tiled GEMM takes too is faster here: its tiles make
// few enough rounds of the chip that reading the operands per tile costs less
// than the GEMM's idle CUs, and with per-block scales than its three bytes a
// weight. Up to 16 tokens it always is (28672 x 4096: 62.0 / 41.6 row scales
// and 89.4 / 48.7 per block); beyond, us of the GEMM / this kernel,
// preparation included, matrices rotated through more than the last cache,
// at tokens (tiles per CU) around where they cross:
//   row scales  4096 x 4096   192 (3.0)  33.4 / 29.7    224 (3.5)  34.2 / 35.0    256 (4.0)  34.1 / 36.4
//               4096 x 14336  160 (2.5)  85.8 / 87.3    192 (3.0)  89.6 / 87.6    224 (3.5)  88.2 / 105.5
//               6144 x 4096   128 (3.0)  39.8 / 34.1    160 (3.8)  40.4 / 39.7    192 (4.5)  40.5 / 45.6
//               2048 x 2048   384 (3.0)  23.9 / 22.4    448 (3.5)  25.0 / 27.1
//               16384 x 2048   64 (4.0)  34.7 / 29.3     96 (6.0)  26.9 / 35.8
//               28672 x 4096   32 (3.5)  63.4 / 48.6     64 (7.0)  59.6 / 67.1
//   per block   4096 x 4096   320 (5.0)  71.5 / 70.8    384 (6.0)  80.3 / 81.5
//               4096 x 14336  320 (5.0) 227.7 / 201.5   384 (6.0) 231.8 / 236.1
//               6144 x 4096   192 (4.5)  69.9 / 68.0    224 (5.3)  75.3 / 76.4
//               16384 x 2048   64 (4.0)  41.9 / 37.4     96 (6.0)  47.5 / 50.1
//               28672 x 4096   32 (3.5)  95.1 / 58.5     64 (7.0)  90.4 / 95.6
// (Up to 64 tokens the GEMM's narrowest workgroup is one token group, partly
// empty, so row scales cross later there.)
static bool few_tiles(const GemvArgs& a) {
    const uint32_t per_cu = a.w.scale_mode == Q8_SCALE_F16 ? 5 : a.tokens <= 64 ? 4 : 3;
    return a.tokens <= 16 ||
           (uint64_t)((a.w.tiles + 1) / 2) * ((a.tokens + 31) / 32) <= (uint64_t)per_cu * (uint32_t)iris_device_cus();
}

// The shape of a launch: tiles of 16 or 32 rows and tokens, and the waves
// that share one's k steps.
struct SkinnyLaunch {
    uint32_t side, waves, row_tiles, tok_tiles;
    // Groups of 8 row tiles, one per XCD, each with its token tiles in turn.
    uint64_t blocks() const { return (uint64_t)(row_tiles + 7) / 8 * 8 * tok_tiles; }
    uint64_t threads() const { return 64 * waves * blocks(); }
};

static SkinnyLaunch skinny_shape(const GemvArgs& a) {
    const bool small = a.tokens <= 16;
    const uint32_t row_tiles = small ? a.w.tiles : (a.w.tiles + 1) / 2, tok_tiles = (a.tokens + 31) / 32;
    return {small ? 16u : 32u, (uint64_t)row_tiles * tok_tiles <= (uint32_t)iris_device_cus() ? 8u : 4u, row_tiles, tok_tiles};
}

bool iris_skinny_applies(const GemvArgs& a) {
    if (!a.planes || !a.token_limbs || a.tokens < 2 || a.w.cols % 64 || a.epilogue == EPI_HEAD_SELECT ||
        a.prologue == PRO_NORM_RES_NORM || a.tokens > 65535)
        return false;
    // A launch holds fewer than 2^32 threads.
    if (skinny_shape(a).threads() >> 32) return false;
    if (a.w.scale_mode == Q8_SCALE_ROW) return a.w.cols < (1u << 17) && few_tiles(a);
    // The planes' only path, whatever the tokens (two shared-shift terms).
    if (a.w.scale_mode == Q16_PLANES)
        return a.w.cols <= 16384 && (a.epilogue == EPI_STORE || a.epilogue == EPI_GELU_MUL);
    // Per-block scales: three weight digits suffice (the upload's bound) and
    // the shared-shift sums stay below 2^31. Without folded planes this is
    // the only matrix-core path, whatever the tokens; work space that is not
    // aligned as the GEMM asks leaves such a product on the vector path.
    if (!a.w.fold_planes && ((uintptr_t)a.planes & 255)) return false;
    return a.w.scale_mode == Q8_SCALE_F16 && a.w.fold_shift && a.w.digits_bound >= 1 && a.w.digits_bound <= 3 &&
           a.w.cols <= 16384 && (few_tiles(a) || !a.w.fold_planes);
}

int iris_skinny_launch(const GemvArgs& a, hipStream_t stream) {
    const SkinnyLaunch s = skinny_shape(a);
    const uint32_t row_tiles = s.row_tiles, tok_tiles = s.tok_tiles;
    const dim3 grid((uint32_t)s.blocks());
    auto launch = [&](auto sh, auto w) {
        constexpr int SH = decltype(sh)::value;
        constexpr uint32_t W = decltype(w)::value;
        if (a.w.scale_mode == Q8_SCALE_ROW)
            hipLaunchKernelGGL((q8_skinny_kernel<SH, Q8_SCALE_ROW, W>), grid, dim3(64 * W), 0, stream, a, row_tiles, tok_tiles);
        else if (a.w.scale_mode == Q16_PLANES)
            hipLaunchKernelGGL((q8_skinny_kernel<SH, Q16_PLANES, W>), grid, dim3(64 * W), 0, stream, a, row_tiles, tok_tiles);
        else
            hipLaunchKernelGGL((q8_skinny_kernel<SH, Q8_SCALE_F16, W>), grid, dim3(64 * W), 0, stream, a, row_tiles, tok_tiles);
    };
    using std::integral_constant;
    if (s.side == 16 && s.waves == 8) launch(integral_constant<int, 16>{}, integral_constant<uint32_t, 8>{});
    else if (s.side == 16) launch(integral_constant<int, 16>{}, integral_constant<uint32_t, 4>{});
    else if (s.waves == 8) launch(integral_constant<int, 32>{}, integral_constant<uint32_t, 8>{});
    else launch(integral_constant<int, 32>{}, integral_constant<uint32_t, 4>{});
    return (int)hipGetLastError();
}

void iris_skinny_route(const GemvArgs& a, char* name, size_t size) {
    const SkinnyLaunch s = skinny_shape(a);
    std::snprintf(name, size, "few %ux%u, %u waves", s.side, s.side, s.waves);
}
