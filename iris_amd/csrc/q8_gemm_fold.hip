// The tiled product of per-block scale matrices and the folding it needs.
#include <cstdio>
#include <mutex>

#include "q8_gemm_row.h"
#include "q8_gemm_tile.h"

namespace {

// ---- per-block scales on the matrix cores ----
//
// A per-block scale matrix is first folded (iris_q8_prepare_fold): with
// s_b = sign_b * m_b * 2^sh_b the exact Q.24 value of block b's f16 scale
// (m_b the integer significand, under 2^11) and R the least sh_b of the
// row's non-zero scales, w' = q * sign_b * (m_b << (sh_b - R)) are integers,
// and dot_row's total sum_b s_b * sum_j q_j x_j equals 2^R * sum_k w'_k x_k
// (crates/det-num/src/q8.rs:56-72). Each w' is split into WP signed byte
// digits like the activations, so every (weight digit p, activation digit
// l) pair is an int8 GEMM with exact int32 sums, and pairs with the same
// p + l share an accumulator (at most five terms of |.| <= K * 2^14 each:
// 5 * 2^28 < 2^31 for K <= 16384). The epilogue recombines the shifts in 128
// bits, shifts by R and rounds once at 24 fraction bits.

constexpr int32_t FOLD_NEGATED = 64;  // in a row's shift (0..29): its w' are kept negated

// The signed byte digits of |v| < 2^47 (six bytes, d_l = byte l as int8,
// v = sum_l 256^l d_l) and how many of them v needs: seven past the largest
// value of six, 0x7f7f7f7f7f7f (the least is -0x808080808080).
__device__ __forceinline__ uint64_t digits6(int64_t v) {
    return (uint64_t)(v + 0x808080808080LL) ^ 0x808080808080ULL;
}
__device__ __forceinline__ int digits6_needed(uint64_t d) {
    return (d >> 48) ? 7 : (d >> 40) ? 6 : (d >> 32) ? 5 : (d >> 24) ? 4 : (d >> 16) ? 3 : (d >> 8) ? 2 : 1;
}

// Per row, the digits its w' need (R the upload's shift[row]) raised into
// *need. sh_b - R <= 29, so |w'| < 2^47, but a weight of -128 under a scale of
// -65280 or more, beside a scale of the least exponent, passes six digits
// (they reach further down than up): such a row is kept negated, marked in
// shift[row], and only one that passes them either way needs the seventh.
__global__ __launch_bounds__(256) void fold_rows_kernel(const uint8_t* qs, const uint16_t* sc16, uint32_t rows,
                                                        uint32_t nb, int32_t* shift, int* need) {
    const uint32_t row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= rows) return;
    const uint32_t tile = row / Q8_TILE_ROWS, r = row % Q8_TILE_ROWS;
    const uint16_t* sc = sc16 + (size_t)tile * nb * Q8_TILE_ROWS + r;
    const int least = shift[row];
    int digits = 1, negated = 1;
    const uint8_t* q = qs + (size_t)tile * nb * Q8_TILE_BLOCK_BYTES + r * 16;
    for (uint32_t b = 0; b < nb; b++) {
        const uint32_t bits = sc[(size_t)b * Q8_TILE_ROWS], e = (bits >> 10) & 0x1f, mant = bits & 0x3ff;
        const int64_t m = (int64_t)(e ? 1024 + mant : mant);
        if (m == 0) continue;
        const int d = (e ? (int)e - 1 : 0) - least;  // 0..29
        // The largest |q| of the block (both signs: digits are asymmetric).
        int qmax = 0, qmin = 0;
        const uint8_t* qb = q + (size_t)b * Q8_TILE_BLOCK_BYTES;
        for (int h = 0; h < 2; h++)
            for (int j = 0; j < 16; j++) {
                const int v = (int8_t)qb[h * 256 + j];
                qmax = max(qmax, v);
                qmin = min(qmin, v);
            }
        const int64_t f = (bits & 0x8000) ? -(m << d) : (m << d);
        for (int64_t wv : {f * qmax, f * qmin}) {
            digits = max(digits, digits6_needed(digits6(wv)));
            negated = max(negated, digits6_needed(digits6(-wv)));
        }
    }
    if (digits > 6 && negated <= 6) {
        shift[row] = least | FOLD_NEGATED;
        digits = negated;
    }
    atomicMax(need, digits);
}

// One thread per (row, block): the block's w' as `nplanes` digit planes in
// the qs tile layout.
__global__ __launch_bounds__(256) void fold_planes_kernel(const uint8_t* qs, const uint16_t* sc16, uint32_t rows,
                                                          uint32_t nb, const int32_t* shift, uint32_t nplanes,
                                                          size_t plane_bytes, int8_t* planes) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)rows * nb) return;
    const uint32_t row = (uint32_t)(idx / nb), b = (uint32_t)(idx % nb);
    const uint32_t tile = row / Q8_TILE_ROWS, r = row % Q8_TILE_ROWS;
    const uint32_t bits = sc16[((size_t)tile * nb + b) * Q8_TILE_ROWS + r], e = (bits >> 10) & 0x1f,
                   mant = bits & 0x3ff;
    const int64_t m = (int64_t)(e ? 1024 + mant : mant);
    const int32_t sh = shift[row];
    const int d = m ? (e ? (int)e - 1 : 0) - (sh & ~FOLD_NEGATED) : 0;
    const int64_t f = !(bits & 0x8000) != !(sh & FOLD_NEGATED) ? -(m << d) : (m << d);
    const size_t off = ((size_t)tile * nb + b) * Q8_TILE_BLOCK_BYTES + r * 16;
    for (int h = 0; h < 2; h++) {
        const uint4 qv = *(const uint4*)(qs + off + h * 256);
        const uint32_t qw[4] = {qv.x, qv.y, qv.z, qv.w};
        uint32_t out[Q8_FOLD_MAX_PLANES][4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            uint64_t dg[4];
#pragma unroll
            for (int k = 0; k < 4; k++) dg[k] = digits6((int64_t)(int8_t)(qw[c] >> (8 * k)) * f);
#pragma unroll
            for (uint32_t p = 0; p < Q8_FOLD_MAX_PLANES; p++) out[p][c] = plane_byte4(dg[0], dg[1], dg[2], dg[3], p);
        }
        for (uint32_t p = 0; p < nplanes; p++)
            *(uint4*)(planes + p * plane_bytes + off + h * 256) = make_uint4(out[p][0], out[p][1], out[p][2], out[p][3]);
    }
}

// Workgroup shape of the folded product: W waves over 128 weight rows and
// 32 * TTWG tokens, each RI row tiles against one token tile; a stage is
// one 64-wide k step of WP weight planes and LG activation planes.
//
// Up to three weight planes: eight waves, two per SIMD, and 128 tokens (two
// passes of 64 where the tokens need four or five digits, whose
// shared-shift accumulators fit only one row tile per wave), or four waves
// and 64 tokens where 128 would leave CUs idle. Four to six planes: four
// waves, 64 rows and 64 tokens.
template <int WP, int LG, uint32_t W, uint32_t RT_>
struct FoldShape {
    static constexpr int RI = WP <= 3 && (W == 4 || LG <= 3) ? 2 : 1;
    static constexpr uint32_t WAVES = W, THREADS = 64 * W, RT = RT_;
    static constexpr uint32_t WR = RT / RI, TTWG = W / WR;
    static constexpr uint32_t CHUNKS = 2 * RT * WP + 2 * LG * TTWG;
    static constexpr uint32_t PER_WAVE = (CHUNKS + WAVES - 1) / WAVES;
    static constexpr uint32_t STAGE = PER_WAVE * WAVES * FRAG;
    static constexpr uint32_t STAGES = 3 * STAGE <= 160 * 1024 ? 3 : 2;
    static constexpr uint32_t PARK = W * RI * PARK_BLOCK * 4;  // the waves' finished blocks
    static constexpr uint32_t SMEM = STAGES * STAGE > PARK ? STAGES * STAGE : PARK;
    static constexpr int NS = WP + LG - 1;
};

template <class G, int WP, int LG>
__device__ __forceinline__ void fold_mainloop(const GemvArgs& a, int8_t* smem, uint32_t rt0, uint32_t tt0,
                                              v16i (&acc)[G::RI][G::NS]) {
    constexpr uint32_t TTWG = G::TTWG, RT = G::RT, CHUNKS = G::CHUNKS, PER_WAVE = G::PER_WAVE;
    constexpr uint32_t STAGES = G::STAGES, STAGE = G::STAGE;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wr = wave % G::WR, wt = wave / G::WR;
    const Q8View& w = a.w;
    const uint32_t KS = w.cols / 64, KB = w.cols / 32, TT = (a.tokens + 31) / 32;
    const size_t lstride = (size_t)TT * KB * FRAG;
    const size_t pstride = (size_t)w.tiles * w.nb * Q8_TILE_BLOCK_BYTES;
    // Wave w copies chunks w, w + W, ...: the first WCH are weight-plane
    // operands (advancing 1 KB of the tile layout per k step), the rest
    // digit-plane operands (2 KB).
    constexpr uint32_t WCH = 2 * RT * WP / G::WAVES;
    static_assert(WCH * G::WAVES == 2 * RT * WP, "whole chunks per wave");
    const int8_t* src[PER_WAVE];
    uint32_t off[WCH];
#pragma unroll
    for (uint32_t i = 0; i < PER_WAVE; i++) {
        const uint32_t c = min(wave + G::WAVES * i, CHUNKS - 1);
        if (i < WCH) {
            const uint32_t p = c / (2 * RT), cw = c % (2 * RT);
            src[i] = weight_operand(w, w.fold_planes + p * pstride, rt0 + cw / 2, cw & 1, lane, off[i]);
        } else {
            const uint32_t b = c - 2 * RT * WP, sub = b & 1, rest = b >> 1, l = rest / TTWG;
            const uint32_t tile = min(tt0 + rest % TTWG, TT - 1);
            src[i] = a.planes + l * lstride + ((size_t)tile * KB + sub) * FRAG;
        }
    }
    const uint32_t ring = __builtin_amdgcn_readfirstlane(lds_offset(smem));
    auto issue = [&](uint32_t ks) {
        const uint32_t base = ring + (ks % STAGES) * STAGE;
#pragma unroll
        for (uint32_t i = 0; i < PER_WAVE; i++)
            copy_to_lds16(src[i] + (size_t)ks * (i < WCH ? FRAG : 2 * FRAG), i < WCH ? off[i] : lane * 16,
                          base + (wave + G::WAVES * i) * FRAG);
    };
#pragma unroll
    for (uint32_t s = 0; s < STAGES - 1; s++)
        if (s < KS) issue(s);
    for (uint32_t ks = 0; ks < KS; ks++) {
        if (STAGES >= 3 && ks + 2 < KS) wait_vmem<(STAGES >= 3 ? 1 : 0) * PER_WAVE>();
        else wait_vmem<0>();
        lds_barrier();
        if (ks + STAGES - 1 < KS) issue(ks + STAGES - 1);
        const int8_t* st = smem + (ks % STAGES) * STAGE + lane * 16;
#pragma unroll
        for (uint32_t sub = 0; sub < 2; sub++) {
            v4i fw[G::RI][WP];
#pragma unroll
            for (int i = 0; i < G::RI; i++)
#pragma unroll
                for (int p = 0; p < WP; p++)
                    fw[i][p] = *(const v4i*)(st + (p * 2 * RT + 2 * (wr * G::RI + i) + sub) * FRAG);
#pragma unroll
            for (int l = 0; l < LG; l++) {
                const v4i fx = *(const v4i*)(st + (2 * RT * WP + 2 * (l * TTWG + wt) + sub) * FRAG);
#pragma unroll
                for (int i = 0; i < G::RI; i++)
#pragma unroll
                    for (int p = 0; p < WP; p++)
                        acc[i][p + l] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx, fw[i][p], acc[i][p + l], 0, 0, 0);
            }
        }
    }
    lds_barrier();
}

// The shared-shift sums recombine into sum_k w'_k x_k, shifted by the row's
// R and rounded once at 24 fraction bits. In double the sum is exact below
// 2^53 and the shift always, so the rounding to the nearest integer is the
// only one; a wave with a larger sum redoes its block in 128 bits. (A negated
// row's sign comes back with the scale.)
template <int NS>
__device__ __forceinline__ void fold_values(const Q8View& w, uint32_t row, const v16i (&acc)[NS], int32_t (&v)[16]) {
    const int32_t marked = row < w.rows ? w.fold_shift[row] : 0, shift = marked & ~FOLD_NEGATED;
    const bool negated = marked & FOLD_NEGATED;
    const double scale = __hiloint2double((negated ? 0x80000000u : 0) | (1023 + shift - 24) << 20, 0);  // +-2^(shift - 24)
    double most = 0;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        // Exact unless past 2^53, and then most says so.
        double tot = (double)acc[NS - 1][e];
#pragma unroll
        for (int s = NS - 2; s >= 0; s--) tot = fma(tot, 256.0, (double)acc[s][e]);
        most = fmax(most, fabs(tot));
        v[e] = round_double_to_i32(tot * scale);
    }
    if (__all(most < 0x1p52)) return;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        dn::i128 tot = 0;
#pragma unroll
        for (int s = 0; s < NS; s++) tot += (dn::i128)((dn::u128)(dn::i128)acc[s][e] << (8 * s));
        if (negated) tot = -tot;
        v[e] = dn::round_to_i32((dn::i128)((dn::u128)tot << shift), 24);
    }
}

template <int WP, int LG, uint32_t W, uint32_t RT>
__device__ __forceinline__ void fold_pass(const GemvArgs& a, int8_t* smem, uint32_t rt0, uint32_t tt0) {
    using G = FoldShape<WP, LG, W, RT>;
    v16i acc[G::RI][G::NS];
#pragma unroll
    for (int i = 0; i < G::RI; i++)
#pragma unroll
        for (int s = 0; s < G::NS; s++) acc[i][s] = v16i{};
    fold_mainloop<G, WP, LG>(a, smem, rt0, tt0, acc);
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t rt = rt0 + (wave % G::WR) * G::RI;
    finish_blocks<G::RI>(a, (int32_t*)smem + wave * G::RI * PARK_BLOCK, rt, tt0 + wave / G::WR,
                         [&](int i, int32_t (&v)[16]) __attribute__((always_inline)) {
                             fold_values<G::NS>(a.w, (rt + i) * 32 + lane % 32, acc[i], v);
                         });
}

// 32 * RT folded weight rows x 32 * TG tokens per workgroup.
template <int WP, uint32_t W, uint32_t RT, uint32_t TG>
__global__ __launch_bounds__(64 * W, 1) void q8_gemm_fold_kernel(const GemvArgs a) {
    static_assert(FoldShape<WP, 3, W, RT>::TTWG == TG && TG % FoldShape<WP, 5, W, RT>::TTWG == 0, "whole passes");
    constexpr uint32_t S3 = FoldShape<WP, 3, W, RT>::SMEM, S5 = FoldShape<WP, 5, W, RT>::SMEM;
    __shared__ __attribute__((aligned(1024))) int8_t smem[S5 > S3 ? S5 : S3];
    const uint32_t TT = (a.tokens + 31) / 32;
    uint32_t rg, tg;
    tile_of_block(blockIdx.x, (a.w.tiles + 2 * RT - 1) / (2 * RT), (TT + TG - 1) / TG, rg, tg);
    const uint32_t rt0 = rg * RT, tt0 = tg * TG;
    const int limbs = tiles_limbs<TG>(a, tt0);
    switch (limbs) {
        case 1: fold_pass<WP, 1, W, RT>(a, smem, rt0, tt0); break;
        case 2: fold_pass<WP, 2, W, RT>(a, smem, rt0, tt0); break;
        case 3: fold_pass<WP, 3, W, RT>(a, smem, rt0, tt0); break;
        case 4:
#pragma unroll 1
            for (uint32_t t = 0; t < TG; t += FoldShape<WP, 4, W, RT>::TTWG) {
                fold_pass<WP, 4, W, RT>(a, smem, rt0, tt0 + t);
                lds_barrier();  // the parked blocks are stored before the ring is refilled
            }
            break;
        default:
#pragma unroll 1
            for (uint32_t t = 0; t < TG; t += FoldShape<WP, 5, W, RT>::TTWG) {
                fold_pass<WP, 5, W, RT>(a, smem, rt0, tt0 + t);
                lds_barrier();
            }
            break;
    }
}

}  // namespace

// The shape of a launch (FoldShape) and its workgroups.
struct FoldLaunch {
    uint32_t rows, tokens, blocks;
};

static FoldLaunch fold_shape(const GemvArgs& a) {
    const uint32_t TT = (a.tokens + 31) / 32, cus = (uint32_t)iris_device_cus();
    if (a.w.fold_nplanes > 3) return {64, 64, (a.w.tiles + 3) / 4 * ((TT + 1) / 2)};
    const uint32_t rg = (a.w.tiles + 7) / 8, n4 = rg * ((TT + 3) / 4), n2 = rg * ((TT + 1) / 2);
    // A 128-token workgroup takes about 8/5 of a 64-token one's time. us per
    // product, preparation included, 128 / 64 tokens, rows x K:
    //   2048 tokens  28672 x 4096  1637 / 1923    4096 x 14336  841 / 959
    //    512 tokens  28672 x 4096   455 / 514     4096 x 14336  327 / 245
    //    128 tokens  28672 x 4096   141 / 158     512 tokens, 4096 x 4096  104 / 78
    const bool wide = a.w.fold_nplanes == 3 && 8 * ((n4 + cus - 1) / cus) <= 5 * ((n2 + cus - 1) / cus);
    return wide ? FoldLaunch{128, 128, n4} : FoldLaunch{128, 64, n2};
}

int iris_gemm_fold_launch(const GemvArgs& a, hipStream_t stream) {
    const FoldLaunch s = fold_shape(a);
    const dim3 grid(s.blocks);
    switch (a.w.fold_nplanes) {
        case 1: hipLaunchKernelGGL((q8_gemm_fold_kernel<1, 4, 4, 2>), grid, dim3(256), 0, stream, a); break;
        case 2: hipLaunchKernelGGL((q8_gemm_fold_kernel<2, 4, 4, 2>), grid, dim3(256), 0, stream, a); break;
        case 3:
            if (s.tokens == 128) hipLaunchKernelGGL((q8_gemm_fold_kernel<3, 8, 4, 4>), grid, dim3(512), 0, stream, a);
            else hipLaunchKernelGGL((q8_gemm_fold_kernel<3, 4, 4, 2>), grid, dim3(256), 0, stream, a);
            break;
        case 4: hipLaunchKernelGGL((q8_gemm_fold_kernel<4, 4, 2, 2>), grid, dim3(256), 0, stream, a); break;
        case 5: hipLaunchKernelGGL((q8_gemm_fold_kernel<5, 4, 2, 2>), grid, dim3(256), 0, stream, a); break;
        default: hipLaunchKernelGGL((q8_gemm_fold_kernel<6, 4, 2, 2>), grid, dim3(256), 0, stream, a); break;
    }
    return (int)hipGetLastError();
}

void iris_gemm_fold_route(const GemvArgs& a, char* name, size_t size) {
    const FoldLaunch s = fold_shape(a);
    std::snprintf(name, size, "folded %ux%u, %u planes", s.rows, s.tokens, a.w.fold_nplanes);
}

int iris_q8_prepare_fold(Q8GpuMatrix* m, hipStream_t stream) {
    static std::mutex lock;  // a matrix is folded once, whichever thread gets there first
    std::lock_guard<std::mutex> guard(lock);
    if (!m || m->fold_tried || m->scale_mode != Q8_SCALE_F16 || !m->sc16 || !m->fold.shift || m->cols % 64) return 0;
    m->fold_tried = true;
    const size_t plane_bytes = (size_t)m->tiles * m->nb * Q8_TILE_BLOCK_BYTES;
    int* d_need = nullptr;
    int need = 0;
    hipError_t st = hipMalloc((void**)&d_need, sizeof(int));
    if (st == hipSuccess) st = hipMemsetAsync(d_need, 0, sizeof(int), stream);
    if (st == hipSuccess) {
        hipLaunchKernelGGL(fold_rows_kernel, dim3((m->rows + 255) / 256), dim3(256), 0, stream, m->qs, m->sc16, m->rows,
                           m->nb, m->fold.shift, d_need);
        st = hipGetLastError();
    }
    if (st == hipSuccess) st = hipMemcpyAsync(&need, d_need, sizeof(int), hipMemcpyDeviceToHost, stream);
    if (st == hipSuccess) st = hipStreamSynchronize(stream);
    hipFree(d_need);
    if (st == hipSuccess && need >= 1 && need <= (int)Q8_FOLD_MAX_PLANES) {
        // Rows past the matrix in its last tile keep zero weights in every plane.
        st = hipMalloc((void**)&m->fold.planes, plane_bytes * need);
        if (st == hipSuccess) st = hipMemsetAsync(m->fold.planes, 0, plane_bytes * need, stream);
        const size_t n = (size_t)m->rows * m->nb;
        if (st == hipSuccess && n) {
            hipLaunchKernelGGL(fold_planes_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, m->qs,
                               m->sc16, m->rows, m->nb, m->fold.shift, (uint32_t)need, plane_bytes, m->fold.planes);
            st = hipGetLastError();
        }
        if (st == hipSuccess) st = hipStreamSynchronize(stream);
        if (st == hipSuccess) {
            m->fold.nplanes = (uint32_t)need;
            m->device_bytes += plane_bytes * need;
            return 0;
        }
    }
    hipFree(m->fold.planes);
    m->fold.planes = nullptr;
    return (int)st;
}

