// The tiled product of row-scale matrices (q8_gemm.hip has the arithmetic,
// the operand layout and the launch rule).
#include <cstdio>

#include "q8_gemm_row.h"
#include "q8_gemm_tile.h"

namespace {

constexpr uint32_t GM_TT = 4;               // 32-token tiles per workgroup (128 tokens)

// The two workgroup shapes: W waves over 32 * W rows and 128 tokens (W = 8: two waves per SIMD, 256 rows, for launches that fill
// the chip; W = 4: one wave per SIMD, 128 rows, for smaller ones). A stage
// is one 64-wide k step: 2W weight operands and up to 24 digit-plane ones.
//
// SPLIT = 2 (four-wave shape only): the workgroup holds two such groups of
// W waves (two waves per SIMD), each walking half of the k steps through a
// two-stage ring of its own; the second group's int32 plane sums are then
// added into the first's (exact: the whole row's sum fits int32), and both
// groups store the block.
template <uint32_t W, uint32_t SPLIT = 1>
struct GemmShape {
    static constexpr uint32_t WAVES = W, RT = W;                     // per k group; RT: 32-row tiles
    static constexpr uint32_t SPLITS = SPLIT, THREADS = 64 * W * SPLIT;
    static constexpr uint32_t STAGE = (2 * W + 24) * FRAG;
    static constexpr uint32_t STAGES = SPLIT == 2 ? 2 : W == 8 ? 3 : 4;
    static constexpr uint32_t RING = STAGES * STAGE;                  // per k group
    static constexpr uint32_t PARK = THREADS / 64 * (SPLIT == 2 ? 2 : 4) * PARK_BLOCK * 4;  // the waves' finished blocks
    static constexpr uint32_t SMEM = SPLIT * RING > PARK ? SPLIT * RING : PARK;
};

// One pass of the workgroup over the whole k range: RT weight tiles of 32
// rows (from 32-row tile rt0) times TTWG token tiles of 32 (from tt0) times
// LG digit planes. Wave (wr, wt) accumulates weight tiles wr*RI.. against
// token tile wt: acc[i][l] is the int32 sum of plane l for its 32 x 32
// block. The loop is held by the LDS as much as by the matrix cores (an
// operand read is 8 cycles of the CU's LDS, a matrix instruction 32 of one
// of its four SIMDs), so a wave takes four weight tiles against one token
// tile where it can: 7 operand reads per 12 instructions at three planes,
// where two tiles against two took 8. A stage holds, for its two 32-wide k blocks s, the
// weight operand of tile r at chunk 2r + s and the plane-l operand of token
// tile j at 2RT + 2(l * TTWG + j) + s (padded to a whole number of chunks
// per wave with copies of the last). Operands past the last tile are clamped
// onto it (read, never stored).
template <class G, int LG, int RI, bool DEEP = false>
__device__ __forceinline__ void gemm_mainloop(const GemvArgs& a, int8_t* smem, uint32_t rt0, uint32_t tt0,
                                              v16i (&acc)[RI][LG]) {
    constexpr uint32_t WR = G::RT / RI, TTWG = G::WAVES / WR;  // token tiles per pass, one per wave
    constexpr uint32_t CHUNKS = 2 * G::RT + 2 * LG * TTWG;  // 1 KB operands per stage
    constexpr uint32_t PER_WAVE = (CHUNKS + G::WAVES - 1) / G::WAVES;
    static_assert(PER_WAVE * G::WAVES * FRAG <= G::STAGE && PER_WAVE >= 2, "stage layout");
    // The ring's stages are as large as this pass's operands, so fewer
    // digit planes leave room for more stages in the same LDS: four where
    // four fit, else the shape's own count; with DEEP (long rows), as many
    // as fit up to four. At three planes and 64 tokens the split four-wave
    // shape then runs three stages instead of two: faster over the 112 k
    // steps of a K=14336 down product (the 512-row prompt pass 20.1-20.2 ->
    // 19.6-19.75 ms), slower over K=4096 (the M=512 product 48.4 -> 49.6 us).
    constexpr uint32_t GM_RT = G::RT, GM_STAGE = PER_WAVE * G::WAVES * FRAG;
    constexpr uint32_t FIT = G::RING / GM_STAGE;
    constexpr uint32_t GM_STAGES = FIT >= 4 ? 4 : DEEP && FIT > G::STAGES ? FIT : G::STAGES;
    static_assert(GM_STAGES * GM_STAGE <= G::RING, "ring layout");
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    // The wave within its k group, the group's ring and k steps [ks0, ks1).
    // Through readfirstlane: uniform, so the k loop's control and the copies'
    // addresses stay in scalar registers.
    const uint32_t id = __builtin_amdgcn_readfirstlane(tid >> 6), half = id / G::WAVES, wave = id % G::WAVES;
    const uint32_t wr = wave % WR, wt = wave / WR;
    const Q8View& w = a.w;
    const uint32_t KS = w.cols / 64, KB = w.cols / 32, TT = (a.tokens + 31) / 32;
    const uint32_t ks0 = half * (KS / G::SPLITS), ks1 = ks0 + KS / G::SPLITS;
    smem += half * G::RING;
    const size_t lstride = (size_t)TT * KB * FRAG;

    // Wave w copies chunks w, w + W, ...: the first two are weight operands
    // (advancing 1 KB of the tile layout per k step), the rest plane
    // operands (advancing 2 KB).
    const int8_t* src[PER_WAVE];
    uint32_t off[2];
#pragma unroll
    for (uint32_t i = 0; i < PER_WAVE; i++) {
        const uint32_t c = min(wave + G::WAVES * i, CHUNKS - 1);
        if (i < 2) {
            src[i] = weight_operand(w, (const int8_t*)w.qs, rt0 + c / 2, c & 1, lane, off[i]);
        } else {
            const uint32_t b = c - 2 * GM_RT, sub = b & 1, rest = b >> 1, l = rest / TTWG;
            const uint32_t tile = min(tt0 + rest % TTWG, TT - 1);
            src[i] = a.planes + l * lstride + ((size_t)tile * KB + sub) * FRAG;
        }
    }
    const uint32_t ring = __builtin_amdgcn_readfirstlane(lds_offset(smem));
    auto issue = [&](uint32_t ks) {
        const uint32_t base = ring + (ks % GM_STAGES) * GM_STAGE;
#pragma unroll
        for (uint32_t i = 0; i < PER_WAVE; i++)
            copy_to_lds16(src[i] + (size_t)ks * (i < 2 ? FRAG : 2 * FRAG), i < 2 ? off[i] : lane * 16,
                          base + (wave + G::WAVES * i) * FRAG);
    };

#pragma unroll
    for (uint32_t s = 0; s < GM_STAGES - 1; s++)
        if (ks0 + s < ks1) issue(ks0 + s);
    // Both k groups take the same number of steps (the launcher's even KS),
    // so their barriers pair up.
    for (uint32_t ks = ks0; ks < ks1; ks++) {
        // This wave's copies for step ks are in LDS once at most the later
        // steps' copies are outstanding; the barrier makes every wave's
        // visible and frees the slot the next copy overwrites (read at ks-1).
        if (GM_STAGES == 2) wait_vmem<0>();
        else if (GM_STAGES >= 4 && ks + 2 < ks1) wait_vmem<(GM_STAGES >= 4 ? 2 : 1) * PER_WAVE>();
        else if (ks + 1 < ks1) wait_vmem<PER_WAVE>();
        else wait_vmem<0>();
        lds_barrier();
        if (ks + GM_STAGES - 1 < ks1) issue(ks + GM_STAGES - 1);
        const int8_t* st = smem + (ks % GM_STAGES) * GM_STAGE + lane * 16;
#pragma unroll
        for (uint32_t sub = 0; sub < 2; sub++) {
            v4i fw[RI];
#pragma unroll
            for (int i = 0; i < RI; i++) fw[i] = *(const v4i*)(st + (2 * (wr * RI + i) + sub) * FRAG);
#pragma unroll
            for (int l = 0; l < LG; l++) {
                const v4i fx = *(const v4i*)(st + (2 * GM_RT + 2 * (l * TTWG + wt) + sub) * FRAG);
#pragma unroll
                for (int i = 0; i < RI; i++)
                    acc[i][l] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx, fw[i], acc[i][l], 0, 0, 0);
            }
        }
    }
    lds_barrier();  // every wave is done with the ring before it is reused
}

// round_to_i32(tot * sc, 24) in 64-bit pieces (q8.rs:94-104).
__device__ __forceinline__ int32_t round_wide(int64_t tot, int64_t sc) {
    const uint64_t lo = (uint64_t)tot * (uint64_t)sc;
    const int64_t hi = __mul64hi(tot, sc), top = hi >> 24;
    const int64_t fl = (int64_t)(((uint64_t)hi << 40) | (lo >> 24));
    if (top != (fl >> 63) || fl >= INT32_MAX || fl < INT32_MIN) 
        return hi < 0 ? INT32_MIN : INT32_MAX;
    return (int32_t)fl + (int32_t)((uint32_t)(lo & 0xffffff) + (uint32_t)(fl & 1) > 0x800000u);
}

// The planes recombine into the row's integer dot product, then
// round_to_i32(tot * scale, 24). In double: a scale of at most 11
// significant bits (every f16's) times |tot| < 2^42 is exact, so the
// rounding to the nearest integer is the only one; about 12 instructions an
// output where 64-bit products with a bit-length test took 55 (14 of a
// workgroup's 123 us at 2048 x 4096 x 4096). A wave with a larger value
// redoes its block in 128 bits.
template <int LG>
__device__ __forceinline__ void row_values(const Q8View& w, uint32_t row, const v16i (&acc)[LG], int32_t (&v)[16]) {
    const int64_t sc = row < w.rows ? w.row_scale[row] : 0;
    const uint64_t as = sc < 0 ? 0 - (uint64_t)sc : (uint64_t)sc;
    const bool narrow = as == 0 || (as >> __builtin_ctzll(as)) < 2048;
    const double scale = (double)sc * 0x1p-24;
    double most = 0;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        // Exact unless past 2^53, and then most says so.
        double tot = (double)acc[LG - 1][e];
#pragma unroll
        for (int l = LG - 2; l >= 0; l--) tot = fma(tot, 256.0, (double)acc[l][e]);
        most = fmax(most, fabs(tot));
        v[e] = round_double_to_i32(tot * scale);
    }
    if (__all(narrow && most < 0x1p42)) return;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        int64_t tot = 0;  // |tot| < K * 2^38
#pragma unroll
        for (int l = 0; l < LG; l++) tot += (int64_t)acc[l][e] * ((int64_t)1 << (8 * l));
        v[e] = round_wide(tot, sc);
    }
}

template <class G, int LG, int RI, bool DEEP>
__device__ __forceinline__ void gemm_pass(const GemvArgs& a, int8_t* smem, uint32_t rt0, uint32_t tt0) {
    constexpr uint32_t WR = G::RT / RI;
    constexpr int NI = RI / G::SPLITS;  // row tiles a wave finishes
    v16i acc[RI][LG];
#pragma unroll
    for (int i = 0; i < RI; i++)
#pragma unroll
        for (int l = 0; l < LG; l++) acc[i][l] = v16i{};
    gemm_mainloop<G, LG, RI, DEEP>(a, smem, rt0, tt0, acc);
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), hw = wave % G::WAVES;
    uint32_t first = 0;
    if constexpr (G::SPLITS == 2) {
        // The k groups' sums meet through LDS, lane-contiguous: the first
        // group finishes the first half of each wave's row tiles, the
        // second the other half.
        constexpr int LS = LG < 3 ? LG : 3;  // planes at a time
        static_assert(2 * G::WAVES * LS * 4096 <= G::SMEM, "exchange fits the LDS");
        const bool second = wave >= G::WAVES;
        int32_t* mine = (int32_t*)smem + (size_t)wave * LS * 1024 + lane;
        const int32_t* theirs = (const int32_t*)smem + (size_t)(wave ^ G::WAVES) * LS * 1024 + lane;
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
            for (int l0 = 0; l0 < LG; l0 += LS) {
#pragma unroll
                for (int l = l0; l < l0 + LS && l < LG; l++)
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        mine[((l - l0) * 16 + e) * 64] = second ? acc[i][l][e] : acc[NI + i][l][e];
                        if (second) acc[i][l][e] = acc[NI + i][l][e];
                    }
                lds_barrier();
#pragma unroll
                for (int l = l0; l < l0 + LS && l < LG; l++)
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[i][l][e] += theirs[((l - l0) * 16 + e) * 64];
                lds_barrier();
            }
        first = second ? NI : 0;
    }
    const uint32_t rt = rt0 + (hw % WR) * RI + first;
    finish_blocks<NI>(a, (int32_t*)smem + wave * NI * PARK_BLOCK, rt, tt0 + hw / WR,
                      [&](int i, int32_t (&v)[16]) __attribute__((always_inline)) {
                          row_values<LG>(a.w, (rt + i) * 32 + lane % 32, acc[i], v);
                      });
}

// 32W weight rows x 32 * TG tokens per workgroup. Up to three digit planes (the
// usual case) are accumulated side by side in one pass; a block whose
// tokens need four or five takes passes of 64 tokens.
template <uint32_t W, uint32_t TG, uint32_t SPLIT = 1, bool DEEP = false>
__global__ __launch_bounds__(64 * W * SPLIT, 1) void q8_gemm_row_kernel(const GemvArgs a) {
    static_assert(TG == 2 || TG == 4, "64 or 128 tokens per workgroup");
    using G = GemmShape<W, SPLIT>;
    __shared__ __attribute__((aligned(1024))) int8_t smem[G::SMEM];
    const uint32_t TT = (a.tokens + 31) / 32;
    uint32_t rg, tg;
    tile_of_block(blockIdx.x, (a.w.tiles + 2 * G::RT - 1) / (2 * G::RT), (TT + TG - 1) / TG, rg, tg);
    const uint32_t rt0 = rg * G::RT, tt0 = tg * TG;

    const int limbs = tiles_limbs<TG>(a, tt0);
    constexpr int RI = TG;  // W waves, one token tile each: W * RI / TG row tiles
    switch (limbs) {
        case 1: gemm_pass<G, 1, RI, DEEP>(a, smem, rt0, tt0); break;
        case 2: gemm_pass<G, 2, RI, DEEP>(a, smem, rt0, tt0); break;
        case 3: gemm_pass<G, 3, RI, DEEP>(a, smem, rt0, tt0); break;
        case 4:
#pragma unroll 1
            for (uint32_t t = 0; t < TG; t += 2) {
                gemm_pass<G, 4, 2, DEEP>(a, smem, rt0, tt0 + t);
                lds_barrier();  // the parked blocks are stored before the ring is refilled
            }
            break;
        default:
#pragma unroll 1
            for (uint32_t t = 0; t < TG; t += 2) {
                gemm_pass<G, 5, 2, DEEP>(a, smem, rt0, tt0 + t);
                lds_barrier();
            }
            break;
    }
}

}  // namespace

// The shape of a launch: `waves` per k group over 32 * waves rows, `tokens`
// tokens, the k steps split between two groups, deep rings, and its workgroups.
struct RowShape {
    uint32_t waves, tokens;
    bool split, deep;
    uint32_t blocks;
};

static RowShape row_shape(const GemvArgs& a) {
    const uint32_t TT = (a.tokens + 31) / 32;
    // The shape whose rounds of workgroups cost least: 256 rows x 128 tokens
    // with two waves per SIMD, or 128 x 128 or 128 x 64 with the k steps
    // split between two wave groups. A round of them takes about 11 : 7 : 4
    // (82, 53 and 30 us at K = 4096 in a full chip). us per product,
    // preparation included, 256 x 128 / 128 x 128 / 128 x 64, rows x K:
    //   2048 tokens  28672 x 4096   639 / 736 / 822    6144 x 4096   178 / 175 / 194
    //   1024 tokens  4096 x 14336   260 / 184 / 214    6144 x 4096    96 / 110 / 104
    //    512 tokens  28672 x 4096   182 / 212 / 215    4096 x 14336  233 / 142 / 106
    //    256 tokens  28672 x 4096    95 / 110 / 123    6144 x 4096    78 /  54 /  37
    //    777 tokens  20000 x 4096   248 / 254 / 245
    const uint32_t n_tg = (TT + GM_TT - 1) / GM_TT, n_tg2 = (TT + 1) / 2;
    const uint32_t cus = (uint32_t)iris_device_cus();
    const uint32_t n8 = (a.w.tiles + 15) / 16 * n_tg, n4 = (a.w.tiles + 7) / 8 * n_tg;
    const uint32_t n42 = (a.w.tiles + 7) / 8 * n_tg2;
    const uint32_t cost8 = 11 * ((n8 + cus - 1) / cus), cost4 = 7 * ((n4 + cus - 1) / cus);
    const uint32_t cost2 = 4 * ((n42 + cus - 1) / cus);
    // The k steps are split only when there is an even number of them (both
    // groups' barriers pair up); else the 128-row shapes have one wave per
    // SIMD and serve launches that leave CUs without a 256-row workgroup.
    const bool split = (a.w.cols / 64) % 2 == 0;
    // Deeper rings for long rows (at least 64 k steps per wave group).
    const bool deep = a.w.cols >= 8192;
    if (split ? cost8 <= (cost4 < cost2 ? cost4 : cost2) : n8 >= cus) return {8, 128, false, false, n8};
    if (n42 != n4 && cost2 <= cost4) return {4, 64, split, split && deep, n42};
    return {4, 128, split, split && deep, n4};
}

int iris_gemm_row_launch(const GemvArgs& a, hipStream_t stream) {
    const RowShape s = row_shape(a);
    const dim3 grid(s.blocks);
    if (s.waves == 8)
        hipLaunchKernelGGL((q8_gemm_row_kernel<8, 4>), grid, dim3(512), 0, stream, a);
    else if (s.tokens == 64) {
        if (s.deep) hipLaunchKernelGGL((q8_gemm_row_kernel<4, 2, 2, true>), grid, dim3(512), 0, stream, a);
        else if (s.split) hipLaunchKernelGGL((q8_gemm_row_kernel<4, 2, 2>), grid, dim3(512), 0, stream, a);
        else hipLaunchKernelGGL((q8_gemm_row_kernel<4, 2>), grid, dim3(256), 0, stream, a);
    } else {
        if (s.deep) hipLaunchKernelGGL((q8_gemm_row_kernel<4, 4, 2, true>), grid, dim3(512), 0, stream, a);
        else if (s.split) hipLaunchKernelGGL((q8_gemm_row_kernel<4, 4, 2>), grid, dim3(512), 0, stream, a);
        else hipLaunchKernelGGL((q8_gemm_row_kernel<4, 4>), grid, dim3(256), 0, stream, a);
    }
    return (int)hipGetLastError();
}

void iris_gemm_row_route(const GemvArgs& a, char* name, size_t size) {
    const RowShape s = row_shape(a);
    std::snprintf(name, size, "tiled %ux%u%s%s", 32 * s.waves, s.tokens, s.split ? " split" : "", s.deep ? " deep" : "");
}
