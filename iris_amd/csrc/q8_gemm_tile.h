// What the tiled multi-token products share (q8_gemm_row.hip,
// q8_gemm_fold.hip): operand copies into LDS, the launch order and the end
// of a wave's output blocks.
//
// The activations are the matrix instruction's A operand and the weights its
// B operand, so output e of lane l of a 32 x 32 block is weight row l % 32,
// token 8 * (e / 4) + 4 * (l / 32) + e % 4: a plain or residual store is
// whole 128-byte runs of a token's row straight from the registers, and a
// lane needs one row scale per block. (With the roles the other way round
// every output went through an LDS block shared by the workgroup, between
// two of its barriers: at 2048 x 4096 x 28672, 34 of a workgroup's 123 us
// came after its matrix work.)
#pragma once

#include "detnum_dev.h"
#include "q8_epilogue.h"
#include "q8_gemm_common.h"
#include "q8_internal.h"

constexpr uint32_t GM_BAND = 8;             // row groups per band of the launch order

template <int N>
__device__ __forceinline__ void wait_vmem() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// 16 bytes per lane from base + off (base the same in every lane: one scalar
// pair per operand, where a 64-bit address per lane and operand held the
// widest shapes at their register limit) into LDS at byte offset lds (the
// wave's base, the same in every lane; lane i writes lds + 16i):
// global_load_lds_dwordx4.
// Written out here because the compiler, lacking alias information, treats
// every copy still in flight as a write to any LDS address a later ds_read
// touches, and in some shapes waited for all of them (vmcnt(0)) before each
// k step's reads, so the next step's copies, issued just before, no longer
// overlapped the step's matrix work. The k loops' own waits (wait_vmem, then
// the barrier) order each copy before the reads of its stage, and the
// compiler's waits for its own loads stay correct: the copies only make its
// vmcnt counts more conservative.
__device__ __forceinline__ void copy_to_lds16(const int8_t* base, uint32_t off, uint32_t lds) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "{m0}"(lds) : "memory");
}

// Where a wave's copies of weight operand (32-row tile rt, first or second
// 32-wide block sub of a k step) start, and each lane's offset from there:
// lane l takes 16 bytes of row l % 32. Tiles past the last are clamped onto
// it (read, never stored).
__device__ __forceinline__ const int8_t* weight_operand(const Q8View& w, const int8_t* qs, uint32_t rt, uint32_t sub,
                                                        uint32_t lane, uint32_t& off) {
    const uint32_t first = min(2 * rt, w.tiles - 1), r = lane % 32, tile = min(2 * rt + r / 16, w.tiles - 1);
    off = (tile - first) * w.nb * Q8_TILE_BLOCK_BYTES + (lane / 32) * 256 + (r % 16) * 16;
    return qs + ((size_t)first * w.nb + sub) * Q8_TILE_BLOCK_BYTES;
}

// The LDS byte offset of a pointer into LDS: a flat address of LDS is the
// aperture above the offset, so its low 32 bits.
__device__ __forceinline__ uint32_t lds_offset(const void* p) { return (uint32_t)(uintptr_t)p; }

// Workgroups are ordered so that each XCD (blocks are dealt to the 8 XCDs in
// turn) takes a contiguous range, walked in bands of 8 row groups with the
// token groups inside a band, so blocks in flight together share operands in
// their XCD's L2. Block b of an n_rg x n_tg grid: row group, token group.
__device__ __forceinline__ void tile_of_block(uint32_t b, uint32_t n_rg, uint32_t n_tg, uint32_t& rg, uint32_t& tg) {
    const uint32_t total = n_rg * n_tg;
    if (total % 8 == 0) b = (b % 8) * (total / 8) + b / 8;
    const uint32_t band = b / (GM_BAND * n_tg), first = band * GM_BAND, rows_in_band = min(GM_BAND, n_rg - first);
    const uint32_t r = b - band * GM_BAND * n_tg;
    rg = first + r % rows_in_band;
    tg = r / rows_in_band;
}

// n <= N ints to dst, 16 bytes at a time where all N are stored and aligned.
template <int N>
__device__ __forceinline__ void store_run(int32_t* dst, const int32_t (&v)[N], uint32_t n) {
    if (n >= N && !((uintptr_t)dst & 15)) {
#pragma unroll
        for (int i = 0; i < N; i += 4) *(int4*)(dst + i) = make_int4(v[i], v[i + 1], v[i + 2], v[i + 3]);
    } else {
#pragma unroll
        for (int i = 0; i < N; i++)
            if (i < (int)n) dst[i] = v[i];
    }
}

// A wave parks a block it cannot store from registers in LDS of its own, as
// 32 lines (one token each, 32 rows and 4 ints of padding: the 16-byte reads
// below then fall on distinct banks), then each lane takes 16 consecutive
// rows (8 pairs) of one token.
constexpr uint32_t PARK_LINE = 36, PARK_BLOCK = 32 * PARK_LINE;  // ints

__device__ __forceinline__ void finish_parked(const GemvArgs& a, int32_t* block, uint32_t rt, uint32_t tt) {
    const Q8View& w = a.w;
    const uint32_t lane = threadIdx.x & 63, t = lane % 32, h = lane / 32;
    const uint32_t row0 = rt * 32 + 16 * h, token = tt * 32 + t;
    int32_t* p = block + (2 * (4 * (t / 8) + t % 4) + (t / 4) % 2) * PARK_LINE + 16 * h;  // this lane's own 16 rows
    const bool valid = token < a.tokens && row0 < w.rows;
    const uint32_t n = row0 < w.rows ? min(16u, w.rows - row0) : 0;
    if (a.epilogue == EPI_SWIGLU || a.epilogue == EPI_GEGLU) {
        // Gate and up rows alternate.
        int32_t o[8];
        if (a.epilogue == EPI_SWIGLU && a.silu_tab) {
            int32_t gate[8], up[8], act[8];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int4 v = *(const int4*)(p + 4 * q);
                gate[2 * q] = v.x, up[2 * q] = v.y, gate[2 * q + 1] = v.z, up[2 * q + 1] = v.w;
            }
            uint32_t slow = 0;
#pragma unroll
            for (int q = 0; q < 8; q++) slow |= (uint32_t)!dn::silu_fast(gate[q], act[q]) << q;
            if (slow) {
#pragma unroll
                for (int q = 0; q < 8; q++)
                    if ((slow >> q) & 1) act[q] = dn::silu_from_tab(gate[q], a.silu_tab[dn::silu_tab_index(gate[q])]);
            }
#pragma unroll
            for (int q = 0; q < 8; q++) o[q] = dn::mul_sat(act[q], up[q]);
        } else {
#pragma unroll 1
            for (int q = 0; q < 8; q++) {  // in place: pair q is read before slot q is written
                const int32_t gate = p[2 * q], up = p[2 * q + 1];
                p[q] = dn::mul_sat(a.epilogue == EPI_SWIGLU ? dn::silu(gate) : dn::gelu(gate), up);
            }
#pragma unroll
            for (int q = 0; q < 8; q++) o[q] = p[q];
        }
        if (a.out && valid) store_run<8>(a.out + (size_t)token * a.out_stride + row0 / 2, o, (n + 1) / 2);
        if (!a.out_gemm_planes) return;
        // The gated values as the next product's digit planes: 8 of the 16
        // bytes of one operand lane per plane, as digit_planes_kernel writes
        // them (zero digits past the last token), and the digits the (k
        // chunk, 32-token tile) needs by atomicMax (the largest in any
        // order; a 32-row tile's 16 pairs lie in one k chunk).
        const uint32_t K = w.rows / 2, pair0 = row0 / 2, TT = (a.tokens + 31) / 32;
        if (rt * 16 >= K || tt >= TT) return;
        uint64_t d[8];
        int need = 1;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            d[q] = digits5(valid ? o[q] : 0);
            need = max(need, limbs_needed(d[q]));
        }
        if (pair0 < K) {
            int8_t* dst = a.out_gemm_planes + ((size_t)tt * (K / 32) + pair0 / 32) * FRAG +
                          (t + 32 * ((pair0 % 32) / 16)) * 16 + pair0 % 16;
#pragma unroll
            for (int l = 0; l < PL_MAX; l++)
                *(uint2*)(dst + l * ((size_t)TT * K * 32)) = make_uint2(plane_byte4(d[0], d[1], d[2], d[3], l),
                                                                        plane_byte4(d[4], d[5], d[6], d[7], l));
        }
        for (int off = 32; off >= 1; off >>= 1) need = max(need, __shfl_xor(need, off));
        if (lane == 0) atomicMax(&a.out_gemm_limbs[a.tokens + rt * 16 / (32 * PLANE_KB) * TT + tt], need);
        return;
    }
    if (!valid) return;
    if (a.epilogue == EPI_ROPE_KV && n == 16 && a.q_rows % 16 == 0 && a.kv_rows % 16 == 0) {
        const uint32_t pos = (uint32_t)*a.d_pos + token;
        int32_t v[16];
        if (row0 < a.q_rows + a.kv_rows && pos != 0) {
            if (a.rope_sc) {
                const int64_t* sc = a.rope_sc + (size_t)token * a.head_dim;
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const uint32_t j = ((row0 + 2 * q) % a.head_dim) / 2;
                    v[2 * q] = p[2 * q], v[2 * q + 1] = p[2 * q + 1];
                    dn::rotate_pair_sc(v[2 * q], v[2 * q + 1], sc[2 * j], sc[2 * j + 1]);
                }
            } else {
#pragma unroll 1
                for (int q = 0; q < 8; q++)
                    dn::rotate_pair_q30(p[2 * q], p[2 * q + 1],
                                        (int64_t)pos * a.inv_freq[((row0 + 2 * q) % a.head_dim) / 2]);
#pragma unroll
                for (int r = 0; r < 16; r++) v[r] = p[r];
            }
        } else {
#pragma unroll
            for (int r = 0; r < 16; r++) v[r] = p[r];
        }
        if (row0 < a.q_rows) {
            store_run<16>(a.out + (size_t)token * a.out_stride + row0, v, 16);
        } else if (row0 < a.q_rows + a.kv_rows) {
            // Lanes are consecutive positions: whole lines of the
            // transposed K cache.
            int32_t* kc = a.k_cache + (size_t)(row0 - a.q_rows) * a.k_pos_stride + pos;
#pragma unroll
            for (int r = 0; r < 16; r++) kc[(size_t)r * a.k_pos_stride] = v[r];
        } else {
            store_run<16>(a.v_cache + (size_t)pos * a.kv_rows + (row0 - a.q_rows - a.kv_rows), v, 16);
        }
        return;
    }
#pragma unroll 1
    for (uint32_t r = 0; r < n; r++) store_output(a, row0 + r, token, p[r], p[r ^ 1]);
}

// A wave's NI finished blocks (32-row tiles rt.., 32-token tile tt), block i
// from values(i, v): from registers for a plain or residual store, else
// through `park` (NI * PARK_BLOCK ints of the wave's own).
template <int NI, class Values>
__device__ __forceinline__ void finish_blocks(const GemvArgs& a, int32_t* park, uint32_t rt, uint32_t tt, Values&& values) {
    const uint32_t lane = threadIdx.x & 63;
    const bool residual = a.epilogue == EPI_RESIDUAL, direct = residual || a.epilogue == EPI_STORE;
#pragma unroll
    for (int i = 0; i < NI; i++) {
        int32_t v[16];
        values(i, v);
        if (direct) {
            const uint32_t row = (rt + i) * 32 + lane % 32, tok0 = tt * 32 + 4 * (lane / 32);
            if (row < a.w.rows) {
                if (residual) {
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        const uint32_t token = min(tok0 + 8 * (e / 4) + e % 4, a.tokens - 1);
                        v[e] = dn::add_sat(v[e], a.residual[(size_t)token * a.residual_stride + row]);
                    }
                }
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const uint32_t token = tok0 + 8 * (e / 4) + e % 4;
                    if (token < a.tokens) a.out[(size_t)token * a.out_stride + row] = v[e];
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < 16; e++) park[i * PARK_BLOCK + (2 * e + lane / 32) * PARK_LINE + lane % 32] = v[e];
        }
    }
    if (direct) return;
    // The wave's own LDS: its accesses stay in order, the compiler keeps them so.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll 1
    for (uint32_t b = 0; b < NI; b++) finish_parked(a, park + b * PARK_BLOCK, rt + b, tt);
}

// The nearest integer to an exact double, ties to even, saturated.
__device__ __forceinline__ int32_t round_double_to_i32(double x) {
    return (int32_t)fmin(fmax(rint(x), -2147483648.0), 2147483647.0);
}
