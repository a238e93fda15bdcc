// mmq_pf.hip — prompt GEMM, third generation: quantized weights x F16 activations on the F16 matrix cores, every byte by LDS-DMA.
//
// Replaces ggml_compute_forward_mul_mat (ggml/src/ggml.c:12377) for prompt-sized batches (what the reference's CUDA plug-in serves with
// dequantize + cuBLAS / mul_mat_q, ggml-cuda.cu:1187-1285, mmq.cuh:2583):   Y[t][n] = sum_k W[n][k] X[t][k].
// Several matrices that share the activations (wq | wk | wv, ffn_gate | ffn_up) are JOBS of one launch, each with its own quant type.
//
// What the second generation (mmq.hip gemm_q_f16_kernel2) lost, by its own counters (profiles/r05_prefill_pmc.txt: MfmaUtil 48 %, waves in
// s_waitcnt): every thread fetched 16-byte weight pieces of its OWN row straight into registers - 512 cache lines touched per instruction
// round, 16 of 128 bytes used, the lines re-requested from L2 by the next three k-steps - and the compiler parked `s_waitcnt vmcnt(0)` in the
// middle of the MFMA stream; the dequantized F16 tile then went through ds_write + barrier + ds_read. Here:
//   * a wave owns 32 weight rows x ALL tokens of the tile (8 waves = 256 rows x 256 tokens; accumulators 8 x 16 = 128 registers). Its
//     weights never meet another wave: the packed bytes travel HBM -> LDS by LDS-DMA into a wave-private area (128 k per piece, two slots),
//     are read back 8 bytes per lane already in MFMA A-operand order (lane = row, k-half) and dequantized IN REGISTERS - packed-F16 math:
//     v_perm_b32 makes the halfs 1024 + q (low nibbles) / 64 + q (high nibbles, no shift), one packed add and one packed fma apply
//     d * sc and dmin * m. No F16 weight tile in LDS, no ds_write, no barrier on the weight path (the wave's own vmcnt orders it).
//   * the F16 activation tile (256 tokens x 64 k = 32 KiB per k-step) travels by LDS-DMA as whole 128-byte lines into a ring of three
//     buffers; the 16-byte chunks of a token row are XOR-swizzled on the SOURCE side (chunk c of token t lands at c ^ ((t >> 1) & 7)) so the
//     sixteen lanes ds_read_b128 serves together hit sixteen different bank groups. One barrier per k-step; step s + 2 is requested at
//     the top of step s, and the first fragments of step s + 1 are read before that barrier, so the matrix pipe never drains at it.
//   * no VGPR-destination global load in the k loop (Q6_K's 2-byte d excepted: once per 256 k): the compiler has nothing to wait for in
//     the MFMA stream; the only vmcnt wait is the explicit one in front of the barrier.
// Numerics: dequantized weight = F16(q * F16(d * sc) - F16(dmin * m)) with ONE rounding in the fma (kernel2 rounded the product first),
// F16 activations, f32 accumulation in k order - the reference's own GPU large-batch numerics (NMSE <= 5e-4, tests/test-backend-ops.cpp:1660;
// measured ~1e-6).
#include "pm355_device.h"
#include "pm355_kernels.h"
#include <stdlib.h>
#include <stdio.h>
#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void * lds_ptr;

constexpr int PF_NTHR = 512, MID_NTHR = 768, PF_MAX_JOBS = 4;

struct PfJob {
    const uint8_t * W; float * Y; _Float16 * Yh; const float * bias; const float * resid; const float * silu_gate;
    long row_stride, ldy; int type, N, tile0;      // tile0: this job's first row tile in the launch's numbering of row tiles
};
struct PfP {
    PfJob job[PF_MAX_JOBS]; int njobs, nt_n, nt_t; const _Float16 * Xh; int K, T; int grp, pair; int splitk, full; float * ws; unsigned long long * trace;
    const uint8_t * Xd, * Xs; int ldt;               // 8-bit activations (pm_q8k_wide): scales, group sums
};
// Ablations (measurement builds only: -DPM_GEMM_ABLATE=1 adds instantiations of the Q4_K 256-token kernel, PM355_GEMM_EXP=<bits> picks one; results are WRONG when set):
// 1 no activation DMA, 2 no weight DMA, 4 no vmcnt wait / barrier, 8 no B fragment reads, 16 no dequantization, 32 no MFMA, 64 no stores;
// 128: s_memtime stamps of super-block 5's second k-step (waves 0 and 4 of workgroup 0), printed by the launcher: the phase timeline
#ifndef PM_GEMM_ABLATE
#define PM_GEMM_ABLATE 0
#endif

// 1 KiB of LDS at byte address `dst` (wave-uniform) <- 64 x 16 bytes, lane l from base (wave-uniform) + its own 32-bit offset. Inline asm, not
// __builtin_amdgcn_global_load_lds: with an LDS-DMA the compiler can see in flight, hipcc (ROCm 7.2) turns every counted `s_waitcnt lgkmcnt(N)` of the
// loop into lgkmcnt(0) - each slice's MFMAs then wait for the fragment reads just issued for the NEXT slice. Invisible to it, the ds_read ladder
// stays counted; the DMA's completion is this kernel's own business (the explicit vmcnt(0) in front of every barrier).
__device__ __forceinline__ void dma16(const uint8_t * base, uint32_t voff, uint32_t dst) {
    unsigned keep;
    dst = (uint32_t) __builtin_amdgcn_readfirstlane((int) dst);          // (provably scalar for the "s" constraint: the compiler keeps some loop counters in VGPRs)
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(voff), "s"(base), "s"(dst) : "memory");
}
__device__ __forceinline__ half2v h2(uint32_t u) { return __builtin_bit_cast(half2v, u); }
__device__ __forceinline__ uint32_t u2(half2v v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ half2v pk_fma(half2v a, half2v b, half2v c) { return __builtin_elementwise_fma(a, b, c); }

template <int TYPE> struct PfT;
// NSTREAM: 1-KiB DMA pieces per 128-k slot (32 rows x 32 bytes each); EXTRA: bytes behind the two header slots (Q5_K: two super-blocks' qh, Q6_K: 8 super-blocks' d)
template <> struct PfT<PM_Q4_K> { static constexpr int NSTREAM = 2, EXTRA = 0; };
template <> struct PfT<PM_Q5_K> { static constexpr int NSTREAM = 2, EXTRA = 2048; };
template <> struct PfT<PM_Q6_K> { static constexpr int NSTREAM = 3, EXTRA = 512; };
// Q8_0 (row-SoA qa[K/32][16] | qb[K/32][16] | half d[K/32]): slots of 64 k = one k-step (two blocks: 1 KiB of qa, 1 KiB of qb per wave), requested two steps ahead
template <> struct PfT<PM_Q8_0> { static constexpr int NSTREAM = 2, EXTRA = 0; };
template <int TYPE> constexpr int pf_wave_bytes() { return 2 * PfT<TYPE>::NSTREAM * 1024 + 1024 + PfT<TYPE>::EXTRA; }

// 8 weights -> one A operand: 16-k slice j of 64-k step ks (may be a run-time value) of 128-k piece mm of a super-block. Written stage by stage over the four independent half2
// chains (and - perm - add - fma): a dependent vector instruction issues ~8-10 cycles after its producer, four chains side by side hide that
template <int TYPE> __device__ __forceinline__ half8 pf_dequant(const u32x2 ql, const u32x2 qh, const int mm, const int ks, const int j, const half2v mul, const half2v add, half8 * low = nullptr) {
    uint32_t v[2];
    half2v t[4];
    if (TYPE == PM_Q8_0) {
        // int8 x -> byte x ^ 0x80 = x + 128 -> F16 1024 + 128 + x (exact) -> - 1152 -> * d: one rounding, dequantize_row_q8_0's d * x (ggml-quants.c:1616)
        const half2v bias = half2v{(_Float16) -1152.0f, (_Float16) -1152.0f};
#pragma unroll
        for (int c = 0; c < 2; ++c) v[c] = ql[c] ^ 0x80808080u;
#pragma unroll
        for (int c = 0; c < 2; ++c) { t[2 * c] = h2(__builtin_amdgcn_perm(0x64646464u, v[c], 0x05010400u)); t[2 * c + 1] = h2(__builtin_amdgcn_perm(0x64646464u, v[c], 0x07030602u)); }
#pragma unroll
        for (int c = 0; c < 4; ++c) t[c] = t[c] + bias;
#pragma unroll
        for (int c = 0; c < 4; ++c) t[c] = t[c] * mul;
    } else if (TYPE == PM_Q4_K || TYPE == PM_Q5_K) {
        const bool hi = j >> 1;                            // slices 2, 3: the unit's second sub-block = high nibbles
        const half2v bias = hi ? half2v{(_Float16) -64.0f, (_Float16) -64.0f} : half2v{(_Float16) -1024.0f, (_Float16) -1024.0f};
        uint32_t ex[2] = {hi ? 0x54545454u : 0x64646464u, hi ? 0x54545454u : 0x64646464u};   // F16 exponent byte: 64 + m / 16 (m = nibble << 4) / 1024 + m
#pragma unroll
        for (int c = 0; c < 2; ++c) v[c] = ql[c] & (hi ? 0xF0F0F0F0u : 0x0F0F0F0Fu);
        if (TYPE == PM_Q5_K) {
            // the 5th bit (bit s of the qh bytes, s = sub-block): low nibbles - bit 4 of the value byte; high nibbles (value byte = q << 4, ulp 1/16) - it is
            // mantissa bit 8 = bit 0 of the half's HIGH byte, which v_perm takes from the exponent operand
            const int sb = 4 * mm + 2 * ks + (j >> 1);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const uint32_t bit = (qh[c] >> sb) & 0x01010101u;
                if (hi) ex[c] |= bit; else v[c] |= bit << 4;
            }
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) { t[2 * c] = h2(__builtin_amdgcn_perm(ex[c], v[c], 0x05010400u)); t[2 * c + 1] = h2(__builtin_amdgcn_perm(ex[c], v[c], 0x07030602u)); }
#pragma unroll
        for (int c = 0; c < 4; ++c) t[c] = t[c] + bias;
#pragma unroll
        for (int c = 0; c < 4; ++c) t[c] = pk_fma(t[c], mul, add);
    } else {
        const half2v bias = half2v{(_Float16) -1056.0f, (_Float16) -1056.0f};  // 1024 + q - 32
        uint32_t lo4[2], hi2[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) lo4[c] = (ql[c] >> (4 * ks)) & 0x0F0F0F0Fu;
#pragma unroll
        for (int c = 0; c < 2; ++c) hi2[c] = (j >> 1 ? (qh[c] >> (4 * ks)) << 2 : (qh[c] >> (4 * ks)) << 4) & 0x30303030u;
#pragma unroll
        for (int c = 0; c < 2; ++c) v[c] = lo4[c] | hi2[c];
#pragma unroll
        for (int c = 0; c < 2; ++c) { t[2 * c] = h2(__builtin_amdgcn_perm(0x64646464u, v[c], 0x05010400u)); t[2 * c + 1] = h2(__builtin_amdgcn_perm(0x64646464u, v[c], 0x07030602u)); }
#pragma unroll
        for (int c = 0; c < 4; ++c) t[c] = t[c] + bias;
        if (low) {                                             // products (whole numbers up to 4096) as 64 x (-64 .. 64) + (-32 .. 32): 1536 + x rounds x to a whole number
            const half2v m64 = mul * half2v{(_Float16) 0.015625f, (_Float16) 0.015625f}, up = {(_Float16) 1536.0f, (_Float16) 1536.0f}, by = {(_Float16) -64.0f, (_Float16) -64.0f};
            half2v q[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) { q[c] = t[c]; t[c] = pk_fma(t[c], m64, up); }
#pragma unroll
            for (int c = 0; c < 4; ++c) t[c] = t[c] - up;
#pragma unroll
            for (int c = 0; c < 4; ++c) q[c] = pk_fma(q[c], mul, t[c] * by);
            *low = __builtin_bit_cast(half8, u32x4{u2(q[0]), u2(q[1]), u2(q[2]), u2(q[3])});
        } else
#pragma unroll
            for (int c = 0; c < 4; ++c) t[c] = t[c] * mul;
    }
    return __builtin_bit_cast(half8, u32x4{u2(t[0]), u2(t[1]), u2(t[2]), u2(t[3])});
}

// a wave's 32 x 32 results (matrix-core layout: token lane % 32, rows 8 g + 4 (lane / 32) .. + 3 in o[g]) -> slab [token][32 rows], through its LDS tile
__device__ __forceinline__ void store_slab(const f32x4 (&o)[4], uint8_t * xe, f32x4 * slab, int lane) {
    const int r = lane & 31, h = lane >> 5;
#pragma unroll
    for (int g = 0; g < 4; ++g) *(f32x4 *) (xe + r * 144 + (8 * g + 4 * h) * 4) = o[g];
#pragma unroll
    for (int q = 0; q < 4; ++q) *(PM_G f32x4 *) (slab + q * 64 + lane) = *(const f32x4 *) (xe + (8 * q + (lane >> 3)) * 144 + (lane & 7) * 16);
}

// the k loop + epilogue of one workgroup tile: rows [n0, n0 + 256) of job jb, tokens [t0, t0 + 32 NT)
// role: 0 plain; 1 / 2 = the gate / up half of a PAIR tile (waves 0-3 multiply ffn_gate's rows [n0, n0 + 128), waves 4-7 the same rows of ffn_up; the gate
// accumulators cross over through LDS after the k loop and the up waves store silu(gate) * up: ffn_gate's result never travels to HBM)
// NL: sub-tiles of the launch's tiles (its slabs)
template <int TYPE, int NT, int EXP, int NL>
__device__ __forceinline__ void pf_body(const PfP & p, const PfJob & jb, const int n0, const int t0, uint8_t * smem, const int role, const int ks, const int S, const int tile_id) {
    constexpr int BBUF = NT * 32 * 128;                       // one activation buffer: 32 NT tokens x 64 halfs
    constexpr int NSTREAM = PfT<TYPE>::NSTREAM, SLOT = NSTREAM * 1024, AW = pf_wave_bytes<TYPE>();   // per wave: two 128-k slots + two 512-byte header slots + EXTRA
    constexpr bool K45 = TYPE == PM_Q4_K || TYPE == PM_Q5_K, Q8 = TYPE == PM_Q8_0;
    constexpr int NQ = NT >= 4 ? NT / 2 : 1;                  // activation DMA instructions per wave and k-step (NT = 2: 64 token rows = one per wave)
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, h = lane >> 5;
    // nb = super-blocks of 256 k the loop walks; Q8_0 rows may end on half of one (K % 256 == 128: Qwen2.5-72B's ffn_down, K = 29568) - the weight operand of
    // the missing half is zeroed, its look-ahead requests are clamped to the last real k-step
    const int K = p.K, nst = K / 64, nb = (K + 255) / 256;
    const bool half_tail = Q8 && (K & 255) != 0;
    constexpr int exp = EXP;
    uint8_t * const aw = smem + 3 * BBUF + wave * AW;
    const uint32_t lds0 = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) uint8_t *) smem;     // LDS byte address of the tile memory
    const uint32_t aw_l = lds0 + 3 * BBUF + wave * AW;

    // ---- DMA sources. weights: lane (row r, 16-byte piece h of the 32 bytes a 128-k slot holds per row and stream)
    const uint8_t * const Wg = jb.W;
    const int nw = n0 + 32 * (role ? wave & 3 : wave);         // first row of this wave
    const uint32_t wrow = (uint32_t) min(nw + r, jb.N - 1) * (uint32_t) jb.row_stride;
    const uint32_t wsrc = wrow + 16u * (uint32_t) h;
    //      activations: instruction q of this wave = token rows 8 (wave + 8 q) .. + 8, lane (row lane / 8, LDS chunk lane % 8 <- global chunk ^ swizzle)
    const uint8_t * const Xg = (const uint8_t *) p.Xh;
    uint32_t xsrc[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int t = 8 * (wave + 8 * q) + (lane >> 3);
        const int c = (lane & 7) ^ ((t >> 1) & 7);
        xsrc[q] = (uint32_t) min(t0 + t, p.T - 1) * (uint32_t) (2 * K) + 16u * (uint32_t) c;
    }
    // ---- fragment reads: B = activations, lane (token r of tile jt, k-half h): chunk 2 j + h of slice j at its swizzled place
    //      (slice j: XOR with j << 5 - the chunk index 2 j + h has j in bits 1..2, and so has the byte offset in bits 5..6)
    const uint32_t boff0 = (uint32_t) (r * 128 + ((h ^ ((r >> 1) & 7)) << 4));
    const uint32_t aoff = (uint32_t) (r * 16 + 8 * h);        // A: 8 bytes of row r in a [32 rows][16] piece image

    // one DMA instruction each (the waits below count them): part q of k-step s's activations, stream st of weight piece m, the header of super-block b
    auto issue_B = [&](int s, uint32_t buf, int q) __attribute__((always_inline)) {
        if (exp & 1) return;
        dma16(Xg, xsrc[q] + (uint32_t) min(s, nst - 1) * 128u, lds0 + buf + (wave + 8 * q) * 1024);
    };
    auto issue_A = [&](int m, int slot, int st) __attribute__((always_inline)) {    // 128-k piece m of the rows -> slot
        if (exp & 2) return;
        if (Q8) {                 // m = k-step: blocks 2 m + h of stream st (0 qa, 1 qb)
            const uint32_t sc = (uint32_t) min(m, nst - 1);
            dma16(Wg, wrow + (st ? (uint32_t) K / 2u : 0u) + (2u * sc + (uint32_t) h) * 16u, aw_l + slot * SLOT + st * 1024);
            return;
        }
        const uint32_t mc = (uint32_t) min(m, 2 * nb - 1);
        if (TYPE == PM_Q5_K)      // native 176-byte blocks: qs at + 48; lane (r, h) = bytes [16 st, + 16) of unit 2 (m % 2) + h
            dma16(Wg, wrow + (mc >> 1) * 176u + 48u + (mc & 1u) * 64u + 32u * (uint32_t) h + 16u * (uint32_t) st, aw_l + slot * SLOT + st * 1024);
        else
            dma16(Wg, wsrc + 32u * mc + (uint32_t) st * (uint32_t) nb * 64u, aw_l + slot * SLOT + st * 1024);
    };
    auto issue_H = [&](int b) __attribute__((always_inline)) {                       // header (Q4_K) / int8 scales (Q6_K) of super-block b
        if (exp & 2) return;
        const uint32_t bc = (uint32_t) min(b, nb - 1);
        const uint32_t off = TYPE == PM_Q4_K ? (uint32_t) nb * 128u + bc * 16u : TYPE == PM_Q5_K ? bc * 176u : Q8 ? (uint32_t) K + bc * 16u /* 8 blocks' d */ : pm_q6k_sc_off((uint32_t) nb, bc);
        if (h == 0) dma16(Wg, wrow + off, aw_l + 2 * SLOT + (b & 1) * 512);
    };
    auto issue_QH = [&](int b) __attribute__((always_inline)) {                      // Q5_K: the 32 qh bytes of super-block b, lane (r, h) = bytes [16 h, + 16)
        if (exp & 2) return;
        dma16(Wg, wrow + (uint32_t) min(b, nb - 1) * 176u + 16u + 16u * (uint32_t) h, aw_l + 2 * SLOT + 1024 + (b & 1) * 1024);
    };
    auto issue_D = [&](int g) __attribute__((always_inline)) {                       // Q6_K: the fp16 d of super-blocks 8 g .. 8 g + 7 (16 bytes per row)
        if (exp & 2) return;
        // (16 bytes from the group's first d: a last group of fewer than 8 super-blocks ends exactly at the 16-byte-rounded row stride, pm_q6k_row_stride)
        if (h == 0) dma16(Wg, wrow + pm_q6k_d_off((uint32_t) nb, (uint32_t) (8 * min(g, (nb - 1) >> 3))), aw_l + 2 * SLOT + 1024);
    };

    // ---- weight path, per 16-k slice i of a super-block (i = 0..15: k-step i / 4, slice j = i % 4; 128-k piece mm = i / 8, k-step ks = (i / 4) % 2 of it)
    struct Raw { u32x2 ql, qh; };
    auto read_raw = [&](int i, int b) __attribute__((always_inline)) {                // slice i of super-block b
        const int mm = (i >> 3) & 1, ks = (i >> 2) & 1, j = i & 3;
        Raw w;
        if (Q8) {
            // block j / 2 of the k-step (slot = the step's parity), its first (qa) or second (qb) sixteen values, bytes [8 h, + 8)
            w.ql = *(const u32x2 *) (aw + ((i >> 2) & 1) * SLOT + (j & 1) * 1024 + (j >> 1) * 512 + aoff);
            w.qh = u32x2{0, 0};
        } else if (K45) {
            // unit ks of the slot: qa = qs[0, 16) / qb = qs[16, 32) of its 64 weights; slices 0, 2 read qa, slices 1, 3 qb
            w.ql = *(const u32x2 *) (aw + mm * SLOT + (j & 1) * 1024 + ks * 512 + aoff);
            w.qh = u32x2{0, 0};
            if (TYPE == PM_Q5_K) w.qh = *(const u32x2 *) (aw + 2 * SLOT + 1024 + (b & 1) * 1024 + (j & 1) * 512 + aoff);   // qh[16 (j & 1) + 8 h, + 8): bit s = 5th bit of sub-block s
        } else {
            // 32-weight group g = 2 ks + j / 2 of the 128-weight half: ql stream (g & 1), piece v = j & 1, nibble ks; qh piece v, bit pair g
            const int v = j & 1, st = j >> 1;
            w.ql = *(const u32x2 *) (aw + mm * SLOT + st * 1024 + v * 512 + aoff);
            w.qh = *(const u32x2 *) (aw + mm * SLOT + 2048 + v * 512 + aoff);
        }
        return w;
    };
    u32x4 hd = {0, 0, 0, 0};                                   // Q4_K: d | dmin | scales[12];  Q6_K: int8 scales[16]
    uint16_t d6h = 0;                                          // Q6_K: the super-block's fp16 d
    auto read_hdr = [&](int b) __attribute__((always_inline)) {
        hd = *(const u32x4 *) (aw + 2 * SLOT + (b & 1) * 512 + r * 16);
        if (TYPE == PM_Q6_K) d6h = *(const uint16_t *) (aw + 2 * SLOT + 1024 + r * 16 + (b & 7) * 2);
    };
    half2v mul = {0, 0}, add = {0, 0}, muln = {0, 0}, addn = {0, 0};
    auto scales = [&](int i, half2v & mul, half2v & add) __attribute__((always_inline)) {   // multiplier / addend of slice i (constant per sub-block / 16-group)
        if (Q8) {
            const int q = i >> 1;                              // block of the super-block: its d is already an F16 number
            const _Float16 dd = __builtin_bit_cast(_Float16, (uint16_t) (hd[q >> 1] >> (16 * (q & 1))));
            mul = half2v{dd, dd};
        } else if (K45) {
            const int s = i >> 1;                              // 32-weight sub-block of the super-block
            int sc, mn;
            k4_scale_min(hd[1], hd[2], hd[3], s, sc, mn);
            const _Float16 ds = (_Float16) (h2f((uint16_t) (hd[0] & 0xFFFF)) * (float) sc), ms = (_Float16) (h2f((uint16_t) (hd[0] >> 16)) * (float) mn);
            mul = half2v{ds, ds}; add = half2v{(_Float16) -ms, (_Float16) -ms};
        } else {
            const int mm = (i >> 3) & 1, ks = (i >> 2) & 1, j = i & 3;
            const int G = 8 * mm + 2 * (2 * ks + (j >> 1)) + (j & 1);               // 16-weight group of the super-block
            const _Float16 dd = (_Float16) (h2f(d6h) * (float) (int) (int8_t) (hd[G >> 2] >> (8 * (G & 3))));
            mul = half2v{dd, dd};
        }
    };
    auto dequant = [&](const Raw & w, int i) __attribute__((always_inline)) { return pf_dequant<TYPE>(w.ql, w.qh, (i >> 3) & 1, (i >> 2) & 1, i & 3, mul, add); };

    float16v acc[NT];
#pragma unroll
    for (int jt = 0; jt < NT; ++jt)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[jt][e] = 0.0f;
    half8 bf[NT], af[2];                                       // B fragments of the slice (re-filled right behind its MFMAs), A operand of this / the next slice
    Raw raw;
    auto read_B = [&](uint32_t buf, int j, int jt) __attribute__((always_inline)) {
        return *(const half8 *) (smem + buf + jt * 4096 + (boff0 ^ (uint32_t) (j << 5)));
    };

    // ---- prologue: super-block 0's header, piece 0, k-steps 0 and 1
    uint32_t rd = 0, nx = BBUF, wr = 2 * BBUF;                 // ring: buffer of step s, s + 1, s + 2
    // split K: slice ks of S takes the super-blocks [b0, b1); all indices below stay absolute (slot parities, look-ahead clamps)
    const int b0 = (int) ((long) ks * nb / S), b1 = (int) ((long) (ks + 1) * nb / S);
    issue_H(b0); if (TYPE == PM_Q6_K) issue_D(b0 >> 3); if (TYPE == PM_Q5_K) issue_QH(b0);
#pragma unroll
    for (int st = 0; st < NSTREAM; ++st) { if (Q8) { issue_A(4 * b0, 0, st); issue_A(4 * b0 + 1, 1, st); } else issue_A(2 * b0, 0, st); }
#pragma unroll
    for (int q = 0; q < NQ; ++q) { issue_B(4 * b0, rd, q); issue_B(4 * b0 + 1, nx, q); }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    read_hdr(b0);
    raw = read_raw(0, b0);
    scales(0, mul, add);
    af[0] = dequant(raw, 0);
    if (TYPE == PM_Q6_K) scales(1, mul, add);
    raw = read_raw(1, b0);
#pragma unroll
    for (int jt = 0; jt < NT; ++jt) bf[jt] = read_B(rd, 0, jt);
    // Two waves share a SIMD (waves w and w + 4): the second group runs HALF A SLICE behind the first, so that on every SIMD one wave is in the memory
    // half of a slice (DMA issue, fragment reads) while the other is in its MFMA half - in lock-step (first version of this kernel) both issued their
    // DMAs, then both read, then both multiplied, and the pieces added up instead of overlapping (profiles/r06_prefill_ablation.txt).
    const bool late = p.grp == 1 ? (wave & 1) : p.grp == 2 ? ((wave >> 1) & 1) : wave >= 4;
    if (late && !(exp & 4)) __builtin_amdgcn_s_barrier();

    unsigned long long ts[17] = {};
    auto stamp = [&](int k, int b) __attribute__((always_inline)) {
        if ((exp & 128) && b == b0 + 5) asm volatile("s_memtime %0" : "=s"(ts[k]));
    };
    for (int b = b0; b < b1; ++b) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int j = i & 3, sq = i >> 2;                  // slice of the k-step, k-step of the super-block
            if (sq == 1) stamp(4 * j, b);
            // ---- memory half of slice i.
            // DMA schedule of k-step s (at most two instructions per slice: an issue blocks the wave for 60-180 cycles): slice j carries part j of step
            // s + 2's activations; the next weight piece's streams ride in slices 1, 2, 3 of steps 0 and 2, the next header in slice 1 of step 1 (Q6_K:
            // the d's of the next eight super-blocks in slice 3 of step 0, when due). Everything requested in step s has landed when step s + 1's
            // slice 2 begins: `vmcnt(N)` there, N = what slices 0 and 1 of step s + 1 issued. For the activations a barrier follows before their first
            // reader (slice 3 of step s + 1 reads the fragments of step s + 2's first slice); the weights are the wave's own.
            if (j == 2 && !(exp & 3)) {
                constexpr int N8[4] = {3, 3, 3, 2}, N4[4] = {2, 2, 2, 1}, Q8N8[4] = {2, 3, 2, 2}, Q8N4[4] = {1, 2, 1, 1};
                const int n = Q8 ? (NT >= 6 ? Q8N8[sq] : Q8N4[sq]) : NT >= 6 ? N8[sq] : N4[sq];
                if (n == 3) asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
                else if (n == 2) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
                else asm volatile("s_waitcnt vmcnt(1)" ::: "memory");
            }
            if (NT == 8 || (NT == 6 && j < 3) || (NT == 4 && (j & 1) == 0) || j == 0) issue_B(4 * b + sq + 2, wr, NT >= 6 ? j : NT == 4 ? j >> 1 : 0);
            // (Q8_0: the 64-k slot of step s is free once its last slice has been read - behind slice 1 - and takes step s + 2's blocks in slices 2 and 3)
            if (Q8) { if (j >= 2) issue_A(4 * b + sq + 2, sq & 1, j - 2); }
            else if ((sq == 0 || sq == 2) && j >= 1 && j - 1 < NSTREAM) issue_A(2 * b + 1 + (sq >> 1), sq == 0 ? 1 : 0, j - 1);
            if (sq == 1 && j == 1) issue_H(b + 1);
            if (TYPE == PM_Q5_K && sq == 1 && j == 2) issue_QH(b + 1);
            // (the slot's last reader - d of super-block 8 g + 7 - ran at slice 13 of super-block 8 g + 6; the first reader of the new group runs at slice 13 of 8 g + 7)
            if (TYPE == PM_Q6_K && sq == 0 && j == 3 && (b & 7) == 7) issue_D((b >> 3) + 1);
            __builtin_amdgcn_sched_barrier(0);
            // the wave's vector work: the F16 operand of slice i + 1. HERE, not between the MFMAs: a packed-F16 instruction next to a wave's own MFMA costs its
            // full 8 cycles of issue (measured: 8 MFMAs + 22 vector instructions = 448 cycles, 56 per MFMA, while this half idled 250 cycles at its barrier)
            // (the multiplier of slice i + 2 is formed next to it, an independent chain: slice i + 1's was formed one slice ago)
            const bool newgrp = TYPE == PM_Q6_K || (i & 1) == 0;
            if (newgrp && !(exp & 16)) scales((i + 2) & 15, muln, addn);
            if (!(exp & 16)) af[(i + 1) & 1] = dequant(raw, (i + 1) & 15);
            if (Q8 && i >= 7 && i < 15 && half_tail && b == nb - 1) af[(i + 1) & 1] = half8{0, 0, 0, 0, 0, 0, 0, 0};      // (k >= K: the row has no such weights)
            if (newgrp) { mul = muln; add = addn; }
            __builtin_amdgcn_sched_barrier(0);
            if (sq == 1) stamp(4 * j + 1, b);
            if (!(exp & 4)) __builtin_amdgcn_s_barrier();
            if (sq == 1) stamp(4 * j + 2, b);
            // ---- MFMA half
            // the slice's MFMAs; fragment jt of slice i + 1 goes into the SAME registers right behind the MFMA that read them (at j == 3: slice 0 of the next
            // step, from the next ring buffer): a 1-KiB read takes the LDS ~13 cycles with four waves reading, well inside an MFMA's 32. The consumers sit
            // behind two barriers, so the scheduler cannot sink the reads to them.
            __builtin_amdgcn_s_setprio(1);
            {
                const uint32_t nbuf = j == 3 ? nx : rd;
#pragma unroll
                for (int jt = 0; jt < NT; ++jt) {
                    if (!(exp & 32)) acc[jt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i & 1], bf[jt], acc[jt], 0, 0, 0);
                    if (!(exp & 8)) bf[jt] = read_B(nbuf, (j + 1) & 3, jt);
                }
#pragma unroll
                for (int jt = 0; jt < NT; ++jt) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // 1 MFMA
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);      // 1 DS read
                }
            }
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
            raw = read_raw((i + 2) & 15, b + ((i + 2) >> 4));                       // (consumed after two barriers: no exposed latency)
            if (i == 13) read_hdr(b + 1);
            if (sq == 1) stamp(4 * j + 3, b);
            if (!(exp & 4)) __builtin_amdgcn_s_barrier();
            if (i == 7) stamp(16, b);
            if (j == 3) { const uint32_t t = rd; rd = nx; nx = wr; wr = t; }
        }
    }

    if ((exp & 128) && p.trace && blockIdx.x == 0 && lane == 0) {
        unsigned hwid;
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID)" : "=s"(hwid));
        p.trace[34 + wave] = hwid;
    }
    if ((exp & 128) && p.trace && blockIdx.x == 0 && (wave == 0 || wave == 4) && lane == 0) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int k = 0; k < 17; ++k) p.trace[(wave >> 2) * 17 + k] = ts[k];
    }
    f32x4 * const xlds = (f32x4 *) smem;
    if (role || S > 1) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // (the last steps' look-ahead DMAs still land in the ring)
        if (!late && !(exp & 4)) __builtin_amdgcn_s_barrier();  // (the second group has passed one barrier more: level)
        __builtin_amdgcn_s_barrier();                           // every wave is out of the k loop: the tile memory is free
    }
    // ---- split K: every slice leaves its partial tile in a slab for pf_reduce_kernel, 32 rows of a token as one line (turned in a wave-private LDS tile [token][32 rows + 4])
    if (S > 1) {
        f32x4 * const mine = (f32x4 *) p.ws + (size_t) (tile_id * S + ks) * (8 * NL * 4 * 64);
#pragma unroll
        for (int jt = 0; jt < NT; ++jt) {
            f32x4 o[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) o[g] = f32x4{acc[jt][4 * g], acc[jt][4 * g + 1], acc[jt][4 * g + 2], acc[jt][4 * g + 3]};
            store_slab(o, smem + wave * (32 * 144), mine + (wave * NL + jt) * 256, lane);
        }
        return;
    }
    // ---- pair tiles: the gate waves park their accumulators in LDS (same lane, same register index as the up wave that needs them)
    if (role) {
        if (role == 1) {
#pragma unroll
            for (int jt = 0; jt < NT; ++jt)
#pragma unroll
                for (int g = 0; g < 4; ++g) xlds[(((wave & 3) * NT + jt) * 4 + g) * 64 + lane] = f32x4{acc[jt][4 * g], acc[jt][4 * g + 1], acc[jt][4 * g + 2], acc[jt][4 * g + 3]};
        }
        __syncthreads();
        if (role == 1) return;
    }
    // ---- epilogue: C[row = (e & 3) + 8 (e >> 2) + 4 h][col = r]; Y[t][n]: 4 consecutive n per float4
#pragma unroll
    for (int jt = 0; jt < NT; ++jt) {
        const int t = t0 + 32 * jt + r;
        if (t >= p.T || (exp & 64)) continue;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int n = nw + 8 * g + 4 * h;
            const long o = (long) t * jb.ldy + n;
            if (role == 2) {                                    // silu(gate) * up, the arithmetic of the separate launches (silu_gate epilogue below)
                const f32x4 gg = xlds[(((wave & 3) * NT + jt) * 4 + g) * 64 + lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[jt][4 * g + e] *= gg[e] / (1.0f + expf(-gg[e]));
            }
            if (n + 3 < jb.N) {
                float4 v = {acc[jt][4 * g], acc[jt][4 * g + 1], acc[jt][4 * g + 2], acc[jt][4 * g + 3]};
                if (jb.bias)  { const float4 bb = ld_g((const float4 *) (jb.bias + n)); v.x += bb.x; v.y += bb.y; v.z += bb.z; v.w += bb.w; }
                if (jb.resid) { const float4 rr = ld_g((const float4 *) (jb.resid + o)); v.x += rr.x; v.y += rr.y; v.z += rr.z; v.w += rr.w; }
                if (jb.silu_gate) {
                    const float4 gg = ld_g((const float4 *) (jb.silu_gate + o));
                    v.x *= gg.x / (1.0f + expf(-gg.x)); v.y *= gg.y / (1.0f + expf(-gg.y)); v.z *= gg.z / (1.0f + expf(-gg.z)); v.w *= gg.w / (1.0f + expf(-gg.w));
                }
                if (jb.Yh) *(PM_G half4v *) (jb.Yh + o) = half4v{(_Float16) v.x, (_Float16) v.y, (_Float16) v.z, (_Float16) v.w};
                else *(PM_G f32x4 *) (jb.Y + o) = f32x4{v.x, v.y, v.z, v.w};
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) if (n + e < jb.N) {
                    float v = acc[jt][4 * g + e];
                    if (jb.bias) v += jb.bias[n + e];
                    if (jb.resid) v += jb.resid[o + e];
                    if (jb.silu_gate) { const float gg = jb.silu_gate[o + e]; v *= gg / (1.0f + expf(-gg)); }
                    if (jb.Yh) jb.Yh[o + e] = (_Float16) v; else jb.Y[o + e] = v;
                }
            }
        }
    }
}

// ---- one round of workgroups (NT = 2 / 3 / 4): 128 rows x 32 NT tokens per workgroup, wave (g, kk) = rows [32 g, + 32) x the kk-th 64 k of every 128-k step ----
// Few tokens leave little to multiply between two barriers. The loop above - 256 rows, two barriers per 16-k slice - spent 860 cycles on a slice of 128 tokens (128 of them in
// MFMAs), half of them in barriers with nothing else left in it, and a launch had 16-64 tiles whose last K slice then read all slabs and stored 16-byte pieces of 32 token rows
// by itself (14 of the 34 us of a 4096 x 4096 launch). Here: one barrier per 128 k; both halves of a step are multiplied side by side and added up through LDS at the end (half the
// slabs of a K split for the same number of workgroups); three activation buffers, weights requested 2 to 4 steps ahead; tiles of 128 rows, so that twice as many
// workgroups share the reduction; results cross LDS once more and are stored as whole 128-byte pieces of a token row.
// Operands are requested by four waves that do nothing else (mid_load); where a kernel's registers leave no room for them, by the ones that multiply, a quarter of a step's behind each slice's
// products. 8B shape, Q4_K at 101 tokens, us, requests by the waves that multiply / by their own: ffn_gate | ffn_up 51.9 / 45.6, ffn_down 28.7 / 26.5, wo 18.0 / 17.0, wq | wk | wv 20.0 / 18.7.
// What bounds it, four layers of that (646 us, 411 without any step): the requests alone 168 of the 235 us of steps - weights 91, whose 32-byte pieces of a line are asked for line by line four
// times over, activations 41 -, LDS reads, dequantization and MFMAs alone 136. Tiles of 96 tokens cost 0.8 of those of 128. Two layers, Q4_K, us, neither / loaders / tiles of 96
// too: 70 tokens 286 / 264 / 241, 90 tokens 290 / 272 / 250, 101 tokens 293 / 276 / 275; 8-bit activations, eight prompts of up to 12 tokens 498 / 494 / 452, of up to 24 706 / 692 / 624, of up to 30 728 / 714 / 645.
// Llama-3-8B's launches at 101 tokens, Q4_K, us in the general tiles / as these were first: wq | wk | wv 37 / 24, wo 34 / 23, ffn_gate | ffn_up 61 / 50, ffn_down 54 / 36.6. Taken back: 64 rows and
// a quarter of the k per wave (half the LDS reads: no change, 1-2 us more for the longer merge); two activation buffers instead of three (2-10 % slower); a step's first fragments read in the
// step before, whose activations then have one step to arrive instead of two (646 -> 680).
template <int TYPE> constexpr int mid_slot() { return TYPE == PM_Q8_0 ? 4096 : PfT<TYPE>::NSTREAM * 1024; }           // 128 k of 32 rows
// weights are requested this many steps ahead (what LDS has room for)
template <int TYPE, bool EX> constexpr int mid_ahead() { return TYPE == PM_Q8_0 || (EX && TYPE == PM_Q5_K) ? 2 : TYPE == PM_Q6_K ? 3 : 4; }
template <int TYPE, bool EX> constexpr int mid_group_bytes() { return (mid_ahead<TYPE, EX>() + 1) * mid_slot<TYPE>() + 2048 + (TYPE == PM_Q5_K ? 4096 : TYPE == PM_Q6_K ? 1024 : 0); }   // + four headers, four qh, two groups of d
// EX, per super-block: 16 group sums (not for Q6_K: no minima) and a scale of every token, two buffers
template <int TYPE, int NT> constexpr int mid_sum_bytes() { return TYPE == PM_Q6_K ? 0 : NT * 32 * 32; }
template <int TYPE, int NT, bool EX> constexpr size_t mid_lds_bytes() { return (size_t) 6 * NT * 32 * 128 + (size_t) 4 * mid_group_bytes<TYPE, EX>() + (EX ? 2 * (mid_sum_bytes<TYPE, NT>() + NT * 32 * 4) : 0); }
// no waves of their own for the requests: where the kernel's registers leave no room for them (168 a wave). 8B shape, 147 tokens of 8-bit activations, wq | wk | wv with a Q6_K wv: 53 us, with loaders
// and 12 registers spilled 68
// PF_SELF (a bit of EXP): or where a loader's requests are the longer part of a step - Q8_0, four pieces of 1 KiB to a row group and 128 k, up to 64 tokens, where half of the chip is idle anyway: less
// than 128 workgroups. us at 64 tokens, four loaders / none: 1024 x 512 10.8 / 10.0, 1024 x 1024 14.3 / 13.4, 2048 x 3072 16.8 / 16.0, 512 x 8192 18.9 / 18.1; from 128 workgroups on 6144 x 4096 20.2 /
// 20.4, 8192 x 8192 29.7 / 30.4. Or where a launch is four steps, K = 512 of the other types at 97..128 tokens: us at 128 tokens, four loaders / none, Q4_K 256 rows 11.7 / 11.2, 32768 rows 14.0 / 13.6, Q5_K
// 4096 rows 12.4 / 12.3, Q6_K 12.6 / 12.1; at 33..64 tokens 0.98-1.00, 1.01-1.05 and 1.00-1.05 of the time, and from K = 1024 on loaders win
constexpr int PF_SELF = 512;
template <int TA, int TB, int NT, bool EX, int EXP = 0> constexpr bool mid_self() { return (EXP & PF_SELF) || (EX && (NT == 4 || TA != TB || TA == PM_Q5_K)); }
template <int N> __device__ __forceinline__ void mid_wait() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory"); }

// A tile's requests. Those of weights and of activations are different waves': requests return in order, and weights come from memory (AHEAD steps ahead), activations mostly from L2 (two steps)
// ... the weights of NG row groups of one wave
template <int TYPE, int NT, bool EX, int NG> struct MidWeights {
    static constexpr int SLOT = mid_slot<TYPE>(), W = SLOT / 1024, AHEAD = mid_ahead<TYPE, EX>(), HDR = (AHEAD + 1) * SLOT, XTRA = HDR + 2048, E = TYPE == PM_Q5_K || TYPE == PM_Q6_K ? 2 : 1;
    const uint8_t * Wg; uint32_t row[NG], ag[NG], sw; int h, K, nsteps, nb;
    // group g0 + u; row n0 + 32 (r0 + u) of the matrix on
    __device__ __forceinline__ void init(const PfP & p, const PfJob & jb, int n0, int g0, int r0, uint32_t lds0, int lane) {
        Wg = jb.W; h = lane >> 5; K = p.K; nsteps = K / 128; nb = (K + 255) / 256; sw = 0;
#pragma unroll
        for (int u = 0; u < NG; ++u) {
            row[u] = (uint32_t) min(n0 + 32 * (r0 + u) + (lane & 31), jb.N - 1) * (uint32_t) jb.row_stride;
            ag[u] = lds0 + (uint32_t) (6 * NT * 32 * 128 + (g0 + u) * mid_group_bytes<TYPE, EX>());
        }
    }
    // part u (0..3) of step s's requests
    __device__ __forceinline__ void issue(int s, bool even, int u) const {
        const uint32_t sc = (uint32_t) min(s, nsteps - 1);
        const int b = s >> 1;
        const uint32_t bc = (uint32_t) min(b, nb - 1);
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            if (u < W) {                                        // stream u
                uint32_t off;
                if (TYPE == PM_Q8_0) off = (u & 1 ? (uint32_t) K / 2u : 0u) + (4u * sc + 2u * (uint32_t) (u >> 1) + (uint32_t) h) * 16u;       // blocks 2 k + h of k-step k = 2 s + u / 2, stream qa / qb
                else if (TYPE == PM_Q5_K) off = (sc >> 1) * 176u + 48u + (sc & 1u) * 64u + 32u * (uint32_t) h + 16u * (uint32_t) u;
                else off = 16u * (uint32_t) h + 32u * sc + (uint32_t) u * (uint32_t) nb * 64u;
                dma16(Wg, row[i] + off, ag[i] + sw + u * 1024);
            }
            if (even && u == 3) {
                const uint32_t off = TYPE == PM_Q4_K ? (uint32_t) nb * 128u + bc * 16u : TYPE == PM_Q5_K ? bc * 176u : TYPE == PM_Q8_0 ? (uint32_t) K + bc * 16u : pm_q6k_sc_off((uint32_t) nb, bc);
                if (h == 0) dma16(Wg, row[i] + off, ag[i] + HDR + (b & 3) * 512);
            }
            if (even && u == 2) {
                if (TYPE == PM_Q5_K) dma16(Wg, row[i] + bc * 176u + 16u + 16u * (uint32_t) h, ag[i] + XTRA + (b & 3) * 1024);
                // (the d's of a group of eight super-blocks: with every one of them, the same bytes again)
                if (TYPE == PM_Q6_K && h == 0) dma16(Wg, row[i] + pm_q6k_d_off((uint32_t) nb, (uint32_t) (8 * min(b >> 3, (nb - 1) >> 3))), ag[i] + XTRA + ((b >> 3) & 1) * 512);
            }
        }
    }
    __device__ __forceinline__ void turn() { sw = sw == AHEAD * SLOT ? 0 : sw + SLOT; }
    // the next step's are there: all but those of the AHEAD - 1 steps behind it
    static __device__ __forceinline__ void wait(bool even) {
        if (even) mid_wait<NG * ((AHEAD - 1) * W + AHEAD / 2 * E)>(); else mid_wait<NG * ((AHEAD - 1) * W + (AHEAD - 1) / 2 * E)>();
    }
};
// ... and the activations, every NW-th request of a step by one of NW waves: (64-k half, token rows 8 q .. + 8), lane (row lane / 8, chunk lane % 8 <- chunk ^ swizzle). EX: group sums and scales of
// every token with an even step, for the next super-block
template <int TYPE, int NT, bool EX, int NW> struct MidActs {
    static constexpr int HB = NT * 32 * 128, BBUF = 2 * HB, NQ = 8 * NT / NW, XSUM = mid_sum_bytes<TYPE, NT>(), XB = XSUM + NT * 32 * 4, XS = 3 * BBUF + 4 * mid_group_bytes<TYPE, EX>(),
                         XP = XSUM / NW, XN = EX ? (XP + 1023) / 1024 + 1 : 0;
    const uint8_t * Xg, * Xd, * Xs; uint32_t src[NQ], lds, bw; int w, lane, nsteps, nb, ldt, t0;
    __device__ __forceinline__ void init(const PfP & p, int t0_, int w_, uint32_t lds0, int lane_) {
        Xg = (const uint8_t *) p.Xh; Xd = p.Xd; Xs = p.Xs; lds = lds0; bw = 0; w = w_; lane = lane_; nsteps = p.K / 128; nb = (p.K + 255) / 256; ldt = p.ldt; t0 = t0_;
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const int q = w + NW * i, t = 8 * (q % (4 * NT)) + (lane >> 3);
            src[i] = (uint32_t) min(t0 + t, p.T - 1) * (uint32_t) (2 * p.K) + 128u * (uint32_t) (q / (4 * NT)) + 16u * (uint32_t) ((lane & 7) ^ ((t >> 1) & 7));
        }
    }
    // requests [from, to) of step s
    __device__ __forceinline__ void issue(int s, int from, int to) const {
        const uint32_t at = (uint32_t) min(s, nsteps - 1) * 256u;
#pragma unroll
        for (int i = from; i < to; ++i) dma16(Xg, src[i] + at, lds + bw + (uint32_t) ((w + NW * i) * 1024));
    }
    __device__ __forceinline__ void issue_x(int b) const {
        const uint32_t at = (uint32_t) min(b, nb - 1) * (uint32_t) ldt + (uint32_t) t0, dst = lds + (uint32_t) (XS + (b & 1) * XB);
#pragma unroll
        for (int o = 0; o < XP; o += 1024) if (o + lane * 16 < XP) dma16(Xs, at * 32u + (uint32_t) (w * XP + o + lane * 16), dst + (uint32_t) (w * XP + o));
        if (lane < 8 * NT / NW) dma16(Xd, at * 4u + (uint32_t) (w * 128 * NT / NW + lane * 16), dst + (uint32_t) (XSUM + w * 128 * NT / NW));
    }
    __device__ __forceinline__ void turn() { bw = bw == 2 * BBUF ? 0 : bw + BBUF; }
    static __device__ __forceinline__ void wait(bool x) { if (x) mid_wait<NQ + XN>(); else mid_wait<NQ>(); }
};
// Four waves of a workgroup that multiply nothing: 0, 1 bring the activations, 2, 3 the weights of two row groups each. (One wave's LDS-DMA moves 61 GB/s, two 119, a CU not much more than
// that: 143. A request holds its wave up for 60-180 cycles while others are at it.)
template <int TYPE, int NT, bool EX>
__device__ __forceinline__ void mid_load(const PfP & p, const PfJob & jb, const int n0, const int t0, uint32_t lds0, const int role, const int b0, const int b1, const int lw, const int lane) {
    const int n = min(2 * b1, p.K / 128) - 2 * b0;              // steps
    auto meet = [&] __attribute__((always_inline)) { __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); };
    if (lw < 2) {
        typedef MidActs<TYPE, NT, EX, 2> A;
        A x;
        x.init(p, t0, lw, lds0, lane);
        if (EX) x.issue_x(b0);
        x.issue(2 * b0, 0, A::NQ); x.turn();
        x.issue(2 * b0 + 1, 0, A::NQ); x.turn();
        A::wait(false);
        meet();
        for (int s = 0; s < n; ++s) {
            const bool with = EX && !(s & 1);
            if (with) x.issue_x(b0 + (s >> 1) + 1);
            x.issue(2 * b0 + s + 2, 0, A::NQ); x.turn();
            A::wait(with);
            meet();
        }
    } else {
        typedef MidWeights<TYPE, NT, EX, 2> M;
        M x;
        x.init(p, jb, n0, 2 * (lw - 2), role ? 0 : 2 * (lw - 2), lds0, lane);
        auto step = [&](int s, bool even) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < 4; ++u) x.issue(s, even, u);
            x.turn();
        };
#pragma unroll
        for (int w = 0; w < M::AHEAD; ++w) step(2 * b0 + w, (w & 1) == 0);
        M::wait(false);
        meet();
        for (int s = 0; s < n; ++s) {
            const bool even = !(s & 1);
            step(2 * b0 + s + M::AHEAD, M::AHEAD & 1 ? !even : even);
            M::wait(even);
            meet();
        }
    }
    mid_wait<0>();                                              // (the look-ahead of the last steps has landed)
}

// EX - 8-bit activations (Q8_K blocks): what the matrix cores add up over a wave's 128 k of a super-block are whole numbers, and exact. B = the 8-bit values as F16, A = quant x 6-bit sub-block
// scale as F16; an f32 accumulator holds whole numbers up to 2^24. Q4_K: at most 945 x 127 x 128, one accumulator. Q5_K: 1953 x 127 x 64 fits, so one accumulator per 64 k, added at the end;
// Q6_K: products of up to 4096 as 64 x hi + lo, two products with an accumulator each (64 x 127 x 128 at most). Their sum is rounded once on its way to f32, as an int32 sum is when it becomes
// one. It is then multiplied by d of the row and d of the token and added in f32, the minima (one product: 16 group sums x minima, exact) by dmin. mmq_i8.hip and mmq_rows.hip do this for all
// 256 k of a super-block at once: here the halves of a super-block meet as f32. Against an integer GEMM: scales per 32 k applied to int32 results cost as much vector work as the products
// take, and scales inside 8-bit operands two products per sub-block (mmq_big.hip); here scale and quant share the multiply that the F16 form needs anyway.
// Bound by the LDS-DMA like the F16 form, by the vector work at a super-block's end (3 x 16 instructions per 32 tokens) and, Q6_K, by twice the products; two sets of accumulators beside the
// running sums leave room for 64 tokens per workgroup, one set and loaders for 96, one set for 128. 8B shape, 147 tokens, us in tiles of 128 / 96 tokens: ffn_gate | ffn_up 112 / 86, wo and ffn_down
// 32.5 / 25.7, wq | wk | wv 31.5 / 24.9; Q6_K ffn_down without loaders / with 84 / 78; wq | wk | wv with a Q6_K wv 53. (Six passes of 28 on mmq_i8.hip: ffn_gate | ffn_up 26.6 each, ffn_down 35.) (Q6_K's product and its remainder in ONE accumulator, 128 tokens: 148 and 84, and sums beyond 2^24 rounded 16 times.)
// Distance from 64 bits (2-norm, normal weights) of mmq_i8.hip / this form: Q4_K 4096 x 4096 1.20e-7 / 0.89e-7, x 14336 1.33e-7 / 1.06e-7, Q5_K 1.20e-7 / 0.88e-7, Q6_K 4096 x 14336 0.81e-7 / 0.79e-7,
// 8192 x 28672 0.92e-7 / 0.86e-7 (running sums over all of a slice's super-blocks: 1.43e-7; minima of a whole super-block by either half in turn: Q4_K x 14336 1.84e-7).
template <int TYPE, int NT, bool EX, bool SELF>
__device__ __forceinline__ void mid_body(const PfP & p, const PfJob & jb, const int n0, const int t0, uint8_t * smem, const int role, const int ks, const int S, const int tile_id) {
    constexpr int HB = NT * 32 * 128, BBUF = 2 * HB;           // activations: 32 NT tokens x 64 halfs, two of them per step
    constexpr int SLOT = mid_slot<TYPE>(), AG = mid_group_bytes<TYPE, EX>(), NH = (NT + 1) / 2, AHEAD = mid_ahead<TYPE, EX>(), HDR = (AHEAD + 1) * SLOT, XTRA = HDR + 2048;
    constexpr int XS = 3 * BBUF + 4 * AG, XSUM = mid_sum_bytes<TYPE, NT>(), XB = XSUM + NT * 32 * 4;      // EX: sums and scales
    constexpr bool K45 = TYPE == PM_Q4_K || TYPE == PM_Q5_K, Q8 = TYPE == PM_Q8_0;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = wave & 3, kk = wave >> 2;       // (waves w and w + 4 share a SIMD)
    const int r = lane & 31, h = lane >> 5;
    const int K = p.K, nsteps = K / 128, nb = (K + 255) / 256;  // (Q8_0 rows may end on half a super-block: one step)
    uint8_t * const ag = smem + 3 * BBUF + g * AG;              // the row group's weights: slots of the steps in turn, header of super-block b % 4
    const uint32_t lds0 = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) uint8_t *) smem;
    const int nw = n0 + 32 * (role ? g & 1 : g);                // first row of this wave
    // split K: slice ks of S takes the super-blocks [b0, b1)
    const int b0 = (int) ((long) ks * nb / S), b1 = (int) ((long) (ks + 1) * nb / S);
    // the waves meet; what they wrote to LDS, and what a loader waited for, is there
    auto meet = [&] __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (!SELF && wave >= 8) {
        mid_load<TYPE, NT, EX>(p, jb, n0, t0, lds0, role, b0, b1, wave - 8, lane);
        meet(); meet(); meet();                                 // the ones behind the loop below
        if (S == 1 && role) meet();
        return;
    }
    const uint32_t boff0 = (uint32_t) (kk * HB + r * 128 + ((h ^ ((r >> 1) & 7)) << 4));
    const uint32_t aoff = (uint32_t) (r * 16 + 8 * h);
    // SELF: requests of the first half's waves for the weights of their rows, of the second half's for the activations, a quarter of a step's behind each slice's products
    struct Own { MidWeights<TYPE, NT, EX, 1> w; MidActs<TYPE, NT, EX, 4> x; };
    struct None {};
    std::conditional_t<SELF, Own, None> own_rq;
    auto request = [&](int s, bool even, int u) __attribute__((always_inline)) {
        if constexpr (SELF) {
            constexpr int Q = decltype(own_rq.x)::NQ / 4, AHEAD = decltype(own_rq.w)::AHEAD;
            if (kk) { if (EX && even && u == 0) own_rq.x.issue_x((s >> 1) + 1); own_rq.x.issue(s + 2, Q * u, Q * u + Q); } else own_rq.w.issue(s + AHEAD, AHEAD & 1 ? !even : even, u);
        }
    };
    // the end of a step: the next one's operands are there (a loader waited for them, or this wave), this wave's LDS reads are through
    auto settle = [&](bool even) __attribute__((always_inline)) {
        if constexpr (SELF) { if (kk) { own_rq.x.wait(even); own_rq.x.turn(); } else { own_rq.w.wait(even); own_rq.w.turn(); } }
        meet();
    };
    if constexpr (SELF) {
        if (kk) {
            own_rq.x.init(p, t0, g, lds0, lane);
            if (EX) own_rq.x.issue_x(b0);
            own_rq.x.issue(2 * b0, 0, 2 * NT); own_rq.x.turn();
            own_rq.x.issue(2 * b0 + 1, 0, 2 * NT);
        } else {
            own_rq.w.init(p, jb, n0, g, role ? g & 1 : g, lds0, lane);
#pragma unroll
            for (int w = 0; w < AHEAD; ++w) {
#pragma unroll
                for (int u = 0; u < 4; ++u) own_rq.w.issue(2 * b0 + w, (w & 1) == 0, u);
                if (w + 1 < AHEAD) own_rq.w.turn();
            }
        }
    }

    float16v acc[NT];
#pragma unroll
    for (int jt = 0; jt < NT; ++jt)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[jt][e] = 0.0f;
    constexpr bool TWO = EX && (TYPE == PM_Q5_K || TYPE == PM_Q6_K);
    static_assert(!TWO || NT == 2, "three sets of accumulators: 64 tokens, or registers spill");
    constexpr bool SUMS = EX && NT == 2;                         // (registers left: running sums of four super-blocks, and those of them)
    float16v run[EX ? NT : 1], ac2[TWO ? NT : 1], tot[SUMS ? NT : 1];
    const float16v zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (EX)
#pragma unroll
        for (int jt = 0; jt < NT; ++jt)
#pragma unroll
            for (int e = 0; e < 16; ++e) { run[jt][e] = 0.0f; if (SUMS) tot[jt][e] = 0.0f; }
    // the 4 slices of this wave's half of the step in buffer bb / slot sl: 128-k half mm of super-block b
    // (addresses that a step or a super-block's end forms anew instead of keeping them in registers, which then spill)
    auto anew = [](uint32_t v) __attribute__((always_inline)) { if (EX && !SELF) asm volatile("" : "+v"(v)); return v; };
    auto multiply = [&](int b, int mm, uint32_t bb, uint32_t sl) __attribute__((always_inline)) {
        const uint32_t bo = anew(boff0);
        half8 bf[2][NT], af[2], al[2];
        auto read_B = [&](int j) __attribute__((always_inline)) {
#pragma unroll
            for (int jt = 0; jt < NT; ++jt) bf[j & 1][jt] = *(const half8 *) (smem + bb + jt * 4096 + (bo ^ (uint32_t) (j << 5)));
        };
        u32x4 hd = {0, 0, 0, 0};
        uint16_t d6 = 0;
        const uint8_t * hp = ag + HDR + (b & 3) * 512 + r * 16;
        if (K45) hd = *(const u32x4 *) hp;
        else hd[0] = *(const uint32_t *) (hp + (2 * mm + kk) * 4);                            // the 4 scales (Q6_K), the 2 d's (Q8_0) of this wave's 64 k
        if (TYPE == PM_Q6_K) d6 = *(const uint16_t *) (ag + XTRA + ((b >> 3) & 1) * 512 + r * 16 + (b & 7) * 2);
        const uint8_t * ap = ag + sl + aoff;
        u32x2 ql[4], qh[2] = {{0, 0}, {0, 0}};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (Q8) ql[j] = *(const u32x2 *) (ap + kk * 2048 + (j & 1) * 1024 + (j >> 1) * 512);
            else if (K45) { if (j < 2) ql[j] = *(const u32x2 *) (ap + j * 1024 + kk * 512); else ql[j] = ql[j - 2]; }   // (slices 2, 3: the high nibbles)
            else ql[j] = *(const u32x2 *) (ap + (j >> 1) * 1024 + (j & 1) * 512);
        }
        if (TYPE == PM_Q5_K)
#pragma unroll
            for (int v = 0; v < 2; ++v) qh[v] = *(const u32x2 *) (ag + XTRA + (b & 3) * 1024 + v * 512 + aoff);
        if (TYPE == PM_Q6_K)
#pragma unroll
            for (int v = 0; v < 2; ++v) qh[v] = *(const u32x2 *) (ap + 2048 + v * 512);
        half2v mul = {0, 0}, add = {0, 0};
        auto operand = [&](int j) __attribute__((always_inline)) {
            if (K45 && (j & 1) == 0) {
                const int sh = 8 * (2 * kk + (j >> 1));                                       // 32-weight sub-block 4 mm + 2 kk + j / 2
                const uint32_t a = hd[1] >> sh, m = hd[2] >> sh, c = hd[3] >> sh;
                const int sc = (int) (mm ? (c & 0x0Fu) | ((a & 0xC0u) >> 2) : a & 63u), mn = (int) (mm ? ((c >> 4) & 0x0Fu) | ((m & 0xC0u) >> 2) : m & 63u);
                if (EX) mul = half2v{(_Float16) sc, (_Float16) sc};
                else {
                const _Float16 ds = (_Float16) (h2f((uint16_t) (hd[0] & 0xFFFF)) * (float) sc), ms = (_Float16) (h2f((uint16_t) (hd[0] >> 16)) * (float) mn);
                mul = half2v{ds, ds}; add = half2v{(_Float16) -ms, (_Float16) -ms};
                }
            } else if (TYPE == PM_Q6_K) {
                const int sc = (int) (int8_t) (hd[0] >> (8 * j));
                const _Float16 dd = EX ? (_Float16) sc : (_Float16) (h2f(d6) * (float) sc);
                mul = half2v{dd, dd};
            } else if (Q8 && (j & 1) == 0) {
                const _Float16 dd = __builtin_bit_cast(_Float16, (uint16_t) (hd[0] >> (16 * (j >> 1))));
                mul = half2v{dd, dd};
            }
            if constexpr (EX && TYPE == PM_Q6_K) af[j & 1] = pf_dequant<TYPE>(ql[j], qh[j & 1], mm, kk, j, mul, add, &al[j & 1]);
            else af[j & 1] = pf_dequant<TYPE>(ql[j], qh[j & 1], mm, kk, j, mul, add);
        };
        read_B(0);
        operand(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j < 3) { read_B(j + 1); operand(j + 1); }
#pragma unroll
            for (int jt = 0; jt < NT; ++jt) {
                if constexpr (TWO && TYPE == PM_Q5_K) {
                    if (mm) ac2[jt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[j & 1], bf[j & 1][jt], j ? ac2[jt] : zero, 0, 0, 0);
                    else    acc[jt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[j & 1], bf[j & 1][jt], j ? acc[jt] : zero, 0, 0, 0);
                } else acc[jt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[j & 1], bf[j & 1][jt], EX && mm + j == 0 ? zero : acc[jt], 0, 0, 0);
            }
            if constexpr (TWO && TYPE == PM_Q6_K)
#pragma unroll
                for (int jt = 0; jt < NT; ++jt) ac2[jt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[j & 1], bf[j & 1][jt], mm + j == 0 ? zero : ac2[jt], 0, 0, 0);
            request(2 * b + mm, mm == 0, j);
        }
    };
    // EX: the whole numbers of super-block b (this wave's half of its k, and the minima of that half: without them the halves' sums are twice as large, and their roundings) onto the running sums
    auto fold = [&](int b) __attribute__((always_inline)) {
        const uint32_t ln = anew((uint32_t) lane), r = ln & 31, h = ln >> 5;
        const uint8_t * const xs = smem + XS + (b & 1) * XB + r * 32 + 16 * h, * const xd = smem + XS + (b & 1) * XB + XSUM + r * 4;
        const uint8_t * const gh = ag + HDR + (b & 3) * 512 + h * 64, * const gd = ag + XTRA + ((b >> 3) & 1) * 512 + h * 64 + (b & 7) * 2;      // the half's first row
        uint32_t dd[16];                                        // d, dmin of the rows (F16)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int row = (e & 3) + 8 * (e >> 2);
            if (K45) dd[e] = *(const uint32_t *) (gh + row * 16);
            else dd[e] = *(const uint16_t *) (gd + row * 16);
        }
        auto d = [&](int e) __attribute__((always_inline)) { return h2f((uint16_t) dd[e]); };
        auto dm = [&](int e) __attribute__((always_inline)) { return h2f((uint16_t) (dd[e] >> 16)); };
        half8 mo = {0, 0, 0, 0, 0, 0, 0, 0};
        if (K45) {                                              // minima of the row's sub-blocks 4 h .. 4 h + 3, each for two groups of 16: 4 h + 2 kk, + 1 are this half's
            const u32x4 hd = *(const u32x4 *) (ag + HDR + (b & 3) * 512 + r * 16);
            const uint32_t m = h ? ((hd[3] >> 4) & 0x0F0F0F0Fu) | ((hd[2] & 0xC0C0C0C0u) >> 2) : hd[2] & 0x3F3F3F3Fu;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const _Float16 v = (_Float16) (int) ((m >> (16 * kk + 8 * (i >> 1))) & 63u);
                mo[i] = kk ? (_Float16) 0.0f : v; mo[4 + i] = kk ? v : (_Float16) 0.0f;
            }
        }
#pragma unroll
        for (int jt = 0; jt < NT; ++jt) {
            if (NT == 4) __builtin_amdgcn_sched_barrier(0);     // (the minima of all four token tiles at once: registers spill)
            const float da = *(const float *) (xd + 128 * jt);
            if constexpr (TWO)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[jt][e] = TYPE == PM_Q6_K ? fmaf(64.0f, acc[jt][e], ac2[jt][e]) : acc[jt][e] + ac2[jt][e];
            if (K45) {
                const float16v am = __builtin_amdgcn_mfma_f32_32x32x16_f16(mo, *(const half8 *) (xs + 1024 * jt), zero, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 16; ++e) run[jt][e] = fmaf(da, fmaf(-dm(e), am[e], d(e) * acc[jt][e]), run[jt][e]);
            } else {
#pragma unroll
                for (int e = 0; e < 16; ++e) run[jt][e] = fmaf(da, d(e) * acc[jt][e], run[jt][e]);
            }
        }
    };

    uint32_t bb = 0, sl = 0;                                    // buffer and slot of the step
    auto turn = [&] __attribute__((always_inline)) { bb = bb == 2 * BBUF ? 0 : bb + BBUF; sl = sl == AHEAD * SLOT ? 0 : sl + SLOT; };
    settle(false);
    for (int b = b0; b < b1; ++b) {
        multiply(b, 0, bb, sl);
        settle(true);
        turn();
        if (Q8 && 2 * b + 1 >= nsteps) break;
        multiply(b, 1, bb, sl);
        if constexpr (EX) fold(b);
        if constexpr (SUMS)
            if (((b - b0) & 3) == 3)
#pragma unroll
                for (int jt = 0; jt < NT; ++jt) {
                    tot[jt] += run[jt]; run[jt] = zero;
                }
        settle(false);
        turn();
    }
    if constexpr (SELF) mid_wait<0>();
    if constexpr (EX)
#pragma unroll
        for (int jt = 0; jt < NT; ++jt) {
            acc[jt] = run[jt];
            if constexpr (SUMS) acc[jt] += tot[jt];
        }
    meet();                                                     // (the loaders: their look-ahead has landed)
    // ---- the two halves of K: every wave keeps its rows' sub-tiles of 32 tokens NH kk, .. (NT = 3: two and one) and takes the partner's sums of them
    f32x4 * const xl = (f32x4 *) smem;
    float16v own[NH];
#pragma unroll
    for (int i = 0; i < NH; ++i) {
        constexpr int LAST = NT - 1;
        if (kk || NH + i < NT) {
            const float16v give = kk ? acc[i] : acc[NH + i < NT ? NH + i : LAST];
#pragma unroll
            for (int q = 0; q < 4; ++q) xl[((wave * NH + i) * 4 + q) * 64 + lane] = f32x4{give[4 * q], give[4 * q + 1], give[4 * q + 2], give[4 * q + 3]};
        }
        own[i] = kk ? acc[NH + i < NT ? NH + i : LAST] : acc[i];
    }
    meet();
#pragma unroll
    for (int i = 0; i < NH; ++i)
        if (!kk || NH + i < NT)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 o = xl[(((wave ^ 4) * NH + i) * 4 + q) * 64 + lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) own[i][4 * q + e] += o[e];
            }
    meet();
    // ---- split K: slabs, as above
    if (S > 1) {
        f32x4 * const mine = (f32x4 *) p.ws + (size_t) (tile_id * S + ks) * (8 * NH * 4 * 64);
#pragma unroll
        for (int i = 0; i < NH; ++i) {
            if (kk && NH + i >= NT) break;
            f32x4 o[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) o[q] = f32x4{own[i][4 * q], own[i][4 * q + 1], own[i][4 * q + 2], own[i][4 * q + 3]};
            store_slab(o, smem + wave * (32 * 144), mine + (wave * NH + i) * 256, lane);
        }
        return;
    }
    // ---- pair tiles: the gate waves park their sums in LDS (same lane, same register index as the up wave that needs them)
    if (role) {
        if (role == 1) {
#pragma unroll
            for (int i = 0; i < NH; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) xl[(((2 * kk + (g & 1)) * NH + i) * 4 + q) * 64 + lane] = f32x4{own[i][4 * q], own[i][4 * q + 1], own[i][4 * q + 2], own[i][4 * q + 3]};
        }
        meet();
        if (role == 1) return;
#pragma unroll
        for (int i = 0; i < NH; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 gg = xl[(((2 * kk + (g & 1)) * NH + i) * 4 + q) * 64 + lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) own[i][4 * q + e] *= gg[e] / (1.0f + expf(-gg[e]));
            }
    }
    // ---- epilogue: C[row = (e & 3) + 8 (e >> 2) + 4 h][token = r] crosses a wave-private LDS tile [token][32 rows + 4]; 8 lanes then hold a token's 32 rows
    uint8_t * const xe = smem + 8 * NH * 4096 + wave * (32 * 144);
#pragma unroll
    for (int i = 0; i < NH; ++i) {
        if (kk && NH + i >= NT) break;
#pragma unroll
        for (int q = 0; q < 4; ++q) *(f32x4 *) (xe + r * 144 + (8 * q + 4 * h) * 4) = f32x4{own[i][4 * q], own[i][4 * q + 1], own[i][4 * q + 2], own[i][4 * q + 3]};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int tr = 8 * q + (lane >> 3), t = t0 + 32 * (kk * NH + i) + tr, n = nw + (lane & 7) * 4;
            f32x4 v = *(const f32x4 *) (xe + tr * 144 + (lane & 7) * 16);
            if (t >= p.T || n >= jb.N) continue;                // (N is a multiple of 4)
            const long o = (long) t * jb.ldy + n;
            if (jb.bias) v += ld_g((const f32x4 *) (jb.bias + n));
            if (jb.resid) v += ld_g((const f32x4 *) (jb.resid + o));
            if (jb.silu_gate) {
                const f32x4 gg = ld_g((const f32x4 *) (jb.silu_gate + o));
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] *= gg[e] / (1.0f + expf(-gg[e]));
            }
            if (jb.Yh) *(PM_G half4v *) (jb.Yh + o) = half4v{(_Float16) v[0], (_Float16) v[1], (_Float16) v[2], (_Float16) v[3]};
            else *(PM_G f32x4 *) (jb.Y + o) = v;
        }
    }
}

// block id -> (row tile, token tile): XCD x = id % 8 takes the row tiles x, x + 8, ..; its consecutive slots sweep the token tiles of one row tile, so the
// workgroups that run together on an XCD share a few row tiles of weights and the activation k-slices in its L2 (mmq_big.hip's mapping)
// PF_CUT (a bit of EXP): the batch's last tile of 256 tokens multiplies the 128 or 192 that are left of it only. us, whole / cut: wo of the 8B shape 640 tokens 50.5 / 47.4, 1400 76.8 / 75.7, 2100 113 / 114
// (in tiles of 192 93), its Q6_K ffn_down 640 114 / 107, 1400 229 / 218, ffn_gate | ffn_up 640 189 / 181, 1800 478 / 471, Q8_0 ffn_down of 72B 640 374 / 345. (Tiles of 192 with a cut last one: wo 2400
// 105 / 110, wq | wk | wv 6001 360 / 379.) A kernel of its own: with the two smaller bodies beside it a launch that cuts nothing took 0.2-0.9 us more (200 tokens of 1024 x 1024 34.2 -> 34.8, Q8_0
// 33.8 -> 34.8; now 33.6, 33.7). Where it is taken: cut_pays. The kernel that cuts nothing has no such choice in its source either: with one of a single body the compiler laid its blocks out otherwise, Q8_0 256 tokens of 512 values
// x 4096 rows 26.9 -> 27.4, of 1024 x 16384 39.0 -> 40.4
constexpr int PF_CUT = 256;
template <int TA, int TB, int NT, bool MID = false, int EXP = 0, bool EX = false>
__global__ __launch_bounds__((MID && !mid_self<TA, TB, NT, EX, EXP>() ? MID_NTHR : PF_NTHR)) void gemm_pf_kernel(PfP p) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t pf_smem[];
    const int id = (int) blockIdx.x, x = id & 7;
    // slots [0, full) of an XCD run whole tiles; the slots behind them are split S ways along K, the slices of a tile neighbours on one XCD.
    // full = 0: every tile split (S = 1: none)
    const int q = id >> 3;
    const int S = q < p.full ? 1 : p.splitk;
    const int ks = q < p.full ? 0 : (q - p.full) % p.splitk, slot = q < p.full ? q : p.full + (q - p.full) / p.splitk;
    const int per_x = (p.nt_n + 7 - x) >> 3;
    if (slot >= per_x * p.nt_t) return;
    const int tile_n = x + 8 * (slot / p.nt_t), tile_t = slot % p.nt_t;
    PfJob jb = p.job[0];                                       // (selected field by field with static indices: a run-time index would put the table into scratch)
    int n0, role = 0;
    constexpr int ROWS = MID ? 128 : 256;
    if (p.pair) {                                              // ROWS / 2-row tiles of job 0 (waves 0-3; mid_body: row groups 0, 1) and job 1
        // (of mid_body's loaders wave 10 brings the weights of job 0, wave 11 those of job 1)
        role = 1 + __builtin_amdgcn_readfirstlane((int) (!MID ? threadIdx.x >> 8 : threadIdx.x < 512 ? (threadIdx.x >> 7) & 1 : (threadIdx.x >> 6) & 1));
        if (role == 2) jb = p.job[1];
        n0 = tile_n * (ROWS / 2);
    } else {
#pragma unroll
        for (int q = 1; q < PF_MAX_JOBS; ++q) if (q < p.njobs && tile_n >= p.job[q].tile0) jb = p.job[q];
        n0 = (tile_n - jb.tile0) * ROWS;
    }
    const int t0 = tile_t * 32 * NT;
    const int tile_id = (slot - p.full) * 8 + x;                 // (split tiles only: slab index)
    if constexpr (!MID && (EXP & PF_CUT)) {
        static_assert(NT == 8, "tiles of 256 tokens");
        auto body = [&](auto nt) __attribute__((always_inline)) {
            constexpr int N = decltype(nt)::value;
            if (TA == TB || jb.type == TA) pf_body<TA, N, EXP & 255, NT>(p, jb, n0, t0, pf_smem, role, ks, S, tile_id);
            else pf_body<TB, N, EXP & 255, NT>(p, jb, n0, t0, pf_smem, role, ks, S, tile_id);
        };
        const int left = p.T - t0;
        if (left <= 128) body(std::integral_constant<int, 4>());
        else if (left <= 192) body(std::integral_constant<int, 6>());
        else body(std::integral_constant<int, 8>());
    } else if constexpr (!MID) {
        if (TA == TB || jb.type == TA) pf_body<TA, NT, EXP, NT>(p, jb, n0, t0, pf_smem, role, ks, S, tile_id);
        else pf_body<TB, NT, EXP, NT>(p, jb, n0, t0, pf_smem, role, ks, S, tile_id);
    } else {
        constexpr bool SELF = mid_self<TA, TB, NT, EX, EXP>();
        if (TA == TB || jb.type == TA) mid_body<TA, NT, EX, SELF>(p, jb, n0, t0, pf_smem, role, ks, S, tile_id);
        else mid_body<TB, NT, EX, SELF>(p, jb, n0, t0, pf_smem, role, ks, S, tile_id);
    }
}

// The slabs of a launch's split tiles, added in slice order, and the epilogue: a wave per 32 rows x 8 tokens, 8 lanes on a token's 32 rows, all S parts on their way at once. Bound by the slabs'
// bytes. A launch of its own because all CUs then share them: the last arriver of a tile (64 of 256 workgroups for 8192 rows x 512 tokens, S = 4) read 1 MB of slabs and stored its tile by
// itself, 48 us behind the last product. us, last arriver (as it was; its loads in fours and the slabs written through) / product + this launch: 512 tokens of 8192 x 8192 Q4_K 107 (102) / 66 + 17,
// 8192 x 28672 264 (245) / 211 + 17, 10240 x 8192 131 (120) / 91 + 15; 101 tokens (mid_body) of 4096 x 4096 23.0 / 18.3 + 4.8, 4096 x 14336 35.9 / 27.7 + 5.9. (A wave per 32 tokens: 18.7 for 16.8 and
// 8.1 for 5.9)
// nt: sub-tiles of 32 tokens in a tile; mid: mid_body's tiles (wave = row group + 4 x token half)
template <int SMAX> __global__ __launch_bounds__(256) void pf_reduce_kernel(PfP p, int mid, int nt, int units) {
    const int u4 = (int) blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), unit = u4 >> 2, k0 = u4 & 3, lane = threadIdx.x & 63;
    if (unit >= units) return;
    const int nti = mid ? (nt + 1) / 2 : nt;                    // sub-tiles of a wave
    const int S = p.splitk, per_tile = (p.pair ? 4 : 8) * nti, tile_id = unit / per_tile, wv = unit % per_tile / nti, i = unit % nti;
    const int x = tile_id & 7, slot = p.full + (tile_id >> 3), per_x = (p.nt_n + 7 - x) >> 3;
    if (slot >= per_x * p.nt_t) return;
    const int tile_n = x + 8 * (slot / p.nt_t), tile_t = slot % p.nt_t;
    PfJob jb = p.job[0];
    int n0 = tile_n * (mid ? 64 : 128), row = wv, half = 0, wave = wv, wave_g = 0;
    if (p.pair) {
        jb = p.job[1];
        if (mid) { row = wv & 1; half = wv >> 1; wave_g = row + 4 * half; wave = wave_g + 2; } else { wave_g = wv; wave = wv + 4; }
    } else {
#pragma unroll
        for (int q = 1; q < PF_MAX_JOBS; ++q) if (q < p.njobs && tile_n >= p.job[q].tile0) jb = p.job[q];
        n0 = (tile_n - jb.tile0) * (mid ? 128 : 256);
        if (mid) { row = wv & 3; half = wv >> 2; }
    }
    if (half * nti + i >= nt) return;
    const int t0 = (tile_t * nt + half * nti + i) * 32 + 8 * k0, t = t0 + (lane >> 3), n = n0 + 32 * row + (lane & 7) * 4;
    if (t0 >= p.T || n >= jb.N) return;                         // (N is a multiple of 4)
    const size_t tile = (size_t) 8 * nti * 256;                 // of f32x4
    const f32x4 * const slab = (const f32x4 *) p.ws + (size_t) tile_id * S * tile + 64 * k0 + lane;
    auto sum = [&](int w) __attribute__((always_inline)) {
        const f32x4 * const at = slab + (size_t) (w * nti + i) * 256;
        f32x4 v[SMAX], o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < SMAX; ++q) v[q] = *(const PM_G f32x4 *) (at + (size_t) (q < S ? q : S - 1) * tile);
#pragma unroll
        for (int q = 0; q < SMAX; ++q) if (q < S) o += v[q];
        return o;
    };
    f32x4 v = sum(wave), gate;
    if (p.pair) gate = sum(wave_g);
    if (t >= p.T) return;
    const long at = (long) t * jb.ldy + n;
    if (p.pair)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= gate[e] / (1.0f + expf(-gate[e]));
    if (jb.bias) v += ld_g((const f32x4 *) (jb.bias + n));
    if (jb.resid) v += ld_g((const f32x4 *) (jb.resid + at));
    if (jb.silu_gate) {
        const f32x4 gg = ld_g((const f32x4 *) (jb.silu_gate + at));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= gg[e] / (1.0f + expf(-gg[e]));
    }
    if (jb.Yh) *(PM_G half4v *) (jb.Yh + at) = half4v{(_Float16) v[0], (_Float16) v[1], (_Float16) v[2], (_Float16) v[3]};
    else *(PM_G f32x4 *) (jb.Y + at) = v;
}

// The same for one matrix of which every tile is split, a workgroup per token, with the RMS norm of the token's new row (rmsnorm_q8k_kernel's expressions in its order, F16): the row does not
// travel to memory and back, and a launch goes. Bound by the slabs. us, both launches / this one: 101 tokens x 4096, S = 4 4.8 + 4.6 / 5.3, S = 8 5.9 + 4.6 / 6.3; 512 x 8192, S = 4 16.8 + 9.9 / 20.8 (28.3
// with 4 waves a token). For up to 512 tokens: beyond, few launches have every tile split
template <int SMAX> __global__ __launch_bounds__(1024) void pf_reduce_norm_kernel(PfP p, int mid, int nt, const float * w, float eps, _Float16 * yh) {
    constexpr int NWV = 16, HOLD = 2;
    __shared__ double red[NWV];
    const int t = blockIdx.x, lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), S = p.splitk;
    const PfJob & jb = p.job[0];
    const int N = jb.N, rows = mid ? 128 : 256, tok = 32 * nt, nti = mid ? (nt + 1) / 2 : nt;
    const int tile_t = t / tok, tt = t % tok / 32, half = mid ? tt / nti : 0, i = mid ? tt % nti : tt;
    const size_t tile = (size_t) 8 * nti * 256;                 // of f32x4
    f32x4 f[HOLD], wt[HOLD];
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < HOLD; ++j) {
        const int n = (wv + NWV * j) * 256 + 4 * lane;
        if (n >= N) continue;
        const int tile_n = n / rows, wave = n % rows / 32 + 4 * half;
        const f32x4 * const at = (const f32x4 *) p.ws + (size_t) (((tile_n >> 3) * p.nt_t + tile_t) * 8 + (tile_n & 7)) * S * tile + (size_t) (wave * nti + i) * 256 + (t & 31) * 8 + (lane & 7);
        f32x4 v[SMAX], o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < SMAX; ++q) v[q] = *(const PM_G f32x4 *) (at + (size_t) (q < S ? q : S - 1) * tile);
        const f32x4 r = jb.resid ? ld_g((const f32x4 *) (jb.resid + (long) t * jb.ldy + n)) : f32x4{0.0f, 0.0f, 0.0f, 0.0f}, b = jb.bias ? ld_g((const f32x4 *) (jb.bias + n)) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        wt[j] = ld_g((const f32x4 *) (w + n));
#pragma unroll
        for (int q = 0; q < SMAX; ++q) if (q < S) o += v[q];
        if (jb.bias) o += b;
        if (jb.resid) o += r;
        f[j] = o;
    }
#pragma unroll
    for (int j = 0; j < HOLD; ++j) {
        const int n = (wv + NWV * j) * 256 + 4 * lane;
        if (n >= N) continue;
        *(PM_G f32x4 *) (jb.Y + (long) t * jb.ldy + n) = f[j];
#pragma unroll
        for (int e = 0; e < 4; ++e) s += (double) (f[j][e] * f[j][e]);
    }
    s = all_sum(s);
    if (lane == 0) red[wv] = s;
    __syncthreads();
    double tot = (red[0] + red[1]) + (red[2] + red[3]);
#pragma unroll
    for (int q = 4; q < NWV; q += 4) tot += (red[q] + red[q + 1]) + (red[q + 2] + red[q + 3]);
    const float scale = 1.0f / sqrtf((float) (tot / N) + eps);
#pragma unroll
    for (int j = 0; j < HOLD; ++j) {
        const int n = (wv + NWV * j) * 256 + 4 * lane;
        if (n >= N) continue;
        const f32x4 v = f[j] * scale * wt[j];
        *(PM_G half4v *) (yh + (size_t) t * N + n) = half4v{(_Float16) v[0], (_Float16) v[1], (_Float16) v[2], (_Float16) v[3]};
    }
}

// The same for wq | wk | wv, with NORM rope (rope_kv_store_kernel's expressions, cos / sin from the pass's table) and the stores of K and V^T into the cache: the launch behind it and two trips of the
// rows go. Bound by the chain of its loads. 101 tokens of 32 + 8 + 8 heads of 128, S = 4: 5.1 + 7.3 us as two launches, 6.4 as this one
template <int SMAX> __global__ __launch_bounds__(1024) void pf_reduce_rope_kernel(PfP p, int mid, int nt, pm_gemm_rope a) {
    constexpr int NWV = 16, HOLD = 3;                           // rows of 256: up to 48
    const int t = blockIdx.x, lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), S = p.splitk;
    const int Nq = p.job[0].N, Nk = p.job[1].N, rows = mid ? 128 : 256, tok = 32 * nt, nti = mid ? (nt + 1) / 2 : nt;
    const int tile_t = t / tok, tt = t % tok / 32, half = mid ? tt / nti : 0, i = mid ? tt % nti : tt;
    const size_t tile = (size_t) 8 * nti * 256;                 // of f32x4
    const int seq = a.seq ? a.seq[a.rows ? t : 0] : 0, pos = a.rows ? a.pos[t] : a.pos[seq] + t;
    uint16_t * const kc = (uint16_t *) a.kc + (long) seq * a.seq_stride + (long) pos * Nk, * const vc = (uint16_t *) a.vc + (long) seq * a.seq_stride + pos;
#pragma unroll
    for (int j = 0; j < HOLD; ++j) {
        const int n0 = (wv + NWV * j) * 256;                    // (a wave's 256 rows are of one matrix)
        if (n0 >= Nq + 2 * Nk) continue;
        const int what = n0 < Nq ? 0 : n0 < Nq + Nk ? 1 : 2, n = n0 - (what == 0 ? 0 : what == 1 ? Nq : Nq + Nk) + 4 * lane;
        const int tile0 = what == 0 ? 0 : what == 1 ? p.job[1].tile0 : p.job[2].tile0;
        const float * const bias = what == 0 ? p.job[0].bias : what == 1 ? p.job[1].bias : p.job[2].bias;
        const int tile_n = tile0 + n / rows, wave = n % rows / 32 + 4 * half, d = n % a.dh;
        const f32x4 * const at = (const f32x4 *) p.ws + (size_t) (((tile_n >> 3) * p.nt_t + tile_t) * 8 + (tile_n & 7)) * S * tile + (size_t) (wave * nti + i) * 256 + (t & 31) * 8 + (lane & 7);
        f32x4 v[SMAX], o = {0.0f, 0.0f, 0.0f, 0.0f}, cs = {1.0f, 0.0f, 1.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < SMAX; ++q) v[q] = *(const PM_G f32x4 *) (at + (size_t) (q < S ? q : S - 1) * tile);
        const f32x4 b = bias ? ld_g((const f32x4 *) (bias + n)) : o;
        if (what < 2 && d < a.n_dims) cs = ld_g((const f32x4 *) (a.tab + (size_t) t * a.n_dims + d));
#pragma unroll
        for (int q = 0; q < SMAX; ++q) if (q < S) o += v[q];
        if (bias) o += b;
        if (what == 2) {
#pragma unroll
            for (int e = 0; e < 4; ++e) vc[(long) (n + e) * a.n_ctx] = f2h(o[e]);
            continue;
        }
        if (d < a.n_dims) o = f32x4{o[0] * cs[0] - o[1] * cs[1], o[0] * cs[1] + o[1] * cs[0], o[2] * cs[2] - o[3] * cs[3], o[2] * cs[3] + o[3] * cs[2]};
        const uint16_t h[4] = {f2h(o[0]), f2h(o[1]), f2h(o[2]), f2h(o[3])};
        if (what == 1) *(PM_G u32x2 *) (kc + n) = u32x2{(uint32_t) h[0] | (uint32_t) h[1] << 16, (uint32_t) h[2] | (uint32_t) h[3] << 16};
        else *(PM_G f32x4 *) (p.job[0].Y + (long) t * Nq + n) = a.round_q ? f32x4{h2f(h[0]), h2f(h[1]), h2f(h[2]), h2f(h[3])} : o;
    }
}

template <int TA, int TB, int NT, bool MID = false, bool EX = false> constexpr size_t pf_lds_bytes() {
    if (!MID) return (size_t) 3 * NT * 32 * 128 + (size_t) 8 * (pf_wave_bytes<TA>() > pf_wave_bytes<TB>() ? pf_wave_bytes<TA>() : pf_wave_bytes<TB>());
    return mid_lds_bytes<TA, NT, EX>() > mid_lds_bytes<TB, NT, EX>() ? mid_lds_bytes<TA, NT, EX>() : mid_lds_bytes<TB, NT, EX>();
}

void pf_allow_lds(const void * kern, size_t lds) {
    struct E { const void * k; int dev; };
    static E done[64]; static int n_done = 0;
    const int dev = pm_cur_dev();
    for (int i = 0; i < n_done && i < 64; ++i) if (done[i].k == kern && done[i].dev == dev) return;
    (void) hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (n_done < 64) { done[n_done].k = kern; done[n_done].dev = dev; ++n_done; }
}

// split-K workspace of a (device, stream): the partial-tile slabs. A product leaves them for the launch behind it, so g_pf_mu is held from here until that one is issued: another host thread's
// product on this stream, or its larger request, comes in front of both launches or behind both
struct PfWs { hipStream_t st; int dev; uint8_t * p; size_t bytes; uint64_t use; };
PfWs g_pf_ws[16] = {};
uint64_t g_pf_tick = 0;
std::mutex g_pf_mu;
uint8_t * pf_workspace(hipStream_t st, size_t need) {
    const int dev = pm_cur_dev();
    PfWs * e = nullptr, * lru = &g_pf_ws[0];
    for (PfWs & c : g_pf_ws) {
        if (c.p && c.st == st && c.dev == dev) { e = &c; break; }
        if (!c.p) lru = &c; else if (lru->p && c.use < lru->use) lru = &c;
    }
    if (e && e->bytes >= need) { e->use = ++g_pf_tick; return e->p; }
    if (!e) e = lru;
    if (e->p) { (void) hipDeviceSynchronize(); (void) hipFree(e->p); e->p = nullptr; e->bytes = 0; }
    need = (need + ((size_t) 32 << 20)) & ~(((size_t) 16 << 20) - 1);     // (grow in steps: a later, larger batch does not reallocate at once)
    if (hipMalloc((void **) &e->p, need) != hipSuccess) { e->p = nullptr; return nullptr; }
    e->st = st; e->dev = dev; e->bytes = need; e->use = ++g_pf_tick;
    return e->p;
}

} // namespace

bool pm_gemm_pf_enabled() {
    static const int force = [] { const char * e = getenv("PM355_GEMM_KERNEL"); return e ? atoi(e) : 0; }();
    return force == 0 || force == 3;
}

// 0 when pm_launch_gemm_pf serves (type, K, N, T)
int pm_gemm_pf_check(int type, int K, int N, int T) {
    if (type != PM_Q4_K && type != PM_Q5_K && type != PM_Q6_K && type != PM_Q8_0) return -1;
    if ((type == PM_Q8_0 ? K % 128 : K % 256) || K < 512 || N < 1 || N % 4 || T < 1) return -2;
    if (type == PM_Q6_K && PM_Q6K_SCD) return -2;               // (the d's travel as 16-byte pieces = 8 super-blocks of the separate-stream row tail)
    if ((size_t) T * (size_t) K * 2 >= ((size_t) 1 << 32) || (size_t) N * pm_weight_row_stride(type, K) >= ((size_t) 1 << 32)) return -2;   // 32-bit lane offsets
    return 0;
}

// The launch geometry of `tiles` row tiles (256 rows, 128 where mid_body runs; pair launches: half of that of each matrix) x T tokens over K on a device of `cus` CUs in 8 XCDs - host
// arithmetic only (tests/test_gemm_plan.py plans the layer shapes without a device). nt: 32-token sub-tiles per workgroup tile (2, 3, 4, 6, 8 = 64, 96, 128, 192, 256 tokens: a dequantized
// operand serves nt MFMAs). Few tiles - wo / ffn_down / wq | wk | wv at the
// reference's default n_ubatch 512 (common/common.h:178) are 64-80 tiles for 256 CUs - are split along K: S slices per tile, the slice count that minimises
// rounds of workgroups x (super-blocks per slice + ~3 for prologue, slab traffic and the launch that adds the slices up). A launch of R full rounds + a short tail (wq | wk | wv
// at 2048 tokens: 320 tiles = 256 + 64; Qwen2.5-72B's ffn_gate | ffn_up: 1848 = 7 x 256 + 56) runs whole tiles in the full rounds and splits ONLY the tail's
// tiles - as many slices as fill the idle CUs of the last round (`full` whole-tile slots per XCD come first in the grid). Splitting every tile instead sends
// every partial tile through memory: 3 x 320 slabs of 256 KB for the qkv launch, 501 us = 685 TFLOP/s against 406 us = 846.
static void plan_tiles(int tiles, int K, int T, int cus, int nt, int force_s, int allow_mixed, pm_gemm_pf_plan_t * out) {
    const int nt_t = (T + 32 * nt - 1) / (32 * nt);
    const long wgs = (long) tiles * nt_t;
    const int nb = (K + 255) / 256;
    if (cus < 8) cus = 8;
    int S = 1, full = 0;
    const int minL = (tiles / 8) * nt_t, maxL = ((tiles + 7) / 8) * nt_t, cpx = cus / 8;      // per-XCD slot counts (XCD x owns the row tiles x, x + 8, ..)
    double best = (double) ((wgs + cus - 1) / cus) * nb;
    for (int q = 2; q <= 8; ++q) {
        if (nb / q < 4 || wgs * q > 16384) break;               // (slabs of 256 KB: 4 GB at most)
        const double c = (double) ((wgs * q + cus - 1) / cus) * ((double) nb / q + 3.0);
        if (c < best * 0.97) { best = c; S = q; }
    }
    const int F = (minL / cpx) * cpx, rem = maxL - F;
    if (allow_mixed && !(force_s >= 1 && force_s <= 8) && F > 0 && rem > 0 && 2 * rem <= cpx) {
        int q = cpx / rem; if (q > 8) q = 8;
        while (q >= 2 && nb / q < 4) --q;
        if (q >= 2) {
            const double c = (double) (F / cpx) * nb + ((double) nb / q + 3.0);
            if (c < best * 0.97) { best = c; S = q; full = F; }
        }
    }
    if (force_s >= 1 && force_s <= 8 && nb / force_s >= 1) { S = force_s; full = 0; }
    out->nt = nt; out->nt_t = nt_t; out->splitk = S; out->full = full; out->grid = 8 * (full + (maxL - full) * S); out->cost = best;
}
// Does a launch whose last tile of 256 tokens is cut gain by it? It saves that tile's part of the steps; what it costs is the same for any K, some 7 us a round of workgroups: two loops of tens of KB
// side by side do not fit the instruction cache that two CUs share. us, whole / cut, by K x sub-tiles saved of 9 / token tiles: 19 (25600 rows of 1024, 3000 tokens) 260 / 294, 76 (8448 of 4096, 3000)
// 243 / 254, 114 (16384 of 1024, 777) 57.0 / 56.5, 152 (8448 of 2048, 1400) 78 / 81, 202 (2100 tokens, 14336 of 4096) 281 / 285, (12800) 261 / 267, 228 (16384 of 2048, 400) 62 / 58, (14336 of 4096, 900)
// 131 / 131, 303 (14336 of 4096, 1400) 206 / 203, 364 (1100) 178 / 172. Where every tile is split along K a cut one has smaller slabs too: 0.89-1.01
static bool cut_pays(int K, int T, int S, int full) {
    const int n = (T + 255) / 256, left = T - 256 * (n - 1), saved = left <= 128 ? 4 : left <= 192 ? 2 : 0;
    return saved && (n == 1 || (S > 1 && !full) || (long) saved * K > 215L * 9 * n);
}
void pm_gemm_pf_plan(const pm_gemm_pf_ask & ask, pm_gemm_pf_plan_t * out) {
    const int tiles = ask.tiles, K = ask.K, T = ask.T, cus = ask.cus, nb = (K + 255) / 256;
    const bool mid = ask.form == PM_PF_ROWS_128, wide = ask.form == PM_PF_WIDE;
    const int nt0 = T <= 64 || ask.form == PM_PF_WIDE_TWO ? 2 : T <= 96 && (mid || wide) ? 3 : T <= 128 || mid || wide ? 4 : 8;
    plan_tiles(tiles, K, T, cus, ask.nt ? ask.nt : nt0, ask.splitk, ask.mixed, out);
    if (ask.nt) return;
    // 8-bit activations of Q4_K: tiles of 96 tokens (with loaders) where they cost less than those of 128 (without: no registers left for them), by rounds of workgroups; the K split stays that of
    // 128 tokens: the sums in one order. 8B shape, whole passes, us, 128 / 96: 79 tokens 716 / 675, 109 738 / 801, 147 935 / 858, 231 1025 / 1095, 316 1279 / 1260, 459 1498 / 1570
    if (wide && T > 64 && !out->full && (T + 95) / 96 * 96 <= ask.ldt) {
        // (rounds of the XCD with the most row tiles. Counted over the chip: 83 row tiles of 2048 values, 231 tokens 31.6 / 45.2, 18 of 4096 27.6 / 36.1, 99 of 8192, 385 tokens 190 / 210 - and 128 where 96 are
        // faster: 84 of 8192, 300 tokens 186 / 141)
        const int cpx = cus / 8;
        const auto cost = [&](int nt) { return ((long) ((tiles + 7) / 8) * ((T + 32 * nt - 1) / (32 * nt)) * out->splitk + cpx - 1) / cpx * (nt + 1); };
        if (cost(3) < cost(4)) plan_tiles(tiles, K, T, cus, 3, out->splitk, 0, out);
    }
    // Tiles of 192 tokens where their rounds of workgroups cost less than those of 256: mostly 129..192, 257..384 and 513..576 tokens, whose rest of a tile of 256 was products of nothing. The K
    // split stays, so every sum keeps its order; in place of a split of the last tiles only, whole ones. Both by full rounds and, as a last round that is not full runs faster, by the work in them, which
    // counts what a cut last tile of 256 leaves out: one round of 256-token workgroups that leaves CUs idle may become up to a tenth more work, as many tiles as much (257..384), others have to save some.
    // us, 256 with the last tile cut / 192: 8B shape ffn_gate | ffn_up Q4_K 150 tokens 64 / 62, 300 110 / 97 (512 129 / 147, 1000 251 / 280, 6001 1425 / 1455: not taken), 70B shape 300 377 / 339, 513
    // 596 / 508, Q6_K ffn_down of 8B 380 74 / 69, Q8_0 ffn_down of 72B 513 319 / 297, wq | wk | wv of 8B 150 36.2 / 34.6, 1500 105 / 93, 6001 379 / 335 (a split tail before), wo 3000 129 / 115, 6001 259 / 226;
    // 33 products of 257..384 tokens and more than a round 0.73-0.97, one 1.01. As much work in more tiles, not taken: 5120 x 13824 pairs 1344 tokens 421 / 450, 8192 x 29568 2112 1871 / 1809
    if (ask.form == PM_PF_ROWS_256 && !ask.splitk && out->nt == 8) {
        const int s6 = out->full ? 1 : out->splitk;
        // rounds of workgroups and work in them, in sub-tiles of 32 tokens + 1; the rounds are those of the XCD with the most row tiles. Counted over the chip, launches whose row tiles do not
        // divide by eight took a round more than with tiles of 256. us, 256 / 192: 1024 rows of 8192, 777 tokens 53 / 62, 2304 of 4096, 4096 tokens 135 / 172, 4352 of 4096, 2100 tokens 115 / 166
        struct Cost { double rounds, work; bool one; };
        const auto cost = [&](int nt) {
            const int n = (T - 1) / (32 * nt), left = T - 32 * nt * n, last = nt == 6 || !n || !cut_pays(K, T, s6, out->full) ? nt : left <= 128 ? 4 : 6;
            const double w = (double) tiles * s6 / cus, x = (double) ((tiles + 7) / 8) * s6 / (cus / 8);
            return Cost{std::ceil(x * (n + 1)) * (nt + 1), w * (n * (nt + 1) + last + 1), w * (n + 1) <= 1.0};
        };
        const Cost c6 = cost(6);
        Cost c8 = cost(8);
        if (out->full) { c8.rounds = c8.work = 9.0 * out->cost / nb; c8.one = false; }
        const double most = c8.one ? 1.1 : !out->full && (T + 191) / 192 == out->nt_t ? 1.001 : 0.97;
        if (c6.rounds < 0.97 * c8.rounds && c6.work < most * c8.work) plan_tiles(tiles, K, T, cus, 6, s6, 0, out);
    }
}

// One launch over njobs <= 4 matrices that share the F16 activations xh [T][K]. Job j: Y_j[t][n] (f32, token stride ldy_j) or Yh_j (F16) =
// W_j . x (+bias)(+resid)(x silu(gate)). 0, or -1 type / -2 shape
int pm_launch_gemm_pf(const pm_gemm_pf_job * jobs, int njobs, const void * xh, int K, int T, hipStream_t st) { return pm_launch_gemm_pf_ex(jobs, njobs, xh, K, T, 0, st); }

// pair != 0: jobs[0] = ffn_gate, jobs[1] = ffn_up (same type, same N; jobs[0]'s outputs are ignored): jobs[1]'s output = silu(W0 . x) * (W1 . x) (+ its own bias / resid
// before the product are NOT applied to the gate). One launch, the gate result stays on the chip.
static int launch_pf(const pm_gemm_pf_job * jobs, int njobs, const void * xh, const pm_q8k_wide * wide, int K, int T, int pair, hipStream_t st, pm_gemm_norm * norm = nullptr, pm_gemm_rope * rope = nullptr) {
    if (njobs < 1 || njobs > PF_MAX_JOBS || !jobs || !xh) return -2;
    if (pair && (njobs != 2 || jobs[0].type != jobs[1].type || jobs[0].N != jobs[1].N || jobs[0].bias || jobs[0].resid || jobs[1].silu_gate)) return -2;
    static const int force_nt = [] { const char * e = getenv("PM355_GEMM_PF_NT"); return e ? atoi(e) : 0; }();
    const int asked_nt = force_nt == 2 || force_nt == 4 || force_nt == 6 || force_nt == 8 ? force_nt : 0;      // (what the 256-row tiles have kernels for)
    const int cus = pm_device_cus();
    // mid_body for up to 128 tokens where its 128-row tiles are one round of workgroups: there a launch is its fixed costs and its K split. us, pf_body / mid_body, Q4_K: 4096 x 4096
    // 101 tokens 28.9 / 22.0, 4096 x 14336 50.4 / 35.7, 32768 x 4096 (256 tiles) 128 tokens 66 / 52. With more tiles the 256-row tiles' fewer bytes per product win: 40960 x 4096 (320)
    // 101 tokens 65.8 / 70, 128256 x 4096 (Q6_K) 209 / 235. Beyond 128 tokens mid_body is still the faster one (4096 x 4096: 256 tokens 55.8 / 26.6, 512 60 / 36) and not taken for its
    // results: it adds the halves of every 128 k in another order, and tokens decoded behind such a prompt then differ from those behind pf_body's by up to 3 % of their logits (eight layers of
    // the 8B shape; their 8-bit roundings turn), although neither is nearer to 64 bits
    bool two = false;                                           // 8-bit activations: tiles of 64 tokens for what needs a second set of accumulators (PM_PF_WIDE_TWO)
    for (int j = 0; j < njobs; ++j) two |= wide && jobs[j].type != PM_Q4_K;
    long mid_wgs = 0;
    for (int j = 0; j < njobs && !(pair && j); ++j) mid_wgs += (jobs[j].N + (pair ? 63 : 127)) / (pair ? 64 : 128);
    // (8-bit activations: mid_body at any size - its tiles side by side -, pf_body's registers are its accumulators')
    const bool mid = wide || (!asked_nt && T <= 128 && mid_wgs <= cus);
    const int rows = mid ? 128 : 256;
    PfP p = {};
    p.pair = pair ? 1 : 0;
    int tiles = 0, ta = jobs[0].type, tb = jobs[0].type;
    for (int j = 0; j < njobs; ++j) {
        const int rc = pm_gemm_pf_check(jobs[j].type, K, jobs[j].N, T);
        if (rc) return rc;
        if (jobs[j].type != ta) { if (tb != ta && jobs[j].type != tb) return -1; tb = jobs[j].type; }
        PfJob & o = p.job[j];
        o.W = (const uint8_t *) jobs[j].W; o.Y = jobs[j].Y; o.Yh = (_Float16 *) jobs[j].Yh; o.bias = jobs[j].bias; o.resid = jobs[j].resid; o.silu_gate = jobs[j].silu_gate;
        o.row_stride = (long) pm_weight_row_stride(jobs[j].type, K); o.ldy = jobs[j].ldy ? jobs[j].ldy : jobs[j].N; o.type = jobs[j].type; o.N = jobs[j].N; o.tile0 = tiles;
        tiles += (jobs[j].N + rows - 1) / rows;
    }
    if (pair) tiles = (jobs[0].N + rows / 2 - 1) / (rows / 2);
    if (ta > tb) { const int t = ta; ta = tb; tb = t; }       // (Q4_K, Q6_K) in that order
    static const int grp = [] { const char * e = getenv("PM355_GEMM_PF_GROUP"); return e ? atoi(e) : 0; }();
    p.grp = grp;
    p.njobs = njobs; p.nt_n = tiles; p.Xh = (const _Float16 *) xh; p.K = K; p.T = T;
    if (wide) { p.Xd = (const uint8_t *) wide->d; p.Xs = (const uint8_t *) wide->s; p.ldt = wide->ldt; }
    static const int force_s = [] { const char * e = getenv("PM355_GEMM_PF_SPLITK"); return e ? atoi(e) : 0; }();
    static const bool no_mixed = [] { const char * e = getenv("PM355_GEMM_PF_MIXED"); return e && e[0] == '0'; }();
    pm_gemm_pf_plan_t pl;
    pm_gemm_pf_plan({tiles, K, T, cus, wide ? (two ? PM_PF_WIDE_TWO : PM_PF_WIDE) : mid ? PM_PF_ROWS_128 : PM_PF_ROWS_256, wide ? wide->ldt : 0, mid ? 0 : asked_nt, force_s, no_mixed ? 0 : 1}, &pl);
    const int nt = pl.nt, S = pl.splitk, full = pl.full, maxL = ((tiles + 7) / 8) * pl.nt_t;
    p.nt_t = pl.nt_t;
    p.splitk = S; p.full = full;
    const int split_slots = maxL - full;                       // per XCD
    std::unique_lock<std::mutex> slabs(g_pf_mu, std::defer_lock);
    if (S > 1) {
        slabs.lock();
        const size_t slab = (size_t) 8 * (mid ? (nt + 1) / 2 : nt) * 4 * 64 * 16, need = (size_t) 8 * split_slots * S * slab;
        p.ws = (float *) pf_workspace(st, need);
        if (!p.ws) return -3;
    }
    const int slots = full + split_slots * S;
    const bool few = mid && !wide && (ta == PM_Q8_0 ? nt == 2 && (long) tiles * pl.nt_t * S < 128 : nt == 4 && K <= 512);      // (PF_SELF)
    const bool self = wide ? nt == 4 || ta != tb || ta == PM_Q5_K : few;                                  // (mid_self of the kernel below)
    auto go = [&](auto kern, size_t lds) {
        pf_allow_lds((const void *) kern, lds);
        hipLaunchKernelGGL(kern, dim3(8 * slots), dim3(mid && !self ? MID_NTHR : PF_NTHR), lds, st, p);
        if (S == 1) return;
        if (norm && !full && T <= 512 && njobs == 1 && jobs[0].Y && !jobs[0].Yh && !jobs[0].silu_gate && p.job[0].ldy == p.job[0].N && jobs[0].N % 256 == 0 && jobs[0].N <= 8192) {
            auto fused = [&](auto k) { hipLaunchKernelGGL(k, dim3(T), dim3(1024), 0, st, p, (int) mid, nt, norm->w, norm->eps, (_Float16 *) norm->yh); };
            if (S <= 4) fused(pf_reduce_norm_kernel<4>); else fused(pf_reduce_norm_kernel<8>);
            norm->done = true;
            return;
        }
        // (a token's V^T is 2-byte pieces n_ctx apart: from 256 tokens on rope_kv_prompt_kernel turns them in tiles)
        bool roped = rope && !full && T < 256 && njobs == 3 && !p.pair && jobs[1].N == jobs[2].N && jobs[1].N == rope->Hkv * rope->dh && jobs[0].N + 2 * jobs[1].N <= 48 * 256 && rope->dh % 4 == 0 && rope->n_dims % 4 == 0;
        for (int j = 0; j < njobs && roped; ++j) roped = jobs[j].N % 256 == 0 && jobs[j].Y && !jobs[j].Yh && !jobs[j].resid && !jobs[j].silu_gate && p.job[j].ldy == p.job[j].N && jobs[j].N % rope->dh == 0;
        if (roped) {
            if (S <= 4) hipLaunchKernelGGL(pf_reduce_rope_kernel<4>, dim3(T), dim3(1024), 0, st, p, (int) mid, nt, *rope);
            else        hipLaunchKernelGGL(pf_reduce_rope_kernel<8>, dim3(T), dim3(1024), 0, st, p, (int) mid, nt, *rope);
            rope->done = true;
            return;
        }
        const int units = 8 * split_slots * (p.pair ? 4 : 8) * (mid ? (nt + 1) / 2 : nt);
        if (S <= 4) hipLaunchKernelGGL(pf_reduce_kernel<4>, dim3(units), dim3(256), 0, st, p, (int) mid, nt, units);
        else        hipLaunchKernelGGL(pf_reduce_kernel<8>, dim3(units), dim3(256), 0, st, p, (int) mid, nt, units);
    };
#if PM_GEMM_ABLATE
    static const int exp_sw = [] { const char * e = getenv("PM355_GEMM_EXP"); return e ? atoi(e) : 0; }();
    if (exp_sw && ta == PM_Q4_K && tb == PM_Q4_K && nt == 8) {
        static unsigned long long * tr = nullptr;
        if (!tr) (void) hipMalloc((void **) &tr, 42 * 8);
        p.trace = tr;
        switch (exp_sw) {
#define PF_AB(E) case E: go(gemm_pf_kernel<PM_Q4_K, PM_Q4_K, 8, false, E>, pf_lds_bytes<PM_Q4_K, PM_Q4_K, 8>()); return 0;
            PF_AB(3) PF_AB(4) PF_AB(8) PF_AB(16) PF_AB(24) PF_AB(27)
#define PF_TR(E) case 128 + E: go(gemm_pf_kernel<PM_Q4_K, PM_Q4_K, 8, false, 128 + E>, pf_lds_bytes<PM_Q4_K, PM_Q4_K, 8>()); break;
            PF_TR(0) PF_TR(3) PF_TR(8) PF_TR(16) PF_TR(24) PF_TR(27)
#undef PF_TR
            default: return -2;
        }
        unsigned long long hst[42];
        (void) hipStreamSynchronize(st);
        (void) hipMemcpy(hst, tr, sizeof hst, hipMemcpyDeviceToHost);
        for (int g = 0; g < 2; ++g) {
            fprintf(stderr, "pf trace exp %d wave %d:", exp_sw & 127, 4 * g);
            for (int k = 1; k < 17; ++k) fprintf(stderr, " %s%lld", k % 4 == 1 ? "| M " : k % 4 == 2 ? "b " : k % 4 == 3 ? "C " : "b ", (long long) (hst[g * 17 + k] - hst[g * 17 + k - 1]));
            fprintf(stderr, "  (A starts %lld after B)\n", (long long) (hst[0] - hst[17]));
        }
        return 0;
    }
#endif
    const bool cut = nt == 8 && cut_pays(K, T, S, full);
    // (an nt that no kernel has stays an error)
#define PF_GO(A, B) do { \
        if (wide) { \
            if (nt == 4)      go(gemm_pf_kernel<PM_Q4_K, PM_Q4_K, 4, true, 0, true>, pf_lds_bytes<PM_Q4_K, PM_Q4_K, 4, true, true>()); \
            else if (nt == 3) go(gemm_pf_kernel<PM_Q4_K, PM_Q4_K, 3, true, 0, true>, pf_lds_bytes<PM_Q4_K, PM_Q4_K, 3, true, true>()); \
            else if (nt == 2) go(gemm_pf_kernel<A, B, 2, true, 0, A != PM_Q8_0>, pf_lds_bytes<A, B, 2, true, A != PM_Q8_0>()); \
            else return -2; \
        } else if (mid) { \
            constexpr int OWN4 = A == PM_Q8_0 ? 0 : PF_SELF; \
            if (nt == 4)      { if (few) go(gemm_pf_kernel<A, B, 4, true, OWN4>, pf_lds_bytes<A, B, 4, true>()); else go(gemm_pf_kernel<A, B, 4, true>, pf_lds_bytes<A, B, 4, true>()); } \
            else if (nt == 3) go(gemm_pf_kernel<A, B, 3, true>, pf_lds_bytes<A, B, 3, true>()); \
            else if (nt == 2) { if (few) go(gemm_pf_kernel<PM_Q8_0, PM_Q8_0, 2, true, PF_SELF>, pf_lds_bytes<PM_Q8_0, PM_Q8_0, 2, true>()); else go(gemm_pf_kernel<A, B, 2, true>, pf_lds_bytes<A, B, 2, true>()); } \
            else return -2; \
        } else if (nt == 8) { \
            if (cut) go(gemm_pf_kernel<A, B, 8, false, PF_CUT>, pf_lds_bytes<A, B, 8>()); else go(gemm_pf_kernel<A, B, 8>, pf_lds_bytes<A, B, 8>()); \
        } \
        else if (nt == 6)     go(gemm_pf_kernel<A, B, 6>, pf_lds_bytes<A, B, 6>()); \
        else if (nt == 4)     go(gemm_pf_kernel<A, B, 4>, pf_lds_bytes<A, B, 4>()); \
        else if (nt == 2)     go(gemm_pf_kernel<A, B, 2>, pf_lds_bytes<A, B, 2>()); \
        else return -2; \
    } while (0)
    if (ta == tb) { if (ta == PM_Q4_K) PF_GO(PM_Q4_K, PM_Q4_K); else if (ta == PM_Q5_K) PF_GO(PM_Q5_K, PM_Q5_K); else if (ta == PM_Q8_0) PF_GO(PM_Q8_0, PM_Q8_0); else PF_GO(PM_Q6_K, PM_Q6_K); }
    else if (ta == PM_Q8_0 || tb == PM_Q8_0) return -1;      // (Q8_0 only as a launch of its own: ffn_down of the files whose n_ff is no multiple of 256)
    else if (ta == PM_Q4_K && tb == PM_Q5_K) PF_GO(PM_Q4_K, PM_Q5_K);
    else if (ta == PM_Q4_K && tb == PM_Q6_K) PF_GO(PM_Q4_K, PM_Q6_K);
    else PF_GO(PM_Q5_K, PM_Q6_K);
#undef PF_GO
    return 0;
}
int pm_launch_gemm_pf_ex(const pm_gemm_pf_job * jobs, int njobs, const void * xh, int K, int T, int pair, hipStream_t st) { return launch_pf(jobs, njobs, xh, nullptr, K, T, pair, st); }

int pm_launch_gemm_pf_rope(const pm_gemm_pf_job * jobs, const void * xh, int K, int T, pm_gemm_rope * rope, hipStream_t st) { rope->done = false; return launch_pf(jobs, 3, xh, nullptr, K, T, 0, st, nullptr, rope); }
int pm_launch_gemm_pf_norm(const pm_gemm_pf_job & job, const void * xh, int K, int T, pm_gemm_norm * norm, hipStream_t st) { norm->done = false; return launch_pf(&job, 1, xh, nullptr, K, T, 0, st, norm); }

int pm_gemm_wide_check(int type, int K, int N, int T) {
    if ((type != PM_Q4_K && type != PM_Q5_K && type != PM_Q6_K) || T < 1 || T > PM_WIDE_MAX_TOKENS) return -1;
    return pm_gemm_pf_check(type, K, N, T);
}
int pm_launch_gemm_wide(const pm_gemm_pf_job * jobs, int njobs, const pm_q8k_wide & x, int K, int T, int pair, hipStream_t st, pm_gemm_rope * rope) {
    if (rope) rope->done = false;
    if (T > PM_WIDE_MAX_TOKENS || !x.q || x.ldt < (T <= 64 ? 64 : (T + 127) / 128 * 128) || x.ldt % 4 || (size_t) (K / 256) * x.ldt * 32 >= ((size_t) 1 << 32)) return -2;
    for (int j = 0; j < njobs; ++j) if (pm_gemm_wide_check(jobs[j].type, K, jobs[j].N, T)) return -1;
    return launch_pf(jobs, njobs, x.q, &x, K, T, pair, st, nullptr, rope);
}
static size_t wide_rows(int rows) { return rows <= 64 ? 64 : (size_t) (rows + 127) / 128 * 128; }
size_t pm_q8k_wide_bytes(int K, int rows) { return wide_rows(rows) * ((size_t) K * 2 + (size_t) (K / 256) * 36); }
pm_q8k_wide pm_q8k_wide_at(void * buf, int K, int rows) {
    const size_t n = wide_rows(rows);
    pm_q8k_wide x;
    x.q = (uint16_t *) buf; x.s = x.q + n * K; x.d = (float *) (x.s + n * (K / 256) * 16); x.ldt = (int) n;
    return x;
}
