// mmq_mid.hip - quantized mat-mul for up to 32 tokens on groups of 32 rows: one matrix or several that share their activations, 9..32 tokens (and fewer where mmq_rows.hip is not the faster
// one, pm_mmq_rows_takes). The arithmetic is mmq_i8.hip's: activations in Q8_K / Q8_0 blocks, exact integer sums per super-block, one f32 multiply-add per super-block.
//
// A workgroup is four CELLS, one per SIMD. A cell has three waves: one LOADER, which does nothing but bring weights, and two that multiply, one half of every pair of super-blocks (512 k) each.
// The loader has two tiles (32 rows x a pair, full 128-byte lines) on their way in its registers and two in LDS, where the others read them in matrix-operand order; the workgroup's twelve waves
// meet once per step. So no multiplying wave ever waits in the issue of a request (with all waves loading their own tiles, each request held its wave up for 60-260 cycles and the waves' loads,
// LDS copies and products added up instead of overlapping: of 7 us per step of 72B's ffn_gate | ffn_up at 23 tokens 5 were products), and LDS tiles are turned by XOR, free of padding.
//   * most often more than 64 rows a workgroup (AL): a cell is a row group, all four work on the same pair; its activations come into LDS once for all of them (each wave for itself out of L2: 12 of 67 us
//     of 57344 x 8192 Q4_K, 20 of 125 of 59136 x 8192 Q6_K)
//   * up to 64 (32), and some others (mmq_mid_rows): two (four) cells share a row group and take pairs next to each other; a pair's activations are needed by one wave only, which loads them straight into operand registers
// Scales come in blocks of up to four pairs, whole lines of them (32 bytes of a line each time, they were a third of the lines that a CU asks for: 14 of 119 us of Q6_K).
// An integer product's results are read behind the next one's start, one v_mad_i32_i24 each (mad24), for up to 8, 16, 24 or 32 tokens.
// Bound by the weights' stream (Q4_K 6.2 TB/s between the first tile, 5 us, and the last sums) and, Q6_K, by vector work (400 instructions per 32 rows x 256 k at 24 tokens).
// us, the form that it replaced (mmq_i8.hip's of then) / here, at 23 tokens: 59136 x 8192 Q6_K 132 / 97, 10240 x 8192 40 / 30, 8192 x 8192 26 / 21, 8192 x 28672 70 / 57; 57344 x 8192 Q4_K
// 78 / 57, 10240 x 8192 23 / 18, 8192 x 28672 40 / 33, 28672 x 4096 27 / 20; 128256 x 4096 Q6_K 160 / 107; 8192 x 29568 Q8_0 76 / 55. Weights out of memory, one matrix of 70..128256 rows, K =
// 512..28672, time here / time there in the geometric mean: Q4_K up to 8 tokens 0.91, 16 0.87, 32 0.85, several matrices 0.83 0.80 0.77; Q6_K 0.89 0.87 0.81, 0.85 0.82 0.76 (slower: Q6_K
// 10240 x 5120 up to 8 tokens 17.4 / 18.0 us, Q4_K 57344 x 14336 at 8 tokens 80.5 / 83)
#include "pm355_device.h"
#include "pm355_kernels.h"
#include "pm355_mmq_rows.h"
#include <algorithm>
#include <type_traits>

namespace {

typedef int      i32x4 __attribute__((ext_vector_type(4)));
typedef int      i32x16 __attribute__((ext_vector_type(16)));
typedef float    f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int CELLS = 4, CW = 8, NT = 64 * (CW + CELLS);

#define PIN __builtin_amdgcn_sched_barrier(0)

__device__ __forceinline__ long pk(uint32_t a, uint32_t b) { return (long) (((uint64_t) b << 32) | a); }
__device__ __forceinline__ u32x4 ld_c16(const void * p) { return *(const PM_G u32x4 *) p; }
__device__ __forceinline__ i32x16 mfma_16k(long a, long b) { const i32x16 z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}; return __builtin_amdgcn_mfma_i32_32x32x16_i8(a, b, z, 0, 0, 0); }
__device__ __forceinline__ i32x16 mfma_32k(u32x4 a, u32x4 b) {
    const i32x16 z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), z, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma_h(u32x4 a, u32x4 b) {
    const f32x16 z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), z, 0, 0, 0);
}
__device__ __forceinline__ uint32_t pk_fma(uint32_t a, _Float16 m, _Float16 c) {
    const f16x2 v = __builtin_bit_cast(f16x2, a), mm = {m, m}, cc = {c, c};
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(v, mm, cc));
}
// the waves meet; what they wrote to LDS is there (requests for memory stay on their way)
__device__ __forceinline__ void meet() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// NV result registers per lane in use: 4 (<= 8 tokens), 8 (<= 16), 12 (<= 24), 16 (<= 32). Sub-blocks per operand register (mmq_i8.hip, ActSrc), products on their way in front of the one
// whose results are read
template <int NV> constexpr int PACK = NV > 8 ? 1 : 16 / NV;
template <int NV> constexpr int AHEAD = NV > 8 ? 1 : NV > 4 ? 2 : 3;
// sum += scale * product, as ONE v_mad_i32_i24 per result (re-associated into mul, mul, add3 it is 1.5). A product's other results stay where they are until then: a register among them that
// is written anew while the product is on its way costs a wait of 12 instructions
template <int NV> __device__ __forceinline__ void mad24(i32x16 & sum, int scale, const i32x16 & acc, int at) {
#pragma unroll
    for (int v = 0; v < NV; ++v) { sum[v] = __mul24(scale, acc[at + v]) + sum[v]; asm("" : "+v"(sum[v])); }
    if constexpr (NV < 16) asm volatile("" :: "v"(acc));
}

// activations of half a pair out of the operand-ordered tables (mmq_i8.hip, ActSrc)
struct ASrc {
    __amdgpu_buffer_rsrc_t rq, rb; uint32_t qo, bo; int n;
    __device__ __forceinline__ u32x4 q(int blk) const { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rq, (int) qo, blk * 1024, 0)); }
    __device__ __forceinline__ u32x4 b(int sb) const { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rb, (int) bo, sb * 1024, 0)); }
};
template <int TYPE, int NV> struct ASet { u32x4 q[8 / PACK<NV>], bs; };
template <int NV> struct ASet<PM_Q8_0, NV> { u32x4 q[4 / PACK<NV>]; };
// request k of half `par` of a pair (behind the last pair: the last one's)
template <int TYPE, int NV> constexpr int NA = TYPE == PM_Q8_0 ? 4 / PACK<NV> : 8 / PACK<NV> + 1;
template <int TYPE, int NV> __device__ __forceinline__ void load_a(ASet<TYPE, NV> & a, const ASrc & s, int pair, int par, int k) {
    if constexpr (TYPE == PM_Q8_0) a.q[k] = s.q(8 * pair + 4 * par + k * PACK<NV>);          // (blocks past the end: zeros)
    else {
        const int sb = min(2 * pair + par, s.n - 1);
        if (k < 8 / PACK<NV>) a.q[k] = s.q(8 * sb + k * PACK<NV>); else a.bs = s.b(sb);
    }
}

// ---- a tile: 32 rows of a pair of super-blocks. In LDS: streams of 128 bytes a row, piece c of row r at c ^ turn(r)
__device__ __forceinline__ int turn(int row) { return ((row >> 1) & 3) | ((row >> 1) & 4); }
// NQ: requests; SLOT: bytes in LDS; HU: bytes of a row's scales of a pair; DT: bytes of a pair's activation scales; NP: kilobytes of a pair's activations
template <int TYPE> struct Fmt;
template <> struct Fmt<PM_Q4_K> { static constexpr int NQ = 8,  SLOT = 8192,  HU = 32, DT = 256,  SUBS = 16; };   // qa[U][16] | qb[U][16] | hdr[nb][16]
template <> struct Fmt<PM_Q5_K> { static constexpr int NQ = 11, SLOT = 32 * 368, HU = 0, DT = 256, SUBS = 16; };  // native 176-byte blocks: 352 bytes a row, 368 in LDS
template <> struct Fmt<PM_Q6_K> { static constexpr int NQ = 12, SLOT = 12288, HU = 32, DT = 256,  SUBS = 16; };   // la[U][16] | lb[U][16] | qh[U][16] | scales[nb][16] | d[nb]
template <> struct Fmt<PM_Q8_0> { static constexpr int NQ = 8,  SLOT = 8192,  HU = 16, DT = 1024, SUBS = 8; };    // qa[nb][16] | qb[nb][16] | d[nb]: 8 blocks
template <int TYPE> struct Tile { u32x4 q[Fmt<TYPE>::NQ], h, dt; uint32_t d; };
// Scales travel in blocks of HP pairs: a row's 32 bytes of a pair are a quarter of the line that they come in
template <int TYPE, int NV, bool AL> constexpr int HP = AL && TYPE == PM_Q6_K ? (NV == 16 ? 1 : 2) : 4;
template <int TYPE, int NV> constexpr int a_bytes() { return Fmt<TYPE>::SUBS * 64 * NV + (TYPE == PM_Q8_0 ? 0 : 128 * NV) + Fmt<TYPE>::DT; }
// LDS of a workgroup: slots (two per cell) | scales (two blocks per row group) | d of Q6_K | activations (AL: two pairs) | sums
template <int TYPE, int NV, bool AL> struct Lds {
    static constexpr int RG = AL ? 4 : 2, H = 32 * Fmt<TYPE>::HU * HP<TYPE, NV, AL>, D = TYPE == PM_Q6_K ? 128 * HP<TYPE, NV, AL> : 0;
    static constexpr int SLOT = Fmt<TYPE>::SLOT + Fmt<TYPE>::DT;
    static constexpr int HDR = CELLS * 2 * SLOT, DD = HDR + RG * 2 * H, ACT = DD + RG * 2 * D, RED = ACT + (AL ? 2 * a_bytes<TYPE, NV>() : 0), BYTES = RED + (AL ? 4 : 8) * NV * 256;
};

// ---- the cell's loader
template <int TYPE, int NV, bool AL> struct Loader {
    typedef Fmt<TYPE> F;
    typedef Lds<TYPE, NV, AL> L;
    static constexpr int hp = HP<TYPE, NV, AL>, NPL = ((F::SUBS + (TYPE == PM_Q8_0 ? 0 : 2) + 1) + 3) / 4;
    const uint8_t * base, * qT, * bsT; const float * dT; uint8_t * smem;     // qT, bsT: with the lane's bytes
    uint32_t stride, rows[4];
    int lane, nb, npair, lim, rl, rgi, kp, cell, n, nround, kl, HS, dt0;      // kl: logarithm of the pairs at a time
    struct Pos { int rd, j; } in, hin, pa;                          // of the next tile, of the block of scales that is asked for, of the next activations
    int hf, at, pf, pb;                                             // pieces of that block asked for; pair of the next tile, piece and block of the next scales to be put down
    __device__ __forceinline__ void rows_of() {
        const int rb = 32 * ((in.rd << rl) + rgi);
        if constexpr (TYPE == PM_Q5_K) rows[0] = (uint32_t) min(rb, lim);
        else {
#pragma unroll
            for (int k = 0; k < 4; ++k) rows[k] = (uint32_t) min(rb + (lane >> 3) + 8 * k, lim) * stride;
        }
    }
    // piece `piece` of the block of scales whose first step is `p`
    __device__ __forceinline__ void load_h(u32x4 & h, uint32_t & d, Pos p, int piece) const {
        if constexpr (F::HU == 0) return;
        constexpr int CH = F::HU / 16 * hp;                         // 16-byte chunks of a row
        const int l = lane & (32 / hp * CH - 1), row = piece * (32 / hp) + l / CH, c = l % CH, e = c / (F::HU / 16);
        auto where = [&](int e, uint32_t & at, int & pair) __attribute__((always_inline)) {
            int j = p.j + (e >> kl), rd = p.rd;
#pragma unroll
            for (int k = 0; k < 3; ++k) if (j >= n) { j -= n; ++rd; }
            pair = min((e & ((1 << kl) - 1)) + (j << kl), npair - 1);
            at = (uint32_t) min(32 * ((min(rd, nround - 1) << rl) + rgi), lim);
        };
        uint32_t first; int pair;
        where(e, first, pair);
        const uint32_t off = (uint32_t) min((int) first + row, lim) * stride;
        if constexpr (TYPE == PM_Q8_0) h = ld_c16(base + (size_t) nb * 32 + (off + (uint32_t) pair * 16u));      // (rows are padded to 16 bytes)
        else {
            const uint32_t sb = (uint32_t) min(2 * pair + (c & 1), nb - 1);
            h = ld_c16(base + (TYPE == PM_Q4_K ? (size_t) nb * 128 : 0) + (off + (TYPE == PM_Q4_K ? sb * 16u : pm_q6k_sc_off((uint32_t) nb, sb))));
        }
        if constexpr (TYPE == PM_Q6_K) {
            const int l2 = lane & 31, row2 = piece * (32 / hp) + l2 / hp;
            where(l2 % hp, first, pair);
            const uint32_t o2 = (uint32_t) min((int) first + row2, lim) * stride, s0 = 2 * (uint32_t) pair, s1 = min(s0 + 1, (uint32_t) nb - 1);
            if constexpr (PM_Q6K_SCD == 0) {
                d = *(const PM_G uint32_t *) (base + (o2 + pm_q6k_d_off((uint32_t) nb, s0)));      // (a last super-block alone: two bytes of the row's padding beside it)
                if (s1 == s0) d &= 0xFFFFu;
            } else d = *(const PM_G uint16_t *) (base + (o2 + pm_q6k_d_off((uint32_t) nb, s0))) | (uint32_t) *(const PM_G uint16_t *) (base + (o2 + pm_q6k_d_off((uint32_t) nb, s1))) << 16;
        }
    }
    __device__ __forceinline__ void put_h(const u32x4 & h, uint32_t d, int buf, int piece) const {
        if constexpr (F::HU == 0) return;
        constexpr int CH = F::HU / 16 * hp;
        const int l = lane & (32 / hp * CH - 1), row = piece * (32 / hp) + l / CH, c = l % CH;
        uint8_t * H = smem + L::HDR + (2 * rgi + buf) * L::H;
        if (lane == l) *(u32x4 *) (H + row * (CH * 16) + ((c ^ (row & (CH - 1))) << 4)) = h;
        if constexpr (TYPE == PM_Q6_K) {
            const int l2 = lane & 31, row2 = piece * (32 / hp) + l2 / hp;
            if (lane < 32) *(uint32_t *) (smem + L::DD + (2 * rgi + buf) * L::D + row2 * (4 * hp) + (l2 % hp) * 4) = d;
        }
    }
    // the next tile, and (HEAD) the next piece of scales. Behind the last one, of no rows or no columns: a few bytes at the start of the slice
    template <bool HEAD> __device__ __forceinline__ void load(Tile<TYPE> & t) {
        const int pair = kp + (in.j << kl), pc = min(pair, npair - 1);
        const uint32_t keep = in.rd < nround && 32 * ((in.rd << rl) + rgi) <= lim && pair < npair ? ~0u : 0u;
        if constexpr (TYPE == PM_Q5_K) {
#pragma unroll
            for (int k = 0; k < 11; ++k) {
                int ci = lane + 64 * k;
                asm("" : "+v"(ci));                                 // (places are computed where they are needed: kept, they cost 22 registers)
                const int row = ci / 22, c = ci - row * 22, sb = min(2 * pc + (c >= 11), nb - 1);
                const uint8_t * at = base + (((uint32_t) min((int) rows[0] + row, lim) * stride + (uint32_t) sb * 176u + (uint32_t) (c >= 11 ? c - 11 : c) * 16u) & keep);
                t.q[k] = AL ? ld_c16(at) : ld_nt16(at);
            }
        } else {
            const uint32_t u = (uint32_t) min(8 * pc + (lane & 7), (TYPE == PM_Q8_0 ? 1 : 4) * nb - 1) * 16u;
            constexpr int NS = TYPE == PM_Q6_K ? 3 : 2;
#pragma unroll
            for (int k = 0; k < F::NQ; ++k) {
                // (AL: rows of Q6_K and Q8_0 may start in the middle of a line; its other half is the next pair's, and stays in L2 until then: ffn_gate | ffn_up of the 72B shape 110 -> 101 us)
                const uint8_t * at = base + (size_t) nb * ((TYPE == PM_Q8_0 ? 16 : 64) * (k % NS)) + ((rows[k / NS] + u) & keep);
                t.q[k] = !AL || TYPE == PM_Q4_K ? ld_nt16(at) : ld_c16(at);
            }
        }
        if constexpr (!AL) t.dt = load_dt(pc);
        if constexpr (HEAD) {
            load_h(t.h, t.d, hin, (hf << kl) + kp);
            if (++hf == HS) {
                hf = 0; hin.j += HS;
#pragma unroll
                for (int k = 0; k < 4; ++k) if (hin.j >= n) { hin.j -= n; ++hin.rd; }
            }
        }
        if (++in.j == n) { in.j = 0; ++in.rd; rows_of(); }
    }
    __device__ __forceinline__ u32x4 load_dt(int pc) const {
        if constexpr (TYPE == PM_Q8_0) return ld_c16(dT + (size_t) min(8 * pc + (lane >> 3), nb - 1) * 32 + dt0);
        else return ld_c16(dT + (size_t) min(2 * pc + ((lane >> 3) & 1), nb - 1) * 32 + dt0);
    }
    __device__ __forceinline__ void put_dt(uint8_t * p, const u32x4 & dt, int pair) const {       // (blocks behind the row, pairs behind the last one: scale 0)
        const u32x4 z = {0, 0, 0, 0};
        if constexpr (TYPE == PM_Q8_0) *(u32x4 *) (p + lane * 16) = 8 * pair + (lane >> 3) < nb ? dt : z;
        else if (lane < 16) *(u32x4 *) (p + lane * 16) = 2 * pair + (lane >> 3) < nb ? dt : z;
    }
    template <bool HEAD> __device__ __forceinline__ void put(const Tile<TYPE> & t, int s) {
        uint8_t * S = smem + (2 * cell + s) * L::SLOT;
        if constexpr (TYPE == PM_Q5_K) {
#pragma unroll
            for (int k = 0; k < 11; ++k) { int ci = lane + 64 * k; asm("" : "+v"(ci)); const int row = ci / 22, c = ci - row * 22; *(u32x4 *) (S + row * 368 + c * 16) = t.q[k]; }
        } else {
            constexpr int NS = TYPE == PM_Q6_K ? 3 : 2;
#pragma unroll
            for (int k = 0; k < F::NQ; ++k) { const int row = (lane >> 3) + 8 * (k / NS); *(u32x4 *) (S + (k % NS) * 4096 + row * 128 + (((lane & 7) ^ turn(row)) << 4)) = t.q[k]; }
        }
        if constexpr (!AL) { put_dt(S + F::SLOT, t.dt, kp + (at << kl)); if (++at == n) at = 0; }
        if constexpr (HEAD) { put_h(t.h, t.d, pb, (pf << kl) + kp); if (++pf == HS) { pf = 0; pb ^= 1; } }
    }
    // activations of a pair: kilobytes cell, cell + 4, ..: sub-blocks, group sums, scales
    __device__ __forceinline__ void load_a(u32x4 (&a)[NPL]) {
        const int pc = pa.j;                                        // (one pair at a time: < npair)
#pragma unroll
        for (int i = 0; i < NPL; ++i) {
            const int k = cell + 4 * i;
            const uint8_t * p;
            if constexpr (TYPE == PM_Q8_0) p = qT + (size_t) min(8 * pc + min(k, 7), nb - 1) * 1024;
            else if (k < 16) p = qT + (size_t) (min(2 * pc + (k >> 3), nb - 1) * 8 + (k & 7)) * 1024;
            else p = bsT + (size_t) min(2 * pc + (k & 1), nb - 1) * 1024;
            if (k == F::SUBS + (TYPE == PM_Q8_0 ? 0 : 2)) a[i] = load_dt(pc); else a[i] = ld_c16(p);
        }
        if (++pa.j == n) pa.j = 0;
    }
    __device__ __forceinline__ void put_a(const u32x4 (&a)[NPL], int s, int pair) const {
        uint8_t * A = smem + L::ACT + s * a_bytes<TYPE, NV>();
        const int t = lane & 31, g = lane >> 5;
#pragma unroll
        for (int i = 0; i < NPL; ++i) {
            const int k = cell + 4 * i;
            constexpr int NK = F::SUBS + (TYPE == PM_Q8_0 ? 0 : 2);
            if (k < NK) { if (t < 2 * NV) *(u32x4 *) (A + (k * 4 * NV + g * 2 * NV + t) * 16) = a[i]; }
            else if (k == NK) put_dt(A + a_bytes<TYPE, NV>() - F::DT, a[i], pair);
        }
    }
};

// ---- products of half `par` of a pair. next(k): operand register k has been read
template <int NV> __device__ __forceinline__ void finish(f32x16 & out, const float * yd_lds, int g, float d, const i32x16 & isum) {
#pragma unroll
    for (int q = 0; q < NV / 4; ++q) {
        const f32x4 yd = *(const f32x4 *) (yd_lds + 8 * q + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) out[4 * q + i] = fmaf(yd[i] * d, (float) isum[4 * q + i], out[4 * q + i]);
    }
}
template <int NV> __device__ __forceinline__ void finish(f32x16 & out, const float * yd_lds, int g, float d, const i32x16 & isum, float dmin, const f32x16 & ms) {
#pragma unroll
    for (int q = 0; q < NV / 4; ++q) {
        const f32x4 yd = *(const f32x4 *) (yd_lds + 8 * q + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int v = 4 * q + i;
            out[v] = fmaf(yd[i] * d, (float) isum[v], fmaf(-(yd[i] * dmin), ms[v], out[v]));
        }
    }
}
struct K4 {                                                        // the eight 6-bit scales and minima, four to a dword (get_scale_min_k4, ggml-quants.c:1898-1906)
    uint32_t sc[2], mn[2];
    __device__ __forceinline__ explicit K4(const u32x4 & hd) {
        sc[0] = hd[1] & 0x3f3f3f3fu; sc[1] = (hd[3] & 0x0f0f0f0fu) | ((hd[1] >> 2) & 0x30303030u);
        mn[0] = hd[2] & 0x3f3f3f3fu; mn[1] = ((hd[3] >> 4) & 0x0f0f0f0fu) | ((hd[2] >> 2) & 0x30303030u);
    }
    __device__ __forceinline__ int scale(int s) const { return (int) ((sc[s >> 2] >> (8 * (s & 3))) & 0xFFu); }
    // as F16, exact (0x6400 | m = 1024 + m)
    __device__ __forceinline__ u32x4 mins() const {
        u32x4 m;
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] = pk_fma(__builtin_amdgcn_perm(mn[i >> 1], 0x64646464u, i & 1 ? 0x00070006u : 0x00050004u), (_Float16) 1.0f, (_Float16) -1024.0f);
        return m;
    }
};
template <int TYPE, int NV, class F>
// L: the tile; H: this row's scales of the half; dd: its d (Q6_K); ds: activation scales of the half
__device__ __forceinline__ void products(ASet<TYPE, NV> & a, const uint8_t * L, const uint8_t * H, const uint8_t * dd, const float * ds, int par, int r, int g, f32x16 & out, F && next) {
    constexpr int AH = AHEAD<NV>, P = PACK<NV>;
    i32x16 acc[AH + 1];
    i32x16 isum = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    if constexpr (TYPE == PM_Q4_K) {
        const u32x4 hd = *(const u32x4 *) H;
        const K4 k(hd);
        const uint8_t * row = L + g * 4096 + r * 128;
        const int tr = turn(r);
        u32x4 w = *(const u32x4 *) (row + (((4 * par) ^ tr) << 4)), wn = w;
#pragma unroll
        for (int s = 0; s < 8 + AH; ++s) {
            if (s < 8 && (s & 1) == 0) {
                if (s) w = wn;
                if (s < 6) wn = *(const u32x4 *) (row + (((4 * par + s / 2 + 1) ^ tr) << 4));
            }
            if (s < 8) { acc[s % (AH + 1)] = mfma_32k(a.q[s / P], (s & 1 ? w >> 4 : w) & 0x0F0F0F0Fu); PIN; if (s % P == P - 1) next(s / P); PIN; }
            const int t = s - AH;
            if (t >= 0) mad24<NV>(isum, k.scale(t), acc[t % (AH + 1)], NV * (t % P));
            if (s < 8) PIN;
        }
        const f32x16 ms = mfma_h(a.bs, k.mins());                  // sum_s min_s * (bsum[2s] + bsum[2s+1]), exact
        PIN; next(8 / P); PIN;
        finish<NV>(out, ds, g, h2f((uint16_t) (hd[0] & 0xFFFF)), isum, h2f((uint16_t) (hd[0] >> 16)), ms);
    } else if constexpr (TYPE == PM_Q5_K) {
        const uint8_t * blk = L + r * 368 + par * 176;
        const u32x4 hd = *(const u32x4 *) blk, qh = *(const u32x4 *) (blk + 16 + 16 * g);       // qh bit s of byte l: fifth bit of weight l of sub-block s (l = 16 g + i)
        const K4 k(hd);
        u32x4 w = *(const u32x4 *) (blk + 48 + 16 * g), wn = w;
#pragma unroll
        for (int s = 0; s < 8 + AH; ++s) {
            if (s < 8 && (s & 1) == 0) {
                if (s) w = wn;
                if (s < 6) wn = *(const u32x4 *) (blk + 48 + 32 * (s / 2 + 1) + 16 * g);
            }
            if (s < 8) { acc[s % (AH + 1)] = mfma_32k(a.q[s / P], ((s & 1 ? w >> 4 : w) & 0x0F0F0F0Fu) | (((qh >> s) & 0x01010101u) << 4)); PIN; if (s % P == P - 1) next(s / P); PIN; }
            const int t = s - AH;
            if (t >= 0) mad24<NV>(isum, k.scale(t), acc[t % (AH + 1)], NV * (t % P));
            if (s < 8) PIN;
        }
        const f32x16 ms = mfma_h(a.bs, k.mins());
        PIN; next(8 / P); PIN;
        finish<NV>(out, ds, g, h2f((uint16_t) (hd[0] & 0xFFFF)), isum, h2f((uint16_t) (hd[0] >> 16)), ms);
    } else if constexpr (TYPE == PM_Q6_K) {
        const u32x4 s16 = *(const u32x4 *) H;
        const float d = h2f(*(const uint16_t *) dd);
        uint32_t lo = 0x0F0F0F0Fu, hi2 = 0x30303030u;              // masks in scalar registers: (x & mask) | y is one v_and_or_b32 then
        asm("" : "+s"(lo)); asm("" : "+s"(hi2));
        const uint8_t * row = L + r * 128 + 8 * g;
        const int tr = turn(r);
        struct Raw { u32x2 la, lb, qh; } raw, ahead;
        auto read = [&](int u) __attribute__((always_inline)) {
            const uint8_t * p = row + (((4 * par + u) ^ tr) << 4);
            return Raw{*(const u32x2 *) p, *(const u32x2 *) (p + 4096), *(const u32x2 *) (p + 8192)};
        };
        ahead = read(0);
        // the offset of every weight first: - 32 sum_G scale_G * bsum_G. Operand slot s of lane group g = scale[2 s + g], times -32 (F16: 1024 + 128 + scale from the bytes)
        const uint32_t sel = g ? 0x00070005u : 0x00060004u;
        u32x4 m;
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] = pk_fma(__builtin_amdgcn_perm(s16[i] ^ 0x80808080u, 0x64646464u, sel), (_Float16) -32.0f, (_Float16) 36864.0f);
        const f32x16 ms = mfma_h(a.bs, m);                          // (multiples of 32 below 2^29: exact)
        PIN; next(8 / P); PIN;
        // A operand of the 16-k product over group G: lane (t, g) needs bytes 8 g .. 8 g + 7 of it; as loaded the lane pair (t, 0) / (t, 1) holds groups 2 s / 2 s + 1 whole
        u32x2 aop[16 / P];
        auto operands = [&](int i) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const u32x2 x = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(a.q[i][e], a.q[i][2 + e], false, false));
                aop[2 * i][e] = x[0]; aop[2 * i + 1][e] = x[1];
            }
        };
        u32x2 qv[4];
#pragma unroll
        for (int i = 0; i < 16 + AH; ++i) {
            const int u = i >> 2, c = i & 3;                         // unit u = (hh, v), group 8 hh + 2 c + v
            if (i < 16 && c == 0) {
                raw = ahead;
                if (u < 3) ahead = read(u + 1);
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                    qv[0][w] = (raw.la[w] & lo) | ((raw.qh[w] << 4) & hi2);
                    qv[1][w] = (raw.lb[w] & lo) | ((raw.qh[w] << 2) & hi2);
                    qv[2][w] = ((raw.la[w] >> 4) & lo) | (raw.qh[w] & hi2);
                    qv[3][w] = ((raw.lb[w] >> 4) & lo) | ((raw.qh[w] >> 2) & hi2);
                }
            }
            if (i < 16) {
                const int s = 4 * (u >> 1) + c;
                if (!(u & 1) && s % P == 0) operands(s / P);
                const u32x2 op = aop[2 * (s / P) + (u & 1)];
                acc[i % (AH + 1)] = mfma_16k(pk(op[0], op[1]), pk(qv[c][0], qv[c][1]));
                PIN;
                if ((u & 1) && s % P == P - 1) next(s / P);
                PIN;
            }
            if (i == 0) {
#pragma unroll
                for (int v = 0; v < NV; ++v) isum[v] = (int) ms[v];
                if constexpr (NV < 16) asm volatile("" :: "v"(ms));
            }
            if (i >= AH) {
                const int j = i - AH, s = 4 * (j >> 3) + (j & 3), G = 2 * s + ((j >> 2) & 1);
                mad24<NV>(isum, (int) (int8_t) (s16[G >> 2] >> (8 * (G & 3))), acc[j % (AH + 1)], NV * (s % P));   // |product| <= 16 * 63 * 127
            }
            if (i < 16) PIN;
        }
        finish<NV>(out, ds, g, d, isum);
    } else {
        const u32x2 d4 = *(const u32x2 *) H;                         // this row's four block scales (f16)
        const uint8_t * row = L + g * 4096 + r * 128;
        const int tr = turn(r);
        u32x4 w = *(const u32x4 *) (row + (((4 * par) ^ tr) << 4)), wn = w;
#pragma unroll
        for (int s = 0; s < 4 + AH; ++s) {
            if (s && s < 4) w = wn;
            if (s < 3) wn = *(const u32x4 *) (row + (((4 * par + s + 1) ^ tr) << 4));
            if (s < 4) { acc[s % (AH + 1)] = mfma_32k(a.q[s / P], w); PIN; if (s % P == P - 1) next(s / P); PIN; }
            const int t = s - AH;
            if (t >= 0) {
                const uint32_t hb = (d4[t >> 1] >> (16 * (t & 1))) & 0xFFFFu;
                const float dw = (hb & 0x7C00u) == 0x7C00u ? 0.0f : h2f((uint16_t) hb);            // (a block past the row: whatever the padding holds, times zero)
#pragma unroll
                for (int q = 0; q < NV / 4; ++q) {
                    const f32x4 yd = *(const f32x4 *) (ds + t * 32 + 8 * q + 4 * g);
#pragma unroll
                    for (int i = 0; i < 4; ++i) out[4 * q + i] = fmaf((float) acc[t % (AH + 1)][NV * (t % P) + 4 * q + i], dw * yd[i], out[4 * q + i]);
                }
                if constexpr (NV < 16) asm volatile("" :: "v"(acc[t % (AH + 1)]));
            }
            if (s < 4) PIN;
        }
    }
}

// a result of a row group: token t, row `row` of the matrix; what is added and where it goes
template <bool EPI> __device__ __forceinline__ void store(const RowsP & p, const RowsJob & job, int ji, float sum, int t, int row, bool live) {
    if constexpr (EPI) {
        if (job.bias) sum += ld_g(job.bias + row);
        const float sp = __shfl_xor(sum, 1);                         // the pair's other row: the neighbouring lane, same token
        if (live) {
            const int seq = p.e_seq ? p.e_seq[p.e_rows ? t : 0] : 0, pos = p.e_rows ? p.e_pos[t] : p.e_pos[seq] + t;
            const long kv = (long) seq * p.e_seq_stride;
            if (ji == 2) p.e_vc[kv + (long) row * p.e_nctx + pos] = f2h(sum);
            else {
                const int dim = row % p.e_dh;
                float o = sum;
                if (dim < p.e_nrot) {
                    const float c = ld_g(p.e_tab + (long) t * p.e_nrot + (dim & ~1)), sn = ld_g(p.e_tab + (long) t * p.e_nrot + (dim & ~1) + 1);
                    o = (dim & 1) ? sp * sn + sum * c : sum * c - sp * sn;
                }
                const uint16_t hv = f2h(o);
                if (ji == 1) p.e_kc[kv + (long) pos * p.e_kvdim + row] = hv;
                else st_g(job.y + (long) t * job.N + row, h2f(hv));
            }
        }
    } else if (live) {
        if (job.bias) sum += ld_g(job.bias + row);
        if (job.resid) sum += ld_g(job.resid + (long) t * job.N + row);
        st_g(job.y + (long) t * job.N + row, sum);
    }
}

template <int TYPE, int NV, bool EPI, bool AL>
__device__ __forceinline__ void mmq_mid_body(const RowsP & p, const RowsJob & job, int r0, int r1, int rl, int ji, uint8_t * smem) {
    typedef Fmt<TYPE> F;
    typedef Lds<TYPE, NV, AL> L;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    constexpr bool Q80 = TYPE == PM_Q8_0;
    const int lim = r1 - r0 - 1, nb = Q80 ? p.K / 32 : p.K / 256, npair = Q80 ? (nb + 7) / 8 : (nb + 1) / 2;
    const int nrg = (r1 - r0 + 31) >> 5, RG = 1 << rl, KP = CELLS >> rl;           // row groups, pairs at a time
    const int n = (npair + KP - 1) / KP, nround = (nrg + RG - 1) >> rl, total = n * nround;
    const int cell = wave & (CELLS - 1), rgi = cell & (RG - 1), kp = cell >> rl, HS = HP<TYPE, NV, AL> >> (2 - rl);
    if (wave >= CW) {
        // ---- the cell's weights: two tiles on their way in registers, two in LDS
        Loader<TYPE, NV, AL> ld;
        ld.stride = (uint32_t) pm_rows_stride<TYPE>(nb); ld.base = job.W + (long) r0 * ld.stride; ld.dT = p.dT; ld.smem = smem;
        ld.qT = p.qT + lane * 16; ld.bsT = p.bsT + lane * 16; ld.dt0 = 4 * (lane & 7);
        ld.lane = lane; ld.nb = nb; ld.npair = npair; ld.lim = lim; ld.rl = rl; ld.rgi = rgi; ld.kp = kp; ld.cell = cell; ld.n = n; ld.nround = nround; ld.kl = 2 - rl; ld.HS = HS;
        ld.in = {0, 0}; ld.hin = {0, 0}; ld.pa = {0, 0}; ld.hf = ld.at = ld.pf = 0; ld.pb = 1;
        Tile<TYPE> T0, T1;
        u32x4 a[Loader<TYPE, NV, AL>::NPL];
        ld.rows_of();
        ld.template load<false>(T0);
        if constexpr (AL) ld.load_a(a);
        u32x4 h[4] = {}; uint32_t d[4] = {};                         // the first block of scales
#pragma unroll
        for (int f = 0; f < HP<TYPE, NV, AL>; ++f) if (f < HS) ld.load_h(h[f], d[f], {0, 0}, (f << ld.kl) + kp);
        ld.hin.j = HS;
#pragma unroll
        for (int k = 0; k < 4; ++k) if (ld.hin.j >= n) { ld.hin.j -= n; ++ld.hin.rd; }
        ld.template load<true>(T1);
        PIN;
        ld.template put<false>(T0, 0);
        int pair = 0;
        if constexpr (AL) ld.put_a(a, 0, 0);
#pragma unroll
        for (int f = 0; f < HP<TYPE, NV, AL>; ++f) if (f < HS) ld.put_h(h[f], d[f], 0, (f << ld.kl) + kp);
        // (up to two steps have no third tile: the products don't wait until its requests, for nothing, are out. Q6_K 10240 x 1536 at 8 tokens 10.5 us, now 9.8)
        if (total <= 2) meet();
        if constexpr (AL) { PIN; ld.load_a(a); }
        PIN;
        ld.template load<true>(T0);
        if (total > 2) meet();
        auto step = [&](Tile<TYPE> & T, int s) __attribute__((always_inline)) {     // (s: where the next tile goes)
            PIN;
            ld.template put<true>(T, s);
            if constexpr (AL) { if (++pair == n) pair = 0; ld.put_a(a, s, pair); PIN; ld.load_a(a); }
            PIN;
            ld.template load<true>(T);
            PIN;
            meet();
            if (n == 1) meet();
        };
        for (int s = 1; s < total; s += 2) {
            step(T1, 1);
            if (s + 1 >= total) break;
            step(T0, 0);
        }
        meet();                                                     // the last tiles' products
        if (n == 1) meet();
        return;
    }
    // ---- products: wave (cell, half of a pair)
    const int par = wave >> 2, r = lane & 31, g = lane >> 5;
    constexpr int RT = 32 / PACK<NV>, P = PACK<NV>;
    const int tq = r / RT, tt = r % RT;
    ASrc as;
    ASet<TYPE, NV> A = {};
    if constexpr (!AL) {
        const bool on = P > 1 ? tt < p.T : r < 2 * NV, on_b = r < 2 * NV;
        as.n = nb;
        as.rq = __builtin_amdgcn_make_buffer_rsrc((void *) p.qT, 0, nb * (Q80 ? 1024 : 8192), 0x00020000);
        as.rb = __builtin_amdgcn_make_buffer_rsrc((void *) p.bsT, 0, Q80 ? 0 : nb * 1024, 0x00020000);
        as.qo = on ? (uint32_t) (tq * 1024 + (32 * g + tt) * 16) : 0x80000000u;
        as.bo = on_b ? (uint32_t) (lane * 16) : 0x80000000u;
#pragma unroll
        for (int k = 0; k < NA<TYPE, NV>; ++k) load_a<TYPE, NV>(A, as, min(kp, npair - 1), par, k);
    }
    const f32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    f32x16 out = zero;
    float * const red = (float *) (smem + L::RED);
    meet();
    int i = 0, rd = 0, hb = 0, hf = 0;
    for (int s = 0; s < total; ++s) {
        const bool last = i + 1 == n;
        const int nxt = min(kp + KP * (last ? 0 : i + 1), npair - 1);
        if (32 * ((rd << rl) + rgi) <= lim) {
            const uint8_t * S = smem + (2 * cell + (s & 1)) * L::SLOT, * AS = smem + L::ACT + (s & 1) * a_bytes<TYPE, NV>();
            constexpr int CH = F::HU / 16 * HP<TYPE, NV, AL>, hp = HP<TYPE, NV, AL>;
            const int e = hf * KP + kp;
            const uint8_t * H = smem + L::HDR + (2 * rgi + hb) * L::H, * dd = smem + L::DD + (2 * rgi + hb) * L::D + r * (4 * hp) + e * 4 + par * 2;
            if constexpr (Q80) H += r * (CH * 16) + ((e ^ (r & (CH - 1))) << 4) + 8 * par;
            else if constexpr (F::HU != 0) H += r * (CH * 16) + (((2 * e + par) ^ (r & (CH - 1))) << 4);
            const float * ds = (const float *) (AL ? AS + a_bytes<TYPE, NV>() - F::DT : S + F::SLOT) + (Q80 ? 128 : 32) * par;
            // this half's operands (AL): sub-blocks of 2 x 2 NV pieces; the second half of them behind the first's use
            auto operand = [&](int k) __attribute__((always_inline)) {
                const int sub0 = (F::SUBS / 2) * par, lt = P > 1 ? tt : min(tt, 2 * NV - 1);
                return *(const u32x4 *) (AS + ((sub0 + k * P + tq) * 4 * NV + g * 2 * NV + lt) * 16);
            };
            if constexpr (AL) {
                const int lb = min(r, 2 * NV - 1);
#pragma unroll
                for (int k = 0; k < (F::SUBS / 2 / P + 1) / 2; ++k) A.q[k] = operand(k);
                if constexpr (!Q80) A.bs = *(const u32x4 *) (AS + ((F::SUBS + par) * 4 * NV + g * 2 * NV + lb) * 16);
            }
            products<TYPE, NV>(A, S, H, dd, ds, par, r, g, out, [&](int k) __attribute__((always_inline)) {
                constexpr int NO = F::SUBS / 2 / P, H0 = (NO + 1) / 2;
                if constexpr (!AL) load_a<TYPE, NV>(A, as, nxt, par, k);
                else if (k < NO - H0) A.q[H0 + k] = operand(H0 + k);
            });
        }
        if (++hf == HS) { hf = 0; hb ^= 1; }
        if (last) {
            if constexpr (AL) {
                if (par) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) red[(cell * NV + v) * 64 + lane] = out[v];
                }
            } else {
#pragma unroll
                for (int v = 0; v < NV; ++v) red[(wave * NV + v) * 64 + lane] = out[v];
            }
        }
        meet();
        if (last) {
            // sums over pairs and halves in a fixed order
            const int base = 32 * (rd << rl);
            if constexpr (AL) {
                if (!par) {
                    float * mine = red + cell * NV * 64 + lane;
#pragma unroll
                    for (int v = 0; v < NV; ++v) mine[v * 64] += out[v];
                    const int row = base + 32 * rgi + r;
#pragma unroll 2
                    for (int v = 0; v < NV; ++v) {
                        const int t = 8 * (v >> 2) + 4 * g + (v & 3);
                        store<EPI>(p, job, ji, mine[v * 64], t, r0 + min(row, lim), t < p.T && row <= lim);
                    }
                }
            } else {
                for (int x = wave; x < RG * NV; x += CW) {           // results (row group, register) one after the other to the waves
                    const int gi = x / NV, v = x - gi * NV;
                    const int t = 8 * (v >> 2) + 4 * g + (v & 3), row = base + 32 * gi + r;
                    float sum = 0.0f;
                    for (int k = 0; k < KP; ++k)
#pragma unroll
                        for (int h = 0; h < 2; ++h) sum += red[((4 * h + gi + (k << rl)) * NV + v) * 64 + lane];
                    store<EPI>(p, job, ji, sum, t, r0 + min(row, lim), t < p.T && row <= lim);
                }
            }
            out = zero;
            i = 0; ++rd;
        } else ++i;
        if (n == 1) meet();
    }
}
// rows of workgroup w: `each`, and one more for the first `more` of them (in pairs for the rotation: they stay inside a workgroup)
template <int TYPE, int NV, bool EPI>
__device__ __forceinline__ void mmq_mid_rows(const RowsP & p, const RowsJob & job, int w, int ji, uint8_t * smem) {
    constexpr int STEP = EPI ? 2 : 1;
    const int r0 = STEP * (w * job.each + min(w, job.more)), r1 = STEP * ((w + 1) * job.each + min(w + 1, job.more));
    const int most = STEP * (job.each + (job.more != 0));          // of the matrix' workgroups: one order of the sums for all its rows
    const int groups = (most + 31) / 32;
    // five or six: rounds of four leave three or two cells without rows every other round; in rounds of two, us of rounds of four / here: Q4_K 33024 x 5120 at 8 tokens 32.6 / 25.3, 36864 x 14336
    // 73 / 54, Q6_K 36864 x 8192 at 24 tokens 86 / 73 (the other lengths and numbers of tokens alike). Three: longer rows of Q4_K over up to 8 tokens, which have little to gain from activations in
    // LDS, one group after the other: 17000 x 14336 34.7 / 31.1, 20480 x 5120 18.7 / 17.2 (512 .. 2048 values 0.84 .. 1.0 of that here, more tokens and Q6_K 0.85 .. 0.95)
    if (TYPE == PM_Q4_K && NV == 4 && groups == 3 && p.K > 4096) mmq_mid_body<TYPE, NV, EPI, false>(p, job, r0, r1, 0, ji, smem);
    else if (groups > 2 && groups != 5 && groups != 6) mmq_mid_body<TYPE, NV, EPI, true>(p, job, r0, r1, 2, ji, smem);
    else mmq_mid_body<TYPE, NV, EPI, false>(p, job, r0, r1, groups > 1 ? 1 : 0, ji, smem);
}

// (TA: the type of all jobs but the last, TB: of the last one; the leading arguments: pm_rows_args)
template <int TA, int TB, int NV, bool EPI>
__global__ __launch_bounds__(NT, 3) void mmq_mid_kernel(const uint8_t * W0, const uint8_t * W1, const uint8_t * W2, const uint8_t * qT, uint32_t first, uint32_t rows0, uint32_t rows1, uint32_t rows2, int K,
                                                        uint32_t tokens, RowsP args) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const RowsStart s = pm_rows_start(W0, W1, W2, first, rows0, rows1, rows2, (int) blockIdx.x);
    RowsP p = args;
    pm_rows_take(p, qT, K, tokens);
    RowsJob job = args.job[s.ji];
    job.W = s.W; job.each = s.each; job.more = s.more;
    if (TA == TB || s.ji < p.njobs - 1) mmq_mid_rows<TA, NV, EPI>(p, job, s.w, s.ji, smem);
    else mmq_mid_rows<TB, NV, EPI>(p, job, s.w, s.ji, smem);
}

template <int TYPE> size_t lds_of(int nv) {
    auto most = [](auto v) { constexpr int NV = decltype(v)::value; static_assert(Lds<TYPE, NV, true>::BYTES <= 160 * 1024 && Lds<TYPE, NV, false>::BYTES <= 160 * 1024, "LDS");
                             return (size_t) std::max(Lds<TYPE, NV, true>::BYTES, Lds<TYPE, NV, false>::BYTES); };
    return nv == 4 ? most(std::integral_constant<int, 4>()) : nv == 8 ? most(std::integral_constant<int, 8>()) : nv == 12 ? most(std::integral_constant<int, 12>()) : most(std::integral_constant<int, 16>());
}
size_t lds_of(int type, int nv) { return type == PM_Q4_K ? lds_of<PM_Q4_K>(nv) : type == PM_Q5_K ? lds_of<PM_Q5_K>(nv) : type == PM_Q6_K ? lds_of<PM_Q6_K>(nv) : lds_of<PM_Q8_0>(nv); }

}  // namespace

int pm_launch_mmq_mid(RowsP p, const int * types, hipStream_t st) {
    if (p.t_off) return -5;                                            // (a pass starts with its tables)
    const int cus = pm_device_cus(), n = p.njobs;
    const int ta = types[0], tb = types[n - 1];
    double bytes[3], all = 0;
    for (int j = 0; j < n; ++j) all += bytes[j] = (double) p.job[j].N * pm_weight_row_stride(types[j], p.K);
    // workgroups by weight bytes, of at least 32 rows each
    const int unit = p.e_on ? 2 : 1;                                   // (N is even then)
    int at = 0, first[3] = {0, INT32_MAX, INT32_MAX}, nw[3] = {};
    auto groups = [&](int j, int w) { return (unit * ((p.job[j].N / unit + w - 1) / w) + 31) / 32; };      // of the longest slice
    for (int j = 0; j < n; ++j) {
        const int most = (p.job[j].N + 31) / 32;
        int want = j == n - 1 && n > 1 ? cus - at : (int) (cus * bytes[j] / all + 0.5);
        if (want > cus - at - (n - 1 - j)) want = cus - at - (n - 1 - j);
        at += nw[j] = want < 1 ? 1 : want > most ? most : want;
    }
    // Slices of the last job that are a row or two longer than whole groups take a group's steps more for them: a few workgroups of the first job then, where its own slices keep their groups
    // (wq | wk | wv of Q4_K, Q4_K, Q5_K, 8192 + 1024 + 1024 x 8192: wv in 31 slices of up to 34 rows 20.4 us at 12 tokens, in 32 of 32 14.9)
    if (const int g = n > 1 ? groups(n - 1, nw[n - 1]) : 1; g > 1) {
        const int up = (p.job[n - 1].N + 32 * (g - 1) - 1) / (32 * (g - 1)), more = up - nw[n - 1];
        if (16 * more <= nw[n - 1] && more < nw[0] && groups(0, nw[0] - more) == groups(0, nw[0]) && groups(n - 1, up) < g) { nw[0] -= more; nw[n - 1] = up; }
    }
    at = 0;
    for (int j = 0; j < n; ++j) {
        RowsJob & b = p.job[j];
        first[j] = at; at += nw[j];
        b.each = b.N / unit / nw[j]; b.more = b.N / unit % nw[j];
    }
    const int nv = p.T <= 8 ? 4 : p.T <= 16 ? 8 : p.T <= 24 ? 12 : 16;
    if (!pm_rows_fit(p)) return -5;
    const size_t lds = std::max(lds_of(ta, nv), lds_of(tb, nv));
    auto go = [&](auto kern) {
        pm_allow_big_lds((const void *) kern, lds);
        const RowsArgs a = pm_rows_args(p, first[1], first[2]);
        hipLaunchKernelGGL(kern, dim3(at), dim3(NT), lds, st, p.job[0].W, p.job[1].W, p.job[2].W, p.qT, a.first, a.rows[0], a.rows[1], a.rows[2], p.K, a.tokens, p);
        return 0;
    };
#define PM_MID_V(TA_, TB_, E_) { return nv == 4 ? go(mmq_mid_kernel<TA_, TB_, 4, E_>) : nv == 8 ? go(mmq_mid_kernel<TA_, TB_, 8, E_>) : nv == 12 ? go(mmq_mid_kernel<TA_, TB_, 12, E_>) : go(mmq_mid_kernel<TA_, TB_, 16, E_>); }
    if (p.e_on) {
        if (ta == PM_Q4_K && tb == PM_Q4_K) PM_MID_V(PM_Q4_K, PM_Q4_K, true)
        if (ta == PM_Q6_K && tb == PM_Q6_K) PM_MID_V(PM_Q6_K, PM_Q6_K, true)
        if (ta == PM_Q4_K && tb == PM_Q6_K) PM_MID_V(PM_Q4_K, PM_Q6_K, true)
        if (ta == PM_Q4_K && tb == PM_Q5_K) PM_MID_V(PM_Q4_K, PM_Q5_K, true)
        return -5;
    }
    if (ta == PM_Q4_K && tb == PM_Q4_K) PM_MID_V(PM_Q4_K, PM_Q4_K, false)
    if (ta == PM_Q6_K && tb == PM_Q6_K) PM_MID_V(PM_Q6_K, PM_Q6_K, false)
    if (ta == PM_Q5_K && tb == PM_Q5_K) PM_MID_V(PM_Q5_K, PM_Q5_K, false)
    if (ta == PM_Q8_0 && tb == PM_Q8_0) PM_MID_V(PM_Q8_0, PM_Q8_0, false)
    if (ta == PM_Q4_K && tb == PM_Q6_K) PM_MID_V(PM_Q4_K, PM_Q6_K, false)
    if (ta == PM_Q4_K && tb == PM_Q5_K) PM_MID_V(PM_Q4_K, PM_Q5_K, false)
#undef PM_MID_V
    return -5;
}
