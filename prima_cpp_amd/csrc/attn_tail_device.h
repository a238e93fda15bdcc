// attn_tail_device.h — single-token attention over cached cells for callers INSIDE a launch that also produced q and this token's cell
// (the QKV launch's tail: mmvq.hip; the persistent engine's attention phase: decode_engine.hip). The arithmetic, its order and its rounding points are
// attn_cached.hip's (ggml.c:12445-12473 K.q rows, :13783-13879 soft_max, F16-rounded probabilities against the F16 V rows: the reference's
// ggml_compute_forward_mul_mat with an F16 src1 conversion) - the outputs are the same bits as attn_cached.hip's OF THE SAME ROUND (up to 256 cells both take attn_whole_lines below);
// what differs is how memory is read: q and the newest
// cell were written by OTHER compute units in this launch, so every load of q / K / V bypasses this XCD's caches (sc0 sc1).
#pragma once
#include "pm355_device.h"

// ---- coherent buffer loads: tracked by the compiler's waitcnt logic, 16 bytes per instruction. `sc0 sc1` (aux 17), not `sc1` alone: a buffer that is
// handed over more than once per launch (the residual stream, q, the attention output, the ffn activation, the partial sums - every layer re-uses
// them) may still sit in THIS XCD's L2 from the previous layer's read, and an sc1 load is served from there: two 70B layers differed by 1e-4 from
// the five launches, one layer by 1e-14 (found on the hardware). The write side stays sc1 write-through (st_act<true>). --------------------------
__device__ __forceinline__ __amdgpu_buffer_rsrc_t coh_rsrc(const void * base) { return __builtin_amdgcn_make_buffer_rsrc((void *) base, 0, 0x7FFFFFF0, 0x00020000); }
__device__ __forceinline__ float4 coh_ld16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    // (the whole vector is re-typed at once: element-wise __builtin_bit_cast(float, t[i]) of the loaded vector compiles to a ONE-dword load that
    //  feeds all four components - ROCm 7.2 clang; found on the hardware, tools/r5)
    const f32x4 t = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int) off, 0, 17));
    return make_float4(t.x, t.y, t.z, t.w);
}
__device__ __forceinline__ u32x4 coh_ld16u(__amdgpu_buffer_rsrc_t r, uint32_t off) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int) off, 0, 17)); }
__device__ __forceinline__ float coh_ld4(__amdgpu_buffer_rsrc_t r, uint32_t off) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int) off, 0, 17)); }


// ---- up to 64 * KPL cells, four waves per head: every load is issued before anything is computed, ONE barrier. What bounds it is the number of cache lines a CU asks for, so an instruction
// takes whole lines: K - DH / 8 lanes hold a key's row, a wave 4 keys of head_dim 128 at once; V^T - 8 KPL lanes hold a dimension's cells, eight each. (A key per lane, and a dimension per
// lane for V - 64 lines an instruction, 8192 for a head of 128 over 256 cells instead of 1024: 7.9 us per launch of 32 heads x 204 cells, now 5.0; 4.3 at 36 cells, now 3.8.)
// Rounding points as everywhere: q, K, V F16, the normalised probabilities rounded to F16, f32 accumulation. n_kv <= 64 * KPL, n_ctx a multiple of 8; DH 64 / 128 (256: KPL = 1).
// COH: q / K / V through cache-bypassing loads, the output written through (callers inside a launch that produced them: attn_tail_head below).
// part: LDS [64 * KPL] floats, pw: [4][64 * KPL]; bar(): barrier of exactly the four waves.
template <int DH, int KPL, bool COH, class Bar>
__device__ __forceinline__ void attn_whole_lines(const float * q_head, const uint16_t * kc, const uint16_t * vc, float * out_head, int hk, int Hkv, int n_ctx, int n_kv,
                                                 float scale, const void * mask, int mask_f16, float * part, float * pw, int lane, int wave, Bar && bar) {
    constexpr int NKEY = 64 * KPL, LPK = DH / 8, KPI = 64 / LPK, NI = NKEY / (4 * KPI), LV = 8 * KPL, DPI = 64 / LV, NV = DH / 4 / DPI, LR = LV < 16 ? LV : 16;
    static_assert(NI <= LPK && NV <= LR, "a lane keeps one result of each kind");
    u32x4 kreg[NI], vreg[NV];
    const __amdgpu_buffer_rsrc_t rk = coh_rsrc(kc), rv = coh_rsrc(vc), rq = coh_rsrc(q_head);
    const int kd = lane % LPK, ks = lane / LPK, c = lane % LV, ve = lane / LV;
    f32x4 q[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        if constexpr (COH) q[j] = __builtin_bit_cast(f32x4, coh_ld16u(rq, (uint32_t) ((8 * kd + 4 * j) * 4)));
        else q[j] = *(const PM_G f32x4 *) (q_head + 8 * kd + 4 * j);
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const long off = (long) min(KPI * (4 * i + wave) + ks, n_kv - 1) * Hkv * DH + (long) hk * DH + 8 * kd;
        if constexpr (COH) kreg[i] = coh_ld16u(rk, (uint32_t) (off * 2));
        else kreg[i] = *(const PM_G u32x4 *) (kc + off);
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const long off = (long) (hk * DH + DH / 4 * wave + DPI * i + ve) * n_ctx + (8 * c < n_kv ? 8 * c : 0);
        if constexpr (COH) vreg[i] = coh_ld16u(rv, (uint32_t) (off * 2));
        else vreg[i] = *(const PM_G u32x4 *) (vc + off);
    }
    float m_add[KPL];
#pragma unroll
    for (int k = 0; k < KPL; ++k) {
        const int key = lane + 64 * k;
        m_add[k] = (mask && key < n_kv) ? (mask_f16 ? h2f(((const PM_G uint16_t *) mask)[key]) : ((const PM_G float *) mask)[key]) : 0.0f;
    }
    // scores: lane kd of a key's lanes keeps the one of instruction kd
    float keep = 0.0f;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        float acc = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t w = kreg[i][t];
            acc = fmaf(h2f((uint16_t) (w & 0xFFFF)), q[t >> 1][2 * (t & 1)], acc);
            acc = fmaf(h2f((uint16_t) (w >> 16)), q[t >> 1][2 * (t & 1) + 1], acc);
        }
        acc += dpp_f<0xB1>(acc); acc += dpp_f<0x4E>(acc); acc += dpp_f<0x141>(acc);
        if constexpr (LPK >= 16) acc += dpp_f<0x140>(acc);
        if constexpr (LPK >= 32) acc += __builtin_bit_cast(float, other_row(__builtin_bit_cast(uint32_t, acc)));
        keep = kd == i ? acc : keep;
    }
    if (kd < NI) part[KPI * (4 * kd + wave) + ks] = keep;
    bar();
    float s_[KPL], mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < KPL; ++k) {
        const int key = lane + 64 * k;
        s_[k] = key < n_kv ? part[key] * scale + m_add[k] : -INFINITY;
        mx = fmaxf(mx, s_[k]);
    }
    mx = all_max(mx);
    float ex[KPL];
    double tot = 0.0;
#pragma unroll
    for (int k = 0; k < KPL; ++k) { ex[k] = lane + 64 * k < n_kv ? expf(s_[k] - mx) : 0.0f; tot += (double) ex[k]; }
    const float inv = (float) (1.0 / all_sum(tot));
#pragma unroll
    for (int k = 0; k < KPL; ++k) pw[wave * NKEY + lane + 64 * k] = h2f(f2h(ex[k] * inv));        // p rounded to F16 (src1 of the V^T.p product)
    __builtin_amdgcn_wave_barrier();                       // (a wave's LDS accesses execute in order: its own copy needs no workgroup barrier)
    const f32x4 p0 = *(const f32x4 *) (pw + wave * NKEY + 8 * c), p1 = *(const f32x4 *) (pw + wave * NKEY + 8 * c + 4);
    keep = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        float o = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t w = vreg[i][t];
            const f32x4 & p = t < 2 ? p0 : p1;
            o = fmaf(h2f((uint16_t) (w & 0xFFFF)), p[2 * (t & 1)], o);
            o = fmaf(h2f((uint16_t) (w >> 16)), p[2 * (t & 1) + 1], o);
        }
        o += dpp_f<0xB1>(o); o += dpp_f<0x4E>(o); o += dpp_f<0x141>(o);
        if constexpr (LV >= 16) o += dpp_f<0x140>(o);
        keep = lane % LR == i ? o : keep;
    }
    if constexpr (LV == 32) keep += __builtin_bit_cast(float, other_row(__builtin_bit_cast(uint32_t, keep)));
    if (lane % LR < NV && (LV < 32 || !(lane & 16))) st_act<COH>(out_head + DH / 4 * wave + DPI * (lane % LR) + ve, keep);
}

struct AttnTailP {
    const float * q; const uint16_t * kc, * vc; const int32_t * pos, * seq; long seq_stride; float * out;
    int H, Hkv, n_ctx; float scale;
};
// LDS bytes of the body for head_dim DH and up to max_keys cells: part[4][256] / pw[4][256] / reductions | qs[DH] | part[256] | sc[max_keys + 8]
static inline __host__ __device__ size_t attn_tail_lds(int dh, int max_keys) { return (size_t) (2048 + 8 + 8) * 4 + (size_t) (dh + 256 + ((max_keys + 15) & ~7)) * 4; }

// head h by FOUR waves (threads 0 .. 255 of the caller's workgroup); bar() = a barrier of exactly those four waves that also orders their LDS traffic.
// attn_cached.hip's short form (up to 256 cells, one barrier) and the cached form of attn_rope_body beyond.
template <int DH, class Bar>
__device__ __forceinline__ void attn_tail_head(const AttnTailP & a, int h, char * smem, Bar && bar) {
    // (the thread id goes through an opaque asm: everything derived from it - dozens of LDS / cache offsets - is then recomputed here instead of being
    //  hoisted to the caller's entry and kept alive, i.e. spilled, across its row loops)
    int tid_ = threadIdx.x;
    asm volatile("" : "+v"(tid_));
    const int tid = tid_, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.H, Hkv = a.Hkv, n_ctx = a.n_ctx;
    const int hk = h / (H / Hkv);
    const float scale = a.scale;
    const int seq = a.seq ? uniform_const_ptr(a.seq)[0] : 0;
    const int n_kv = uniform_const_ptr(a.pos)[seq] + 1;
    const long soff = (long) seq * a.seq_stride;
    const __amdgpu_buffer_rsrc_t rk = coh_rsrc(a.kc + soff), rv = coh_rsrc(a.vc + soff), rq = coh_rsrc(a.q);
    float * part = (float *) smem;                         // [4][256]
    float * pw = part + 1024;                              // [4][256]
    float * redf = pw + 1024;                              // [8]
    double * redd = (double *) (redf + 8);                 // [4]
    float * body = (float *) (redd + 4);                   // general path: qs[DH] | part[256] | sc[max_keys]
    // ---- up to 256 cells (the same function attn_cached.hip calls: same bits)
    const float * qh = a.q + (long) h * DH;
    float * oh = a.out + (long) h * DH;
    if (n_kv <= 64) { attn_whole_lines<DH, 1, true>(qh, a.kc + soff, a.vc + soff, oh, hk, Hkv, n_ctx, n_kv, scale, nullptr, 0, part, pw, lane, wave, bar); return; }
    if constexpr (DH <= 128) {
        if (n_kv <= 128) { attn_whole_lines<DH, 2, true>(qh, a.kc + soff, a.vc + soff, oh, hk, Hkv, n_ctx, n_kv, scale, nullptr, 0, part, pw, lane, wave, bar); return; }
        if (n_kv <= 256) { attn_whole_lines<DH, 4, true>(qh, a.kc + soff, a.vc + soff, oh, hk, Hkv, n_ctx, n_kv, scale, nullptr, 0, part, pw, lane, wave, bar); return; }
    }
    // ---- general cached body (attn_rope_body<DH, COH, 0, true>): thread per key, three 4-wave reductions
    constexpr int PARTS = 256 / DH, KQ = DH / 8;
    float * qs = body, * part2 = qs + DH, * sc = part2 + 256;
    if (tid < DH) qs[tid] = coh_ld4(rq, (uint32_t) (((long) h * DH + tid) * 4));
    const int ve = tid % DH, vpt = tid / DH;
    const int n_pad = (n_kv + 7) & ~7;
    bar();
    float lmax = -INFINITY;
#pragma unroll 1
    for (int i = tid; i < n_kv; i += 256) {
        // (the key's row in two halves: same accumulation order as one pass, half the registers)
        float acc = 0.0f;
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            u32x4 kk[KQ / 2];
#pragma unroll
            for (int j = 0; j < KQ / 2; ++j) kk[j] = coh_ld16u(rk, (uint32_t) (((long) i * Hkv * DH + (long) hk * DH + 8 * (hf * (KQ / 2) + j)) * 2));
#pragma unroll
            for (int jj = 0; jj < KQ / 2; ++jj)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    acc += h2f((uint16_t) (kk[jj][j] & 0xFFFF)) * qs[8 * (hf * (KQ / 2) + jj) + 2 * j];
                    acc += h2f((uint16_t) (kk[jj][j] >> 16)) * qs[8 * (hf * (KQ / 2) + jj) + 2 * j + 1];
                }
        }
        const float s_ = acc * scale;
        sc[i] = s_;
        lmax = fmaxf(lmax, s_);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) lmax = fmaxf(lmax, __shfl_xor(lmax, off));
    if (lane == 0) redf[wave] = lmax;
    bar();
    const float mx = fmaxf(fmaxf(redf[0], redf[1]), fmaxf(redf[2], redf[3]));
    double lsum = 0.0;
    for (int i = tid; i < n_kv; i += 256) {
        const float e = expf(sc[i] - mx);
        sc[i] = e;
        lsum += (double) e;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off);
    if (lane == 0) redd[wave] = lsum;
    bar();
    const double tot = (redd[0] + redd[1]) + (redd[2] + redd[3]);
    const float inv = (float) (1.0 / tot);
    bar();
    for (int i = tid; i < n_pad; i += 256) sc[i] = i < n_kv ? h2f(f2h(sc[i] * inv)) : 0.0f;
    bar();
    {
        float acc = 0.0f;
        const long vrow = (long) (hk * DH + ve) * n_ctx;
#pragma unroll 1
        for (int i = vpt * 8; i < n_pad; i += PARTS * 8) {
            const u32x4 vv = coh_ld16u(rv, (uint32_t) ((vrow + i) * 2));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc += h2f((uint16_t) (vv[j] & 0xFFFF)) * sc[i + 2 * j];
                acc += h2f((uint16_t) (vv[j] >> 16)) * sc[i + 2 * j + 1];
            }
        }
        part2[tid] = acc;
    }
    bar();
    if (tid < DH) {
        float acc = 0.0f;
#pragma unroll
        for (int pt = 0; pt < PARTS; ++pt) acc += part2[pt * DH + tid];
        st_act<true>(a.out + (long) h * DH + tid, acc);
    }
}

