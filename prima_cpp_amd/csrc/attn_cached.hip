// attn_cached.hip — single-token attention over cells that are ALL in the cache, for the decode path whose wq | wk | wv launch has
// already applied RoPE, rounded q to F16 and stored the token's K row / V column (QkvEpi, mmvq_device.h), plus the per-token
// cos / sin table that launch reads.
//
// Replaces (with the QKV epilogue) the same reference nodes as attn_rope_fused_kernel: ROPE x2 (ggml.c:14143), CPY F32->F16 x2
// (llm_build_kv_store, src/llama.cpp:9673-9718), MUL_MAT(K, q) with q converted to F16 (ggml.c:12445-12473), SOFT_MAX_EXT
// (ggml.c:13783-13879), MUL_MAT(V^T, p) with p converted to F16, same rounding points.
//
// Why a second kernel: at short contexts the fused kernel is a chain of dependent latencies (position -> rope -> LDS -> barrier ->
// 128-term dot per THREAD -> two block reductions -> P.V -> reduction): 7.4 us per 70B layer for ~0 bytes. Here
//   * up to 256 cells (head sizes up to 128; 64 cells for 256), where the cache has as many as the form takes: attn_short, every load issued first, ONE workgroup barrier.
//   * the rest (up to the long-context threshold): the per-head body of attn_device.h in its CACHED form.
#include "attn_device.h"
#include "pm355_kernels.h"
#include "pm355_layer_ops.h"
#include "pm355_q8k.h"
#include <algorithm>
#include <type_traits>

namespace {

// this token's (cos, sin) per rotation pair: one launch per token serves every layer's wq | wk | wv epilogue
__global__ __launch_bounds__(128) void rope_table_kernel(RopeP r, const int32_t * pos_ptr, const int32_t * seq_ptr, const float * freq_factors, float * tab, int rows) {
    // (blockIdx.x: token of a small batch, its table n_dims floats further on)
    const int pos = rows ? pos_ptr[blockIdx.x] : pos_ptr[seq_ptr ? *seq_ptr : 0] + (int) blockIdx.x;
    tab += (size_t) blockIdx.x * r.n_dims;
    for (int pair = threadIdx.x; pair < r.n_dims / 2; pair += blockDim.x) {
        float c, s;
        rope_cs(r, (float) pos, pair, freq_factors, c, s);
        tab[2 * pair] = c; tab[2 * pair + 1] = s;
    }
}

// What a wave of attn_short stages, bytes: rows of 16 KPL keys, then the same memory for its DH / 4 rows of V^T (16 bytes more than the data: consecutive rows start 4 banks on)
template <int DH, int KPL> struct ShortLds {
    static constexpr int K_PITCH = 2 * DH + 16, V_PITCH = 128 * KPL + 16, K = 16 * KPL * K_PITCH, V = DH / 4 * V_PITCH, STAGE = K > V ? K : V;
    static constexpr int BYTES = 64 * KPL * (4 + 4 * 2) + 4 * (STAGE + DH * 4);   // scores | probabilities of each wave | q and stage of each wave
};
// Up to 64 * KPL cells, four waves per head. What bounds it is the number of cache lines a CU asks for, so an instruction takes whole lines: K - DH / 8 lanes hold a key's row, V^T - 8 KPL lanes a
// dimension's cells - a wave a quarter of the keys and a quarter of the dimensions. They are multiplied out of LDS, which a wave fills for itself (no barrier): the sums of a decoded token stay
// what a lane per key and a lane per dimension make them - the dimensions of a quarter in a row, the quarters as (0 + 1) + (2 + 3); the cells of a dimension in 64 / (DH / 4) rows, one lane each.
// us per launch of 32 heads of 128 over 36 / 100 / 204 cells: a lane's own key and dimension straight from memory 3.3 / 4.4 / 7.0, this 2.8 / 3.7 / 5.7 (multiplied in the registers that the
// lines arrive in, sums over lanes, 2.6 / 3.1 / 4.5: one other bit here turns 8-bit roundings behind it, 3 % of the logits of eight layers of the 8B shape).
// Rounding points as everywhere: q, K, V F16, the normalised probabilities rounded to F16, f32 accumulation. n_kv <= 64 * KPL <= n_ctx; DH 64 / 128 (256: KPL = 1).
// out: the head's result in memory, or a function of (dimension, value).
template <int DH, int KPL, class Out>
__device__ __forceinline__ void attn_short(const float * q_head, const uint16_t * kc, const uint16_t * vc, Out out, int hk, int Hkv, int n_ctx, int n_kv, float scale, const void * mask,
                                           int mask_f16, char * smem, int lane, int wave, unsigned long long * ts) {
    unsigned long long tsv[6] = {PM_TS_NOW(), 0, 0, 0, 0, 0};
    typedef ShortLds<DH, KPL> S;
    constexpr int NKEY = 64 * KPL, NKW = NKEY / 4, LPK = DH / 8, KPI = 64 / LPK, NI = NKW / KPI, DPW = DH / 4, LV = 8 * KPL, DPI = 64 / LV, NV = DPW / DPI, KPP = NKEY * DPW / 64;
    float * const part = (float *) smem, * const qs = (float *) (smem + 12 * NKEY) + DH * wave;
    uint16_t * const pw = (uint16_t *) (part + NKEY) + NKEY * wave;
    char * const st = smem + 12 * NKEY + 4 * DH * 4 + S::STAGE * wave;
    const int kd = lane % LPK, ks = lane / LPK, c = lane % LV, ve = lane / LV;
    const f32x4 q4 = *(const PM_G f32x4 *) (q_head + 4 * (lane % DPW));
    u32x4 kreg[NI], vreg[NV];
#pragma unroll
    for (int i = 0; i < NI; ++i) kreg[i] = *(const PM_G u32x4 *) (kc + (long) max(min(KPI * (4 * i + wave) + ks, n_kv - 1), 0) * Hkv * DH + (long) hk * DH + 8 * kd);
#pragma unroll
    for (int i = 0; i < NV; ++i) vreg[i] = *(const PM_G u32x4 *) (vc + (long) (hk * DH + DPW * wave + DPI * i + ve) * n_ctx + (8 * c < n_kv ? 8 * c : 0));
    float m_add[KPL];
#pragma unroll
    for (int k = 0; k < KPL; ++k) m_add[k] = lane + 64 * k < n_kv ? attn_mask_at(mask, mask_f16, lane + 64 * k) : 0.0f;
    auto staged = []() __attribute__((always_inline)) {        // (a wave's LDS accesses execute in order: what it wrote is there for its other lanes, what it has read may be overwritten)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    if (lane < DPW) *(f32x4 *) (qs + 4 * lane) = q4;
#pragma unroll
    for (int i = 0; i < NI; ++i) *(u32x4 *) (st + (KPI * i + ks) * S::K_PITCH + 16 * kd) = kreg[i];
    staged();
    tsv[1] = PM_TS_NOW();                                      // loads back
    // ---- scores: lane = (key l of the wave, quarters u0 .. u0 + KPL - 1 of the head)
    const int l = lane % NKW, u0 = KPL * (lane / NKW);
    float acc[KPL];
#pragma unroll
    for (int u = 0; u < KPL; ++u) acc[u] = 0.0f;
#pragma unroll
    for (int j = 0; j < DPW / 8; ++j)
#pragma unroll
        for (int u = 0; u < KPL; ++u) {
            const int d = DPW * (u0 + u) + 8 * j;
            const u32x4 w = *(const u32x4 *) (st + l * S::K_PITCH + 2 * d);
            const f32x4 q[2] = {*(const f32x4 *) (qs + d), *(const f32x4 *) (qs + d + 4)};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                acc[u] = fmaf(h2f((uint16_t) (w[t] & 0xFFFF)), q[t >> 1][2 * (t & 1)], acc[u]);
                acc[u] = fmaf(h2f((uint16_t) (w[t] >> 16)), q[t >> 1][2 * (t & 1) + 1], acc[u]);
            }
        }
    float s = acc[0];
    if constexpr (KPL == 1) s += __builtin_bit_cast(float, other_row(__builtin_bit_cast(uint32_t, s)));
    else s += acc[1];
    if constexpr (KPL == 4) s += acc[2] + acc[3];
    else s += __builtin_bit_cast(float, other_half(__builtin_bit_cast(uint32_t, s)));
    if (lane < NKW) part[KPI * (4 * (l / KPI) + wave) + l % KPI] = s;
    staged();
#pragma unroll
    for (int i = 0; i < NV; ++i) *(u32x4 *) (st + (DPI * i + ve) * S::V_PITCH + 16 * c) = vreg[i];
    __syncthreads();                                           // the only workgroup barrier of this path
    tsv[2] = PM_TS_NOW();                                      // scores
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
    for (int k = 0; k < KPL; ++k) pw[lane + 64 * k] = f2h(ex[k] * inv);            // p rounded to F16 (src1 of the V^T.p product)
    staged();
    tsv[3] = PM_TS_NOW();                                      // softmax
    // ---- P.V: lane = (dimension e, part kp of the cells). Pieces without an attended cell repeat the row's first one, against probabilities of zero
    const int e = lane % DPW, kp = lane / DPW;
    float o = 0.0f;
#pragma unroll
    for (int j = 0; j < KPP / 8; ++j) {
        const u32x4 w = *(const u32x4 *) (st + e * S::V_PITCH + 2 * (KPP * kp + 8 * j));
        const u32x4 p = *(const u32x4 *) (pw + KPP * kp + 8 * j);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            o = fmaf(h2f((uint16_t) (w[t] & 0xFFFF)), h2f((uint16_t) (p[t] & 0xFFFF)), o);
            o = fmaf(h2f((uint16_t) (w[t] >> 16)), h2f((uint16_t) (p[t] >> 16)), o);
        }
    }
    tsv[4] = PM_TS_NOW();                                      // P.V
    if constexpr (DPW <= 16) o += __builtin_bit_cast(float, other_row(__builtin_bit_cast(uint32_t, o)));
    if constexpr (DPW <= 32) o += __builtin_bit_cast(float, other_half(__builtin_bit_cast(uint32_t, o)));
    if (lane < DPW) {
        if constexpr (std::is_pointer_v<Out>) st_g(out + DPW * wave + lane, o);
        else out(DPW * wave + lane, o);
    }
    tsv[5] = PM_TS_NOW();
    pm_ts_store(ts, 2, tsv);
}

// What leads to the first loads - positions and sequences, queries and caches, the KV head without a division - leads the arguments, in registers when a launch starts: inv = 2^32 / (heads per KV head),
// rounded up (0: one), how: 1 rows of several sequences, 2 a length from the graph (dyn). us, 8B shape: eight rows of up to 36 cells
// 5.05 / 4.77, 169 rows of prompts 24.6 / 22.2; a token of eight layers behind 203 cells 428.2 / 426.6 a pass
struct CachedArgs { uint32_t heads, inv; int how; };
static CachedArgs cached_args(const AttnP & a) {
    const uint64_t R = (uint64_t) (a.H / a.Hkv);
    return CachedArgs{(uint32_t) a.H | (uint32_t) a.Hkv << 16, R == 1 ? 0u : (uint32_t) (((1ull << 32) + R - 1) / R), (a.rows ? 1 : 0) | (a.dyn ? 2 : 0)};
}
__device__ __forceinline__ int kv_head(int h, uint32_t inv) { return inv ? (int) __umulhi((uint32_t) h, inv) : h; }      // (exact: heads x heads per KV head < 2^32)
// MANY: more heads than 16 bits of an argument hold, and the division
template <int DH, int VM, bool MANY = false>
__global__ __launch_bounds__(256) void attn_cached_kernel(const float * q0, uint16_t * kc0, uint16_t * vc0, const int32_t * pos0, const int32_t * seq0, uint32_t heads, uint32_t inv, int n_ctx0, int how, AttnP a_in) {
    // grid.y = tokens of a small batch (engine: 2..64-token steps after rope_kv_store has rotated / rounded q and stored every token's K / V):
    // token t attends cells [0, pos0 + t], its q / out rows are t * H * DH further on
    // (the leading arguments: CachedArgs; the rest, dyn and the output among them, is read behind the first loads)
    AttnP a = a_in;
    a.q = q0; a.kc = kc0; a.vc = vc0; a.pos0_ptr = pos0; a.seq_ptr = seq0; a.n_ctx = n_ctx0; a.rows = how & 1;
    if constexpr (!MANY) { a.H = (int) (heads & 65535); a.Hkv = (int) (heads >> 16); }
    a.tok = (int) blockIdx.y;
    a.q += (long) a.tok * a.H * DH; a.out += (long) a.tok * a.H * DH;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ float redf[8];
    __shared__ double redd[4];
    const int h = blockIdx.x;
    if constexpr (VM == 0) {
        const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int Hkv = a.Hkv, hk = MANY ? h / (a.H / Hkv) : kv_head(h, inv), n_ctx = a.n_ctx;
        int seq = 0, n_kv;
        if (how & 2) n_kv = uniform_const_ptr(a.dyn)[1];
        else {
            seq = a.seq_ptr ? uniform_const_ptr(a.seq_ptr)[a.rows ? a.tok : 0] : 0;
            n_kv = uniform_const_ptr(a.pos0_ptr)[a.rows ? a.tok : seq] + 1 + (a.rows ? 0 : a.tok);
        }
        const uint16_t * kc = a.kc + (long) seq * a.seq_stride, * vc = a.vc + (long) seq * a.seq_stride;
        auto go = [&](auto kpl) __attribute__((always_inline)) {
            attn_short<DH, decltype(kpl)::value>(a.q + (long) h * DH, kc, vc, a.out + (long) h * DH, hk, Hkv, n_ctx, n_kv, a.scale, a.mask, a.mask_f16, smem, lane, wave, a.ts);
        };
        // (caches that hold fewer cells than the form takes: the general body, as it always was - its sums are in another order)
        if (n_kv <= 64 && n_ctx >= 64) return go(std::integral_constant<int, 1>());
        if constexpr (DH <= 128) {
            if (n_kv <= 128 && n_ctx >= 128) return go(std::integral_constant<int, 2>());
            if (n_kv <= 256 && n_ctx >= 256) return go(std::integral_constant<int, 4>());
        }
    }
    attn_rope_body<DH, false, VM, true>(a, h, smem, redf, redd);
}

// The same for rows of up to 256 cells and two heads of 128 per workgroup, whose results meet in LDS and leave as a Q8_K block (the wo product's activations) - no f32 rows and no launch that
// quantizes them: 8 sequences of the 8B shape, 4.0 + 3.2 us and the gap between them, now 6.4
__global__ __launch_bounds__(512) void attn_cached_q8k_kernel(const float * q0, uint16_t * kc0, uint16_t * vc0, const int32_t * pos0, const int32_t * seq0, uint32_t heads, uint32_t inv, int n_ctx0, float scale0, AttnP a,
                                                              pm_q8k_out y) {
    a.q = q0; a.kc = kc0; a.vc = vc0; a.pos0_ptr = pos0; a.seq_ptr = seq0; a.H = (int) (heads & 65535); a.Hkv = (int) (heads >> 16); a.n_ctx = n_ctx0; a.scale = scale0;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ __attribute__((aligned(16))) float row[256];
    const int tid = threadIdx.x, lane = tid & 63, w8 = __builtin_amdgcn_readfirstlane(tid >> 6), half = w8 >> 2, wave = w8 & 3;
    const int t = blockIdx.y, blk = blockIdx.x, h = 2 * blk + half, hk = kv_head(h, inv), seq = uniform_const_ptr(a.seq_ptr)[t], n_kv = uniform_const_ptr(a.pos0_ptr)[t] + 1;
    auto go = [&](auto kpl) __attribute__((always_inline)) {     // (chosen by the row's own cells, as above: the sums do not depend on what else is in the batch)
        constexpr int KPL = decltype(kpl)::value;
        attn_short<128, KPL>(a.q + ((long) t * a.H + h) * 128, a.kc + (long) seq * a.seq_stride, a.vc + (long) seq * a.seq_stride, [&](int d, float v) __attribute__((always_inline)) { row[128 * half + d] = v; },
                             hk, a.Hkv, a.n_ctx, n_kv, a.scale, nullptr, 0, smem + ShortLds<128, KPL>::BYTES * half, lane, wave, nullptr);
    };
    if (n_kv <= 64) go(std::integral_constant<int, 1>());
    else if (n_kv <= 128) go(std::integral_constant<int, 2>());
    else go(std::integral_constant<int, 4>());
    __syncthreads();
    if (w8) return;
    const f32x4 f = *(const f32x4 *) (row + 4 * lane);
    const float v[4] = {f[0], f[1], f[2], f[3]};
    const int K = a.H * 128;
    q8k_block_from_regs(v, lane, y.y + (size_t) t * y.row_bytes, K, blk, y.tab, t);
}

} // namespace

int pm_launch_attn_cached_q8k(const float * q, void * kc, void * vc, const int32_t * pos, const int32_t * seq, long seq_stride, int H, int Hkv, int dh, int n_ctx, float scale, hipStream_t st,
                              int max_cells, int n_tok, const pm_q8k_out & out) {
    const int kpl = max_cells <= 64 ? 1 : max_cells <= 128 ? 2 : 4;
    if (dh != 128 || Hkv < 1 || H < Hkv || H > 65535 || H % 2 || n_ctx % 8 || n_tok < 1 || max_cells < 1 || max_cells > 256 || n_ctx < 64 * kpl || !pos || !seq) return -1;
    AttnP a = {q, nullptr, nullptr, (uint16_t *) kc, (uint16_t *) vc, pos, seq, seq_stride, nullptr, nullptr, H, Hkv, n_ctx, scale, RopeP(), nullptr, nullptr, 0, nullptr, 0, 1};
    const size_t lds = 2 * (size_t) (kpl == 1 ? ShortLds<128, 1>::BYTES : kpl == 2 ? ShortLds<128, 2>::BYTES : ShortLds<128, 4>::BYTES);
    pm_allow_big_lds((const void *) attn_cached_q8k_kernel, lds);
    const CachedArgs c = cached_args(a);
    hipLaunchKernelGGL(attn_cached_q8k_kernel, dim3(H / 2, n_tok), dim3(512), lds, st, a.q, a.kc, a.vc, a.pos0_ptr, a.seq_ptr, c.heads, c.inv, a.n_ctx, a.scale, a, out);
    return 0;
}

void pm_launch_rope_table(const pm_rope_cfg & c, const int32_t * pos, const int32_t * seq, const float * freq_factors, float * tab, hipStream_t st, int n_tok, int rows) {
    RopeP r;
    r.n_dims = c.n_dims; r.mode = c.mode; r.n_ctx_orig = c.n_ctx_orig; r.theta_scale = c.theta_scale;
    r.freq_scale = c.freq_scale; r.ext_factor = c.ext_factor; r.attn_factor = c.attn_factor; r.corr0 = c.corr0; r.corr1 = c.corr1;
    hipLaunchKernelGGL(rope_table_kernel, dim3(n_tok < 1 ? 1 : n_tok), dim3(128), 0, st, r, pos, seq, freq_factors, tab, rows);
}

// q = rotated, F16-rounded query rows; caches already hold this token. Same arguments as pm_launch_attn_rope_fused otherwise.
int pm_launch_attn_cached(const float * q, void * kc, void * vc, const int32_t * pos0, const int32_t * seq, long seq_stride, float * out,
                          int H, int Hkv, int dh, int n_ctx, float scale, hipStream_t st, const int32_t * dyn, const void * mask,
                          int max_keys, int v_rowmajor, int mask_f16, int n_tok, int rows) {
    if ((dh != 64 && dh != 128 && dh != 256) || Hkv < 1 || H < Hkv || n_ctx % 8 || n_tok < 1 || (n_tok > 1 && dyn) || (rows && (dyn || !seq || !pos0))) return -1;
    size_t lds = (size_t) (4 * dh + (v_rowmajor ? 2048 : 256) + (max_keys > 0 ? ((max_keys + 7) & ~7) : n_ctx) + 8) * 4;
    if (lds > 150 * 1024) return -1;
    // (two workgroups of the largest short form per CU, as many as their registers allow)
    const int kpl = v_rowmajor || n_ctx < 64 ? 0 : n_ctx < 128 || dh > 128 ? 1 : n_ctx < 256 ? 2 : 4;
    if (kpl) lds = std::max(lds, (size_t) (dh == 256 ? ShortLds<256, 1>::BYTES : dh == 128 ? kpl == 1 ? ShortLds<128, 1>::BYTES : kpl == 2 ? ShortLds<128, 2>::BYTES : ShortLds<128, 4>::BYTES :
                                           kpl == 1 ? ShortLds<64, 1>::BYTES : kpl == 2 ? ShortLds<64, 2>::BYTES : ShortLds<64, 4>::BYTES));
    RopeP r = {};
    if (!pos0) pos0 = dyn;                       // ggml-graph mode: cells come from dyn; keep every pointer the kernel may touch valid
    if (!pos0) return -1;
    auto launch = [&](auto kern) {
        pm_allow_big_lds((const void *) kern, lds);
        AttnP a = {q, nullptr, nullptr, (uint16_t *) kc, (uint16_t *) vc, pos0, seq, seq_stride, nullptr, out, H, Hkv, n_ctx, scale, r, dyn,
                   (const float *) mask, mask_f16, pm_ts_next_slot(), 0, rows};
        const CachedArgs c = cached_args(a);
        hipLaunchKernelGGL(kern, dim3(H, n_tok), dim3(256), lds, st, a.q, a.kc, a.vc, a.pos0_ptr, a.seq_ptr, c.heads, c.inv, a.n_ctx, c.how, a);
    };
    auto go = [&](auto few, auto many) { if (H > 65535) launch(many); else launch(few); };
    if (v_rowmajor) {
        if (dh == 64) go(attn_cached_kernel<64, 1>, attn_cached_kernel<64, 1, true>);
        else if (dh == 128) go(attn_cached_kernel<128, 1>, attn_cached_kernel<128, 1, true>);
        else go(attn_cached_kernel<256, 1>, attn_cached_kernel<256, 1, true>);
    } else if (dh == 64) go(attn_cached_kernel<64, 0>, attn_cached_kernel<64, 0, true>);
    else if (dh == 128) go(attn_cached_kernel<128, 0>, attn_cached_kernel<128, 0, true>);
    else go(attn_cached_kernel<256, 0>, attn_cached_kernel<256, 0, true>);
    return 0;
}
