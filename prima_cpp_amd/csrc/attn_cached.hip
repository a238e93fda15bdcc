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
//   * up to 256 cells (head sizes up to 128; 64 cells for 256): attn_whole_lines (attn_tail_device.h), every load issued first, ONE workgroup barrier.
//   * more cells (up to the long-context threshold): the per-head body of attn_device.h in its CACHED form.
#include "attn_device.h"
#include "attn_tail_device.h"
#include "pm355_layer_ops.h"
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

template <int DH, int VM>
__global__ __launch_bounds__(256) void attn_cached_kernel(AttnP a_in) {
    // grid.y = tokens of a small batch (engine: 2..64-token steps after rope_kv_store has rotated / rounded q and stored every token's K / V):
    // token t attends cells [0, pos0 + t], its q / out rows are t * H * DH further on
    AttnP a = a_in;
    a.tok = (int) blockIdx.y;
    a.q += (long) a.tok * a.H * DH; a.out += (long) a.tok * a.H * DH;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ float redf[8];
    __shared__ double redd[4];
    __shared__ __attribute__((aligned(16))) float part[256], pw[4][256];       // scores, probabilities by wave (attn_whole_lines)
    const int h = blockIdx.x;
    if constexpr (VM == 0) {
        const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int Hkv = a.Hkv, hk = h / (a.H / Hkv), n_ctx = a.n_ctx;
        int seq = 0, n_kv;
        if (a.dyn) n_kv = uniform_const_ptr(a.dyn)[1];
        else {
            seq = a.seq_ptr ? uniform_const_ptr(a.seq_ptr)[a.rows ? a.tok : 0] : 0;
            n_kv = uniform_const_ptr(a.pos0_ptr)[a.rows ? a.tok : seq] + 1 + (a.rows ? 0 : a.tok);
        }
        const uint16_t * kc = a.kc + (long) seq * a.seq_stride, * vc = a.vc + (long) seq * a.seq_stride;
        auto bar = [&]() __attribute__((always_inline)) { __syncthreads(); };
        auto whole = [&](auto kpl) __attribute__((always_inline)) {
            attn_whole_lines<DH, decltype(kpl)::value, false>(a.q + (long) h * DH, kc, vc, a.out + (long) h * DH, hk, Hkv, n_ctx, n_kv, a.scale, a.mask, a.mask_f16, part, &pw[0][0], lane, wave, bar);
        };
        if (n_kv <= 64) return whole(std::integral_constant<int, 1>());
        if constexpr (DH <= 128) {
            if (n_kv <= 128) return whole(std::integral_constant<int, 2>());
            if (n_kv <= 256) return whole(std::integral_constant<int, 4>());
        }
    }
    attn_rope_body<DH, false, VM, true>(a, h, smem, redf, redd);
}

} // namespace

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
    if ((dh != 64 && dh != 128 && dh != 256) || n_ctx % 8 || n_tok < 1 || (n_tok > 1 && dyn) || (rows && (dyn || !seq || !pos0))) return -1;
    const size_t lds = (size_t) (4 * dh + (v_rowmajor ? 2048 : 256) + (max_keys > 0 ? ((max_keys + 7) & ~7) : n_ctx) + 8) * 4;
    if (lds > 150 * 1024) return -1;
    RopeP r = {};
    if (!pos0) pos0 = dyn;                       // ggml-graph mode: cells come from dyn; keep every pointer the kernel may touch valid
    if (!pos0) return -1;
    auto launch = [&](auto kern) {
        if (lds > 48 * 1024) (void) hipFuncSetAttribute((const void *) kern, hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024);
        AttnP a = {q, nullptr, nullptr, (uint16_t *) kc, (uint16_t *) vc, pos0, seq, seq_stride, nullptr, out, H, Hkv, n_ctx, scale, r, dyn,
                   (const float *) mask, mask_f16, pm_ts_next_slot(), 0, rows};
        hipLaunchKernelGGL(kern, dim3(H, n_tok), dim3(256), lds, st, a);
    };
    if (v_rowmajor) {
        if (dh == 64) launch(attn_cached_kernel<64, 1>);
        else if (dh == 128) launch(attn_cached_kernel<128, 1>);
        else launch(attn_cached_kernel<256, 1>);
    } else if (dh == 64) launch(attn_cached_kernel<64, 0>);
    else if (dh == 128) launch(attn_cached_kernel<128, 0>);
    else launch(attn_cached_kernel<256, 0>);
    return 0;
}
