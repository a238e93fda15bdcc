// attn_blocks.hip — the two attention launches of a small batch that end in the wo product's 8-bit blocks, beside the same attention stored as f32 rows and quantized by its own launch: both write rows
// of Q8_K and the small-batch mat-mul's tables (tests/test_gpu_ops.py compares them byte for byte; linked with the product's own objects).
#include "pm355_device.h"
#include "pm355_kernels.h"
#include "pm355_layer_ops.h"

static pm_q8k_tables tables(void * tab, void * q, int K) {
    pm_q8k_tables t;
    t.base = (uint8_t *) tab; t.nsb = K / 256; t.tab_bytes = (size_t) t.nsb * (1024 + 128); t.qbase = (uint8_t *) q;
    return t;
}
// rows != 0: every token a row of its own sequence, pos[t] + 1 cells (max_cells the most of them); 0: consecutive tokens of sequence seq[0] from pos[0] on. q, f32: [n_tok][H * 128]; y, y2: n_tok Q8_K
// rows; tab, tab2: tables of 32 tokens; kc, vc: caches of sequences of `stride` values
extern "C" __attribute__((visibility("default"))) int pm355_probe_attn_blocks(const float * q, void * kc, void * vc, const int32_t * pos, const int32_t * seq, int64_t stride, int H, int Hkv, int n_ctx, float scale, int rows, int max_cells,
                                       int n_tok, void * y, void * tab, void * tq, float * f32, void * y2, void * tab2, void * tq2, void * st_) {
    hipStream_t st = (hipStream_t) st_;
    const int K = H * 128;
    const pm_q8k_out out = {(uint8_t *) y, pm_q8k_row_bytes(K), tables(tab, tq, K)};
    int rc = rows ? pm_launch_attn_cached_q8k(q, kc, vc, pos, seq, stride, H, Hkv, 128, n_ctx, scale, st, max_cells, n_tok, out)
                  : pm_launch_attn_prefill_q8k(q, kc, vc, pos, seq, stride, n_tok, H, Hkv, 128, n_ctx, scale, st, nullptr, 0, out);
    if (rc) return rc;
    rc = rows ? pm_launch_attn_cached(q, kc, vc, pos, seq, stride, f32, H, Hkv, 128, n_ctx, scale, st, nullptr, nullptr, max_cells, 0, 0, n_tok, 1)
              : pm_launch_attn_prefill(q, kc, vc, pos, seq, stride, f32, n_tok, H, Hkv, 128, n_ctx, scale, st);
    if (rc) return rc;
    pm_launch_quantize_q8k(f32, y2, K, n_tok, st, tables(tab2, tq2, K));
    return hipGetLastError() == hipSuccess ? 0 : -2;
}
