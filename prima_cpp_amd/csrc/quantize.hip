// quantize.hip — activation quantizers for the decode path (gfx950).
//
//   f32 row -> Q8_K  (reference: quantize_row_q8_K_ref, ggml/src/ggml-quants.c:3785-3826)
//   f32 row -> Q8_0  (reference: quantize_row_q8_0_ref, ggml/src/ggml-quants.c:848-871)
//   rms_norm(x) * w -> f32 and/or Q8_K in one pass
//              (reference: ggml_compute_forward_rms_norm_f32 ggml.c:11950 + ggml_compute_forward_mul_f32 :10077)
//
// Bit-exact with the reference for q / bsums / d: same float operations in the same order per
// element (iscale = -127/max; nearest_int(iscale*x); d = 1/iscale), and the same "first element with
// the largest |x| decides the sign" rule, implemented as (wave max) + (wave min over candidate index).
//
// Device layout of a quantized activation row ("row-SoA", internal to this library; K values):
//   Q8_K : int8 qs[K] | float d[K/256] | int16 bsums[K/16]       -> pm_q8k_row_bytes(K)
//   Q8_0 : int8 qs[K] | half  d[K/32]                            -> pm_q80_row_bytes(K)
// HBM-bound, trivially small (K <= 32k): one wave per 256-value block, 4 values per lane (16-B loads).
#include "pm355_device.h"
#include "pm355_kernels.h"
#include "pm355_q8k.h"

// (Grids of rows x groups of four blocks, below of rows x 1024 values: by one index, split into row and block in 64 bits, every launch began with a division of a few hundred instructions in front of
// its first load. us a pass before / now: eight sequences of the 8B shape, 96 launches of 8 rows of 14336 9056 / 9036;
// two layers of the 72B shape at 23 tokens, silu_mul_q80_tab_kernel, 451.1 / 449.9)
// FLAT: rows that fill less than half of a workgroup, by one index all the same (a division of 32 bits). us, rows x groups / flat: Q8_0 200000 rows of 32 45.7 / 6.9,
// 8192 of 64 3.7 / 2.3, 8192 of 256 4.0 / 3.3, Q8_K 200000 of 256 65.0 / 52.9. From 512 values on rows x groups are faster (Q8_0 8192 of 512 4.6, by one index and 64 bits 5.2). And from 2^24 rows on, where a grid of rows ends
template <bool FLAT>
__global__ __launch_bounds__(256) void quantize_q8k_kernel(const float * __restrict__ x, uint8_t * __restrict__ y,
                                                           int K, int rows, size_t y_row_bytes, pm_q8k_tables tb, pm_q8k_wide wd) {
    const int lane = threadIdx.x & 63;
    int row = (int) blockIdx.x, blk = (int) blockIdx.y * 4 + __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
    if constexpr (FLAT) {
        const uint32_t nblk = (uint32_t) K / PM_QK_K, w = blockIdx.x * 4 + (uint32_t) __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
        row = (int) (w / nblk); blk = (int) (w % nblk);
        if (row >= rows) return;
    } else if (blk >= K / PM_QK_K) return;
    const float4 f = ((const float4 *) (x + (size_t) row * K + (size_t) blk * PM_QK_K))[lane];
    const float v[4] = {f.x, f.y, f.z, f.w};
    q8k_block_from_regs(v, lane, y ? y + (size_t) row * y_row_bytes : nullptr, K, blk, tb, row, wd);
}

// silu(gate) * up (ggml_silu + ggml_mul of llm_build_ffn, src/llama.cpp:9804; same f32 expressions as layer_ops.hip's silu_mul_kernel) fused with
// the Q8_K quantization of the product: the ffn_down activations of a small batch, without the f32 round trip through HBM
__global__ __launch_bounds__(256) void silu_mul_q8k_kernel(const float * __restrict__ gate, const float * __restrict__ up, uint8_t * __restrict__ y,
                                                           int K, size_t y_row_bytes, pm_q8k_tables tb) {
    const int lane = threadIdx.x & 63;
    const int row = (int) blockIdx.x, blk = (int) blockIdx.y * 4 + __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
    if (blk >= K / PM_QK_K) return;
    const float4 g = ((const float4 *) (gate + (size_t) row * K + (size_t) blk * PM_QK_K))[lane];
    const float4 u = ((const float4 *) (up + (size_t) row * K + (size_t) blk * PM_QK_K))[lane];
    const float v[4] = {g.x / (1.0f + expf(-g.x)) * u.x, g.y / (1.0f + expf(-g.y)) * u.y, g.z / (1.0f + expf(-g.z)) * u.z, g.w / (1.0f + expf(-g.w)) * u.w};
    q8k_block_from_regs(v, lane, y + (size_t) row * y_row_bytes, K, blk, tb, row);
}

// Q8_0: 32-value blocks, 8 lanes x 4 values; amax over the 8-lane group.
template <bool FLAT>
__global__ __launch_bounds__(256) void quantize_q80_kernel(const float * __restrict__ x, uint8_t * __restrict__ y,
                                                           int K, int rows, size_t y_row_bytes) {
    int row = (int) blockIdx.x, i4 = (int) blockIdx.y * 256 + (int) threadIdx.x;        // one thread = 4 values
    if constexpr (FLAT) {
        const uint32_t per_row = (uint32_t) K / 4, t = blockIdx.x * 256 + threadIdx.x;
        row = (int) (t / per_row); i4 = (int) (t % per_row);
        if (row >= rows) return;
    } else if (i4 >= K / 4) return;
    const float4 f = ((const float4 *) (x + (size_t) row * K))[i4];
    float amax = fmaxf(fmaxf(fabsf(f.x), fabsf(f.y)), fmaxf(fabsf(f.z), fabsf(f.w)));
    amax = group8_max(amax);
    const float d  = amax / 127;
    const float id = d ? 1.0f / d : 0.0f;
    uint8_t * ro = y + (size_t) row * y_row_bytes;
    const float v[4] = {f.x, f.y, f.z, f.w};
    uint32_t packed = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) packed |= (uint32_t) ((int) roundf(v[i] * id) & 0xFF) << (8 * i);
    ((uint32_t *) ro)[i4] = packed;
    if ((i4 & 7) == 0) ((uint16_t *) (ro + K))[i4 >> 3] = f2h(d);
}

// silu(gate) * up fused with the Q8_0 quantization of the product, written STRAIGHT into the small-batch mat-mul's activation tables (mmq_i8.hip, Q8_0 weights:
// per 32-token pass [blk][64 lanes][16 B] values in A-operand order + [blk][32] f32 scales) - the ffn_down activations of the files whose n_ff is no multiple of
// 256 (Qwen2.5-72B: K = 29568 falls back to Q8_0, src/llama.cpp:19447). Replaces three launches (silu_mul, quantize_q80, the mat-mul's table prologue).
// Rows T .. 32 * passes - 1 write scale 0 (their values are never loaded).
__global__ __launch_bounds__(256) void silu_mul_q80_tab_kernel(const float * __restrict__ gate, const float * __restrict__ up, uint8_t * __restrict__ tab,
                                                               int K, int rows, size_t pass_bytes, size_t qtab_bytes) {
    const int row = (int) blockIdx.x, i4 = (int) blockIdx.y * 256 + (int) threadIdx.x;        // one thread = 4 values, 8 lanes = one block
    if (i4 >= K / 4) return;
    const int blk = i4 >> 3, sub = i4 & 7;
    uint8_t * base = tab + (size_t) (row >> 5) * pass_bytes;
    float * dslot = (float *) (base + qtab_bytes) + ((size_t) blk * 32 + (row & 31));
    if (row >= rows) { if (sub == 0) *dslot = 0.0f; return; }
    const float4 g = ((const float4 *) (gate + (size_t) row * K))[i4];
    const float4 u = ((const float4 *) (up + (size_t) row * K))[i4];
    const float v[4] = {g.x / (1.0f + expf(-g.x)) * u.x, g.y / (1.0f + expf(-g.y)) * u.y, g.z / (1.0f + expf(-g.z)) * u.z, g.w / (1.0f + expf(-g.w)) * u.w};
    float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
    amax = group8_max(amax);
    const float d  = amax / 127;
    const float id = d ? 1.0f / d : 0.0f;
    uint32_t packed = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) packed |= (uint32_t) ((int) roundf(v[i] * id) & 0xFF) << (8 * i);
    // lane (token slot row % 32, half g = sub / 4) of block blk holds bytes [16 g, 16 g + 16) of the block
    *(uint32_t *) (base + (size_t) blk * 1024 + (size_t) (32 * (sub >> 2) + (row & 31)) * 16 + 4 * (sub & 3)) = packed;
    if (sub == 0) *dslot = h2f(f2h(d));
}

// rms_norm (+ weight) fused with Q8_K quantization. One 256-thread workgroup per row.
// Optionally also writes the normalised f32 row (ynorm != nullptr).
// NWV waves per row: 4 for many rows (prompts: small workgroups, several per CU), 16 while every row has a CU to itself - the launch is then ONE latency chain per row: load, reduce,
// quantize block after block. us with 4 / 16 waves, K = 4096: 101 rows 5.1 / 3.9, 256 rows 5.3 / 4.2, 300 rows 5.4 / 6.0; K = 8192: 101 rows 7.9 / 4.9, 256 rows 8.2 / 5.4, 512 rows 9.3 / 8.5,
// 700 rows 11.1 / 11.4. (8 rows 3.8 -> 3.6 with the sum by DPP and the weights asked for with the row.)
// SPLIT: two workgroups to a row of 17 .. 32 blocks, each adds the whole row up (the same sum) and writes one half of it. Two blocks one after the other in every wave, four waves on a SIMD, were
// 2.0 of a launch's 3.9 us (stamps, 8 rows of 8192): three layers of the 70B shape at 8 tokens, six such launches, 391 -> 388 us. (One block in every wave, 1.25 of 3.1, in two or four workgroups: no
// change. A workgroup's share by gridDim.y and a division: 0.6 us more on every launch, the grid's size is another load.)
template <int NWV, bool SPLIT = false>
__global__ __launch_bounds__(64 * NWV) void rmsnorm_q8k_kernel(const float * __restrict__ x, const float * __restrict__ w,
                                                          float * __restrict__ ynorm, uint8_t * __restrict__ yq,
                                                          int K, float eps, size_t yq_row_bytes, _Float16 * __restrict__ yh, pm_q8k_tables tb, pm_q8k_wide wd) {
    __shared__ double red[NWV];
    const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int nblk = K / PM_QK_K;
    const float * xr = x + (size_t) row * K;
    // A wave's blocks (wv, wv + 4, ...) are loaded ONCE, all loads in flight together, and stay in registers between the two passes
    // (K <= 8192: 8 blocks per wave). With few rows (decode batches) the kernel is one latency chain per row: the former form - one
    // dependent load per block and pass - took 12 us for K = 8192.
    constexpr int HOLD = NWV == 4 ? 8 : 2;
    const bool held = nblk <= NWV * HOLD;
    float4 f[HOLD], wt[HOLD];                                          // (a handful of rows: the weights too, behind the sum they were a second round of latency)
    constexpr bool WT = NWV > 4;
    if (held) {
#pragma unroll
        for (int i = 0; i < HOLD; ++i) {
            const int blk = min(wv + NWV * i, nblk - 1);
            f[i] = ((const float4 *) (xr + (size_t) blk * PM_QK_K))[lane];
            if constexpr (WT) wt[i] = w ? ((const float4 *) (w + (size_t) blk * PM_QK_K))[lane] : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
        }
    }
    // pass 1: sum of squares; products rounded to f32 like the reference, accumulated in f64 (same order as before: blocks ascending)
    double s = 0.0;
    if (held) {
#pragma unroll
        for (int i = 0; i < HOLD; ++i) if (wv + NWV * i < nblk) {
            s += (double) (f[i].x * f[i].x); s += (double) (f[i].y * f[i].y); s += (double) (f[i].z * f[i].z); s += (double) (f[i].w * f[i].w);
        }
    } else {
        for (int blk = wv; blk < nblk; blk += NWV) {
            const float4 g = ((const float4 *) (xr + (size_t) blk * PM_QK_K))[lane];
            s += (double) (g.x * g.x); s += (double) (g.y * g.y); s += (double) (g.z * g.z); s += (double) (g.w * g.w);
        }
    }
    s = all_sum(s);
    if (lane == 0) red[wv] = s;
    __syncthreads();
    double tot = (red[0] + red[1]) + (red[2] + red[3]);
#pragma unroll
    for (int i = 4; i < NWV; i += 4) tot += (red[i] + red[i + 1]) + (red[i + 2] + red[i + 3]);
    const float mean  = (float) (tot / K);
    const float scale = 1.0f / sqrtf(mean + eps);
    // pass 2: normalise (+weight), write f32 and/or quantize
    auto emit = [&](const float4 & fx, int blk, const float4 * held_w = nullptr) __attribute__((always_inline)) {
        float v[4] = {fx.x * scale, fx.y * scale, fx.z * scale, fx.w * scale};
        if (w) {
            const float4 g = held_w ? *held_w : ((const float4 *) (w + (size_t) blk * PM_QK_K))[lane];
            v[0] *= g.x; v[1] *= g.y; v[2] *= g.z; v[3] *= g.w;
        }
        if (ynorm) ((float4 *) (ynorm + (size_t) row * K + (size_t) blk * PM_QK_K))[lane] = make_float4(v[0], v[1], v[2], v[3]);
        if (yh) {                                // F16 copy for the MFMA GEMMs (RNE, the rounding their conversion pass applies)
            typedef _Float16 h4 __attribute__((ext_vector_type(4)));
            ((h4 *) (yh + (size_t) row * K + (size_t) blk * PM_QK_K))[lane] = h4{(_Float16) v[0], (_Float16) v[1], (_Float16) v[2], (_Float16) v[3]};
        }
        if (yq || wd.q) q8k_block_from_regs(v, lane, yq ? yq + (size_t) row * yq_row_bytes : nullptr, K, blk, tb, row, wd);
    };
    if (held) {
#pragma unroll
        for (int i = 0; i < HOLD; ++i) if ((!SPLIT || i == (int) blockIdx.y) && wv + NWV * i < nblk) emit(f[i], wv + NWV * i, WT ? &wt[i] : nullptr);
    } else {
        for (int blk = wv; blk < nblk; blk += NWV) emit(((const float4 *) (xr + (size_t) blk * PM_QK_K))[lane], blk);
    }
}

// (a row whose results lie on the input is one workgroup's: of two, one may store its half before the other has read the row)
static bool norm_split(const float * x, const float * ynorm, const void * yq, const void * yh, int K, int rows) {
    if (K <= 16 * PM_QK_K || K > 32 * PM_QK_K || 2 * rows > pm_device_cus()) return false;
    const size_t n = (size_t) rows * K;
    const auto meets = [&](const void * y, size_t bytes) { return y && (uintptr_t) y < (uintptr_t) (x + n) && (uintptr_t) x < (uintptr_t) y + bytes; };
    return !meets(ynorm, n * 4) && !meets(yq, rows * pm_q8k_row_bytes(K)) && !meets(yh, n * 2);
}

static dim3 q8k_grid(int K, int rows) { return dim3(rows, (K / PM_QK_K + 3) / 4); }
static bool flat(int K, int rows) { return K < 512 || rows >= 1 << 24; }

// ---- host launchers -------------------------------------------------------------------------------
static void launch_quantize_q8k(const float * x, void * y, int K, int rows, hipStream_t st, size_t y_row_bytes, const pm_q8k_tables & tab, const pm_q8k_wide & wd) {
    if (flat(K, rows)) hipLaunchKernelGGL(quantize_q8k_kernel<true>, dim3((unsigned) (((long) rows * (K / PM_QK_K) + 3) / 4)), dim3(256), 0, st, x, (uint8_t *) y, K, rows, y_row_bytes, tab, wd);
    else               hipLaunchKernelGGL(quantize_q8k_kernel<false>, q8k_grid(K, rows), dim3(256), 0, st, x, (uint8_t *) y, K, rows, y_row_bytes, tab, wd);
}
void pm_launch_quantize_q8k(const float * x, void * y, int K, int rows, hipStream_t st, pm_q8k_tables tab) {
    launch_quantize_q8k(x, y, K, rows, st, pm_q8k_row_bytes(K), tab, pm_q8k_wide());
}
void pm_launch_quantize_wide(const float * x, const pm_q8k_wide & y, int K, int rows, hipStream_t st) { launch_quantize_q8k(x, nullptr, K, rows, st, 0, pm_q8k_tables(), y); }
void pm_launch_silu_mul_q8k(const float * gate, const float * up, void * y, int K, int rows, hipStream_t st, pm_q8k_tables tab) {
    hipLaunchKernelGGL(silu_mul_q8k_kernel, q8k_grid(K, rows), dim3(256), 0, st, gate, up, (uint8_t *) y, K, pm_q8k_row_bytes(K), tab);
}
void pm_launch_silu_mul_q80_tab(const float * gate, const float * up, void * tab, size_t qtab_bytes, size_t dtab_bytes, int K, int rows, hipStream_t st) {
    hipLaunchKernelGGL(silu_mul_q80_tab_kernel, dim3((rows + 31) / 32 * 32, (K / 4 + 255) / 256), dim3(256), 0, st, gate, up, (uint8_t *) tab, K, rows,
                       qtab_bytes + dtab_bytes, qtab_bytes);
}
void pm_launch_quantize_q80(const float * x, void * y, int K, int rows, hipStream_t st) {
    if (flat(K, rows)) hipLaunchKernelGGL(quantize_q80_kernel<true>, dim3((unsigned) (((long) rows * (K / 4) + 255) / 256)), dim3(256), 0, st, x, (uint8_t *) y, K, rows, pm_q80_row_bytes(K));
    else               hipLaunchKernelGGL(quantize_q80_kernel<false>, dim3(rows, (K / 4 + 255) / 256), dim3(256), 0, st, x, (uint8_t *) y, K, rows, pm_q80_row_bytes(K));
}
void pm_launch_rmsnorm_q8k(const float * x, const float * w, float * ynorm, void * yq, int K, int rows, float eps, hipStream_t st, void * ynorm_f16, pm_q8k_tables tab) {
    if (norm_split(x, ynorm, yq, ynorm_f16, K, rows)) hipLaunchKernelGGL((rmsnorm_q8k_kernel<16, true>), dim3(rows, 2), dim3(1024), 0, st, x, w, ynorm, (uint8_t *) yq, K, eps, pm_q8k_row_bytes(K), (_Float16 *) ynorm_f16, tab, pm_q8k_wide());
    else if (rows <= pm_device_cus()) hipLaunchKernelGGL(rmsnorm_q8k_kernel<16>, dim3(rows), dim3(1024), 0, st, x, w, ynorm, (uint8_t *) yq, K, eps, pm_q8k_row_bytes(K), (_Float16 *) ynorm_f16, tab, pm_q8k_wide());
    else            hipLaunchKernelGGL(rmsnorm_q8k_kernel<4>, dim3(rows), dim3(256), 0, st, x, w, ynorm, (uint8_t *) yq, K, eps, pm_q8k_row_bytes(K), (_Float16 *) ynorm_f16, tab, pm_q8k_wide());
}
void pm_launch_rmsnorm_wide(const float * x, const float * w, const pm_q8k_wide & y, int K, int rows, float eps, hipStream_t st) {
    if (norm_split(x, nullptr, nullptr, nullptr, K, rows)) hipLaunchKernelGGL((rmsnorm_q8k_kernel<16, true>), dim3(rows, 2), dim3(1024), 0, st, x, w, (float *) nullptr, (uint8_t *) nullptr, K, eps, 0, (_Float16 *) nullptr, pm_q8k_tables(), y);
    else if (rows <= pm_device_cus()) hipLaunchKernelGGL(rmsnorm_q8k_kernel<16>, dim3(rows), dim3(1024), 0, st, x, w, (float *) nullptr, (uint8_t *) nullptr, K, eps, 0, (_Float16 *) nullptr, pm_q8k_tables(), y);
    else             hipLaunchKernelGGL(rmsnorm_q8k_kernel<4>, dim3(rows), dim3(256), 0, st, x, w, (float *) nullptr, (uint8_t *) nullptr, K, eps, 0, (_Float16 *) nullptr, pm_q8k_tables(), y);
}
