// attn_prefill.hip — causal multi-token (prefill) attention on the MFMA matrix cores of gfx950.
//
// Replaces, for n_tokens >= 16, the three nodes of llm_build_kqv without flash-attn (src/llama.cpp:10032-10110):
//   kq  = MUL_MAT(K F16, q)            ggml_compute_forward_mul_mat with vec_dot_type F16: q is converted to F16, f32 accumulate
//   p   = SOFT_MAX_EXT(kq, mask, scale) ggml_compute_forward_soft_max_f32 (ggml.c:13783): max, expf, sum, scale by 1/sum
//   kqv = MUL_MAT(V^T F16, p)          p converted to F16, f32 accumulate
// with q and p rounded to F16, K / V F16, f32 accumulation. The per-token kernel (attn_decode_kernel) needs O(n_tokens^2) scalar work: 9.2 ms per layer for a 2048-token
// prompt on the 70B shape, more than all GEMMs of the layer together.
//
// Design. Everything is computed TRANSPOSED so that a query is a COLUMN of the MFMA result: S^T = K Q^T (keys x queries) and O^T = V^T P^T. In the 32x32 accumulator layout a lane
// then holds 16 keys of ONE query (column = lane & 31): the softmax statistics are in-lane reductions plus one exchange with the partner lane (lane ^ 32), and P^T never leaves the
// registers. attn_prompt_kernel serves the transposed V cache of the default graphs, attn_rowmajor_kernel the row-major one of the flash-attention graphs.
#include "pm355_device.h"
#include "pm355_dense.h"
#include "pm355_kernels.h"
#include "pm355_layer_ops.h"
#include "pm355_q8k.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));

struct PfP {
    const float * q; const uint16_t * kc; const uint16_t * vc; const int32_t * pos0_ptr; const int32_t * seq_ptr; long seq_stride;
    float * out; int T, H, Hkv, n_ctx; float scale;
    // ggml-graph mode (mask != nullptr; pm355_attn_prefill_masked): every query attends cells [0, n_kv) with the additive F32 KQ_mask
    // row of its token (0 / -inf; llama_set_inputs src/llama.cpp:17379-17420) instead of the causal rule "cell <= position"
    const float * mask; long mask_stride; int n_kv;
    int mask_f16;                                // the mask rows are F16
    _Float16 * out_h;                            // optional: the result as F16 [T][H*DH] (activations of the wo GEMM) instead of `out`
    const int32_t * tiles; int n_tiles;          // optional: tiles {row, queries, position, sequence} of several sequences; else consecutive tokens from pos0 on
};

// Flash-attention graphs (FLASH_ATTN_EXT, llm_build_kqv src/llama.cpp:10075-10095): V cache [n_ctx][Hkv*DH] like K, always masked. One workgroup = 128 queries of one head, 4 waves x
// 32. K and V tiles (32 keys) travel global -> registers -> LDS once per workgroup, double-buffered; V is transposed on its way. Row strides are padded so that the fragment reads
// (lane = key / channel, 16 bytes) are conflict-free: K rows DH + 8 halves (68 dwords: lane i -> bank 4 i), V^T rows 40 halves (20 dwords: 16 lanes cover the 64 banks once). Two
// passes over the keys, because p is rounded to F16 after the division by the full row sum: pass 1 = row max and sum (online), pass 2 = recompute S, p = exp(s - max) / sum -> F16,
// accumulate O. P is rounded to F16 here as well (it is an MFMA operand; the reference keeps it f32 and rounds its F16 accumulator instead).
template <int DH>
__global__ __launch_bounds__(256, 2) void attn_rowmajor_kernel(PfP p) {
    constexpr int KK = DH / 16;                  // k-steps of the S^T MFMAs
    constexpr int DT = DH / 32;                  // 32-row tiles of O^T
    constexpr int KS = DH + 8, VS = 40;          // LDS row strides (halves)
    constexpr int UPR = DH / 8;                  // 16-byte units per K row
    constexpr int NU = DH / 64;                  // units per thread and tile (K: 32 * UPR / 256; V^T: 4 * DH / 256)
    __shared__ __attribute__((aligned(16))) _Float16 ks[2][32 * KS];
    __shared__ __attribute__((aligned(16))) _Float16 vs[2][DH * VS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 31, hf = lane >> 5;
    const int h = blockIdx.y, hk = h / (p.H / p.Hkv);
    const long krow = (long) p.Hkv * DH;
    const uint16_t * kc = p.kc + (long) hk * DH, * vc = p.vc + (long) hk * DH;         // K, V [key][Hkv*DH]
    const int qb = (int) blockIdx.x;
    const int tq0 = qb * 128 + wave * 32;                                              // first query token of this wave
    const bool wave_live = tq0 < p.T;
    const int tq = min(tq0 + col, p.T - 1);                                            // this lane's query (clamped)
    const int n_wg = (p.n_kv + 31) / 32, n_tiles = wave_live ? n_wg : 0;                // (every wave takes part in the staging and the barriers)
    const float * mrow = !p.mask_f16 ? p.mask + (long) tq * p.mask_stride : nullptr;
    const uint16_t * mrow16 = p.mask_f16 ? (const uint16_t *) p.mask + (long) tq * p.mask_stride : nullptr;

    // ---- staging: global -> registers (fetch) -> LDS (put)
    u32x4 kg[NU], vg[NU];
    auto fetch_k = [&](int j) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int u = tid + 256 * i, key = min(j * 32 + u / UPR, p.n_ctx - 1), piece = u % UPR;
            kg[i] = *(const u32x4 *) (kc + (long) key * krow + 8 * piece);
        }
    };
    auto fetch_v = [&](int j) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int u = tid + 256 * i, key = min(j * 32 + u / UPR, p.n_ctx - 1), piece = u % UPR;
            vg[i] = *(const u32x4 *) (vc + (long) key * krow + 8 * piece);
        }
    };
    auto put_k = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NU; ++i) { const int u = tid + 256 * i; *(u32x4 *) (ks[b] + (u / UPR) * KS + 8 * (u % UPR)) = kg[i]; }
    };
    auto put_v = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int u = tid + 256 * i, key = u / UPR, piece = u % UPR;      // V[key][8 piece .. +8] -> V^T rows 8 piece .. +8, column key
            uint16_t * d = (uint16_t *) vs[b] + (8 * piece) * VS + key;
#pragma unroll
            for (int e = 0; e < 4; ++e) { d[(2 * e) * VS] = (uint16_t) (vg[i][e] & 0xFFFF); d[(2 * e + 1) * VS] = (uint16_t) (vg[i][e] >> 16); }
        }
    };

    // Q^T as B operand: lane (col = query, hf) holds q[query][16 kk + 8 hf .. +8], rounded to F16 like the reference
    half8 qf[KK];
    {
        const float * qr = p.q + ((long) tq * p.H + h) * DH + 8 * hf;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const float4 a = *(const float4 *) (qr + 16 * kk), b = *(const float4 *) (qr + 16 * kk + 4);
            qf[kk] = half8{(_Float16) a.x, (_Float16) a.y, (_Float16) a.z, (_Float16) a.w, (_Float16) b.x, (_Float16) b.y, (_Float16) b.z, (_Float16) b.w};
        }
    }
    // S^T tile (32 keys x 32 queries) of key tile j out of LDS buffer b: A = K rows (lane: key = col, dh slice 16 kk + 8 hf)
    auto scores = [&](int j, int b, float (&s)[16]) __attribute__((always_inline)) {
        float16v acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
        const _Float16 * kr = ks[b] + col * KS + 8 * hf;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const half8 *) (kr + 16 * kk), qf[kk], acc, 0, 0, 0);
#pragma unroll
        for (int g = 0; g < 4; ++g) {                            // registers 4g .. 4g+3 = keys j*32 + 8g + 4hf .. +4: one float4 of the mask row
                const int k0 = j * 32 + 8 * g + 4 * hf;
                float4 mv = float4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
                if (k0 + 3 < p.n_kv) {
                    if (mrow) mv = *(const float4 *) (mrow + k0);
                    else { const u32x2 mh = *(const u32x2 *) (mrow16 + k0); mv = float4{h2f((uint16_t) (mh[0] & 0xFFFF)), h2f((uint16_t) (mh[0] >> 16)), h2f((uint16_t) (mh[1] & 0xFFFF)), h2f((uint16_t) (mh[1] >> 16))}; }
                }
                s[4 * g + 0] = acc[4 * g + 0] * p.scale + mv.x; s[4 * g + 1] = acc[4 * g + 1] * p.scale + mv.y;
                s[4 * g + 2] = acc[4 * g + 2] * p.scale + mv.z; s[4 * g + 3] = acc[4 * g + 3] * p.scale + mv.w;
            }
    };

    // ---- pass 1: row max and sum of exp (online within the lane, merged with the partner lane at the end)
    // exp = v_exp_f32 (__expf, ~1 ulp): the probabilities are rounded to F16 right after, and the reference's own SIMD builds use a
    // polynomial expf (ggml_v_expf, ggml.c:2370); libm's expf was ~30 VALU instructions x 33 per lane and key tile - most of the kernel
    float m = -INFINITY, l = 0.0f;
    fetch_k(0);
    put_k(0);
    __syncthreads();
    for (int j = 0; j < n_wg; ++j) {
        const bool more = j + 1 < n_wg;
        if (more) fetch_k(j + 1);
        if (j < n_tiles) {
            float s[16];
            scores(j, j & 1, s);
            float mt = s[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) mt = fmaxf(mt, s[r]);
            const float mn = fmaxf(m, mt);
            if (mn != -INFINITY) {
                float acc = 0.0f;
#pragma unroll
                for (int r = 0; r < 16; ++r) acc += __expf(s[r] - mn);
                l = l * __expf(m - mn) + acc;     // m == -inf: l == 0 and expf(-inf) == 0
                m = mn;
            }
        }
        if (more) put_k((j + 1) & 1);
        __syncthreads();
    }
    {
        const float mo = __shfl_xor(m, 32), lo = __shfl_xor(l, 32);
        const float mn = fmaxf(m, mo);           // key 0 is always visible: mn is finite
        l = (m == -INFINITY ? 0.0f : l * expf(m - mn)) + (mo == -INFINITY ? 0.0f : lo * expf(mo - mn));
        m = mn;
    }
    const float inv = 1.0f / l;

    // ---- pass 2: p = exp(s - m) * inv -> F16;  O^T (dh x queries) += V^T tile (dh x keys) . P^T tile (keys x queries)
    float16v o[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
    fetch_k(0); fetch_v(0);
    put_k(0); put_v(0);
    __syncthreads();
    for (int j = 0; j < n_wg; ++j) {
        const bool more = j + 1 < n_wg;
        if (more) { fetch_k(j + 1); fetch_v(j + 1); }
        if (j < n_tiles) {
            float s[16];
            scores(j, j & 1, s);
            half4 pk[4];                         // pk[g] = the 4 keys 8 g + 4 hf .. +4 of this query
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int i = 0; i < 4; ++i) pk[g][i] = (_Float16) (__expf(s[4 * g + i] - m) * inv);
            // B operand of k-step kk (keys 16 kk .. +16): lane half hf wants keys 16 kk + 8 hf .. +8 = two groups of 4, one of
            // which sits in the partner lane (lane ^ 32)
            half8 pf[2];
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                const half4 mine = hf ? pk[2 * kk + 1] : pk[2 * kk];         // keys this lane keeps
                const half4 send = hf ? pk[2 * kk] : pk[2 * kk + 1];         // keys the partner needs
                uint32_t s0 = ((const uint32_t *) &send)[0], s1 = ((const uint32_t *) &send)[1];
                s0 = (uint32_t) __shfl_xor((int) s0, 32); s1 = (uint32_t) __shfl_xor((int) s1, 32);
                half4 got;
                ((uint32_t *) &got)[0] = s0; ((uint32_t *) &got)[1] = s1;
                const half4 lo = hf ? got : mine, hi = hf ? mine : got;      // ascending key order
                pf[kk] = half8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            }
            const _Float16 * vb = vs[j & 1] + col * VS + 8 * hf;
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int kk = 0; kk < 2; ++kk)
                    o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const half8 *) (vb + (32 * d) * VS + 16 * kk), pf[kk], o[d], 0, 0, 0);
        }
        if (more) { put_k((j + 1) & 1); put_v((j + 1) & 1); }
        __syncthreads();
    }
    // ---- O^T[dh = 32 d + acc_row(r, hf)][query = col] -> out[t][h*DH + dh]
    if (wave_live && tq0 + col < p.T) {
        float * orow = p.out + ((long) tq * p.H + h) * DH;
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *(float4 *) (orow + 32 * d + 8 * g + 4 * hf) = float4{o[d][4 * g], o[d][4 * g + 1], o[d][4 * g + 2], o[d][4 * g + 3]};
    }
}

// ---- the default graphs' layout: V transposed ---------------------------------------------------------------------------------------------------------------------------------
// One workgroup = QW * 32 consecutive queries of one head; QW query waves x KW = 8 / QW key groups, and four waves that bring the keys and values (a request holds its wave up for 60-180 cycles: a
// stage's eight per wave were 0.9 of the 1.5 us that a stage of 128 keys took; now 1.2, the requests' own time and their latency). Per stage KS keys of K ([KS][DH]) and V^T ([DH][KS]) travel by LDS-DMA
// (double-buffered, 16-byte chunks XOR-swizzled on the source side so that the sixteen lanes a fragment read serves hit sixteen bank groups); key group kw multiplies keys
// kw * KT .. + KT of every stage and keeps an online softmax of its own, the groups are merged through LDS at the end. Rows of a K tile are read with bits 2 and 3 of the row
// index swapped: the accumulators of S^T then ARE the B operand of the P.V product.
// ONE pass over the keys: the probabilities are rounded to F16 before the division by their sum (which adds the unrounded ones), where the reference rounds behind it - the same
// relative error per probability (2^-11 at most; smaller where p would be subnormal), without the second K.q product and the second exponential of every score: 2.0e-4 of the result from
// float64 with two passes, 1.6e-4 with one.
// Bound by the LDS reads of the fragments (32 queries per wave: 32 KiB per 64 keys and wave at ~80 bytes per cycle and CU, about the time of the 32 matrix instructions) and the
// exponentials beside them. Against the two-pass form with 4 waves x 32 queries, 32-key tiles through registers: 6001 tokens x 32 heads 870 -> 393 us (752 TFLOP/s), 512 x 64 behind
// 1024 cached cells 102 -> 38, 101 x 32 behind 300 29.8 -> 11.7, 2048 x 32 144 -> 55. Requests by the waves that multiply / by their own, whole passes: 70B shape, three layers, 8 tokens behind 403
// cells 408 / 406, 72B shape, two layers, 23 tokens 461 / 459, 8B shape, four layers and head, 6001 13255 / 13215. (Both stages asked for at once in front, keys behind the last one left out: no change.)
// PLAIN: caches that do not start on 16 bytes, by loads and LDS stores instead of DMA
// PAIR: tiles of up to 32 queries, the two query waves of a key group are two heads of one KV head; their results leave as Q8_K blocks (the wo product's activations) - no f32 rows and no launch that
// quantizes them: 8 tokens x 64 heads behind 403 cells 11.3 + 5.0 us, with this ending 13.3, with waves that bring 12.0; 23 tokens and no other cells 11.8 / 9.0
// SELF: no waves that bring, each of the eight requests its share of the next stage (launch_prompt says where)
template <int DH, int QW, int KS, bool MASK, bool PLAIN = false, bool PAIR = false, bool SELF = false>
__global__ __launch_bounds__(SELF ? 512 : 768, !SELF ? 3 : DH == 64 ? 4 : 2) void attn_prompt_kernel(PfP p, pm_q8k_out y) {
    static_assert(!PAIR || !SELF, "the waves that bring store rows too");
    static_assert(!PAIR || (DH == 128 && QW == 2 && !MASK && !PLAIN), "two heads are a block");
    constexpr int KW = 8 / QW, KT = KS / KW, ST = KT / 32;            // keys per wave and stage, 32-key score tiles
    constexpr int KK = DH / 16, DT = DH / 32, CK = DH / 8, CV = KS / 8;      // k-steps of a score tile, output tiles, 16-byte chunks per K row / V^T row
    constexpr int STAGE = KS * DH * 4, OS = DH + 4;
    constexpr float LOG2E = 1.4426950408889634f;
    // the maxima below are in units of log2, with a mask in natural units - a mask entry times log2 e may overflow (the lowest f32 value), which would hide a cell that a row of such
    // entries attends - and start from the lowest value there is
    constexpr float NONE = MASK ? -INFINITY : -1e30f, UNIT = MASK ? LOG2E : 1.0f;
    static_assert(KT % 32 == 0, "whole score tiles");
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), lane = threadIdx.x & 63, lr = lane & 31, hf = lane >> 5;
    const int qw = wave % QW, kw = wave / QW;
    // an XCD (blockIdx % 8) keeps to its share of the heads: the query heads of a KV head meet in one L2. Tiles with the most keys first: the short ones fill the tail
    int h, tile;
    const int n_h = PAIR ? p.H / 2 : p.H;                         // (heads, or pairs of them)
    if (n_h % 8 == 0) { const int per = n_h / 8, j = blockIdx.x >> 3; h = (blockIdx.x & 7) * per + j % per; tile = j / per; }
    else { h = blockIdx.x % n_h; tile = blockIdx.x / n_h; }
    const int pair = h;
    if (PAIR) h = 2 * h + qw;
    tile = p.n_tiles - 1 - tile;
    const int hk = h / (p.H / p.Hkv);
    int row0 = tile * QW * 32, nq = min(QW * 32, p.T - row0), pos0 = 0, seq = 0;                 // the workgroup's first row, its queries, the first one's position
    if (!MASK && p.tiles) { row0 = p.tiles[4 * tile]; nq = p.tiles[4 * tile + 1]; pos0 = p.tiles[4 * tile + 2]; seq = p.tiles[4 * tile + 3]; }
    else { seq = p.seq_ptr ? *p.seq_ptr : 0; if (!MASK) pos0 = p.pos0_ptr[seq] + row0; }
    const long krow = (long) p.Hkv * DH;
    const uint16_t * kc = p.kc + (long) seq * p.seq_stride + (long) hk * DH;                     // K[key][Hkv*DH]
    const uint16_t * vc = p.vc + (long) seq * p.seq_stride + (long) hk * DH * p.n_ctx;           // V^T[hk*DH + e][n_ctx]
    const int q0 = PAIR ? 0 : qw * 32, tq0 = row0 + q0;                                                     // first query of this wave: in the workgroup, and its row
    const bool live = q0 < nq;
    const int qi = min(q0 + lr, nq - 1), tq = row0 + qi, qpos = pos0 + qi;
    const int w_first = pos0 + q0, w_last = pos0 + min(q0 + 31, nq - 1);                         // positions of the wave's first and last query
    const int n_keys = MASK ? p.n_kv : pos0 + nq;                                                // cells the workgroup's last query sees
    const int n_it = (n_keys + KS - 1) / KS;
    // cells this wave's queries see together
    const int seen = MASK ? p.n_kv : w_last + 1;

    const uint32_t lds0 = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) char *) smem;
    auto bring = [&](const char * base, uint32_t off, int to) __attribute__((always_inline)) {
        if constexpr (PLAIN) { u32x4 v; __builtin_memcpy(&v, base + off, 16); *(u32x4 *) (smem + to + lane * 16) = v; }
        else pm_dma16(base, off, lds0 + to);
    };
    // a stage: every RW-th piece of 1 KiB by each of the waves that request
    constexpr int RW = SELF ? 8 : 4;
    const int rw = SELF ? wave : wave - 8;
    auto request = [&](int it, int stage) __attribute__((always_inline)) {
        const char * kb = (const char *) (kc + (long) it * KS * krow), * vb = (const char *) vc;
        const int key0 = it * KS, kmax = p.n_ctx - 1 - key0, vmax = p.n_ctx - 8 - key0;          // (cells behind the cache: its last ones, masked)
#pragma unroll
        for (int i = 0; i < KS * DH * 2 / (1024 * RW); ++i) {
            const int o = (rw + i * RW) * 64 + lane, row = o / CK, ch = o % CK;
            bring(kb, (uint32_t) min(row, kmax) * (uint32_t) (krow * 2) + (uint32_t) (ch ^ (CK == 8 ? (row >> 1) & 7 : row & 15)) * 16u, stage * STAGE + (rw + i * RW) * 1024);
        }
#pragma unroll
        for (int i = 0; i < KS * DH * 2 / (1024 * RW); ++i) {
            const int o = (rw + i * RW) * 64 + lane, row = o / CV, ch = o % CV;
            const int key = key0 + min((ch ^ (CV == 8 ? (row >> 1) & 7 : row & 15)) * 8, vmax);
            bring(vb, (uint32_t) row * (uint32_t) (p.n_ctx * 2) + (uint32_t) key * 2u, stage * STAGE + KS * DH * 2 + (rw + i * RW) * 1024);
        }
    };
    float * const ex = (float *) smem, * const ml = ex + 8 * 32 * OS;      // behind the loop: [wave][query][DH + 4], [wave][query]{m, l}
    // PAIR: a wave per token, lanes 0 .. 31 the first head, 32 .. 63 the second
    auto rows_of_pair = [&] __attribute__((always_inline)) {
        for (int r = wave; r < nq; r += 12) {
            float4 a = *(const float4 *) (ex + (hf * 32 + r) * OS + 4 * lr);
#pragma unroll
            for (int g = 1; g < KW; ++g) {
                const float4 b = *(const float4 *) (ex + ((g * QW + hf) * 32 + r) * OS + 4 * lr);
                a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
            }
            const float v[4] = {a.x, a.y, a.z, a.w};
            q8k_block_from_regs(v, lane, y.y + (size_t) (row0 + r) * y.row_bytes, p.H * DH, pair, y.tab, row0 + r);
        }
    };
    if constexpr (SELF) request(0, 0);
    else if (wave >= 8) {
        request(0, 0);
        for (int it = 0; it < n_it; ++it) {
            pm_vm_drain();
            __syncthreads();
            if (it + 1 < n_it) request(it + 1, (it & 1) ^ 1);
        }
        __syncthreads();
        if (KW > 1) __syncthreads();
        __syncthreads();
        if constexpr (PAIR) rows_of_pair();
        return;
    }

    // Q^T as B operand: lane (query lr, hf) holds q[query][16 kk + 8 hf .. + 8], rounded to F16 like the reference
    half8 q[KK];
    {
        const float * qr = p.q + ((long) tq * p.H + h) * DH + 8 * hf;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const float4 a = *(const float4 *) (qr + 16 * kk), b = *(const float4 *) (qr + 16 * kk + 4);
            q[kk] = half8{(_Float16) a.x, (_Float16) a.y, (_Float16) a.z, (_Float16) a.w, (_Float16) b.x, (_Float16) b.y, (_Float16) b.z, (_Float16) b.w};
        }
    }
    if (!(p.scale > 0.0f)) {                                      // (the queries carry the sign of the scale: hidden scores are -inf in front of the positive factor c)
        const _Float16 sg = p.scale == 0.0f ? (_Float16) 0.0f : (_Float16) -1.0f;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) q[kk] *= sg;
    }
    const float * mrow = (const float *) p.mask + (long) tq * p.mask_stride;
    const uint16_t * mrow16 = (const uint16_t *) p.mask + (long) tq * p.mask_stride;
    float16v o[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
    float m = NONE, l = 0.0f;
    const float sc = p.scale == 0.0f ? 1.0f : fabsf(p.scale), c = sc * LOG2E;
    const int kr = (lr & ~12) | ((lr & 4) << 1) | ((lr & 8) >> 1);
    for (int it = 0; it < n_it; ++it) {
        const int stage = it & 1;
        if constexpr (SELF) pm_vm_drain();
        __syncthreads();
        if constexpr (SELF) if (it + 1 < n_it) request(it + 1, stage ^ 1);
        const int key0 = it * KS + kw * KT;
        if (!live || key0 >= seen) continue;
        // cells behind the last attended one: a probability of 0 does not undo what they hold (0 x NaN), so they become zeros in LDS. Every wave of a key group writes the same bytes and
        // waits for its own only. (The last stage's work: kept small and out of the loop's registers - unrolled, with addresses that the loop carries, it cost every stage the second set of
        // registers that its reads of K alternate between: 2 x 12000 cells of 64 heads 127 -> 135 us)
        if (key0 + KT > n_keys) {
            int row = lane;
            asm volatile("" : "+v"(row));
            const int n = max(n_keys - key0, 0);                   // attended cells of the key group: chunks n / 8 and behind
#pragma unroll 1
            for (; row < DH; row += 64) {
                char * at = smem + stage * STAGE + KS * DH * 2 + row * (KS * 2);
                const int sw = CV == 8 ? (row >> 1) & 7 : row & 15;
                u32x4 v = *(const u32x4 *) (at + ((kw * (KT / 8) + n / 8) ^ sw) * 16);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] &= n % 8 >= 2 * e + 2 ? 0xFFFFFFFFu : n % 8 == 2 * e + 1 ? 0xFFFFu : 0u;
#pragma unroll 1
                for (int ch = n / 8; ch < KT / 8; ++ch) { *(u32x4 *) (at + ((kw * (KT / 8) + ch) ^ sw) * 16) = v; v = u32x4{0, 0, 0, 0}; }
            }
        }
        const char * ks = smem + stage * STAGE, * vs = ks + KS * DH * 2;
        float16v s[ST];
#pragma unroll
        for (int t = 0; t < ST; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[t][r] = 0.0f;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
#pragma unroll
            for (int t = 0; t < ST; ++t) {
                const int row = kw * KT + t * 32 + kr;
                const half8 k = *(const half8 *) (ks + row * (DH * 2) + ((kk * 2 + hf) ^ (CK == 8 ? (row >> 1) & 7 : row & 15)) * 16);
                s[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(k, q[kk], s[t], 0, 0, 0);
            }
        float mx = NONE;
        if (MASK) {
#pragma unroll
            for (int t = 0; t < ST; ++t)
#pragma unroll
                for (int g = 0; g < 4; ++g) {                     // registers 4 g .. + 4 = keys 16 (g >> 1) + 8 hf + 4 (g & 1) .. + 4
                    const int k0 = key0 + t * 32 + 16 * (g >> 1) + 8 * hf + 4 * (g & 1);
                    if (k0 >= p.n_kv) {                           // (n_kv is a multiple of 4; whatever a cell behind n_kv holds, its score does not count)
                        s[t][4 * g + 0] = s[t][4 * g + 1] = s[t][4 * g + 2] = s[t][4 * g + 3] = -INFINITY;
                        continue;
                    }
                    float4 mv;
                    if (!p.mask_f16) mv = *(const float4 *) (mrow + k0);
                    else { const u32x2 mh = *(const u32x2 *) (mrow16 + k0); mv = float4{h2f((uint16_t) (mh[0] & 0xFFFF)), h2f((uint16_t) (mh[0] >> 16)), h2f((uint16_t) (mh[1] & 0xFFFF)), h2f((uint16_t) (mh[1] >> 16))}; }
                    s[t][4 * g + 0] = fmaf(s[t][4 * g + 0], sc, mv.x); s[t][4 * g + 1] = fmaf(s[t][4 * g + 1], sc, mv.y);
                    s[t][4 * g + 2] = fmaf(s[t][4 * g + 2], sc, mv.z); s[t][4 * g + 3] = fmaf(s[t][4 * g + 3], sc, mv.w);
                }
        } else if (key0 + KT - 1 > w_first) {                     // (keys that some query of the wave does not see)
#pragma unroll
            for (int t = 0; t < ST; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (key0 + t * 32 + 16 * (r >> 3) + 8 * hf + (r & 7) > qpos) s[t][r] = -INFINITY;
        }
#pragma unroll
        for (int t = 0; t < ST; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[t][r]);
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        if (!MASK) mx = fmaxf(mx * c, NONE);                      // (scores are scaled where the exponent is formed; c > 0)
        const float mn = fmaxf(m, mx), mr = MASK && mn == -INFINITY ? 0.0f : mn;      // (nothing visible so far: every exponent below is -inf)
        if (__any(mn > m)) {
            const float corr = __builtin_amdgcn_exp2f((m - mr) * UNIT);
            l *= corr; m = mn;
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[d][r] *= corr;
        }
        half8 pr[2 * ST];
#pragma unroll
        for (int t = 0; t < ST; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float e = __builtin_amdgcn_exp2f(MASK ? (s[t][r] - mr) * LOG2E : fmaf(s[t][r], c, -m));
                l += e;
                pr[2 * t + (r >> 3)][r & 7] = (_Float16) e;
            }
#pragma unroll
        for (int j = 0; j < 2 * ST; ++j) {
            if (ST > 1 && j == 2 && key0 + 32 >= seen) break;      // (nor do the later tokens' cells belong to the queries of this wave)
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const int row = d * 32 + lr, ch = kw * (KT / 8) + 2 * j + hf;
                const half8 v = *(const half8 *) (vs + row * (KS * 2) + (ch ^ (CV == 8 ? (row >> 1) & 7 : row & 15)) * 16);
                o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, pr[j], o[d], 0, 0, 0);
            }
        }
    }
    l += __shfl_xor(l, 32);
    __syncthreads();                                              // (the stages become the exchange of the results)
    float f = 1.0f / l;
    if (KW > 1) {
        if (hf == 0) { ml[(wave * 32 + lr) * 2] = m; ml[(wave * 32 + lr) * 2 + 1] = l; }
        __syncthreads();
        float M = NONE, L = 0.0f;
#pragma unroll
        for (int g = 0; g < KW; ++g) M = fmaxf(M, ml[((g * QW + qw) * 32 + lr) * 2]);
#pragma unroll
        for (int g = 0; g < KW; ++g) L += ml[((g * QW + qw) * 32 + lr) * 2 + 1] * __builtin_amdgcn_exp2f((ml[((g * QW + qw) * 32 + lr) * 2] - M) * UNIT);
        f = __builtin_amdgcn_exp2f((m - M) * UNIT) / L;
    }
    // O^T[d][query]: queries are columns; through LDS, then a wave stores whole rows
    if (q0 + lr < nq)
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *(float4 *) (ex + (wave * 32 + lr) * OS + d * 32 + 8 * g + 4 * hf) = float4{o[d][4 * g] * f, o[d][4 * g + 1] * f, o[d][4 * g + 2] * f, o[d][4 * g + 3] * f};
    __syncthreads();
    if constexpr (PAIR) { rows_of_pair(); return; }
    constexpr int RL = DH / 4, RP = 64 / RL;                       // lanes per row (4 values each), rows per pass
    for (int r = kw * (32 / KW) + lane / RL; r < (kw + 1) * (32 / KW); r += RP) {
        if (q0 + r >= nq) break;
        float4 a = *(const float4 *) (ex + (qw * 32 + r) * OS + 4 * (lane % RL));
#pragma unroll
        for (int g = 1; g < KW; ++g) {
            const float4 b = *(const float4 *) (ex + ((g * QW + qw) * 32 + r) * OS + 4 * (lane % RL));
            a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
        }
        const long at = ((long) (tq0 + r) * p.H + h) * DH + 4 * (lane % RL);
        if (p.out_h) *(half4 *) (p.out_h + at) = half4{(_Float16) a.x, (_Float16) a.y, (_Float16) a.z, (_Float16) a.w};
        else *(float4 *) (p.out + at) = a;
    }
}

template <int DH, int QW, int KS, bool MASK, bool PLAIN = false, bool PAIR = false, bool SELF = false> void launch_form(const PfP & p, hipStream_t st, const pm_q8k_out & y) {
    constexpr size_t stages = 2 * (size_t) KS * DH * 4, ex = (size_t) 8 * 32 * (DH + 4) * 4 + 8 * 32 * 2 * 4, lds = stages > ex ? stages : ex;
    pm_allow_big_lds((const void *) attn_prompt_kernel<DH, QW, KS, MASK, PLAIN, PAIR, SELF>, lds);
    hipLaunchKernelGGL((attn_prompt_kernel<DH, QW, KS, MASK, PLAIN, PAIR, SELF>), dim3(p.n_tiles * (PAIR ? p.H / 2 : p.H)), dim3(SELF ? 512 : 768), lds, st, p, y);
}
// Heads of 64: eight waves of up to 128 registers and half of the LDS leave room for a second workgroup on a CU, eight waves and four that bring do not. Where there are more workgroups than CUs, two
// at a time win. us, waves that bring / two workgroups: 48 heads x 640 tokens 15.1 / 14.1, 64 x 1000 27.5 / 25.6, 96 x 2048
// 92.0 / 83.5, with a mask 48 x 512 behind 1024 cells 57.4 / 43.9. With a mask, tiles of 128 and 256 queries took 130 and 136 registers, one workgroup: 64 x 1000 66.2, with waves that bring 65.1
// Heads of 128 with a mask, tiles of 128 and 256 queries: 168 registers a wave, what waves that bring leave, are too few (186 and 196 without). us, with them (two spilled) / without: 64 heads
// x 1000 tokens 85.3 / 87.4, 64 x 512 behind 1024 cells 64.6 / 64.4, 48 x 2500 417 / 406, 64 x 2500 583 / 571, 128 x 2500 1168 / 1013
template <int DH, int QW, int KS, bool MASK, bool PLAIN = false, bool PAIR = false> void launch_prompt(PfP p, hipStream_t st, const pm_q8k_out & y = {}) {
    if (!p.tiles) p.n_tiles = (p.T + QW * 32 - 1) / (QW * 32);
    if constexpr (DH == 64 && (!MASK || QW == 2)) if ((long) p.n_tiles * p.H > pm_device_cus()) return launch_form<DH, QW, KS, MASK, PLAIN, PAIR, true>(p, st, y);
    launch_form<DH, QW, KS, MASK, PLAIN, PAIR, DH == 128 && MASK && QW != 2>(p, st, y);
}
// Which tile: a CU holds one workgroup. 256 queries share a stage where that still makes two rounds of workgroups (2048 tokens x 64 heads: 102 us, 110 with 128 queries; x 32 heads
// = one round whose longest tile decides: 80 against 57); 128 queries where they make one (512 x 64 behind 1024 cached: 38 against 50 with 64); below that 64 queries with four key
// groups each (101 x 32 behind 300: 11.7 against 14.9).
int tile_of(int n_tok, int H) {
    const int cus = pm_device_cus();
    return (n_tok + 255) / 256 * H >= 2 * cus ? 256 : (n_tok + 127) / 128 * H >= cus ? 128 : 64;
}
template <int DH, bool MASK> void launch_prompt_dh(const PfP & p, int tile_q, hipStream_t st) {
    if (((uintptr_t) p.kc | (uintptr_t) p.vc) & 15) launch_prompt<DH, 2, 128, MASK, true>(p, st);
    else if (tile_q == 256) launch_prompt<DH, 8, 64, MASK>(p, st);
    else if (tile_q == 128) launch_prompt<DH, 4, 128, MASK>(p, st);
    else launch_prompt<DH, 2, 128, MASK>(p, st);
}

} // namespace

int pm_attn_prefill_tile(int n_tok, int H) { return tile_of(n_tok, H); }

// n_ctx % 32 == 0 and head_dim 64 / 128 only (callers fall back to the per-token kernel otherwise)
int pm_launch_attn_prefill(const float * q, const void * kc, const void * vc, const int32_t * pos0, const int32_t * seq,
                           long seq_stride, float * out, int n_tok, int H, int Hkv, int dh, int n_ctx, float scale, hipStream_t st,
                           const float * mask, long mask_stride, int n_kv, int v_rowmajor, int mask_f16, void * out_f16, const int32_t * tiles, int n_tiles, int tile_q) {
    if ((dh != 64 && dh != 128) || n_ctx % 32 || n_tok < 1) return -1;
    if (mask && (n_kv < 1 || n_kv > n_ctx || n_kv % 4 || mask_stride % 4)) return -1;
    if ((v_rowmajor || mask_f16) && !mask) return -1;                 // the flash-attention form exists in ggml-graph mode only
    PfP p = {q, (const uint16_t *) kc, (const uint16_t *) vc, pos0, seq, seq_stride, out, n_tok, H, Hkv, n_ctx, scale, mask, mask_stride, n_kv, mask_f16 ? 1 : 0, (_Float16 *) out_f16, tiles, n_tiles};
    if (tiles && (mask || n_tiles < 1 || (((uintptr_t) kc | (uintptr_t) vc) & 15))) return -1;
    if (!tiles) tile_q = tile_of(n_tok, H);
    if (v_rowmajor) {
        if (out_f16 || seq) return -1;
        const dim3 grid((n_tok + 127) / 128, H);
        if (dh == 128) hipLaunchKernelGGL(attn_rowmajor_kernel<128>, grid, dim3(256), 0, st, p);
        else           hipLaunchKernelGGL(attn_rowmajor_kernel<64>, grid, dim3(256), 0, st, p);
    } else if (dh == 128) {
        if (mask) launch_prompt_dh<128, true>(p, tile_q, st); else launch_prompt_dh<128, false>(p, tile_q, st);
    } else {
        if (mask) launch_prompt_dh<64, true>(p, tile_q, st); else launch_prompt_dh<64, false>(p, tile_q, st);
    }
    return 0;
}

int pm_launch_attn_prefill_q8k(const float * q, const void * kc, const void * vc, const int32_t * pos0, const int32_t * seq, long seq_stride, int n_tok, int H, int Hkv, int dh, int n_ctx,
                               float scale, hipStream_t st, const int32_t * tiles, int n_tiles, const pm_q8k_out & out) {
    if (dh != 128 || n_ctx % 32 || n_tok < 1 || n_tok > 32 || H / Hkv % 2 || (tiles && n_tiles < 1) || (((uintptr_t) kc | (uintptr_t) vc) & 15)) return -1;
    const PfP p = {q, (const uint16_t *) kc, (const uint16_t *) vc, pos0, seq, seq_stride, nullptr, n_tok, H, Hkv, n_ctx, scale, nullptr, 0, 0, 0, nullptr, tiles, n_tiles};
    launch_prompt<128, 2, 128, false, false, true>(p, st, out);
    return 0;
}
