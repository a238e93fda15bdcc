// dense_small.hip — y[t][n] = act(W[n] . x[t] + bias) for up to 64 tokens per pass over dense weights: every weight is read once per 64 tokens, straight from HBM into
// the A operand of 16 x 16 matrix-core tiles (rows of W = rows of the tile, tokens = its columns). HBM-bound: a workgroup owns 16 or 32 rows, its eight waves take
// interleaved 64-k blocks of them and add up through LDS. Both number formats: bf16 (v_mfma_f32_16x16x32_bf16) and f32 (v_mfma_f32_16x16x4_f32); the order of k inside a
// block is the one in which a lane's 16-byte loads lie (both operands agree on it).
// With a few tokens the prologue x + norm(y) runs in every workgroup (one launch less; the residual row is written by the first).
// The same body serves one matrix per attention head (groups of rows with activations of their own) and experts: with a few tokens one workgroup row per (token, expert)
// pair, which routes its token in the prologue where no launch has, and a down product over the concatenation of a token's experts; with more one row per expert that has tokens.
#include "pm355_dense.h"
#include "pm355_kernels.h"
#include "pm355_route.h"
#include <algorithm>
#include "../../include/prima_mi355.h"

namespace {

enum { DENSE = 0, PAIR = 1, CONCAT = 2, SORTED = 3 };
struct SmallP {
    const void * W; const void * act; void * y; const float * bias; pm_add_norm pro;
    int K, T, lda, ldy, y_type, n_store, act_fn;
    int group, g_act, g_out, g_store; pm_split_merge merge;
    // experts: values between two of them; SORTED: rows in / out are sorted pairs (in_sorted / out_sorted) or tokens / pairs
    pm_route r; int64_t e_stride; int in_sorted, out_sorted, weigh;
};
// The norm prologue pays where a launch is short: up to this width x tokens (rounded up to a power of two). Wider rows cost every workgroup more than one norm launch does
// (width 2048: 8.3 us against 6.7 + 3.0; 4096: 20.8 against 15.5 + 4.2; 8192: 87 against 57 + 7)
constexpr int PRO_MAX = 2048;

template <typename T> struct Frag;                         // one 16-byte load per lane
template <> struct Frag<uint16_t> {
    static constexpr int PER_BLOCK = 2;                    // loads per lane and 64-k block
    static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
};
template <> struct Frag<float> {
    static constexpr int PER_BLOCK = 4;
    static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
        const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
        for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], c, 0, 0, 0);
        return c;
    }
};

__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
    v |= (uint32_t) dpp_i<0xB1>((int) v); v |= (uint32_t) dpp_i<0x4E>((int) v); v |= (uint32_t) dpp_i<0x141>((int) v); v |= (uint32_t) dpp_i<0x140>((int) v);
    v |= other_row(v);
    return (uint32_t) __builtin_amdgcn_readfirstlane((int) (v | other_half(v)));
}

// x + norm(y) of token wave / (8 / TP) in VP values per lane: everything the rows need is requested before the first weights (loads return in order), the sums run
// while those are on their way. Result -> LDS (T, stride ldl) and, from workgroup 0, the residual stream.
template <typename T, int TP> struct AddNorm {
    static constexpr int NW = 8 / TP, VP = PRO_MAX / 512;
    float y[VP], x[VP], w[VP], b[VP], w2[VP];
    int t, l;
    __device__ __forceinline__ void request(const SmallP & p, int wave, int lane) {
        const pm_add_norm & q = p.pro;
        t = wave / NW; l = (wave % NW) * 64 + lane;
        const int tt = t < p.T ? t : 0;
#pragma unroll
        for (int i = 0; i < VP; ++i) {
            const int c = i * NW * 64 + l, cc = c < q.width ? c : q.width - 1;
            y[i] = ld_g(q.y + (size_t) tt * q.ldy + cc);
            x[i] = q.x ? ld_g(q.x + (size_t) tt * q.ldx + cc) : 0.0f;
            w[i] = ld_g(q.w + cc);
            b[i] = q.b ? ld_g(q.b + cc) : 0.0f;
            w2[i] = q.w2 ? ld_g(q.w2 + cc) : 1.0f;
        }
    }
    __device__ __forceinline__ float token_sum(float s, float * red, int wave, int lane) const {
        s = wave_sum(s);
        if (lane == 0) red[wave] = s;
        __syncthreads();
        float o = 0.0f;
#pragma unroll
        for (int i = 0; i < NW; ++i) o += red[t * NW + i];
        return o;
    }
    __device__ __forceinline__ void finish(const SmallP & p, T * rows, int ldl, float * red, int wave, int lane) {
        const pm_add_norm & q = p.pro;
        float s = 0.0f, mean = 0.0f;
        if (!q.rms) {
#pragma unroll
            for (int i = 0; i < VP; ++i) s += i * NW * 64 + l < q.width ? y[i] : 0.0f;
            mean = token_sum(s, red, wave, lane) / (float) q.width;
        }
        float s2 = 0.0f;
#pragma unroll
        for (int i = 0; i < VP; ++i) { const float d = i * NW * 64 + l < q.width ? y[i] - mean : 0.0f; s2 = fmaf(d, d, s2); }
        const float rs = 1.0f / sqrtf(token_sum(s2, red + 8, wave, lane) / (float) q.width + q.eps);
        float s3 = 0.0f;
#pragma unroll
        for (int i = 0; i < VP; ++i) { x[i] += (y[i] - mean) * rs * w[i] + b[i]; s3 += i * NW * 64 + l < q.width ? x[i] * x[i] : 0.0f; }
        const float r2 = q.w2 ? 1.0f / sqrtf(token_sum(s3, red + 16, wave, lane) / (float) q.width + q.eps) : 1.0f;
        if (t < p.T) {
#pragma unroll
            for (int i = 0; i < VP; ++i) {
                const int c = i * NW * 64 + l;
                const T v = from_f<T>(x[i] * (r2 * w2[i]));
                if (c < q.width) {
                    rows[t * ldl + c] = v;
                    if (blockIdx.x == 0 && q.x_out) q.x_out[(size_t) t * q.ldo + c] = x[i];
                    if (blockIdx.x == 0 && q.act_out) ((T *) q.act_out)[(size_t) t * q.ld_act + c] = v;
                } else if (c < p.K) rows[t * ldl + c] = from_f<T>(0.0f);
            }
        }
        for (int c = NW * VP * 64 + l; c < p.K && t < p.T; c += NW * 64) rows[t * ldl + c] = from_f<T>(0.0f);
        __syncthreads();
    }
};

// SRC, where the activations come from: 0 global memory (they ride in the load groups: the vector-memory counter is in order, a later load must not be waited for in front
// of an earlier one), -1 LDS (copied once), 1 / 2 / 4 the norm prologue for that many tokens (LDS).
// LINE (bf16, activations in LDS, up to 8 tokens): the 16 tile rows are 8 rows of W x 2 halves of a 64-k block and the 16 columns 8 tokens x the same 2 halves, so that one
// load instruction covers whole 128-byte lines (a line that two instructions touch is requested twice); of the result the blocks with equal halves count.
template <typename T, int NT, int RM, int SRC, int EXP> __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void dense_small_kernel(SmallP p) {
    constexpr bool LINE = sizeof(T) == 2 && SRC != 0;
    constexpr int ROWS = LINE ? 8 : 16, TOK = LINE ? 8 : 16, EPL = 16 / sizeof(T);
    // PB loads per lane and 64-k block, U blocks per load group: about eight 16-byte weight loads per lane, two groups in flight
    constexpr int PB = LINE ? 1 : Frag<T>::PER_BLOCK, NB = SRC == 0 ? NT : 0, UG = 8 / (PB * (RM + NB)), U = UG < 1 ? 1 : UG;
    constexpr bool TWO = NB < 4;                           // (NT = 4: one group, its registers are taken by the products)
    extern __shared__ __attribute__((aligned(16))) char smem[];
    float * red = (float *) smem;                                                                  // [8 waves][NT][RM][16 columns][16 rows]
    const int wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), lane = threadIdx.x & 63, lr = lane & 15, g = lane >> 4;
    const int r0 = blockIdx.x * ROWS * RM;
    // this workgroup's matrix, activations and tokens
    const T * W = (const T *) p.W, * act = (const T *) p.act;
    int t0 = blockIdx.y * TOK * NT, n_tok = p.T, base = 0;
    float weight = 1.0f;
    const int32_t * cat = nullptr;                         // CONCAT: the token's experts
    (void) cat;
    if constexpr (EXP == PAIR) {                           // base: the pair, which is also its row of y
        __shared__ int ids[64]; __shared__ float w[64];
        const int top = p.r.top, t = blockIdx.y / top, k = blockIdx.y % top;
        if (wave == 0) {
            if (p.r.logits) {
                route_token([&](int e) { return ld_g(p.r.logits + (size_t) t * p.r.ldl + e); }, p.r.E, top, p.r.groups, p.r.keep, (float *) smem, (float *) smem + 1024, ids, w);
                if (blockIdx.x == 0 && k == 0 && lane < top) { p.r.id[t * top + lane] = ids[lane]; p.r.w[t * top + lane] = w[lane]; }
            } else if (lane == k) { ids[k] = ld_g(p.r.id + blockIdx.y); w[k] = ld_g(p.r.w + blockIdx.y); }
        }
        __syncthreads();
        W += (size_t) __builtin_amdgcn_readfirstlane(ids[k]) * p.e_stride;
        weight = w[k]; base = blockIdx.y; act += (size_t) t * p.lda; t0 = 0; n_tok = 1;
    }
    if constexpr (EXP == CONCAT) { const int t = blockIdx.y; cat = uniform_const_ptr(p.r.id + t * p.r.top); base = t; act += (size_t) t * p.lda; t0 = 0; n_tok = 1; }
    __shared__ int local[EXP == SORTED ? PM_ROUTE_PAIRS : 1];          // SORTED without tables: the expert's pairs
    // SORTED: the workgroup's experts are the blockIdx.y-th, (blockIdx.y + gridDim.y)-th, .. that have pairs
    constexpr int G = EXP == SORTED ? PM_ROUTE_PAIRS / 64 : 1;
    int mine_e[G], ye = blockIdx.y, n_on = 0;
    uint64_t on = 0;
    if constexpr (EXP == SORTED) {
        if (p.r.logits) n_on = __builtin_amdgcn_readfirstlane(ld_g(p.r.active));
        else {
            // up to PM_ROUTE_PAIRS pairs of up to 64 experts: a lane per pair, 64 at a time. (One round of loads in front of the weights instead of three, one behind the other, and no launch that
            // sorts; every wave finds the same)
            const int pairs = p.T * p.r.top;
#pragma unroll
            for (int i = 0; i < G; ++i) { mine_e[i] = 64; if (i * 64 < pairs && i * 64 + lane < pairs) mine_e[i] = ld_g(p.r.id + i * 64 + lane); }       // (64: no expert)
            uint32_t has[2] = {0, 0};
#pragma unroll
            for (int i = 0; i < G; ++i)
                if (i * 64 < pairs) { has[0] |= mine_e[i] < 32 ? 1u << mine_e[i] : 0u; has[1] |= mine_e[i] >= 32 && mine_e[i] < 64 ? 1u << (mine_e[i] - 32) : 0u; }
            on = (p.r.E > 32 ? (uint64_t) wave_or(has[1]) << 32 : 0) | wave_or(has[0]);
            n_on = __popcll(on);
        }
        if (ye >= n_on) return;
    }
    auto take = [&]() __attribute__((always_inline)) {                  // the ye-th of them
        int e;
        if (p.r.logits) {
            e = __builtin_amdgcn_readfirstlane(ld_g(p.r.active + 1 + ye));
            base = __builtin_amdgcn_readfirstlane(ld_g(p.r.off + e)); n_tok = __builtin_amdgcn_readfirstlane(ld_g(p.r.off + e + 1)) - base;
        } else {
            e = __builtin_ctzll(__builtin_amdgcn_ballot_w64((on >> lane & 1) && __popcll(on & ((1ull << lane) - 1)) == ye));
            base = 0; n_tok = 0;
#pragma unroll
            for (int i = 0; i < G; ++i) {
                if (i * 64 >= p.T * p.r.top) break;
                const uint64_t its = __builtin_amdgcn_ballot_w64(mine_e[i] == e);
                base += __popcll(__builtin_amdgcn_ballot_w64(mine_e[i] < e));
                if (its >> lane & 1) local[n_tok + __popcll(its & ((1ull << lane) - 1))] = i * 64 + lane;
                n_tok += __popcll(its);
            }
            wave_fence();
        }
        W = (const T *) p.W + (size_t) e * p.e_stride; t0 = 0;
    };
    if constexpr (EXP == SORTED) take();
    // sorted pair base + t
    auto pair_at = [&](int t) __attribute__((always_inline)) -> int { return EXP == SORTED && !p.r.logits ? local[t] : ld_g(p.r.order + base + t); };
    if (EXP == DENSE && p.group) act += (size_t) (r0 / p.group) * p.g_act;
    // activation row of the tile's token t (< n_tok)
    auto row_in = [&](int t) __attribute__((always_inline)) -> const T * {
        if constexpr (EXP == PAIR || EXP == CONCAT) return act;
        if constexpr (EXP == SORTED) return act + (size_t) (p.in_sorted ? base + t : pair_at(t) / p.r.top) * p.lda;
        return act + (size_t) t * p.lda;
    };
    const int nb1 = p.K >> 6, nblk = EXP == CONCAT ? nb1 * p.r.top : nb1, mine = (nblk - wave + 7) >> 3;      // 64-k blocks wave, wave + 8, ..
    const int koff = (LINE ? (lr >> 3) * 32 : 0) + g * EPL;
    const T * wrow[RM];
    auto w_at = [&](int blk) __attribute__((always_inline)) -> int64_t {      // of a 64-k block in a row of W
        if constexpr (EXP == CONCAT) { const int s = blk / nb1; return (int64_t) cat[s] * p.e_stride + ((blk - s * nb1) << 6); }
        return blk << 6;
    };
    do {
#pragma unroll
    for (int m = 0; m < RM; ++m) wrow[m] = W + (size_t) (r0 + m * ROWS + lr % ROWS) * p.K + koff;
    const T * arow[NT];
    if (SRC == 0) {
#pragma unroll
        for (int n = 0; n < NT; ++n) { const int t = t0 + n * 16 + lr; arow[n] = row_in(t < n_tok ? t : n_tok - 1) + koff; }
    }
    struct Group { u32x4 w[U][RM][PB], x[U][NB ? NB : 1][PB]; };
    auto load = [&](Group & a, int grp) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = grp * U + u, blk = wave + (i < mine ? i : mine - 1) * 8, k = blk << 6;   // (past the end: the last block again, not multiplied)
            const int64_t wk = w_at(blk);
#pragma unroll
            for (int s = 0; s < PB; ++s) {
#pragma unroll
                for (int n = 0; n < NB; ++n) a.x[u][n][s] = *(const PM_G u32x4 *) (arow[n] + k + s * (64 / PB));
#pragma unroll
                for (int m = 0; m < RM; ++m) a.w[u][m][s] = ld_nt16(wrow[m] + wk + s * (64 / PB));
            }
        }
    };
    AddNorm<T, SRC < 1 ? 1 : SRC> norm;
    if (SRC > 0) norm.request(p, wave, lane);
    Group ga, gb;
    (void) gb;
    if (mine > 0) load(ga, 0);                             // the first weights are on their way while the activations are made
    if (SRC != 0) {
        const int kk = nblk << 6, ldl = kk + EPL;
        T * rows = (T *) (smem + 8 * NT * RM * 1024);
        const int here = n_tok - t0 < TOK ? n_tok - t0 : TOK;
        if (SRC > 0) norm.finish(p, rows, ldl, red, wave, lane);
        else if (EXP == DENSE && sizeof(T) == 2 && p.merge.part) {
            // the activations are sums over key splits (wave t: the shares of token t's splits)
            __shared__ float share[8 * 64];
            const int h = r0 / p.group < p.merge.H ? r0 / p.group : p.merge.H - 1;
            const size_t ht = (p.merge.H + 15) / 16;
            const pm_split_merge & q = p.merge;
            if (wave < here) {
                const size_t slot = (size_t) (t0 + wave) * ht + h / 16;
                const float * ml = q.ml + ((slot * q.splits + (lane < q.splits ? lane : 0)) * 16 + h % 16) * 2;
                const float m = lane < q.splits ? ld_g(ml) : -1e30f, l = lane < q.splits ? ld_g(ml + 1) : 0.0f, f = __builtin_amdgcn_exp2f(m - wave_max(m));
                share[wave * 64 + lane] = f / wave_sum(l * f);
            }
            __syncthreads();
            const int n2 = kk / 2;
            for (int i = threadIdx.x; i < here * n2; i += 512) {
                const int t = i / n2, c = (i - t * n2) * 2;
                const float * src = q.part + ((((size_t) (t0 + t) * ht + h / 16) * q.splits) * 16 + h % 16) * kk + c;
                float a0 = 0.0f, a1 = 0.0f;
                for (int s0 = 0; s0 < q.splits; s0 += 16) {
                    float2 v[16];
#pragma unroll
                    for (int s = 0; s < 16; ++s) v[s] = __builtin_bit_cast(float2, *(const PM_G u32x2 *) (src + (size_t) (s0 + s < q.splits ? s0 + s : 0) * 16 * kk));
#pragma unroll
                    for (int s = 0; s < 16; ++s) { const float w = s0 + s < q.splits ? share[t * 64 + s0 + s] : 0.0f; a0 = fmaf(v[s].x, w, a0); a1 = fmaf(v[s].y, w, a1); }
                }
                rows[t * ldl + c] = from_f<T>(a0); rows[t * ldl + c + 1] = from_f<T>(a1);
            }
            __syncthreads();
        } else {
            const int n16 = kk / EPL;
            for (int t = 0; t < here; ++t) {
                const T * src = row_in(t0 + t);
                for (int i = threadIdx.x; i < n16; i += 512) *(u32x4 *) (rows + t * ldl + i * EPL) = *(const PM_G u32x4 *) (src + i * EPL);
            }
            __syncthreads();
        }
        const int t = lr % TOK;
        arow[0] = rows + (t < here ? t : here - 1) * ldl + koff;
    }
    f32x4 acc[NT][RM];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < RM; ++m) acc[n][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto mma = [&](const Group & a, int grp, bool full) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = grp * U + u, k = (wave + i * 8) << 6;
            if (!full && i >= mine) break;
#pragma unroll
            for (int s = 0; s < PB; ++s)
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    u32x4 x;
                    if (NB) x = a.x[u][n][s]; else x = *(const u32x4 *) (arow[n] + k + s * (64 / PB));
#pragma unroll
                    for (int m = 0; m < RM; ++m) acc[n][m] = Frag<T>::mma(a.w[u][m][s], x, acc[n][m]);
                }
        }
    };
    // two register sets, the next group's loads in front of this group's products
    const int ng = (mine + U - 1) / U;
    int i = 0;
    if (!TWO) for (; i < ng; ++i) { if (i) load(ga, i); mma(ga, i, false); }
    else for (; i + 2 < ng; i += 2) { load(gb, i + 1); mma(ga, i, true); load(ga, i + 2); mma(gb, i + 1, true); }
    if (TWO && ng - i == 2) { load(gb, i + 1); mma(ga, i, true); mma(gb, i + 1, false); }
    else if (TWO && ng - i == 1) mma(ga, i, false);
    // A wave with nothing left to multiply comes here by a jump, and behind one of those jumps ROCm 7.2's compiler left out the wait states between a product and the store
    // that reads it (seen in the assembly of the sorted-experts kernels, and in their results): they are spelled out. 20 states: the longest such wait there is
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < RM; ++m) asm volatile("" : "+v"(acc[n][m]));
    asm volatile("s_nop 15\n\ts_nop 3");
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < RM; ++m) asm volatile("" : "+v"(acc[n][m]));
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < RM; ++m) *(f32x4 *) (red + (((wave * NT + n) * RM + m) * 16 + lr) * 16 + g * 4) = acc[n][m];
    __syncthreads();
    for (int o = threadIdx.x; o < NT * RM * ROWS * TOK; o += 512) {
        const int r = o % ROWS, m = o / ROWS % RM, t = o / ROWS / RM, n = t / TOK, tt = t % TOK;      // rows fastest: a token's rows are stored as one segment
        const int row = r0 + m * ROWS + r;
        int tok = t0 + t, col = row;
        if (tok >= n_tok) continue;
        if (EXP == DENSE && p.group) {
            const int h = row / p.group, hr = row - h * p.group;
            if (hr >= p.g_store) continue;
            col = h * p.g_out + hr;
        }
        if (col >= p.n_store) continue;
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < 8; ++w) {
            const float * q = red + (((w * NT + n) * RM + m) * 16 + tt) * 16 + r;
            v += q[0];
            if (LINE) v += q[8 * 16 + 8];
        }
        if (p.bias) v += p.bias[row];
        v = act_apply(p.act_fn, v);
        if constexpr (EXP == PAIR) { v *= weight; tok = base; }
        if constexpr (EXP == CONCAT) tok = base;
        if constexpr (EXP == SORTED) {
            const int pair = pair_at(tok);
            if (p.weigh) v *= ld_g(p.r.w + pair);
            tok = p.out_sorted ? base + tok : pair;
        }
        st_type(p.y, (size_t) tok * p.ldy + col, p.y_type, v);
    }
    if constexpr (EXP == SORTED) {
        t0 += TOK * NT;
        __syncthreads();
        if (t0 >= n_tok && (ye += gridDim.y) < n_on) take();
    }
    } while (EXP == SORTED && t0 < n_tok);
}

// The same product over ONE bf16 matrix for up to 8 tokens: workgroups that stay (two per CU) take the row tiles blockIdx.x, + gridDim.x, .. one after another. A workgroup per
// tile copies all activations for every 8 or 16 rows - six tokens of 4096 values are 48 KB against 64 KB of weights -, behind a barrier, and has nothing on its way while it
// starts and while it adds up; what bounds the product is the read of the weights. Here the load groups of all tiles are one sequence, two of them in flight, the next one
// requested right behind the products that free its registers, also across the end of a tile. TP = 4 or 8: the activations of that many tokens are copied to LDS once, by DMA and
// by the wave that multiplies them (a wave has every 8th 64-k block of all rows: no barrier). TP = 0: they do not fit and ride in the load groups; 16 rows share them, one workgroup
// per CU with twice the registers. The bias rides there too (loads return in order: one of its own would wait for the weights in flight).
// Weights from memory, in us before / now: 14336 x 4096 3 tokens 27.9 / 22.5, 6 30.4 / 22.7 (5.2 TB/s); 4096 x 14336 6 tokens 33.2 / 24.3; 32000 x 4096 6 tokens 59 / 45.7 (5.7 TB/s);
// 28672 x 8192 5 tokens 133 / 77 (6.1 TB/s). What the first loads need stands first among the arguments (in registers when the launch starts) and the tiles of a
// workgroup are counted by the host (no division, no grid size from memory): 108 launches of a pass of 6 tokens of 36 layers, 5219 -> 5178 us a pass. Taken back: two sum buffers in turn for one barrier less (spills at RM = 2, 32000 x 2048 25.1 -> 26.6).
template <int RM, int TP> __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(TP == 0 && RM == 2 ? 2 : 4))) void dense_rows_kernel(const void * W0, const void * act0, int K0, int T0, int lda0, int G, int each, int rest, SmallP p) {
    p.W = W0; p.act = act0; p.K = K0; p.T = T0; p.lda = lda0;
    constexpr int U = TP ? 8 / RM : 4, NL = U * (RM + (TP ? 0 : 1)) + 1, ROWS = 8 * RM;            // 64-k blocks and loads of a group
    extern __shared__ __attribute__((aligned(16))) char smem[];
    float * red = (float *) smem;                                                                  // [8 waves][RM][16 columns][16 rows]
    const int wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), lane = threadIdx.x & 63, lr = lane & 15, g = lane >> 4;
    const int nblk = p.K >> 6, mine = (nblk - wave + 7) >> 3, ng = mine > U ? (mine + U - 1) / U : 1;      // 64-k blocks wave, wave + 8, .. ; load groups per tile
    const int my_tiles = each + ((int) blockIdx.x < rest), total = my_tiles * ng;      // (tiles = each G + rest)
    const uint16_t * W = (const uint16_t *) p.W;
    const uint32_t at = (uint32_t) ((lr >> 3) * 32 + g * 8), tok = (lr & 7) < p.T ? lr & 7 : p.T - 1;
    uint32_t w_off[RM];
#pragma unroll
    for (int m = 0; m < RM; ++m) w_off[m] = ((uint32_t) (m * 8 + (lr & 7)) * (uint32_t) p.K + at) * 2;
    // the element of a tile that this thread stores: rows fastest, a token's rows are one segment
    const int o_row = threadIdx.x % ROWS, o_tok = threadIdx.x / ROWS;
    // this wave's blocks of the activations: [block][TP tokens][8 pieces of 16 bytes, piece p in place p ^ token / 2]
    char * xs = smem + 8 * RM * 1024 + (size_t) wave * ((nblk + 7) >> 3) * (TP * 128);
    if constexpr (TP != 0) {
        constexpr int PER = 8 / TP;                                                                // blocks per request
        const int t = lane >> 3 & (TP - 1), b = lane >> 3 >> (TP == 8 ? 3 : 2);
        const uint32_t src = ((uint32_t) t * (uint32_t) p.lda + (uint32_t) (((lane & 7) ^ (t >> 1)) * 8)) * 2 + (uint32_t) (wave + b * 8) * 128, dst = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) char *) xs;
        for (int i = 0; i < mine; i += PER)
            if (t < p.T && i + b < mine) pm_dma16(p.act, src + (uint32_t) i * 1024, dst + (uint32_t) i * (TP * 128));
    }
    const char * x_at = xs + (TP ? (tok * 128 + (((lr >> 3) * 4 + g) ^ (tok >> 1)) * 16) : 0);
    const uint32_t x_off = (tok * (uint32_t) p.lda + at) * 2;
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *) p.bias, 0, p.bias ? p.n_store * 4 : 0, 0x00020000);
    struct Group { u32x4 w[U][RM], x[TP ? 1 : U]; float bias; };
    int l_tile = (int) blockIdx.x, l_grp = 0;                                                      // the next group to be requested
    auto load = [&](Group & a) __attribute__((always_inline)) {
        const uint16_t * at_tile = W + (size_t) l_tile * ROWS * p.K;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // past the end of a row: out of the bounds of an empty buffer, no traffic (the last block again would be waited for)
            const int i = l_grp * U + u, in = i < mine, soff = in ? (wave + i * 8) * 128 : 0;
            if (TP == 0) {
                const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *) p.act, 0, in ? ((p.T - 1) * p.lda + p.K) * 2 : 0, 0x00020000);
                a.x[TP ? 0 : u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, (int) x_off, soff, 0));
            }
            const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *) at_tile, 0, in ? ROWS * p.K * 2 : 0, 0x00020000);
#pragma unroll
            for (int m = 0; m < RM; ++m) a.w[u][m] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, (int) w_off[m], soff, 2));      // (2: streamed past the caches)
        }
        a.bias = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, (l_tile * ROWS + o_row) * 4, 0, 0));       // (past n_store, without a bias: 0)
        if (++l_grp == ng) { l_grp = 0; l_tile += G; }
    };
    Group ga, gb;
    load(ga);
    if (total > 1) load(gb);
    // the activations are in LDS (a wave reads its own blocks only), the weights on their way
    if constexpr (TP != 0) {
        if (total > 1) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * NL) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" : : "n"(NL) : "memory");
    }
    f32x4 acc[RM];
#pragma unroll
    for (int m = 0; m < RM; ++m) acc[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    int c_tile = (int) blockIdx.x, c_grp = 0;              // the group that is multiplied
    auto step = [&](const Group & a) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = c_grp * U + u;
            // (read on every path: a register that may still be on its way would be waited for where it is loaded again)
            if (TP == 0) asm volatile("" : : "v"(a.x[TP ? 0 : u]));
#pragma unroll
            for (int m = 0; m < RM; ++m) asm volatile("" : : "v"(a.w[u][m]));
            if (i >= mine) continue;
            const u32x4 x = TP ? *(const u32x4 *) (x_at + i * (TP * 128)) : a.x[TP ? 0 : u];
#pragma unroll
            for (int m = 0; m < RM; ++m) acc[m] = Frag<uint16_t>::mma(a.w[u][m], x, acc[m]);
        }
        const float bias = a.bias;
        asm volatile("" : : "v"(bias));
        if (++c_grp < ng) return;
        c_grp = 0;
        // (the wait states between a product and the store that reads it, spelled out as in the kernel above)
#pragma unroll
        for (int m = 0; m < RM; ++m) asm volatile("" : "+v"(acc[m]));
        asm volatile("s_nop 15\n\ts_nop 3");
#pragma unroll
        for (int m = 0; m < RM; ++m) asm volatile("" : "+v"(acc[m]));
#pragma unroll
        for (int m = 0; m < RM; ++m) { *(f32x4 *) (red + ((wave * RM + m) * 16 + lr) * 16 + g * 4) = acc[m]; acc[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f}; }
        __syncthreads();
        const int row = c_tile * ROWS + o_row;
        if (o_tok < p.T && row < p.n_store) {
            float v = 0.0f;
#pragma unroll
            for (int w = 0; w < 8; ++w) { const float * q = red + ((w * RM + o_row / 8) * 16 + o_tok) * 16 + o_row % 8; v += q[0]; v += q[8 * 16 + 8]; }
            st_type(p.y, (size_t) o_tok * p.ldy + row, p.y_type, act_apply(p.act_fn, v + bias));
        }
        c_tile += G;
        __syncthreads();
    };
    if (total == 1) { step(ga); return; }
    int left = total - 2;
    for (; left > 1; left -= 2) { step(ga); load(ga); step(gb); load(gb); }
    step(ga);
    if (left) { load(ga); step(gb); step(ga); }
    else step(gb);
}
size_t rows_lds(int rm, int tp, int K) { return (size_t) 8 * rm * 1024 + (size_t) (K / 64 + 7) / 8 * 8 * tp * 128; }
template <int RM, int TP> int launch_rows(const SmallP & p, int N, hipStream_t st) {
    const int tiles = N / (8 * RM), cus = pm_device_cus();
    const size_t lds = rows_lds(RM, TP, p.K);
    const int per = (TP == 0 && RM == 2) || lds > 80 * 1024 ? 1 : 2, grid = tiles < per * cus ? tiles : per * cus;
    pm_allow_big_lds((const void *) dense_rows_kernel<RM, TP>, lds);
    hipLaunchKernelGGL((dense_rows_kernel<RM, TP>), dim3(grid), dim3(512), lds, st, p.W, p.act, p.K, p.T, p.lda, grid, tiles / grid, tiles % grid, p);
    return 0;
}

// The same for the experts' products behind pm_launch_route_stream (up to PM_ROUTE_PAIRS pairs of up to 64 experts): a workgroup keeps its rows and takes the experts blockIdx.y, + ny, .. of those
// that have pairs, up to 8 of an expert's pairs at a time. One by one (dense_small_kernel), an item's 64 KB of weights were asked for when the item in front was stored: nothing was on its way while a
// workgroup fetched activations, added up and stored. Here the load groups of all items are one sequence, two of them in flight, and the activations of the next item follow the last products
// of this one, by DMA into the waves' own LDS. 20 pairs of 32 experts of 2048 x 2048: 22.5 us a launch, now 21.2 (5.4 TB/s), a pass of
// 5 sequences of such layers 6112 -> 5984.
// The pairs: a lane per pair, 64 at a time, every wave for itself (no launch that sorts, no barrier). inv: 65536 / experts per token + 1. Sums in dense_small_kernel's order.
template <int RM> __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void dense_experts_kernel(const void * W0, const void * act0, const int32_t * id, const float * pair_w, int64_t e_stride,
                                                                                                                    int K, int lda, uint32_t pairs_ny, uint32_t inv, SmallP p) {
    constexpr int U = 8 / RM, ROWS = 8 * RM, G = PM_ROUTE_PAIRS / 64;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ int list[8][8];
    __shared__ float weight[PM_ROUTE_PAIRS];
    float * red = (float *) smem;                                                                  // [8 waves][RM][16 columns][16 rows]
    const int wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), lane = threadIdx.x & 63, lr = lane & 15, g = lane >> 4, pairs = (int) (pairs_ny & 65535), ny = (int) (pairs_ny >> 16);
    const int nblk = K >> 6, mine = (nblk - wave + 7) >> 3, ng = mine > U ? (mine + U - 1) / U : 1, r0 = (int) blockIdx.x * ROWS;
    int pe[G];                                                                                     // the experts of pairs lane, 64 + lane, .. (64: no pair)
    float pw[G];
#pragma unroll
    for (int i = 0; i < G; ++i) { pe[i] = 64; pw[i] = 0.0f; if (i * 64 < pairs && i * 64 + lane < pairs) { pe[i] = ld_g(id + i * 64 + lane); pw[i] = ld_g(pair_w + i * 64 + lane); } }
    uint32_t has[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < G; ++i) if (i * 64 < pairs) { has[0] |= pe[i] < 32 ? 1u << pe[i] : 0u; has[1] |= pe[i] >= 32 && pe[i] < 64 ? 1u << (pe[i] - 32) : 0u; }
    const uint64_t on = (uint64_t) wave_or(has[1]) << 32 | wave_or(has[0]), below = (1ull << lane) - 1;
    const int n_on = __popcll(on);
    if ((int) blockIdx.y >= n_on) return;
    auto nth = [&](int k) __attribute__((always_inline)) { return (int) __builtin_ctzll(__builtin_amdgcn_ballot_w64((on >> lane & 1) && __popcll(on & below) == k)); };
    auto pairs_of = [&](int e) __attribute__((always_inline)) {
        int n = 0;
#pragma unroll
        for (int i = 0; i < G; ++i) if (i * 64 < pairs) n += __popcll(__builtin_amdgcn_ballot_w64(pe[i] == e));
        return n;
    };
    const uint32_t at = (uint32_t) ((lr >> 3) * 32 + g * 8);
    uint32_t w_off[RM];
#pragma unroll
    for (int m = 0; m < RM; ++m) w_off[m] = ((uint32_t) (m * 8 + (lr & 7)) * (uint32_t) K + at) * 2;
    const int o_row = threadIdx.x % ROWS, o_tok = threadIdx.x / ROWS;                              // the element of an item that this thread stores
    // ---- the weights: the next group to be requested
    struct Group { u32x4 w[U][RM]; };
    int l_k = blockIdx.y, l_e = nth(l_k), l_left = (pairs_of(l_e) + 7) >> 3, l_grp = 0;             // (l_left 0: no more)
    auto load = [&](Group & a) __attribute__((always_inline)) {
        const uint16_t * at_rows = (const uint16_t *) W0 + (size_t) l_e * e_stride + (size_t) r0 * K;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // past the end of a row: out of the bounds of an empty buffer, no traffic
            const int i = l_grp * U + u, in = i < mine, soff = in ? (wave + i * 8) * 128 : 0;
            const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *) at_rows, 0, in ? ROWS * K * 2 : 0, 0x00020000);
#pragma unroll
            for (int m = 0; m < RM; ++m) a.w[u][m] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, (int) w_off[m], soff, 2));      // (2: streamed past the caches)
        }
        if (++l_grp < ng) return;
        l_grp = 0;
        if (--l_left) return;
        l_k += ny;
        if (l_k < n_on) { l_e = nth(l_k); l_left = (pairs_of(l_e) + 7) >> 3; }
    };
    // ---- the activations: up to 8 pairs of an expert, this wave's blocks of them: [block][8 pairs][8 pieces of 16 bytes, piece p in place p ^ pair / 2]
    char * const xs = smem + 8 * RM * 1024 + (size_t) wave * ((nblk + 7) >> 3) * 1024;
    const uint32_t dst = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) char *) xs;
    struct Item { int at, here, pair; float w; };                                                   // first sorted pair, pairs; this thread's pair and its weight
    int a_k = blockIdx.y, a_e = l_e, a_n = pairs_of(a_e), a_t = 0;                                  // the next item (a_n 0: no more)
    auto fetch = [&]() __attribute__((always_inline)) {
        Item x;
        int first = 0, seen = -a_t;
#pragma unroll
        for (int i = 0; i < G; ++i) {
            if (i * 64 >= pairs) break;
            const uint64_t its = __builtin_amdgcn_ballot_w64(pe[i] == a_e);
            first += __popcll(__builtin_amdgcn_ballot_w64(pe[i] < a_e));
            const int place = seen + __popcll(its & below);
            if ((its >> lane & 1) && place >= 0 && place < 8) list[wave][place] = i * 64 + lane;
            seen += __popcll(its);
        }
        wave_fence();
        x.here = a_n - a_t < 8 ? a_n - a_t : 8; x.at = first + a_t;
        const int t = lane >> 3, last = x.here - 1;
        const uint32_t row = p.in_sorted ? (uint32_t) (x.at + t) : (uint32_t) list[wave][t < last ? t : last] * inv >> 16;
        x.pair = list[wave][o_tok < last ? o_tok : last]; x.w = weight[x.pair];
        const uint32_t src = (row * (uint32_t) lda + (uint32_t) (((lane & 7) ^ (t >> 1)) * 8)) * 2 + (uint32_t) wave * 128;
        wave_fence();
        for (int i = 0; i < mine; ++i) if (t < x.here) pm_dma16(act0, src + (uint32_t) i * 1024, dst + (uint32_t) i * 1024);
        a_t += 8;
        if (a_t >= a_n) {
            a_k += ny; a_t = 0; a_n = 0;
            if (a_k < n_on) { a_e = nth(a_k); a_n = pairs_of(a_e); }
        }
        return x;
    };
#pragma unroll
    for (int i = 0; i < G; ++i) if (i * 64 < pairs) weight[i * 64 + lane] = pw[i];                  // (every wave the same; each reads what it has written itself)
    wave_fence();
    Group ga, gb;
    load(ga);
    Item now = fetch(), next = now;
    bool behind = l_left != 0;                                                                     // a group was asked for behind the item's activations
    if (behind) load(gb);
    f32x4 acc[RM];
#pragma unroll
    for (int m = 0; m < RM; ++m) acc[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    int c_grp = 0;
    auto step = [&](Group & a) __attribute__((always_inline)) -> bool {                             // the next group; false: it was the last one
        if (c_grp == 0) {
            if (behind) asm volatile("s_waitcnt vmcnt(8)" : : : "memory"); else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        }
        const int tok = (lr & 7) < now.here ? lr & 7 : now.here - 1;
        const char * x_at = xs + tok * 128 + (((lr >> 3) * 4 + g) ^ (tok >> 1)) * 16;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = c_grp * U + u;
#pragma unroll
            for (int m = 0; m < RM; ++m) asm volatile("" : : "v"(a.w[u][m]));
            if (i >= mine) continue;
            const u32x4 x = *(const u32x4 *) (x_at + i * 1024);
#pragma unroll
            for (int m = 0; m < RM; ++m) acc[m] = Frag<uint16_t>::mma(a.w[u][m], x, acc[m]);
        }
        const bool end = ++c_grp == ng, more = a_n != 0;
        if (end && more) next = fetch();
        behind = l_left != 0;
        if (behind) load(a);
        if (!end) return true;
        c_grp = 0;
        // (the wait states between a product and the store that reads it, spelled out as in the kernel above)
#pragma unroll
        for (int m = 0; m < RM; ++m) asm volatile("" : "+v"(acc[m]));
        asm volatile("s_nop 15\n\ts_nop 3");
#pragma unroll
        for (int m = 0; m < RM; ++m) asm volatile("" : "+v"(acc[m]));
#pragma unroll
        for (int m = 0; m < RM; ++m) { *(f32x4 *) (red + ((wave * RM + m) * 16 + lr) * 16 + g * 4) = acc[m]; acc[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f}; }
        __syncthreads();
        const int row = r0 + o_row;
        if (o_tok < now.here && row < p.n_store) {
            float v = 0.0f;
#pragma unroll
            for (int w = 0; w < 8; ++w) { const float * q = red + ((w * RM + o_row / 8) * 16 + o_tok) * 16 + o_row % 8; v += q[0]; v += q[8 * 16 + 8]; }
            v = act_apply(p.act_fn, v);
            if (p.weigh) v *= now.w;
            st_type(p.y, (size_t) (p.out_sorted ? now.at + o_tok : now.pair) * p.ldy + row, p.y_type, v);
        }
        if (!more) return false;
        now = next;
        __syncthreads();
        return true;
    };
    while (step(ga) && step(gb)) {}
}
template <int RM> int launch_sorted(const SmallP & p, int N, int experts, hipStream_t st) {
    const int tiles = N / (8 * RM), y = std::min(experts, (2 * pm_device_cus() + tiles - 1) / tiles);      // (two workgroups per CU: the figures at launch() below)
    const size_t lds = rows_lds(RM, 8, p.K);
    pm_allow_big_lds((const void *) dense_experts_kernel<RM>, lds);
    hipLaunchKernelGGL(dense_experts_kernel<RM>, dim3(tiles, y), dim3(512), lds, st, p.W, p.act, (const int32_t *) p.r.id, (const float *) p.r.w, p.e_stride, p.K, p.lda,
                       (uint32_t) (p.T * p.r.top) | (uint32_t) y << 16, 65536u / (uint32_t) p.r.top + 1, p);
    return 0;
}

// One bf16 matrix per group of rows (attention head) with short rows: NB 64-k blocks, a wave per 16 rows and 16 tokens, everything it needs requested at once and no sums over waves. (Above,
// eight waves share a row's blocks: of 64 k seven have none. 16384 rows of 64, 5 tokens: 8.4 us, now 3.2 .. 5.0)
template <int NB> __global__ __launch_bounds__(256) void dense_group_kernel(SmallP p, int rows, int whole) {
    const int wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), lane = threadIdx.x & 63, lr = lane & 15, g = lane >> 4;
    const int r0 = ((int) blockIdx.x * 4 + wave) * 16, t0 = blockIdx.y * 16;
    if (r0 >= rows) return;
    const int h = r0 / p.group, hr = r0 - h * p.group + g * 4, t = t0 + lr;
    const uint16_t * w = (const uint16_t *) p.W + (size_t) (r0 + lr) * (NB * 64) + g * 8, * x = (const uint16_t *) p.act + (size_t) h * p.g_act + (size_t) (t < p.T ? t : p.T - 1) * p.lda + g * 8;
    u32x4 a[2 * NB], b[2 * NB];
#pragma unroll
    for (int i = 0; i < 2 * NB; ++i) { a[i] = *(const PM_G u32x4 *) (w + i * 32); b[i] = *(const PM_G u32x4 *) (x + i * 32); }
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 2 * NB; ++i) acc = Frag<uint16_t>::mma(a[i], b[i], acc);
    if (t >= p.T) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = act_apply(p.act_fn, acc[e]);
    const size_t at = (size_t) t * p.ldy + h * p.g_out + hr;
    if (whole) {                                           // (four neighbours of a row of y, wanted and on their boundary)
        if (p.y_type == PM_F32) *(PM_G f32x4 *) ((float *) p.y + at) = acc;
        else *(PM_G u32x2 *) ((uint16_t *) p.y + at) = u32x2{(uint32_t) f2bf(acc[0]) | (uint32_t) f2bf(acc[1]) << 16, (uint32_t) f2bf(acc[2]) | (uint32_t) f2bf(acc[3]) << 16};
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) if (hr + e < p.g_store && h * p.g_out + hr + e < p.n_store) st_type(p.y, at + e, p.y_type, acc[e]);
}
template <int NB> int launch_group(const SmallP & p, int N, hipStream_t st) {
    const int whole = p.g_store % 16 == 0 && p.g_store == p.group && p.g_out % 4 == 0 && p.ldy % 4 == 0 && ((uintptr_t) p.y & 15) == 0 && (N / p.group - 1) * p.g_out + p.g_store <= p.n_store;
    hipLaunchKernelGGL(dense_group_kernel<NB>, dim3((N + 63) / 64, (p.T + 15) / 16), dim3(256), 0, st, p, N, whole);
    return 0;
}

template <typename T, int NT, int RM, int SRC, int EXP = DENSE> int launch(const SmallP & p, int N, int y, hipStream_t st) {
    constexpr bool LINE = sizeof(T) == 2 && SRC != 0;
    constexpr int rows = (LINE ? 8 : 16) * RM, toks = (LINE ? 8 : 16) * NT;
    const int here = EXP == PAIR || EXP == CONCAT ? 1 : EXP == SORTED || p.T > toks ? toks : p.T;
    size_t lds = (size_t) 8 * NT * RM * 1024 + (SRC ? (size_t) here * ((size_t) p.K * (EXP == CONCAT ? p.r.top : 1) * sizeof(T) + 16) : 0);
    if (EXP == PAIR && lds < 8192) lds = 8192;
    pm_allow_big_lds((const void *) dense_small_kernel<T, NT, RM, SRC, EXP>, lds);
    // Sorted experts: two workgroups per CU, which take their experts in turn. One per row tile and expert that there could be (`y`), most of them without tokens, were 14336 of 512 threads for 8 tokens
    // of 32 experts of 4096 x 3584: 102 us with tables and 112 without, 96 so; of 2048 x 2048 at 24 tokens 56 and 56, now 47. (768 .. 4096 of them: up to 20 % more, whole rounds or not)
    if (EXP == SORTED) y = std::min(y, (2 * pm_device_cus() + N / rows - 1) / (N / rows));
    hipLaunchKernelGGL((dense_small_kernel<T, NT, RM, SRC, EXP>), dim3(N / rows, EXP == DENSE ? (p.T + toks - 1) / toks : y), dim3(512), lds, st, p);
    return 0;
}
// a wave's load group should not outgrow its share of K
int rows_per_lane(int K) { return (K / 64 + 7) / 8 >= 8 ? 1 : 2; }
constexpr size_t LDS_ACT = 72 * 1024;

template <typename T> int launch_type(const pm_dense_args & a, const SmallP & p, hipStream_t st) {
    const int N = a.group ? a.N : (a.n_store + 63) / 64 * 64;
    const int rm = rows_per_lane(a.K);
    if (a.pro) {
        if (!pm_dense_pro_ok(a.T, a.pro->width)) return PM355_E_UNSUPPORTED;
        if constexpr (sizeof(T) == 2) if (rm == 2) return a.T == 1 ? launch<T, 1, 2, 1>(p, N, 0, st) : a.T == 2 ? launch<T, 1, 2, 2>(p, N, 0, st) : launch<T, 1, 2, 4>(p, N, 0, st);
        return a.T == 1 ? launch<T, 1, 1, 1>(p, N, 0, st) : a.T == 2 ? launch<T, 1, 1, 2>(p, N, 0, st) : launch<T, 1, 1, 4>(p, N, 0, st);
    }
    // One matrix per group, short rows: up to 256 values a wave's operands fit its registers, and eight waves on a row have at most half a block each
    if constexpr (sizeof(T) == 2)
        if (a.group && !a.merge && a.T <= 64 && a.K <= 256 && (((uintptr_t) p.W | (uintptr_t) p.act) & 15) == 0 && p.lda % 8 == 0 && p.g_act % 8 == 0 && N % p.group == 0) {
            if (a.K == 64) return launch_group<1>(p, N, st);
            if (a.K == 128) return launch_group<2>(p, N, st);
            return a.K == 192 ? launch_group<3>(p, N, st) : launch_group<4>(p, N, st);
        }
    // One matrix, up to 8 tokens: the workgroups that stay, with the activations in LDS where they fit (150 KB: 16 bytes per value for 5..8 tokens, 8 for less), from memory above that
    // (5 tokens of 4096 values, 14336 rows: 22.7 us against 27 from memory). One token of shorter rows stays with a workgroup per tile, which has less to do before its first and after
    // its last weight (32000 x 2048: 23.6 us against 25.1, 4096 x 5120: 10.2 / 10.9; the other way round from 6144 values: 5120 x 6144 16.8 / 15.2, 2048 x 8192 10.3 / 9.0). DMA and buffer loads
    // of 16 bytes want operands that start on 16 bytes
    if constexpr (sizeof(T) == 2)
        if (a.T <= 8 && (((uintptr_t) p.W | (uintptr_t) p.act) & 15) == 0 && !a.group && !a.merge && (a.T > 1 || a.K >= 6144) && (int64_t) p.T * p.lda < (1 << 28) && a.K < (1 << 26)) {
            const int tp = a.T <= 4 ? 4 : 8;
            if (rows_lds(rm, tp, a.K) > 150 * 1024) return launch_rows<2, 0>(p, N, st);
            if (tp == 4) return rm == 1 ? launch_rows<1, 4>(p, N, st) : launch_rows<2, 4>(p, N, st);
            return rm == 1 ? launch_rows<1, 8>(p, N, st) : launch_rows<2, 8>(p, N, st);
        }
    if constexpr (sizeof(T) == 2)
        if (a.T <= 8 && (size_t) a.T * (a.K * 2 + 16) <= LDS_ACT) return rm == 1 ? launch<T, 1, 1, -1>(p, N, 0, st) : launch<T, 1, 2, -1>(p, N, 0, st);
    const bool wide = N / 32 >= 512;
    if (a.merge) return PM355_E_SHAPE;                     // (pm_dense_merge_ok)
    if (a.T <= 16) return wide ? launch<T, 1, 2, 0>(p, N, 0, st) : launch<T, 1, 1, 0>(p, N, 0, st);
    if (a.T <= 32) return wide ? launch<T, 2, 2, 0>(p, N, 0, st) : launch<T, 2, 1, 0>(p, N, 0, st);
    if constexpr (sizeof(T) == 2) if (wide) return launch<T, 4, 2, 0>(p, N, 0, st);
    return launch<T, 4, 1, 0>(p, N, 0, st);
}
// one product of the experts: N rows of K values per expert
template <typename T, int EXP> int launch_experts(const SmallP & p, int N, int y, hipStream_t st) {
    if constexpr (sizeof(T) == 2) {
        const size_t one = (size_t) p.K * (EXP == CONCAT ? p.r.top : 1) * 2 + 16;
        // (the same line as below; buffer loads and DMA of 16 bytes want operands that start on 16 bytes, 32-bit offsets)
        if (EXP == SORTED && !p.r.logits && one * 8 <= LDS_ACT && (((uintptr_t) p.W | (uintptr_t) p.act) & 15) == 0 && p.lda % 8 == 0 && p.e_stride % 8 == 0 && (int64_t) p.T * p.r.top * p.lda < (1 << 30))
            return rows_per_lane(p.K) == 1 ? launch_sorted<1>(p, N, y, st) : launch_sorted<2>(p, N, y, st);
        if (one * (EXP == SORTED ? 8 : 1) <= LDS_ACT) return rows_per_lane(EXP == CONCAT ? p.K * p.r.top : p.K) == 1 ? launch<T, 1, 1, -1, EXP>(p, N, y, st) : launch<T, 1, 2, -1, EXP>(p, N, y, st);
    }
    return launch<T, 1, 1, 0, EXP>(p, N, y, st);
}
template <typename T> int experts_type(const pm_expert_args & a, hipStream_t st) {
    SmallP p = {};
    p.r = a.r;
    const int pairs = a.T * a.r.top, few = a.r.E < pairs ? a.r.E : pairs;
    // up: hid = weight * act(W_up x)
    p.W = a.up; p.e_stride = a.up_stride; p.act = a.x; p.lda = a.ldx; p.K = a.width_p; p.y = a.hid; p.ldy = a.ffp; p.y_type = a.type; p.n_store = a.ffp; p.act_fn = a.act_fn; p.T = a.T;
    p.in_sorted = 0; p.out_sorted = 1; p.weigh = 1;
    int rc = a.T <= PM_ROUTE_PAIR_MAX ? launch_experts<T, PAIR>(p, a.ffp, pairs, st) : launch_experts<T, SORTED>(p, a.ffp, few, st);
    if (rc) return rc;
    p.W = a.down; p.e_stride = a.down_stride; p.act = a.hid; p.K = a.ffp; p.y = a.y; p.ldy = a.ldy; p.y_type = a.y_type; p.n_store = a.width; p.act_fn = PM355_ACT_NONE;
    p.in_sorted = 1; p.out_sorted = 0; p.weigh = 0;
    if (a.T <= PM_ROUTE_PAIR_MAX) { p.lda = a.ffp * a.r.top; return launch_experts<T, CONCAT>(p, a.width_p, a.T, st); }
    p.lda = a.ffp;
    return launch_experts<T, SORTED>(p, a.width_p, few, st);
}

} // namespace

// (every workgroup of a head merges that head's sums again: with more tokens a launch of its own costs less)
bool pm_dense_merge_ok(int T, int K) { return T <= 2 && (size_t) T * (K * 2 + 16) <= LDS_ACT; }
bool pm_dense_pro_ok(int T, int width) { return T >= 1 && T <= 4 && width * (T == 1 ? 1 : T == 2 ? 2 : 4) <= PRO_MAX; }

int pm_launch_dense_small(const pm_dense_args & a, hipStream_t st) {
    SmallP p = {};
    p.W = a.W; p.act = a.act; p.y = a.y; p.bias = a.bias; p.K = a.K; p.T = a.T; p.lda = a.lda; p.ldy = a.ldy; p.y_type = a.y_type; p.n_store = a.n_store; p.act_fn = a.act_fn;
    p.group = a.group; p.g_act = a.g_act; p.g_out = a.g_out; p.g_store = a.g_store;
    if (a.pro) p.pro = *a.pro;
    if (a.merge) p.merge = *a.merge;
    if (a.merge && (!a.group || a.type != PM_BF16 || a.merge->splits < 1 || a.merge->splits > 64 || !pm_dense_merge_ok(a.T, a.K))) return PM355_E_SHAPE;
    if (a.K % 64 || a.N % 64 || (!a.group && a.n_store > a.N) || a.T < 1 || (a.type != PM_BF16 && a.type != PM_F32)) return PM355_E_SHAPE;
    if (a.group && (a.group % 32 || a.pro || a.bias || (size_t) a.g_act * pm_dense_bytes(a.type) % 16)) return PM355_E_SHAPE;
    return a.type == PM_BF16 ? launch_type<uint16_t>(a, p, st) : launch_type<float>(a, p, st);
}

int pm_launch_experts_small(const pm_expert_args & a, hipStream_t st) {
    if (a.T < 1 || a.width_p % 64 || a.ffp % 64 || a.r.E < 1 || a.r.E > 1024 || a.r.top < 1 || a.r.top > 64 || a.r.groups > 1024 || (a.type != PM_BF16 && a.type != PM_F32)) return PM355_E_SHAPE;
    return a.type == PM_BF16 ? experts_type<uint16_t>(a, st) : experts_type<float>(a, st);
}
