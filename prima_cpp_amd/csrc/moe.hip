// moe.hip — routing of a step's tokens to experts, in one of three forms:
// - few pairs of up to 64 experts behind a bf16 model's RMS norm (pm_route_stream_ok): norm, router product and choice in one launch, a workgroup per token; the expert products find their own pairs
// - up to 64 tokens otherwise: one workgroup scores, selects and sorts (expert by expert, tokens in order)
// - more: a wave per token selects and takes a place in its expert's list, then every workgroup sorts its share of the pairs (the order inside an expert does not enter any sum)
#include "pm355_route.h"
#include "pm355_kernels.h"

namespace {

// exclusive prefix of the experts' counts in LDS: off[0 .. E]; one wave
__device__ __forceinline__ void prefix(const int * count, int E, int * off) {
    const int lane = threadIdx.x & 63;
    int carry = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
        const int v = e0 + lane < E ? count[e0 + lane] : 0;
        int s = v;
        for (int o = 1; o < 64; o *= 2) { const int u = __shfl_up(s, o); if (lane >= o) s += u; }
        if (e0 + lane < E) off[e0 + lane] = carry + s - v;
        carry += __shfl(s, 63);
    }
    if (lane == 0) off[E] = carry;
}
// which experts have pairs, and their tiles; one wave
__device__ __forceinline__ void lists(const int * off, const pm_route & r, int want_tiles) {
    const int lane = threadIdx.x & 63;
    int n_act = 0, n_tile = 0;
    for (int e0 = 0; e0 < r.E; e0 += 64) {
        const int e = e0 + lane, n = e < r.E ? off[e + 1] - off[e] : 0;
        const uint64_t on = __builtin_amdgcn_ballot_w64(n > 0);
        if (n > 0) r.active[1 + n_act + __popcll(on & ((1ull << lane) - 1))] = e;
        n_act += __popcll(on);
        if (!want_tiles) continue;
        const int tiles = (n + r.tile - 1) / r.tile;
        int s = tiles;
        for (int o = 1; o < 64; o *= 2) { const int u = __shfl_up(s, o); if (lane >= o) s += u; }
        for (int i = 0; i < tiles; ++i) {
            int32_t * t = r.tiles + 1 + 3 * (n_tile + s - tiles + i);
            t[0] = e; t[1] = off[e] + i * r.tile; t[2] = n - i * r.tile < r.tile ? n - i * r.tile : r.tile;
        }
        n_tile += __shfl(s, 63);
    }
    if (lane == 0) { r.active[0] = n_act; if (want_tiles) r.tiles[0] = n_tile; }
}

// T <= 64 tokens. LDS: [16 waves][E] scores, [16][groups], count[E], off[E + 1], ids [T * top]
__global__ __launch_bounds__(1024) void route_one_kernel(pm_route r, int T, int want_tiles) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, pairs = T * r.top;
    float * s = sm + wave * r.E, * gs = sm + 16 * r.E + wave * r.groups;
    int * off = (int *) (sm + 16 * (r.E + r.groups)), * count = off + r.E + 1, * ids = count + r.E;
    float * ws = (float *) (ids + pairs);
    for (int t = wave; t < T; t += 16) {
        route_token([&](int e) { return ld_g(r.logits + (size_t) t * r.ldl + e); }, r.E, r.top, r.groups, r.keep, s, gs, ids + t * r.top, ws + t * r.top);
        for (int k = lane; k < r.top; k += 64) { r.id[t * r.top + k] = ids[t * r.top + k]; r.w[t * r.top + k] = ws[t * r.top + k]; }
    }
    __syncthreads();
    // few pairs: a wave per expert, a lane per pair (a thread per expert reads the pairs one after the other, a trip to LDS each: 5 tokens x 4 of 32 experts 8.2 us, now 7.3; 7.1 with the maximum by DPP)
    const bool few = pairs <= 256;
    if (few) {
        for (int e = wave; e < r.E; e += 16) {
            int n = 0;
            for (int i = lane; i - lane < pairs; i += 64) n += __popcll(__builtin_amdgcn_ballot_w64(i < pairs && ids[i < pairs ? i : 0] == e));
            if (lane == 0) count[e] = n;
        }
    } else for (int e = threadIdx.x; e < r.E; e += 1024) {
        int n = 0;
        for (int i = 0; i < pairs; ++i) n += ids[i] == e;
        count[e] = n;
    }
    __syncthreads();
    if (wave == 0) prefix(count, r.E, off);
    __syncthreads();
    if (wave == 0) lists(off, r, want_tiles);
    if (few)
        for (int e = wave; e < r.E; e += 16) {
            int at = off[e];
            if (!count[e]) continue;
            for (int i = lane; i - lane < pairs; i += 64) {
                const bool is = i < pairs && ids[i < pairs ? i : 0] == e;
                const uint64_t on = __builtin_amdgcn_ballot_w64(is);
                if (is) r.order[at + __popcll(on & ((1ull << lane) - 1))] = i;
                at += __popcll(on);
            }
        }
    for (int e = threadIdx.x; e <= r.E; e += 1024) {
        int at = off[e];
        r.off[e] = at;
        if (!few && e < r.E && count[e]) for (int i = 0; i < pairs; ++i) if (ids[i] == e) r.order[at++] = i;
    }
}

// Up to 64 tokens of a bf16 model with RMS norms: the residual stream's norm, the router product and the choice of experts, one workgroup per token. Three launches otherwise, whose time is the way to their first
// byte and from their last one: 5 tokens of 2048 values, 32 experts, 4 each: 4.2 + 4.5 + 7.1 us and the gaps between them, now 8.3 and one gap (all tokens in one workgroup, which then also sorts the
// pairs: 16.7 us, the vector pipe of one CU; the expert products find their pairs themselves, dense_small.hip). A wave has every 16th 64-value block of the row: it norms those columns and
// multiplies them, the router's weights of all its blocks on their way from the start (in its registers: that bounds the width and the experts), so that the workgroup meets for the norm's
// sums and for the logits only. 16 tile rows = 8 rows of W x 2 halves of a block (whole 128-byte lines, as in dense_small.hip), the halves in columns 0 and 8 of the result.
struct StreamP { const float * y; float * x; const uint16_t * W; uint16_t * xb; int ld, K; };       // y, x, xb: rows of ld values; W: rows of K
template <int VP, int ET> __global__ __launch_bounds__(1024) void route_stream_kernel(pm_route r, pm_norm_args q, StreamP p) {      // VP: 64-value blocks per wave; ET: tiles of 8 experts
    __shared__ __attribute__((aligned(16))) float red[2][16], part[16][2][8 * ET];
    __shared__ __attribute__((aligned(16))) uint16_t act[16][VP * 64];
    __shared__ float s_group[2][64];
    const int wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), lane = threadIdx.x & 63, lr = lane & 15, g = lane >> 4, nblk = p.K >> 6, t = blockIdx.x;
    const float * y_row = p.y + (size_t) t * p.ld;
    float * x_row = p.x + (size_t) t * p.ld;
    float y[VP], x[VP], w[VP], w2[VP];
    u32x4 W[VP][ET];
#pragma unroll
    for (int v = 0; v < VP; ++v) {                         // (past the row: its last column)
        const int c = (wave + 16 * v) * 64 + lane, cc = c < q.width ? c : q.width - 1;
        y[v] = ld_g(y_row + cc); x[v] = ld_g(x_row + cc); w[v] = ld_g(q.w + cc);
        w2[v] = q.w2 ? ld_g(q.w2 + cc) : 1.0f;
    }
#pragma unroll
    for (int v = 0; v < VP; ++v) {
        const int blk = wave + 16 * v < nblk ? wave + 16 * v : nblk - 1;
#pragma unroll
        for (int e = 0; e < ET; ++e) W[v][e] = *(const PM_G u32x4 *) (p.W + (size_t) (e * 8 + (lr & 7)) * p.K + blk * 64 + (lr >> 3) * 32 + g * 8);
    }
    auto in = [&](int v) __attribute__((always_inline)) { return (wave + 16 * v) * 64 + lane < q.width; };
    auto row_sum = [&](float s, int i) __attribute__((always_inline)) {
        s = wave_sum(s);
        if (lane == 0) red[i][wave] = s;
        __syncthreads();
        float o = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k) { const f32x4 f = ((const f32x4 *) red[i])[k]; o += (f[0] + f[1]) + (f[2] + f[3]); }
        return o;
    };
    float s = 0.0f;
#pragma unroll
    for (int v = 0; v < VP; ++v) s = in(v) ? fmaf(y[v], y[v], s) : s;
    const float rs = 1.0f / sqrtf(row_sum(s, 0) / (float) q.width + q.eps);
    s = 0.0f;
#pragma unroll
    for (int v = 0; v < VP; ++v) {
        x[v] += y[v] * rs * w[v];
        s = in(v) ? fmaf(x[v], x[v], s) : s;
    }
    const float r2 = q.w2 ? 1.0f / sqrtf(row_sum(s, 1) / (float) q.width + q.eps) : 1.0f;
#pragma unroll
    for (int v = 0; v < VP; ++v) {
        const int c = (wave + 16 * v) * 64 + lane;
        const uint16_t o = in(v) ? f2bf(x[v] * (r2 * w2[v])) : (uint16_t) 0;
        act[wave][v * 64 + lane] = o;
        if (in(v)) { st_g(x_row + c, x[v]); st_g(p.xb + (size_t) t * p.ld + c, o); }
    }
    wave_fence();                                          // (a wave reads its own blocks)
    f32x4 acc[ET];
#pragma unroll
    for (int e = 0; e < ET; ++e) acc[e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int v = 0; v < VP; ++v) {
        if (wave + 16 * v >= nblk) continue;
        const u32x4 a = *(const u32x4 *) (act[wave] + v * 64 + (lr >> 3) * 32 + g * 8);
#pragma unroll
        for (int e = 0; e < ET; ++e) acc[e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, W[v][e]), __builtin_bit_cast(bf16x8, a), acc[e], 0, 0, 0);
    }
    // (a wave without a block comes here by a jump: the wait states between a product and the store that reads it are spelled out, as in dense_small.hip)
#pragma unroll
    for (int e = 0; e < ET; ++e) asm volatile("" : "+v"(acc[e]));
    asm volatile("s_nop 15\n\ts_nop 3");
#pragma unroll
    for (int e = 0; e < ET; ++e) asm volatile("" : "+v"(acc[e]));
    if (lr == (g >> 1) * 8) {                              // rows 4 g .. + 4: half g / 2 of W's rows 4 (g % 2) ..
#pragma unroll
        for (int e = 0; e < ET; ++e) *(f32x4 *) (part[wave][g >> 1] + e * 8 + (g & 1) * 4) = acc[e];
    }
    __syncthreads();
    if (wave) return;
    float z = 0.0f;
#pragma unroll
    for (int k = 0; k < 32; ++k) z += part[k >> 1][k & 1][lane & (8 * ET - 1)];
    route_token([&](int) { return z; }, r.E, r.top, r.groups, r.keep, s_group[0], s_group[1], r.id + t * r.top, r.w + t * r.top);
}

// 32 tokens per workgroup: places among its own pairs by LDS counters, then one global counter update per expert
constexpr int SEL_TOK = 32;
__global__ __launch_bounds__(1024) void route_select_kernel(pm_route r, int T) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    const int wave = threadIdx.x >> 6, t0 = blockIdx.x * SEL_TOK, n = (T - t0 < SEL_TOK ? T - t0 : SEL_TOK) * r.top;
    int * count = (int *) sm, * ids = count + r.E;
    float * w = (float *) (ids + SEL_TOK * r.top), * s = w + SEL_TOK * r.top + wave * (r.E + r.groups);
    for (int e = threadIdx.x; e < r.E; e += 1024) count[e] = 0;
    for (int i = wave; i < SEL_TOK && t0 + i < T; i += 16)
        route_token([&](int e) { return ld_g(r.logits + (size_t) (t0 + i) * r.ldl + e); }, r.E, r.top, r.groups, r.keep, s, s + r.E, ids + i * r.top, w + i * r.top);
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 1024) {
        r.id[t0 * r.top + i] = ids[i]; r.w[t0 * r.top + i] = w[i];
        ((int *) w)[i] = atomicAdd(count + ids[i], 1);     // (the weight has been stored: its place takes over)
    }
    __syncthreads();
    for (int e = threadIdx.x; e < r.E; e += 1024) if (count[e]) count[e] = atomicAdd(r.count + e, count[e]);
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 1024) r.pos[t0 * r.top + i] = count[ids[i]] + ((int *) w)[i];
}
__global__ __launch_bounds__(256) void route_place_kernel(pm_route r, int pairs, int want_tiles) {
    extern __shared__ __attribute__((aligned(16))) int cnt[];
    int * off = cnt + r.E;
    for (int e = threadIdx.x; e < r.E; e += 256) cnt[e] = r.count[e];
    __syncthreads();
    if (threadIdx.x < 64) prefix(cnt, r.E, off);
    __syncthreads();
    if (blockIdx.x == 0) {
        if (threadIdx.x < 64) lists(off, r, want_tiles);
        for (int e = threadIdx.x; e <= r.E; e += 256) r.off[e] = off[e];
    }
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p < pairs) r.order[off[r.id[p]] + r.pos[p]] = p;
}

} // namespace

void pm_launch_route(const pm_route & r, int T, int want_tiles, hipStream_t st) {
    const int pairs = T * r.top;
    if (T <= PM_ROUTE_ONE_MAX) {
        const size_t lds = (size_t) 16 * (r.E + r.groups) * 4 + (size_t) (2 * r.E + 1 + 2 * pairs) * 4;
        pm_allow_big_lds((const void *) route_one_kernel, lds);
        if (lds <= 150 * 1024) { hipLaunchKernelGGL(route_one_kernel, dim3(1), dim3(1024), lds, st, r, T, want_tiles); return; }
    }
    const size_t lds = ((size_t) r.E + 2 * SEL_TOK * r.top + 16 * (r.E + r.groups)) * 4;      // (at most 150 KB: E, groups <= 1024, top <= 64)
    pm_allow_big_lds((const void *) route_select_kernel, lds);
    hipLaunchKernelGGL(route_select_kernel, dim3((T + SEL_TOK - 1) / SEL_TOK), dim3(1024), lds, st, r, T);
    hipLaunchKernelGGL(route_place_kernel, dim3((pairs + 255) / 256), dim3(256), (size_t) (2 * r.E + 1) * 4, st, r, pairs, want_tiles);
}

// what a workgroup's registers hold: 64 blocks of 32 experts, 32 of 64; the pairs that the small products find for themselves (dense_small.hip)
bool pm_route_stream_ok(const pm_route & r, const pm_norm_args & q, int K, int T) {
    return T <= PM_ROUTE_ONE_MAX && T * r.top <= PM_ROUTE_PAIRS && r.E <= 64 && K <= (r.E <= 32 ? 4096 : 2048) && q.width <= K && q.rms && !q.b && !q.parts && q.y_type == PM_F32;
}
void pm_launch_route_stream(const pm_route & r, const pm_norm_args & q, float * x, const float * y, const void * W, int K, void * xb, int ld, int T, hipStream_t st) {
    const StreamP p{y, x, (const uint16_t *) W, (uint16_t *) xb, ld, K};
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(T), dim3(1024), 0, st, r, q, p); };
    if (r.E > 32) go(route_stream_kernel<2, 8>);
    else if (K > 2048) go(route_stream_kernel<4, 4>);
    else go(route_stream_kernel<2, 4>);
}
