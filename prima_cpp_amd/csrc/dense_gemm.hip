// dense_gemm.hip — y[t][n] = act(W[n] . x[t] + bias) for prompt-sized batches, bf16 x bf16 with f32 accumulation on the matrix cores.
// Both operands travel by LDS-DMA as whole 128-byte lines (64 k per stage) into two stages; 16-byte chunks are XOR-swizzled on the source side (chunk c of row r at
// c ^ ((r >> 1) & 7): the sixteen lanes a ds_read_b128 serves hit sixteen bank groups). One barrier per stage: behind it the stage of the previous step is free and takes
// the next k-step's DMA, which has this step's MFMAs to land. Tiles of one XCD form compact blocks of the output so that its L2 serves both operands.
// dense_tile_kernel: one matrix, tiles of 128 .. 256 tokens x 128 or 256 rows, chosen by the time their rounds take; experts with many pairs. dense_gemm_kernel: 128 x 128 and 256 x 256 tiles where
// they are the quickest; experts (token tiles from the routing tables, rows gathered and scattered by pair); latent cache pages into keys and transposed values.
#include "pm355_dense.h"
#include "pm355_kernels.h"
#include "../../include/prima_mi355.h"
#include <algorithm>
#include <iterator>
#include <type_traits>

namespace {

enum { DENSE = 0, EXPERTS = 1, KEYS = 2, VALUES = 3 };
struct GemmP {
    const uint16_t * W; const uint16_t * X; void * y; const float * bias;
    int K, N, T, lda, ldy, y_type, n_store, act_fn, nt, nn;      // nt, nn: token / row tiles
    // EXPERTS: tiles = [count, {expert, first sorted pair, pairs} ..]; input rows are tokens (gather) or sorted pairs, output rows sorted pairs or pairs (scatter)
    const int32_t * tiles, * order; const float * weight; int64_t e_stride; int top, gather, scatter;
    // KEYS: X rows are those of cache pages; VALUES: the rows of W are (tokens become the columns of the output)
    const int32_t * pages; int H, per, rows_h, pad;              // heads, values per head, rows of W per head, padded head size of the output
    int splits, split_steps, rows;                               // dense_tile_kernel: k ranges of so many 64-k steps; with more than one, y = f32 sums [splits][T][ldy] (reduce_kernel), or [T][splits][ldy] (rows)
};

template <int N> __device__ __forceinline__ void vm_wait() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }

template <int BM, int BN, int WM, int WN, int STAGES, int KIND> __global__ __launch_bounds__(BM / WM * (BN / WN) * 64) void dense_gemm_kernel(GemmP p) {
    constexpr int WAVES = BM / WM * (BN / WN), MI = WM / 32, NI = WN / 32, PIECES = (BM + BN) / 8 / WAVES, STAGE = (BM + BN) * 128;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), lane = threadIdx.x & 63, lr = lane & 31, h_ = lane >> 5;
    const int wm = wave / (BN / WN), wn = wave % (BN / WN);
    // tile order: XCD x = blockIdx % 8 takes a contiguous run of tiles; runs walk blocks of 8 token tiles column by column
    const int nt = KIND == EXPERTS ? __builtin_amdgcn_readfirstlane(ld_g(p.tiles)) : p.nt;      // (the grid has room for the most tiles there can be)
    const int total = nt * p.nn, per = (total + 7) / 8;
    const int slot = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (slot >= total || (int) (blockIdx.x >> 3) >= per) return;
    const int band = slot / (8 * p.nn), left = nt - band * 8, bh = left < 8 ? left : 8, in = slot - band * 8 * p.nn;
    int t0 = (band * 8 + in % bh) * BM, n_tok = p.T;
    const int n0 = (in / bh) * BN;
    const uint16_t * W = p.W;
    if constexpr (KIND == EXPERTS) {                       // t0, n_tok: sorted pairs of this tile
        const int32_t * tt = p.tiles + 1 + 3 * (band * 8 + in % bh);
        W += (int64_t) __builtin_amdgcn_readfirstlane(ld_g(tt)) * p.e_stride;
        t0 = __builtin_amdgcn_readfirstlane(ld_g(tt + 1)); n_tok = t0 + __builtin_amdgcn_readfirstlane(ld_g(tt + 2));
    }

    // DMA pieces of this wave (8 rows of 128 bytes each): the first half of the waves brings the tokens, the second half the rows of W
    static_assert(STAGES == 2 || STAGES == 4, "stages are found by a mask, waits are spelled for these");
    static_assert(BM == BN, "a wave's pieces belong to one operand");
    const bool tok = wave < WAVES / 2;
    const char * base = tok ? (const char *) (KIND == VALUES ? W + (size_t) t0 * p.K : p.X + (KIND == EXPERTS ? 0 : (size_t) t0 * p.lda)) : (const char *) (W + (size_t) n0 * p.K);
    const int last = tok ? n_tok - 1 - t0 : p.N - 1 - n0;
    const bool paged = KIND == KEYS ? tok : KIND == VALUES ? !tok : false;
    const char * pbase[PIECES];                            // (paged: a piece's eight rows lie in one page)
    (void) pbase;
    const uint32_t pitch = (uint32_t) (tok && KIND != VALUES ? p.lda : p.K) * 2u;
    const uint32_t lds0 = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) char *) smem + (uint32_t) wave * PIECES * 1024u;
    uint32_t off[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int r = (wave * PIECES + i) * 8 + (lane >> 3), rr = tok ? r : r - BM;
        int row = rr < last ? rr : last;
        if constexpr (KIND == EXPERTS) if (tok) { row += t0; if (p.gather) row = ld_g(p.order + row) / p.top; }
        const uint32_t swz = (uint32_t) ((lane & 7) ^ ((r >> 1) & 7)) * 16u;
        if (KIND >= KEYS && paged) {
            const int at = (tok ? t0 : n0) + (wave * PIECES + i) * 8 - (tok ? 0 : BM), lim = (tok ? n_tok : p.N) - 8, a8 = at < lim ? at : lim;      // (whole pages: a multiple of 8)
            pbase[i] = (const char *) p.X + ((size_t) __builtin_amdgcn_readfirstlane(ld_g(p.pages + a8 / PM_PAGE)) * PM_PAGE + a8 % PM_PAGE) * (size_t) p.lda * 2;
            off[i] = (uint32_t) (lane >> 3) * (uint32_t) p.lda * 2u + swz;
        } else off[i] = (uint32_t) row * pitch + swz;
    }
    auto request = [&](int k, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) pm_dma16((KIND >= KEYS && paged ? pbase[i] : base) + (size_t) k * 128, off[i], lds0 + (uint32_t) stage * STAGE + (uint32_t) i * 1024u);
    };
    f32x16 acc[MI][NI];
#pragma unroll
    for (int m = 0; m < MI; ++m)
#pragma unroll
        for (int n = 0; n < NI; ++n)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[m][n][e] = 0.0f;
    uint32_t arow[MI], brow[NI]; int asw[MI], bsw[NI];
#pragma unroll
    for (int m = 0; m < MI; ++m) { const int r = wm * WM + m * 32 + lr; arow[m] = (uint32_t) r * 128u; asw[m] = (r >> 1) & 7; }
#pragma unroll
    for (int n = 0; n < NI; ++n) { const int r = BM + wn * WN + n * 32 + lr; brow[n] = (uint32_t) r * 128u; bsw[n] = (r >> 1) & 7; }

    float bias[NI];
#pragma unroll
    for (int n = 0; n < NI; ++n) { const int col = n0 + wn * WN + n * 32 + lr; bias[n] = KIND == DENSE && p.bias && col < p.n_store ? ld_g(p.bias + col) : 0.0f; }
    const int steps = p.K >> 6;
#pragma unroll
    for (int i = 0; i < STAGES - 1; ++i) if (i < steps) request(i, i);
    for (int k = 0; k < steps; ++k) {
        const int ahead = steps - 1 - k;                   // this step's lines have landed (requests complete in order) ..
        if (STAGES > 2 && ahead >= STAGES - 2) vm_wait<PIECES * (STAGES - 2)>();
        else if (STAGES > 3 && ahead == 1) vm_wait<PIECES>();
        else vm_wait<0>();
        __syncthreads();                                   // .. for every wave, and every wave is done with the stage in front of this one
        if (k + STAGES - 1 < steps) request(k + STAGES - 1, (k + STAGES - 1) & (STAGES - 1));
        const char * s = smem + (k & (STAGES - 1)) * STAGE;
        // fragments of the next 16 k are on their way while this 16 k's products run
        bf16x8 a[2][MI], b[2][NI];
        auto read = [&](int j) __attribute__((always_inline)) {
#pragma unroll
            for (int n = 0; n < NI; ++n) b[j & 1][n] = *(const bf16x8 *) (s + brow[n] + (uint32_t) (((j * 2 + h_) ^ bsw[n]) * 16));
#pragma unroll
            for (int m = 0; m < MI; ++m) a[j & 1][m] = *(const bf16x8 *) (s + arow[m] + (uint32_t) (((j * 2 + h_) ^ asw[m]) * 16));
        };
        read(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j < 3) read(j + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < MI; ++m)
#pragma unroll
                for (int n = 0; n < NI; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[j & 1][m], b[j & 1][n], acc[m][n], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    int * s_pair = (int *) smem;
    float * s_weight = (float *) (smem + BM * 4);
    if constexpr (KIND == EXPERTS) {                       // what the stores need about their rows
        __syncthreads();
        for (int i = threadIdx.x; i < BM; i += WAVES * 64) {
            const int pair = ld_g(p.order + (t0 + i < n_tok ? t0 + i : n_tok - 1));
            s_pair[i] = p.scatter ? pair : t0 + i;
            s_weight[i] = p.weight ? ld_g(p.weight + pair) : 1.0f;
        }
        __syncthreads();
    }
    // tokens are the tile's rows, W rows its columns: a register's 32 lanes store 32 consecutive outputs of one token
#pragma unroll
    for (int n = 0; n < NI; ++n) {
        const int col = n0 + wn * WN + n * 32 + lr;
        const bool ok = col < p.n_store;
        // (32 rows of the tile lie in one page, or belong to one head)
        if constexpr (KIND == KEYS) {                      // K[page][head][slot][pad]
            const int h = col / p.per, d = col - h * p.per;
#pragma unroll
            for (int m = 0; m < MI; ++m) {
                const int tok0 = t0 + wm * WM + m * 32;
                uint16_t * o = (uint16_t *) p.y + (((size_t) (tok0 / PM_PAGE) * p.H + h) * PM_PAGE + tok0 % PM_PAGE) * p.pad + d;
                if (!ok || tok0 >= p.T) continue;          // (whole pages)
#pragma unroll
                for (int e = 0; e < 16; ++e) st_g(o + (size_t) ((e & 3) + 8 * (e >> 2) + 4 * h_) * p.pad, f2bf(acc[m][n][e]));
            }
            continue;
        }
        if constexpr (KIND == VALUES) {                    // V[page][head][pad][slot]: rows of the tile are W's, columns the keys
#pragma unroll
            for (int m = 0; m < MI; ++m) {
                const int row0 = t0 + wm * WM + m * 32, h = row0 / p.rows_h, d0 = row0 - h * p.rows_h;
                uint16_t * o = (uint16_t *) p.y + (((size_t) (col / PM_PAGE) * p.H + h) * p.pad + d0) * PM_PAGE + col % PM_PAGE;
                if (!ok || h >= p.H) continue;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int in = (e & 3) + 8 * (e >> 2) + 4 * h_;
                    if (d0 + in < p.per) st_g(o + (size_t) in * PM_PAGE, f2bf(acc[m][n][e]));
                }
            }
            continue;
        }
        (void) ok;
    }
    if constexpr (KIND <= EXPERTS) {
        // (everything the stores need is in registers or LDS: a load among them would wait for the stores in front of it)
#pragma unroll
        for (int n = 0; n < NI; ++n) asm volatile("" : "+v"(bias[n]));
#pragma unroll
        for (int m = 0; m < MI; ++m)
#pragma unroll
            for (int n = 0; n < NI; ++n)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[m][n][e] += bias[n];
        if (p.act_fn) {
#pragma unroll
            for (int m = 0; m < MI; ++m)
#pragma unroll
                for (int n = 0; n < NI; ++n)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[m][n][e] = act_apply(p.act_fn, acc[m][n][e]);
        }
        auto put = [&](auto * y, bool whole) __attribute__((always_inline)) {
#pragma unroll
            for (int m = 0; m < MI; ++m)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int in = wm * WM + m * 32 + (e & 3) + 8 * (e >> 2) + 4 * h_;
                    if (!whole && t0 + in >= n_tok) continue;
                    float w = 1.0f;
                    int tok = t0 + in;
                    if constexpr (KIND == EXPERTS) { w = s_weight[in]; tok = s_pair[in]; }
                    auto * row = y + (size_t) tok * p.ldy + n0 + wn * WN + lr;
#pragma unroll
                    for (int n = 0; n < NI; ++n)
                        if (whole || n0 + wn * WN + n * 32 + lr < p.n_store) st_g(row + n * 32, from_f<std::remove_reference_t<decltype(*y)>>(KIND == EXPERTS ? acc[m][n][e] * w : acc[m][n][e]));
                }
        };
        const bool whole = t0 + BM <= n_tok && n0 + BN <= p.n_store;
        if (p.y_type == PM_BF16) { if (whole) put((uint16_t *) p.y, true); else put((uint16_t *) p.y, false); }
        else { if (whole) put((float *) p.y, true); else put((float *) p.y, false); }
    }
}

// One matrix over many tokens (or experts: sorted pairs, 256 per tile): tiles of 32 MI tokens x 64 NI rows, eight waves of 16 MI x 16 NI, so that tiles can be cut to what a batch has (835 tokens are 3.3 tiles of 256 and 3.7 of 224, and
// 10240 rows 40 tiles of 256 - 160 workgroups - and 54 of 192). v_mfma_f32_16x16x32_bf16 (the rate of 32 x 32 x 16 per bit of operand): rows of W are the tile's rows, so that a lane holds
// four neighbouring outputs of a token and stores them together. Both operands by LDS-DMA as in the kernel above, as many stages as fit.
// What bounds it: a step of 64 k of a 256 x 256 tile takes 1.65 us - its products and the LDS reads for them 1.4, its lines from the L2s 1.45 beside that -, in proportion to the tile's area.
template <int MI, int NI> struct Tile { static constexpr int BM = 32 * MI, BN = 64 * NI, STAGE = (BM + BN) * 128, STAGES = (160 * 1024 - 1) / STAGE; };
template <int MI, int NI, bool EXP> __global__ __launch_bounds__(512) void dense_tile_kernel(GemmP p) {
    typedef Tile<MI, NI> S;
    constexpr int BM = S::BM, BN = S::BN, STAGE = S::STAGE, STAGES = S::STAGES, ALL = (BM + BN) / 8, PIECES = (ALL + 7) / 8;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), lane = threadIdx.x & 63, lr = lane & 15, g = lane >> 4;
    const int wm = wave >> 2, wn = wave & 3;
    const int nt = EXP ? __builtin_amdgcn_readfirstlane(ld_g(p.tiles)) : p.nt;               // (the grid has room for the most tiles there can be)
    const int tiles = nt * p.nn, total = EXP ? tiles : tiles * p.splits, per = (total + 7) / 8;      // (order of the tiles: as above)
    int slot = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (slot >= total || (int) (blockIdx.x >> 3) >= per) return;
    const int split = EXP ? 0 : slot / tiles;
    slot -= split * tiles;
    const int band = slot / (8 * p.nn), left = nt - band * 8, bh = left < 8 ? left : 8, in = slot - band * 8 * p.nn;
    int t0 = (band * 8 + in % bh) * BM, n_tok = p.T;
    const int n0 = (in / bh) * BN, k0 = EXP ? 0 : split * p.split_steps;
    const int steps = !EXP && p.split_steps < (p.K >> 6) - k0 ? p.split_steps : (p.K >> 6) - k0;
    const uint16_t * W = p.W;
    if constexpr (EXP) {                                   // t0 .. n_tok: sorted pairs of this tile
        const int32_t * tt = p.tiles + 1 + 3 * (band * 8 + in % bh);
        W += (int64_t) __builtin_amdgcn_readfirstlane(ld_g(tt)) * p.e_stride;
        t0 = __builtin_amdgcn_readfirstlane(ld_g(tt + 1)); n_tok = t0 + __builtin_amdgcn_readfirstlane(ld_g(tt + 2));
    }
    // pieces of 8 rows x 128 bytes, wave, wave + 8, .. (a wave without a last one brings the last one again: the same bytes to the same place)
    const char * xb = (const char *) (EXP ? p.X : p.X + (size_t) t0 * p.lda), * wb = (const char *) (W + (size_t) n0 * p.K);
    const int x_last = n_tok - 1 - t0, w_last = p.N - 1 - n0;
    const uint32_t lds0 = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) char *) smem;
    uint32_t off[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int q = min(wave + 8 * i, ALL - 1), r = q * 8 + (lane >> 3);
        const bool tok = q < BM / 8;
        int row = tok ? min(r, x_last) : min(r - BM, w_last);
        if constexpr (EXP) if (tok) { row += t0; if (p.gather) row = ld_g(p.order + row) / p.top; }
        off[i] = (uint32_t) row * (uint32_t) (tok ? p.lda : p.K) * 2u + (uint32_t) ((lane & 7) ^ ((r >> 1) & 7)) * 16u;
    }
    auto request = [&](int k, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int q = min(wave + 8 * i, ALL - 1);
            pm_dma16((q < BM / 8 ? xb : wb) + (size_t) (k0 + k) * 128, off[i], lds0 + (uint32_t) (stage * STAGE) + (uint32_t) q * 1024u);
        }
    };
    f32x4 acc[NI][MI];
#pragma unroll
    for (int n = 0; n < NI; ++n)
#pragma unroll
        for (int m = 0; m < MI; ++m) acc[n][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // (rows of one operand's blocks are 16 apart: the swizzle is the lane's own)
    const uint32_t x_at = (uint32_t) (wm * 16 * MI + lr) * 128u, w_at = (uint32_t) (BM + wn * 16 * NI + lr) * 128u, sw = (uint32_t) (lr >> 1) & 7u;
#pragma unroll
    for (int i = 0; i < STAGES - 1; ++i) if (i < steps) request(i, i);
    int stage = 0, next = STAGES - 1;
    for (int k = 0; k < steps; ++k) {
        const int ahead = steps - 1 - k;                   // (as in the kernel above)
        static_assert(STAGES >= 2 && STAGES <= 5, "the waits are spelled for these");
        if (STAGES > 2 && ahead >= STAGES - 2) vm_wait<PIECES * (STAGES - 2)>();
        else if (STAGES > 4 && ahead == 2) vm_wait<PIECES * 2>();
        else if (STAGES > 3 && ahead == 1) vm_wait<PIECES>();
        else vm_wait<0>();
        __syncthreads();
        if (k + STAGES - 1 < steps) request(k + STAGES - 1, next);
        const char * s = smem + stage * STAGE;
        bf16x8 x[2][MI], w[2][NI];
        auto read = [&](int j) __attribute__((always_inline)) {                  // 32 k of the stage
            const uint32_t c = ((uint32_t) (j * 4 + g) ^ sw) * 16u;
#pragma unroll
            for (int n = 0; n < NI; ++n) w[j][n] = *(const bf16x8 *) (s + w_at + n * 2048 + c);
#pragma unroll
            for (int m = 0; m < MI; ++m) x[j][m] = *(const bf16x8 *) (s + x_at + m * 2048 + c);
        };
        read(0);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (j == 0) read(1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < MI; ++m)
#pragma unroll
                for (int n = 0; n < NI; ++n) acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j][n], x[j][m], acc[n][m], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        stage = stage == STAGES - 1 ? 0 : stage + 1;
        next = next == STAGES - 1 ? 0 : next + 1;
    }
    f32x4 bias[NI];
#pragma unroll
    for (int n = 0; n < NI; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) { const int col = n0 + (wn * NI + n) * 16 + g * 4 + e; bias[n][e] = p.bias && split == 0 && col < p.n_store ? ld_g(p.bias + col) : 0.0f; }
#pragma unroll
    for (int n = 0; n < NI; ++n) asm volatile("" : "+v"(bias[n]));
    int pair[EXP ? MI : 1];
    float weight[EXP ? MI : 1];
    if constexpr (EXP) {                                   // what the stores need about their rows
#pragma unroll
        for (int m = 0; m < MI; ++m) {
            const int i = t0 + (wm * MI + m) * 16 + lr;
            pair[m] = ld_g(p.order + (i < n_tok ? i : n_tok - 1));
            weight[m] = p.weight ? ld_g(p.weight + pair[m]) : 1.0f;
        }
#pragma unroll
        for (int m = 0; m < MI; ++m) asm volatile("" : "+v"(pair[m]), "+v"(weight[m]));
    }
    const bool four = p.ldy % 4 == 0 && ((uintptr_t) p.y & 15) == 0;      // (four outputs together where rows and their start allow it)
    auto put = [&](auto * y, bool whole) __attribute__((always_inline)) {
        typedef std::remove_reference_t<decltype(*y)> Y;
#pragma unroll
        for (int m = 0; m < MI; ++m) {
            int tok = t0 + (wm * MI + m) * 16 + lr;
            if (tok >= n_tok) continue;
            if constexpr (EXP) { if (p.scatter) tok = pair[m]; }
            Y * row = y + (EXP ? (size_t) tok : p.rows ? (size_t) tok * p.splits + split : (size_t) split * p.T + tok) * p.ldy + n0 + wn * 16 * NI + g * 4;
#pragma unroll
            for (int n = 0; n < NI; ++n) {
                f32x4 v = acc[n][m] + bias[n];
                if (p.act_fn) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = act_apply(p.act_fn, v[e]);
                }
                if constexpr (EXP) v *= weight[m];
                const int col = n0 + (wn * NI + n) * 16 + g * 4;
                if (whole || (four && col + 4 <= p.n_store)) {
                    if constexpr (sizeof(Y) == 4) *(PM_G f32x4 *) (row + n * 16) = v;
                    else *(PM_G u32x2 *) (row + n * 16) = u32x2{(uint32_t) f2bf(v[0]) | (uint32_t) f2bf(v[1]) << 16, (uint32_t) f2bf(v[2]) | (uint32_t) f2bf(v[3]) << 16};
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) if (col + e < p.n_store) st_g(row + n * 16 + e, from_f<Y>(v[e]));
                }
            }
        }
    };
    const bool whole = four && n0 + BN <= p.n_store;
    if (p.y_type == PM_BF16) { if (whole) put((uint16_t *) p.y, true); else put((uint16_t *) p.y, false); }
    else { if (whole) put((float *) p.y, true); else put((float *) p.y, false); }
}
template <int MI, int NI, bool EXP = false> int launch_tile(GemmP p, hipStream_t st) {
    typedef Tile<MI, NI> S;
    if (p.splits < 1) { p.splits = 1; p.split_steps = p.K >> 6; }
    if (!EXP) p.nt = (p.T + S::BM - 1) / S::BM;
    p.nn = (p.n_store + S::BN - 1) / S::BN;
    const size_t lds = (size_t) S::STAGES * S::STAGE;
    pm_allow_big_lds((const void *) dense_tile_kernel<MI, NI, EXP>, lds);
    hipLaunchKernelGGL((dense_tile_kernel<MI, NI, EXP>), dim3((p.nt * p.nn * p.splits + 7) / 8 * 8), dim3(512), lds, st, p);
    return 0;
}

// sums of k ranges -> act(sum + bias)
__global__ __launch_bounds__(256) void reduce_kernel(const float * part, int splits, int T, int ldp, const float * bias, int act_fn, void * y, int ldy, int y_type, int n_store) {
    const int quads = ldp / 4;
    const long i = (long) blockIdx.x * 256 + threadIdx.x;
    if (i >= (long) T * quads) return;
    const int t = (int) (i / quads), c = (int) (i - (long) t * quads) * 4;
    const float * src = part + (size_t) t * ldp + c;
    f32x4 v = *(const PM_G f32x4 *) src;
    for (int s = 1; s < splits; s += 4) {                  // four loads at a time
        f32x4 r[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] = *(const PM_G f32x4 *) (src + (size_t) (s + j < splits ? s + j : 0) * T * ldp);
#pragma unroll
        for (int j = 0; j < 4; ++j) if (s + j < splits) v += r[j];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) if (c + e < n_store) st_type(y, (size_t) t * ldy + c + e, y_type, act_apply(act_fn, v[e] + (bias ? ld_g(bias + c + e) : 0.0f)));
}

template <int BM, int BN, int WM, int WN, int STAGES, int KIND> int launch_stages(GemmP p, hipStream_t st) {
    constexpr int threads = BM / WM * (BN / WN) * 64;
    if (KIND != EXPERTS) p.nt = (p.T + BM - 1) / BM;
    p.nn = (p.n_store + BN - 1) / BN;
    const size_t lds = (size_t) STAGES * (BM + BN) * 128;
    pm_allow_big_lds((const void *) dense_gemm_kernel<BM, BN, WM, WN, STAGES, KIND>, lds);
    const int per = (p.nt * p.nn + 7) / 8;
    hipLaunchKernelGGL((dense_gemm_kernel<BM, BN, WM, WN, STAGES, KIND>), dim3(per * 8), dim3(threads), lds, st, p);
    return 0;
}
// up to one tile per CU: twice the stages hide the memory's latency; more: two tiles share a CU
template <int KIND> int launch_128(const GemmP & p, hipStream_t st) {
    if constexpr (KIND != EXPERTS) if ((long) ((p.T + 127) / 128) * ((p.n_store + 127) / 128) <= 256) return launch_stages<128, 128, 64, 64, 4, KIND>(p, st);
    return launch_stages<128, 128, 64, 64, 2, KIND>(p, st);
}

// Forms of one matrix and the us they take: c per round of workgroups, out32 (out16) per MB of f32 (bf16) results, `rag` where the last token tile is not full, and per 64-k step `step`, of which
// `fill` also where a workgroup runs alone, and `weights` for lines of W that no other token tile asks for. Least squares of the logarithms over 25 matrices of 512..14336 x 1024..32000, 65..4096
// tokens, either type of results, up to 32 k ranges, weights out of memory and out of the last-level cache (residuals 5 to 10 %; the last three by 1 .. 3 % less, they are what the choice was between
// before there were tiles). Choices are 0.5 .. 2 % in the mean from the best form of all; of 1752 products without ranges 30 are more than 3 % (12 % at most) behind the former choice, the mean is
// 0.95 of its time.
// The last three are dense_gemm_kernel's: two workgroups per CU, whose stores and steps overlap (257 x 8192 x 14336 out of the cache 92 us, in 160 x 256 tiles 125); 256 x 256 and 128 x 128 tiles of
// short rows, which it stores in half the time (2048 x 1024 x 14336 68.7 us, dense_tile_kernel's 70.8; 128 x 512 x 8192 8.3 / 9.5)
struct Form {
    int bm, bn, per_cu; bool tile; float c, step, fill, weights, out32, out16, rag;
    float us(int T, int nt, int64_t all, int64_t room, int steps, float values, bool f32) const {
        const int64_t full = all / room, last = all % room;
        const float part = (float) last / (float) room;
        return (float) ((all + room - 1) / room) * c + values * (f32 ? 4e-6f * out32 : 2e-6f * out16) + (T % bm ? rag : 0.0f) +
               (float) steps * ((float) full * (step + weights / nt) + (last ? step * (fill + (1.0f - fill) * part) + weights * part / nt : 0.0f));
    }
};
constexpr Form forms[] = {{128, 128, 1, true, 4.8f, 0.468f, 0.911f, 0.177f, 0.139f, 0.0f, 0.33f}, {160, 256, 1, true, 7.8f, 0.953f, 0.896f, 0.123f, 0.13f, 0.072f, 0.0f},
                          {224, 256, 1, true, 3.8f, 1.283f, 0.87f, 0.0f, 0.154f, 0.208f, 4.0f}, {256, 256, 1, true, 8.2f, 1.378f, 0.892f, 0.0f, 0.144f, 0.187f, 0.0f},
                          {128, 128, 2, false, 1.4f, 0.87f, 0.474f, 0.53f, 0.116f, 0.14f, 1.44f}, {256, 256, 1, false, 5.0f, 1.49f, 0.792f, 0.083f, 0.09f, 0.075f, 1.65f},
                          {128, 128, 1, false, 3.3f, 0.53f, 0.892f, 0.138f, 0.046f, 0.0f, 1.67f}};

} // namespace

int pm_launch_dense_small(const pm_dense_args & a, hipStream_t st);

int pm_launch_dense_gemm(const pm_dense_args & a, hipStream_t st) {
    if (a.type != PM_BF16 || a.K % 64 || a.N % 64 || a.n_store > a.N || a.T < 1 || a.pro) return PM355_E_SHAPE;
    GemmP p = {};
    p.W = (const uint16_t *) a.W; p.X = (const uint16_t *) a.act; p.y = a.y; p.bias = a.bias; p.K = a.K; p.N = a.N; p.T = a.T; p.lda = a.lda; p.ldy = a.ldy; p.y_type = a.y_type;
    p.n_store = a.n_store; p.act_fn = a.act_fn;
    // The tile whose rounds take the least time. With too few tiles for the chip ranges of k go to different workgroups; their f32 sums are written, and added up by a launch of their own or by the
    // norm behind the product (a workgroup per token, which reads 15 KB of them in a us).
    // Measured on 835 tokens, in a pass between other launches: 10240 x 4096 98 us in 160 tiles of 256 x 256, 79 in 240 of 160 x 256; 14336 x 4096 107 (224 of 256 x 256) / 100 (224 of 224 x
    // 256); 4096 x 14336 135 (224 of 128 x 128, four waves) / 90 and 6 more in the norm behind it (64 of 224 x 256 in four ranges); 4096 x 4096 44 / 41 (128 x 128 tiles by eight waves)
    const int steps = a.K >> 6, ldp = a.parts ? a.ldy : (a.n_store + 3) / 4 * 4;
    const bool may_split = a.split && (!a.parts || a.act_fn == PM355_ACT_NONE);
    auto summed = [&](int s) { return 3.7f + (float) (s + 1) * a.T * ldp * 4.6e-7f; };                                              // us of the launch that adds them up, and
    auto normed = [&](int s) { return std::max((float) (s - 1) * ldp / 3900, (float) (s - 1) * a.T * ldp * 6.7e-7f); };             // of what the norm takes longer
    int form = 0, splits = 1;
    float best = INFINITY;
    for (int f = 0; f < (int) std::size(forms); ++f) {
        const int nt = (a.T + forms[f].bm - 1) / forms[f].bm;
        const int64_t tiles = (int64_t) nt * ((a.n_store + forms[f].bn - 1) / forms[f].bn), room = (int64_t) pm_device_cus() * forms[f].per_cu;
        if (forms[f].per_cu > 1 && tiles <= pm_device_cus()) continue;
        for (int s = 1; s == 1 || (forms[f].tile && may_split && s * tiles <= room && s * 4 <= steps && (size_t) s * a.T * ldp <= a.split_floats); ++s) {
            float t = forms[f].us(a.T, nt, tiles * s, room, (steps + s - 1) / s, (float) s * a.T * ldp, s > 1 || a.y_type == PM_F32);
            if (s > 1) t += a.parts ? std::min(summed(s), normed(s)) : summed(s);
            if (t < best) { best = t; form = f; splits = s; }
        }
    }
    auto go = [&]() -> int {
        switch (form) {
            case 0: return launch_tile<4, 2>(p, st);
            case 1: return launch_tile<5, 4>(p, st);
            case 2: return launch_tile<7, 4>(p, st);
            case 3: return launch_tile<8, 4>(p, st);
            case 4: return launch_stages<128, 128, 64, 64, 2, DENSE>(p, st);
            case 5: return launch_stages<256, 256, 128, 64, 2, DENSE>(p, st);
            default: return launch_stages<128, 128, 64, 64, 4, DENSE>(p, st);
        }
    };
    if (a.parts) *a.parts = 0;
    if (splits > 1) {
        p.split_steps = (steps + splits - 1) / splits; p.splits = (steps + p.split_steps - 1) / p.split_steps;
        p.y = a.split; p.ldy = ldp; p.y_type = PM_F32; p.act_fn = PM355_ACT_NONE;
        if (a.parts && normed(p.splits) <= summed(p.splits)) { *a.parts = p.splits; p.rows = 1; return go(); }
        p.bias = nullptr;
        go();
        hipLaunchKernelGGL(reduce_kernel, dim3((unsigned) (((long) a.T * (ldp / 4) + 255) / 256)), dim3(256), 0, st, a.split, p.splits, a.T, ldp, a.bias, a.act_fn, a.y, a.ldy, a.y_type, a.n_store);
        return 0;
    }
    return go();
}

int pm_launch_dense(const pm_dense_args & a, hipStream_t st) {
    return a.pro || a.group || a.type != PM_BF16 || a.T <= 64 ? pm_launch_dense_small(a, st) : pm_launch_dense_gemm(a, st);
}

int pm_launch_experts_gemm(const pm_expert_args & a, hipStream_t st) {
    const int64_t pairs = (int64_t) a.T * a.r.top;
    if (a.type != PM_BF16 || a.T < 1 || a.width_p % 64 || a.ffp % 64 || (int64_t) a.T * a.ldx * 2 >= 1ll << 32 || pairs * a.ffp * 2 >= 1ll << 32) return PM355_E_SHAPE;
    GemmP p = {};
    p.tiles = a.r.tiles; p.order = a.r.order; p.top = a.r.top;
    if (a.r.tile != 128 && a.r.tile != 256) return PM355_E_SHAPE;
    auto go = [&]() { return a.r.tile == 256 ? launch_tile<8, 4, true>(p, st) : launch_128<EXPERTS>(p, st); };
    p.nt = (int) (pairs / a.r.tile + (a.r.E < pairs ? a.r.E : pairs));                  // (most tiles there can be: every expert's last one may be short)
    p.W = (const uint16_t *) a.up; p.e_stride = a.up_stride; p.X = (const uint16_t *) a.x; p.lda = a.ldx; p.K = a.width_p; p.N = p.n_store = a.ffp; p.y = a.hid; p.ldy = a.ffp;
    p.y_type = PM_BF16; p.act_fn = a.act_fn; p.gather = 1; p.weight = a.r.w;
    go();
    p.W = (const uint16_t *) a.down; p.e_stride = a.down_stride; p.X = (const uint16_t *) a.hid; p.lda = a.ffp; p.K = a.ffp; p.N = a.width_p; p.n_store = a.width; p.y = a.y; p.ldy = a.ldy;
    p.y_type = a.y_type; p.act_fn = PM355_ACT_NONE; p.gather = 0; p.scatter = 1; p.weight = nullptr;
    return go();
}

int pm_launch_latent_expand(const pm_latent_expand & x, hipStream_t st) {
    if (x.n_pages < 1 || x.kvp % 64 || x.ld % 64) return PM355_E_SHAPE;
    GemmP p = {};
    p.pages = x.pages; p.X = (const uint16_t *) x.cache; p.lda = x.ld; p.K = x.kvp; p.H = x.H;
    GemmP k = p;
    k.W = (const uint16_t *) x.Wk; k.T = x.n_pages * PM_PAGE; k.n_store = x.H * x.dim; k.N = pm_dense_pad(k.n_store); k.y = x.K; k.per = x.dim; k.pad = x.dkp;
    launch_128<KEYS>(k, st);
    p.W = (const uint16_t *) x.Wv; p.T = pm_dense_pad(x.H * x.vrows); p.N = p.n_store = x.n_pages * PM_PAGE; p.y = x.V; p.per = x.vdim; p.rows_h = x.vrows; p.pad = x.dvp;
    return launch_128<VALUES>(p, st);
}
