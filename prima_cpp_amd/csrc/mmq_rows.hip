// mmq_rows.hip - quantized mat-mul for 1..8 tokens, some shapes and types up to 32 (pm_mmq_rows_takes: the rest is mmq_i8.hip's and mmq_mid.hip's): weights from memory straight into the operands of v_mfma_i32_16x16x64_i8 / 16x16x32_i8, no LDS on their way.
//
// The arithmetic is mmq_i8.hip's (activations in Q8_K / Q8_0 blocks, exact integer sums per super-block, one f32 multiply-add per super-block): what differs is where the bytes go. A workgroup
// owns a slice of the rows of one matrix, its eight waves share K: a wave takes PAIRS of super-blocks, pair w, w + 8, ..., for all rows of the slice, 16 at a time. So
//   * a pair's activations are loaded once per wave and serve every row group (mmq_i8.hip's waves own row groups: each loads all activations of its K range again),
//   * row groups are 16 rows, so a matrix of 4096 rows has one for each of the 256 CUs (32-row groups: half of them stood still),
//   * the order of the sums depends on K only - the same bits whatever the launch, its row split or the number of tokens.
// Operands: B = weights, lane (r = lane % 16, kg = lane / 16) of row r; A = activations, operand row a = (h = a / 8, t = a % 8). kg = 0, 1 hold the first, kg = 2, 3 the second super-block of
// the pair, and operand rows of h = 0 are zero for kg = 2, 3 and the other way round: one product is one scale group of BOTH, and result lane (r, g) holds tokens 4 (g % 2) + i of super-block
// h = g / 2, next to that super-block's scales of its own row.
// Bound by the weights' stream (alone 6.4 TB/s on the large shapes) and, a fifth above it, by what else asks for lines and by the vector work (190 instructions per 16 rows x 512 k of Q4_K, 340
// of Q6_K). Launches of 8 tokens, us, mmq_i8.hip's form of them / here: 8B shape wq | wk | wv 9.6 / 7.8, wo 7.6 / 5.7, ffn_gate | ffn_up 19.2 / 17.4, ffn_down 13.3 / 12.8 (Q4_K), 25.2 / 18.0
// (Q6_K), head 119 / 97; 70B shape 19.3 / 16.0, 17.9 / 18.2 (wo and Q4_K ffn_down), 52.0 / 47.4, Q6_K ffn_down 49.9 / 47.3; Q8_0 8192 x 29568 54 / 52.
#include "pm355_device.h"
#include "pm355_kernels.h"
#include "pm355_mmq_rows.h"
#include <algorithm>

namespace {

typedef int      i32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int KW = 8, NT = 64 * KW;                                // waves of a workgroup = pairs of a step

__device__ __forceinline__ i32x4 mfma_64(u32x4 a, u32x4 b) { const i32x4 z = {0, 0, 0, 0}; return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), z, 0, 0, 0); }
__device__ __forceinline__ i32x4 mfma_32(u32x2 a, u32x2 b) { const i32x4 z = {0, 0, 0, 0}; return __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, a), __builtin_bit_cast(long, b), z, 0, 0, 0); }
__device__ __forceinline__ f32x4 mfma_h(u32x4 a, u32x4 b) { const f32x4 z = {0, 0, 0, 0}; return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), z, 0, 0, 0); }
// rows (of 16 lanes) 1, 3 of x change places with rows 0, 2 of y
__device__ __forceinline__ void swap16(u32x4 & x, u32x4 & y) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t a = x[i], b = y[i];
        const u32x2 r = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(a, b, false, false));
        x[i] = r[0]; y[i] = r[1];
    }
}
// the same for the halves of a 16-byte piece: lanes kg = 0, 1 (2, 3) then hold the first one's piece in x[0..1], the second one's in x[2..3], eight bytes each
__device__ __forceinline__ void swap16h(u32x4 & x) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t a = x[i], b = x[2 + i];
        const u32x2 r = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(a, b, false, false));
        x[i] = r[0]; x[2 + i] = r[1];
    }
}
__device__ __forceinline__ uint32_t pk_fma(uint32_t a, _Float16 m, _Float16 c) {
    const f16x2 v = __builtin_bit_cast(f16x2, a), mm = {m, m}, cc = {c, c};
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(v, mm, cc));
}
__device__ __forceinline__ u32x4 ld_c16(const void * p) { return *(const PM_G u32x4 *) p; }
__device__ __forceinline__ u32x4 ld_buf(__amdgpu_buffer_rsrc_t r, uint32_t lane, int at) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int) lane, at, 0)); }

// first super-block that a pair's registers hold: an odd last pair moves back by one, whose half then has activation scales of zero (as have both of a pair past the end: every wave takes
// the same number of pairs, without a branch)
__device__ __forceinline__ int first_of(int pair, int nsb) { return min(2 * pair, nsb - 2); }

// Full lines: the eight 16-byte pieces of a 128-byte line of a stream (a pair's) are fetched by ONE instruction - x by rows 0..7, y by rows 8..15 of the sixteen, lane (l = lane % 16, kg):
// x: row l % 8, piece piece_of(kg, l / 8); y: row 8 + l % 8, piece piece_of(kg, 1 - l / 8). (64 bytes per row and instruction, two instructions to a line: 57344 x 8192 Q4_K 88 us instead of
// 62 - what limits a CU is the number of lines it asks for.) Then x gets pieces piece_of(kg, 0) of all sixteen rows, y pieces piece_of(kg, 1).
__device__ __forceinline__ int piece_of(int kg, int half) { return (kg & 1) + 4 * (kg >> 1) + 2 * half; }
__device__ __forceinline__ void halves(u32x4 & x, u32x4 & y) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int a = (int) x[i], b = (int) y[i];
        const int t = __builtin_amdgcn_update_dpp(0, b, 0x128 /*row_ror:8*/, 0xF, 0xF, true);
        y[i] = (uint32_t) __builtin_amdgcn_update_dpp(t, a, 0x128, 0xF, 0x3, false);
        x[i] = (uint32_t) __builtin_amdgcn_update_dpp(a, b, 0xE4 /*quad_perm 0 1 2 3*/, 0xF, 0xC, false);
    }
}

// ---- activations: a lane's operands of a pair (K-quants: sub-block j of either super-block; Q8_0: blocks j and 4 + j of eight) ------------------------------------------------
template <int TYPE> struct ASet { u32x4 q[8], bs; f32x4 yd; };
template <> struct ASet<PM_Q8_0> { u32x4 q[4]; f32x4 yd[4]; };
// from the tables that the quantizers (or mmq_i8.hip's prologue) write; lane offsets are out of range - zeros, no traffic - where the operand row is empty
// (g: the group of eight tokens; only the last one may have fewer)
struct ASrc { __amdgpu_buffer_rsrc_t rq, rb, rd; uint32_t qo[2], bo[2], dd; int n; };
template <int TYPE, int NG> __device__ __forceinline__ ASrc source_a(const RowsP & p, int nb, int lr, int kg) {
    constexpr bool Q80 = TYPE == PM_Q8_0;
    const int t = lr & 7, hk = kg >> 1;
    const bool on = (lr >> 3) == hk, on_last = on && t + 8 * (NG - 1) < p.T;
    ASrc s;
    s.n = nb;
    s.rq = __builtin_amdgcn_make_buffer_rsrc((void *) p.qT, 0, nb * (Q80 ? 1024 : 8192), 0x00020000);
    s.rb = __builtin_amdgcn_make_buffer_rsrc((void *) p.bsT, 0, nb * 1024, 0x00020000);
    s.rd = __builtin_amdgcn_make_buffer_rsrc((void *) p.dT, 0, nb * 128, 0x00020000);
    const uint32_t qo = (uint32_t) (hk * (Q80 ? 4096 : 8192) + (32 * (kg & 1) + t + p.t_off) * 16), bo = (uint32_t) (hk * 1024 + (32 * (kg & 1) + t + p.t_off) * 16);
    s.qo[0] = on ? qo : 0x80000000u; s.qo[1] = on_last ? qo : 0x80000000u;
    s.bo[0] = on ? bo : 0x80000000u; s.bo[1] = on_last ? bo : 0x80000000u;
    s.dd = (uint32_t) (hk * (Q80 ? 512 : 128) + 16 * (kg & 1) + 4 * p.t_off);
    return s;
}
template <int TYPE> __device__ __forceinline__ void load_q(ASet<TYPE> & a, const ASrc & s, int g, bool last, int pair, int j) {
    const uint32_t o = s.qo[last] + (uint32_t) (128 * g);
    if constexpr (TYPE == PM_Q8_0) a.q[j] = ld_buf(s.rq, o + (uint32_t) (j * 1024), min(pair, (s.n + 7) / 8 - 1) * 8192);
    else a.q[j] = ld_buf(s.rq, o + (uint32_t) ((j & 3) * 1024), first_of(pair, s.n) * 8192 + (j >> 2) * 4096);
}
template <int TYPE> __device__ __forceinline__ void load_yd(ASet<TYPE> & a, const ASrc & s, int g, bool last, int pair, int hk) {
    if constexpr (TYPE == PM_Q8_0) {
        // blocks behind the last one of a row (and pairs behind the last one): scale 0
        const int pc = min(pair, (s.n + 7) / 8 - 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) a.yd[j] = __builtin_bit_cast(f32x4, ld_buf(s.rd, 8 * pair + 4 * hk + j < s.n ? s.dd + (uint32_t) (j * 128 + 32 * g) : 0x80000000u, pc * 1024));
    } else {
        const int sb = first_of(pair, s.n);
        a.bs = ld_buf(s.rb, s.bo[last] + (uint32_t) (128 * g), sb * 1024);
        a.yd = __builtin_bit_cast(f32x4, ld_buf(s.rd, sb + hk >= 2 * pair ? s.dd + (uint32_t) (32 * g) : 0x80000000u, sb * 128));
    }
}
// All activations in LDS, 8 tokens of each super-block: where the waves go over them several times (more rows per workgroup than one pass takes)
//   K-quants: values [nb][8 sub-blocks][2][8 t][16] | group sums [nb][2][8 t][8 F16] | scales [nb][8];  Q8_0 (per 8 blocks): values [8][2][8 t][16] | - | scales [8][8]
// in front of them 2 KiB of zeros, which the lanes of empty operand rows read
template <int TYPE> struct ALds {
    static constexpr int Q = 2048, B = TYPE == PM_Q8_0 ? 0 : 256, D = TYPE == PM_Q8_0 ? 256 : 32, ZERO = 2048;
    static size_t bytes(int n) { return ZERO + (size_t) n * (Q + B + D); }     // n super-blocks
};
// (two parts: the pieces of the first round - all of them up to 32 super-blocks - are asked for in front of the first weights and stored behind those requests: loads return in order, so the
// store waits for the activations alone. Asked for and stored kind by kind before the first weight was, they were three rounds of latency: ffn_gate | ffn_up of the 8B shape at 8 tokens, this and
// the arguments in registers, 16.7 us, now 15.3; of the 70B shape 44.9 / 44.5, the 8B head 97.1 / 95.5)
template <int TYPE> struct StageA { u32x4 q[8], b, d; };
template <int TYPE> __device__ __forceinline__ u32x4 stage_q(const RowsP & p, int lim, int i) {
    return ld_c16(p.qT + (size_t) min(i >> 4, lim - 1) * 1024 + (32 * ((i >> 3) & 1) + (i & 7) + p.t_off) * 16);
}
__device__ __forceinline__ u32x4 stage_b(const RowsP & p, int n, int i) { return ld_c16(p.bsT + (size_t) min(i >> 4, n - 1) * 1024 + (32 * ((i >> 3) & 1) + (i & 7) + p.t_off) * 16); }
__device__ __forceinline__ u32x4 stage_d(const RowsP & p, int rows, int i) { return ld_c16(p.dT + (size_t) min(i >> 1, rows - 1) * 32 + 4 * (i & 1) + p.t_off); }
template <int TYPE> __device__ __forceinline__ void load_stage(StageA<TYPE> & a, const RowsP & p, int n) {
    const int tid = threadIdx.x, lim = TYPE == PM_Q8_0 ? p.K / 32 : n * 8;         // sub-blocks / blocks of the row
#pragma unroll
    for (int u = 0; u < 8; ++u) a.q[u] = stage_q<TYPE>(p, lim, min(tid + u * NT, n * 128 - 1));
    if constexpr (TYPE != PM_Q8_0) a.b = stage_b(p, n, tid);
    a.d = stage_d(p, TYPE == PM_Q8_0 ? lim : n, tid);
}
template <int TYPE> __device__ __forceinline__ void store_stage(uint8_t * L, const StageA<TYPE> & a, const RowsP & p, int n) {
    typedef ALds<TYPE> S;
    const int tid = threadIdx.x;
    const u32x4 z = {0, 0, 0, 0};
    const int lim = TYPE == PM_Q8_0 ? p.K / 32 : n * 8, rows = TYPE == PM_Q8_0 ? lim : n;
    uint8_t * const Lq = L + S::ZERO, * const Lb = Lq + (size_t) n * S::Q, * const Ld = Lb + (size_t) n * S::B;
    for (int i = tid; i < S::ZERO / 16; i += NT) *(u32x4 *) (L + i * 16) = z;
#pragma unroll
    for (int u = 0; u < 8; ++u) { const int i = tid + u * NT; if (i < n * 128) *(u32x4 *) (Lq + (size_t) i * 16) = (i >> 4) < lim ? a.q[u] : z; }
    if constexpr (TYPE != PM_Q8_0) if (tid < n * 16) *(u32x4 *) (Lb + tid * 16) = a.b;
    if (tid < n * S::D / 16) *(u32x4 *) (Ld + tid * 16) = (tid >> 1) < rows ? a.d : z;
    // longer rows: the rest
    for (int i = tid + 8 * NT; i < n * 128; i += NT) *(u32x4 *) (Lq + (size_t) i * 16) = (i >> 4) < lim ? stage_q<TYPE>(p, lim, i) : z;
    if constexpr (TYPE != PM_Q8_0) for (int i = tid + NT; i < n * 16; i += NT) *(u32x4 *) (Lb + i * 16) = stage_b(p, n, i);
    for (int i = tid + NT; i < n * S::D / 16; i += NT) *(u32x4 *) (Ld + i * 16) = (i >> 1) < rows ? stage_d(p, rows, i) : z;
}
struct ALane { uint32_t q, qi, b, bi, d; };                        // the lane's addresses in it, and what a super-block adds to them (0: an empty row)
template <int TYPE> __device__ __forceinline__ ALane lane_a(int n, int lr, int kg) {
    typedef ALds<TYPE> S;
    const int t = lr & 7, hk = kg >> 1;
    const bool on = (lr >> 3) == hk;
    ALane l;
    l.q = on ? S::ZERO + hk * (TYPE == PM_Q8_0 ? 1024 : S::Q) + (kg & 1) * 128 + t * 16 : 0; l.qi = on ? S::Q : 0;
    l.b = on ? S::ZERO + n * S::Q + hk * S::B + (kg & 1) * 128 + t * 16 : 0; l.bi = on ? S::B : 0;
    l.d = S::ZERO + n * (S::Q + S::B) + (TYPE == PM_Q8_0 ? hk * 128 : hk * S::D) + 16 * (kg & 1);
    return l;
}
template <int TYPE> __device__ __forceinline__ void read_a(ASet<TYPE> & a, const uint8_t * L, const ALane & l, int pair, int n, int hk) {
    typedef ALds<TYPE> S;
    const int sb = TYPE == PM_Q8_0 ? min(pair, n - 1) : first_of(pair, n);
    const bool live = TYPE == PM_Q8_0 ? pair < n : sb + hk >= 2 * pair;
    const uint8_t * q = L + (l.q + l.qi * (uint32_t) sb), * d = L + (live ? l.d + (uint32_t) S::D * (uint32_t) sb : 0);
    if constexpr (TYPE == PM_Q8_0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) { a.q[j] = *(const u32x4 *) (q + j * 256); a.yd[j] = *(const f32x4 *) (d + j * 32); }
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) a.q[j] = *(const u32x4 *) (q + j * 256);
        a.bs = *(const u32x4 *) (L + (l.b + l.bi * (uint32_t) sb));
        a.yd = *(const f32x4 *) d;
    }
}

// ---- weights ----------------------------------------------------------------------------------------------------------------------------------------------------------------
// where a wave's weights come from: the (scalar) start of the slice, blocks per row; the lane's offsets x / y (above)
struct WSrc { const uint8_t * base; int nb; };
struct Off { uint32_t x, y; };
// The scales of a step - all waves' pairs of all its rows - come in whole lines too, one 16-byte element a thread, through LDS: element (row, j) = super-block j of the step's 16 (Q8_0: pair j
// of 8: eight block scales). One step ahead, behind the barrier that ends a step. (By the lanes that need them: sixteen lines of 32 bytes per wave and row group, 7.6 us of 67 on that matrix.)
template <int TYPE> struct Scales {                                // Q4_K: headers (d, dmin, 6-bit scales and mins)
    static constexpr int PER_ROW = 16, PITCH = 272;
    u32x4 v;
    __device__ __forceinline__ void load(const WSrc & s, uint32_t row, int it, int j) { v = ld_c16(s.base + (size_t) s.nb * 128 + (row + 16u * (uint32_t) (first_of(KW * it + (j >> 1), s.nb) + (j & 1)))); }
    __device__ __forceinline__ void store(uint8_t * L, int row, int j) const { *(u32x4 *) (L + row * PITCH + j * 16) = v; }
};
template <> struct Scales<PM_Q6_K> {                               // int8 scales, behind them d
    static constexpr int PER_ROW = 16, PITCH = 304;
    u32x4 v; uint16_t d;
    __device__ __forceinline__ void load(const WSrc & s, uint32_t row, int it, int j) {
        const uint32_t sb = (uint32_t) (first_of(KW * it + (j >> 1), s.nb) + (j & 1));
        v = ld_c16(s.base + (row + pm_q6k_sc_off((uint32_t) s.nb, sb)));
        d = *(const PM_G uint16_t *) (s.base + (row + pm_q6k_d_off((uint32_t) s.nb, sb)));
    }
    __device__ __forceinline__ void store(uint8_t * L, int row, int j) const { *(u32x4 *) (L + row * PITCH + j * 16) = v; *(uint16_t *) (L + row * PITCH + 256 + 2 * j) = d; }
};
template <> struct Scales<PM_Q8_0> {
    static constexpr int PER_ROW = 8, PITCH = 144;
    u32x4 v;
    __device__ __forceinline__ void load(const WSrc & s, uint32_t row, int it, int j) { v = ld_c16(s.base + (size_t) s.nb * 32 + (row + 16u * (uint32_t) min(KW * it + j, (s.nb + 7) / 8 - 1))); }   // (rows are padded to 16 bytes)
    __device__ __forceinline__ void store(uint8_t * L, int row, int j) const { *(u32x4 *) (L + row * PITCH + j * 16) = v; }
};
template <> struct Scales<PM_Q5_K> {                               // (inside the native blocks)
    static constexpr int PER_ROW = 0, PITCH = 0;
    __device__ __forceinline__ void load(const WSrc &, uint32_t, int, int) {}
    __device__ __forceinline__ void store(uint8_t *, int, int) const {}
};
template <int TYPE> struct Tile;

// Q4_K / Q5_K: sum += scale_j * (w . a), scales and mins four to a dword (get_scale_min_k4, ggml-quants.c:1898-1906)
template <int NG> struct K4 {
    uint32_t sc[2], mn[2], dm; i32x4 sum[NG];
    __device__ __forceinline__ explicit K4(const u32x4 & hd) : dm(hd[0]), sum{} {
        sc[0] = hd[1] & 0x3f3f3f3fu; sc[1] = (hd[3] & 0x0f0f0f0fu) | ((hd[1] >> 2) & 0x30303030u);
        mn[0] = hd[2] & 0x3f3f3f3fu; mn[1] = ((hd[3] >> 4) & 0x0f0f0f0fu) | ((hd[2] >> 2) & 0x30303030u);
    }
    __device__ __forceinline__ void add(const i32x4 & acc, int g, int j) {
        const int s = (int) ((sc[j >> 2] >> (8 * (j & 3))) & 0xFFu);
#pragma unroll
        for (int i = 0; i < 4; ++i) { sum[g][i] = __mul24(s, acc[i]) + sum[g][i]; asm("" : "+v"(sum[g][i])); }   // (keeps it ONE v_mad_i32_i24)
    }
    // ... and the minima, exact: as F16 (0x6400 | m = 1024 + m), integer sums below 2^24 in f32
    template <class A> __device__ __forceinline__ void finish(const A (&a)[NG], f32x4 (&out)[NG]) const {
        u32x4 m;
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] = pk_fma(__builtin_amdgcn_perm(mn[i >> 1], 0x64646464u, i & 1 ? 0x00070006u : 0x00050004u), (_Float16) 1.0f, (_Float16) -1024.0f);
        const float d = h2f((uint16_t) (dm & 0xFFFF)), dmin = h2f((uint16_t) (dm >> 16));
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const f32x4 ms = mfma_h(a[g].bs, m);
#pragma unroll
            for (int i = 0; i < 4; ++i) out[g][i] = fmaf(a[g].yd[i] * d, (float) sum[g][i], fmaf(-(a[g].yd[i] * dmin), ms[i], out[g][i]));
        }
    }
};

// mul: L - the lane's row in the step's scales, kw - the wave's pair in the step; used(g, j): operand j of the activations of token group g has been read
// ---- Q4_K: qa[U][16] | qb[U][16] | hdr[nb][16] (unit u: bytes of sub-blocks 2 u in the low, 2 u + 1 in the high nibbles)
template <> struct Tile<PM_Q4_K> {
    u32x4 qa[2], qb[2];
    __device__ __forceinline__ void load(const WSrc & s, const Off & o, int, int pair) {
        const uint8_t * pa = s.base + (uint32_t) first_of(pair, s.nb) * 64u, * pb = pa + (size_t) s.nb * 64;
        qa[0] = ld_nt16(pa + o.x); qb[0] = ld_nt16(pb + o.x);
        qa[1] = ld_nt16(pa + o.y); qb[1] = ld_nt16(pb + o.y);
    }
    template <int NG, class F> __device__ __forceinline__ void mul(ASet<PM_Q4_K> (&a)[NG], const uint8_t * L, int kw, int kg, f32x4 (&out)[NG], F && used) {
        K4<NG> k(*(const u32x4 *) (L + (2 * kw + (kg >> 1)) * 16));
        halves(qa[0], qa[1]); halves(qb[0], qb[1]);
        swap16(qa[0], qb[0]); swap16(qa[1], qb[1]);                // units 0, 1, 2, 3
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const u32x4 & w = (j >> 1) & 1 ? qb[j >> 2] : qa[j >> 2];
            const u32x4 b = (j & 1 ? w >> 4 : w) & 0x0F0F0F0Fu;
#pragma unroll
            for (int g = 0; g < NG; ++g) { k.add(mfma_64(a[g].q[j], b), g, j); used(g, j); }
        }
        k.finish(a, out);
    }
};

// ---- Q5_K: native 176-byte blocks (d, dmin | scales[12] | qh[32] | qs[128]): loaded in operand order (wv of some layers: 2 % of a file). o.x: the lane's own row
template <> struct Tile<PM_Q5_K> {
    u32x4 q[4], qh, hd;
    __device__ __forceinline__ void load(const WSrc & s, const Off & o, int kg, int pair) {
        const uint8_t * p = s.base + (uint32_t) first_of(pair, s.nb) * 176u;
        const uint32_t at = o.x + 176u * (kg >> 1);
        hd = ld_c16(p + at);
        qh = ld_c16(p + 16 + (at + 16u * (kg & 1)));
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = ld_c16(p + 48 + 32 * u + (at + 16u * (kg & 1)));
    }
    template <int NG, class F> __device__ __forceinline__ void mul(ASet<PM_Q5_K> (&a)[NG], const uint8_t *, int, int, f32x4 (&out)[NG], F && used) {
        K4<NG> k(hd);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const u32x4 & w = q[j >> 1];
            const u32x4 b = ((j & 1 ? w >> 4 : w) & 0x0F0F0F0Fu) | (((qh >> j) & 0x01010101u) << 4);
#pragma unroll
            for (int g = 0; g < NG; ++g) { k.add(mfma_64(a[g].q[j], b), g, j); used(g, j); }
        }
        k.finish(a, out);
    }
};

// ---- Q6_K: la[U][16] | lb[U][16] | qh[U][16] | scales[nb][16] | d[nb]. Unit (hh, v): groups 8 hh + 2 c + v, c = 0..3. A scale group is 16 weights = one lane's piece: the swap works on
// its halves, so that a lane pair holds first a group of unit v = 0 whole, then one of v = 1; the products are 32 k wide
template <> struct Tile<PM_Q6_K> {
    u32x4 la[2], lb[2], qh[2];
    __device__ __forceinline__ void load(const WSrc & s, const Off & o, int, int pair) {
        const uint8_t * pa = s.base + (uint32_t) first_of(pair, s.nb) * 64u, * pb = pa + (size_t) s.nb * 64, * ph = pb + (size_t) s.nb * 64;
        la[0] = ld_nt16(pa + o.x); lb[0] = ld_nt16(pb + o.x); qh[0] = ld_nt16(ph + o.x);
        la[1] = ld_nt16(pa + o.y); lb[1] = ld_nt16(pb + o.y); qh[1] = ld_nt16(ph + o.y);
    }
    template <int NG, class F> __device__ __forceinline__ void mul(ASet<PM_Q6_K> (&a)[NG], const uint8_t * L, int kw, int kg, f32x4 (&out)[NG], F && used) {
        const u32x4 S = *(const u32x4 *) (L + (2 * kw + (kg >> 1)) * 16);
        const float d = h2f(*(const uint16_t *) (L + 256 + 2 * (2 * kw + (kg >> 1))));
        halves(la[0], la[1]); halves(lb[0], lb[1]); halves(qh[0], qh[1]);
        i32x4 sum[NG] = {};
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            swap16h(la[hh]); swap16h(lb[hh]); swap16h(qh[hh]);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
#pragma unroll
                for (int v = 0; v < 2; ++v) {
                    const u32x2 l = c & 1 ? u32x2{lb[hh][2 * v], lb[hh][2 * v + 1]} : u32x2{la[hh][2 * v], la[hh][2 * v + 1]}, h = {qh[hh][2 * v], qh[hh][2 * v + 1]};
                    const u32x2 q = ((c >> 1 ? l >> 4 : l) & 0x0F0F0F0Fu) | ((c == 0 ? h << 4 : c == 1 ? h << 2 : c == 2 ? h : h >> 2) & 0x30303030u);
                    const int G = 8 * hh + 2 * c + v, s = (int) (int8_t) (S[G >> 2] >> (8 * (G & 3)));
#pragma unroll
                    for (int g = 0; g < NG; ++g) {
                        const i32x4 acc = mfma_32(u32x2{a[g].q[4 * hh + c][2 * v], a[g].q[4 * hh + c][2 * v + 1]}, q);
#pragma unroll
                        for (int i = 0; i < 4; ++i) { sum[g][i] = __mul24(s, acc[i]) + sum[g][i]; asm("" : "+v"(sum[g][i])); }   // |acc| <= 16 * 63 * 127
                        if (v == 1) used(g, 4 * hh + c);
                    }
                }
            }
        }
        // - 32 sum_G scale_G * bsum_G (the offset of every weight): operand slot s of lane kg = scale of group 2 s + kg % 2, times -32 (F16: 1024 + 128 + scale from the bytes)
        const uint32_t sel = kg & 1 ? 0x00070005u : 0x00060004u;
        u32x4 m;
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] = pk_fma(__builtin_amdgcn_perm(S[i] ^ 0x80808080u, 0x64646464u, sel), (_Float16) -32.0f, (_Float16) 36864.0f);
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const f32x4 ms = mfma_h(a[g].bs, m);                       // (multiples of 32 below 2^29: exact)
#pragma unroll
            for (int i = 0; i < 4; ++i) out[g][i] = fmaf(a[g].yd[i] * d, (float) (sum[g][i] + (int) ms[i]), out[g][i]);
        }
    }
};

// ---- Q8_0: qa[nb][16] | qb[nb][16] | d[nb], blocks of 32; a pair is 8 blocks. Blocks past the row: the last one again, against activations and scales of zero
template <> struct Tile<PM_Q8_0> {
    u32x4 qa[2], qb[2];
    __device__ __forceinline__ void load(const WSrc & s, const Off & o, int kg, int pair) {
        const int l8 = (int) (threadIdx.x >> 3) & 1, px = piece_of(kg, l8), py = piece_of(kg, 1 - l8);
        const uint32_t ox = o.x + 16u * (uint32_t) (min(8 * pair + px, s.nb - 1) - px), oy = o.y + 16u * (uint32_t) (min(8 * pair + py, s.nb - 1) - py);
        const uint8_t * pb = s.base + (size_t) s.nb * 16;
        qa[0] = ld_nt16(s.base + ox); qb[0] = ld_nt16(pb + ox);
        qa[1] = ld_nt16(s.base + oy); qb[1] = ld_nt16(pb + oy);
    }
    template <int NG, class F> __device__ __forceinline__ void mul(ASet<PM_Q8_0> (&a)[NG], const uint8_t * L, int kw, int kg, f32x4 (&out)[NG], F && used) {
        const u32x2 d4 = *(const u32x2 *) (L + kw * 16 + 8 * (kg >> 1));
        halves(qa[0], qa[1]); halves(qb[0], qb[1]);
        swap16(qa[0], qb[0]); swap16(qa[1], qb[1]);                // blocks 0 | 4, 1 | 5, 2 | 6, 3 | 7
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t hb = (d4[j >> 1] >> (16 * (j & 1))) & 0xFFFFu;
            const float dw = (hb & 0x7C00u) == 0x7C00u ? 0.0f : h2f((uint16_t) hb);      // (padding behind the row, times zero)
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                const i32x4 acc = mfma_64(a[g].q[j], j & 1 ? qb[j >> 1] : qa[j >> 1]);
                used(g, j);
#pragma unroll
                for (int i = 0; i < 4; ++i) out[g][i] = fmaf((float) acc[i], dw * a[g].yd[j][i], out[g][i]);
            }
        }
    }
};

// A step: KW = 8 pairs, one per wave, of 16 R rows, times NG groups of eight tokens. D steps of weights are in flight; AL: activations from LDS
template <int TYPE, int NG, int R, int D, bool AL, bool EPI>
__device__ __forceinline__ void rows_body(const RowsP & p, const RowsJob & job, int w, int ji, uint8_t * smem) {
    constexpr int ROWS = 16 * R;
    typedef Scales<TYPE> SC;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lr = lane & 15, kg = lane >> 4, hk = kg >> 1;
    constexpr bool Q80 = TYPE == PM_Q8_0;
    // rows of workgroup w: `each`, and one more for the first `more` of them (in pairs for the rotation: they stay inside a workgroup)
    constexpr int STEP = EPI ? 2 : 1;
    const int r0 = STEP * (w * job.each + min(w, job.more)), r1 = STEP * ((w + 1) * job.each + min(w + 1, job.more));
    const int nb = Q80 ? p.K / 32 : p.K / 256, npair = Q80 ? (nb + 7) / 8 : (nb + 1) / 2, na = Q80 ? npair : nb;
    const int nit = (npair + KW - 1) / KW;                         // steps per pass over ROWS rows
    const int npass = (r1 - r0 + ROWS - 1) / ROWS, nstep = nit * npass;
    if (npass <= 0) return;
    // LDS: partial sums of two passes | scales of two steps | activations
    float * red = (float *) smem;
    uint8_t * scl = smem + 2 * KW * R * NG * 512;
    uint8_t * act = scl + 2 * ROWS * SC::PITCH;
    const ASrc as = source_a<TYPE, NG>(p, nb, lr, kg);
    WSrc ws;
    ws.nb = nb;
    const uint32_t stride = (uint32_t) pm_rows_stride<TYPE>(nb);
    ws.base = job.W + (long) r0 * stride;
    const int lim = r1 - r0 - 1;
    Tile<TYPE> W[D][R];
    ASet<TYPE> A[NG];
    Off off[R];
    const uint32_t px = TYPE == PM_Q5_K ? 0 : 16u * (uint32_t) piece_of(kg, lr >> 3), py = 16u * (uint32_t) piece_of(kg, 1 - (lr >> 3));
    // the step whose weights are asked for next (behind the last one: the slice's first row, sixteen times)
    struct { int pass, it; } wn = {0, 0};
    auto rows_of = [&](int pass) __attribute__((always_inline)) {
        const uint32_t keep = pass < npass ? ~0u : 0u;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int at = ROWS * pass + 16 * r + (TYPE == PM_Q5_K ? lr : lr & 7);
            off[r].x = (((uint32_t) min(at, lim) * stride) & keep) + px;
            off[r].y = (((uint32_t) min(at + 8, lim) * stride) & keep) + py;
        }
    };
    auto advance = [&]() __attribute__((always_inline)) { if (++wn.it == nit) { wn.it = 0; rows_of(++wn.pass); } };
    // scales: element e = tid, tid + NT, .. of the step
    constexpr int NE = SC::PER_ROW ? (ROWS * SC::PER_ROW + NT - 1) / NT : 1;
    SC sc[NE];
    auto load_scales = [&](int pass, int it) __attribute__((always_inline)) {
        if constexpr (SC::PER_ROW) {
#pragma unroll
            for (int i = 0; i < NE; ++i) {
                const int el = tid + i * NT, row = el / SC::PER_ROW, j = el % SC::PER_ROW;
                sc[i].load(ws, (uint32_t) min(ROWS * pass + row, lim) * stride, it, j);
            }
        }
    };
    auto store_scales = [&](int buf) __attribute__((always_inline)) {
        if constexpr (SC::PER_ROW) {
#pragma unroll
            for (int i = 0; i < NE; ++i) {
                const int el = tid + i * NT, row = el / SC::PER_ROW, j = el % SC::PER_ROW;
                if (ROWS * SC::PER_ROW % NT == 0 || row < ROWS) sc[i].store(scl + buf * (ROWS * SC::PITCH), row, j);
            }
        }
    };
    // a thread's element of a pass' results: row 16 rg + rr, token t; what the end of the pass adds is asked for behind the first weights (at its use it was a round of latency on its own, in
    // the rotation's case three). No branches: rows and tokens past the end ask for the last one's, absent operands for some bytes of the matrix
    constexpr int NEL = (R * NG * 128 + NT - 1) / NT;
    struct End { float add, resid, c, sn; int seq, pos; } end[NEL];
    struct El { int rr, rg, g, t; };
    auto el_of = [&](int i) __attribute__((always_inline)) { const int x = tid + i * NT; return El{x & 15, (x >> 7) % R, (x >> 7) / R, 8 * ((x >> 7) / R) + ((x >> 4) & 7)}; };
    auto load_end = [&](int pass) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NEL; ++i) {
            const El x = el_of(i);
            End & e = end[i];
            const int lrow = min(r0 + ROWS * pass + 16 * x.rg + x.rr, r1 - 1), tt = min(x.t, p.T - 1);
            e.add = ld_g((job.bias ? job.bias : (const float *) job.W) + lrow);
            if constexpr (EPI) {
                const int dim = min(lrow % p.e_dh, p.e_nrot - 1);
                e.seq = ld_g((p.e_seq ? p.e_seq : p.e_pos) + (p.e_rows ? tt : 0)); e.seq = p.e_seq ? e.seq : 0;
                e.pos = ld_g(p.e_pos + tt * p.e_rows);
                e.c = ld_g(p.e_tab + (long) tt * p.e_nrot + (dim & ~1)); e.sn = ld_g(p.e_tab + (long) tt * p.e_nrot + (dim & ~1) + 1);
            } else e.resid = ld_g((job.resid ? job.resid : (const float *) job.W) + (long) tt * job.N + lrow);
        }
    };
    constexpr int NQ = Q80 ? 4 : 8;
    rows_of(0);
    load_scales(0, 0);
    StageA<TYPE> sa;
    if constexpr (AL) { load_stage<TYPE>(sa, p, na); __builtin_amdgcn_sched_barrier(0); }
#pragma unroll
    for (int d = 0; d < D; ++d) {
#pragma unroll
        for (int r = 0; r < R; ++r) W[d][r].load(ws, off[r], kg, wave + KW * wn.it);
        advance();
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!AL) if (d == 0) {
#pragma unroll
            for (int g = 0; g < NG; ++g) {
#pragma unroll
                for (int j = 0; j < NQ; ++j) load_q<TYPE>(A[g], as, g, g == NG - 1, wave, j);
                load_yd<TYPE>(A[g], as, g, g == NG - 1, wave, hk);
            }
        }
    }
    load_end(0);
    if constexpr (AL) { __builtin_amdgcn_sched_barrier(0); store_stage<TYPE>(act, sa, p, na); }
    store_scales(0);
    __syncthreads();
    ALane al;
    if constexpr (AL) al = lane_a<TYPE>(na, lr, kg);
    int e_pos0 = 0;
    if constexpr (EPI) if (!p.e_rows) e_pos0 = p.e_pos[p.e_seq ? p.e_seq[0] : 0];      // (scalar loads)
    f32x4 out[R][NG] = {};
    int pass = 0, it = 0;
    for (int step = 0; step < nstep; ) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const bool wrap = it + 1 == nit;
            const int itn = wrap ? 0 : it + 1, next = wave + KW * itn;
            load_scales(wrap ? min(pass + 1, npass - 1) : pass, itn);
            if constexpr (AL) read_a<TYPE>(A[0], act, al, wave + KW * it, na, hk);
            __builtin_amdgcn_sched_barrier(0);
            const uint8_t * L = scl + (step & 1) * (ROWS * SC::PITCH) + lr * SC::PITCH;
            if constexpr (TYPE == PM_Q6_K) {
#pragma unroll
                for (int g = 0; g < NG; ++g)
#pragma unroll
                    for (int j = 0; j < NQ; ++j) swap16h(A[g].q[j]);
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                auto used = [&](int g, int j) __attribute__((always_inline)) {
                    if constexpr (!AL) if (r == R - 1) { __builtin_amdgcn_sched_barrier(0); load_q<TYPE>(A[g], as, g, g == NG - 1, next, j); __builtin_amdgcn_sched_barrier(0); }
                };
                if (r == 0 || ROWS * pass + 16 * r <= lim) W[d][r].mul(A, L + 16 * r * SC::PITCH, wave, kg, out[r], used);
                else {                                                 // (the last pass: no such rows)
#pragma unroll
                    for (int j = 0; j < NQ; ++j)
#pragma unroll
                        for (int g = 0; g < NG; ++g) used(g, j);
                }
                // (the sums now: sunk behind the requests below, they keep the old activations alive beside the new ones - copies at the end of the step that wait for every request)
#pragma unroll
                for (int g = 0; g < NG; ++g)
#pragma unroll
                    for (int i = 0; i < 4; ++i) { float v = out[r][g][i]; asm volatile("" : "+v"(v)); out[r][g][i] = v; }
                __builtin_amdgcn_sched_barrier(0);
                W[d][r].load(ws, off[r], kg, wave + KW * wn.it);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (!AL) {
#pragma unroll
                for (int g = 0; g < NG; ++g) load_yd<TYPE>(A[g], as, g, g == NG - 1, next, hk);
                __builtin_amdgcn_sched_barrier(0);
            }
            advance();
            if (wrap) {
                // sums over the waves and the two super-blocks of a pair, in a fixed order: the latter here, 32 lanes of either
                float * buf = red + (pass & 1) * (KW * R * NG * 128);
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int g = 0; g < NG; ++g) {
                        f32x4 s;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float o = out[r][g][i];
                            const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, o), __builtin_bit_cast(uint32_t, o), false, false));
                            const uint32_t lo = v[0], hi = v[1];               // (a bit cast of a vector's element takes element 0 here)
                            s[i] = __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
                        }
                        if (lane < 32) *(f32x4 *) (buf + (((wave * NG + g) * R + r) * 32 + lane) * 4) = s;
                        out[r][g] = f32x4{0, 0, 0, 0};
                    }
            }
            store_scales((step + 1) & 1);
            __syncthreads();
            if (wrap) {
                const float * buf = red + (pass & 1) * (KW * R * NG * 128);
#pragma unroll
                for (int i = 0; i < NEL; ++i) {
                    if (R * NG * 128 % NT != 0 && tid + i * NT >= R * NG * 128) continue;
                    const El x = el_of(i);
                    const End & e = end[i];
                    float s = 0.0f;
#pragma unroll
                    for (int k = 0; k < KW; ++k) s += buf[(((k * NG + x.g) * R + x.rg) * 32 + 16 * ((x.t >> 2) & 1) + x.rr) * 4 + (x.t & 3)];
                    const int lrow = r0 + ROWS * pass + 16 * x.rg + x.rr;
                    const bool live = x.t < p.T && lrow < r1;
                    if (job.bias) s += e.add;
                    if constexpr (EPI) {
                        const float sp = __shfl_xor(s, 1);                  // the pair's other row: the neighbouring lane, same token
                        if (live) {
                            const long kv = (long) e.seq * p.e_seq_stride;
                            const int pos = p.e_rows ? e.pos : e_pos0 + x.t;
                            if (ji == 2) p.e_vc[kv + (long) lrow * p.e_nctx + pos] = f2h(s);
                            else {
                                const int dim = lrow % p.e_dh;
                                float v = s;
                                if (dim < p.e_nrot) v = (dim & 1) ? sp * e.sn + s * e.c : s * e.c - sp * e.sn;
                                const uint16_t hv = f2h(v);
                                if (ji == 1) p.e_kc[kv + (long) pos * p.e_kvdim + lrow] = hv;
                                else st_g(job.y + (long) x.t * job.N + lrow, h2f(hv));
                            }
                        }
                    } else if (live) st_g(job.y + (long) x.t * job.N + lrow, job.resid ? s + e.resid : s);
                }
                if (pass + 1 < npass) load_end(pass + 1);
                ++pass;
            }
            it = itn;
            if (++step >= nstep) break;
        }
    }
}

// TA: the type of all jobs but the last, TB: of the last one. What the first loads need leads the arguments and is in registers when the kernel starts (pm_rows_args)
template <int TA, int TB, int NG, int R, int D, bool AL, bool EPI>
__global__ __launch_bounds__(NT, 2) void mmq_rows_kernel(const uint8_t * W0, const uint8_t * W1, const uint8_t * W2, const uint8_t * qT, uint32_t first, uint32_t rows0, uint32_t rows1, uint32_t rows2, int K,
                                                         uint32_t tokens, RowsP args) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const RowsStart s = pm_rows_start(W0, W1, W2, first, rows0, rows1, rows2, (int) blockIdx.x);
    RowsP p = args;
    pm_rows_take(p, qT, K, tokens);
    RowsJob job = args.job[s.ji];
    job.W = s.W; job.each = s.each; job.more = s.more;
    if (TA == TB || s.ji < p.njobs - 1) rows_body<TA, NG, R, D, AL, EPI>(p, job, s.w, s.ji, smem);
    else rows_body<TB, NG, R, D, AL, EPI>(p, job, s.w, s.ji, smem);
}
template <int TYPE> size_t lds_of(int NG, int R, bool AL, int K) {
    const int n = TYPE == PM_Q8_0 ? (K / 32 + 7) / 8 : K / 256;
    return (size_t) 2 * KW * R * NG * 512 + (size_t) 2 * 16 * R * Scales<TYPE>::PITCH + (AL ? ALds<TYPE>::bytes(n) : 0);
}
constexpr size_t LDS_MOST = 150 * 1024;
size_t lds_of(int type, int NG, int R, bool AL, int K) {
    return type == PM_Q4_K ? lds_of<PM_Q4_K>(NG, R, AL, K) : type == PM_Q5_K ? lds_of<PM_Q5_K>(NG, R, AL, K) : type == PM_Q6_K ? lds_of<PM_Q6_K>(NG, R, AL, K) : lds_of<PM_Q8_0>(NG, R, AL, K);
}

}  // namespace

// Where this form is the faster one, by rows per CU (groups of 16) and K. Its workgroup takes all of K at once, eight pairs of super-blocks a step: with one row group the chip is full where
// 32-row groups fill half of it, with more it pays for the steps' empty pairs (K = 2048: four of eight), for a round of sums over the waves per pass, and for a last pass of few rows (passes of 48
// rows, of 64 where the activations fit LDS). Weights out of memory, time here / time of mmq_i8.hip's kernel
// (for Q4_K and Q6_K that was the form before mmq_mid.hip's, which takes 0.91 and 0.89 of its time in the mean up to 8 tokens: divide by these to compare with what a shape not taken here gets now):
//   8 tokens, one matrix, N = 4096 / 8192 / 12288 / 16384 / 36864 / 128256: Q4_K K = 1024 0.96 1.15 1.23 1.37 1.37 1.51, 2048 0.91 1.07 1.16 1.25 1.14 1.22, 3072 0.84 0.99 1.00 1.11 0.97 0.92,
//   4096 0.82 0.94 0.94 1.03 0.89 0.87, 5120 0.87 1.13 1.09 1.21 1.07 1.05, 8192 0.86 1.02 0.93 0.98 0.88, 14336 0.92 1.12 0.99 1.24 0.95; Q6_K 1024 0.96 1.24 1.40 1.65 1.60 1.65, 4096 0.74 0.95
//   0.94 1.07 0.86 0.82, 5120 0.86 1.20 1.13 1.30 1.07, 8192 0.76 1.04 0.90 0.98 0.80, 14336 0.76 1.08 0.93 1.09 0.82; Q5_K 2048 0.89 1.07 1.19 1.36 1.29 1.32, 4096 0.75 1.01 1.03 1.07 1.00,
//   8192 0.84 1.17 1.04 1.10 0.98; Q8_0 1024 1.00 1.19 1.20 1.27 1.17, 2048 0.92 1.05 1.06 1.09 0.97 0.89, 4096 0.92 1.07 1.04 1.02 0.95, 8192 0.89 1.09 0.97 0.98 0.98
//   several matrices of one type (mmq_i8.hip looks their rows up one by one), N in all 6144 / 8192 / 16384 / 28672: Q4_K 2048 0.99 0.98 1.12 1.12, 3072 0.89 0.90 1.02 0.94, 4096 0.87 0.87 0.94
//   0.88, 5120 1.01 1.02 1.13 1.04, 8192 0.96 0.96 0.94 0.88; Q6_K 4096 0.84 0.88 1.00 0.89; two types, 6144 / 10240 / 16384: 2048 0.95 1.11 1.16, 3072 0.84 0.98 1.00, 5120 0.99 1.06 1.14, 8192
//   0.91 0.93 0.88
//   12 / 20 tokens, one row group: Q4_K K = 1024 1.05 1.07, 2048 1.02 1.02, 3072 0.89 0.88, 8192 0.90 0.88; Q6_K 1024 1.05 1.06, 2048 0.98 0.96, 4096 0.79 0.75; Q5_K 1024 0.96 0.69, 4096 0.83 0.55
//   (32 tokens 0.62); Q8_0 1024 1.09 0.76, 4096 1.01 0.67 (32: 0.71), 8192 0.98 0.64. Q4_K and Q6_K stop at 24 tokens: with four groups of them registers spill
//   20 tokens, more rows (Q5_K and Q8_0, which mmq_i8.hip takes 16 tokens at a time): N = 8192 / 16384 / 49152 Q5_K 1024 0.84 1.02 1.31, 2048 0.84 1.04 1.07, 3072 0.71 0.84 0.79, 8192 0.73 0.78 0.74; Q8_0
//   512 0.95 1.11 1.27, 1024 0.90 0.94 0.93, 4096 0.81 0.80 0.78. (32 tokens there spill)
bool pm_mmq_rows_takes(int type, long N, int K, int T, int form) {
    const int cus = pm_device_cus();
    const long rows = (N + cus - 1) / cus, groups = (rows + 15) / 16;
    const bool q5 = type == PM_Q5_K, q8 = type == PM_Q8_0;
    if (T > 8) {
        if (form != PM_ROWS_ONE || T > (q5 || q8 ? 32 : 24)) return false;
        if (groups == 1) return q5 || (q8 && T > 16) || K >= (q8 ? 7168 : type == PM_Q6_K ? 2048 : 3072);
        return (q5 || q8) && T > 16 && T <= 24 && (groups == 2 || K >= (q5 ? 3072 : 1024));
    }
    if (groups == 1) return !q8 || K >= 1024;
    if (q5) return groups == 2 && K >= 3072 && K <= 4096;
    const int pairs = (K + (q8 ? 255 : 511)) / (q8 ? 256 : 512), steps = (pairs + 7) / 8;
    const bool lds = groups > 3 && lds_of(type, 1, 4, true, K) <= LDS_MOST;         // passes of 64 rows
    // rows of the passes that are there, per cent
    const long filled = groups <= 3 ? 100 : lds ? 100 * rows / (64 * ((rows + 63) / 64)) : 100 * rows / (48 * ((rows + 47) / 48));
    if (q8) return filled >= (lds ? 70 : 80) && ((groups >= 3 && K >= 5120) || (groups >= 9 && K >= 1536));
    if (pairs == 6) return groups <= (form == PM_ROWS_ONE && type == PM_Q6_K ? 2 : 3) || (form == PM_ROWS_ONE ? groups >= 9 : form == PM_ROWS_SEVERAL && groups >= 7);
    if (form == PM_ROWS_MIXED) return pairs == 8 * steps || (pairs >= 7 * steps && K <= 9216) || (rows <= 24 && pairs >= 4);
    // (at least 7 of 8 pairs; Q4_K whose activations do not fit LDS 9 of 10)
    if ((!lds && filled < (type == PM_Q6_K ? 75 : 80)) || 10 * pairs < (type == PM_Q4_K && K > 9216 ? 72 : 70) * steps) return false;
    if (form == PM_ROWS_ONE && groups == 2) return K <= 4096 || (type == PM_Q6_K && K > 16384);
    return form != PM_ROWS_ONE || groups != 4 || K >= 8192;
}

int pm_launch_mmq_rows(RowsP p, const int * types, hipStream_t st) {
    const int cus = pm_device_cus(), n = p.njobs;
    const int ta = types[0], tb = types[n - 1];
    double bytes[3], all = 0;
    for (int j = 0; j < n; ++j) all += bytes[j] = (double) p.job[j].N * pm_weight_row_stride(types[j], p.K);
    // workgroups by weight bytes, of at least 16 rows each
    int at = 0, big = 0, first[3] = {0, INT32_MAX, INT32_MAX};
    for (int j = 0; j < n; ++j) {
        RowsJob & b = p.job[j];
        const int most = (b.N + 15) / 16;
        int want = j == n - 1 && n > 1 ? cus - at : (int) (cus * bytes[j] / all + 0.5);
        if (want > cus - at - (n - 1 - j)) want = cus - at - (n - 1 - j);
        const int nw = want < 1 ? 1 : want > most ? most : want;
        first[j] = at; at += nw;
        const int unit = p.e_on ? 2 : 1;                               // (N is even then)
        b.each = b.N / unit / nw; b.more = b.N / unit % nw;
        const int groups = (unit * (b.each + (b.more != 0)) + 15) / 16;
        if (groups > big) big = groups;
    }
    if (!pm_rows_fit(p)) return -5;
    // up to 48 rows a workgroup: one pass, activations by the wave that multiplies them; more: passes of 64 rows over activations in LDS where they fit (K up to 9 k: two thirds of it), else
    // again passes of 48
    const auto lds = [&](int g, int r, bool al) { return std::max(lds_of(ta, g, r, al, p.K), lds_of(tb, g, r, al, p.K)); };
    const int ng = (p.T + 7) / 8;
    const bool al = ng == 1 && big > 3 && lds(1, 4, true) <= LDS_MOST, deep = p.K > 4096;
    auto go = [&](auto kern, size_t bytes) {
        pm_allow_big_lds((const void *) kern, bytes);
        const RowsArgs a = pm_rows_args(p, first[1], first[2]);
        hipLaunchKernelGGL(kern, dim3(at), dim3(NT), bytes, st, p.job[0].W, p.job[1].W, p.job[2].W, p.qT, a.first, a.rows[0], a.rows[1], a.rows[2], p.K, a.tokens, p);
        return 0;
    };
#define PM_ROWS_GO(TA_, TB_, G_, R_, D_, AL_, E_) go(mmq_rows_kernel<TA_, TB_, G_, R_, D_, AL_, E_>, lds(G_, R_, AL_))
#define PM_ROWS_R(TA_, TB_, E_) { if (al) return PM_ROWS_GO(TA_, TB_, 1, 4, 1, true, E_); \
                                  switch (big) { case 1: return deep ? PM_ROWS_GO(TA_, TB_, 1, 1, 2, false, E_) : PM_ROWS_GO(TA_, TB_, 1, 1, 1, false, E_); \
                                                 case 2: return deep ? PM_ROWS_GO(TA_, TB_, 1, 2, 2, false, E_) : PM_ROWS_GO(TA_, TB_, 1, 2, 1, false, E_); \
                                                 default: return PM_ROWS_GO(TA_, TB_, 1, 3, 1, false, E_); } }
#define PM_ROWS_G(T_, G_, R_) go(mmq_rows_kernel<T_, T_, G_, R_, 1, false, false>, lds(G_, R_, false))
    if (ng > 1) {
        if (n > 1 || !pm_mmq_rows_takes(ta, p.job[0].N, p.K, p.T)) return -5;
        if (big > 1) return ta == PM_Q5_K ? PM_ROWS_G(PM_Q5_K, 3, 2) : PM_ROWS_G(PM_Q8_0, 3, 2);
        if (ta == PM_Q4_K) return ng == 2 ? PM_ROWS_G(PM_Q4_K, 2, 1) : PM_ROWS_G(PM_Q4_K, 3, 1);
        if (ta == PM_Q6_K) return ng == 2 ? PM_ROWS_G(PM_Q6_K, 2, 1) : PM_ROWS_G(PM_Q6_K, 3, 1);
        if (ta == PM_Q5_K) return ng == 2 ? PM_ROWS_G(PM_Q5_K, 2, 1) : ng == 3 ? PM_ROWS_G(PM_Q5_K, 3, 1) : PM_ROWS_G(PM_Q5_K, 4, 1);
        return ng == 2 ? PM_ROWS_G(PM_Q8_0, 2, 1) : ng == 3 ? PM_ROWS_G(PM_Q8_0, 3, 1) : PM_ROWS_G(PM_Q8_0, 4, 1);
    }
    if (p.e_on) {
        if (ta == PM_Q4_K && tb == PM_Q4_K) PM_ROWS_R(PM_Q4_K, PM_Q4_K, true)
        if (ta == PM_Q6_K && tb == PM_Q6_K) PM_ROWS_R(PM_Q6_K, PM_Q6_K, true)
        if (ta == PM_Q4_K && tb == PM_Q6_K) PM_ROWS_R(PM_Q4_K, PM_Q6_K, true)
        if (ta == PM_Q4_K && tb == PM_Q5_K) PM_ROWS_R(PM_Q4_K, PM_Q5_K, true)
        return -5;
    }
    if (ta == PM_Q4_K && tb == PM_Q4_K) PM_ROWS_R(PM_Q4_K, PM_Q4_K, false)
    if (ta == PM_Q6_K && tb == PM_Q6_K) PM_ROWS_R(PM_Q6_K, PM_Q6_K, false)
    if (ta == PM_Q5_K && tb == PM_Q5_K) {                             // (up to two groups)
        if (big > 2) return -5;
        return big == 2 ? PM_ROWS_GO(PM_Q5_K, PM_Q5_K, 1, 2, 1, false, false) : deep ? PM_ROWS_GO(PM_Q5_K, PM_Q5_K, 1, 1, 2, false, false) : PM_ROWS_GO(PM_Q5_K, PM_Q5_K, 1, 1, 1, false, false);
    }
    if (ta == PM_Q8_0 && tb == PM_Q8_0) PM_ROWS_R(PM_Q8_0, PM_Q8_0, false)
    if (ta == PM_Q4_K && tb == PM_Q6_K) PM_ROWS_R(PM_Q4_K, PM_Q6_K, false)
    if (ta == PM_Q4_K && tb == PM_Q5_K) PM_ROWS_R(PM_Q4_K, PM_Q5_K, false)
#undef PM_ROWS_R
#undef PM_ROWS_G
#undef PM_ROWS_GO
    return -5;
}
