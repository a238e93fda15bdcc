// pm355_mmq_rows.h - launches of the quantized mat-mul of few tokens (mmq_rows.hip, mmq_mid.hip) on activation tables that are already written
#pragma once
#include "pm355_device.h"
#include "pm355_kernels.h"

struct RowsJob { const uint8_t * W; float * y; const float * bias, * resid; int N, each, more; };      // each, more: rows of its workgroups (filled in by the launch)
struct RowsP {
    RowsJob job[3]; int njobs, K, T, t_off;                        // t_off: first slot of these tokens in the tables' 32
    // K-quants: values in operand order [nsb][8][64][16], F16 group sums [nsb][64][8], scales [nsb][32]; Q8_0: values [nb][64][16], scales [nb][32] (pm_q8k_tables, mmq_i8.hip)
    const uint8_t * qT, * bsT; const float * dT;
    // the jobs are wq, wk, wv: NORM rope and the KV store in the epilogue (pm_qkv_epi)
    int e_on; const float * e_tab; const int32_t * e_pos, * e_seq; long e_seq_stride; uint16_t * e_kc, * e_vc; int e_dh, e_nctx, e_nrot, e_kvdim, e_rows;
};
// What a launch's first loads need travels as leading arguments of 14 dwords, which the hardware places in registers before a wave starts; read from memory with the rest they stood in front of every
// first load. us per launch at 8 tokens, before / now: 8B shape wq | wk | wv 7.9 / 7.0 (with a Q6_K wv 10.1 / 9.0), wo 5.7 / 5.3, ffn_down 12.6 / 10.9 (Q6_K 18.0 / 16.5); 70B shape wo and ffn_down
// 16.6 / 16.3, wq | wk | wv 15.5 / 14.9. first: first workgroups of the second and third job, 16 bits each (65535: none); rows: each | more << 24; tokens: T | t_off << 8 | njobs << 16
struct RowsArgs { uint32_t first, rows[3], tokens; };
inline RowsArgs pm_rows_args(const RowsP & p, int first1, int first2) {
    RowsArgs a;
    a.first = (uint32_t) (first1 < 65535 ? first1 : 65535) | (uint32_t) (first2 < 65535 ? first2 : 65535) << 16;
    for (int j = 0; j < 3; ++j) a.rows[j] = (uint32_t) p.job[j].each | (uint32_t) p.job[j].more << 24;
    a.tokens = (uint32_t) p.T | (uint32_t) p.t_off << 8 | (uint32_t) p.njobs << 16;
    return a;
}
// (more < workgroups of the matrix, at most one per CU. A row is at least 288 bytes, 512 values of Q4_K: a workgroup's 16 M rows, 4.8 GB, beside its 255 others' would be four times the device's memory)
inline bool pm_rows_fit(const RowsP & p) {
    for (int j = 0; j < p.njobs; ++j) if (p.job[j].each >= 1 << 24 || p.job[j].more >= 1 << 8) return false;
    return true;
}
struct RowsStart { const uint8_t * W; int ji, w, each, more; };
__device__ __forceinline__ RowsStart pm_rows_start(const uint8_t * W0, const uint8_t * W1, const uint8_t * W2, uint32_t first, uint32_t rows0, uint32_t rows1, uint32_t rows2, int b) {
    const int first1 = (int) (first & 65535), first2 = (int) (first >> 16), ji = (b >= first1) + (b >= first2);
    const uint32_t rows = ji == 0 ? rows0 : ji == 1 ? rows1 : rows2;
    return RowsStart{ji == 0 ? W0 : ji == 1 ? W1 : W2, ji, b - (ji == 0 ? 0 : ji == 1 ? first1 : first2), (int) (rows & 0xFFFFFF), (int) (rows >> 24)};
}
__device__ __forceinline__ void pm_rows_take(RowsP & p, const uint8_t * qT, int K, uint32_t tokens) { p.qT = qT; p.K = K; p.T = (int) (tokens & 255); p.t_off = (int) (tokens >> 8 & 255); p.njobs = (int) (tokens >> 16); }
template <int TYPE> __device__ __forceinline__ size_t pm_rows_stride(int nb) {
    return TYPE == PM_Q4_K ? (size_t) nb * 144 : TYPE == PM_Q5_K ? (size_t) nb * 176 : TYPE == PM_Q6_K ? pm_q6k_row_stride((size_t) nb) : (size_t) nb * 32 + (((size_t) nb * 2 + 15) & ~(size_t) 15);
}
// one or several matrices of one K (types[0]; only the last may be of another type) over 1..8 tokens, one matrix over more; -5: not served
enum { PM_ROWS_ONE, PM_ROWS_SEVERAL, PM_ROWS_MIXED };               // one matrix; several of one type; two types
// whether a pass over T tokens of N rows in all is one for it (else mmq_mid.hip's kernel, or mmq_i8.hip's); type: of the first matrix
bool pm_mmq_rows_takes(int type, long N, int K, int T, int form = PM_ROWS_ONE);
int pm_launch_mmq_rows(RowsP p, const int * types, hipStream_t st);
// mmq_mid.hip: one or several matrices of one K (types[0]; only the last may be of another type) over 1..32 tokens, t_off 0; -5: not served
int pm_launch_mmq_mid(RowsP p, const int * types, hipStream_t st);
