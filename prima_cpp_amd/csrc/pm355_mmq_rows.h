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
