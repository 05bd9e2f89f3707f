// The decode stages' launches over question rows (2^qsh query rows per sequence; layout in
// oa_common.h), shared by the one-row entry points (qsh = 0) and oa_step.  rows = (kv_rows << qsh) * 4;
// the arguments are otherwise those of the entry points of the same names.
#pragma once
#include <stdint.h>

namespace oa_rows {

int qgs_prep(const void* q, long q_stride, const float* U, const float* scale, int kv_rows, int8_t* limbs,
             int* fexp, int qsh, void* stream);

int scan_heads(const int8_t* codes, int kv_rows, int Lmax, const int8_t* limbs, const int* fexp, uint16_t* H,
               long h_stride, float* TM, long tm_stride, float* TMn, const int* n_dev, int ns, int nl, int qsh,
               void* stream);

int topk_select_heads(uint16_t* H, long h_stride, const float* TM, long tm_stride, int rows, int ntiles,
                      int32_t* sel, long sel_stride, const int* n_dev, int ns, int nl, int k_top,
                      const int8_t* codes, int kv_rows, int Lmax, const int8_t* limbs, const int* fexp,
                      int qsh, void* stream);

int topk_gate_fill(uint16_t* H, long h_stride, const float* TM, long tm_stride, int ntiles, const int* n_dev,
                   int ns, int nl, int k_top, const int8_t* codes, int Lmax, const int8_t* limbs,
                   const int* fexp, const void* q, long q_stride, const void* K, long k_stride_b,
                   long k_stride_s, int rows, int kv_rows, int head_dim, const int32_t* asg, long asg_stride,
                   int32_t* sel, long sel_stride, const float* Sk, const float* Sk2, const float* nb, int C,
                   float sm_scale, float sm_scale_sq, int budget, float* score, float* n_t, float* quota,
                   float* qsk, int qsh, void* stream);

int topq_heads(const uint16_t* H, long h_stride, const uint8_t* asg8, long asg8_stride, const float* quota,
               int rows, int C, int Lmax, int32_t* exp_idx, int E, const int* n_dev, const int8_t* codes,
               int kv_rows, const int8_t* limbs, const int* fexp, float* S32, long s32_stride, const float* TM,
               const float* TMn, long tm_stride, int path, int qsh, void* stream);

int residual_flash(const void* q, long q_stride, const void* K, const void* V, long kv_stride_b,
                   long kv_stride_s, int rows, int kv_rows, const int32_t* asg, long asg_stride,
                   const int32_t* sel, long sel_stride, int n_sel, const int32_t* exp_idx, int E,
                   const float* quota, const float* n_t, const float* Sk, const float* Sv, int C,
                   float sm_scale, void* out, long out_stride, int out_is_f32, const float* qsk, int qsh,
                   void* stream);

}  // namespace oa_rows
