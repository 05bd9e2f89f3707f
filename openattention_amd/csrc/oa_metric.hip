// The a10 query metric of every query-head row of a build, on the device: the moment of the
// row's question rows advanced to the decode position, trace-normalised and blended with the
// (per head) rotated static metric, and each KV row's group mean (methods_eager.py:510-519;
// static_top_k.py:185-194).  For question row q_p (p over the picked rows, P of them), advanced
// by its own RoPE angle,
//   r_p = s (cos_p * q_p + sin_p * rotate_half(q_p))                     (fp64)
//   Mq  = fp32((sum_p r_p r_p^T) / P)                                    (fp64 sums over p in order)
//   M   = mst_half + 0.5 (Mq / max(tr Mq, 1e-12))                        (fp32; tr summed in order)
//   Mg  = (M_0 + M_1 + ... + M_{G-1}) / G over a KV row's G query rows   (fp32, in order)
// mst_half = 1/2 nt(the rotated static metric) is formed once per layer on the host side.
// S 256-thread workgroups per KV row, each 128 / S rows of the matrices: the picked rows of one query
// row at a time in LDS (fp64), each thread a TR x TC block of the slice's moment, and the whole
// diagonal (for the trace) formed in every slice.  One KV row's four heads are a serial chain of
// loads and fp64 products (150 us with one workgroup), so that few KV rows take eight slices, which
// repeat the rotation of the question rows but not the products: 8 or 16 KV rows 150 -> 42 us,
// 256 KV rows 167 -> 104 us.
#include "oa_common.h"

namespace {

constexpr int kN = 128;
constexpr int kMaxP = 64;
constexpr int kThreads = 256;

template <bool BF16>
__device__ __forceinline__ double q_at(const void* q, long idx) {
  if (BF16) return (double)oa::bf16_to_f32(static_cast<const uint16_t*>(q)[idx]);
  return (double)static_cast<const float*>(q)[idx];
}

template <bool BF16, int S>
__global__ __launch_bounds__(kThreads) void query_metric_kernel(
    const void* __restrict__ q, long q_sr, long q_sp, int G, const int* __restrict__ pick, int P,
    const double* __restrict__ cosv, const double* __restrict__ sinv, double scaling,
    const float* __restrict__ mst_half, int heads, float* __restrict__ gm_out,
    float* __restrict__ m_out) {
  constexpr int TC = S <= 2 ? 8 : 4, kColT = kN / TC;         // columns per thread, column threads
  constexpr int TR = kN / S / (kThreads / kColT);             // rows per thread
  __shared__ __align__(16) double s_r[kMaxP * kN];
  __shared__ float s_diag[kN];
  __shared__ float s_tr;
  const int kvr = blockIdx.x;
  const int t = threadIdx.x;
  const int i0 = blockIdx.y * (kN / S) + (t / kColT) * TR, j0 = (t % kColT) * TC;
  float gm[TR][TC];
  for (int h = 0; h < G; ++h) {
    const int row = kvr * G + h;
    if (h) __syncthreads();             // the previous row's reads of s_r and s_tr are done
    // dims d and d + 64 of a picked row together: each is the other's rotated half
#pragma unroll 4
    for (int e = t; e < P * (kN / 2); e += kThreads) {
      const int p = e / (kN / 2), d = e % (kN / 2);
      const long base = (long)row * q_sr + (long)pick[p] * q_sp;
      const double x = q_at<BF16>(q, base + d), y = q_at<BF16>(q, base + d + kN / 2);
      const double c0 = cosv[p * kN + d] * x, s0 = sinv[p * kN + d] * -y;
      const double c1 = cosv[p * kN + d + kN / 2] * y, s1 = sinv[p * kN + d + kN / 2] * x;
      s_r[p * kN + d] = scaling * (c0 + s0);
      s_r[p * kN + d + kN / 2] = scaling * (c1 + s1);
    }
    __syncthreads();
    if (t < kN) {                       // the diagonal's own sums (the same chains as the blocks')
      double acc = 0.0;
#pragma unroll 8
      for (int p = 0; p < P; ++p) acc = fma(s_r[p * kN + t], s_r[p * kN + t], acc);
      s_diag[t] = (float)(acc / (double)P);
    }
    double acc[TR][TC];
#pragma unroll
    for (int a = 0; a < TR; ++a)
#pragma unroll
      for (int b = 0; b < TC; ++b) acc[a][b] = 0.0;
#pragma unroll 2
    for (int p = 0; p < P; ++p) {
      double ra[TR], rb[TC];
#pragma unroll
      for (int k = 0; k < TR; k += 2) {
        const double2 x = *reinterpret_cast<const double2*>(&s_r[p * kN + i0 + k]);
        ra[k] = x.x; ra[k + 1] = x.y;
      }
#pragma unroll
      for (int k = 0; k < TC; k += 2) {
        const double2 y = *reinterpret_cast<const double2*>(&s_r[p * kN + j0 + k]);
        rb[k] = y.x; rb[k + 1] = y.y;
      }
#pragma unroll
      for (int a = 0; a < TR; ++a)
#pragma unroll
        for (int b = 0; b < TC; ++b) acc[a][b] = fma(ra[a], rb[b], acc[a][b]);
    }
    __syncthreads();
    if (t == 0) {
      float tr = 0.f;
#pragma unroll 16
      for (int i = 0; i < kN; ++i) tr = tr + s_diag[i];
      s_tr = fmaxf(tr, 1e-12f);
    }
    __syncthreads();
    const float tr = s_tr;
    const float* ms = mst_half + (long)(row % heads) * kN * kN;
    float* mo = m_out + (long)row * kN * kN;
#pragma unroll
    for (int a = 0; a < TR; ++a) {
      float v[TC];
#pragma unroll
      for (int b = 0; b < TC; ++b) {
        const float mq = (float)(acc[a][b] / (double)P);
        v[b] = ms[(i0 + a) * kN + j0 + b] + 0.5f * (mq / tr);
        gm[a][b] = h ? gm[a][b] + v[b] : v[b];
      }
#pragma unroll
      for (int b = 0; b < TC; b += 4)
        *reinterpret_cast<float4*>(mo + (i0 + a) * kN + j0 + b) = make_float4(v[b], v[b + 1], v[b + 2], v[b + 3]);
    }
  }
  float* go = gm_out + (long)kvr * kN * kN;
#pragma unroll
  for (int a = 0; a < TR; ++a)
#pragma unroll
    for (int b = 0; b < TC; b += 4)
      *reinterpret_cast<float4*>(go + (i0 + a) * kN + j0 + b) =
          make_float4(gm[a][b] / (float)G, gm[a][b + 1] / (float)G, gm[a][b + 2] / (float)G, gm[a][b + 3] / (float)G);
}

}  // namespace

extern "C" int oa_query_metric(const void* q, int q_bf16, long q_stride_row, long q_stride_pos, int rows,
                               int G, const int32_t* pick, int P, const double* cosv, const double* sinv,
                               double scaling, const float* mst_half, int heads, float* gm_out,
                               float* m_out, void* stream) {
  if (rows <= 0 || G <= 0 || G > 8 || rows % G || P < 1 || P > kMaxP || heads <= 0 || !q || !pick ||
      !cosv || !sinv || !mst_half || !gm_out || !m_out || q_stride_pos < kN ||
      (reinterpret_cast<uintptr_t>(gm_out) & 15) || (reinterpret_cast<uintptr_t>(m_out) & 15))
    return OA_EINVAL;
  const int kv_rows = rows / G;
  // slices: eight while they are at most two workgroups per compute unit (64 KB of LDS each), else
  // the most that are
  auto launch = [&](auto kernel, int slices) {
    hipLaunchKernelGGL(kernel, dim3(kv_rows, slices), dim3(kThreads), 0, (hipStream_t)stream, q, q_stride_row,
                       q_stride_pos, G, pick, P, cosv, sinv, scaling, mst_half, heads, gm_out, m_out);
  };
#define OA_METRIC(S) q_bf16 ? launch(query_metric_kernel<true, S>, S) : launch(query_metric_kernel<false, S>, S)
  if (kv_rows <= 64) OA_METRIC(8);
  else if (kv_rows <= 128) OA_METRIC(4);
  else if (kv_rows <= 256) OA_METRIC(2);
  else OA_METRIC(1);
#undef OA_METRIC
  return OA_LAUNCH_STATUS();
}
