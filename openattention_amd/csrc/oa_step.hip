// One decode step, or one group of question rows, as a single call: the stages of the deployed step
// (ours_graph.py:290-347) launched in order on one stream.
//
// Question rows (the reference's estimator over a question chunk, multibin.py:2875-2970): row i of a
// group attends the n + i keys before it, so its cluster statistics are those of all n_keys keys with
// the keys n_keys - 1, ..., n + i taken back, in that order (index_downdate's fp32 terms).
// rows_stats_kernel writes every row's statistics at once, and the 2^qsh rows of every sequence then
// run through each stage as one launch.  One row of one sequence holds 32 of the 256 compute units
// for a chain of five launches: 64 of them one after the other took 64 x 78 us of device time, and take
// 0.4 ms in two groups of 32.
#include "oa_common.h"
#include "oa_rows.h"

namespace {

constexpr int kMaxQsh = 10;

// (the statistics are aligned as floats, K and V as bf16)
typedef float floatx2a4 __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t __attribute__((aligned(2))) uint32a2;

struct StatsArgs {
  const uint16_t* K; const uint16_t* V; long kv_sb; long kv_ss;
  const int32_t* asg; long asg_stride;
  const float* nb; const float* Sk; const float* Sk2; const float* Sv;
  float* rnb; float* rSk; float* rSk2; float* rSv;
  const int* n_dev; int C; int qsh; int later;
};

// One wave per (query-head row of the index, cluster): the cluster's statistics walk back from those
// given (of all keys, or of an earlier group's first row) to the group's first row, lane l holding dims 2 l, 2 l + 1, and are written out at every row of
// the group.  Bound by the writes (1540 bytes per row and cluster).
__global__ void __launch_bounds__(256) rows_stats_kernel(StatsArgs a) {
  const int r = blockIdx.y;
  const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (c >= a.C) return;
  const int kv = r >> 2, nq = 1 << a.qsh;
  const int n0 = *a.n_dev;                          // keys of the group's first row
  const uint16_t* kb = a.K + (long)kv * a.kv_sb + 2 * lane;
  const uint16_t* vb = a.V + (long)kv * a.kv_sb + 2 * lane;
  const int32_t* ar = a.asg + (long)r * a.asg_stride;
  const long sb = ((long)r * a.C + c) * OA_D + 2 * lane;
  floatx2a4 sk = *reinterpret_cast<const floatx2a4*>(a.Sk + sb);
  floatx2a4 s2 = *reinterpret_cast<const floatx2a4*>(a.Sk2 + sb);
  floatx2a4 sv = *reinterpret_cast<const floatx2a4*>(a.Sv + sb);
  float nb = a.nb[(long)r * a.C + c];
  const int top = nq - 1 + a.later;                 // keys above the first row's
  // 64 cluster ids at a time, lane l holding that of key n0 + base + l
  for (int base = top & ~63; base >= 0; base -= 64) {
    const int mine = base + lane < top ? ar[n0 + base + lane] : -1;
    for (int j = min(63, top - base); j >= 0; --j) {
      const int i = base + j;                       // statistics of keys [0, n0 + i)
      if (i < nq) {
        const long v = (((((long)kv << a.qsh) + i) << 2) | (r & 3)) * a.C + c;
        const long o = v * OA_D + 2 * lane;
        *reinterpret_cast<floatx2a4*>(a.rSk + o) = sk;
        *reinterpret_cast<floatx2a4*>(a.rSk2 + o) = s2;
        *reinterpret_cast<floatx2a4*>(a.rSv + o) = sv;
        if (lane == 0) a.rnb[v] = nb;
      }
      // the key before leaves on the way to row i - 1 (at j = 0 it is the next 64's last)
      if (i == 0) break;
      const int id = j > 0 ? __builtin_amdgcn_readlane(mine, j - 1) : ar[n0 + i - 1];
      if (id == c) {
        const uint32_t kw = *reinterpret_cast<const uint32a2*>(kb + (long)(n0 + i - 1) * a.kv_ss);
        const uint32_t vw = *reinterpret_cast<const uint32a2*>(vb + (long)(n0 + i - 1) * a.kv_ss);
        const float k0 = __uint_as_float(kw << 16), k1 = __uint_as_float(kw & 0xffff0000u);
        sk.x = sk.x - k0; sk.y = sk.y - k1;
        s2.x = s2.x - k0 * k0; s2.y = s2.y - k1 * k1;
        sv.x = sv.x - __uint_as_float(vw << 16);
        sv.y = sv.y - __uint_as_float(vw & 0xffff0000u);
        nb = nb - 1.0f;
      }
    }
  }
}

}  // namespace

extern "C" int oa_step(const oa_step_args* p, void* stream) {
  if (!p) return OA_EINVAL;
  const oa_step_args& a = *p;
  const int qsh = a.qshift;
  if (a.head_dim != OA_D || a.kv_rows <= 0 || qsh < 0 || qsh > kMaxQsh || a.later < 0 ||
      a.rows != (a.kv_rows << qsh) * 4 || a.C <= 0 || a.C > 256 || a.Lmax <= 0 || !a.q || !a.K || !a.V ||
      !a.codes || !a.U || !a.scale || !a.asg || !a.asg8 || !a.nb || !a.Sk || !a.Sk2 || !a.Sv || !a.limbs ||
      !a.fexp || !a.TM || !a.n_dev || a.q_stride % 8 || (a.update && (qsh || a.later)))
    return OA_EINVAL;
  const bool rowed = qsh > 0 || a.later > 0;
  if (rowed && (!a.rnb || !a.rSk || !a.rSk2 || !a.rSv || a.kv_stride_b % 2 || a.kv_stride_s % 2))
    return OA_EINVAL;
  int st;
  if (a.update) {
    st = oa_index_prep(a.K, a.V, a.kv_stride_b, a.kv_stride_s, a.rows, a.kv_rows, a.head_dim, a.codes, a.Lmax,
                       32, a.U, a.scale, a.W, a.colmean, 16, a.cent, a.C, a.asg, a.asg_stride, a.asg8,
                       a.asg8_stride, a.nb, a.Sk, a.Sk2, a.Sv, a.reclist, a.reccnt, a.rmax, a.n_dev, a.q,
                       a.q_stride, a.limbs, a.fexp, stream);
  } else {
    if (rowed) {
      StatsArgs s;
      s.K = (const uint16_t*)a.K; s.V = (const uint16_t*)a.V; s.kv_sb = a.kv_stride_b; s.kv_ss = a.kv_stride_s;
      s.asg = a.asg; s.asg_stride = a.asg_stride;
      s.nb = a.nb; s.Sk = a.Sk; s.Sk2 = a.Sk2; s.Sv = a.Sv;
      s.rnb = a.rnb; s.rSk = a.rSk; s.rSk2 = a.rSk2; s.rSv = a.rSv;
      s.n_dev = a.n_dev; s.C = a.C; s.qsh = qsh; s.later = a.later;
      hipLaunchKernelGGL(rows_stats_kernel, dim3((a.C + 3) / 4, a.kv_rows * 4), dim3(256), 0,
                         (hipStream_t)stream, s);
      st = OA_LAUNCH_STATUS();
      if (st) return st;
    }
    st = oa_rows::qgs_prep(a.q, a.q_stride, a.U, a.scale, a.kv_rows, a.limbs, a.fexp, qsh, stream);
  }
  if (st) return st;
  const float* nb = rowed ? a.rnb : a.nb;
  const float* Sk = rowed ? a.rSk : a.Sk;
  const float* Sk2 = rowed ? a.rSk2 : a.Sk2;
  const float* Sv = rowed ? a.rSv : a.Sv;
  st = oa_rows::scan_heads(a.codes, a.kv_rows, a.Lmax, a.limbs, a.fexp, a.H, a.h_stride, a.TM, a.tm_stride,
                           a.TMn, a.n_dev, a.ns, a.nl, qsh, stream);
  if (st) return st;
  st = oa_rows::topk_gate_fill(a.H, a.h_stride, a.TM, a.tm_stride, a.ntiles, a.n_dev, a.ns, a.nl, a.k_top,
                               a.codes, a.Lmax, a.limbs, a.fexp, a.q, a.q_stride, a.K, a.kv_stride_b,
                               a.kv_stride_s, a.rows, a.kv_rows, a.head_dim, a.asg, a.asg_stride, a.sel,
                               a.sel_stride, Sk, Sk2, nb, a.C, a.sm_scale, a.sm_scale_sq, a.budget, a.score, a.n_t,
                               a.quota, a.qsk, qsh, stream);
  if (st) return st;
  st = oa_rows::topq_heads(a.H, a.h_stride, a.asg8, a.asg8_stride, a.quota, a.rows, a.C, a.Lmax, a.exp_idx,
                           a.E, a.n_dev, a.codes, a.kv_rows, a.limbs, a.fexp, a.S32, a.s32_stride,
                           a.TMn ? a.TM : nullptr, a.TMn, a.TMn ? a.tm_stride : 0, 0, qsh, stream);
  if (st) return st;
  return oa_rows::residual_flash(a.q, a.q_stride, a.K, a.V, a.kv_stride_b, a.kv_stride_s, a.rows, a.kv_rows,
                                 a.asg, a.asg_stride, a.sel, a.sel_stride, a.ns + a.nl + a.k_top, a.exp_idx,
                                 a.E, a.quota, a.n_t, Sk, Sv, a.C, a.sm_scale, a.out, a.out_stride,
                                 a.out_is_f32, a.qsk, qsh, stream);
}
