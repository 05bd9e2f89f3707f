// Top eigenpairs of symmetric positive semi-definite 128 x 128 fp32 matrices: the a10 bases at
// prefill (U = the top-32 eigenvectors of each KV head's group-mean metric, W from the top-16
// eigenpairs of each query head's metric), which the reference obtains from torch.linalg.eigh
// (inference/methods_eager.py:519-528).
//
// Method: one-sided (Hestenes) Jacobi.  Pairs of columns (a, b) of A are rotated,
//   [a b] <- [a b] [[c, s], [-s, c]],  tan = t, t^2 + 2 zeta t - 1 = 0 (the smaller root),
//   zeta = (|b|^2 - |a|^2) / (2 a.b),
// which makes the pair orthogonal.  Repeated over every pair until each is orthogonal to a
// relative tolerance, A V = B holds with mutually orthogonal columns.  For A = Q diag(lambda) Q^T
// positive semi-definite, B = Q diag(lambda) (the columns are lambda_j q_j): the eigenvalues are
// the column norms and the eigenvectors the normalised columns, so V is never formed.  Only the
// lower triangle of M is read (torch.linalg.eigh's default).
//
// Schedule: 64 lanes hold 64 column pairs (a, b), one step rotates them at once.  A sweep of 127
// steps meets every two columns once, by recursive halving: at level l = 0..6 the columns form 2^l
// blocks, each split into halves H0 | H1 held as (a, b) by h = 64 >> l pairs, and the block meets
// H0 x H1 in h steps, its b columns moving one pair along after each step.  Between levels the
// first h/2 pairs of a block hand their b column to pair i + h/2 for its a column, so each new
// block again holds one column of each of its halves per pair.
// Each column's squared norm travels with it (recomputed at every sweep start), so a step forms
// one dot product, a.b, per pair; a pair counts as orthogonal when |a.b| <= kTol |a| |b| or when
// both columns are below 1e-6 |A|_F (numerically in the null space, where fp32 cannot resolve
// their angle).  Sweeps repeat until one applies no rotation (at most kMaxSweeps).  Every matrix
// runs the same fixed schedule on its own workgroup: results do not depend on the batch a
// matrix is in.
//
// Layout: one workgroup per matrix, lane l of every wave pair l, each wave a share of the rows.  A
// b column moves one pair along by one cross-lane move per register (DPP; one LDS permutation at
// level 1), a trade between levels is one lane swap, and only the waves' partial dot products pass
// through LDS (one float per pair and wave, one barrier a step, two buffers in turn).  With the
// rows of a pair in one quad of lanes, whole b columns went through LDS at every step (16 16-byte
// operations per lane and two barriers).  What bounds a step is vector issue, and a lone wave
// issues only every second slot, so few matrices are split over eight waves (the even and the odd
// rows of each 32, the two halves of a dot product's fixed order) and many over four, which
// repeats the rotation angles less often.  Against quads of lanes and LDS columns, same bits: 40
// matrices 1275 -> 892 us, 1280 matrices 2975 -> 2463 us.
#include "oa_common.h"

namespace {

constexpr int kN = 128;
constexpr int kPairs = 64;
constexpr int kChunks = 4;                     // row chunks of 32, summed (c0 + c1) + (c2 + c3)
constexpr int kChunkRows = kN / kChunks;
constexpr int kOutCols = 32;                   // output columns staged at a time
constexpr int kOutStride = kN + 1;             // floats per staged output column
constexpr int kMaxSweeps = 40;
constexpr int kMaxK = 64;
constexpr float kTol = 1e-5f;                  // |a.b| <= kTol |a| |b| counts as orthogonal

// element (r, c) of the symmetric matrix from the lower triangle of row-major M
__device__ __forceinline__ float sym_at(const float* M, int r, int c) {
  return r >= c ? M[r * kN + c] : M[c * kN + r];
}

// two rows rotated in place: (a, b) <- (fma(c, a, -(s b)), fma(s, a, c b)).  Written out so that the
// results stay in the rows' own registers: the compiler's order kept 32 products beside the 64 row
// values and then copied the rows back (34 moves a step).
__device__ __forceinline__ void rotate2(float& a0, float& b0, float& a1, float& b1, float c, float s) {
  float t0, t1, u0, u1;
  asm("v_mul_f32 %4, %9, %1\n\tv_mul_f32 %5, %9, %3\n\t"
      "v_mul_f32 %6, %8, %1\n\tv_mul_f32 %7, %8, %3\n\t"
      "v_fma_f32 %1, %9, %0, %6\n\tv_fma_f32 %3, %9, %2, %7\n\t"
      "v_fma_f32 %0, %8, %0, -%4\n\tv_fma_f32 %2, %8, %2, -%5"
      : "+v"(a0), "+v"(b0), "+v"(a1), "+v"(b1), "=&v"(t0), "=&v"(t1), "=&v"(u0), "=&v"(u1)
      : "v"(c), "v"(s));
}

// the value of the next pair (circular within H pairs; H = 32: of the interleaved order)
template <int H>
__device__ __forceinline__ float next_pair(float v, int lane) {
  if (H == 64) return oa::dpp_f32<0x134>(v);            // wave_rol:1
  if (H == 32) return oa::dpp_f32<0x134>(oa::dpp_f32<0x134>(v));
  if (H == 16) return oa::dpp_f32<0x12F>(v);            // row_ror:15
  if (H == 8) {
    const float n = oa::dpp_f32<0x12F>(v), w = oa::dpp_f32<0x127>(v);   // row_ror:7: lanes 7, 15
    return (lane & 7) == 7 ? w : n;
  }
  if (H == 4) return oa::dpp_f32<0x39>(v);              // quad_perm [1,2,3,0]
  return oa::dpp_f32<0xB1>(v);                          // quad_perm [1,0,3,2]
}

// trade between levels: pairs with bit HB clear give b for the a of pair ^ HB (HB = 16: in the
// interleaved order, where pair ^ 16 is 32 lanes away)
template <int HB>
__device__ __forceinline__ void trade(float& a, float& b, int lane) {
  if (HB == 32 || HB == 16) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
    return;
  }
  const bool low = (lane & HB) == 0;
  const float give = low ? b : a;
  const float got = HB == 8 ? oa::dpp_f32<0x128>(give)                      // row_ror:8
                    : HB == 4 ? oa::dpp_f32<0x1B>(oa::dpp_f32<0x141>(give))   // ^ 7, then ^ 3
                    : HB == 2 ? oa::dpp_f32<0x4E>(give)                       // quad_perm [2,3,0,1]
                              : oa::dpp_f32<0xB1>(give);                      // quad_perm [1,0,3,2]
  a = low ? a : got;
  b = low ? got : b;
}

// SPLIT = 1: wave w holds rows 32 w .. 32 w + 31; SPLIT = 2: rows 32 (w / 2) + 2 j + w % 2
template <int SPLIT>
struct Jacobi {
  static constexpr int kWaves = kChunks * SPLIT;
  static constexpr int kThreads = kWaves * OA_WAVE;
  static constexpr int kRows = kChunkRows / SPLIT;

  float a[kRows], b[kRows];   // this lane's rows of pair `lane`
  float al, be;               // the columns' squared norms
  float floor2;
  int lane, wave;
  float (*part)[kWaves][kPairs];   // LDS: two buffers of partial dot products
  int buf;

  // the waves' partials of one dot product, summed in the fixed order; every wave returns the sum
  __device__ __forceinline__ float join(float v) {
    part[buf][wave][lane] = v;
    __syncthreads();
    float c[kChunks];
#pragma unroll
    for (int i = 0; i < kChunks; ++i)
      c[i] = SPLIT == 2 ? part[buf][2 * i][lane] + part[buf][2 * i + 1][lane] : part[buf][i][lane];
    // a buffer is written again two joins later, past the barrier that follows these reads
    buf ^= 1;
    return (c[0] + c[1]) + (c[2] + c[3]);
  }
  // x . y over this lane's rows: the even rows' chain and the odd rows' (SPLIT = 2 holds one of them)
  __device__ __forceinline__ float dot(const float (&x)[kRows], const float (&y)[kRows]) {
    float s0 = 0.f, s1 = 0.f;
    if (SPLIT == 2) {
#pragma unroll
      for (int j = 0; j < kRows; ++j) s0 = fmaf(x[j], y[j], s0);
      return s0;
    }
#pragma unroll
    for (int j = 0; j < kRows; j += 2) {
      s0 = fmaf(x[j], y[j], s0);
      s1 = fmaf(x[j + 1], y[j + 1], s1);
    }
    return s0 + s1;
  }

  // one Jacobi rotation of every pair, whose squared norms al, be are carried along and updated as
  // al - t ga, be + t ga (the rotated pair's Gram diagonal); the lanes that were not yet orthogonal.
  // The rotation itself is skipped when no pair needs one.
  __device__ __forceinline__ unsigned long long rotate() {
    const float ga = join(dot(a, b));
    // orthogonal to the tolerance, or both columns negligible against the matrix (their norms
    // below 1e-6 |A|_F: they cannot move the leading eigenvectors)
    const bool on = ga * ga > (kTol * kTol) * (al * be) && al + be > floor2;
    const unsigned long long any = __ballot(on);
    if (any == 0ull) return 0ull;
    // the angle from the hardware reciprocal and square roots (about 1 ulp): an error there only
    // changes which orthogonal rotation is applied (c^2 + s^2 = 1 to about 2 ulp either way); for
    // ga = 0 the quotients are inf or NaN and the pair is not rotated
    const float zeta = (be - al) * __builtin_amdgcn_rcpf(2.f * ga);
    const float t = copysignf(
        __builtin_amdgcn_rcpf(fabsf(zeta) + __builtin_amdgcn_sqrtf(fmaf(zeta, zeta, 1.f))), zeta);
    const float cr = __builtin_amdgcn_rsqf(fmaf(t, t, 1.f));
    const float c = on ? cr : 1.f;
    const float s = on ? cr * t : 0.f;
    const float tg = on ? t * ga : 0.f;
    al = fmaxf(al - tg, 0.f);
    be = be + tg;
#pragma unroll
    for (int j = 0; j < kRows; j += 2) rotate2(a[j], b[j], a[j + 1], b[j + 1], c, s);
    return any;
  }

  // every lane takes the pair of lane src / 4.  Level 1 runs its two blocks of 32 pairs in alternate
  // lanes, where the next pair is two lanes away: two DPP moves, against an LDS permutation of every
  // b register at every step (570 cycles a step)
  __device__ __forceinline__ void reorder(int src) {
    auto take = [&](float& v) {
      v = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(v)));
    };
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      take(a[j]);
      take(b[j]);
    }
    take(al);
    take(be);
  }

  // level of H pairs per block (H steps), then the trade that starts the next level
  template <int H>
  __device__ __forceinline__ unsigned long long level() {
    unsigned long long any = 0;
    if (H == 32) reorder(4 * ((lane & 1) * 32 + (lane >> 1)));
#pragma unroll 1
    for (int t = 0; t < H; ++t) {
      any |= rotate();
      if (t + 1 < H) {
#pragma unroll
        for (int j = 0; j < kRows; ++j) b[j] = next_pair<H>(b[j], lane);
        be = next_pair<H>(be, lane);
      }
    }
    if (H > 1) {
#pragma unroll
      for (int j = 0; j < kRows; ++j) trade<H / 2>(a[j], b[j], lane);
      trade<H / 2>(al, be, lane);
    }
    if (H == 32) reorder(4 * (2 * (lane & 31) + (lane >> 5)));
    return any;
  }
};

template <int SPLIT>
__global__ __launch_bounds__(Jacobi<SPLIT>::kThreads, SPLIT == 2 ? 4 : 5) void sym_eig_top_kernel(
    const float* __restrict__ M, long m_stride, int k, float* __restrict__ ev, float* __restrict__ evec,
    int* __restrict__ sweeps_out) {
  typedef Jacobi<SPLIT> J;
  constexpr int kRows = J::kRows, kThreads = J::kThreads;
  // partial products; at the end the odd rows (SPLIT = 2), then the staged output columns
  constexpr int kOdd = SPLIT == 2 ? kChunks * 2 * kRows * kPairs : 0;
  __shared__ float s_part[2][J::kWaves][kPairs];
  __shared__ float s_x[kOdd > kOutCols * kOutStride ? kOdd : kOutCols * kOutStride];
  __shared__ double s_sum[2][kChunks][kPairs];   // fp64 squared norms: a columns, b columns
  const int m = blockIdx.x;
  const int tid = threadIdx.x;
  const float* A = M + (long)m * m_stride;
  J p;
  p.lane = tid & (OA_WAVE - 1);
  p.wave = __builtin_amdgcn_readfirstlane(tid / OA_WAVE);
  p.part = s_part;
  p.buf = 0;
  const int lane = p.lane;
  const int chunk = p.wave / SPLIT, r0 = chunk * kChunkRows + p.wave % SPLIT;   // rows r0 + SPLIT j
#pragma unroll
  for (int j = 0; j < kRows; ++j) {
    p.a[j] = sym_at(A, r0 + SPLIT * j, lane);
    p.b[j] = sym_at(A, r0 + SPLIT * j, lane + kPairs);
  }
  // |A|_F^2: each pair's two columns over 32 rows in order, the chunks, then 16 pairs at a time
  {
    float f = 0.f;
    if (SPLIT == 1 || p.wave < kChunks) {
#pragma unroll
      for (int j = 0; j < kChunkRows; ++j) {
        const int r = (SPLIT == 1 ? r0 : p.wave * kChunkRows) + j;
        const float x = SPLIT == 1 ? p.a[j % kRows] : sym_at(A, r, lane);
        const float y = SPLIT == 1 ? p.b[j % kRows] : sym_at(A, r, lane + kPairs);
        f = fmaf(x, x, fmaf(y, y, f));
      }
      s_part[0][p.wave][lane] = f;
    }
    __syncthreads();
    f = (s_part[0][0][lane] + s_part[0][1][lane]) + (s_part[0][2][lane] + s_part[0][3][lane]);
    f = oa::group16_sum(f);
    auto at = [&](int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), l)); };
    p.floor2 = 1e-12f * ((at(0) + at(16)) + (at(32) + at(48)));
    p.buf = 1;   // buffer 0 is read above: it is written again past the next join's barrier
  }

  int sweep = 0;
  bool more = true;
  while (more && sweep < kMaxSweeps) {
    p.al = p.join(p.dot(p.a, p.a));
    p.be = p.join(p.dot(p.b, p.b));
    unsigned long long any = p.template level<64>();
    any |= p.template level<32>();
    any |= p.template level<16>();
    any |= p.template level<8>();
    any |= p.template level<4>();
    any |= p.template level<2>();
    any |= p.template level<1>();
    ++sweep;
    more = any != 0ull;   // the same in every wave: the sums that decide are
  }

  // column norms in fp64 (slot l: pair l's a column, slot 64 + l: its b column), a chunk's rows in
  // order; the waves with the odd rows hand them to those with the even ones
  if (SPLIT == 2) {
    if (p.wave & 1) {
#pragma unroll
      for (int j = 0; j < kRows; ++j) {
        s_x[((chunk * 2 + 0) * kRows + j) * kPairs + lane] = p.a[j];
        s_x[((chunk * 2 + 1) * kRows + j) * kPairs + lane] = p.b[j];
      }
    }
    __syncthreads();
  }
  if (SPLIT == 1 || (p.wave & 1) == 0) {
    double pa = 0.0, pb = 0.0;
    // (scheduling barriers every 8 rows keep the fp64 conversions from being hoisted all at once)
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      pa = fma((double)p.a[j], (double)p.a[j], pa);
      pb = fma((double)p.b[j], (double)p.b[j], pb);
      if (SPLIT == 2) {
        const double oa_ = (double)s_x[((chunk * 2 + 0) * kRows + j) * kPairs + lane];
        const double ob = (double)s_x[((chunk * 2 + 1) * kRows + j) * kPairs + lane];
        pa = fma(oa_, oa_, pa);
        pb = fma(ob, ob, pb);
      }
      if ((j & 7) == 7) __builtin_amdgcn_sched_barrier(0);
    }
    s_sum[0][chunk][lane] = pa;
    s_sum[1][chunk][lane] = pb;
  }
  __syncthreads();
  auto norm = [&](int ab, int l) {
    return sqrt((s_sum[ab][0][l] + s_sum[ab][1][l]) + (s_sum[ab][2][l] + s_sum[ab][3][l]));
  };
  const double na = norm(0, lane), nb = norm(1, lane);
  // rank in descending norm, ties to the lower slot (every wave counts the same)
  int ra = 0, rb = 0;
#pragma unroll 1
  for (int j = 0; j < kPairs; ++j) {
    const double x = __longlong_as_double(
        ((long long)__builtin_amdgcn_readlane((int)(__double_as_longlong(na) >> 32), j) << 32) |
        (unsigned)__builtin_amdgcn_readlane((int)__double_as_longlong(na), j));
    const double y = __longlong_as_double(
        ((long long)__builtin_amdgcn_readlane((int)(__double_as_longlong(nb) >> 32), j) << 32) |
        (unsigned)__builtin_amdgcn_readlane((int)__double_as_longlong(nb), j));
    ra += (x > na) || (x == na && j < lane);
    ra += y > na;
    rb += x >= nb;
    rb += (y > nb) || (y == nb && j < lane);
  }
  const float ia = na > 0.0 ? (float)(1.0 / na) : 0.f, ib = nb > 0.0 ? (float)(1.0 / nb) : 0.f;
  if (p.wave == 0) {
    if (ra < k) ev[(long)m * k + k - 1 - ra] = (float)na;
    if (rb < k) ev[(long)m * k + k - 1 - rb] = (float)nb;
  }
  // the k largest, ascending (the largest in position k - 1), staged kOutCols output columns at a
  // time for a coalesced store; a zero column (a zero eigenvalue among the k) is stored as zeros
  float* out = evec + (long)m * kN * k;
  for (int c0 = 0; c0 < k; c0 += kOutCols) {
    const int nc = min(kOutCols, k - c0);
    auto stage = [&](const float (&v)[kRows], int rank, float inv) {
      const int c = k - 1 - rank - c0;
      if (c < 0 || c >= nc) return;
#pragma unroll
      for (int j = 0; j < kRows; ++j) s_x[c * kOutStride + r0 + SPLIT * j] = v[j] * inv;
    };
    stage(p.a, ra, ia);
    stage(p.b, rb, ib);
    __syncthreads();
    for (int e = tid; e < kN * nc; e += kThreads) {
      const int row = e / nc, c = e - row * nc;
      out[(long)row * k + c0 + c] = s_x[c * kOutStride + row];
    }
    __syncthreads();
  }
  if (sweeps_out && tid == 0) sweeps_out[m] = more ? -sweep : sweep;
}

}  // namespace

// matrices up to which eight waves per matrix are the faster: with one matrix per compute unit the
// four waves of SPLIT = 1 leave half of the issue slots empty (40 matrices 1025 -> 892 us, 256
// matrices 1039 -> 913 us); with more, the angles repeated in eight waves cost more (512 matrices
// 1253 -> 1296 us, 1280 matrices 2463 -> 2714 us)
static constexpr int kSplitBatch = 256;

extern "C" int oa_sym_eig_top(const float* M, long m_stride, int batch, int n, int k, float* evals,
                              float* evecs, int* sweeps, void* stream) {
  if (batch < 0 || n != kN || k < 1 || k > kMaxK || m_stride < (long)kN * kN || !M || !evals ||
      !evecs)
    return OA_EINVAL;
  if (batch == 0) return 0;
  if (batch <= kSplitBatch)
    hipLaunchKernelGGL(sym_eig_top_kernel<2>, dim3(batch), dim3(Jacobi<2>::kThreads), 0, (hipStream_t)stream,
                       M, m_stride, k, evals, evecs, sweeps);
  else
    hipLaunchKernelGGL(sym_eig_top_kernel<1>, dim3(batch), dim3(Jacobi<1>::kThreads), 0, (hipStream_t)stream,
                       M, m_stride, k, evals, evecs, sweeps);
  return OA_LAUNCH_STATUS();
}
