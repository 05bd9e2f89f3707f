// Prefill index build on gfx950: QGS codes, QGC projection, k-means (assign / update), and the
// cluster statistics with their CSR member lists.  One request (batch row) at a time: kv_rows
// KV-head rows and rows = G * kv_rows query-head rows; query row r reads KV row r / G.
//
// Reference: the fast build of inference/ours_fastbuild.py:236-304 and the eager build of
// inference/methods_eager.py:505-555, with the accuracy-path semantics where they differ:
//   codes    zc = k U (fp32), scale = max(max_t |zc| / 127, 1e-12) per (KV head, coordinate),
//            codes = clamp(rint(zc / scale), -127, 127)  (static_top_k.py:174-181)
//   project  zP = bf16(k W) - colmean, colmean = mean_t bf16(k W)  (methods_eager.py:526-531,
//            ours_fastbuild.py:264-275)
//   assign   a_t = argmax_c bf16(bf16(bf16(zP_t) . bf16(c)) - bf16(|c|^2 / 2)), ties to the lower
//            cluster  (ours_fastbuild.py:52-82, methods_eager.py:536-540)
//   update   c = mean of the members, an empty cluster keeps its initial point
//            (ours_fastbuild.py:85-108, methods_eager.py:541-547)
//   sums     n_c, Sk_c = sum k, Sk2_c = sum k*k, Sv_c = sum v over the members; member lists =
//            stable argsort of the assignment  (ours_fastbuild.py:111-139, 293-301)
//
// Orders.  The reference leaves every summation order to its libraries.  This build fixes one
// wherever a CPU restatement has to match it bit for bit:
//   codes    zc_r = fma chain over d = 0..127 in fp32 (z = fma(k_d, U_dr, z), from z = 0);
//   colmean  per 64-token tile an fp64 sum in a fixed lane order, the tiles summed in order,
//            then one rounding of sum / T to fp32;
//   update   per cluster the sum of the members, one rounding of sum / count to fp32: in fp64 in position
//            order in oa_kmeans_update; in oa_kmeans_step exact over 2048 tokens (kmeans_assign_kernel
//            says how), then in fp64 in order;
//   sums     per cluster fp64 sums of k, k*k and v over the members, a fixed order that the row's length
//            and cluster count give (cluster_sums_kernel), one rounding to fp32.
// The two matrix products of the QGC step (k W and zP . c) run on the bf16 matrix cores with
// fp32 accumulation, as the reference's bf16 matmuls do; their fp32 partial rounding is the
// hardware's, so the CPU restatement matches them up to an agreement rate (ties of the bf16
// result), not bit for bit.
#include <algorithm>
#include <cfloat>
#include <type_traits>

#include "oa_common.h"

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short short4v;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float float4v;

constexpr int kD = 128;
constexpr int kRQ = 32;       // QGS rank
constexpr int kRC = 16;       // QGC rank
constexpr int kMaxC = 256;

__device__ __forceinline__ __bf16 bits_bf16(uint16_t h) { return __builtin_bit_cast(__bf16, h); }

// ---------------------------------------------------------------------------------- codes
// zc of one token (one lane) against U in LDS (U[d][r], 128 x 32 floats): fma chain over d
__device__ __forceinline__ void token_zc(const uint16_t* krow, const float* sU, float z[kRQ]) {
#pragma unroll
  for (int r = 0; r < kRQ; ++r) z[r] = 0.f;
  for (int d0 = 0; d0 < kD; d0 += 8) {
    const uint4 w = *reinterpret_cast<const uint4*>(krow + d0);
    float kv[8];
    oa::unpack8(w, kv);
#pragma unroll
    for (int dd = 0; dd < 8; ++dd) {
      const float4* u4 = reinterpret_cast<const float4*>(sU + (d0 + dd) * kRQ);
#pragma unroll
      for (int r4 = 0; r4 < kRQ / 4; ++r4) {
        const float4 u = u4[r4];
        z[4 * r4] = fmaf(kv[dd], u.x, z[4 * r4]);
        z[4 * r4 + 1] = fmaf(kv[dd], u.y, z[4 * r4 + 1]);
        z[4 * r4 + 2] = fmaf(kv[dd], u.z, z[4 * r4 + 2]);
        z[4 * r4 + 3] = fmaf(kv[dd], u.w, z[4 * r4 + 3]);
      }
    }
  }
}

constexpr int kCodeThreads = 256;

__global__ void __launch_bounds__(64) clear_u32_kernel(uint32_t* p, int n) {
  for (int i = threadIdx.x + blockIdx.x * 64; i < n; i += 64 * gridDim.x) p[i] = 0u;
}

// pass 1: per (KV row, coordinate) the maximum |zc| over the tokens, as float bits (|zc| >= 0,
// so the unsigned maximum of the bits is the float maximum); zc itself into zc_ws when given
// (128 bytes per token), so that pass 2 quantizes without a second fma chain.
// The fma chains run on the fp32 matrix cores: v_mfma_f32_32x32x1_2b_f32 adds one product per output
// with one rounding, an fma, so that 128 of them over d = 0..127 are token_zc's chains bit for bit
// (subnormal products included) at twice the vector rate.  A is U (coordinate lane % 32), B dimension d
// of the wave's 64 tokens (token lane), and a lane ends with coordinates 8 (r / 4) + 4 (lane / 32) + r % 4
// of tokens lane % 32 and 32 + lane % 32.  U lies in LDS by fours of d: as 128 registers it left two
// waves per SIMD, the next keys went through scratch and the matrix cores waited for them (1229 us
// against the figure below).  The key rows reach LDS 64 dims at a time in coalesced 128-byte segments
// (rows padded to 144 bytes: a 16-lane phase of row reads hits distinct banks), the next segment
// requested while one is used; a wave takes up to kZcTiles tiles of 64 tokens.  At 256 rows of 32767
// tokens: 1310 us with the chains on the vector units, 731 us now, 3.2 GB of keys and zc at 4.4 TB/s
// beside 0.5 ms of matrix instructions; at 16 rows of 10007 tokens 42 -> 26 us.
constexpr int kZcDims = 64;                    // dims staged per segment
constexpr int kZcRowQ = kZcDims / 8 + 1;       // uint4 per staged row (8 + 1 pad)
constexpr int kZcTiles = 8;                    // 64-token tiles per wave
typedef __attribute__((__vector_size__(32 * sizeof(float)))) float float32v;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t uint32x4v;

__global__ void __launch_bounds__(kCodeThreads, 3) codes_amax_kernel(const uint16_t* __restrict__ K, long ksh,
                                                                     long kst, int T,
                                                                     const float* __restrict__ U,
                                                                     uint32_t* __restrict__ amax,
                                                                     float* __restrict__ zc_ws, int tiles) {
  __shared__ uint32_t s_m[kRQ];
  __shared__ uint4 s_k[kCodeThreads / 64][64 * kZcRowQ];
  __shared__ float4 s_u[kD / 4][kRQ];
  const int h = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int hi = lane >> 5, n32 = lane & 31;
  const float* Uh = U + (long)h * kD * kRQ;
  if (threadIdx.x < kRQ) s_m[threadIdx.x] = 0u;
  for (int i = threadIdx.x; i < kD / 4 * kRQ; i += kCodeThreads) {
    const float* up = Uh + (i / kRQ) * 4 * kRQ + i % kRQ;
    s_u[i / kRQ][i % kRQ] = make_float4(up[0], up[kRQ], up[2 * kRQ], up[3 * kRQ]);
  }
  __syncthreads();
  const uint16_t* kh = K + (long)h * ksh;
  const int ntiles = (T + 63) / 64;
  const int tile0 = (blockIdx.x * (kCodeThreads / 64) + wave) * tiles;
  const int tend = min(ntiles, tile0 + tiles);
  // a segment's 512 16-byte words: lane takes word lane % 8 of rows lane / 8 + 8 j
  uint32x4v seg[8];
  auto fetch = [&](int tile, int half) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      seg[j] = *reinterpret_cast<const uint32x4v*>(kh + (long)min(tile * 64 + (lane >> 3) + 8 * j, T - 1) * kst +
                                                   half * kZcDims + 8 * (lane & 7));
  };
  uint32_t mx[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) mx[r] = 0u;
  if (tile0 < tend) fetch(tile0, 0);
#pragma unroll 1
  for (int tile = tile0; tile < tend; ++tile) {
    float32v acc = {};
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      // (one wave's LDS: its reads of the last segment precede these writes in order)
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 8; ++j)
        *reinterpret_cast<uint32x4v*>(&s_k[wave][((lane >> 3) + 8 * j) * kZcRowQ + (lane & 7)]) = seg[j];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
      fetch(min(tile + half, ntiles - 1), half ^ 1);
#pragma unroll
      for (int c = 0; c < kZcDims / 8; ++c) {
        float kv[8];
        oa::unpack8(s_k[wave][lane * kZcRowQ + c], kv);
        const float4 ua = s_u[half * (kZcDims / 4) + 2 * c][n32], ub = s_u[half * (kZcDims / 4) + 2 * c + 1][n32];
        const float u[8] = {ua.x, ua.y, ua.z, ua.w, ub.x, ub.y, ub.z, ub.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x1f32(u[e], kv[e], acc, 0, 0, 0);
      }
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int t = tile * 64 + 32 * b + n32;
      if (t < T) {
#pragma unroll
        for (int r = 0; r < 16; ++r) mx[r] = max(mx[r], __float_as_uint(fabsf(acc[16 * b + r])));
        if (zc_ws) {
          float4* zo = reinterpret_cast<float4*>(zc_ws + ((long)h * T + t) * kRQ + 4 * hi);
#pragma unroll
          for (int g = 0; g < 4; ++g)
            zo[2 * g] = make_float4(acc[16 * b + 4 * g], acc[16 * b + 4 * g + 1], acc[16 * b + 4 * g + 2],
                                    acc[16 * b + 4 * g + 3]);
        }
      }
    }
  }
  __syncthreads();                               // s_m is cleared
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    // the maximum over the 32 lanes that hold this coordinate
    uint32_t v = mx[r];
    v = max(v, oa::dpp_u32<0xB1, 0xf>(v));
    v = max(v, oa::dpp_u32<0x4E, 0xf>(v));
    v = max(v, oa::dpp_u32<0x141, 0xf>(v));
    v = max(v, oa::dpp_u32<0x140, 0xf>(v));
    const auto x = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = max((uint32_t)x[0], (uint32_t)x[1]);
    if (n32 == 0) atomicMax(&s_m[8 * (r >> 2) + 4 * hi + (r & 3)], v);
  }
  __syncthreads();
  if (threadIdx.x < kRQ) atomicMax(&amax[h * kRQ + threadIdx.x], s_m[threadIdx.x]);
}

// pass 2: the codes (32 bytes per token) and, from the first block of each KV row, the scale
__global__ void __launch_bounds__(kCodeThreads) codes_write_kernel(const uint16_t* K, long ksh, long kst,
                                                                   int T, const float* U,
                                                                   const uint32_t* amax, int8_t* codes,
                                                                   long csh, float* scale,
                                                                   const float* zc_ws) {
  __shared__ float sU[kD * kRQ];
  __shared__ float s_sc[kRQ];
  const int h = blockIdx.y;
  for (int i = threadIdx.x; i < kD * kRQ; i += kCodeThreads) sU[i] = U[(long)h * kD * kRQ + i];
  if (threadIdx.x < kRQ) {
    const float sc = fmaxf(__uint_as_float(amax[h * kRQ + threadIdx.x]) / 127.0f, 1e-12f);
    s_sc[threadIdx.x] = sc;
    if (blockIdx.x == 0) scale[h * kRQ + threadIdx.x] = sc;
  }
  __syncthreads();
  const int t = blockIdx.x * kCodeThreads + threadIdx.x;
  if (t >= T) return;
  float z[kRQ];
  if (zc_ws) {
    const float4* zi = reinterpret_cast<const float4*>(zc_ws + ((long)h * T + t) * kRQ);
#pragma unroll
    for (int r4 = 0; r4 < kRQ / 4; ++r4) {
      const float4 v = zi[r4];
      z[4 * r4] = v.x; z[4 * r4 + 1] = v.y; z[4 * r4 + 2] = v.z; z[4 * r4 + 3] = v.w;
    }
  } else {
    token_zc(K + (long)h * ksh + (long)t * kst, sU, z);
  }
  uint32_t packed[kRQ / 4];
#pragma unroll
  for (int r4 = 0; r4 < kRQ / 4; ++r4) {
    uint32_t w = 0u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float q = fminf(fmaxf(rintf(z[4 * r4 + j] / s_sc[4 * r4 + j]), -127.f), 127.f);
      w |= ((uint32_t)(uint8_t)(int8_t)(int)q) << (8 * j);
    }
    packed[r4] = w;
  }
  uint4* dst = reinterpret_cast<uint4*>(codes + (long)h * csh + (long)t * kRQ);
  dst[0] = make_uint4(packed[0], packed[1], packed[2], packed[3]);
  dst[1] = make_uint4(packed[4], packed[5], packed[6], packed[7]);
}

// ---------------------------------------------------------------------------------- projection
constexpr int kProjTiles = 8;    // 64-token tiles per wave (the row's W operands loaded once)
// One wave per (8 64-token tiles, query row or KV row).  Four 16-token blocks, each 16 tokens x 16 columns
// from four v_mfma_f32_16x16x32_bf16 over d = 0..127 (A: token rows of K, B: the row's W).
// Output layout of a 16x16 block: lane l holds tokens 4*(l/16) + i (i = 0..3) of column l % 16.
// zraw = bf16(acc) is written (as fp32) into zP, and the tile's column sums (fp64, lane order
// below) into tsum[row][tile][16].
// NG query rows per wave (NG == G: a KV row's query rows, whose K blocks are then loaded once for
// all of them; NG == 1: blockIdx.y is the query row).
template <int NG>
__global__ void __launch_bounds__(64) qgc_project_kernel(const uint16_t* K, long ksh, long kst, int G,
                                                         int T, const uint16_t* W, float* zP,
                                                         long zps, uint16_t* zraw_out, double* tsum,
                                                         int ntiles, uint32_t* wmax) {
  __shared__ uint4 s_z[NG][64 * kRC / 8];         // the tile's bf16(k W), token rows of 32 bytes
  const int lane = threadIdx.x;
  const int row0 = NG == 1 ? (int)blockIdx.y : (int)blockIdx.y * G;
  const uint16_t* krow = K + (long)(row0 / G) * ksh;
  // B operand of chunk ch: column j = lane % 16, dims ch*32 + 8*(lane/16) + e, e = 0..7
  bf16x8 bw[NG][4];
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int ch = 0; ch < 4; ++ch)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        bw[g][ch][e] = bits_bf16(W[(long)(row0 + g) * kD * kRC + (ch * 32 + 8 * (lane >> 4) + e) * kRC + (lane & 15)]);
  const int tend = min(ntiles, (int)(blockIdx.x + 1) * kProjTiles);
  uint32_t mx[NG];   // this lane's column: the largest |bf16(k W)|, as float bits
#pragma unroll
  for (int g = 0; g < NG; ++g) mx[g] = 0u;
#pragma unroll 1
  for (int tile = blockIdx.x * kProjTiles; tile < tend; ++tile) {
  double cs[NG];   // this lane's column (lane % 16) partial over its tokens, in block order
#pragma unroll
  for (int g = 0; g < NG; ++g) cs[g] = 0.0;
#pragma unroll
  for (int blk = 0; blk < 4; ++blk) {
    const int t0 = tile * 64 + blk * 16;
    const int ta = min(t0 + (lane & 15), T - 1);          // A row: token t0 + lane % 16
    uint4 av[4];
#pragma unroll
    for (int ch = 0; ch < 4; ++ch)
      av[ch] = *reinterpret_cast<const uint4*>(krow + (long)ta * kst + ch * 32 + 8 * (lane >> 4));
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      float4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ch = 0; ch < 4; ++ch)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av[ch]), bw[g][ch], acc, 0, 0, 0);
      uint16_t* s_zh = reinterpret_cast<uint16_t*>(s_z[g]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = t0 + 4 * (lane >> 4) + i;
        const uint16_t hb = oa::f32_to_bf16_rn(acc[i]);
        const float v = oa::bf16_to_f32(hb);
        s_zh[(blk * 16 + 4 * (lane >> 4) + i) * kRC + (lane & 15)] = hb;
        if (t < T) {
          if (zP) zP[(long)(row0 + g) * zps + (long)t * kRC + (lane & 15)] = v;
          cs[g] += (double)v;
          mx[g] = max(mx[g], __float_as_uint(fabsf(v)));
        }
      }
    }
  }
  // the tile's rows out through LDS: lane l writes token l's 32 bytes
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (zraw_out) {
    const int t = tile * 64 + lane;
    if (t < T) {
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        uint4* dst = reinterpret_cast<uint4*>(zraw_out + (long)(row0 + g) * zps + (long)t * kRC);
        dst[0] = s_z[g][lane * 2];
        dst[1] = s_z[g][lane * 2 + 1];
      }
    }
  }
  // lanes j, 16 + j, 32 + j, 48 + j hold column j: ((g0 + g1) + (g2 + g3))
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    double c = cs[g];
    c += __shfl_xor(c, 16, 64);
    c += __shfl_xor(c, 32, 64);
    if (lane < 16) tsum[((long)(row0 + g) * ntiles + tile) * kRC + lane] = c;
  }
  // the next tile's stores to s_z wait for these reads
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  }
  if (wmax)
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const auto r16 = __builtin_amdgcn_permlane16_swap(mx[g], mx[g], false, false);
      const uint32_t v = max(r16[0], r16[1]);
      const auto r32 = __builtin_amdgcn_permlane32_swap(v, v, false, false);
      if (lane < 16) wmax[((long)(row0 + g) * gridDim.x + blockIdx.x) * kRC + lane] = max(r32[0], r32[1]);
    }
}

// A column's bound word: the bits of a largest |bf16(k W)| that is finite, with kOddColumn where some
// value of the column is not
constexpr uint32_t kOddColumn = 0x80000000u;

// colmean from the tile sums (tiles in order, fp64): one wave per row, lane j < 16 a column; the
// sums of 16 tiles are requested together and then added in tile order (one load in flight at a
// time left the pass bound by memory latency: 0.21 ms at 512 tiles, 0.44 ms at 2048)
// Lanes 16 .. 31: the bound word of column lane - 16 from the nw waves' maxima (a value that is not finite
// makes the column's mean so too, and every zP: what is finite beside it does not matter then).
__global__ void __launch_bounds__(64) qgc_colmean_kernel(int T, const double* tsum, int ntiles,
                                                         float* colmean, const uint32_t* wmax, int nw,
                                                         uint32_t* zmax) {
  constexpr int kBatch = 16;
  const int row = blockIdx.x;
  const int j = threadIdx.x;
  if (j < kRC) {
    const double* p = tsum + (long)row * ntiles * kRC + j;
    double s = 0.0;
    int k = 0;
    for (; k + kBatch <= ntiles; k += kBatch) {
      double x[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) x[u] = p[(long)(k + u) * kRC];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) s += x[u];
    }
    for (; k < ntiles; ++k) s += p[(long)k * kRC];
    colmean[row * kRC + j] = (float)(s / (double)T);
  } else if (zmax && j < 2 * kRC) {
    const uint32_t* p = wmax + (long)row * nw * kRC + j - kRC;
    uint32_t m = 0u;
#pragma unroll 8
    for (int k = 0; k < nw; ++k) m = max(m, p[(long)k * kRC]);
    zmax[row * kRC + j - kRC] = m < 0x7f800000u ? m : kOddColumn | 0x7f7f0000u;
  }
}

// zP -= colmean in place (float4 per thread: four columns of one token)
__global__ void __launch_bounds__(256) qgc_center_kernel(float* zP, long zps, int T,
                                                         const float* colmean) {
  const int row = blockIdx.y;
  const float* cm = colmean + row * kRC;
  float4* z = reinterpret_cast<float4*>(zP + (long)row * zps);
  const long n4 = (long)T * (kRC / 4);
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n4; i += (long)gridDim.x * 256) {
    const int c4 = (int)(i & 3) * 4;
    float4 v = z[i];
    v.x = v.x - cm[c4];
    v.y = v.y - cm[c4 + 1];
    v.z = v.z - cm[c4 + 2];
    v.w = v.w - cm[c4 + 3];
    z[i] = v;
  }
}

// ---------------------------------------------------------------------------------- k-means
// two fp32 values rounded to bf16 (nearest even) in one conversion: a in the low half
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2v;
__device__ __forceinline__ uint32_t cvt_pk_bf16(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2v));
}

// bf16(b) above the high half of `tag`, which comes from a scalar register: left to the compiler, every
// distinct tag took a vector register
__device__ __forceinline__ uint32_t cvt_pk_bf16_tag(uint32_t tag, float b) {
  uint32_t r;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "s"(tag), "v"(b));
  return r;
}

// One 256-thread workgroup per (4 x tiles_per_wave 64-token tiles, query row).  The row's centroids
// (bf16) are the A operand of v_mfma_f32_16x16x16bf16_1k and 16 tokens the B operand, so that a lane
// holds distances of one token: centroids 16 cb + 4 (lane / 16) + i of token lane % 16 for the
// centroid blocks cb, kept in registers with their bf16(|c|^2 / 2) for all of the wave's tiles.
//
// A distance bf16(bf16(dot) - half) is ranked as one integer: the conversion that rounds it to bf16
// puts it above a 16-bit tag that is larger for a lower cluster (v_cvt_pk_bf16_f32 with a constant
// for the low half).  As a signed integer that order is the distance's own wherever the best one is
// positive, as it is for most tokens once the centroids are means; a block of 16 tokens with a best
// distance that is not a positive finite number is ranked again with the negative distances' order
// set right (two instructions more per distance), and so are the blocks after it until one would not
// have needed it.  A row with a centroid of half = +0 (only there can bf16(x - half) be -0, which
// ranks as +0) is ranked with a third order.
//
// Bound by vector issue: 3.5 instructions per distance and about 26 per 16 tokens; with tokens as
// rows a distance took about 8 (keys and tags formed apart) and each block of 16 tokens a 16-lane
// maximum of four registers.  32 sequences of 32767 tokens, 64 clusters: 725 -> 432 us per
// assignment; two of 10007 tokens, 256 clusters: 109 -> 38 us.
constexpr int kAsgThreads = 256;
constexpr int kAsgMaxTiles = 8;                // tiles per wave where the grid is full without
constexpr uint32_t kTag = 0x3f00u;             // low half of a ranked distance: kTag | 63 - (4 cb + i)
//
// ACC (a whole Lloyd iteration): each token's zP also joins its cluster's sum, in LDS per workgroup,
// and the workgroup's sums and counts go to ll for kmeans_mean_kernel; asg and asg8 may be null.  No
// order of the tokens shows in the centroids, nor how many tiles a wave takes (a segment of kSegTiles
// tiles is summed exactly, and the segments are added in order):
//   fp64     where every column of the row has |zP| <= 2^17 |colmean| =: 2^17 m.  Every zP is a multiple
//            of half of m's last place (of m's 2^-25 at least), and 2048 of them stay below 2^28 m = 2^53
//            times that, so that every partial sum is exact.
//   wholes   else (a column whose mean is small against its values, or one with values that are not
//            finite): a value counts in units of 2^-51 of a power of two above the row's largest |zP| in
//            the column.  x + 1.5 * 2^52 holds the whole number in its low bits, and the bits are added
//            as 64-bit integers (the constant's share comes off by the count).  A value keeps all of its
//            24 bits down to 2^-27 of the largest.  Infinities and NaN are noted per cluster and column.
// (fp64 atomics alone: a column of +-2^20 in pairs beside 2^-22 gave other centroids at every call.  Whole
// numbers for every row: 9.17 ms for a build of 32 sequences of 32767 tokens, 8.79 so, 8.71 before.)
// |zP| is bounded by |bf16(k W)| + |colmean| of the column (rounding keeps the order).  Before, the ids of
// every iteration were sorted into member lists and each cluster's rows gathered again: 0.14 + 0.44 ms
// per iteration at 32 sequences.
constexpr int kAccStride = kRC + 1;            // sums per cluster in LDS (spread over the banks)
constexpr int kSegTiles = kAsgThreads / 64 * kAsgMaxTiles;
constexpr double kWhole = 6755399441055744.0;  // 1.5 * 2^52

struct LloydArgs {                             // a whole iteration's inputs and partial results
  const uint32_t* zmax;                        // bound words (rows, 16)
  unsigned long long* part;                    // sums (rows, workgroups, C, 16), fp64 or whole numbers
  int32_t* pcnt;                               // counts (rows, workgroups, C)
  uint32_t* pbad;                              // (rows, workgroups, C): 2 bits a column, +inf and -inf (NaN: both)
  int32_t* pexp;                               // (rows, 16): kFp64Sums, or the unit is 2^-pexp
};
constexpr int kFp64Sums = 0x7fffffff;

template <int CB, bool ACC>
__global__ void __launch_bounds__(kAsgThreads, CB <= 4 ? 6 : CB <= 12 || !ACC ? 4 : 3) kmeans_assign_kernel(const uint16_t* zraw,
                                                                    const float* colmean, long zps, int T,
                                                                    const float* cent, int C,
                                                                    int32_t* asg, long as,
                                                                    uint8_t* asg8, long a8s,
                                                                    int tiles_per_wave, LloydArgs ll) {
  __shared__ __align__(16) uint16_t s_cb[CB * 16 * kRC];
  __shared__ __align__(16) float s_half[CB * 16];
  __shared__ unsigned long long s_acc[ACC ? CB * 16 * kAccStride : 1];   // (0 in either form)
  __shared__ int s_cnt[ACC ? CB * 16 : 1];
  __shared__ uint32_t s_bad[ACC ? CB * 16 : 1];
  if (ACC) {
    for (int i = threadIdx.x; i < CB * 16 * kAccStride; i += kAsgThreads) s_acc[i] = 0ull;
    for (int i = threadIdx.x; i < CB * 16; i += kAsgThreads) { s_cnt[i] = 0; s_bad[i] = 0u; }
  }
  const int lane = threadIdx.x & 63, grp = lane >> 4;
  const int wave = threadIdx.x >> 6;
  const int row = blockIdx.y;
  const int ntiles = (T + 63) / 64;
  const float* cr = cent + (long)row * C * kRC;
  // four centroid values per thread and iteration (C * kRC is a multiple of 4)
  for (int i = 4 * threadIdx.x; i < CB * 16 * kRC; i += 4 * kAsgThreads) {
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i < C * kRC) x = *reinterpret_cast<const float4*>(cr + i);
    s_cb[i] = oa::f32_to_bf16(x.x);
    s_cb[i + 1] = oa::f32_to_bf16(x.y);
    s_cb[i + 2] = oa::f32_to_bf16(x.z);
    s_cb[i + 3] = oa::f32_to_bf16(x.w);
  }
  int zero_half = 0;          // this thread staged a real centroid with bf16(|c|^2 / 2) = +0
  for (int c = threadIdx.x; c < CB * 16; c += kAsgThreads) {
    uint16_t hv = 0x7f80u;   // padding centroids: +inf, a distance of -inf ranks below every real one
    if (c < C) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < kRC; ++j) {
        const float x = cr[c * kRC + j];
        s = s + x * x;
      }
      hv = oa::f32_to_bf16(0.5f * s);
      zero_half |= hv == 0;
    }
    s_half[c] = oa::bf16_to_f32(hv);
  }
  const bool plain = __syncthreads_or(zero_half) == 0;
  short4v ca[CB];
  float4 hf[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    ca[cb] = *reinterpret_cast<const short4v*>(s_cb + (cb * 16 + (lane & 15)) * kRC + 4 * grp);
    hf[cb] = *reinterpret_cast<const float4*>(s_half + cb * 16 + 4 * grp);
  }
  // zP = bf16(k W) - colmean, formed from the stored bf16 projection (the same fp32 values)
  float cm[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) cm[e] = colmean[row * kRC + 4 * grp + e];
  int ex[4] = {0, 0, 0, 0};                    // |zP| < 2^(51 - ex)
  bool wholes = false;                         // (uniform: every wave holds all columns)
  if (ACC) {
    bool far = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t w = ll.zmax[row * kRC + 4 * grp + e];
      const float m = fabsf(cm[e]);
      float b = __uint_as_float(w & ~kOddColumn) + (m < INFINITY ? m : 0.f);
      if (!(b < INFINITY)) b = FLT_MAX;
      far |= (w & kOddColumn) || !(b <= 131072.f * m && m < INFINITY);
      ex[e] = 177 - (int)(__float_as_uint(b) >> 23);       // b < 2^(field - 126)
    }
    wholes = __any(far);
    if (blockIdx.x == 0 && wave == 0 && (lane & 15) == 0)
#pragma unroll
      for (int e = 0; e < 4; ++e) ll.pexp[row * kRC + 4 * grp + e] = wholes ? ex[e] : kFp64Sums;
  }
  const uint16_t* zr = zraw + (long)row * zps + 4 * grp;
  auto load = [&](uint2 (&z)[4], int tile) {
#pragma unroll
    for (int blk = 0; blk < 4; ++blk)
      z[blk] = *reinterpret_cast<const uint2*>(zr + (long)min(tile * 64 + blk * 16 + (lane & 15), T - 1) * kRC);
  };
  const int tile0 = (blockIdx.x * (kAsgThreads / 64) + wave) * tiles_per_wave;
  const int tend = min(ntiles, tile0 + tiles_per_wave);
  uint2 z[4];
  if (tile0 < tend) load(z, tile0);
  bool positive = plain;     // the last block's best distances were: try the cheap order on the next
#pragma unroll 1
  for (int tile = tile0; tile < tend; ++tile) {
    uint2 zn[4];
    load(zn, min(tile + 1, ntiles - 1));
    int mine = 0;              // the ranked best of this lane's token of the tile (token lane)
#pragma unroll 1
    for (int blk = 0; blk < 4; ++blk) {
      const float zp[4] = {__uint_as_float(z[0].x << 16) - cm[0], __uint_as_float(z[0].x & 0xffff0000u) - cm[1],
                           __uint_as_float(z[0].y << 16) - cm[2], __uint_as_float(z[0].y & 0xffff0000u) - cm[3]};
      const uint2 w = make_uint2(cvt_pk_bf16(zp[0], zp[1]), cvt_pk_bf16(zp[2], zp[3]));
      const short4v tok = __builtin_bit_cast(short4v, w);
      z[0] = z[1]; z[1] = z[2]; z[2] = z[3];
      // the token's best: 0 as the bits stand (right where it is positive), 1 in the distances' order,
      // 2 the same with -0 as +0
      auto rank = [&](auto mode_c) {
        constexpr int MODE = decltype(mode_c)::value;
        int best = (int)0x80000000u;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          float4v acc = {0.f, 0.f, 0.f, 0.f};
          acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ca[cb], tok, acc, 0, 0, 0);
          const float h[4] = {hf[cb].x, hf[cb].y, hf[cb].z, hf[cb].w};
          int v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float d = __uint_as_float(cvt_pk_bf16(0.f, acc[i])) - h[i];
            if (MODE == 2) d = __uint_as_float(cvt_pk_bf16(0.f, d)) + 0.f;
            v[i] = (int)cvt_pk_bf16_tag((kTag | (63 - (4 * cb + i))) << 16, d);
            if (MODE) v[i] ^= (v[i] >> 31) & 0x7fff0000;   // a negative distance's magnitude reversed
          }
          best = max(max(best, v[0]), v[1]);
          best = max(max(best, v[2]), v[3]);
        }
        // tag 63 - (4 cb + i) of lane group g -> 255 - (16 cb + 4 g + i), then the best of the groups
        const uint32_t u = (uint32_t)best;
        best = (int)((u & 0xffff0000u) | ((u & 0x3cu) << 2) | (u & 3u) | (uint32_t)(4 * (3 - grp)));
        const auto r16 = __builtin_amdgcn_permlane16_swap((uint32_t)best, (uint32_t)best, false, false);
        best = max((int)r16[0], (int)r16[1]);
        const auto r32 = __builtin_amdgcn_permlane32_swap((uint32_t)best, (uint32_t)best, false, false);
        return max((int)r32[0], (int)r32[1]);
      };
      int best = 0;
      if (positive) best = rank(std::integral_constant<int, 0>());
      if (!positive || __ballot(best <= 0 || best >= 0x7f800000) != 0ull) {
        best = plain ? rank(std::integral_constant<int, 1>()) : rank(std::integral_constant<int, 2>());
        positive = plain && __ballot(best <= 0 || best >= 0x7f800000) == 0ull;
      }
      mine = grp == blk ? best : mine;
      if (ACC && tile * 64 + blk * 16 + (lane & 15) < T) {
        const int cid = 255 - (best & 0xff);          // of token lane % 16, in every lane group
        if (!wholes) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            __hip_atomic_fetch_add(reinterpret_cast<double*>(&s_acc[cid * kAccStride + 4 * grp + e]), (double)zp[e],
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float v = zp[e];
            if (!(fabsf(v) < INFINITY)) {
              atomicOr(&s_bad[cid], (v > 0.f ? 1u : v < 0.f ? 2u : 3u) << (2 * (4 * grp + e)));
              v = 0.f;
            }
            const double x = (double)__builtin_amdgcn_ldexpf(v, ex[e]) + kWhole;
            __hip_atomic_fetch_add(&s_acc[cid * kAccStride + 4 * grp + e], (unsigned long long)__double_as_longlong(x),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          }
        }
        if (grp == 0) atomicAdd(&s_cnt[cid], 1);
      }
    }
    const int t = tile * 64 + lane;
    if (t < T && (!ACC || asg)) {
      const int cid = 255 - (mine & 0xff);
      asg[(long)row * as + t] = cid;
      asg8[(long)row * a8s + t] = (uint8_t)cid;
    }
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) z[blk] = zn[blk];
  }
  if (ACC) {
    __syncthreads();
    const long g = ((long)row * gridDim.x + blockIdx.x) * C;
    const unsigned long long base = wholes ? (unsigned long long)__double_as_longlong(kWhole) : 0ull;
    for (int i = threadIdx.x; i < C * kRC; i += kAsgThreads)
      ll.part[g * kRC + i] = s_acc[(i / kRC) * kAccStride + i % kRC] - s_cnt[i / kRC] * base;
    for (int i = threadIdx.x; i < C; i += kAsgThreads) {
      ll.pcnt[g + i] = s_cnt[i];
      ll.pbad[g + i] = s_bad[i];
    }
  }
}

// The centroids from the workgroups' sums: one thread per value, its partials 8 at a time in flight.  A
// segment's (of wgs workgroups) are added exactly, then the segments in order, in fp64; an empty
// cluster keeps its initial point.
__global__ void __launch_bounds__(256) kmeans_mean_kernel(LloydArgs ll, int nwg, int wgs, int C,
                                                          const uint16_t* zraw, const float* colmean, long zps,
                                                          const int32_t* init_idx, float* cent) {
  const int row = blockIdx.y;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= C * kRC) return;
  const int c = i / kRC, j = i % kRC;
  const unsigned long long* p = ll.part + (long)row * nwg * C * kRC + i;
  const int32_t* q = ll.pcnt + (long)row * nwg * C + c;
  const uint32_t* b = ll.pbad + (long)row * nwg * C + c;
  const int ex = ll.pexp[row * kRC + j];
  double acc = 0.0, sum = 0.0;
  unsigned long long whole = 0ull;
  int cnt = 0;
  uint32_t bad = 0u;
  for (int g0 = 0; g0 < nwg; g0 += 8) {        // (wgs divides 8)
    unsigned long long px[8];
    int pq[8];
    uint32_t pb[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int g = min(g0 + u, nwg - 1);
      px[u] = p[(long)g * C * kRC];
      pq[u] = q[(long)g * C];
      pb[u] = ex != kFp64Sums ? b[(long)g * C] : 0u;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (g0 + u < nwg) {
        sum += __longlong_as_double((long long)px[u]);
        whole += px[u];                        // (two's complement, below 2^62: 2048 values)
        cnt += pq[u];
        bad |= pb[u];
        if ((u + 1) % wgs == 0 || g0 + u == nwg - 1) {
          acc += ex == kFp64Sums ? sum : __builtin_amdgcn_ldexp((double)(long long)whole, -ex);
          sum = 0.0;
          whole = 0ull;
        }
      }
  }
  bad = bad >> (2 * j) & 3u;
  if (bad) acc = bad == 3u ? NAN : bad == 1u ? INFINITY : -INFINITY;
  cent[(long)row * C * kRC + i] =
      cnt > 0 ? (float)(acc / (double)cnt)
              : oa::bf16_to_f32(zraw[(long)row * zps + (long)init_idx[c] * kRC + j]) - colmean[row * kRC + j];
}

// The bound words of a projection that came without them: one workgroup per row reads it once, a thread
// 8 columns of every 128th token.
__global__ void __launch_bounds__(256) column_max_kernel(const uint16_t* zraw, long zps, int T, uint32_t* zmax) {
  typedef uint32_t uint32x4a8 __attribute__((ext_vector_type(4), aligned(8)));
  __shared__ uint32_t s_mx[kRC], s_odd[kRC];
  const int row = blockIdx.x, half = threadIdx.x & 1;
  if (threadIdx.x < kRC) s_mx[threadIdx.x] = s_odd[threadIdx.x] = 0u;
  __syncthreads();
  uint32_t mx[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u}, odd = 0u;
#pragma unroll 4
  for (int t = threadIdx.x >> 1; t < T; t += 128) {
    const uint32x4a8 x = *reinterpret_cast<const uint32x4a8*>(zraw + (long)row * zps + (long)t * kRC + 8 * half);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t y = (k & 1 ? x[k >> 1] : x[k >> 1] << 16) & 0x7fff0000u;
      if (y < 0x7f800000u) mx[k] = max(mx[k], y);
      else odd |= 1u << k;
    }
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    atomicMax(&s_mx[8 * half + k], mx[k]);
    if (odd >> k & 1u) s_odd[8 * half + k] = kOddColumn;
  }
  __syncthreads();
  if (threadIdx.x < kRC) zmax[row * kRC + threadIdx.x] = s_mx[threadIdx.x] | s_odd[threadIdx.x];
}

// a wave copies 1 <= n <= (the LDS array's size) member positions into LDS, eight loads per lane
// in flight at a time (one at a time, each copy waited on its load)
__device__ __forceinline__ void stage_members(int* s_pos, const int32_t* ml, int n, int lane) {
  for (int b = 0; b < n; b += 512) {
    int v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = ml[min(b + lane + 64 * u, n - 1)];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (b + lane + 64 * u < n) s_pos[b + lane + 64 * u] = v[u];
  }
}

// One wave per (cluster, query row): the members in position order (the row's member lists of
// csr_sort_kernel), their zP rows staged kUB at a time through LDS (the next batch requested
// while one is summed) and summed in fp64 by lanes 0..15 (one column each) in that order;
// centroid = fp32(sum / count), or the initial point when the cluster is empty.
__global__ void __launch_bounds__(64) kmeans_update_kernel(const uint16_t* zraw, const float* colmean,
                                                           long zps, int C, const int32_t* mem, long ms,
                                                           const int32_t* cstart, const int32_t* clen,
                                                           const int32_t* init_idx, float* cent,
                                                           float* cnt_out) {
  constexpr int kUB = 64;                      // members per staged batch
  constexpr int kUpdBuf = 512;                 // member positions staged at a time (6 KB of LDS
                                               // per wave: about 26 waves per compute unit)
  __shared__ int s_pos[kUpdBuf];
  __shared__ float4 s_stage[kUB * (kRC / 4)];
  const int lane = threadIdx.x;
  // the C workgroups of a row run on one XCD (workgroups are dealt to the 8 XCDs in turn), so the
  // row's projection lines, each holding the rows of members of several clusters, are fetched
  // into that XCD's L2 once rather than by every XCD
  int c, row;
  {
    const int b = blockIdx.x, rows = gridDim.x / C;
    if (rows % 8 == 0) {
      const int k = b >> 3;
      row = (k / C) * 8 + (b & 7);
      c = k % C;
    } else {
      row = b / C;
      c = b % C;
    }
  }
  const int32_t* ml = mem + (long)row * ms + cstart[row * C + c];
  const int cl = clen[row * C + c];
  const uint16_t* zr = zraw + (long)row * zps;
  // zP = bf16(k W) - colmean from the stored bf16 projection: this lane's quarter of a row
  float cq[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) cq[e] = colmean[row * kRC + 4 * (lane & 3) + e];
  double acc = 0.0;
  int cnt = 0;
  // lane l reads member quarter l % 4 of members l / 4 + 16 b of a batch; a slot past the last
  // member reads the last member's row again (never summed), so the loads issue without branches
  auto load = [&](uint2* w, int k0, int n) {
#pragma unroll
    for (int b = 0; b < kUB / 16; ++b) {
      const int m = min(k0 + (lane >> 2) + 16 * b, n - 1);
      w[b] = *reinterpret_cast<const uint2*>(zr + (long)s_pos[m] * kRC + 4 * (lane & 3));
    }
  };
  for (int i0 = 0; i0 < cl; i0 += kUpdBuf) {
    const int n = min(kUpdBuf, cl - i0);
    stage_members(s_pos, ml + i0, n, lane);
    __syncthreads();
    uint2 w[kUB / 16];
    if (n > 0) load(w, 0, n);
    for (int k0 = 0; k0 < n; k0 += kUB) {
#pragma unroll
      for (int b = 0; b < kUB / 16; ++b)
        s_stage[((lane >> 2) + 16 * b) * 4 + (lane & 3)] =
            make_float4(__uint_as_float(w[b].x << 16) - cq[0], __uint_as_float(w[b].x & 0xffff0000u) - cq[1],
                        __uint_as_float(w[b].y << 16) - cq[2], __uint_as_float(w[b].y & 0xffff0000u) - cq[3]);
      __syncthreads();
      // the next batch's rows are requested while this one is summed
      if (k0 + kUB < n) load(w, k0 + kUB, n);
      if (lane < kRC) {
        // 16 staged values read together, then added in member order (a slot past the last
        // member adds +0, which leaves the sum as it is: it is never -0 starting from +0)
        const float* st = reinterpret_cast<const float*>(s_stage);
        const int mm = min(kUB, n - k0);
        for (int m0 = 0; m0 < mm; m0 += 16) {
          float v[16];
#pragma unroll
          for (int u = 0; u < 16; ++u) v[u] = st[(m0 + u) * kRC + lane];   // m0 + u < kUB
#pragma unroll
          for (int u = 0; u < 16; ++u) v[u] = m0 + u < mm ? v[u] : 0.f;
#pragma unroll
          for (int u = 0; u < 16; ++u) acc += (double)v[u];
        }
      }
      __syncthreads();
    }
    cnt += n;
  }
  if (lane < kRC) {
    const float v = cnt > 0 ? (float)(acc / (double)cnt)
                            : oa::bf16_to_f32(zr[(long)init_idx[c] * kRC + lane]) - colmean[row * kRC + lane];
    cent[((long)row * C + c) * kRC + lane] = v;
  }
  if (lane == 0 && cnt_out) cnt_out[row * C + c] = (float)cnt;
}

// ---------------------------------------------------------------------------------- sums + CSR
// One 1024-thread workgroup per query row: nb, clen (member counts), cstart (exclusive prefix)
// and mem, every cluster's members in position order (a stable counting sort of the row's ids).
// The row is taken 1024 positions at a time, wave w holding positions 64 w .. 64 w + 63 of the
// step.  A lane's equal-id lanes are the AND over the 8 id bits of that bit's ballot (or its
// complement); its rank among them orders it, their count goes to LDS per (cluster, wave), and
// a 16-lane scan per cluster turns the counts into the waves' starts in wave order -- so equal
// ids keep their position order inside a step, and the steps follow each other.
constexpr int kSortThreads = 1024;
constexpr int kSortStage = 32768;   // rows of at most this many ids are staged in LDS by the sort
constexpr int kSortWaves = kSortThreads / 64;
__global__ void __launch_bounds__(kSortThreads) csr_sort_kernel(int T, const uint8_t* asg8, long a8s, int C,
                                                               float* nb, int32_t* cstart, int32_t* clen,
                                                               int32_t* mem, long ms, int staged) {
  __shared__ int s_base[kMaxC];
  __shared__ int s_wcnt[kMaxC][kSortWaves];
  __shared__ __align__(16) uint8_t s_ids[kSortStage];   // the row's ids when staged (T <= kSortStage)
  const int row = blockIdx.x;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const uint8_t* ar = asg8 + (long)row * a8s;
  int32_t* mr = mem + (long)row * ms;
  for (int c = tid; c < kMaxC; c += kSortThreads) s_base[c] = 0;
  __syncthreads();
  if (staged) {
    // 16 ids per thread and load (rows 16-byte aligned, their stride a multiple of 16), kept in
    // LDS for the scatter pass
    const int T16 = (T + 15) / 16;
    for (int i = tid; i < T16; i += kSortThreads) {
      const uint4 w = reinterpret_cast<const uint4*>(ar)[i];
      *reinterpret_cast<uint4*>(s_ids + 16 * i) = w;
      const uint32_t q[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int b = 0; b < 16; ++b)
        if (16 * i + b < T) atomicAdd(&s_base[(q[b >> 2] >> (8 * (b & 3))) & 0xffu], 1);
    }
  } else {
    for (int t = tid; t < T; t += kSortThreads) atomicAdd(&s_base[ar[t]], 1);
  }
  __syncthreads();
  if (wave == 0) {
    int v[4], loc = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) { v[i] = s_base[lane * 4 + i]; loc += v[i]; }
    const int incl = oa::wave_incl_scan_i32(loc);
    int run = incl - loc;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = lane * 4 + i;
      if (c < C) {
        cstart[row * C + c] = run;
        clen[row * C + c] = v[i];
        if (nb) nb[row * C + c] = (float)v[i];
      }
      s_base[c] = run;
      run += v[i];
    }
  }
  const unsigned long long lower = (1ull << lane) - 1ull;
  for (int p0 = 0; p0 < T; p0 += kSortThreads) {
    for (int i = tid; i < kSortWaves * kMaxC; i += kSortThreads) (&s_wcnt[0][0])[i] = 0;
    __syncthreads();
    const int p = p0 + tid;
    const bool valid = p < T;
    const int x = valid ? (int)(staged ? s_ids[p] : ar[p]) : 0;
    unsigned long long m = __ballot(valid);
#pragma unroll
    for (int bit = 0; bit < 8; ++bit) {
      const unsigned long long bb = __ballot((x >> bit) & 1);
      m &= ((x >> bit) & 1) ? bb : ~bb;
    }
    const int rank = __popcll(m & lower);
    if (valid && rank == 0) s_wcnt[x][wave] = __popcll(m);
    __syncthreads();
    // the waves' starts per cluster: thread (c, w) of 16-lane groups, an inclusive scan over w
    for (int e = tid; e < C * kSortWaves; e += kSortThreads) {
      const int c = e >> 4, w = e & 15;
      const int v = s_wcnt[c][w];
      int incl = v;
      incl += __builtin_amdgcn_update_dpp(0, incl, 0x111, 0xf, 0xf, true);   // row_shr:1
      incl += __builtin_amdgcn_update_dpp(0, incl, 0x112, 0xf, 0xf, true);   // row_shr:2
      incl += __builtin_amdgcn_update_dpp(0, incl, 0x114, 0xf, 0xf, true);   // row_shr:4
      incl += __builtin_amdgcn_update_dpp(0, incl, 0x118, 0xf, 0xf, true);   // row_shr:8
      const int base = s_base[c];
      s_wcnt[c][w] = base + incl - v;
      if (w == kSortWaves - 1) s_base[c] = base + incl;
    }
    __syncthreads();
    if (valid) mr[s_wcnt[x][wave] + rank] = p;
    __syncthreads();
  }
}

// The fp64 sums of k, k*k and v of one (cluster, query row) by W waves: a lane holds 8 dims (16-byte
// loads) of the members its 16-lane group takes, every (4 W)-th of the list, 4 at a time in flight;
// the groups' sums are joined by two lane swaps and (W > 1) through LDS.  A group adds its members in
// position order.  Sums of up to 2^15 bf16 values are exact in fp64 where these span at most 2^30, of
// their squares (16 bits, twice the span) where the values span at most 2^11; beyond, the order shows in
// what rounding leaves, so that W follows from the row alone, not from the batch: the same row gives the
// same bits in every call.
// Bound by vector issue: 14 fp64 and conversion instructions per member and lane of 8 dims.  With a
// lane on 2 dims (4-byte loads, a row address per member for every lane) and one wave 32 sequences of
// 32767 tokens in 64 clusters took 2215 us, with 8 dims 2086 (by the counters 15 GB of the 17 GB gathered
// miss the L2s: waves of clusters of different sizes drift apart in position), with four waves 1782; one
// such sequence 206 us, and with four waves 78.
typedef uint32_t uint32x4a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float floatx4a4 __attribute__((ext_vector_type(4), aligned(4)));
template <int W>
__global__ void __launch_bounds__(64 * W) cluster_sums_kernel(const uint16_t* K, const uint16_t* V, long ksh,
                                                              long kst, int G, int C, const int32_t* cstart,
                                                              const int32_t* clen, float* Sk, float* Sk2,
                                                              float* Sv, const int32_t* mem, long ms,
                                                              float* nb) {
  constexpr int kGroups = 4 * W, U = 4;
  __shared__ double s_part[W > 1 ? W - 1 : 1][3][kD];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int grp = threadIdx.x >> 4, d0 = 8 * (lane & 15);
  // every token's K and V rows are read once per query row of its KV row (each query row has its
  // own clusters).  The G * C workgroups of a KV row run on one XCD, its query rows interleaved,
  // so that they walk the KV row's positions together and the later reads of a row hit that
  // XCD's L2 (workgroups are dealt to the 8 XCDs in turn)
  int c, row;
  {
    const int b = blockIdx.x, rows = gridDim.x / C, kv_rows = rows / G;
    if (kv_rows % 8 == 0) {
      const int k = b >> 3, per = G * C;
      const int j = k % per;
      row = ((k / per) * 8 + (b & 7)) * G + j % G;
      c = j / G;
    } else {
      row = b / C;
      c = b % C;
    }
  }
  const uint16_t* kr = K + (long)(row / G) * ksh + d0;
  const uint16_t* vr = V + (long)(row / G) * ksh + d0;
  const int32_t* ml = mem + (long)row * ms + cstart[row * C + c];
  const int cl = clen[row * C + c];
  if (nb && threadIdx.x == 0) nb[row * C + c] = (float)cl;   // (when the sort did not write it)
  double ks[8], qs[8], vs[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) ks[e] = qs[e] = vs[e] = 0.0;
  // this group's members grp, grp + kGroups, ...: U positions requested a batch ahead of their rows
  int pos[U];
  auto next = [&](int m0) {
#pragma unroll
    for (int u = 0; u < U; ++u) pos[u] = ml[min(m0 + u * kGroups, cl - 1)];
  };
  if (cl > 0) next(grp);
  for (int m0 = grp; m0 < cl; m0 += U * kGroups) {
    uint32x4a4 kw[U], vw[U];                     // (K, V rows are 4-byte aligned)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const long off = (long)pos[u] * kst;
      kw[u] = *reinterpret_cast<const uint32x4a4*>(kr + off);
      vw[u] = *reinterpret_cast<const uint32x4a4*>(vr + off);
    }
    next(m0 + U * kGroups);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (m0 + u * kGroups < cl) {
        float k[8], v[8];
        oa::unpack8(make_uint4(kw[u][0], kw[u][1], kw[u][2], kw[u][3]), k);
        oa::unpack8(make_uint4(vw[u][0], vw[u][1], vw[u][2], vw[u][3]), v);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const double x = (double)k[e];
          ks[e] += x;
          qs[e] = fma(x, x, qs[e]);                // (the square of a bf16 value is exact)
          vs[e] += (double)v[e];
        }
      }
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    ks[e] = oa::swap32_sum(oa::swap16_sum(ks[e]));
    qs[e] = oa::swap32_sum(oa::swap16_sum(qs[e]));
    vs[e] = oa::swap32_sum(oa::swap16_sum(vs[e]));
  }
  if (W > 1) {
    if (wave > 0 && lane < 16) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        s_part[wave - 1][0][d0 + e] = ks[e];
        s_part[wave - 1][1][d0 + e] = qs[e];
        s_part[wave - 1][2][d0 + e] = vs[e];
      }
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < W - 1; ++w)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        ks[e] += s_part[w][0][d0 + e];
        qs[e] += s_part[w][1][d0 + e];
        vs[e] += s_part[w][2][d0 + e];
      }
  }
  // lane group 0 writes Sk, 1 Sk2, 2 Sv (every group holds all three)
  if (lane >= 48) return;
  float* out = (lane < 16 ? Sk : lane < 32 ? Sk2 : Sv) + ((long)row * C + c) * kD + d0;
  floatx4a4 o[2];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e / 4][e % 4] = (float)(lane < 16 ? ks[e] : lane < 32 ? qs[e] : vs[e]);
  reinterpret_cast<floatx4a4*>(out)[0] = o[0];
  reinterpret_cast<floatx4a4*>(out)[1] = o[1];
}

}  // namespace

extern "C" int oa_qgs_codes(const void* K, long k_stride_h, long k_stride_t, int kv_rows, int T,
                            const float* U, int8_t* codes, long codes_stride_h, float* scale,
                            uint32_t* amax_ws, float* zc_ws, void* stream) {
  if (kv_rows <= 0 || T <= 0 || !K || !U || !codes || !scale || !amax_ws || k_stride_t < kD ||
      k_stride_t % 8 || k_stride_h % 8 || codes_stride_h < (long)T * kRQ || codes_stride_h % 16 ||
      (reinterpret_cast<uintptr_t>(K) & 15) || (reinterpret_cast<uintptr_t>(codes) & 15) ||
      (reinterpret_cast<uintptr_t>(zc_ws) & 15))
    return OA_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  const uint16_t* k = reinterpret_cast<const uint16_t*>(K);
  hipLaunchKernelGGL(clear_u32_kernel, dim3(std::min(64, (kv_rows * kRQ + 63) / 64)), dim3(64), 0, s,
                     amax_ws, kv_rows * kRQ);
  const dim3 grid((T + kCodeThreads - 1) / kCodeThreads, kv_rows);
  // tiles per wave: eight spread the block's load of U; fewer where the grid would leave a SIMD with
  // less than four waves
  const int ntiles = (T + 63) / 64;
  const int tiles = (int)std::min<long>(kZcTiles, std::max<long>(1, (long)ntiles * kv_rows / 4096));
  const int per = kCodeThreads / 64 * tiles;
  hipLaunchKernelGGL(codes_amax_kernel, dim3((ntiles + per - 1) / per, kv_rows), dim3(kCodeThreads), 0, s, k,
                     k_stride_h, k_stride_t, T, U, amax_ws, zc_ws, tiles);
  hipLaunchKernelGGL(codes_write_kernel, grid, dim3(kCodeThreads), 0, s, k, k_stride_h, k_stride_t, T, U,
                     amax_ws, codes, codes_stride_h, scale, zc_ws);
  return OA_LAUNCH_STATUS();
}

static int qgc_project(const void* K, long k_stride_h, long k_stride_t, int rows, int G, int T,
                              const void* W, float* zP, long zp_stride, float* colmean,
                              double* tile_ws, uint16_t* zraw_out, uint32_t* wmax, uint32_t* zmax, void* stream) {
  if (rows <= 0 || G <= 0 || rows % G || T <= 0 || !K || !W || (!zP && !zraw_out) || !colmean ||
      !tile_ws || k_stride_t < kD || k_stride_t % 8 || k_stride_h % 8 || zp_stride < (long)T * kRC ||
      zp_stride % 4 || (reinterpret_cast<uintptr_t>(K) & 15) || (reinterpret_cast<uintptr_t>(zP) & 15) ||
      (reinterpret_cast<uintptr_t>(zraw_out) & 15) || (zraw_out && zp_stride % 8))
    return OA_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  const int ntiles = (T + 63) / 64;
  const int nx = (ntiles + kProjTiles - 1) / kProjTiles;
  if (G == 4)   // a KV row's four query rows per wave: each K block loaded once for all four
    hipLaunchKernelGGL(qgc_project_kernel<4>, dim3(nx, rows / 4), dim3(64), 0, s,
                       reinterpret_cast<const uint16_t*>(K), k_stride_h, k_stride_t, G, T,
                       reinterpret_cast<const uint16_t*>(W), zP, zp_stride, zraw_out, tile_ws, ntiles, wmax);
  else
    hipLaunchKernelGGL(qgc_project_kernel<1>, dim3(nx, rows), dim3(64), 0, s,
                       reinterpret_cast<const uint16_t*>(K), k_stride_h, k_stride_t, G, T,
                       reinterpret_cast<const uint16_t*>(W), zP, zp_stride, zraw_out, tile_ws, ntiles, wmax);
  hipLaunchKernelGGL(qgc_colmean_kernel, dim3(rows), dim3(64), 0, s, T, tile_ws, ntiles, colmean,
                     wmax, nx, zmax);
  if (zP) {
    const int nb = std::min(16, (T * (kRC / 4) + 255) / 256);
    hipLaunchKernelGGL(qgc_center_kernel, dim3(nb, rows), dim3(256), 0, s, zP, zp_stride, T, colmean);
  }
  return OA_LAUNCH_STATUS();
}

extern "C" int oa_qgc_project(const void* K, long k_stride_h, long k_stride_t, int rows, int G, int T,
                              const void* W, float* zP, long zp_stride, float* colmean, double* tile_ws,
                              uint16_t* zraw_out, void* stream) {
  return qgc_project(K, k_stride_h, k_stride_t, rows, G, T, W, zP, zp_stride, colmean, tile_ws, zraw_out, nullptr,
                     nullptr, stream);
}

extern "C" int oa_qgc_project_max(const void* K, long k_stride_h, long k_stride_t, int rows, int G, int T,
                                  const void* W, float* zP, long zp_stride, float* colmean, double* tile_ws,
                                  uint16_t* zraw_out, uint32_t* max_ws, uint32_t* zmax, void* stream) {
  if (!max_ws || !zmax) return OA_EINVAL;
  return qgc_project(K, k_stride_h, k_stride_t, rows, G, T, W, zP, zp_stride, colmean, tile_ws, zraw_out, max_ws,
                     zmax, stream);
}

// tiles per wave: up to eight spread the centroids' staging; fewer, a power of two so that workgroups
// share a segment evenly, where the grid would not give every SIMD eight waves
static int asg_tiles_per_wave(int rows, int T) {
  const long want = (long)((T + 63) / 64) * rows / 8192;
  return want >= kAsgMaxTiles ? kAsgMaxTiles : want >= 4 ? 4 : want >= 2 ? 2 : 1;
}

template <bool ACC>
static void launch_assign(const uint16_t* zraw, const float* colmean, long z_stride, int rows, int T,
                          const float* cent, int C, int32_t* asg, long asg_stride, uint8_t* asg8,
                          long asg8_stride, int tpw, LloydArgs ll, hipStream_t stream) {
  const int ntiles = (T + 63) / 64, per = kAsgThreads / 64 * tpw;
  const dim3 grid((ntiles + per - 1) / per, rows), block(kAsgThreads);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, stream, zraw, colmean, z_stride, T, cent, C, asg, asg_stride, asg8,
                       asg8_stride, tpw, ll);
  };
  // the centroid blocks a wave holds: the least of these that covers C (padding ranks below)
  const int cb = (C + 15) / 16;
  if (cb <= 1) launch(kmeans_assign_kernel<1, ACC>);
  else if (cb <= 2) launch(kmeans_assign_kernel<2, ACC>);
  else if (cb <= 4) launch(kmeans_assign_kernel<4, ACC>);
  else if (cb <= 8) launch(kmeans_assign_kernel<8, ACC>);
  else if (cb <= 12) launch(kmeans_assign_kernel<12, ACC>);
  else launch(kmeans_assign_kernel<16, ACC>);
}

extern "C" int oa_kmeans_assign(const uint16_t* zraw, const float* colmean, long z_stride, int rows,
                                int T, const float* cent, int C, int32_t* asg, long asg_stride,
                                uint8_t* asg8, long asg8_stride, void* stream) {
  if (rows <= 0 || T <= 0 || C <= 0 || C > kMaxC || !zraw || !colmean || !cent || !asg || !asg8 ||
      z_stride < (long)T * kRC || z_stride % 4 || asg_stride < T || asg8_stride < T ||
      (reinterpret_cast<uintptr_t>(zraw) & 7))
    return OA_EINVAL;
  const int tpw = asg_tiles_per_wave(rows, T);
  launch_assign<false>(zraw, colmean, z_stride, rows, T, cent, C, asg, asg_stride, asg8, asg8_stride, tpw,
                       LloydArgs{}, (hipStream_t)stream);
  return OA_LAUNCH_STATUS();
}

// a whole Lloyd iteration: the workspace holds the sums, counts and flags of each of the grid's
// workgroups, each row's units and bound words
static int step_groups(int rows, int T) {
  const int per = kAsgThreads / 64 * asg_tiles_per_wave(rows, T);
  return ((T + 63) / 64 + per - 1) / per;
}

extern "C" long oa_kmeans_step_ws(int rows, int T, int C) {
  if (rows <= 0 || T <= 0 || C <= 0 || C > kMaxC) return OA_EINVAL;
  return (long)rows * (step_groups(rows, T) * (long)C * (kRC * 8 + 8) + kRC * 8);
}

// zmax NULL: the bound words are formed here
extern "C" int oa_kmeans_step_max(const uint16_t* zraw, const float* colmean, const uint32_t* zmax, long z_stride,
                                  int rows, int T, float* cent, int C, const int32_t* init_idx, int32_t* asg,
                                  long asg_stride, uint8_t* asg8, long asg8_stride, void* ws, long ws_bytes,
                                  void* stream) {
  if (rows <= 0 || T <= 0 || C <= 0 || C > kMaxC || !zraw || !colmean || !cent || !init_idx || !ws ||
      z_stride < (long)T * kRC || z_stride % 4 || (!asg != !asg8) || (asg && (asg_stride < T || asg8_stride < T)) ||
      (reinterpret_cast<uintptr_t>(zraw) & 7) || (reinterpret_cast<uintptr_t>(ws) & 7) ||
      ws_bytes < oa_kmeans_step_ws(rows, T, C))
    return OA_EINVAL;
  const int nwg = step_groups(rows, T), tpw = asg_tiles_per_wave(rows, T);
  hipStream_t s = (hipStream_t)stream;
  LloydArgs ll;
  ll.part = static_cast<unsigned long long*>(ws);
  ll.pcnt = reinterpret_cast<int32_t*>(ll.part + (long)rows * nwg * C * kRC);
  ll.pbad = reinterpret_cast<uint32_t*>(ll.pcnt + (long)rows * nwg * C);
  ll.pexp = reinterpret_cast<int32_t*>(ll.pbad + (long)rows * nwg * C);
  ll.zmax = zmax;
  if (!zmax) {
    uint32_t* own = reinterpret_cast<uint32_t*>(ll.pexp + (long)rows * kRC);
    hipLaunchKernelGGL(column_max_kernel, dim3(rows), dim3(256), 0, s, zraw, z_stride, T, own);
    ll.zmax = own;
  }
  launch_assign<true>(zraw, colmean, z_stride, rows, T, cent, C, asg, asg_stride, asg8, asg8_stride, tpw, ll, s);
  hipLaunchKernelGGL(kmeans_mean_kernel, dim3((C * kRC + 255) / 256, rows), dim3(256), 0, s, ll, nwg,
                     kAsgMaxTiles / tpw, C, zraw, colmean, z_stride, init_idx, cent);
  return OA_LAUNCH_STATUS();
}

extern "C" int oa_kmeans_step(const uint16_t* zraw, const float* colmean, long z_stride, int rows, int T,
                              float* cent, int C, const int32_t* init_idx, int32_t* asg, long asg_stride,
                              uint8_t* asg8, long asg8_stride, void* ws, long ws_bytes, void* stream) {
  return oa_kmeans_step_max(zraw, colmean, nullptr, z_stride, rows, T, cent, C, init_idx, asg, asg_stride, asg8,
                            asg8_stride, ws, ws_bytes, stream);
}

// the sort stages a row's ids in LDS with 16-byte loads when the row fits and its rows are
// 16-byte aligned with a stride that is a multiple of 16 (it then reads up to the next multiple of
// 16 of T, inside the row's stride)
static int sort_staged(int T, const uint8_t* asg8, long asg8_stride) {
  return T <= kSortStage && asg8_stride % 16 == 0 && (reinterpret_cast<uintptr_t>(asg8) & 15) == 0;
}

extern "C" int oa_kmeans_update(const uint16_t* zraw, const float* colmean, long z_stride, int rows,
                                int T, const uint8_t* asg8, long asg8_stride, int C,
                                const int32_t* init_idx, float* cent, float* cnt_out, int32_t* mem_ws,
                                long mem_stride, int32_t* cstart_ws, int32_t* clen_ws, void* stream) {
  if (rows <= 0 || T <= 0 || C <= 0 || C > kMaxC || !zraw || !colmean || !asg8 || !init_idx || !cent ||
      !mem_ws || !cstart_ws || !clen_ws || mem_stride < T || z_stride < (long)T * kRC ||
      z_stride % 4 || (reinterpret_cast<uintptr_t>(zraw) & 7) || asg8_stride < T)
    return OA_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(csr_sort_kernel, dim3(rows), dim3(kSortThreads), 0, s, T, asg8, asg8_stride, C,
                     nullptr, cstart_ws, clen_ws, mem_ws, mem_stride, sort_staged(T, asg8, asg8_stride));
  hipLaunchKernelGGL(kmeans_update_kernel, dim3(C * rows), dim3(64), 0, s, zraw, colmean, z_stride, C,
                     mem_ws, mem_stride, cstart_ws, clen_ws, init_idx, cent, cnt_out);
  return OA_LAUNCH_STATUS();
}

// Waves per (cluster, row) by a row's mean members, whatever the batch: four from 256 up, where a
// cluster of several times the mean holds a wave for long, else one (four waves' joins cost more than
// they save).  On built indexes, one wave against four: 32, 8 and 1 sequences of 32767 tokens in 64
// clusters 2123 / 1799, 611 / 477 and 146 / 81 us; in 192 clusters (170 members) 1702 / 2020, 461 / 518
// and 87 / 72; 8 of 4096 in 256 clusters 96 / 247.
static void launch_sums(const void* K, const void* V, long ksh, long kst, int rows, int G, int T, int C,
                        const int32_t* cstart, const int32_t* clen, float* Sk, float* Sk2, float* Sv,
                        const int32_t* mem, long ms, float* nb, hipStream_t s) {
  const uint16_t* k = reinterpret_cast<const uint16_t*>(K);
  const uint16_t* v = reinterpret_cast<const uint16_t*>(V);
  if (T < 256L * C)
    hipLaunchKernelGGL(cluster_sums_kernel<1>, dim3(C * rows), dim3(64), 0, s, k, v, ksh, kst, G, C, cstart,
                       clen, Sk, Sk2, Sv, mem, ms, nb);
  else
    hipLaunchKernelGGL(cluster_sums_kernel<4>, dim3(C * rows), dim3(256), 0, s, k, v, ksh, kst, G, C, cstart,
                       clen, Sk, Sk2, Sv, mem, ms, nb);
}

extern "C" int oa_cluster_build(const void* K, const void* V, long kv_stride_h, long kv_stride_t, int rows,
                                int G, int T, const uint8_t* asg8, long asg8_stride, int C, float* nb,
                                float* Sk, float* Sk2, float* Sv, int32_t* mem, long mem_stride,
                                int32_t* cstart, int32_t* clen, void* stream) {
  if (rows <= 0 || G <= 0 || rows % G || T <= 0 || C <= 0 || C > kMaxC || !K || !V || !asg8 || !nb ||
      !Sk || !Sk2 || !Sv || !mem || !cstart || !clen || kv_stride_t < kD || kv_stride_t % 2 ||
      kv_stride_h % 2 || asg8_stride < T || mem_stride < T || (reinterpret_cast<uintptr_t>(K) & 3) ||
      (reinterpret_cast<uintptr_t>(V) & 3))
    return OA_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(csr_sort_kernel, dim3(rows), dim3(kSortThreads), 0, s, T, asg8, asg8_stride, C, nb,
                     cstart, clen, mem, mem_stride, sort_staged(T, asg8, asg8_stride));
  launch_sums(K, V, kv_stride_h, kv_stride_t, rows, G, T, C, cstart, clen, Sk, Sk2, Sv, mem, mem_stride, nullptr, s);
  return OA_LAUNCH_STATUS();
}

extern "C" int oa_cluster_sums(const void* K, const void* V, long kv_stride_h, long kv_stride_t, int rows,
                               int G, int T, int C, float* nb, float* Sk, float* Sk2, float* Sv,
                               const int32_t* mem, long mem_stride, const int32_t* cstart,
                               const int32_t* clen, void* stream) {
  if (rows <= 0 || G <= 0 || rows % G || T <= 0 || C <= 0 || C > kMaxC || !K || !V || !nb || !Sk ||
      !Sk2 || !Sv || !mem || !cstart || !clen || kv_stride_t < kD || kv_stride_t % 2 ||
      kv_stride_h % 2 || mem_stride < T || (reinterpret_cast<uintptr_t>(K) & 3) ||
      (reinterpret_cast<uintptr_t>(V) & 3))
    return OA_EINVAL;
  launch_sums(K, V, kv_stride_h, kv_stride_t, rows, G, T, C, cstart, clen, Sk, Sk2, Sv, mem, mem_stride, nb,
              (hipStream_t)stream);
  return OA_LAUNCH_STATUS();
}
