// Dense causal attention of a prompt on the bf16 matrix cores (the prefill branch of the deployed
// attention hook, graph_runner.py:472-475): every position attends itself and what is before it,
// fp32 scores and softmax, bf16 weights into the value product, fp32 sums.
//
// One workgroup of four waves takes 32 positions of one KV head, wave w its query head w: the four
// waves share every key and value tile and the causal limit.  Two workgroups run on a compute unit,
// two waves per SIMD: one wave alone issues only every second slot (a wave of 64 queries, which would
// halve the LDS reads per product, ran at 861 TFLOP/s alone on its SIMD).
//   scores   S^T = K Q^T by v_mfma_f32_32x32x16_bf16: a lane holds 16 of 32 keys' scores of one query,
//            so that a row maximum or sum is 16 registers and one lane swap;
//   values   O^T = V^T P^T: a lane's weights are the B operand as they stand once the keys of the A
//            operand are taken in the order the scores left them (4 h + 0..3, 8 + 4 h + 0..3 for lane
//            half h); V^T comes out of the row-major tile by the LDS transpose reads.
// The loop is a pipeline over 32-key tiles: iteration i issues the products of S(i + 1) and of
// O += V(i - 1) P(i - 1) interleaved with the softmax of S(i), which none of them needs.  O^T is
// rescaled only in tiles where a query of the wave meets a new maximum (about 1 in 7 at 32768
// positions).  Letting scores pass the maximum by up to 2^8 first would save 4% and lose precision: the
// largest weight is then not exactly 1 in bf16 (errors against fp64 over rows near a stored key, 1024 /
// 32768 positions: 1.81e-3 / 2.13e-3 that way, 1.71e-3 / 1.987e-3 as it is, 1.71e-3 / 1.994e-3 for
// the library kernel it replaces).
// Tiles: rows of 256 bytes whose 16-byte chunks c lie at c ^ f(row), f = (row % 4) * 4 + row / 4 % 4:
// 16 rows read at one chunk (K) and 4 rows read at four chunks (V^T) both meet every bank once.
//
// Bound by vector issue beside the products: 16 exponentials and about 70 other vector instructions per
// 32 x 32 scores of a wave against 512 matrix cycles.  32768 positions, 32 heads: 9.2 ms, 953 TFLOP/s
// (a large bf16 product reaches 1326 on this card); the library kernel it replaces took 16.9 ms and
// another 0.34 ms to expand the KV heads.
#include <cfloat>
#include <type_traits>

#include "oa_common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef unsigned int uint4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4v lds_short4v;

constexpr int kThreads = 256;
constexpr int kQ = 32;                   // queries per wave
constexpr int kKeys = 32;                // keys per tile
constexpr int kRowB = OA_D * 2;          // bytes per tile row
constexpr int kTileB = kKeys * kRowB;    // 8 KB
constexpr int kAhead = 2;              // steps whose LDS operands are requested ahead (1, 2, 3 measured alike)
constexpr float kLog2e = 1.4426950408889634f;

struct PrefillArgs {
  const uint16_t* q; long q_sh, q_st;
  const uint16_t* k; long k_sh, k_st;
  const uint16_t* v; long v_sh, v_st;
  uint16_t* out; long o_sh, o_st;
  int T, kv_heads, ntiles;
  float c;                               // softmax scale * log2 e
};

__device__ __forceinline__ float16v mfma(bf16x8 a, bf16x8 b, float16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  const f32x2 x = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2));
}

struct Weights {                         // P^T of a 32-key tile, 16 keys per operand
  uint4v w[2];
};

__global__ void __launch_bounds__(kThreads, 2) prefill_attn_kernel(PrefillArgs a) {
  __shared__ __align__(16) char s_t[4 * kTileB];          // K even, K odd, V even, V odd tiles
  char* const s_k = s_t;
  char* const s_v = s_t + 2 * kTileB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n32 = lane & 31, h = lane >> 5;
  // the longest rows first; consecutive workgroups (XCDs in turn) on different KV heads, so that an
  // XCD's L2 serves few heads' tiles
  const int kvh = blockIdx.x % a.kv_heads;
  const int q0 = (a.ntiles - 1 - (int)blockIdx.x / a.kv_heads) * kQ;
  const int T = a.T;

  // staging: 16-byte chunks tid and tid + 256 of a tile (rows of 16 chunks); row r + 16 has row r's f
  const int srow = tid >> 4, sc = tid & 15;
  auto fsw = [](int r) { return ((r & 3) << 2) | ((r >> 2) & 3); };
  const int sdst = srow * kRowB + ((sc ^ fsw(srow)) << 4);
  // a tile's rows from a scalar base and fixed 32-bit offsets; rows past the last one read it again
  // (their keys are masked and their weights 0)
  const char* const kb = reinterpret_cast<const char*>(a.k + (long)kvh * a.k_sh);
  const char* const vb = reinterpret_cast<const char*>(a.v + (long)kvh * a.v_sh);
  const uint32_t koff = (uint32_t)srow * (uint32_t)a.k_st * 2 + 16 * sc, koff16 = koff + 32 * (uint32_t)a.k_st;
  const uint32_t voff = (uint32_t)srow * (uint32_t)a.v_st * 2 + 16 * sc, voff16 = voff + 32 * (uint32_t)a.v_st;
  uint4v ks0, ks1, vs0, vs1;
  auto fetch = [&](uint4v& x0, uint4v& x1, const char* base, long st, uint32_t o0, uint32_t o16, int tile) {
    if ((tile + 1) * kKeys <= T) {
      const char* p = base + (long)tile * kKeys * st * 2;
      x0 = *reinterpret_cast<const uint4v*>(p + o0);
      x1 = *reinterpret_cast<const uint4v*>(p + o16);
    } else {
      const int r = tile * kKeys + srow;
      x0 = *reinterpret_cast<const uint4v*>(base + (long)min(r, T - 1) * st * 2 + 16 * sc);
      x1 = *reinterpret_cast<const uint4v*>(base + (long)min(r + 16, T - 1) * st * 2 + 16 * sc);
    }
  };
  auto fetch_k = [&](int tile) { fetch(ks0, ks1, kb, a.k_st, koff, koff16, tile); };
  auto fetch_v = [&](int tile) { fetch(vs0, vs1, vb, a.v_st, voff, voff16, tile); };
  auto put = [&](char* tile, uint4v x0, uint4v x1) {
    *reinterpret_cast<uint4v*>(tile + sdst) = x0;
    *reinterpret_cast<uint4v*>(tile + sdst + 16 * kRowB) = x1;
  };

  // operand addresses (bytes in a tile)
  const int kad = n32 * kRowB + ((h ^ fsw(n32)) << 4);                     // ^ (step << 5)
  const int lr = (lane & 15) >> 2, lc = lane & 3, dsub = (lane >> 4) & 1;
  const int vad = (4 * h + lr) * kRowB + ((((lr << 2) | ((dsub * 2 + (lc >> 1)) ^ h)) << 4) | ((lc & 1) << 3));
  auto key_op = [&](const char* tile, int step) {
    return *reinterpret_cast<const bf16x8*>(tile + (kad ^ (step << 5)));
  };
  // V^T of d block db (32 dims) and keys 16 kk..: two transposed reads of 4 keys
  auto val_op = [&](char* tile, int db, int kk) {
    const int ad = vad ^ (db << 6);
    const short4v x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4v*)(tile + ad + kk * 16 * kRowB));
    const short4v y = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_short4v*)(tile + (ad ^ 32) + kk * 16 * kRowB + 8 * kRowB));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  // this wave's queries: B operands of every 16 dims
  bf16x8 Q[8];
  {
    const uint16_t* qr =
        a.q + (long)(kvh * 4 + wave) * a.q_sh + (long)min(q0 + n32, T - 1) * a.q_st + 8 * h;
#pragma unroll
    for (int s = 0; s < 8; ++s) Q[s] = *reinterpret_cast<const bf16x8*>(qr + 16 * s);
  }
  const int n = q0 / kKeys + 1;          // tiles; the last holds the diagonal
  fetch_k(0);
  put(s_k, ks0, ks1);
  fetch_k(1);
  put(s_k + kTileB, ks0, ks1);
  put(s_v + kTileB, uint4v(0u), uint4v(0u));               // V(-1): its weights are 0
  fetch_k(2);
  fetch_v(0);
  oa::lds_barrier();

  float16v O[4], S0 = float16v(0.f), S1;
  Weights P0, P1;
  P1.w[0] = P1.w[1] = uint4v(0u);
#pragma unroll
  for (int d = 0; d < 4; ++d) O[d] = float16v(0.f);
#pragma unroll
  for (int s = 0; s < 8; ++s) S0 = mfma(key_op(s_k, s), Q[s], S0);
  float m = -FLT_MAX, l = 0.f;           // running maximum (scaled by c) and sum of the lane's keys
  bool big = false;                      // a lane's maximum is past 2^24 (uniform)
  oa::lds_barrier();                     // K(0) has been read: its place takes K(2)

  // iteration i (parity odd = i & 1): K(i + 1), V(i - 1) are in the other parity's tiles
  auto body = [&](auto mask_c, auto odd_c, int i, float16v& S, float16v& Sn, const Weights& Pp, Weights& Pn) {
    constexpr bool MASK = decltype(mask_c)::value;
    constexpr int kOdd = decltype(odd_c)::value;
    char* const kt = s_k + (1 - kOdd) * kTileB;
    char* const vt = s_v + (1 - kOdd) * kTileB;
    put(s_k + kOdd * kTileB, ks0, ks1);                               // K(i + 2)
    put(s_v + kOdd * kTileB, vs0, vs1);                               // V(i)
    fetch_k(i + 3);
    fetch_v(i + 1);
    float mx = -INFINITY, alpha = 1.f, p0 = 0.f;
    bool moved = false;
    Sn = float16v(0.f);
    bf16x8 kop[8], vop[8];               // (kAhead steps' operands in flight)
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
      kop[s] = key_op(kt, s);
      vop[s] = val_op(vt, s >> 1, s & 1);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      if (s + kAhead < 8) {
        kop[s + kAhead] = key_op(kt, s + kAhead);
        vop[s + kAhead] = val_op(vt, (s + kAhead) >> 1, (s + kAhead) & 1);
      }
      Sn = mfma(kop[s], Q[s], Sn);
      O[s >> 1] = mfma(vop[s], __builtin_bit_cast(bf16x8, Pp.w[s & 1]), O[s >> 1]);
      if (s == 0) {                      // the tile's maximum
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          // (a masked tile's scores are scaled here: -inf times a scale of 0 would be NaN)
          if (MASK) S[r] = i * kKeys + 8 * (r >> 2) + 4 * h + (r & 3) <= q0 + n32 ? S[r] * a.c : -INFINITY;
          mx = fmaxf(mx, S[r]);
        }
      } else if (s == 1) {
        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1])) * (MASK ? 1.f : a.c);
        moved = __any(mx > m);
        if (moved) {
          const float mn = fmaxf(m, mx);
          alpha = __builtin_amdgcn_exp2f(m - mn);
          l *= alpha;
          m = mn;
          // m rounds S c, so that the fma below leaves up to half its last place: past 2^24 more than
          // the exponential should see, and an infinity in time.  There S c is rounded first, as m is
          big = __any(fabsf(m) >= 16777216.f);
        }
        if (!MASK && big) {
#pragma unroll
          for (int r = 0; r < 16; ++r) S[r] *= a.c;
        }
      } else {
#pragma unroll
        for (int r = (s - 2) * 16 / 6; r < (s - 1) * 16 / 6; ++r) {
          const float p1 = __builtin_amdgcn_exp2f(MASK ? S[r] - m : fmaf(S[r], big ? 1.f : a.c, -m));
          l += p1;
          if (r & 1) {                   // (pinned here: left alone they all sink below the products)
            uint32_t w = pack2(p0, p1);
            asm volatile("" : "+v"(w));
            Pn.w[r >> 3][(r & 7) >> 1] = w;
          }
          p0 = p1;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (moved) {                         // (after O += V(i - 1) P(i - 1), whose weights had the old maximum)
#pragma unroll
      for (int d = 0; d < 4; ++d) O[d] *= alpha;
    }
    oa::lds_barrier();
  };
  typedef std::integral_constant<int, 0> even_t;
  typedef std::integral_constant<int, 1> odd_t;
  auto finish = [&](int parity, const Weights& P) {        // V(n - 1) P(n - 1)
#pragma unroll
    for (int s = 0; s < 8; ++s)
      O[s >> 1] = mfma(val_op(s_v + parity * kTileB, s >> 1, s & 1), __builtin_bit_cast(bf16x8, P.w[s & 1]), O[s >> 1]);
  };

  int i = 0;
#pragma unroll 1
  for (; i + 2 < n; i += 2) {
    body(std::false_type(), even_t(), i, S0, S1, P1, P0);
    body(std::false_type(), odd_t(), i + 1, S1, S0, P0, P1);
  }
  if (n & 1) {
    body(std::true_type(), even_t(), i, S0, S1, P1, P0);
    finish(0, P0);
  } else {
    body(std::false_type(), even_t(), i, S0, S1, P1, P0);
    body(std::true_type(), odd_t(), i + 1, S1, S0, P0, P1);
    finish(1, P1);
  }

  const auto lx = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
  const float inv = 1.f / (__uint_as_float(lx[0]) + __uint_as_float(lx[1]));
  const int t = q0 + n32;
  if (t >= T) return;
  uint16_t* o = a.out + (long)(kvh * 4 + wave) * a.o_sh + (long)t * a.o_st + 4 * h;
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<uint2*>(o + 32 * d + 8 * g) = make_uint2(
          pack2(O[d][4 * g] * inv, O[d][4 * g + 1] * inv), pack2(O[d][4 * g + 2] * inv, O[d][4 * g + 3] * inv));
}

}  // namespace

extern "C" int oa_prefill_attn(const void* q, long q_stride_h, long q_stride_t, const void* k, long k_stride_h,
                               long k_stride_t, const void* v, long v_stride_h, long v_stride_t, int heads,
                               int kv_heads, int T, int head_dim, float sm_scale, void* out, long out_stride_h,
                               long out_stride_t, void* stream) {
  auto bad = [](const void* p, long sh, long st, int align) {
    return !p || (reinterpret_cast<uintptr_t>(p) & (2 * align - 1)) || sh % align || st % align || st < OA_D;
  };
  if (head_dim != OA_D || kv_heads <= 0 || heads != 4 * kv_heads || T <= 0 || T > (1 << 24) || !(sm_scale >= 0.f) ||
      bad(q, q_stride_h, q_stride_t, 8) || bad(k, k_stride_h, k_stride_t, 8) ||
      bad(v, v_stride_h, v_stride_t, 8) || bad(out, out_stride_h, out_stride_t, 4))
    return OA_EINVAL;
  PrefillArgs a;
  a.q = (const uint16_t*)q; a.q_sh = q_stride_h; a.q_st = q_stride_t;
  a.k = (const uint16_t*)k; a.k_sh = k_stride_h; a.k_st = k_stride_t;
  a.v = (const uint16_t*)v; a.v_sh = v_stride_h; a.v_st = v_stride_t;
  a.out = (uint16_t*)out; a.o_sh = out_stride_h; a.o_st = out_stride_t;
  a.T = T; a.kv_heads = kv_heads; a.ntiles = (T + kQ - 1) / kQ;
  a.c = sm_scale * kLog2e;
  if ((long)a.ntiles * kv_heads > 0x7fffffffL || k_stride_t > (1L << 24) || v_stride_t > (1L << 24)) return OA_EINVAL;
  hipLaunchKernelGGL(prefill_attn_kernel, dim3(a.ntiles * kv_heads), dim3(kThreads), 0, (hipStream_t)stream, a);
  return OA_LAUNCH_STATUS();
}
