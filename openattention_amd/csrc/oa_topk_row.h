// Exact top-k of one query-head row by one wave, register variant (rows of at most 64 * TPL
// score tiles, k <= KR), shared by the top-k launch and the small-batch top-k + gate + fill launch.
//
// Reference semantics: StaticTopKMasker.add_mask (static_top_k.py:221-262: top-k over positions
// not already taken by the sink/local maskers), deployed select kernel graph_runner.py:100-159;
// ties break to the lower position (graph_runner.py:127-151).
#pragma once
#include "oa_common.h"
#include "oa_score.h"

namespace oa_sel {

constexpr int GQ = 4;    // query heads per KV head (limb rows = GQ * 4 = 16)
constexpr int kMaxTop = 64;

__device__ __forceinline__ unsigned long long tile_key(float v, int t) {
  return ((unsigned long long)oa::float_key(v) << 32) | (0xffffffffu - (unsigned)t);
}

// With HEADS the score rows hold 16-bit key heads: the candidate tiles' exact scores are
// recomputed from the codes (oa::qgs_score, the scan's arithmetic), and the selected tokens'
// heads are set to that of -inf.
struct Rescore {
  const int8_t* codes; long lmax;   // (BH, Lmax, 32)
  const int8_t* limbs;              // (BH, 16, 32)
  const int* fexp;                  // (R,)
  int qsh = 0;                      // question rows per KV row (oa_common.h)
};

template <bool HEADS>
__device__ __forceinline__ void mark_selected(void* Sv, long s_stride, int row, int pos) {
  if (HEADS) static_cast<uint16_t*>(Sv)[(long)row * s_stride + pos] = oa::kNegInfHead;
  else static_cast<float*>(Sv)[(long)row * s_stride + pos] = -INFINITY;
}
// the row's limb words (HEADS only) and 2^-F
template <bool HEADS>
__device__ __forceinline__ double load_limbs(const Rescore& rs, int row, int* lw) {
  if (!HEADS) return 0.0;
  const int* p = oa::limb_words(rs.limbs, row / GQ, row % GQ);
#pragma unroll
  for (int w = 0; w < 32; ++w) lw[w] = p[w];
  return ldexp(1.0, -rs.fexp[row]);
}

// The wave's list of candidate keys (one per lane at most), in its own 64 LDS words.  lanes_below: the
// set bits of m below this lane.
constexpr int kTopList = 64;
__device__ __forceinline__ int lanes_below(unsigned long long m) {
  return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}
__device__ __forceinline__ void list_sync() {      // one wave's LDS: in order, the compiler told
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ void list_push(unsigned long long* list, int& m, bool in, unsigned long long x) {
  const unsigned long long bal = __ballot(in);
  if (!bal) return;                                 // uniform
  const int i = m + lanes_below(bal);
  if (in && i < kTopList) list[i] = x;
  m += __popcll(bal);
}
// the rank of this lane's key among the list's m <= 64 distinct keys (entries past m are 0)
__device__ __forceinline__ int list_rank(const unsigned long long* list, int m, unsigned long long x) {
  int r0 = 0, r1 = 0;
  for (int i = 0; i < m; i += 4) {
    const ulonglong2 u = reinterpret_cast<const ulonglong2*>(list)[i >> 1];
    const ulonglong2 v = reinterpret_cast<const ulonglong2*>(list)[(i >> 1) + 1];
    r0 += (u.x > x ? 1 : 0) + (u.y > x ? 1 : 0);
    r1 += (v.x > x ? 1 : 0) + (v.y > x ? 1 : 0);
  }
  return r0 + r1;
}

// Lane l holds the maxima of tiles l, l + 64, ...; the chosen tiles and then the selected tokens come
// from a short list instead of repeated wave maxima over every lane's registers:
//   tiles    the k-th of the distinct lane maxima bounds the k-th tile key from below (k wave maxima of
//            one 32-bit register a lane), so that the tiles at or above it -- k and a few -- hold the k best;
//            each takes a lane and its rank is the number of larger keys of the list;
//   tokens   a chosen tile's greatest score is some token's, so the k-th best token reaches the k-th
//            chosen tile's maximum: the tokens of the chosen tiles that do (by key head with HEADS) are
//            listed, scored exactly, one per lane, and ranked the same way.
// Keys carry the position, so they are distinct and ranks are a permutation.  A list of more than 64
// keys (many equal scores) or one that does not settle the k tokens (fewer than k scores above -inf)
// takes the repeated maxima, 900 cycles a step on a lone wave.  At 32 rows of 512 tiles, k = 9, the row's
// top-k went from 20000 to 9700 cycles.
// Writes sel = [0..ns) ++ [n-nl..n) ++ top and marks the selected scores.  list: kTopList words of LDS
// of this wave.  lds_sel, when not null, receives the same sel row (for the rest of the workgroup).
template <int TPL, int KR, bool HEADS>
__device__ __forceinline__ void topk_reg_row(void* __restrict__ Sv, long s_stride,
                                             const float* __restrict__ TM, long tm_stride,
                                             int ntiles, int32_t* __restrict__ sel, long sel_stride,
                                             int n, int ns, int nl, int k_top, const Rescore& rs,
                                             int row, int lane, unsigned long long* list,
                                             int32_t* lds_sel = nullptr) {
  int lw[HEADS ? 32 : 1];
  const double inv = load_limbs<HEADS>(rs, row, lw);
  float tv[TPL];
#pragma unroll
  for (int j = 0; j < TPL; ++j) tv[j] = TM[(long)row * tm_stride + min(j * 64 + lane, ntiles - 1)];
  int my_pos = 0;                // lane i < k_top: the i-th selected position
  if (k_top > 0) {
    // ---- the chosen tiles
    uint32_t cur = 0u;
#pragma unroll
    for (int j = 0; j < TPL; ++j) cur = max(cur, j * 64 + lane < ntiles ? oa::float_key(tv[j]) : 0u);
    uint32_t bound = 0u;
    for (int i = 0; i < k_top; ++i) {
      bound = oa::wave_max_u32(cur);
      cur = cur == bound ? 0u : cur;
    }
    list[lane] = 0ull;
    list_sync();
    int m = 0;
#pragma unroll
    for (int j = 0; j < TPL; ++j) {
      const int t = j * 64 + lane;
      list_push(list, m, t < ntiles && oa::float_key(tv[j]) >= bound, tile_key(tv[j], t));
    }
    list_sync();
    int my_tile = 0;             // lane i < k_top: the i-th chosen tile
    uint32_t kth;                // the score key of the k-th chosen tile's maximum
    if (m <= kTopList) {
      const unsigned long long x = list[lane];
      const int rank = list_rank(list, m, x);       // lanes past m: m (>= k_top)
      my_tile = __builtin_amdgcn_ds_permute(rank << 2, (int)(0xffffffffu - (unsigned)x));
      kth = (uint32_t)__builtin_amdgcn_readlane((int)(x >> 32), __ffsll(__ballot(rank == k_top - 1)) - 1);
    } else {
      kth = 0u;
      unsigned long long last = ~0ull;              // the next tile: the greatest key below the last
      for (int i = 0; i < k_top; ++i) {
        unsigned long long mine = 0ull;
#pragma unroll
        for (int j = 0; j < TPL; ++j) {
          const unsigned long long x = j * 64 + lane < ntiles ? tile_key(tv[j], j * 64 + lane) : 0ull;
          mine = x < last && x > mine ? x : mine;
        }
        last = oa::wave_max_u64(mine);
        if (lane == i) my_tile = (int)(0xffffffffu - (unsigned)last);
        kth = (uint32_t)(last >> 32);
      }
    }
    // ---- candidates: column lane of the k chosen tiles.  With HEADS only those whose key head
    // reaches that of the k-th tile maximum can be in the top k (heads are non-decreasing in the
    // score): their exact scores are recomputed, the others count as -inf
    const int dead_hi = n - nl;
    const int kvr = oa::row_kv(row, rs.qsh);
    uint32_t hv[KR];             // heads, or the scores' bits
#pragma unroll
    for (int j = 0; j < KR; ++j) {
      const long at = (long)row * s_stride + __builtin_amdgcn_readlane(my_tile, min(j, k_top - 1)) * 64 + lane;
      hv[j] = HEADS ? (uint32_t)static_cast<const uint16_t*>(Sv)[at]
                    : __float_as_uint(static_cast<const float*>(Sv)[at]);
    }
    list[lane] = 0ull;
    list_sync();
    m = 0;
#pragma unroll
    for (int j = 0; j < KR; ++j) {
      if (j >= k_top) continue;                     // uniform
      const int pos = __builtin_amdgcn_readlane(my_tile, j) * 64 + lane;
      if (HEADS) list_push(list, m, hv[j] >= (kth >> 16) && pos >= ns && pos < dead_hi, (unsigned long long)pos);
      else list_push(list, m, oa::float_key(__uint_as_float(hv[j])) >= kth, tile_key(__uint_as_float(hv[j]), pos));
    }
    list_sync();
    bool done = m >= k_top && m <= kTopList;
    if (done) {
      unsigned long long x = list[lane];
      if (HEADS) {
        const int pos = max(min((int)x, dead_hi - 1), 0);
        x = lane < m ? tile_key(oa::qgs_score(rs.codes, rs.lmax, kvr, pos, lw, inv), pos) : 0ull;
        list_sync();
        list[lane] = x;
        list_sync();
      }
      const int rank = list_rank(list, m, x);
      my_pos = __builtin_amdgcn_ds_permute(rank << 2, (int)(0xffffffffu - (unsigned)x));
      // a token that is not listed scores -inf: the k listed ones must be above it
      done = !HEADS || __ballot(rank < k_top && (uint32_t)(x >> 32) <= oa::float_key(-INFINITY)) == 0ull;
    }
    if (!done) {
      // the repeated maxima over every candidate
      unsigned long long ck[KR] = {};
#pragma unroll 1
      for (int j = 0; j < k_top; ++j) {
        const int pos = __builtin_amdgcn_readlane(my_tile, j) * 64 + lane;
        uint32_t h = 0u;
        float v = -INFINITY;
#pragma unroll
        for (int u = 0; u < KR; ++u) h = u == j ? hv[u] : h;
        if (!HEADS) v = __uint_as_float(h);
        else if (h >= (kth >> 16) && pos >= ns && pos < dead_hi)
          v = oa::qgs_score(rs.codes, rs.lmax, kvr, pos, lw, inv);
        const unsigned long long x = tile_key(v, pos);
#pragma unroll
        for (int u = 0; u < KR; ++u) ck[u] = u == j ? x : ck[u];
      }
      unsigned long long last = ~0ull;
      for (int i = 0; i < k_top; ++i) {
        unsigned long long mine = 0ull;
#pragma unroll
        for (int j = 0; j < KR; ++j) mine = j < k_top && ck[j] < last && ck[j] > mine ? ck[j] : mine;
        last = oa::wave_max_u64(mine);
        if (lane == i) my_pos = (int)(0xffffffffu - (unsigned)last);
      }
    }
  }
  int32_t* sr = sel + (long)row * sel_stride;
  if (lane < ns) sr[lane] = lane;
  if (lane < nl) sr[ns + lane] = n - nl + lane;
  if (lane < k_top) {
    sr[ns + nl + lane] = my_pos;
    mark_selected<HEADS>(Sv, s_stride, row, my_pos);
  }
  if (lds_sel) {
    if (lane < ns) lds_sel[lane] = lane;
    if (lane < nl) lds_sel[ns + lane] = n - nl + lane;
    if (lane < k_top) lds_sel[ns + nl + lane] = my_pos;
  }
}

}  // namespace oa_sel
