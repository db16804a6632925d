// Backward of the block-sparse prefill attention (fsi_sparse_attn) on MI355X
// (gfx950), without materialising any (T, T) tensor.
//
//   out[t] = sum_s w(t, s) exp(scale q_t . k_s - m_t) v_s / l_t,
//   l_t = sum_s w(t, s) exp(scale q_t . k_s - m_t)
//
// with the key weights of the forward: FSI_SATTN_LOCAL_REMOTE (attention.py:
// 148-218) w = 1 where t - W < s <= t or the page of s is listed for the query
// block of t (a union), FSI_SATTN_BLOCK_LIST (triton_ops.py:26-93) w = the
// number of times the block of s is listed for the block of t.  Gradients, with
// P_ts = w exp(scale q_t . k_s - m_t) / l_t and D_t = dout_t . out_t:
//   dV_s = sum_t P_ts dout_t,      dP_ts = dout_t . v_s,
//   dS_ts = P_ts (dP_ts - D_t),    dQ_t = scale sum_s dS_ts k_s,
//   dK_s = scale sum_t dS_ts q_t   (GQA: summed over the group's query heads).
//
// Three kernels on tiles of 64 queries x 64 keys (bf16 inputs with head_dim 32 / 64 / 128:
// the sab_*_bf kernels below, every product on bf16 MFMA; otherwise fp32 arithmetic on
// v_mfma_f32_16x16x4_f32):
//   1. sab_map_kernel: for every (query block, key block) pair of the pattern's
//      block size, its weight class: mode LOCAL_REMOTE 1 = the window reaches
//      it, 2 = listed (every key counts); mode BLOCK_LIST the listing count.
//      Tiles whose pairs are all 0 are skipped below.
//   2. sab_q_kernel: per (sequence, query head, 64-query tile), two passes over
//      the key tiles: the row maxima and sums, then dQ; writes m, l and D per
//      query row.
//   3. sab_kv_kernel: per (sequence, KV head, 64-key tile), every query tile and
//      query head of the group: dV and dK accumulated in registers, no atomics.
#include "fsi_common.h"

namespace {

using namespace fsi;

constexpr int AB_T = 64;        // queries / keys per tile
constexpr int AB_THREADS = 256;

template <typename T>
__device__ __forceinline__ float ldv(const T* p, int64_t i);
template <>
__device__ __forceinline__ float ldv<float>(const float* p, int64_t i) { return p[i]; }
template <>
__device__ __forceinline__ float ldv<bf16_t>(const bf16_t* p, int64_t i) { return bf16_to_f32(p[i]); }

struct AbParams {
  const void* q;
  int64_t qs_b, qs_h, qs_t;
  const void* k;
  int64_t ks_b, ks_h, ks_t;
  const void* v;
  int64_t vs_b, vs_h, vs_t;
  const void* o;
  int64_t os_b, os_h, os_t;
  const void* dout;
  int64_t ds_b, ds_h, ds_t;
  int B, Hq, Hkv, T, hd, block, mode, window;
  const int32_t* lists;
  int64_t ls_b, ls_q;
  int cap;
  const int32_t* counts;
  int64_t cs_b, cs_q;
  float scale;
  int nb;             // blocks of the pattern: ceil(T / block)
  int64_t tp;         // T rounded up to whole tiles
  bool vec4;          // head_dim one of the tile widths (16 / 32 / 64 / 128), rows 4-element aligned
  int32_t* map;       // (B, nb, nb) weight classes
  float* stat_m;      // (B, Hq, T); the bf16 kernels: lse2 and D, (B, Hq, tp)
  float* stat_l;
  float* stat_d;
  float* dq;          // (B, Hq, T, hd) fp32, contiguous
  float* dk;          // (B, Hkv, T, hd) fp32
  float* dv;
  int* err;
};

// 1. Weight classes of query block qb against every key block.
__global__ __launch_bounds__(AB_THREADS) void sab_map_kernel(AbParams P) {
  const int qb = blockIdx.x, b = blockIdx.y;
  int32_t* row = P.map + (static_cast<int64_t>(b) * P.nb + qb) * P.nb;
  const int t_lo = qb * P.block, t_hi = min(P.T, t_lo + P.block) - 1;
  for (int kb = threadIdx.x; kb < P.nb; kb += AB_THREADS) {
    int w = 0;
    if (P.mode == FSI_SATTN_LOCAL_REMOTE) {
      const int s_lo = kb * P.block, s_hi = min(P.T, s_lo + P.block) - 1;
      // some s <= t and s > t - W with t, s in the two blocks
      if (s_lo <= t_hi && s_hi > t_lo - P.window) w = 1;
    }
    row[kb] = w;
  }
  __syncthreads();
  int cnt = P.counts[b * P.cs_b + qb * P.cs_q];
  cnt = cnt < 0 ? 0 : (cnt > P.cap ? P.cap : cnt);
  const int32_t* list = P.lists ? P.lists + b * P.ls_b + qb * P.ls_q : nullptr;
  bool bad = false;
  for (int j = threadIdx.x; j < cnt; j += AB_THREADS) {
    const int pg = list[j];
    if (pg < 0 || pg >= P.nb) {
      bad = true;
      continue;
    }
    if (P.mode == FSI_SATTN_LOCAL_REMOTE) atomicOr(row + pg, 2);
    else atomicAdd(row + pg, 1);
  }
  if (bad) set_error(P.err, FSI_ERR_INDEX_RANGE);
}

// Class of the block pair (query t, key s), both < T.
__device__ __forceinline__ int sab_class(const AbParams& P, const int32_t* map_b, int t, int s) {
  return map_b[static_cast<int64_t>(t / P.block) * P.nb + s / P.block];
}

// Weight of key s for query t (both < T) given the class of their blocks.
__device__ __forceinline__ float sab_weight(const AbParams& P, int cls, int t, int s) {
  if (P.mode == FSI_SATTN_LOCAL_REMOTE) return ((cls & 2) || (s <= t && s > t - P.window)) ? 1.f : 0.f;
  return static_cast<float>(cls);
}

// Class of the tile of queries [t0, t0 + 64) and keys [s0, s0 + 64), the
// same for every thread: the block class (> 0) when the tile lies in one block
// pair, 0 when every block pair it touches has class 0 (nothing to do), -1
// when it spans several block pairs and some is non-zero (classes then looked
// up per element).
__device__ __forceinline__ int sab_tile_class(const AbParams& P, const int32_t* map_b, int t0, int s0) {
  const int qb0 = t0 / P.block, qb1 = (min(P.T, t0 + AB_T) - 1) / P.block;
  const int kb0 = s0 / P.block, kb1 = (min(P.T, s0 + AB_T) - 1) / P.block;
  const int nq = qb1 - qb0 + 1, nk = kb1 - kb0 + 1;
  if (nq == 1 && nk == 1) return map_b[static_cast<int64_t>(qb0) * P.nb + kb0];
  int live = 0;
  for (int i = threadIdx.x; i < nq * nk; i += AB_THREADS)
    live |= map_b[static_cast<int64_t>(qb0 + i / nk) * P.nb + kb0 + i % nk] != 0;
  return __syncthreads_or(live) != 0 ? -1 : 0;
}

// Weight of key s for query t (both < T) in a tile of class tcls (as returned by
// sab_tile_class, non-zero); the block map is read only for a mixed tile.
__device__ __forceinline__ float sab_tile_weight(const AbParams& P, const int32_t* map_b, int tcls, int t, int s) {
  if (tcls < 0) return sab_weight(P, sab_class(P, map_b, t, s), t, s);
  return sab_weight(P, tcls, t, s);
}

// Logits of keys s0 + 16 t + 4 kg + e against query tq (S^T accumulators st),
// with the weight folded in (exp(x - m) = w exp(scale q.k - m)); -inf where the
// weight is 0 or the query / key is past T.  A tile of one block pair takes its
// weight from the class (one log per tile); a local tile of the local/remote
// pattern tests the window per element.
__device__ __forceinline__ void sab_logits(const AbParams& P, const int32_t* map_b, int tq, int kg, int s0, int tcls,
                                           f32x4_t (&st)[4]) {
  if (tcls > 0 && (P.mode == FSI_SATTN_BLOCK_LIST || (tcls & 2))) {
    // one weight for the whole tile: keys below lim are valid
    const float lw = P.mode == FSI_SATTN_BLOCK_LIST ? __logf(static_cast<float>(tcls)) : 0.f;
    const int lim = tq < P.T ? P.T : 0;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int sk = s0 + 16 * t + 4 * kg + e;
        st[t][e] = sk < lim ? st[t][e] * P.scale + lw : -INFINITY;
      }
  } else if (tcls > 0) {
    // local/remote tile reached by the window only: tq - W < sk <= tq (< T)
    const int hi = tq < P.T ? tq : -1, lo = tq - P.window;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int sk = s0 + 16 * t + 4 * kg + e;
        st[t][e] = sk <= hi && sk > lo ? st[t][e] * P.scale : -INFINITY;
      }
  } else {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int sk = s0 + 16 * t + 4 * kg + e;
        float x = -INFINITY;
        if (tq < P.T && sk < P.T) {
          const float w = sab_tile_weight(P, map_b, tcls, tq, sk);
          if (w > 0.f) x = st[t][e] * P.scale + __logf(w);
        }
        st[t][e] = x;
      }
  }
}

// 64 rows of a (T, hd) matrix at row stride rs into an LDS tile of row stride
// HD + 4 floats (rows past T and columns past hd read as 0).  The 4-float pad
// puts the 8 rows a 128-bit read serves at once on distinct bank groups, and
// the 16 rows of a column read on two halves of the banks.
// vec: head_dim == HD and every row starts 4-element aligned (host-checked), so
// a thread moves 4 consecutive elements at once.
template <typename T>
__device__ __forceinline__ f32x4_t ld4(const T* p);
template <>
__device__ __forceinline__ f32x4_t ld4<float>(const float* p) { return *reinterpret_cast<const f32x4_t*>(p); }
template <>
__device__ __forceinline__ f32x4_t ld4<bf16_t>(const bf16_t* p) {
  const uint2 w = *reinterpret_cast<const uint2*>(p);
  return f32x4_t{__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u), __uint_as_float(w.y << 16),
                 __uint_as_float(w.y & 0xffff0000u)};
}
template <typename T, int HD>
__device__ __forceinline__ void sab_load_tile(const T* base, int64_t rs, int r0, int nrows, int hd, float* tile,
                                              bool vec) {
  if (vec) {
    for (int i = threadIdx.x; i < AB_T * HD / 4; i += AB_THREADS) {
      const int r = i / (HD / 4), d = 4 * (i % (HD / 4));
      f32x4_t x = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (r0 + r < nrows) x = ld4<T>(base + static_cast<int64_t>(r0 + r) * rs + d);
      *reinterpret_cast<f32x4_t*>(&tile[r * (HD + 4) + d]) = x;
    }
    return;
  }
  for (int i = threadIdx.x; i < AB_T * HD; i += AB_THREADS) {
    const int r = i / HD, d = i % HD;
    tile[r * (HD + 4) + d] =
        r0 + r < nrows && d < hd ? ldv<T>(base, static_cast<int64_t>(r0 + r) * rs + d) : 0.f;
  }
}

// Row `row` (< T) of a (T, hd) matrix as this lane's MFMA k-operand: dims
// 16 dg + 4 kg .. +4 of every 16-dim group (0 past hd).
template <typename T, int HD>
__device__ __forceinline__ void sab_row_frag(const T* base, int64_t rs, int row, int hd, int kg,
                                             f32x4_t (&f)[HD / 16]) {
#pragma unroll
  for (int dg = 0; dg < HD / 16; ++dg)
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int d = 16 * dg + 4 * kg + kk;
      f[dg][kk] = d < hd ? ldv<T>(base, static_cast<int64_t>(row) * rs + d) : 0.f;
    }
}

__device__ __forceinline__ f32x4_t ab_mfma(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Two floats holding bf16 values as one packed bf16 pair (their upper halves).
__device__ __forceinline__ uint32_t ab_pk(float x, float y) {
  return __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u);
}
// 8 consecutive floats of an LDS row (bf16 values) as a bf16 MFMA operand.
__device__ __forceinline__ u32x4_t ab_pack8(const float* p) {
  const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p);
  const f32x4_t b = *reinterpret_cast<const f32x4_t*>(p + 4);
  return u32x4_t{ab_pk(a[0], a[1]), ab_pk(a[2], a[3]), ab_pk(b[0], b[1]), ab_pk(b[2], b[3])};
}
// Row `row` of a bf16 (T, hd) matrix as this lane's bf16 MFMA operand: dims
// 32 ks + 8 kg .. +8 of every 32-dim step (0 past hd).
template <typename T, int HD>
__device__ __forceinline__ void sab_row_frag_bf(const T* base, int64_t rs, int row, int hd, int kg,
                                                u32x4_t (&f)[HD / 32]) {
#pragma unroll
  for (int ks = 0; ks < HD / 32; ++ks) {
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int d = 32 * ks + 8 * kg + j;
      x[j] = d < hd ? ldv<T>(base, static_cast<int64_t>(row) * rs + d) : 0.f;
    }
    f[ks] = u32x4_t{ab_pk(x[0], x[1]), ab_pk(x[2], x[3]), ab_pk(x[4], x[5]), ab_pk(x[6], x[7])};
  }
}

// 2. dQ and the row statistics for one (b, h, 64-query tile).  Wave w owns
//    queries t0 + 16 w .. +16 and keeps their Q and dout rows as the B operand
//    of S^T = K Q^T and dP^T = V dout^T (v_mfma_f32_16x16x4_f32, k-step kk taking
//    dims 4 (lane / 16) + kk of each 16-dim group); lane (r, kg) then holds keys
//    16 t + 4 kg + e of query r, so dS^T's element kk is the B operand of
//    dQ^T = K^T dS^T for the keys 16 t + 4 kg + kk (K^T read by column from LDS).
template <typename T, int HD>
__global__ __launch_bounds__(AB_THREADS) void sab_q_kernel(AbParams P) {
  constexpr int DG = HD / 16, R = HD + 4;
  __shared__ float Ks[AB_T * R], Vs[AB_T * R];
  // heads fastest and the latest query tiles first: under a causal pattern they
  // reach the most key tiles, so the longest blocks start first
  const int t0 = ((P.T + AB_T - 1) / AB_T - 1 - static_cast<int>(blockIdx.x / P.Hq)) * AB_T;
  const int b = blockIdx.y, h = blockIdx.x % P.Hq;
  const int g = h / (P.Hq / P.Hkv);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, kg = lane >> 4;
  const int tq = t0 + 16 * wave + r;             // this lane's query
  const int tql = tq < P.T ? tq : P.T - 1;       // rows past T read row T - 1, never stored
  const T* q = static_cast<const T*>(P.q) + b * P.qs_b + h * P.qs_h;
  const T* o = static_cast<const T*>(P.o) + b * P.os_b + h * P.os_h;
  const T* dout = static_cast<const T*>(P.dout) + b * P.ds_b + h * P.ds_h;
  const T* k = static_cast<const T*>(P.k) + b * P.ks_b + g * P.ks_h;
  const T* v = static_cast<const T*>(P.v) + b * P.vs_b + g * P.vs_h;
  const int32_t* map_b = P.map + static_cast<int64_t>(b) * P.nb * P.nb;

  // bf16 inputs: S^T and dP^T on v_mfma_f32_16x16x32_bf16 (products of bf16 values
  // are exact in fp32, so this loses nothing against the fp32 form)
  constexpr bool BFR = sizeof(T) == 2 && HD >= 32;
  constexpr int KS32 = HD >= 32 ? HD / 32 : 1;
  f32x4_t qf[DG], df[DG];
  sab_row_frag<T, HD>(q, P.qs_t, tql, P.hd, kg, qf);
  sab_row_frag<T, HD>(dout, P.ds_t, tql, P.hd, kg, df);
  u32x4_t qb[KS32], db[KS32];
  if constexpr (BFR) {
    sab_row_frag_bf<T, HD>(q, P.qs_t, tql, P.hd, kg, qb);
    sab_row_frag_bf<T, HD>(dout, P.ds_t, tql, P.hd, kg, db);
  }
  float dd;  // D = dout . out of query r
  {
    f32x4_t of[DG];
    sab_row_frag<T, HD>(o, P.os_t, tql, P.hd, kg, of);
    float part = 0.f;
#pragma unroll
    for (int dg = 0; dg < DG; ++dg)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) part = fmaf(df[dg][kk], of[dg][kk], part);
    dd = sum_rows4(part);
  }

  auto logits = [&](int s0, int tcls, f32x4_t (&st)[4]) { sab_logits(P, map_b, tq, kg, s0, tcls, st); };
  // S^T tiles of the 64 keys in Ks against this wave's queries
  auto scores = [&](f32x4_t (&st)[4], const float* Xs, const f32x4_t (&bf)[DG], const u32x4_t (&bb)[KS32]) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      st[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if constexpr (BFR) {
#pragma unroll
        for (int ks = 0; ks < KS32; ++ks)
          st[t] = mfma16x16x32(ab_pack8(&Xs[(16 * t + r) * R + 32 * ks + 8 * kg]), bb[ks], st[t]);
      } else {
#pragma unroll
        for (int dg = 0; dg < DG; ++dg) {
          const f32x4_t a = *reinterpret_cast<const f32x4_t*>(&Xs[(16 * t + r) * R + 16 * dg + 4 * kg]);
#pragma unroll
          for (int kk = 0; kk < 4; ++kk) st[t] = ab_mfma(a[kk], bf[dg][kk], st[t]);
        }
      }
    }
  };

  // pass 1: row maximum and sum over every live key tile (the sum kept per lane
  // and reduced over the lane group at the end)
  float m = -INFINITY, lpart = 0.f;
  for (int s0 = 0; s0 < P.T; s0 += AB_T) {
    const int tcls = sab_tile_class(P, map_b, t0, s0);
    if (tcls == 0) continue;
    sab_load_tile<T, HD>(k, P.ks_t, s0, P.T, P.hd, Ks, P.vec4);
    __syncthreads();
    f32x4_t st[4];
    scores(st, Ks, qf, qb);
    logits(s0, tcls, st);
    float cm = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) cm = fmaxf(cm, st[t][e]);
    cm = max_rows4(cm);
    if (cm > -INFINITY) {
      const float mn = fmaxf(m, cm);
      float add = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) add += __expf(st[t][e] - mn);
      lpart = (m > -INFINITY ? lpart * __expf(m - mn) : 0.f) + add;
      m = mn;
    }
    __syncthreads();
  }
  const float l = sum_rows4(lpart);
  const float il = l > 0.f ? 1.f / l : 0.f;

  // pass 2: dQ^T[dim][query] = scale sum_key K[key][dim] dS[query][key]
  f32x4_t dqa[DG];
#pragma unroll
  for (int dt = 0; dt < DG; ++dt) dqa[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < P.T; s0 += AB_T) {
    const int tcls = sab_tile_class(P, map_b, t0, s0);
    if (tcls == 0) continue;
    sab_load_tile<T, HD>(k, P.ks_t, s0, P.T, P.hd, Ks, P.vec4);
    sab_load_tile<T, HD>(v, P.vs_t, s0, P.T, P.hd, Vs, P.vec4);
    __syncthreads();
    f32x4_t st[4], dp[4];
    scores(st, Ks, qf, qb);
    scores(dp, Vs, df, db);  // dP^T = V dout^T
    logits(s0, tcls, st);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p = l > 0.f ? __expf(st[t][e] - m) * il : 0.f;  // exp(-inf) = 0 where w = 0
        st[t][e] = p * (dp[t][e] - dd);                            // dS^T
      }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const float* krow = &Ks[(16 * t + 4 * kg + kk) * R + r];
#pragma unroll
        for (int dt = 0; dt < DG; ++dt) dqa[dt] = ab_mfma(krow[16 * dt], st[t][kk], dqa[dt]);
      }
    __syncthreads();
  }
  // lane (r, kg) holds dQ[query r][dims 16 dt + 4 kg + e]
  const int64_t rowbase = (static_cast<int64_t>(b) * P.Hq + h) * P.T;
  if (tq < P.T) {
#pragma unroll
    for (int dt = 0; dt < DG; ++dt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int d = 16 * dt + 4 * kg + e;
        if (d < P.hd) P.dq[(rowbase + tq) * P.hd + d] = dqa[dt][e] * P.scale;
      }
    if (kg == 0) {
      P.stat_m[rowbase + tq] = m;
      P.stat_l[rowbase + tq] = l;
      P.stat_d[rowbase + tq] = dd;
    }
  }
}

// 3. dK and dV for one (b, g, 64-key tile) over every query tile and query
//    head of the group.  Wave w owns keys s0 + 16 w .. +16 and keeps their K and
//    V rows as the B operand of S = Q K^T and dP = dout V^T; lane (r, kg) then
//    holds queries 16 qt + 4 kg + e of key r, so the elements of P and dS are the
//    B operands of dV^T = dout^T P and dK^T = Q^T dS (dout^T, Q^T read by column
//    from LDS).  Accumulated in registers, no atomics.
template <typename T, int HD>
__global__ __launch_bounds__(AB_THREADS) void sab_kv_kernel(AbParams P) {
  constexpr int DG = HD / 16, R = HD + 4;
  __shared__ float Qs[AB_T * R], Ds[AB_T * R];
  __shared__ float row_m[AB_T], row_il[AB_T], row_d[AB_T];
  // heads fastest and the earliest key tiles first: under a causal pattern the
  // most query tiles reach them, so the longest blocks start first
  const int s0 = static_cast<int>(blockIdx.x / P.Hkv) * AB_T;
  const int b = blockIdx.y, g = blockIdx.x % P.Hkv;
  const int G = P.Hq / P.Hkv;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, kg = lane >> 4;
  const int sk = s0 + 16 * wave + r;       // this lane's key
  const int skl = sk < P.T ? sk : P.T - 1;
  const T* k = static_cast<const T*>(P.k) + b * P.ks_b + g * P.ks_h;
  const T* v = static_cast<const T*>(P.v) + b * P.vs_b + g * P.vs_h;
  const int32_t* map_b = P.map + static_cast<int64_t>(b) * P.nb * P.nb;
  constexpr bool BFR = sizeof(T) == 2 && HD >= 32;  // S and dP on bf16 MFMA (exact products)
  constexpr int KS32 = HD >= 32 ? HD / 32 : 1;
  f32x4_t kf[BFR ? 1 : DG], vf[BFR ? 1 : DG];
  u32x4_t kb[KS32], vb[KS32];
  if constexpr (BFR) {
    sab_row_frag_bf<T, HD>(k, P.ks_t, skl, P.hd, kg, kb);
    sab_row_frag_bf<T, HD>(v, P.vs_t, skl, P.hd, kg, vb);
  } else {
    sab_row_frag<T, HD>(k, P.ks_t, skl, P.hd, kg, kf);
    sab_row_frag<T, HD>(v, P.vs_t, skl, P.hd, kg, vf);
  }
  f32x4_t dka[DG], dva[DG];
#pragma unroll
  for (int dt = 0; dt < DG; ++dt) dka[dt] = dva[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  for (int t0 = 0; t0 < P.T; t0 += AB_T) {
    const int tcls = sab_tile_class(P, map_b, t0, s0);
    if (tcls == 0) continue;
    // weight of the whole tile when it lies in one block pair and needs no window test
    const float wall = tcls > 0 && (P.mode == FSI_SATTN_BLOCK_LIST || (tcls & 2))
                           ? (P.mode == FSI_SATTN_BLOCK_LIST ? static_cast<float>(tcls) : 1.f)
                           : 0.f;
    for (int hh = 0; hh < G; ++hh) {
      const int h = g * G + hh;
      const T* q = static_cast<const T*>(P.q) + b * P.qs_b + h * P.qs_h;
      const T* dout = static_cast<const T*>(P.dout) + b * P.ds_b + h * P.ds_h;
      const int64_t rowbase = (static_cast<int64_t>(b) * P.Hq + h) * P.T;
      sab_load_tile<T, HD>(q, P.qs_t, t0, P.T, P.hd, Qs, P.vec4);
      sab_load_tile<T, HD>(dout, P.ds_t, t0, P.T, P.hd, Ds, P.vec4);
      if (tid < AB_T) {
        const int t = t0 + tid;
        const float lq = t < P.T ? P.stat_l[rowbase + t] : 0.f;
        row_m[tid] = t < P.T ? P.stat_m[rowbase + t] : -INFINITY;
        row_il[tid] = lq > 0.f ? 1.f / lq : 0.f;
        row_d[tid] = t < P.T ? P.stat_d[rowbase + t] : 0.f;
      }
      __syncthreads();
#pragma unroll 1
      for (int qt = 0; qt < 4; ++qt) {  // not unrolled: K, V, dK and dV already hold 128 registers
        f32x4_t s = f32x4_t{0.f, 0.f, 0.f, 0.f}, dp = s;
        if constexpr (BFR) {
#pragma unroll
          for (int ks = 0; ks < KS32; ++ks) {
            s = mfma16x16x32(ab_pack8(&Qs[(16 * qt + r) * R + 32 * ks + 8 * kg]), kb[ks], s);
            dp = mfma16x16x32(ab_pack8(&Ds[(16 * qt + r) * R + 32 * ks + 8 * kg]), vb[ks], dp);
          }
        } else {
#pragma unroll
          for (int dg = 0; dg < DG; ++dg) {
            const f32x4_t a = *reinterpret_cast<const f32x4_t*>(&Qs[(16 * qt + r) * R + 16 * dg + 4 * kg]);
            const f32x4_t c = *reinterpret_cast<const f32x4_t*>(&Ds[(16 * qt + r) * R + 16 * dg + 4 * kg]);
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
              s = ab_mfma(a[kk], kf[dg][kk], s);
              dp = ab_mfma(c[kk], vf[dg][kk], dp);
            }
          }
        }
        // s[e], dp[e]: query 16 qt + 4 kg + e, key r
        f32x4_t pp, ds;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int rq = 16 * qt + 4 * kg + e, t = t0 + rq;
          float p = 0.f;
          const float il = row_il[rq];
          if (t < P.T && sk < P.T && il > 0.f) {
            const float w = wall > 0.f ? wall : sab_tile_weight(P, map_b, tcls, t, sk);
            if (w > 0.f) p = w * __expf(s[e] * P.scale - row_m[rq]) * il;
          }
          pp[e] = p;
          ds[e] = p * (dp[e] - row_d[rq]);
        }
        // dV^T[dim][key] += dout[query][dim] P[query][key], dK^T += Q[query][dim] dS[query][key]
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          const float* drow = &Ds[(16 * qt + 4 * kg + kk) * R + r];
          const float* qrow = &Qs[(16 * qt + 4 * kg + kk) * R + r];
#pragma unroll
          for (int dt = 0; dt < DG; ++dt) {
            dva[dt] = ab_mfma(drow[16 * dt], pp[kk], dva[dt]);
            dka[dt] = ab_mfma(qrow[16 * dt], ds[kk], dka[dt]);
          }
        }
      }
      __syncthreads();
    }
  }
  // lane (r, kg) holds dK, dV [key r][dims 16 dt + 4 kg + e]
  const int64_t kbase = (static_cast<int64_t>(b) * P.Hkv + g) * P.T;
  if (sk < P.T) {
#pragma unroll
    for (int dt = 0; dt < DG; ++dt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int d = 16 * dt + 4 * kg + e;
        if (d >= P.hd) continue;
        P.dk[(kbase + sk) * P.hd + d] = dka[dt][e] * P.scale;
        P.dv[(kbase + sk) * P.hd + d] = dva[dt][e];
      }
  }
}

// ---------------------------------------------------------------------------
// bf16 inputs with head_dim 32 / 64 / 128 and 8-element-aligned rows: every product on
// v_mfma_f32_16x16x32_bf16 over 64-row tiles moved straight into LDS (no staging
// registers), double-buffered: the next tile's loads run while this one is used.
//
// An operand fragment is 1 KiB (8 LDS clocks) and feeds a 16-clock MFMA on one of four SIMDs,
// so a fragment has to serve two MFMAs at least or LDS bounds the kernel.  Each wave therefore
// owns 32 rows (two 16-row operands in registers) of its side, and P / dS enter their products as
// a pair of bf16 operands hi + lo (hi = the value rounded to bf16, lo = the remainder rounded;
// ~2^-17 relative, the other operand an exact bf16 input, fp32 accumulation), which makes it four
// there.  With that no unit is full (sab_q | sab_kv: MFMA 0.37 | 0.41 busy, VALU 0.55 | 0.44, LDS
// 0.30 | 0.29 with half of it bank conflicts): what bounds them is the chain product, softmax
// and split, product of every tile, at the two waves per SIMD that registers (204 | 256) and
// LDS (64 | 65 KiB a workgroup) leave.
// The tiles are stored row-major only: products that contract over a tile's rows read it
// with ds_read_b64_tr_b16, so no transposed copy is written.
// 8192 tokens, 32 / 8 heads of 128, window 1024 + 32 pages: sab_q 1521 -> 1026 us,
// sab_kv 1763 -> 1125 us against 16 rows a wave over padded row-major and
// transposed tiles staged in registers (four heads a workgroup in sab_q: 2 % slower).
// Sub-tile classes: block 16, 2 x 4096 tokens, 8 / 2 heads of 128 2480 -> 925 us.
//
// 16-byte piece p of row r sits at piece p ^ sab_swz(r): the 8 rows a 128-bit read serves
// at once fall on distinct bank quads, and the 4 rows x 32 bytes that 16 lanes of a
// transposing read cover fill one bank period (head_dim 32: two rows share a period and
// the transposing reads conflict pairwise).
//
// A lane's k slots of a 32-row product: rows 4 kg + e (e < 4) and 16 + 4 kg + e - 4
// (e >= 4), i.e. the rows its two 16 x 16 accumulators of P / dS hold, so those enter the
// MFMA where they are; the transposing reads take the same rows.
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(3))) void ab_lds_t;
typedef __attribute__((address_space(1))) void ab_glb_t;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short s16x4_t;
typedef __attribute__((address_space(3))) s16x4_t ab_tr_t;

template <int HD>
__device__ __forceinline__ int sab_swz(int row) {
  return HD >= 64 ? ((row & 3) << 1) | ((row >> 2) & 1) : (row >> 1) & 3;
}

template <int HD>
constexpr int sab_tile_bytes() { return AB_T * HD * 2; }

// Rows [r0, r0 + 64) of a (T, HD) bf16 matrix at row stride rs into the LDS tile, by NT
// threads; rows past T re-read row T - 1 (every product that uses them is multiplied by a
// zero P / dS or never stored, so they only need to be finite).  Row strides are below
// 2^24 elements (host-checked): a scalar row base and 32-bit lane offsets.
template <int HD, int NT>
__device__ __forceinline__ void sab_dma(const bf16_t* base, int64_t rs, int r0, int T, char* tile) {
  constexpr int PC = HD / 8, ROWS = NT / PC, N = AB_T / ROWS > 0 ? AB_T / ROWS : 1;
  static_assert(ROWS % 8 == 0, "a thread's rows share their swizzle");
  if (NT > AB_T * PC && threadIdx.x >= AB_T * PC) return;
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // offsets are formed here, not kept in registers over the caller's loop
  const int row = tid / PC, lp = (tid % PC) ^ sab_swz<HD>(row);
  const uint32_t rsb = static_cast<uint32_t>(rs) * 2u;
  const char* rb = reinterpret_cast<const char*>(base + static_cast<int64_t>(r0) * rs);
  char* dst = tile + (threadIdx.x & ~63u) * 16;
  if (r0 + AB_T <= T) {
    // scalar bases and one lane offset: nothing else is kept in registers over the loop
    const uint32_t lo = static_cast<uint32_t>(row) * rsb + 16u * static_cast<uint32_t>(lp);
#pragma unroll
    for (int j = 0; j < N; ++j)
      __builtin_amdgcn_global_load_lds((ab_glb_t*)(rb + static_cast<uint64_t>(j * ROWS) * rsb + lo),
                                       (ab_lds_t*)(dst + j * NT * 16), 16, 0, 0);
  } else {
    const int last = T - 1 - r0;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const uint32_t lo = static_cast<uint32_t>(min(j * ROWS + row, last)) * rsb + 16u * static_cast<uint32_t>(lp);
      __builtin_amdgcn_global_load_lds((ab_glb_t*)(rb + lo), (ab_lds_t*)(dst + j * NT * 16), 16, 0, 0);
    }
  }
}

// LDS byte offsets of a lane's reads inside a tile: every fragment's address is one of
// these plus the tile's, xored with its step's piece, plus a constant, so a loop keeps two
// registers of them and not one per fragment.
//   row: row (lane & 15) of the 128-bit operand reads (32-dim step ks in bits 6 and up);
//   tr: row 4 kg + r / 4, 4-dim group r % 4 of the transposing reads (dims 16 dt in bits 5 and up).
template <int HD>
__device__ __forceinline__ uint32_t sab_row_off(int r, int kg) {
  return r * (HD * 2) + 16 * (kg ^ sab_swz<HD>(r));
}
template <int HD>
__device__ __forceinline__ uint32_t sab_tr_off(int r, int kg) {
  const int row = 4 * kg + (r >> 2);
  return row * (HD * 2) + 16 * (((r >> 1) & 1) ^ sab_swz<HD>(row)) + 8 * (r & 1);
}
// The operand at a row offset (16 rows from a multiple of 16, `at` the constant part) for step ks.
__device__ __forceinline__ u32x4_t sab_row(const char* smem, uint32_t off, int ks, int at) {
  typedef __attribute__((address_space(3))) const u32x4_t lds_u32x4_t;
  typedef __attribute__((address_space(3))) const char lds_char_t;
  return *(lds_u32x4_t*)((lds_char_t*)smem + ((off ^ (64u * (ks & 1))) + 128 * (ks >> 1) + at));
}
// Dims 16 dt + (lane & 15) at the lane's k slots of 32 rows.
template <int HD>
__device__ __forceinline__ u32x4_t sab_trow(char* smem, uint32_t off, int dt, int at) {
  typedef __attribute__((address_space(3))) char lds_char_t;
  lds_char_t* p = (lds_char_t*)smem + ((off ^ (32u * (dt & 3))) + 128 * (dt >> 2) + at);
  const u32x2_t x = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((ab_tr_t*)p));
  const u32x2_t y = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((ab_tr_t*)(p + 16 * HD * 2)));
  return u32x4_t{x[0], x[1], y[0], y[1]};
}

// Class of the tile pair (queries [t0, t0 + 64), keys [s0, s0 + 64)) computed by
// one thread (sab_tile_class without the workgroup reduction).
__device__ __forceinline__ int sab_pair_class(const AbParams& P, const int32_t* map_b, int t0, int s0) {
  const int qb0 = t0 / P.block, qb1 = (min(P.T, t0 + AB_T) - 1) / P.block;
  const int kb0 = s0 / P.block, kb1 = (min(P.T, s0 + AB_T) - 1) / P.block;
  if (qb0 == qb1 && kb0 == kb1) return map_b[static_cast<int64_t>(qb0) * P.nb + kb0];
  int live = 0;
  for (int qb = qb0; qb <= qb1; ++qb)
    for (int kb = kb0; kb <= kb1; ++kb) live |= map_b[static_cast<int64_t>(qb) * P.nb + kb] != 0;
  return live ? -1 : 0;
}

// The live tiles of one tile row (ROW: the query tile at fixed0, key tiles vary) or column,
// ascending: next() moves to the next one and returns false after the last.  Every wave
// walks the same list (64 classes a time in a register, the live ones a ballot), so no LDS
// and no barrier is spent on it.
template <bool ROW>
struct SabTiles {
  const AbParams& P;
  const int32_t* map_b;
  int fixed0, ntiles, c0, cls_lane;
  uint64_t live;
  int tile, cls;
  __device__ SabTiles(const AbParams& p, const int32_t* m, int f0, int n) : P(p), map_b(m), fixed0(f0), ntiles(n) {
    c0 = -64;
    live = 0;
  }
  __device__ __forceinline__ bool next() {
    while (live == 0) {
      c0 += 64;
      if (c0 >= ntiles) return false;
      const int i = c0 + static_cast<int>(threadIdx.x & 63);
      cls_lane = 0;
      if (i < ntiles)
        cls_lane = ROW ? sab_pair_class(P, map_b, fixed0, i * AB_T) : sab_pair_class(P, map_b, i * AB_T, fixed0);
      live = __ballot(cls_lane != 0);
    }
    const int i = __builtin_ctzll(live);
    live &= live - 1;
    tile = c0 + i;
    cls = __builtin_amdgcn_readlane(cls_lane, i);
    return true;
  }
};

// How a 64 x 64 tile's weights are found (by the pattern's block, host-chosen): one block
// pair per tile; one per 16 x 16 sub-tile (block a multiple of 16, the class a scalar load);
// or looked up per element.
enum SabMix : int { SAB_TILE = 0, SAB_SUB = 1, SAB_ELEM = 2 };
template <int MIX>
using sab_mix_t = std::integral_constant<int, MIX>;

// Class of the 16 x 16 sub-tile at queries t0, keys s0 (both wave-uniform); 0 past T.  The
// constant address space makes it a scalar load, which the vector loads in flight don't delay.
__device__ __forceinline__ int sab_sub_class(const AbParams& P, const int32_t* map_b, int t0, int s0) {
  typedef __attribute__((address_space(4))) const int32_t const_i32_t;
  if (t0 >= P.T || s0 >= P.T) return 0;
  return ((const_i32_t*)map_b)[static_cast<int64_t>(t0 / P.block) * P.nb + s0 / P.block];
}

// Logits in log2 units of 4 keys sb + e against query tq (S^T accumulator st) in a tile or
// sub-tile of class cls > 0: x2 = scale log2(e) q.k + log2(w) (sl2 = scale log2(e)), -inf where
// the weight is 0 or the query / key is past T.  inner: all of it lies inside T; one weight
// then takes one fma per score.
__device__ __forceinline__ void sab_logits4(const AbParams& P, int tq, int sb, int cls, bool inner, float sl2,
                                            f32x4_t& st) {
  if (P.mode == FSI_SATTN_BLOCK_LIST || (cls & 2)) {
    const float lw2 = P.mode == FSI_SATTN_BLOCK_LIST ? __log2f(static_cast<float>(cls)) : 0.f;
    if (inner) {
#pragma unroll
      for (int e = 0; e < 4; ++e) st[e] = fmaf(st[e], sl2, lw2);
    } else {
      const int lim = tq < P.T ? P.T : 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) st[e] = sb + e < lim ? fmaf(st[e], sl2, lw2) : -INFINITY;
    }
  } else {
    const int hi = tq < P.T ? tq : -1, lo = tq - P.window;
#pragma unroll
    for (int e = 0; e < 4; ++e) st[e] = sb + e <= hi && sb + e > lo ? st[e] * sl2 : -INFINITY;
  }
}

// How the weights of a tile or sub-tile of class cls >= 0 are applied: one weight (all, its
// log2 lw2), the window only (win), or nothing attended.
struct SabWeight {
  bool all, win;
  float lw2;
};
__device__ __forceinline__ SabWeight sab_weight_of(const AbParams& P, int cls) {
  const bool list = P.mode == FSI_SATTN_BLOCK_LIST;
  const bool all = cls > 0 && (list || (cls & 2));
  return {all, cls > 0 && !all, all && list ? __log2f(static_cast<float>(cls)) : 0.f};
}
// P of query t and key sk from the raw score and the query's log2 denominator (+inf past T: P = 0).
__device__ __forceinline__ float sab_p(const AbParams& P, const SabWeight& w, int t, int sk, bool inner, float sl2,
                                       float lse, float s) {
  float p = 0.f;
  if (w.all) {
    p = __builtin_amdgcn_exp2f(fmaf(s, sl2, w.lw2 - lse));
    if (!inner) p = sk < P.T ? p : 0.f;
  } else if (w.win) {
    const float x = __builtin_amdgcn_exp2f(fmaf(s, sl2, -lse));
    p = sk <= t && sk > t - P.window ? x : 0.f;
  }
  return p;
}

// sab_logits4 for keys sb + 16 t + 4 kg + e of a tile of class tcls against query tq0 + r.
template <int N, int MIX>
__device__ __forceinline__ void sab_logits2(const AbParams& P, const int32_t* map_b, int tq0, int r, int kg, int sb,
                                            int tcls, bool inner, float sl2, f32x4_t (&st)[N]) {
  const int tq = tq0 + r;
#pragma unroll
  for (int t = 0; t < N; ++t) {
    const int s0 = sb + 16 * t;
    if (MIX == SAB_TILE || tcls > 0) {
      sab_logits4(P, tq, s0 + 4 * kg, tcls, inner, sl2, st[t]);
    } else if constexpr (MIX == SAB_SUB) {
      const int cls = sab_sub_class(P, map_b, tq0, s0);
      if (cls > 0) sab_logits4(P, tq, s0 + 4 * kg, cls, inner, sl2, st[t]);
      else st[t] = f32x4_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int sk = s0 + 4 * kg + e;
        float x = -INFINITY;
        if (tq < P.T && sk < P.T) {
          const float w = sab_tile_weight(P, map_b, tcls, tq, sk);
          if (w > 0.f) x = fmaf(st[t][e], sl2, __log2f(w));
        }
        st[t][e] = x;
      }
    }
  }
}

__device__ __forceinline__ uint32_t bf_cvt2(float a, float b) {
  typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_t;
  const bf16x2_t v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  return __builtin_bit_cast(uint32_t, v);
}
// The lane's 8 k-slot values (4 of accumulator a, then 4 of b) as hi + lo bf16 operands.
__device__ __forceinline__ void bf_split8(const f32x4_t& a, const f32x4_t& b, u32x4_t& hi, u32x4_t& lo) {
  float x[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const uint32_t h = bf_cvt2(x[2 * w], x[2 * w + 1]);
    hi[w] = h;
    lo[w] = bf_cvt2(x[2 * w] - __uint_as_float(h << 16), x[2 * w + 1] - __uint_as_float(h & 0xffff0000u));
  }
}

// dQ and the row statistics (as sab_q_kernel).  A workgroup is HP query heads of one KV head
// (they share the K / V tiles and the block lists) at 64 queries; wave (head, half) owns 32
// of them.  With one head (an odd number of them per KV head) four waves share it too: wave
// (key half, query half) takes 32 keys of every tile, and the halves' statistics and dQ meet
// in LDS.  Two waves a workgroup leave one wave per SIMD: whole backward, 32 / 32 heads of 128,
// 8192 tokens 2583 us with two and 2095 with four; 4 x 2048 tokens, 4 / 4 heads of 32, blocks of
// 10 (classes per element) 667 and 427.  Consecutive workgroups are consecutive KV heads (one
// XCD each when there are eight), the latest query tiles first.
template <int HD, int HP, int MIX>
__global__ __launch_bounds__(AB_THREADS, 2) void sab_q_bf_kernel(AbParams P) {
  constexpr int DG = HD / 16, KS32 = HD / 32, NT = AB_THREADS, TB = sab_tile_bytes<HD>();
  static_assert(HP == 1 || HP == 2, "four waves: two heads or two key halves");
  constexpr int JN = HP;  // 32-key parts of a tile that a wave takes
  // one array: separate ones get alias scopes, and every LDS read would then wait for the
  // direct loads in flight
  __shared__ __attribute__((aligned(1024))) char smem[4 * TB];  // [stage][K, V]
  const int ntiles = (P.T + AB_T - 1) / AB_T, nhp = P.Hq / HP;
  const int t0 = (ntiles - 1 - static_cast<int>(blockIdx.x) / nhp) * AB_T;
  const int hp = static_cast<int>(blockIdx.x) % nhp, g = hp % P.Hkv;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.y, h = g * (P.Hq / P.Hkv) + hp / P.Hkv * HP + (HP == 2 ? wave >> 1 : 0);
  const int j0 = HP == 2 ? 0 : wave >> 1;  // first of them
  const int r = lane & 15, kg = lane >> 4;
  const int tw = t0 + 32 * (wave & 1);  // this wave's queries tw + 16 i + r
  const bf16_t* q = static_cast<const bf16_t*>(P.q) + b * P.qs_b + h * P.qs_h;
  const bf16_t* o = static_cast<const bf16_t*>(P.o) + b * P.os_b + h * P.os_h;
  const bf16_t* dout = static_cast<const bf16_t*>(P.dout) + b * P.ds_b + h * P.ds_h;
  const bf16_t* k = static_cast<const bf16_t*>(P.k) + b * P.ks_b + g * P.ks_h;
  const bf16_t* v = static_cast<const bf16_t*>(P.v) + b * P.vs_b + g * P.vs_h;
  const int32_t* map_b = P.map + static_cast<int64_t>(b) * P.nb * P.nb;

  u32x4_t qb[2][KS32], db[2][KS32];
  float dd[2];  // D = dout . out of query tw + 16 i + r
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int tq = tw + 16 * i + r, tql = tq < P.T ? tq : P.T - 1;
    sab_row_frag_bf<bf16_t, HD>(q, P.qs_t, tql, HD, kg, qb[i]);
    sab_row_frag_bf<bf16_t, HD>(dout, P.ds_t, tql, HD, kg, db[i]);
    f32x4_t of[DG], df[DG];
    sab_row_frag<bf16_t, HD>(o, P.os_t, tql, HD, kg, of);
    sab_row_frag<bf16_t, HD>(dout, P.ds_t, tql, HD, kg, df);
    float part = 0.f;
#pragma unroll
    for (int d = 0; d < DG; ++d)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) part = fmaf(df[d][kk], of[d][kk], part);
    dd[i] = sum_rows4(part);
  }
  const uint32_t row_off = sab_row_off<HD>(r, kg), tr_off = sab_tr_off<HD>(r, kg);
  // S^T (dP^T) of 32 keys of a tile against this wave's queries
  auto scores = [&](f32x4_t (&st)[2][2], uint32_t off, const u32x4_t (&bb)[2][KS32]) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      st[0][t] = st[1][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS32; ++ks) {
        const u32x4_t a = sab_row(smem, off, ks, 16 * t * HD * 2);
        st[0][t] = mfma16x16x32(a, bb[0][ks], st[0][t]);
        st[1][t] = mfma16x16x32(a, bb[1][ks], st[1][t]);
      }
    }
  };

  // pass 1: row maximum and sum (log2 units) over the live key tiles
  const float sl2 = P.scale * 1.4426950408889634f;
  float m[2] = {-INFINITY, -INFINITY}, lpart[2] = {0.f, 0.f};
  {
    SabTiles<true> it(P, map_b, t0, ntiles);
    bool more = it.next();
    if (more) sab_dma<HD, NT>(k, P.ks_t, it.tile * AB_T, P.T, smem);
    int stage = 0;
    __syncthreads();
    while (more) {
      const int s0 = it.tile * AB_T, tcls = it.cls;
      const uint32_t ko = row_off + stage * 2 * TB;
      stage ^= 1;
      more = it.next();
      if (more) sab_dma<HD, NT>(k, P.ks_t, it.tile * AB_T, P.T, smem + stage * 2 * TB);
      const bool inner = t0 + AB_T <= P.T && s0 + AB_T <= P.T;
      f32x4_t st[2][2 * JN];
#pragma unroll
      for (int j = 0; j < JN; ++j) {
        f32x4_t x[2][2];
        scores(x, ko + 32 * (j0 + j) * HD * 2, qb);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          st[i][2 * j] = x[i][0];
          st[i][2 * j + 1] = x[i][1];
        }
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        sab_logits2<2 * JN, MIX>(P, map_b, tw + 16 * i, r, kg, s0 + 32 * j0, tcls, inner, sl2, st[i]);
        float cm = -INFINITY;
#pragma unroll
        for (int t = 0; t < 2 * JN; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) cm = fmaxf(cm, st[i][t][e]);
        cm = max_rows4(cm);
        if (cm > -INFINITY) {
          const float mn = fmaxf(m[i], cm);
          float add = 0.f;
#pragma unroll
          for (int t = 0; t < 2 * JN; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) add += __builtin_amdgcn_exp2f(st[i][t][e] - mn);
          lpart[i] = (m[i] > -INFINITY ? lpart[i] * __builtin_amdgcn_exp2f(m[i] - mn) : 0.f) + add;
          m[i] = mn;
        }
      }
      __syncthreads();
    }
  }
  // log2 of the row's softmax denominator: P = exp2(x2 - lse2); +inf for a row with no key
  // or past T (every P 0, no NaN)
  float lse2[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) lpart[i] = sum_rows4(lpart[i]);
  if constexpr (HP == 1) {  // [key half][max, sum][query]
    float* sums = reinterpret_cast<float*>(smem) + 32 * (wave & 1) + r;
    if (kg == 0)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        sums[2 * j0 * AB_T + 16 * i] = m[i];
        sums[(2 * j0 + 1) * AB_T + 16 * i] = lpart[i];
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float* s = sums + 16 * i;
      const float m0 = s[0], m1 = s[2 * AB_T];
      m[i] = fmaxf(m0, m1);
      lpart[i] = (m0 > -INFINITY ? s[AB_T] * __builtin_amdgcn_exp2f(m0 - m[i]) : 0.f) +
                 (m1 > -INFINITY ? s[3 * AB_T] * __builtin_amdgcn_exp2f(m1 - m[i]) : 0.f);
    }
    __syncthreads();  // the tiles take the memory
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float l = lpart[i];
    lse2[i] = l > 0.f && tw + 16 * i + r < P.T ? m[i] + __log2f(l) : INFINITY;
  }

  // pass 2: dQ^T[dim][query] = sum_key K^T[dim][key] dS^T[key][query]
  f32x4_t dqa[2][DG];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int dt = 0; dt < DG; ++dt) dqa[i][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  {
    SabTiles<true> it(P, map_b, t0, ntiles);
    auto load = [&](int stage) {
      sab_dma<HD, NT>(k, P.ks_t, it.tile * AB_T, P.T, smem + stage * 2 * TB);
      sab_dma<HD, NT>(v, P.vs_t, it.tile * AB_T, P.T, smem + stage * 2 * TB + TB);
    };
    bool more = it.next();
    if (more) load(0);
    int stage = 0;
    __syncthreads();
    while (more) {
      const int s0 = it.tile * AB_T, tcls = it.cls;
      const int cur = stage * 2 * TB;
      stage ^= 1;
      more = it.next();
      if (more) load(stage);
      const bool inner = t0 + AB_T <= P.T && s0 + AB_T <= P.T;
#pragma unroll 1
      for (int j = j0; j < j0 + JN; ++j) {  // 32 keys at a time (not unrolled: register budget)
        f32x4_t st[2][2], dp[2][2];
        const uint32_t at = cur + 32 * j * HD * 2;
        scores(st, row_off + at, qb);
        scores(dp, row_off + at + TB, db);  // dP^T = V dout^T
        u32x4_t hi[2], lo[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          sab_logits2<2, MIX>(P, map_b, tw + 16 * i, r, kg, s0 + 32 * j, tcls, inner, sl2, st[i]);
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              st[i][t][e] = __builtin_amdgcn_exp2f(st[i][t][e] - lse2[i]) * (dp[i][t][e] - dd[i]);  // dS^T
          bf_split8(st[i][0], st[i][1], hi[i], lo[i]);
        }
#pragma unroll
        for (int dt = 0; dt < DG; ++dt) {
          const u32x4_t a = sab_trow<HD>(smem, tr_off + at, dt, 0);
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            dqa[i][dt] = mfma16x16x32(a, hi[i], dqa[i][dt]);
            dqa[i][dt] = mfma16x16x32(a, lo[i], dqa[i][dt]);
          }
        }
      }
      __syncthreads();
    }
  }
  if constexpr (HP == 1) {  // the second key half hands its sums over, the first stores
    f32x4_t* part = reinterpret_cast<f32x4_t*>(smem) + (wave & 1) * (2 * DG * 64) + lane;
    if (j0 == 1)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int dt = 0; dt < DG; ++dt) part[(i * DG + dt) * 64] = dqa[i][dt];
    __syncthreads();
    if (j0 == 1) return;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int dt = 0; dt < DG; ++dt) dqa[i][dt] += part[(i * DG + dt) * 64];
  }
  const int64_t row0 = static_cast<int64_t>(b) * P.Hq + h;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int tq = tw + 16 * i + r;
    if (tq < P.T) {
#pragma unroll
      for (int dt = 0; dt < DG; ++dt)
        *reinterpret_cast<f32x4_t*>(&P.dq[(row0 * P.T + tq) * HD + 16 * dt + 4 * kg]) = dqa[i][dt] * P.scale;
    }
    if (kg == 0) {  // statistics of whole tiles: rows past T get P = 0
      P.stat_m[row0 * P.tp + tq] = lse2[i];
      P.stat_d[row0 * P.tp + tq] = dd[i];
    }
  }
}

// dK and dV (as sab_kv_kernel): wave (query half, key half) owns 32 keys and, of every
// query tile, 32 queries; the two query halves' sums meet in LDS at the end.
template <int HD, int MIX>
__global__ __launch_bounds__(AB_THREADS, 2) void sab_kv_bf_kernel(AbParams P) {
  constexpr int DG = HD / 16, KS32 = HD / 32, TB = sab_tile_bytes<HD>();
  constexpr int STAGE = 2 * TB + 2 * AB_T * 4;  // Q, dout, then lse2 and D of the rows
  constexpr int SUMS = 2 * 2 * 2 * DG * 64 * 16;  // two waves' dK and dV accumulators
  __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE > SUMS ? 2 * STAGE : SUMS];
  const int ntiles = (P.T + AB_T - 1) / AB_T;
  const int s0 = static_cast<int>(blockIdx.x / P.Hkv) * AB_T;
  const float sl2 = P.scale * 1.4426950408889634f;
  const int b = blockIdx.y, g = blockIdx.x % P.Hkv;
  const int G = P.Hq / P.Hkv;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, kg = lane >> 4;
  const int wq = wave >> 1, sw = s0 + 32 * (wave & 1);  // this wave's keys sw + 16 kt + r
  const bf16_t* k = static_cast<const bf16_t*>(P.k) + b * P.ks_b + g * P.ks_h;
  const bf16_t* v = static_cast<const bf16_t*>(P.v) + b * P.vs_b + g * P.vs_h;
  const int32_t* map_b = P.map + static_cast<int64_t>(b) * P.nb * P.nb;
  u32x4_t kb[2][KS32], vb[2][KS32];
  f32x4_t dka[2][DG], dva[2][DG];
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
    const int sk = sw + 16 * kt + r, skl = sk < P.T ? sk : P.T - 1;
    sab_row_frag_bf<bf16_t, HD>(k, P.ks_t, skl, HD, kg, kb[kt]);
    sab_row_frag_bf<bf16_t, HD>(v, P.vs_t, skl, HD, kg, vb[kt]);
#pragma unroll
    for (int dt = 0; dt < DG; ++dt) dka[kt][dt] = dva[kt][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  const uint32_t row_off = sab_row_off<HD>(r, kg) + 32 * wq * HD * 2;
  const uint32_t tr_off = sab_tr_off<HD>(r, kg) + 32 * wq * HD * 2;
  // (live query tile, query head of the group) pairs
  SabTiles<false> it(P, map_b, s0, ntiles);
  int hh = G - 1;
  auto next = [&]() {
    if (++hh < G) return true;
    hh = 0;
    return it.next();
  };
  auto load = [&](int stage) {
    char* S = smem + stage * STAGE;
    const int h = g * G + hh, t0 = it.tile * AB_T;
    sab_dma<HD, AB_THREADS>(static_cast<const bf16_t*>(P.q) + b * P.qs_b + h * P.qs_h, P.qs_t, t0, P.T, S);
    sab_dma<HD, AB_THREADS>(static_cast<const bf16_t*>(P.dout) + b * P.ds_b + h * P.ds_h, P.ds_t, t0, P.T, S + TB);
    if (wave < 2) {  // the statistics cover whole tiles
      const float* st = (wave ? P.stat_d : P.stat_m) + (static_cast<int64_t>(b) * P.Hq + h) * P.tp + t0 + lane;
      __builtin_amdgcn_global_load_lds((ab_glb_t*)st, (ab_lds_t*)(S + 2 * TB + wave * AB_T * 4), 4, 0, 0);
    }
  };
  bool more = next();
  if (more) load(0);
  int stage = 0;
  __syncthreads();
  while (more) {
    const int t0 = it.tile * AB_T, tcls = it.cls;
    const bool inner = t0 + AB_T <= P.T && s0 + AB_T <= P.T;
    const SabWeight wt = sab_weight_of(P, tcls);
    const int cur = stage * STAGE;
    stage ^= 1;
    more = next();
    if (more) load(stage);
    f32x4_t s[2][2], dp[2][2];  // [key half][16-query part]: query 32 wq + 16 i + 4 kg + e, key r
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      s[0][i] = s[1][i] = dp[0][i] = dp[1][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS32; ++ks) {
        const u32x4_t aq = sab_row(smem, row_off + cur, ks, 16 * i * HD * 2);
        const u32x4_t ad = sab_row(smem, row_off + cur, ks, 16 * i * HD * 2 + TB);
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
          s[kt][i] = mfma16x16x32(aq, kb[kt][ks], s[kt][i]);
          dp[kt][i] = mfma16x16x32(ad, vb[kt][ks], dp[kt][i]);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // register budget: keep the phases apart
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int rq = 32 * wq + 16 * i + 4 * kg;
      const float* rows = reinterpret_cast<const float*>(smem + cur + 2 * TB) + rq;
      const f32x4_t lse = *reinterpret_cast<const f32x4_t*>(rows);  // +inf past T: P = 0
      const f32x4_t rd = *reinterpret_cast<const f32x4_t*>(rows + AB_T);
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const int sk0 = sw + 16 * kt, sk = sk0 + r, t = t0 + rq;
        SabWeight w = wt;
        if (MIX == SAB_SUB && tcls < 0)
          w = sab_weight_of(P, sab_sub_class(P, map_b, t0 + 32 * wq + 16 * i, sk0));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float p;
          if (MIX == SAB_ELEM && tcls < 0) {
            p = 0.f;
            if (t + e < P.T && sk < P.T) {
              const float we = sab_tile_weight(P, map_b, tcls, t + e, sk);
              if (we > 0.f) p = __builtin_amdgcn_exp2f(fmaf(s[kt][i][e], sl2, __log2f(we) - lse[e]));
            }
          } else {
            p = sab_p(P, w, t + e, sk, inner, sl2, lse[e], s[kt][i][e]);
          }
          s[kt][i][e] = p;
          dp[kt][i][e] = p * (dp[kt][i][e] - rd[e]);  // dS
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // register budget: keep the phases apart
    // dV^T[dim][key] += dout^T[dim][query] P[query][key], dK^T += Q^T dS
    u32x4_t ph[2], pl[2], dh[2], dl[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      bf_split8(s[kt][0], s[kt][1], ph[kt], pl[kt]);
      bf_split8(dp[kt][0], dp[kt][1], dh[kt], dl[kt]);
    }
#pragma unroll
    for (int dt = 0; dt < DG; ++dt) {
      const u32x4_t ad = sab_trow<HD>(smem, tr_off + cur, dt, TB);
      const u32x4_t aq = sab_trow<HD>(smem, tr_off + cur, dt, 0);
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        dva[kt][dt] = mfma16x16x32(ad, ph[kt], dva[kt][dt]);
        dva[kt][dt] = mfma16x16x32(ad, pl[kt], dva[kt][dt]);
        dka[kt][dt] = mfma16x16x32(aq, dh[kt], dka[kt][dt]);
        dka[kt][dt] = mfma16x16x32(aq, dl[kt], dka[kt][dt]);
      }
    }
    __syncthreads();
  }
  // the second query half hands its sums over, the first stores
  f32x4_t* sums = reinterpret_cast<f32x4_t*>(smem) + (wave & 1) * (4 * DG * 64) + lane;
  if (wq == 1) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int dt = 0; dt < DG; ++dt) {
        sums[(2 * (kt * DG + dt)) * 64] = dka[kt][dt];
        sums[(2 * (kt * DG + dt) + 1) * 64] = dva[kt][dt];
      }
  }
  __syncthreads();
  if (wq == 1) return;
  const int64_t kbase = (static_cast<int64_t>(b) * P.Hkv + g) * P.T;
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
    const int sk = sw + 16 * kt + r;
    if (sk >= P.T) continue;
#pragma unroll
    for (int dt = 0; dt < DG; ++dt) {
      const int64_t at = (kbase + sk) * HD + 16 * dt + 4 * kg;
      *reinterpret_cast<f32x4_t*>(&P.dk[at]) = (dka[kt][dt] + sums[(2 * (kt * DG + dt)) * 64]) * P.scale;
      *reinterpret_cast<f32x4_t*>(&P.dv[at]) = dva[kt][dt] + sums[(2 * (kt * DG + dt) + 1) * 64];
    }
  }
}

// Workspace: the counter area (left untouched), the block map, then m, l, D.
size_t sab_map_bytes(int64_t B, int64_t T, int64_t block) {
  const int64_t nb = (T + block - 1) / block;
  return fsi_host::align_up(sizeof(int32_t) * static_cast<size_t>(B * nb * nb), 256);
}

// One statistic of every query row, T rounded up to whole tiles.
size_t sab_stat_bytes(int64_t B, int64_t Hq, int64_t T) {
  return fsi_host::align_up(sizeof(float) * static_cast<size_t>(B * Hq * ((T + AB_T - 1) / AB_T * AB_T)), 256);
}

}  // namespace

extern "C" {

FSI_API size_t fsi_sparse_attn_bwd_workspace_size(int64_t B, int64_t Hq, int64_t T, int64_t block) {
  if (B <= 0 || Hq <= 0 || T <= 0 || block <= 0) return 0;
  return FSI_WORKSPACE_COUNTER_BYTES + sab_map_bytes(B, T, block) + 3 * sab_stat_bytes(B, Hq, T);
}

FSI_API int fsi_sparse_attn_bwd(const void* q, int64_t qs_b, int64_t qs_h, int64_t qs_t, const void* k, int64_t ks_b,
                                int64_t ks_h, int64_t ks_t, const void* v, int64_t vs_b, int64_t vs_h, int64_t vs_t,
                                const void* out, int64_t os_b, int64_t os_h, int64_t os_t, const void* dout,
                                int64_t ds_b, int64_t ds_h, int64_t ds_t, int64_t B, int64_t Hq, int64_t Hkv,
                                int64_t T, int64_t head_dim, int64_t block, int mode, int64_t window,
                                const int32_t* lists, int64_t ls_b, int64_t ls_q, int64_t capacity,
                                const int32_t* counts, int64_t cs_b, int64_t cs_q, float scale, int dtype, float* dq,
                                float* dk, float* dv, void* workspace, size_t workspace_bytes, int* err,
                                void* stream) {
  using namespace fsi_host;
  FSI_CHECK_ARG(dtype == FSI_DTYPE_F32 || dtype == FSI_DTYPE_BF16, FSI_ERR_DTYPE, "sparse_attn_bwd: dtype %d", dtype);
  FSI_CHECK_ARG(mode == FSI_SATTN_LOCAL_REMOTE || mode == FSI_SATTN_BLOCK_LIST, FSI_ERR_INVALID_ARG,
                "sparse_attn_bwd: mode %d", mode);
  FSI_CHECK_ARG(head_dim >= 1 && head_dim <= 128, FSI_ERR_SHAPE, "sparse_attn_bwd: head_dim %lld (1..128)",
                (long long)head_dim);
  FSI_CHECK_ARG(B > 0 && T > 0 && Hkv > 0 && Hq > 0 && Hq % Hkv == 0 && block > 0, FSI_ERR_SHAPE,
                "sparse_attn_bwd: B=%lld T=%lld Hq=%lld Hkv=%lld block=%lld", (long long)B, (long long)T,
                (long long)Hq, (long long)Hkv, (long long)block);
  FSI_CHECK_ARG(T <= (int64_t(1) << 30) && B <= 65535 && (T + AB_T - 1) / AB_T * Hq <= 0x7fffffff, FSI_ERR_SHAPE,
                "sparse_attn_bwd: sizes beyond range");
  const int64_t nb = (T + block - 1) / block;
  FSI_CHECK_ARG(nb <= 65535 && B * nb * nb <= (int64_t(1) << 31), FSI_ERR_SHAPE,
                "sparse_attn_bwd: %lld blocks per sequence beyond the block map", (long long)nb);
  FSI_CHECK_ARG(capacity >= 0 && capacity <= 4096, FSI_ERR_CAPACITY, "sparse_attn_bwd: capacity %lld",
                (long long)capacity);
  FSI_CHECK_ARG(mode != FSI_SATTN_LOCAL_REMOTE || window > 0, FSI_ERR_SHAPE, "sparse_attn_bwd: window %lld",
                (long long)window);
  FSI_CHECK_ARG(q && k && v && out && dout && counts && (lists || capacity == 0) && dq && dk && dv, FSI_ERR_INVALID_ARG,
                "sparse_attn_bwd: null pointer");
  const size_t need = fsi_sparse_attn_bwd_workspace_size(B, Hq, T, block);
  FSI_CHECK_ARG(workspace && workspace_bytes >= need && reinterpret_cast<uintptr_t>(workspace) % 16 == 0,
                FSI_ERR_WORKSPACE, "sparse_attn_bwd: workspace %zu < %zu (or misaligned)", workspace_bytes, need);
  AbParams P{};
  P.q = q;
  P.qs_b = qs_b;
  P.qs_h = qs_h;
  P.qs_t = qs_t;
  P.k = k;
  P.ks_b = ks_b;
  P.ks_h = ks_h;
  P.ks_t = ks_t;
  P.v = v;
  P.vs_b = vs_b;
  P.vs_h = vs_h;
  P.vs_t = vs_t;
  P.o = out;
  P.os_b = os_b;
  P.os_h = os_h;
  P.os_t = os_t;
  P.dout = dout;
  P.ds_b = ds_b;
  P.ds_h = ds_h;
  P.ds_t = ds_t;
  P.B = (int)B;
  P.Hq = (int)Hq;
  P.Hkv = (int)Hkv;
  P.T = (int)T;
  P.hd = (int)head_dim;
  P.block = (int)block;
  P.mode = mode;
  P.window = (int)(window < 0x7fffffff ? window : 0x7fffffff);
  P.lists = lists;
  P.ls_b = ls_b;
  P.ls_q = ls_q;
  P.cap = (int)capacity;
  P.counts = counts;
  P.cs_b = cs_b;
  P.cs_q = cs_q;
  P.scale = scale;
  P.nb = (int)nb;
  {
    const int64_t esz = dtype == FSI_DTYPE_F32 ? 4 : 2;
    auto al = [&](const void* p, int64_t sb, int64_t sh, int64_t st) {
      return reinterpret_cast<uintptr_t>(p) % (4 * esz) == 0 && sb % 4 == 0 && sh % 4 == 0 && st % 4 == 0;
    };
    P.vec4 = (head_dim == 16 || head_dim == 32 || head_dim == 64 || head_dim == 128) && al(q, qs_b, qs_h, qs_t) && al(k, ks_b, ks_h, ks_t) && al(v, vs_b, vs_h, vs_t) &&
             al(dout, ds_b, ds_h, ds_t);
  }
  char* ws = static_cast<char*>(workspace) + FSI_WORKSPACE_COUNTER_BYTES;
  P.map = reinterpret_cast<int32_t*>(ws);
  P.tp = (T + AB_T - 1) / AB_T * AB_T;
  const size_t st_bytes = sab_stat_bytes(B, Hq, T);
  P.stat_m = reinterpret_cast<float*>(ws + sab_map_bytes(B, T, block));
  P.stat_l = reinterpret_cast<float*>(ws + sab_map_bytes(B, T, block) + st_bytes);
  P.stat_d = reinterpret_cast<float*>(ws + sab_map_bytes(B, T, block) + 2 * st_bytes);
  P.dq = dq;
  P.dk = dk;
  P.dv = dv;
  P.err = err;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  sab_map_kernel<<<dim3(static_cast<unsigned>(nb), static_cast<unsigned>(B)), AB_THREADS, 0, st>>>(P);
  const unsigned ntiles = static_cast<unsigned>((T + AB_T - 1) / AB_T);
  const dim3 gq(ntiles * static_cast<unsigned>(Hq), static_cast<unsigned>(B)),
      gkv(ntiles * static_cast<unsigned>(Hkv), static_cast<unsigned>(B));
  auto run = [&](auto hd_tag) {
    constexpr int HD = decltype(hd_tag)::value;
    if (dtype == FSI_DTYPE_F32) {
      sab_q_kernel<float, HD><<<gq, AB_THREADS, 0, st>>>(P);
      sab_kv_kernel<float, HD><<<gkv, AB_THREADS, 0, st>>>(P);
    } else {
      if constexpr (HD >= 32) {
        // the bf16 kernels move 16-byte pieces and address a tile's rows with 32-bit
        // offsets: rows 8-element aligned, row strides below 2^24
        auto al8 = [&](const void* p, int64_t sb, int64_t sh, int64_t stt) {
          return reinterpret_cast<uintptr_t>(p) % 16 == 0 && sb % 8 == 0 && sh % 8 == 0 && stt % 8 == 0 &&
                 stt >= 0 && stt < (int64_t(1) << 24);
        };
        const bool out16 = reinterpret_cast<uintptr_t>(dq) % 16 == 0 && reinterpret_cast<uintptr_t>(dk) % 16 == 0 &&
                           reinterpret_cast<uintptr_t>(dv) % 16 == 0;
        if (head_dim == HD && out16 && al8(q, qs_b, qs_h, qs_t) && al8(k, ks_b, ks_h, ks_t) &&
            al8(v, vs_b, vs_h, vs_t) && al8(dout, ds_b, ds_h, ds_t)) {
          auto launch = [&](auto mix_tag) {
            constexpr int MIX = decltype(mix_tag)::value;
            if ((Hq / Hkv) % 2 == 0) sab_q_bf_kernel<HD, 2, MIX><<<dim3(gq.x / 2, gq.y), AB_THREADS, 0, st>>>(P);
            else sab_q_bf_kernel<HD, 1, MIX><<<gq, AB_THREADS, 0, st>>>(P);
            sab_kv_bf_kernel<HD, MIX><<<gkv, AB_THREADS, 0, st>>>(P);
          };
          if (block % AB_T == 0) launch(sab_mix_t<SAB_TILE>{});
          else if (block % 16 == 0) launch(sab_mix_t<SAB_SUB>{});
          else launch(sab_mix_t<SAB_ELEM>{});
          return;
        }
      }
      sab_q_kernel<bf16_t, HD><<<gq, AB_THREADS, 0, st>>>(P);
      sab_kv_kernel<bf16_t, HD><<<gkv, AB_THREADS, 0, st>>>(P);
    }
  };
  if (head_dim <= 16) run(std::integral_constant<int, 16>{});
  else if (head_dim <= 32) run(std::integral_constant<int, 32>{});
  else if (head_dim <= 64) run(std::integral_constant<int, 64>{});
  else run(std::integral_constant<int, 128>{});
  FSI_HIP_LAUNCH_CHECK("sparse_attn_bwd");
  return FSI_OK;
}

}  // extern "C"
