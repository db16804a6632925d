// Training path of FovealPattentionMLP around its library GEMMs
// (foveal_indexer/foveal_pattention.py:257-262, 292-307, 328-342):
//
//   router    z = rms_norm(q), s = z . keys^T / 4 per token, p = softmax(s / T),
//             context = p . keys, and the active list [0 .. base) ++ topk(mean_tokens(s)[base:])
//   gather    the active blocks' rows of k_gate and k_up as one matrix and of v as another,
//             so gate and up are one GEMM forward, and one for x and one for the weights back
//   swiglu    act = silu(g) u of the [g | u] rows, and its backward
//   scatter   the active rows' weight gradients into the dense ones, zero elsewhere
//
// Everything here is bound by memory or, at the usual micro-batch, by launches: as torch ops
// the same steps are some 70 launches (index_put sorts among them) beside the GEMMs.  2048
// tokens of the default layer (2048 hidden, 24 of 96 blocks), forward and backward: 92 -> 25
// launches, 650 -> 330 us of kernels (210 of them GEMMs), 1.28 -> 0.58 .. 0.80 ms a pass,
// which the host now sets (about 20 us for each library GEMM call).
#include <type_traits>

#include "fsi_common.h"

using namespace fsi;

namespace {

template <typename T>
__device__ __forceinline__ float ldf(const T* p, int64_t i) {
  if constexpr (sizeof(T) == 2) return bf16_to_f32(p[i]);
  else return p[i];
}
template <typename T>
__device__ __forceinline__ void stf(T* p, int64_t i, float v) {
  if constexpr (sizeof(T) == 2) p[i] = f32_to_bf16(v);
  else p[i] = v;
}
template <typename T>
__device__ __forceinline__ float round_to(float v) {
  if constexpr (sizeof(T) == 2) return round_bf16(v);
  else return v;
}

constexpr int RT_DIM = 16;     // index dimension
constexpr int RT_TOK = 16;     // tokens per tile: 16 lanes of a wave each
constexpr int RT_MAX_NB = 256; // blocks: keys and two coefficients per token and block within 64 KiB of LDS
constexpr int RT_MAX_WG = 256;
constexpr int RT_THREADS = 256;

__device__ __forceinline__ float sum16(float v) {
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 16);
  return v;
}
__device__ __forceinline__ float max16(float v) {
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 16));
  return v;
}

struct RouteArgs {
  const void* q;        // (M, 16) projected queries
  const void* keys;     // (nb, 16)
  int M, nb;
  float inv_t;          // 1 / temperature
  void* scores;         // (M, nb)
  void* ctx;            // (M, 16)
  float* part;          // (workgroups, nb) sums of the rounded scores; backward: (workgroups, nb, 16)
  const void* dscores;  // (M, nb) or null
  const void* dctx;     // (M, 16) or null
  void* dq;             // (M, 16)
};

// Scores are rounded where torch's ops round them (rms_norm, the product, the division), as
// the routing decides on them.
template <typename T>
__device__ __forceinline__ void route_z(const T* q, int64_t m, float (&x)[RT_DIM], float (&z)[RT_DIM], float& inv) {
  float ss = 0.f;
#pragma unroll
  for (int d = 0; d < RT_DIM; ++d) {
    x[d] = ldf<T>(q, m * RT_DIM + d);
    ss = fmaf(x[d], x[d], ss);
  }
  inv = rsqrtf(ss * (1.f / RT_DIM) + 1.1920929e-07f);
#pragma unroll
  for (int d = 0; d < RT_DIM; ++d) z[d] = round_to<T>(x[d] * inv);
}
template <typename T>
__device__ __forceinline__ float route_score(const float (&z)[RT_DIM], const float* key) {
  float s = 0.f;
#pragma unroll
  for (int d = 0; d < RT_DIM; ++d) s = fmaf(z[d], key[d], s);
  return round_to<T>(round_to<T>(s) * 0.25f);
}

constexpr int RT_KS = RT_DIM + 1;  // key row stride: the 16 lanes of a token read distinct banks

// 16 lanes a token (lane j: blocks j, j + 16, ..); a workgroup walks tiles of 16 tokens and
// sums its rounded scores per block, in token order, for the routing's mean.
template <typename T>
__global__ __launch_bounds__(RT_THREADS) void train_route_kernel(RouteArgs A) {
  extern __shared__ float lds[];
  float* keys = lds;                       // nb x RT_KS
  float* tile = lds + A.nb * RT_KS;        // RT_TOK x nb scores
  for (int i = threadIdx.x; i < A.nb * RT_DIM; i += RT_THREADS)
    keys[i / RT_DIM * RT_KS + i % RT_DIM] = ldf<T>(static_cast<const T*>(A.keys), i);
  const int j = threadIdx.x & 15, t = threadIdx.x >> 4;
  float col[RT_MAX_NB / RT_THREADS] = {};
  __syncthreads();
  for (int64_t m0 = static_cast<int64_t>(blockIdx.x) * RT_TOK; m0 < A.M; m0 += static_cast<int64_t>(gridDim.x) * RT_TOK) {
    const int64_t m = m0 + t;
    const bool live = m < A.M;
    float x[RT_DIM], z[RT_DIM], inv;
    route_z<T>(static_cast<const T*>(A.q), live ? m : A.M - 1, x, z, inv);
    float mx = -INFINITY;
    for (int b = j; b < A.nb; b += 16) {
      const float s = route_score<T>(z, keys + b * RT_KS);
      tile[t * A.nb + b] = live ? s : 0.f;
      if (live) stf<T>(static_cast<T*>(A.scores), m * A.nb + b, s);
      mx = fmaxf(mx, s);
    }
    mx = max16(mx);
    float l = 0.f, c[RT_DIM] = {};
    for (int b = j; b < A.nb; b += 16) {
      const float* key = keys + b * RT_KS;
      const float p = expf((route_score<T>(z, key) - mx) * A.inv_t);
      l += p;
#pragma unroll
      for (int d = 0; d < RT_DIM; ++d) c[d] = fmaf(p, key[d], c[d]);
    }
    l = sum16(l);
    float mine = 0.f;  // lane j keeps dimension j
#pragma unroll
    for (int d = 0; d < RT_DIM; ++d) {
      const float v = sum16(c[d]);
      mine = d == j ? v : mine;
    }
    if (live) stf<T>(static_cast<T*>(A.ctx), m * RT_DIM + j, mine / l);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RT_MAX_NB / RT_THREADS; ++i) {
      const int b = i * RT_THREADS + threadIdx.x;
      if (b < A.nb)
#pragma unroll
        for (int r = 0; r < RT_TOK; ++r) col[i] += tile[r * A.nb + b];
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < RT_MAX_NB / RT_THREADS; ++i) {
    const int b = i * RT_THREADS + threadIdx.x;
    if (b < A.nb) A.part[static_cast<int64_t>(blockIdx.x) * A.nb + b] = col[i];
  }
}

// Largest-first order of floats as integers, NaN first (torch.topk's order).
__device__ __forceinline__ uint32_t order_key(float f) {
  if (f != f) return 0xffffffffu;
  const uint32_t u = __float_as_uint(f == 0.f ? 0.f : f);
  return u & 0x80000000u ? ~u : u | 0x80000000u;
}

// Token means (workgroup sums in order), rounded as torch's mean, and the ranks of the
// remote ones (equal means: lower block first).  One workgroup.
template <typename T>
__global__ __launch_bounds__(RT_MAX_NB) void train_topk_kernel(const float* __restrict__ part, int n_wg, int M, int nb,
                                                               int base, int remote, int32_t* __restrict__ active) {
  __shared__ uint32_t key[RT_MAX_NB];
  const int b = threadIdx.x;
  if (b < nb) {
    float s = 0.f;
#pragma unroll 16
    for (int w = 0; w < n_wg; ++w) s += part[static_cast<int64_t>(w) * nb + b];
    key[b] = order_key(round_to<T>(s / static_cast<float>(M)));
  }
  __syncthreads();
  if (b < base) active[b] = b;
  if (b >= base && b < nb) {
    const uint32_t mine = key[b];
    int rank = 0;
    for (int o = base; o < nb; ++o) rank += key[o] > mine || (key[o] == mine && o < b);
    if (rank < remote) active[base + rank] = b;
  }
}

// dq of every token and this workgroup's dkeys.  Per token, with g_b = keys_b . dctx:
//   ds_b = p_b (g_b - sum p g) / T + dscores_b,  dz = sum_b ds_b keys_b / 4, dq through rms_norm;
//   dkeys_b = sum_tokens p_b dctx + ds_b z / 4, accumulated per thread over (block, dim) pairs
// from the tile's p and ds in LDS, in token order.
template <typename T, int NACC>
__global__ __launch_bounds__(RT_THREADS) void train_route_bwd_kernel(RouteArgs A) {
  extern __shared__ float lds[];
  float* keys = lds;                        // nb x RT_KS
  float* ps = lds + A.nb * RT_KS;           // RT_TOK x nb
  float* dss = ps + RT_TOK * A.nb;          // RT_TOK x nb
  float* zs = dss + RT_TOK * A.nb;          // RT_TOK x 16, then dctx
  float* cs = zs + RT_TOK * RT_DIM;
  for (int i = threadIdx.x; i < A.nb * RT_DIM; i += RT_THREADS)
    keys[i / RT_DIM * RT_KS + i % RT_DIM] = ldf<T>(static_cast<const T*>(A.keys), i);
  const int j = threadIdx.x & 15, t = threadIdx.x >> 4;
  float acc[NACC] = {};
  __syncthreads();
  for (int64_t m0 = static_cast<int64_t>(blockIdx.x) * RT_TOK; m0 < A.M; m0 += static_cast<int64_t>(gridDim.x) * RT_TOK) {
    const int64_t m = m0 + t;
    const bool live = m < A.M;
    const int64_t ml = live ? m : A.M - 1;
    float x[RT_DIM], z[RT_DIM], dc[RT_DIM], inv;
    route_z<T>(static_cast<const T*>(A.q), ml, x, z, inv);
#pragma unroll
    for (int d = 0; d < RT_DIM; ++d)
      dc[d] = A.dctx && live ? ldf<T>(static_cast<const T*>(A.dctx), ml * RT_DIM + d) : 0.f;
    float mx = -INFINITY;
    for (int b = j; b < A.nb; b += 16) mx = fmaxf(mx, route_score<T>(z, keys + b * RT_KS));
    mx = max16(mx);
    float l = 0.f, pg = 0.f;
    for (int b = j; b < A.nb; b += 16) {
      const float* key = keys + b * RT_KS;
      const float e = expf((route_score<T>(z, key) - mx) * A.inv_t);
      float g = 0.f;
#pragma unroll
      for (int d = 0; d < RT_DIM; ++d) g = fmaf(key[d], dc[d], g);
      ps[t * A.nb + b] = e;
      dss[t * A.nb + b] = g;
      l += e;
      pg = fmaf(e, g, pg);
    }
    l = sum16(l);
    pg = sum16(pg) / l;
    float dz[RT_DIM] = {};
    for (int b = j; b < A.nb; b += 16) {
      const float* key = keys + b * RT_KS;
      const float p = ps[t * A.nb + b] / l;
      float ds = p * (dss[t * A.nb + b] - pg) * A.inv_t;
      if (A.dscores) ds += ldf<T>(static_cast<const T*>(A.dscores), ml * A.nb + b);
      ds = live ? ds * 0.25f : 0.f;
      ps[t * A.nb + b] = live ? p : 0.f;
      dss[t * A.nb + b] = ds;
#pragma unroll
      for (int d = 0; d < RT_DIM; ++d) dz[d] = fmaf(ds, key[d], dz[d]);
    }
    float dot = 0.f, mine = 0.f, xj = 0.f, zj = 0.f, cj = 0.f;
#pragma unroll
    for (int d = 0; d < RT_DIM; ++d) {
      const float v = sum16(dz[d]);
      dot = fmaf(v, x[d], dot);
      mine = d == j ? v : mine;
      xj = d == j ? x[d] : xj;
      zj = d == j ? z[d] : zj;
      cj = d == j ? dc[d] : cj;
    }
    // z = x inv: dx = inv dz - x inv^3 (dz . x) / 16
    if (live) stf<T>(static_cast<T*>(A.dq), m * RT_DIM + j, inv * (mine - xj * inv * inv * dot * (1.f / RT_DIM)));
    zs[t * RT_DIM + j] = zj;
    cs[t * RT_DIM + j] = cj;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NACC; ++i) {
      const int e = i * RT_THREADS + threadIdx.x, b = e / RT_DIM, d = e % RT_DIM;
      if (b < A.nb)
#pragma unroll
        for (int r = 0; r < RT_TOK; ++r)
          acc[i] += ps[r * A.nb + b] * cs[r * RT_DIM + d] + dss[r * A.nb + b] * zs[r * RT_DIM + d];
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < NACC; ++i) {
    const int e = i * RT_THREADS + threadIdx.x;
    if (e < A.nb * RT_DIM) A.part[static_cast<int64_t>(blockIdx.x) * A.nb * RT_DIM + e] = acc[i];
  }
}

template <typename T>
__global__ __launch_bounds__(256) void train_dkeys_kernel(const float* __restrict__ part, int n_wg, int n,
                                                          T* __restrict__ dkeys) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
#pragma unroll 16
  for (int w = 0; w < n_wg; ++w) s += part[static_cast<int64_t>(w) * n + i];
  stf<T>(dkeys, i, s);
}

// 16-byte vectors (38 MB moved in 11 us at the size above, the scatter 110 MB in 18).  Gather: kgu rows [0, n) are k_gate's active rows, [n, 2 n) k_up's (n =
// active channels); vs is v's active rows (n, D), or with v_t (v stored (D, N_p)) its active
// columns (D, n).
struct RowsArgs {
  const void *gate, *up, *v;
  int64_t ldk, ldv;
  void *kgu, *vs;
  const int32_t* active;
  int n_active, block, n_blocks, D;
  bool v_t;
};
template <int ES>
__global__ __launch_bounds__(256) void train_gather_kernel(RowsArgs A) {
  constexpr int V = 16 / ES;
  const int64_t n = static_cast<int64_t>(A.n_active) * A.block;
  const int64_t rowv = A.D / V, colv = n / V, per = n * rowv;
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x, step = static_cast<int64_t>(gridDim.x) * 256;
  for (int64_t i = i0; i < 3 * per; i += step) {
    const int which = static_cast<int>(i / per);
    const int64_t k = i - which * per;
    u32x4_t val = u32x4_t{0u, 0u, 0u, 0u};
    if (which < 2 || !A.v_t) {
      const int64_t c = k / rowv, d = k % rowv * V;
      const int blk = A.active[c / A.block];
      const int64_t ld = which < 2 ? A.ldk : A.ldv;
      const char* src = static_cast<const char*>(which == 0 ? A.gate : which == 1 ? A.up : A.v);
      if (blk >= 0 && blk < A.n_blocks)
        val = *reinterpret_cast<const u32x4_t*>(src + ((static_cast<int64_t>(blk) * A.block + c % A.block) * ld + d) * ES);
      char* dst = which < 2 ? static_cast<char*>(A.kgu) + (which * n + c) * A.D * ES : static_cast<char*>(A.vs) + c * A.D * ES;
      *reinterpret_cast<u32x4_t*>(dst + d * ES) = val;
    } else {
      const int64_t d = k / colv, c = k % colv * V;
      const int blk = A.active[c / A.block];
      if (blk >= 0 && blk < A.n_blocks)
        val = *reinterpret_cast<const u32x4_t*>(static_cast<const char*>(A.v) +
                                                (d * A.ldv + static_cast<int64_t>(blk) * A.block + c % A.block) * ES);
      *reinterpret_cast<u32x4_t*>(static_cast<char*>(A.vs) + (d * n + c) * ES) = val;
    }
  }
}

// Dense weight gradients (contiguous (N_p, D), v's as (D, N_p) with v_t) from the active
// rows' ones: each output vector is written once, zero for a block that is not listed.
struct ScatterArgs {
  const void *dkgu, *dvs;
  void *dgate, *dup, *dv;  // null: not wanted
  const int32_t* active;
  int n_active, block, n_blocks, D;
  bool v_t;
};
template <int ES>
__global__ __launch_bounds__(256) void train_scatter_kernel(ScatterArgs A) {
  constexpr int V = 16 / ES;
  __shared__ int32_t slot[4096];  // list position of every block, -1 none
  for (int i = threadIdx.x; i < A.n_blocks; i += 256) slot[i] = -1;
  __syncthreads();
  for (int i = threadIdx.x; i < A.n_active; i += 256) {
    const int b = A.active[i];
    if (b >= 0 && b < A.n_blocks) slot[b] = i;
  }
  __syncthreads();
  const int64_t n = static_cast<int64_t>(A.n_active) * A.block, np = static_cast<int64_t>(A.n_blocks) * A.block;
  const int64_t rowv = A.D / V, colv = np / V, per = np * rowv;
  const int which = blockIdx.y;
  char* out = static_cast<char*>(which == 0 ? A.dgate : which == 1 ? A.dup : A.dv);
  if (!out) return;
  const int64_t step = static_cast<int64_t>(gridDim.x) * 256;
  for (int64_t k = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; k < per; k += step) {
    u32x4_t val = u32x4_t{0u, 0u, 0u, 0u};
    if (which < 2 || !A.v_t) {
      const int64_t c = k / rowv, d = k % rowv * V;
      const int s = slot[c / A.block];
      if (s >= 0) {
        const int64_t row = static_cast<int64_t>(s) * A.block + c % A.block + (which == 1 ? n : 0);
        val = *reinterpret_cast<const u32x4_t*>(static_cast<const char*>(which < 2 ? A.dkgu : A.dvs) + (row * A.D + d) * ES);
      }
      *reinterpret_cast<u32x4_t*>(out + (c * A.D + d) * ES) = val;
    } else {
      const int64_t d = k / colv, c = k % colv * V;
      const int s = slot[c / A.block];
      if (s >= 0)
        val = *reinterpret_cast<const u32x4_t*>(static_cast<const char*>(A.dvs) +
                                                (d * n + static_cast<int64_t>(s) * A.block + c % A.block) * ES);
      *reinterpret_cast<u32x4_t*>(out + (d * np + c) * ES) = val;
    }
  }
}

// act[m][c] = silu(g) u from gu[m] = [g | u] (n each); backward: dgu[m] = [dg | du] with
// s = sigmoid(g), du = d g s, dg = d u s (1 + g (1 - s)).  fp32, one rounding.
template <typename T>
struct Vec {
  static constexpr int N = 16 / static_cast<int>(sizeof(T));
  float v[N];
  __device__ __forceinline__ explicit Vec(const T* p) {
    const u32x4_t w = *reinterpret_cast<const u32x4_t*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (sizeof(T) == 2) {
        v[2 * i] = lo_bf16(w[i]);
        v[2 * i + 1] = hi_bf16(w[i]);
      } else {
        v[i] = __uint_as_float(w[i]);
      }
    }
  }
  __device__ __forceinline__ void store(T* p) const {
    u32x4_t w;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (sizeof(T) == 2) w[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
      else w[i] = __float_as_uint(v[i]);
    }
    *reinterpret_cast<u32x4_t*>(p) = w;
  }
};
template <typename T>
__global__ __launch_bounds__(256) void swiglu_pair_kernel(const T* __restrict__ gu, int64_t M, int64_t n,
                                                          T* __restrict__ act) {
  constexpr int V = Vec<T>::N;
  const int64_t nv = n / V, step = static_cast<int64_t>(gridDim.x) * 256;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < M * nv; i += step) {
    const int64_t m = i / nv, c = i % nv * V;
    Vec<T> g(gu + m * 2 * n + c);
    const Vec<T> u(gu + m * 2 * n + n + c);
#pragma unroll
    for (int e = 0; e < V; ++e) g.v[e] = silu_f32(g.v[e]) * u.v[e];
    g.store(act + m * n + c);
  }
}
template <typename T>
__global__ __launch_bounds__(256) void swiglu_pair_bwd_kernel(const T* __restrict__ dact, const T* __restrict__ gu,
                                                              int64_t M, int64_t n, T* __restrict__ dgu) {
  constexpr int V = Vec<T>::N;
  const int64_t nv = n / V, step = static_cast<int64_t>(gridDim.x) * 256;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < M * nv; i += step) {
    const int64_t m = i / nv, c = i % nv * V;
    const Vec<T> d(dact + m * n + c);
    Vec<T> g(gu + m * 2 * n + c), u(gu + m * 2 * n + n + c);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const float s = 1.0f / (1.0f + expf(-g.v[e]));
      const float du = d.v[e] * (g.v[e] * s);
      g.v[e] = d.v[e] * u.v[e] * (s * (1.0f + g.v[e] * (1.0f - s)));
      u.v[e] = du;
    }
    g.store(dgu + m * 2 * n + c);
    u.store(dgu + m * 2 * n + n + c);
  }
}

int route_wgs(int64_t M) {
  const int64_t t = (M + RT_TOK - 1) / RT_TOK;
  return static_cast<int>(t < RT_MAX_WG ? t : RT_MAX_WG);
}
unsigned copy_grid(int64_t vecs) {
  const int64_t g = (vecs + 255) / 256;
  return static_cast<unsigned>(g < 1 ? 1 : g < 8192 ? g : 8192);
}
bool al16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace

extern "C" {

FSI_API size_t fsi_mlp_train_route_workspace_size(int64_t M, int64_t n_blocks, int backward) {
  if (M <= 0 || n_blocks <= 0) return FSI_WORKSPACE_COUNTER_BYTES;
  return FSI_WORKSPACE_COUNTER_BYTES +
         sizeof(float) * static_cast<size_t>(route_wgs(M)) * static_cast<size_t>(n_blocks) * (backward ? RT_DIM : 1);
}

#define TRAIN_ROUTE_CHECKS(what)                                                                                   \
  FSI_CHECK_ARG(dtype == FSI_DTYPE_BF16 || dtype == FSI_DTYPE_F32, FSI_ERR_DTYPE, what ": dtype %d", dtype);       \
  FSI_CHECK_ARG(M > 0 && M <= 0x7fffffff && n_blocks > 0 && temperature > 0.f, FSI_ERR_SHAPE,                      \
                what ": M=%lld n_blocks=%lld", (long long)M, (long long)n_blocks);                                 \
  FSI_CHECK_ARG(n_blocks <= RT_MAX_NB, FSI_ERR_CAPACITY, what ": %lld blocks > %d", (long long)n_blocks, RT_MAX_NB)

FSI_API int fsi_mlp_train_route(const void* q, const void* keys, int64_t M, int64_t n_blocks, int64_t base_blocks,
                                int64_t remote_blocks, float temperature, int dtype, void* scores, void* ctx,
                                int32_t* active, void* workspace, size_t workspace_bytes, void* stream) {
  TRAIN_ROUTE_CHECKS("mlp_train_route");
  FSI_CHECK_ARG(base_blocks >= 0 && remote_blocks >= 0 && base_blocks + remote_blocks <= n_blocks, FSI_ERR_SHAPE,
                "mlp_train_route: %lld + %lld of %lld blocks", (long long)base_blocks, (long long)remote_blocks,
                (long long)n_blocks);
  FSI_CHECK_ARG(q && keys && scores && ctx && active, FSI_ERR_INVALID_ARG, "mlp_train_route: null pointer");
  FSI_CHECK_ARG(workspace && workspace_bytes >= fsi_mlp_train_route_workspace_size(M, n_blocks, 0), FSI_ERR_WORKSPACE,
                "mlp_train_route: workspace %zu", workspace_bytes);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  RouteArgs A{};
  A.q = q;
  A.keys = keys;
  A.M = (int)M;
  A.nb = (int)n_blocks;
  A.inv_t = 1.f / temperature;
  A.scores = scores;
  A.ctx = ctx;
  A.part = reinterpret_cast<float*>(static_cast<char*>(workspace) + FSI_WORKSPACE_COUNTER_BYTES);
  const int wg = route_wgs(M);
  const size_t lds = sizeof(float) * n_blocks * (RT_KS + RT_TOK);
  if (dtype == FSI_DTYPE_BF16) {
    train_route_kernel<bf16_t><<<wg, RT_THREADS, lds, st>>>(A);
    train_topk_kernel<bf16_t><<<1, RT_MAX_NB, 0, st>>>(A.part, wg, A.M, A.nb, (int)base_blocks, (int)remote_blocks, active);
  } else {
    train_route_kernel<float><<<wg, RT_THREADS, lds, st>>>(A);
    train_topk_kernel<float><<<1, RT_MAX_NB, 0, st>>>(A.part, wg, A.M, A.nb, (int)base_blocks, (int)remote_blocks, active);
  }
  FSI_HIP_LAUNCH_CHECK("mlp_train_route");
  return FSI_OK;
}

FSI_API int fsi_mlp_train_route_bwd(const void* q, const void* keys, const void* dscores, const void* dctx, int64_t M,
                                    int64_t n_blocks, float temperature, int dtype, void* dq, void* dkeys,
                                    void* workspace, size_t workspace_bytes, void* stream) {
  TRAIN_ROUTE_CHECKS("mlp_train_route_bwd");
  FSI_CHECK_ARG(q && keys && dq && dkeys, FSI_ERR_INVALID_ARG, "mlp_train_route_bwd: null pointer");
  FSI_CHECK_ARG(workspace && workspace_bytes >= fsi_mlp_train_route_workspace_size(M, n_blocks, 1), FSI_ERR_WORKSPACE,
                "mlp_train_route_bwd: workspace %zu", workspace_bytes);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  RouteArgs A{};
  A.q = q;
  A.keys = keys;
  A.M = (int)M;
  A.nb = (int)n_blocks;
  A.inv_t = 1.f / temperature;
  A.dscores = dscores;
  A.dctx = dctx;
  A.dq = dq;
  A.part = reinterpret_cast<float*>(static_cast<char*>(workspace) + FSI_WORKSPACE_COUNTER_BYTES);
  const int wg = route_wgs(M), n = A.nb * RT_DIM;
  const size_t lds = sizeof(float) * (n_blocks * (RT_KS + 2 * RT_TOK) + 2 * RT_TOK * RT_DIM);
  auto run = [&](auto tag, auto acc) {
    using T = decltype(tag);
    train_route_bwd_kernel<T, decltype(acc)::value><<<wg, RT_THREADS, lds, st>>>(A);
    train_dkeys_kernel<T><<<(n + 255) / 256, 256, 0, st>>>(A.part, wg, n, static_cast<T*>(dkeys));
  };
  auto sized = [&](auto tag) {  // (block, dim) pairs a thread accumulates
    if (n_blocks <= 128) run(tag, std::integral_constant<int, 8>{});
    else run(tag, std::integral_constant<int, 16>{});
  };
  if (dtype == FSI_DTYPE_BF16) sized(bf16_t{});
  else sized(float{});
  FSI_HIP_LAUNCH_CHECK("mlp_train_route_bwd");
  return FSI_OK;
}

#define TRAIN_ROWS_CHECKS(what)                                                                                     \
  const int64_t es = dtype == FSI_DTYPE_F32 ? 4 : 2, V = 16 / es;                                                  \
  FSI_CHECK_ARG(dtype == FSI_DTYPE_BF16 || dtype == FSI_DTYPE_F32, FSI_ERR_DTYPE, what ": dtype %d", dtype);        \
  FSI_CHECK_ARG(n_active > 0 && block > 0 && n_blocks > 0 && n_blocks <= 4096 && n_active <= 4096 && D > 0 &&       \
                    D <= 0x7fffffff && block <= 0x7fffffff,                                                        \
                FSI_ERR_SHAPE, what ": n_active=%lld block=%lld n_blocks=%lld D=%lld", (long long)n_active,         \
                (long long)block, (long long)n_blocks, (long long)D);                                              \
  FSI_CHECK_ARG(D % V == 0 && block % V == 0, FSI_ERR_ALIGN, what ": rows and blocks of whole 16-byte vectors")

FSI_API int fsi_mlp_train_gather(const void* k_gate, const void* k_up, int64_t ldk, const void* v, int64_t ldv,
                                 int v_transposed, const int32_t* active, int64_t n_active, int64_t block,
                                 int64_t n_blocks, int64_t D, int dtype, void* kgu, void* vs, void* stream) {
  TRAIN_ROWS_CHECKS("mlp_train_gather");
  FSI_CHECK_ARG(k_gate && k_up && v && active && kgu && vs, FSI_ERR_INVALID_ARG, "mlp_train_gather: null pointer");
  FSI_CHECK_ARG(ldk >= D && ldv >= (v_transposed ? n_blocks * block : D) && ldk % V == 0 && ldv % V == 0 &&
                    al16(k_gate) && al16(k_up) && al16(v) && al16(kgu) && al16(vs),
                FSI_ERR_ALIGN, "mlp_train_gather: 16-byte aligned rows");
  RowsArgs A{k_gate, k_up, v, ldk, ldv, kgu, vs, active, (int)n_active, (int)block, (int)n_blocks, (int)D, v_transposed != 0};
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const unsigned g = copy_grid(3 * n_active * block * (D / V));
  if (es == 2) train_gather_kernel<2><<<g, 256, 0, st>>>(A);
  else train_gather_kernel<4><<<g, 256, 0, st>>>(A);
  FSI_HIP_LAUNCH_CHECK("mlp_train_gather");
  return FSI_OK;
}

FSI_API int fsi_mlp_train_scatter(const void* dkgu, const void* dvs, int v_transposed, const int32_t* active,
                                  int64_t n_active, int64_t block, int64_t n_blocks, int64_t D, int dtype, void* dgate,
                                  void* dup, void* dv, void* stream) {
  TRAIN_ROWS_CHECKS("mlp_train_scatter");
  FSI_CHECK_ARG(active && (dkgu || (!dgate && !dup)) && (dvs || !dv), FSI_ERR_INVALID_ARG,
                "mlp_train_scatter: null pointer");
  FSI_CHECK_ARG(al16(dkgu) && al16(dvs) && al16(dgate) && al16(dup) && al16(dv), FSI_ERR_ALIGN,
                "mlp_train_scatter: 16-byte aligned rows");
  ScatterArgs A{dkgu, dvs, dgate, dup, dv, active, (int)n_active, (int)block, (int)n_blocks, (int)D, v_transposed != 0};
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 g(copy_grid((n_blocks * block * (D / V) + 3) / 4), 3);  // about four vectors a thread
  if (es == 2) train_scatter_kernel<2><<<g, 256, 0, st>>>(A);
  else train_scatter_kernel<4><<<g, 256, 0, st>>>(A);
  FSI_HIP_LAUNCH_CHECK("mlp_train_scatter");
  return FSI_OK;
}

FSI_API int fsi_swiglu_pair(const void* gu, int64_t M, int64_t n, int dtype, void* act, void* stream) {
  FSI_CHECK_ARG(dtype == FSI_DTYPE_BF16 || dtype == FSI_DTYPE_F32, FSI_ERR_DTYPE, "swiglu_pair: dtype %d", dtype);
  FSI_CHECK_ARG(M > 0 && n > 0 && n % (dtype == FSI_DTYPE_F32 ? 4 : 8) == 0, FSI_ERR_SHAPE, "swiglu_pair: M=%lld n=%lld",
                (long long)M, (long long)n);
  FSI_CHECK_ARG(gu && act && al16(gu) && al16(act), FSI_ERR_ALIGN, "swiglu_pair: null or misaligned pointer");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const unsigned g = copy_grid(M * n / (dtype == FSI_DTYPE_F32 ? 4 : 8));
  if (dtype == FSI_DTYPE_BF16)
    swiglu_pair_kernel<bf16_t><<<g, 256, 0, st>>>(static_cast<const bf16_t*>(gu), M, n, static_cast<bf16_t*>(act));
  else
    swiglu_pair_kernel<float><<<g, 256, 0, st>>>(static_cast<const float*>(gu), M, n, static_cast<float*>(act));
  FSI_HIP_LAUNCH_CHECK("swiglu_pair");
  return FSI_OK;
}

FSI_API int fsi_swiglu_pair_bwd(const void* dact, const void* gu, int64_t M, int64_t n, int dtype, void* dgu,
                                void* stream) {
  FSI_CHECK_ARG(dtype == FSI_DTYPE_BF16 || dtype == FSI_DTYPE_F32, FSI_ERR_DTYPE, "swiglu_pair_bwd: dtype %d", dtype);
  FSI_CHECK_ARG(M > 0 && n > 0 && n % (dtype == FSI_DTYPE_F32 ? 4 : 8) == 0, FSI_ERR_SHAPE,
                "swiglu_pair_bwd: M=%lld n=%lld", (long long)M, (long long)n);
  FSI_CHECK_ARG(dact && gu && dgu && al16(dact) && al16(gu) && al16(dgu), FSI_ERR_ALIGN,
                "swiglu_pair_bwd: null or misaligned pointer");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const unsigned g = copy_grid(M * n / (dtype == FSI_DTYPE_F32 ? 4 : 8));
  if (dtype == FSI_DTYPE_BF16)
    swiglu_pair_bwd_kernel<bf16_t><<<g, 256, 0, st>>>(static_cast<const bf16_t*>(dact), static_cast<const bf16_t*>(gu),
                                                      M, n, static_cast<bf16_t*>(dgu));
  else
    swiglu_pair_bwd_kernel<float><<<g, 256, 0, st>>>(static_cast<const float*>(dact), static_cast<const float*>(gu), M,
                                                     n, static_cast<float*>(dgu));
  FSI_HIP_LAUNCH_CHECK("swiglu_pair_bwd");
  return FSI_OK;
}

}  // extern "C"
