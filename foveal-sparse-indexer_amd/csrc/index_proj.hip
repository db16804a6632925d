// The products around the 16-D index on MI355X (foveal_indexer/core.py:214-250, 288-312):
// the projections of hidden states to 16 dimensions, their weights' gradients, and the
// additive stream's projection back with its repetition over each block's elements.
//
// All of them are one pass over the hidden states (or over their gradient) with 16 or 32
// columns on the other side, so memory bounds them; a library GEMM of that shape costs as
// much host time as the pass takes, and each projection read the states for itself.  One
// distillation step over 16384 hidden states of 2048 in fp32 (128 MiB): keys and values
// 47 -> 33 us, their weights' gradients 133 -> 49 (3.0 TB/s of x), the stream 55 -> 25 (5.4
// TB/s written) and its backward 53 -> 51 us, the whole step's kernels 500 -> 250 us and its
// issue from the host 0.67 -> 0.33 .. 0.48 ms.
#include <type_traits>

#include "fsi_common.h"

using namespace fsi;

namespace {

constexpr int IP_D = 16;
constexpr int IP_CT = 128;      // columns per wave of the weight gradients
constexpr int IP_SPLITS = 32;   // row ranges of the weight gradients, at most

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
__device__ __forceinline__ f32x4_t mfma_f32(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

struct ProjArgs {
  const void* x;          // row m = (b, t) at x + b xs_b + t xs_t, D contiguous elements
  int64_t xs_b, xs_t;
  int64_t M;
  int tokens, D;          // rows per batch entry (FLAT kernels: row m at x + m xs_t)
  const void* w[2];       // (16, D) each
  void* y[2];             // (M, 16) each
  const void* g[2];       // (M, 16): gradients of y
  float* part;            // (splits, NW, 16, D)
  int rows;               // rows per split
};
template <bool FLAT>
__device__ __forceinline__ int64_t proj_row(const ProjArgs& A, int64_t m) {
  m = m < A.M ? m : A.M - 1;
  if (FLAT) return m * A.xs_t;
  const int64_t b = m / A.tokens;
  return b * A.xs_b + (m - b * A.tokens) * A.xs_t;
}

// y = x W^T for NW weights.  A workgroup takes 16 TT rows; its waves share the columns in
// chunks of 128 bytes of a row (A = W, B = x^T, both straight from memory in the MFMA's k
// order) and add up in LDS.  TT = 4 lets a fragment of W serve four tiles where rows are
// many; TT = 1 with eight waves keeps a few rows' chain short.
template <typename T, int NW, int TT, int WAVES, bool FLAT>
__global__ __launch_bounds__(64 * WAVES) void proj_kernel(ProjArgs A) {
  constexpr int V = 16 / static_cast<int>(sizeof(T));  // elements per lane and piece
  constexpr int CH = 128 / static_cast<int>(sizeof(T));
  __shared__ f32x4_t red[WAVES][NW * TT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, kg = lane >> 4;
  const int64_t m0 = static_cast<int64_t>(blockIdx.x) * 16 * TT;
  const T* xr[TT];
#pragma unroll
  for (int t = 0; t < TT; ++t) xr[t] = static_cast<const T*>(A.x) + proj_row<FLAT>(A, m0 + 16 * t + r) + V * kg;
  const T* wr[NW];
#pragma unroll
  for (int w = 0; w < NW; ++w) wr[w] = static_cast<const T*>(A.w[w]) + static_cast<int64_t>(r) * A.D + V * kg;
  f32x4_t acc[NW][TT];
#pragma unroll
  for (int w = 0; w < NW; ++w)
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[w][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
  for (int c = wave; c < A.D / CH; c += WAVES) {
    u32x4_t xv[2][TT], wv[2][NW];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int d = c * CH + h * 4 * V;
#pragma unroll
      for (int t = 0; t < TT; ++t) xv[h][t] = *reinterpret_cast<const u32x4_t*>(xr[t] + d);
#pragma unroll
      for (int w = 0; w < NW; ++w) wv[h][w] = *reinterpret_cast<const u32x4_t*>(wr[w] + d);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int t = 0; t < TT; ++t) {
          if constexpr (sizeof(T) == 2) {
            acc[w][t] = mfma16x16x32(wv[h][w], xv[h][t], acc[w][t]);
          } else {
#pragma unroll
            for (int k = 0; k < 4; ++k)
              acc[w][t] = mfma_f32(__uint_as_float(wv[h][w][k]), __uint_as_float(xv[h][t][k]), acc[w][t]);
          }
        }
  }
#pragma unroll
  for (int w = 0; w < NW; ++w)
#pragma unroll
    for (int t = 0; t < TT; ++t) red[wave][w * TT + t][lane] = acc[w][t];
  __syncthreads();
  for (int i = wave; i < NW * TT; i += WAVES) {
    f32x4_t s = red[0][i][lane];
#pragma unroll
    for (int v = 1; v < WAVES; ++v) s += red[v][i][lane];
    const int64_t m = m0 + 16 * (i % TT) + r;  // components 4 kg + e of row m
    if (m < A.M)
#pragma unroll
      for (int e = 0; e < 4; ++e) stf<T>(static_cast<T*>(A.y[i / TT]), m * IP_D + 4 * kg + e, s[e]);
  }
}

// Partial dW[c][d] = sum_m g[m][c] x[m][d] over one range of rows and 128 columns, on the
// fp32 matrix unit for either type (bf16 rows would need a transpose to contract over; the
// 2 M D 32 operations fit under the pass over x).  Wave w takes every fourth group of 4 rows:
// A = g^T, B = x with column tile n = columns V r + j of a 16-byte piece.
template <typename T, int NW, bool FLAT>
__global__ __launch_bounds__(256) void proj_dw_kernel(ProjArgs A) {
  constexpr int V = 16 / static_cast<int>(sizeof(T)), P = IP_CT / (16 * V), NT = IP_CT / 16;  // pieces, column tiles
  __shared__ f32x4_t red[3][NW * NT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, kg = lane >> 4;
  const int d0 = blockIdx.x * IP_CT;
  const int64_t ma = static_cast<int64_t>(blockIdx.y) * A.rows;
  const int64_t mb = ma + A.rows < A.M ? ma + A.rows : A.M;
  f32x4_t acc[NW][NT];
#pragma unroll
  for (int w = 0; w < NW; ++w)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[w][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int64_t m = ma + 4 * wave; m < mb; m += 16) {
    const int64_t row = m + kg;
    const bool live = row < mb;
    const T* xp = static_cast<const T*>(A.x) + proj_row<FLAT>(A, row) + d0 + V * r;
    u32x4_t xv[P];
#pragma unroll
    for (int p = 0; p < P; ++p) xv[p] = *reinterpret_cast<const u32x4_t*>(xp + 16 * V * p);
    float g[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float v = ldf<T>(static_cast<const T*>(A.g[w]), (live ? row : mb - 1) * IP_D + r);
      g[w] = live ? v : 0.f;
    }
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int j = 0; j < V; ++j) {
        float x;
        if constexpr (sizeof(T) == 2) x = j & 1 ? hi_bf16(xv[p][j / 2]) : lo_bf16(xv[p][j / 2]);
        else x = __uint_as_float(xv[p][j]);
        x = live ? x : 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) acc[w][p * V + j] = mfma_f32(g[w], x, acc[w][p * V + j]);
      }
  }
  if (wave)
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
      for (int n = 0; n < NT; ++n) red[wave - 1][w * NT + n][lane] = acc[w][n];
  __syncthreads();
  if (wave) return;
#pragma unroll
  for (int w = 0; w < NW; ++w)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int v = 0; v < 3; ++v) acc[w][n] += red[v][w * NT + n][lane];
  // lane (r, kg), tile n = p V + j, element e: component 4 kg + e, column d0 + 16 V p + V r + j
#pragma unroll
  for (int w = 0; w < NW; ++w)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float* out = A.part + ((static_cast<int64_t>(blockIdx.y) * NW + w) * IP_D + 4 * kg + e) * A.D + d0 + V * r;
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int q = 0; q < V / 4; ++q)
          *reinterpret_cast<f32x4_t*>(out + 16 * V * p + 4 * q) =
              f32x4_t{acc[w][p * V + 4 * q][e], acc[w][p * V + 4 * q + 1][e], acc[w][p * V + 4 * q + 2][e],
                      acc[w][p * V + 4 * q + 3][e]};
    }
}

// dw[w] = sum over the splits, in order.  n = 16 D elements per weight.
template <typename T>
__global__ __launch_bounds__(256) void split_sum_kernel(const float* __restrict__ part, int splits, int nw, int64_t n,
                                                        T* __restrict__ a, T* __restrict__ b) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i >= nw * n) return;
  f32x4_t s = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int k = 0; k < splits; ++k) s += *reinterpret_cast<const f32x4_t*>(part + k * nw * n + i);
  T* out = i < n ? a + i : b + (i - n);
#pragma unroll
  for (int e = 0; e < 4; ++e) stf<T>(out, e, s[e]);
}

// w[d .. d + V) (16 components each, 16-byte aligned) against c: one dot product per column.
template <typename T, int V>
__device__ __forceinline__ void dot_rows(const T* w, const float (&c)[IP_D], float (&y)[V]) {
  constexpr int E = 16 / static_cast<int>(sizeof(T));
#pragma unroll
  for (int j = 0; j < V; ++j) {
    y[j] = 0.f;
#pragma unroll
    for (int h = 0; h < IP_D / E; ++h) {
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(w + j * IP_D + h * E);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (sizeof(T) == 2) {
          y[j] = fmaf(c[h * E + 2 * i], lo_bf16(v[i]), y[j]);
          y[j] = fmaf(c[h * E + 2 * i + 1], hi_bf16(v[i]), y[j]);
        } else {
          y[j] = fmaf(c[h * E + i], __uint_as_float(v[i]), y[j]);
        }
      }
    }
  }
}
// c += s[j] w[d + j] over the V columns.
template <typename T, int V>
__device__ __forceinline__ void add_rows(const T* w, const float (&s)[V], float (&c)[IP_D]) {
  constexpr int E = 16 / static_cast<int>(sizeof(T));
#pragma unroll
  for (int j = 0; j < V; ++j)
#pragma unroll
    for (int h = 0; h < IP_D / E; ++h) {
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(w + j * IP_D + h * E);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (sizeof(T) == 2) {
          c[h * E + 2 * i] = fmaf(s[j], lo_bf16(v[i]), c[h * E + 2 * i]);
          c[h * E + 2 * i + 1] = fmaf(s[j], hi_bf16(v[i]), c[h * E + 2 * i + 1]);
        } else {
          c[h * E + i] = fmaf(s[j], __uint_as_float(v[i]), c[h * E + i]);
        }
      }
    }
}

// out[p bs + t][d] = ctx[p] . w[d] for every element t of block p: each product is formed
// once and written bs times.  Thread = one 16-byte piece of the row.
template <typename T>
__global__ __launch_bounds__(256) void expand_kernel(const T* __restrict__ ctx, const T* __restrict__ w, int bs, int D,
                                                     T* __restrict__ out) {
  constexpr int V = 16 / static_cast<int>(sizeof(T));
  const int64_t p = blockIdx.x;
  const int d = (blockIdx.y * 256 + threadIdx.x) * V;
  if (d >= D) return;
  float c[IP_D];
#pragma unroll
  for (int k = 0; k < IP_D; ++k) c[k] = ldf<T>(ctx, p * IP_D + k);
  u32x4_t val;
  float y[V];
  dot_rows<T, V>(w + static_cast<int64_t>(d) * IP_D, c, y);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (sizeof(T) == 2) val[i] = pack_bf16x2(y[2 * i], y[2 * i + 1]);
    else val[i] = __float_as_uint(y[i]);
  }
  T* o = out + p * bs * D + d;
  for (int t = 0; t < bs; ++t) *reinterpret_cast<u32x4_t*>(o + static_cast<int64_t>(t) * D) = val;
}

// Backward: sums[p][d] = sum_t dy[p bs + t][d] (fp32) and dctx[p] = sums[p] . w.  One
// workgroup per block, a thread a 16-byte piece of the row.
template <typename T>
__global__ __launch_bounds__(512) void expand_sum_kernel(const T* __restrict__ dy, const T* __restrict__ w, int bs,
                                                         int D, float* __restrict__ sums, T* __restrict__ dctx) {
  constexpr int V = 16 / static_cast<int>(sizeof(T));
  __shared__ float red[8][IP_D];
  const int64_t p = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float c[IP_D] = {};
  for (int d = threadIdx.x * V; d < D; d += 512 * V) {
    float s[V] = {};
    const T* src = dy + p * bs * D + d;
#pragma unroll 8
    for (int t = 0; t < bs; ++t) {
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(src + static_cast<int64_t>(t) * D);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (sizeof(T) == 2) {
          s[2 * i] += lo_bf16(v[i]);
          s[2 * i + 1] += hi_bf16(v[i]);
        } else {
          s[i] += __uint_as_float(v[i]);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < V; j += 4)
      *reinterpret_cast<f32x4_t*>(sums + p * D + d + j) = f32x4_t{s[j], s[j + 1], s[j + 2], s[j + 3]};
    add_rows<T, V>(w + static_cast<int64_t>(d) * IP_D, s, c);
  }
#pragma unroll
  for (int k = 0; k < IP_D; ++k) {
    const float v = wave_sum(c[k]);
    if (lane == 0) red[wave][k] = v;
  }
  __syncthreads();
  if (threadIdx.x < IP_D) {
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) v += red[i][threadIdx.x];
    stf<T>(dctx, p * IP_D + threadIdx.x, v);
  }
}

// dw[d][k] = sum_p sums[p][d] ctx[p][k]: 32 columns a workgroup, eight threads a column.
constexpr int ED_COLS = 32, ED_PH = 8;
template <typename T>
__global__ __launch_bounds__(ED_COLS * ED_PH) void expand_dw_kernel(const float* __restrict__ sums,
                                                                   const T* __restrict__ ctx, int64_t n_pool, int D,
                                                                   T* __restrict__ dw) {
  __shared__ float red[ED_PH - 1][ED_COLS][IP_D + 1];
  const int col = threadIdx.x % ED_COLS, ph = threadIdx.x / ED_COLS;
  const int d = blockIdx.x * ED_COLS + col;
  float acc[IP_D] = {};
  if (d < D) {
#pragma unroll 4
    for (int64_t p = ph; p < n_pool; p += ED_PH) {
      const float s[1] = {sums[p * D + d]};
      add_rows<T, 1>(ctx + p * IP_D, s, acc);
    }
  }
  if (ph)
#pragma unroll
    for (int k = 0; k < IP_D; ++k) red[ph - 1][col][k] = acc[k];
  __syncthreads();
  if (ph || d >= D) return;
#pragma unroll
  for (int k = 0; k < IP_D; ++k) {
#pragma unroll
    for (int i = 0; i < ED_PH - 1; ++i) acc[k] += red[i][col][k];
    stf<T>(dw, static_cast<int64_t>(d) * IP_D + k, acc[k]);
  }
}

int dw_splits(int64_t M) {
  const int64_t s = (M + 63) / 64;
  return static_cast<int>(s < IP_SPLITS ? s : IP_SPLITS);
}
bool al16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// The element type and whether rows are evenly spaced over the batch (no division per row).
template <typename F>
void by_rows(int dtype, int64_t B, int64_t T, int64_t xs_b, int64_t xs_t, F run) {
  const bool flat = B == 1 || xs_b == T * xs_t;
  if (dtype == FSI_DTYPE_BF16) flat ? run(bf16_t{}, std::true_type{}) : run(bf16_t{}, std::false_type{});
  else flat ? run(float{}, std::true_type{}) : run(float{}, std::false_type{});
}

int proj_checks(const char* what, const void* x, int64_t xs_b, int64_t xs_t, int64_t B, int64_t T, int64_t D,
                int dtype) {
  FSI_CHECK_ARG(dtype == FSI_DTYPE_BF16 || dtype == FSI_DTYPE_F32, FSI_ERR_DTYPE, "%s: dtype %d", what, dtype);
  const int64_t V = dtype == FSI_DTYPE_F32 ? 4 : 8;
  FSI_CHECK_ARG(B > 0 && T > 0 && D > 0 && D % IP_CT == 0 && D <= (1 << 24) && T <= 0x7fffffff &&
                    B * T <= (int64_t(1) << 35),
                FSI_ERR_SHAPE, "%s: B=%lld T=%lld D=%lld", what, (long long)B, (long long)T, (long long)D);
  FSI_CHECK_ARG(x && al16(x) && xs_b % V == 0 && xs_t % V == 0, FSI_ERR_ALIGN, "%s: 16-byte aligned rows", what);
  return FSI_OK;
}

}  // namespace

extern "C" {

FSI_API int fsi_index_proj(const void* x, int64_t xs_b, int64_t xs_t, int64_t B, int64_t T, int64_t D, const void* w0,
                           const void* w1, int dtype, void* y0, void* y1, void* stream) {
  const int rc = proj_checks("index_proj", x, xs_b, xs_t, B, T, D, dtype);
  if (rc != FSI_OK) return rc;
  FSI_CHECK_ARG(w0 && y0 && !w1 == !y1 && al16(w0) && al16(w1), FSI_ERR_INVALID_ARG, "index_proj: null pointer");
  ProjArgs A{};
  A.x = x;
  A.xs_b = xs_b;
  A.xs_t = xs_t;
  A.M = B * T;
  A.tokens = (int)T;
  A.D = (int)D;
  A.w[0] = w0;
  A.w[1] = w1;
  A.y[0] = y0;
  A.y[1] = y1;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  auto run = [&](auto tag, auto flat) {
    using E = decltype(tag);
    constexpr bool F = decltype(flat)::value;
    // 16 rows a workgroup as long as all of them run at once (two of eight waves on each of 256
    // compute units), 64 rows beyond.  us with 64 | 16, keys and values of 2048 columns in
    // fp32: 4096 rows 27.3 | 13.5, 8192 27.5 | 23.9, 12288 27.8 | 34.4, 16384 28.1 | 45.2; bf16 14.1 |
    // 12.4, 14.3 | 13.6, 14.6 | 19.0, 14.8 | 24.2.
    if (A.M > 8192) {
      const unsigned g = static_cast<unsigned>((A.M + 63) / 64);
      if (w1) proj_kernel<E, 2, 4, 4, F><<<g, 256, 0, st>>>(A);
      else proj_kernel<E, 1, 4, 4, F><<<g, 256, 0, st>>>(A);
    } else {
      const unsigned g = static_cast<unsigned>((A.M + 15) / 16);
      if (w1) proj_kernel<E, 2, 1, 8, F><<<g, 512, 0, st>>>(A);
      else proj_kernel<E, 1, 1, 8, F><<<g, 512, 0, st>>>(A);
    }
  };
  by_rows(dtype, B, T, xs_b, xs_t, run);
  FSI_HIP_LAUNCH_CHECK("index_proj");
  return FSI_OK;
}

FSI_API size_t fsi_index_proj_dw_workspace_size(int64_t M, int64_t D, int n_weights) {
  if (M <= 0 || D <= 0 || n_weights <= 0) return FSI_WORKSPACE_COUNTER_BYTES;
  return FSI_WORKSPACE_COUNTER_BYTES + sizeof(float) * static_cast<size_t>(dw_splits(M)) * n_weights * IP_D * D;
}

FSI_API int fsi_index_proj_dw(const void* x, int64_t xs_b, int64_t xs_t, int64_t B, int64_t T, int64_t D,
                              const void* g0, const void* g1, int dtype, void* dw0, void* dw1, void* workspace,
                              size_t workspace_bytes, void* stream) {
  const int rc = proj_checks("index_proj_dw", x, xs_b, xs_t, B, T, D, dtype);
  if (rc != FSI_OK) return rc;
  FSI_CHECK_ARG(g0 && dw0 && !g1 == !dw1, FSI_ERR_INVALID_ARG, "index_proj_dw: null pointer");
  const int nw = g1 ? 2 : 1;
  FSI_CHECK_ARG(workspace && al16(workspace) && workspace_bytes >= fsi_index_proj_dw_workspace_size(B * T, D, nw),
                FSI_ERR_WORKSPACE, "index_proj_dw: workspace %zu", workspace_bytes);
  ProjArgs A{};
  A.x = x;
  A.xs_b = xs_b;
  A.xs_t = xs_t;
  A.M = B * T;
  A.tokens = (int)T;
  A.D = (int)D;
  A.g[0] = g0;
  A.g[1] = g1;
  A.part = reinterpret_cast<float*>(static_cast<char*>(workspace) + FSI_WORKSPACE_COUNTER_BYTES);
  const int splits = dw_splits(A.M);
  const int64_t rows = (A.M + splits - 1) / splits;
  FSI_CHECK_ARG(rows <= 0x7fffffff, FSI_ERR_SHAPE, "index_proj_dw: too many rows");
  A.rows = (int)rows;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid(static_cast<unsigned>(D / IP_CT), static_cast<unsigned>(splits));
  const int64_t n = IP_D * D;
  const unsigned rg = static_cast<unsigned>((nw * n / 4 + 255) / 256);
  auto run = [&](auto tag, auto flat) {
    using E = decltype(tag);
    constexpr bool F = decltype(flat)::value;
    if (nw == 2) proj_dw_kernel<E, 2, F><<<grid, 256, 0, st>>>(A);
    else proj_dw_kernel<E, 1, F><<<grid, 256, 0, st>>>(A);
    split_sum_kernel<E><<<rg, 256, 0, st>>>(A.part, splits, nw, n, static_cast<E*>(dw0), static_cast<E*>(dw1));
  };
  by_rows(dtype, B, T, xs_b, xs_t, run);
  FSI_HIP_LAUNCH_CHECK("index_proj_dw");
  return FSI_OK;
}

#define EXPAND_CHECKS(what)                                                                                        \
  FSI_CHECK_ARG(dtype == FSI_DTYPE_BF16 || dtype == FSI_DTYPE_F32, FSI_ERR_DTYPE, what ": dtype %d", dtype);       \
  FSI_CHECK_ARG(n_pool > 0 && n_pool <= 0x7fffffff && block > 0 && block <= 0x7fffffff && D > 0 && D % 8 == 0 &&   \
                    D <= (1 << 24),                                                                                \
                FSI_ERR_SHAPE, what ": n_pool=%lld block=%lld D=%lld", (long long)n_pool, (long long)block,         \
                (long long)D)

FSI_API int fsi_index_expand(const void* ctx, const void* w, int64_t n_pool, int64_t block, int64_t D, int dtype,
                             void* out, void* stream) {
  EXPAND_CHECKS("index_expand");
  FSI_CHECK_ARG(ctx && w && out && al16(out) && al16(w), FSI_ERR_INVALID_ARG, "index_expand: null or misaligned pointer");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int64_t per = 256 * (dtype == FSI_DTYPE_F32 ? 4 : 8);
  const dim3 grid(static_cast<unsigned>(n_pool), static_cast<unsigned>((D + per - 1) / per));
  if (dtype == FSI_DTYPE_BF16)
    expand_kernel<bf16_t><<<grid, 256, 0, st>>>(static_cast<const bf16_t*>(ctx), static_cast<const bf16_t*>(w),
                                                (int)block, (int)D, static_cast<bf16_t*>(out));
  else
    expand_kernel<float><<<grid, 256, 0, st>>>(static_cast<const float*>(ctx), static_cast<const float*>(w), (int)block,
                                               (int)D, static_cast<float*>(out));
  FSI_HIP_LAUNCH_CHECK("index_expand");
  return FSI_OK;
}

FSI_API size_t fsi_index_expand_bwd_workspace_size(int64_t n_pool, int64_t D) {
  if (n_pool <= 0 || D <= 0) return FSI_WORKSPACE_COUNTER_BYTES;
  return FSI_WORKSPACE_COUNTER_BYTES + sizeof(float) * static_cast<size_t>(n_pool) * D;
}

FSI_API int fsi_index_expand_bwd(const void* dy, const void* ctx, const void* w, int64_t n_pool, int64_t block,
                                 int64_t D, int dtype, void* dctx, void* dw, void* workspace, size_t workspace_bytes,
                                 void* stream) {
  EXPAND_CHECKS("index_expand_bwd");
  FSI_CHECK_ARG(dy && ctx && w && dctx && dw && al16(dy) && al16(ctx) && al16(w), FSI_ERR_INVALID_ARG,
                "index_expand_bwd: null or misaligned pointer");
  FSI_CHECK_ARG(workspace && workspace_bytes >= fsi_index_expand_bwd_workspace_size(n_pool, D), FSI_ERR_WORKSPACE,
                "index_expand_bwd: workspace %zu", workspace_bytes);
  float* sums = reinterpret_cast<float*>(static_cast<char*>(workspace) + FSI_WORKSPACE_COUNTER_BYTES);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const unsigned n = static_cast<unsigned>(n_pool), gd = static_cast<unsigned>((D + ED_COLS - 1) / ED_COLS);
  auto run = [&](auto tag) {
    using E = decltype(tag);
    expand_sum_kernel<E><<<n, 512, 0, st>>>(static_cast<const E*>(dy), static_cast<const E*>(w), (int)block, (int)D,
                                            sums, static_cast<E*>(dctx));
    expand_dw_kernel<E><<<gd, 256, 0, st>>>(sums, static_cast<const E*>(ctx), n_pool, (int)D, static_cast<E*>(dw));
  };
  if (dtype == FSI_DTYPE_BF16) run(bf16_t{});
  else run(float{});
  FSI_HIP_LAUNCH_CHECK("index_expand_bwd");
  return FSI_OK;
}

}  // extern "C"
