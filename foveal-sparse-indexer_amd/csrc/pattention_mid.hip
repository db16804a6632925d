// Pattention of 65 .. 255 bf16 tokens (short prompts, drafts to verify) on MI355X:
// out = (silu(x K_gate[S]^T) * (x K_up[S]^T)) V[S] over the active blocks S, from the
// parameters in place (V stored [D_out, N_p]).
//
// Too few tokens for 256 x 256 tiles, too many for one 64-token tile: with a workgroup per
// 16 weight rows and 64 tokens, every workgroup read its tokens' whole rows (x, then H),
// 590 MB through the L2s at 150 tokens of the 8B layer for 96 MB of weights.  Here a
// workgroup holds all the tokens against NT tiles of 16 weight rows and a range of the
// contraction, so the token rows it reads are K / splits long:
//   mid_gemm_kernel   fp32 partial sums (splits, M, N); N in tiles of 16, gate and up tiles
//                     in turn, or the output columns
//   mid_act_kernel    sums the splits, SwiGLU with the caller's rounding -> H (bf16)
//   mid_out_kernel    sums the splits -> out
// The partials cost 30 MB of traffic each way at that size, less than the rows they save.
// 150 tokens of the 8B layer (4096 hidden, 64 of 224 blocks): 92 -> 63 us, the two GEMMs
// 31 and 21 (2.1 - 2.4 TB/s of weights: the vector memory counter is in order, so waiting for a
// step's token rows, loaded two steps ahead, also waits for the weight stages issued before
// them, and two stages of the ring stay in flight).
#include "fsi_common.h"

using namespace fsi;

namespace {

constexpr int MD_WAVES = 8;
constexpr int MD_THREADS = 64 * MD_WAVES;
constexpr int MD_K = 64;          // contraction per step: 128 bytes of a row
constexpr int MD_MAX_STEPS = 64;  // steps of one split (their columns held one per lane)

typedef __attribute__((address_space(3))) void md_lds_t;
typedef __attribute__((address_space(1))) void md_glb_t;

struct MidArgs {
  const bf16_t* a;   // (M, lda): x or H
  int64_t lda;
  int M;
  const bf16_t* w0;  // k_gate or V^T
  const bf16_t* w1;  // k_up
  int64_t ldw;
  const int32_t* active;  // list channel block -> block; null: all
  int log2bn, n_blocks;
  int steps;         // per split
  int64_t n;         // 16 x tiles
  float* part;       // (splits, M, n)
  int* err;
};

// Parameter row of list channel c, or -1 (id out of range).
__device__ __forceinline__ int64_t mid_row(const MidArgs& A, int c) {
  if (!A.active) return c;
  const int b = A.active[c >> A.log2bn];
  if (b < 0 || b >= A.n_blocks) return -1;
  return (static_cast<int64_t>(b) << A.log2bn) + (c & ((1 << A.log2bn) - 1));
}

// At most N vector loads in flight, and every LDS read of this wave done (its stage may be
// overwritten after the barrier).
template <int N>
__device__ __forceinline__ void md_wait() {
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4));
}

// GATEUP: tile 2 c is gate channels 16 c .. + 16, tile 2 c + 1 the up ones; else tile c is
// output columns 16 c .. (rows of V^T) and the contraction runs over list channels.
// Wave w owns token tiles w, w + 8 (MT of them): their rows go straight to registers, two
// steps ahead; the weight tiles go straight to LDS (a ring of STAGES steps), rows of 128
// bytes with 16-byte piece p at p ^ (row & 7), and serve all eight waves.
template <bool GATEUP, int NT, int MT>
__global__ __launch_bounds__(MD_THREADS, 2) void mid_gemm_kernel(MidArgs A) {
  constexpr int STAGE = NT * 2048, STAGES = 8, UNITS = 2 * NT / MD_WAVES > 0 ? 2 * NT / MD_WAVES : 1;
  __shared__ __attribute__((aligned(1024))) char ring[STAGES * STAGE];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int t0 = blockIdx.x * NT;       // first weight tile
  const int s0 = blockIdx.y * A.steps;  // first step

  // ---- this lane's weight rows: unit u of a stage is 8 rows of tile u / 2 -----------
  const bf16_t* wrow[UNITS];
  bool loads = true;
#pragma unroll
  for (int i = 0; i < UNITS; ++i) {
    const int u = wave * UNITS + i;
    loads = u < 2 * NT;
    const int tile = t0 + (loads ? u >> 1 : 0), row = 8 * (u & 1) + (lane >> 3);
    const int piece = (lane & 7) ^ (row & 7);
    if (GATEUP) {
      const int c = 16 * (tile >> 1) + row;
      int64_t pr = mid_row(A, c);
      if (pr < 0) {  // its H is zeroed by mid_act_kernel; any row will do
        if (blockIdx.y == 0) set_error(A.err, FSI_ERR_INDEX_RANGE);
        pr = 0;
      }
      wrow[i] = (tile & 1 ? A.w1 : A.w0) + pr * A.ldw + 8 * piece;
    } else {
      wrow[i] = A.w0 + static_cast<int64_t>(16 * tile + row) * A.ldw + 8 * piece;
    }
  }
  // column of step i of this split (lane i), for the down projection's gathered contraction
  int col = 0;
  if (!GATEUP && lane < A.steps) {
    const int64_t c = mid_row(A, (s0 + lane) * MD_K);
    col = c < 0 ? 0 : static_cast<int>(c);  // H is zero there
  }
  auto issue = [&](int step) {
    if (!loads) return;
    const int k = GATEUP ? (s0 + step) * MD_K : __builtin_amdgcn_readlane(col, step);
    char* dst = ring + (step % STAGES) * STAGE + wave * UNITS * 1024;
#pragma unroll
    for (int i = 0; i < UNITS; ++i)
      __builtin_amdgcn_global_load_lds((md_glb_t*)(wrow[i] + k), (md_lds_t*)(dst + i * 1024), 16, 0, 0);
  };

  // ---- token rows -----------------------------------------------------------------
  const bf16_t* arow[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int t = 16 * (wave + MD_WAVES * m) + r;
    arow[m] = A.a + static_cast<int64_t>(t < A.M ? t : A.M - 1) * A.lda + static_cast<int64_t>(s0) * MD_K + 8 * q;
  }
  u32x4_t av[3][MT][2];
  auto load_a = [&](u32x4_t (&x)[MT][2], int step) {
    step = step < A.steps ? step : A.steps - 1;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int h = 0; h < 2; ++h) x[m][h] = *reinterpret_cast<const u32x4_t*>(arow[m] + step * MD_K + 32 * h);
  };

  f32x4_t acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[m][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  for (int p = 0; p < STAGES - 1 && p < A.steps; ++p) issue(p);
  load_a(av[0], 0);
  load_a(av[1], 1);
  // One step: refill the stage read in the previous one, then multiply.  Counting the direct
  // loads alone (the token rows in flight make the wait stricter), the stage of `step`
  // has landed once at most the STAGES - 2 later steps' are outstanding.
  auto run = [&](int step, u32x4_t (&x)[MT][2], u32x4_t (&next)[MT][2]) {
    if (step + STAGES - 2 < A.steps) md_wait<UNITS * (STAGES - 2)>();
    else md_wait<0>();
    asm volatile("s_barrier" ::: "memory");
    if (step + STAGES - 1 < A.steps) issue(step + STAGES - 1);
    load_a(next, step + 2);
    const char* S = ring + (step % STAGES) * STAGE;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const u32x4_t w = *reinterpret_cast<const u32x4_t*>(S + t * 2048 + r * 128 + 16 * ((4 * h + q) ^ (r & 7)));
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m][t] = mfma16x16x32(w, x[m][h], acc[m][t]);
      }
  };
  int step = 0;
  for (; step + 2 < A.steps; step += 3) {
    run(step, av[0], av[2]);
    run(step + 1, av[1], av[0]);
    run(step + 2, av[2], av[1]);
  }
  if (step < A.steps) run(step, av[0], av[2]);
  if (step + 1 < A.steps) run(step + 1, av[1], av[0]);

  // lane (r, q) of acc[m][t]: columns 4 q .. + 4 of tile t, token r of tile m
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int tok = 16 * (wave + MD_WAVES * m) + r;
    if (tok >= A.M) continue;
    float* out = A.part + (static_cast<int64_t>(blockIdx.y) * A.M + tok) * A.n + 16 * t0 + 4 * q;
#pragma unroll
    for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4_t*>(out + 16 * t) = acc[m][t];
  }
}

__device__ __forceinline__ f32x4_t sum_splits(const float* p, int splits, int64_t stride) {
  f32x4_t s = *reinterpret_cast<const f32x4_t*>(p);
  for (int i = 1; i < splits; ++i) s += *reinterpret_cast<const f32x4_t*>(p + i * stride);
  return s;
}

// H[m][c .. c + 4) from the gate and up sums; zero on channels of an out-of-range block.
__global__ __launch_bounds__(256) void mid_act_kernel(MidArgs A, int splits, int64_t n_ch, int rounding,
                                                      bf16_t* __restrict__ h) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x, per = n_ch / 4;
  if (i >= A.M * per) return;
  const int64_t m = i / per;
  const int c = static_cast<int>(i % per) * 4;
  const float* p = A.part + m * A.n + 32 * (c >> 4) + (c & 15);
  const f32x4_t g = sum_splits(p, splits, A.M * A.n), u = sum_splits(p + 16, splits, A.M * A.n);
  const bool ok = mid_row(A, c) >= 0;
  float y[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = ok ? pattention_act<ACT_SWIGLU>(g[e], u[e], rounding) : 0.f;
  *reinterpret_cast<uint2*>(h + m * n_ch + c) = make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
}

__global__ __launch_bounds__(256) void mid_out_kernel(const float* __restrict__ part, int splits, int64_t M, int64_t D,
                                                      bf16_t* __restrict__ out, int64_t ldo) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x, per = D / 4;
  if (i >= M * per) return;
  const int64_t m = i / per, d = i % per * 4;
  const f32x4_t s = sum_splits(part + m * D + d, splits, M * D);
#pragma unroll
  for (int e = 0; e < 4; ++e) out[m * ldo + d + e] = f32_to_bf16(s[e]);
}

// Weight tiles per workgroup and splits of `steps` contraction steps.  Eight tiles a workgroup
// read the token rows half as often as four, if four splits of them still give three
// quarters of the compute units a workgroup; more splits cost more in partial sums than the
// shorter rows save (8B layer, 150 tokens: gate and up 8 tiles x 4 splits 72.6 us a pass, 4 x
// 4 76.1, 4 x 2 78.0, 8 x 8 88.2; down 4 x 4 61.0, 8 x 4 64.5, 4 x 2 72.3).
struct MidPlan {
  int nt, splits;
};
bool mid_plan(int64_t tiles, int64_t steps, MidPlan& p) {
  for (int nt : {8, 4}) {
    if (tiles % nt) continue;
    p = MidPlan{nt, 0};
    for (int s = 1; s <= 4 && tiles / nt * p.splits < 192; s *= 2)
      if (steps % s == 0 && steps / s >= 4 && steps / s <= MD_MAX_STEPS) p.splits = s;
    if (tiles / nt * p.splits >= (nt == 8 ? 192 : 64)) return true;
  }
  return false;
}

// Elements of one weight matrix's active rows from which these kernels are the faster ones at
// every token count: below, the caches hold the weights that every 64-token workgroup of the
// other kernels reads again, and the partials weigh more.  At 8.4 M five of six points are
// 3 to 13 % faster here, but one is 3 % slower and the line keeps it from losing.  us a pass, there -> here, for 65 / 150 / 255 tokens: 4096 x 4096 (16.8 M) 59 / 92 /
// 111 -> 44 / 63 / 77; 4096 x 2048 and 2048 x 4096 (8.4 M) 36 / 54 / 61 -> 33 / 47 / 59 and
// 38 / 53 / 60 -> 36 / 50 / 62; 2048 x 1536 (3.1 M) 22 / 30 / 32 -> 23 / 35 / 45.
constexpr int64_t MD_MIN_WEIGHT = 12 << 20;

struct MidWs {
  size_t h, part, end;
};
MidWs mid_ws(int64_t M, int64_t n_ch, int64_t D, const MidPlan& a, const MidPlan& b) {
  MidWs o{};
  o.h = FSI_WORKSPACE_COUNTER_BYTES;
  o.part = o.h + fsi_host::align_up(static_cast<size_t>(M * n_ch) * 2, 256);
  const int64_t pa = a.splits * M * 2 * n_ch, pb = b.splits * M * D;
  o.end = o.part + static_cast<size_t>(pa > pb ? pa : pb) * 4;
  return o;
}
bool mid_plans(int64_t M, int64_t K, int64_t n_ch, int64_t D, MidPlan& a, MidPlan& b) {
  return M > 64 && M < 256 && K * n_ch >= MD_MIN_WEIGHT && K % MD_K == 0 && n_ch % MD_K == 0 && D % 16 == 0 && n_ch <= (1 << 24) &&
         mid_plan(2 * n_ch / 16, K / MD_K, a) && mid_plan(D / 16, n_ch / MD_K, b);
}

template <bool GATEUP>
void mid_launch(const MidArgs& A, const MidPlan& p, int64_t tiles, hipStream_t st) {
  const dim3 g(static_cast<unsigned>(tiles / p.nt), static_cast<unsigned>(p.splits));
  const bool one = A.M <= 16 * MD_WAVES;
  if (p.nt == 8) {
    if (one) mid_gemm_kernel<GATEUP, 8, 1><<<g, MD_THREADS, 0, st>>>(A);
    else mid_gemm_kernel<GATEUP, 8, 2><<<g, MD_THREADS, 0, st>>>(A);
  } else {
    if (one) mid_gemm_kernel<GATEUP, 4, 1><<<g, MD_THREADS, 0, st>>>(A);
    else mid_gemm_kernel<GATEUP, 4, 2><<<g, MD_THREADS, 0, st>>>(A);
  }
}

}  // namespace

namespace fsi_mid {

// 0 where the shape has no plan here.
size_t workspace_bytes(int64_t M, int64_t K, int64_t D_out, int64_t n_channels) {
  MidPlan a, b;
  return mid_plans(M, K, n_channels, D_out, a, b) ? mid_ws(M, n_channels, D_out, a, b).end : 0;
}

// 0: done, 1: not a shape for these kernels, -1: launch failed.  block_n a power of two >= 64
// dividing N_p, 16-byte aligned rows.
int run(const bf16_t* x, int64_t ldx, const bf16_t* kg, const bf16_t* ku, int64_t ldk, const bf16_t* vt, int64_t ldv,
        const int32_t* active, int64_t n_blocks, int log2bn, int64_t M, int64_t K, int64_t n_ch, int64_t D, int rounding,
        bf16_t* out, int64_t ldo, void* workspace, size_t ws_bytes, int* err, hipStream_t st) {
  MidPlan a, b;
  if (!mid_plans(M, K, n_ch, D, a, b)) return 1;
  const MidWs o = mid_ws(M, n_ch, D, a, b);
  if (ws_bytes < o.end) return 1;
  char* ws = static_cast<char*>(workspace);
  bf16_t* h = reinterpret_cast<bf16_t*>(ws + o.h);
  MidArgs A{};
  A.a = x;
  A.lda = ldx;
  A.M = (int)M;
  A.w0 = kg;
  A.w1 = ku;
  A.ldw = ldk;
  A.active = active;
  A.log2bn = log2bn;
  A.n_blocks = (int)n_blocks;
  A.steps = (int)(K / MD_K) / a.splits;
  A.n = 2 * n_ch;
  A.part = reinterpret_cast<float*>(ws + o.part);
  A.err = err;
  mid_launch<true>(A, a, 2 * n_ch / 16, st);
  mid_act_kernel<<<static_cast<unsigned>((M * n_ch / 4 + 255) / 256), 256, 0, st>>>(A, a.splits, n_ch, rounding, h);
  A.a = h;
  A.lda = n_ch;
  A.w0 = vt;
  A.w1 = nullptr;
  A.ldw = ldv;
  A.steps = (int)(n_ch / MD_K) / b.splits;
  A.n = D;
  mid_launch<false>(A, b, D / 16, st);
  mid_out_kernel<<<static_cast<unsigned>((M * D / 4 + 255) / 256), 256, 0, st>>>(A.part, b.splits, M, D, out, ldo);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace fsi_mid
