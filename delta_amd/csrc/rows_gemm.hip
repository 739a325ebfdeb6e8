// Decode-batch GEMM for gfx950 at 33-128 token rows: out[m, n] = sum_k x[m, k] W[n, k] (+ bias[n]).
//
// At these batches a projection still reads its weight once per step (2 M <= 256 flops per 2 bytes),
// so the weight stream from HBM is its floor, but x is no longer small: every block reads all M rows
// of x for its k range, at 128 rows as many bytes as W for a block of 128 columns.  What bounds the
// kernel is the CU's vector memory path: it keeps about 32 KiB of requests in flight and returns them
// in order, so a CU draws 40-47 GB/s while x and W requests alternate (x alone, from L2: 110 GB/s; W
// alone at 216 blocks: 6.3 TB/s in all).  Hence:
//   * all loads go straight to LDS (global_load_lds, no registers held), x in slabs of SK k steps at
//     once and W in a ring of WS steps, so x's L2 hits come in runs instead of queueing one by one
//     behind W's misses;
//   * block tiles as wide as the grid allows (128 or 192 W rows) and K split over the grid (S splits,
//     fp32 partials summed by the consumer) until nearly every CU has a block;
//   * a block's 8 waves split every k step in two halves (kg), so each wave reads 64 rows x 64 bytes
//     of both operands: 64 KiB of LDS reads a step at 128 x 128, against 96 KiB for 8 waves of 64 x 32.
// Measured against hipBLASLt (x @ W.T, graph replays over rotating weights, us; S > 1 without the
// consumer's sum): 128 rows, Qwen2.5-14B w2 34.9 vs 73.9, wo 18.9 vs 32.1, w1|w3 with SiLU-mul 65-73
// vs 73 and a 5 us SiLU-mul launch; Llama-3-8B w2 30.4 vs 75.2; 64 rows, DeepSeek-R1-Distill-Qwen-1.5B
// w2 9.8 vs 25.4, wo 4.9 vs 7.5, w1|w3 18.2 vs 18.7 + 5.  W in registers with producer waves for x
// (one consumer wave per SIMD) was slower (w2 40.4), and so was staging x step by step beside W
// (w1|w3 69-71).
#include "delta_common.h"

namespace delta {
namespace {

struct RowsArgs {
  const uint16_t *x;
  int64_t ldx;
  const uint16_t *w;
  int64_t ldw;
  const uint16_t *bias;
  uint16_t *out;  // one split
  int64_t ldo;
  float *part;    // several splits: [S][M][N]
  int M, N, K;
  int inter;      // GLU: W = [gate rows; up rows], out [M][inter]
};

// A block: kg (2) x WM x WN waves; wave (kg, wm, wn) computes TM x TN tiles of 16 tokens x 16 W rows over
// the k half kg of every 64-wide k step.
template <int DT, int WM, int TM, int WN, int TN, int SK, int WS, bool GLU>
__global__ void __launch_bounds__(128 * WM * WN) gemm_rows_kernel(RowsArgs a) {
  using E = Elem<DT>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  static_assert(!GLU || TN % 2 == 0, "a GLU wave owns gate tiles and the matching up tiles");
  constexpr int NW = 2 * WM * WN;
  constexpr int kRows = 16 * TM * WM;      // token rows per block
  constexpr int kCols = 16 * TN * WN;      // W rows per block
  constexpr int kOutCols = GLU ? kCols / 2 : kCols;
  constexpr int kXStep = kRows * 128, kWStage = kCols * 128;  // LDS bytes
  constexpr int kXSlab = SK * kXStep;
  static_assert(kRows % (8 * NW) == 0 || (8 * NW) % kRows == 0, "x loads");
  constexpr int LX = SK * kRows / 8 / NW;  // 1 KiB loads per wave: x slab, W stage
  constexpr int LW = kCols / 8 / NW;
  static_assert(SK * kRows % (8 * NW) == 0 && kCols % (8 * NW) == 0, "loads per wave");
  static_assert(WS >= 3 && WS - 2 < SK, "one x slab among the loads behind a W stage");
  constexpr int XG = kRows / 8 >= NW ? kRows / 8 / NW : 1;  // row groups a wave loads per k step

  const int wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int kg = wave & 1, wm = (wave >> 1) % WM, wn = (wave >> 1) / WM;
  const int c = lane >> 4, t = lane & 15;
  const int steps = a.K / 64;
  const int sp = blockIdx.y, ns = gridDim.y;
  const int s_beg = (int)((int64_t)steps * sp / ns), s_end = (int)((int64_t)steps * (sp + 1) / ns);
  const int total = s_end - s_beg;
  const int n0 = blockIdx.x * kOutCols;

  // A load covers 8 tile rows x 128 bytes, whole cache lines: lane l takes row l / 8, 16-byte chunk
  // (l % 8) ^ ((row / 2) % 8), which makes the 16-row fragment reads conflict-free.
  uint32_t xoff[XG], woff[LW];
#pragma unroll
  for (int j = 0; j < XG; ++j) {
    const int tr = 8 * ((wave + NW * j) % (kRows / 8)) + (lane >> 3);
    xoff[j] = (uint32_t)(((int64_t)(tr < a.M ? tr : a.M - 1) * a.ldx + 8 * ((lane & 7) ^ ((tr >> 1) & 7))) * 2);
  }
#pragma unroll
  for (int j = 0; j < LW; ++j) {
    const int wr = 8 * (wave + NW * j) + (lane >> 3);
    int64_t r;
    if (GLU) {
      constexpr int half = 8 * TN;  // a wave column's gate rows, then its up rows
      const int col = n0 + wr / (2 * half) * half + wr % half;
      r = (col < a.inter ? col : a.inter - 1) - n0 + (wr % (2 * half) >= half ? (int64_t)a.inter : 0);
    } else {
      r = (n0 + wr < a.N ? n0 + wr : a.N - 1) - n0;
    }
    woff[j] = (uint32_t)((r * a.ldw + 8 * ((lane & 7) ^ ((wr >> 1) & 7))) * 2);
  }
  const char *xb = reinterpret_cast<const char *>(a.x + (int64_t)s_beg * 64);
  const char *wb = reinterpret_cast<const char *>(a.w + (int64_t)n0 * a.ldw + (int64_t)s_beg * 64);
  const uint32_t lds_x = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
  const uint32_t lds_w = lds_x + 2 * kXSlab;
  auto issue_x = [&](int slab) {
    const uint32_t dst = lds_x + (uint32_t)(slab & 1) * kXSlab;
#pragma unroll
    for (int j = 0; j < LX; ++j) {
      const int q = wave + NW * j;
      int s = slab * SK + q / (kRows / 8);
      s = s < total ? s : total - 1;  // past the end: the last step again, never read
      load_lds_1k(dst + q * 1024, xb + (int64_t)s * 128, xoff[j % XG]);
    }
  };
  auto issue_w = [&](int s) {
    const uint32_t dst = lds_w + (uint32_t)(s % WS) * kWStage;
#pragma unroll
    for (int j = 0; j < LW; ++j) load_lds_1k<true>(dst + (wave + NW * j) * 1024, wb + (int64_t)s * 128, woff[j]);
  };

  f32x4 acc[TN][TM];
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int fo = t * 128 + 16 * ((4 * kg + c) ^ ((t >> 1) & 7));  // the lane's bytes in a 16-row tile
  auto compute = [&](int s, int slab, int p) {
    const char *xs = smem + (slab & 1) * kXSlab + p * kXStep + TM * wm * 2048 + fo;
    const char *ws = smem + 2 * kXSlab + (s % WS) * kWStage + TN * wn * 2048 + fo;
    u32x4 xf[TM], wf[TN];
#pragma unroll
    for (int m = 0; m < TM; ++m) xf[m] = *reinterpret_cast<const u32x4 *>(xs + m * 2048);
#pragma unroll
    for (int n = 0; n < TN; ++n) wf[n] = *reinterpret_cast<const u32x4 *>(ws + n * 2048);
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int m = 0; m < TM; ++m) acc[n][m] = E::mfma(wf[n], xf[m], acc[n][m]);
  };

  // Issue order: x(0), W(0 .. WS-2); then at step s (after its barrier): x(slab + 1) if s starts a
  // slab, then W(s + WS - 1).  W(s) has landed when at most the loads issued after it are pending:
  // WS - 2 stages, and one x slab when one was issued at steps s - WS + 2 .. s - 1.
  if (total > 0) {
    issue_x(0);
#pragma unroll
    for (int s = 0; s < WS - 1; ++s)
      if (s < total) issue_w(s);
  }
  int slab = 0;
  for (int s0 = 0; s0 < total; s0 += SK, ++slab) {
    const bool more_x = s0 + SK < total;
#pragma unroll
    for (int p = 0; p < SK; ++p) {
      const int s = s0 + p;
      if (s < total) {
        const int left = total - 1 - s;  // W stages after s
        if (left >= WS - 2) {
          if (p >= 1 && p <= WS - 2 && more_x)
            wait_loads<(WS - 2) * LW + LX>();
          else
            wait_loads<(WS - 2) * LW>();
        } else {
          wait_loads<0>();
        }
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (p == 0 && more_x) issue_x(slab + 1);
        if (s + WS - 1 < total) issue_w(s + WS - 1);
        compute(s, slab, p);
      }
    }
  }

  // The k halves meet in LDS: waves kg = 1 park their tiles, waves kg = 0 add them.
  f32x4 *red = reinterpret_cast<f32x4 *>(smem) + (wave >> 1) * (TM * TN * 64) + lane;
  __syncthreads();
  if (kg == 1) {
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int m = 0; m < TM; ++m) red[(n * TM + m) * 64] = acc[n][m];
  }
  __syncthreads();
  if (kg == 1) return;
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[n][m] += red[(n * TM + m) * 64];

  // Lane (c, t) holds W rows 4c + r (4 consecutive columns) of token t of each tile.
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int row = 16 * (TM * wm + m) + t;
    if (row >= a.M) continue;
#pragma unroll
    for (int n = 0; n < (GLU ? TN / 2 : TN); ++n) {
      const int col = n0 + 16 * ((GLU ? TN / 2 : TN) * wn + n) + 4 * c;
      if (col >= (GLU ? a.inter : a.N)) continue;
      f32x4 v = acc[n][m];
      if (GLU) {
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float gr = E::lo(E::from_float(v[i])), ur = E::lo(E::from_float(acc[n + TN / 2][m][i]));
          const float h = E::lo(E::from_float(gr / (1.f + expf(-gr))));
          o[i] = E::from_float(h * ur);
        }
        *reinterpret_cast<uint2 *>(a.out + (int64_t)row * a.ldo + col) = uint2{o[0] | (o[1] << 16), o[2] | (o[3] << 16)};
      } else {
        if (a.bias && sp == 0) {
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] += E::lo(a.bias[col + i]);
        }
        if (ns == 1)
          *reinterpret_cast<uint2 *>(a.out + (int64_t)row * a.ldo + col) =
              uint2{E::from_float(v[0]) | (E::from_float(v[1]) << 16), E::from_float(v[2]) | (E::from_float(v[3]) << 16)};
        else
          *reinterpret_cast<f32x4 *>(a.part + ((int64_t)sp * a.M + row) * a.N + col) = v;
      }
    }
  }
}

template <int DT, int WM, int TM, int WN, int TN, int SK, int WS, bool GLU>
void launch_rows(const RowsArgs &a, int splits, hipStream_t stream) {
  constexpr size_t loop = 2ull * SK * 16 * TM * WM * 128 + (size_t)WS * 16 * TN * WN * 128;
  constexpr size_t red = (size_t)WM * WN * TM * TN * 1024;
  constexpr size_t bytes = loop > red ? loop : red;
  static_assert(bytes <= 160 * 1024, "LDS");
  constexpr int cols = 16 * TN * WN / (GLU ? 2 : 1);
  const dim3 grid((unsigned)ceil_div(GLU ? a.inter : a.N, cols), splits);
  hipLaunchKernelGGL((gemm_rows_kernel<DT, WM, TM, WN, TN, SK, WS, GLU>), grid, dim3(128 * WM * WN), bytes, stream, a);
}

// Tile and K splits.  Up to 64 rows: 64-column blocks (two fit a CU) when some power-of-two split
// count <= 16 brings them to 192-256 blocks, else 128-column ones; past 64 rows: 128 or 192 columns,
// whichever splits to more blocks <= 256 (14B w2 at 128 rows: 160 blocks of 128 columns 45.1 us, 216 of
// 192 columns 34.9).  A split keeps at least 3 k steps.
struct RowsPlan {
  int cols, splits;
};
int rows_splits(int64_t n, int cols, int steps) {
  const int64_t cb = ceil_div(n, cols);
  int s = 1;
  while (s < 16 && cb * s * 2 <= 256 && steps >= 6 * s) s *= 2;
  return s;
}
RowsPlan rows_plan(int M, int N, int K) {
  const int steps = K / 64;
  const int a = M <= 64 ? 64 : 128, b = M <= 64 ? 128 : 192;
  const int sa = rows_splits(N, a, steps), sb = rows_splits(N, b, steps);
  const int64_t na = ceil_div(N, a) * sa, nb = ceil_div(N, b) * sb;
  if (M <= 64) return na >= 192 && na <= 256 ? RowsPlan{a, sa} : RowsPlan{b, sb};
  return nb > na && nb <= 256 ? RowsPlan{b, sb} : RowsPlan{a, sa};
}

template <int DT>
void launch_plain(const RowsArgs &a, const RowsPlan &p, hipStream_t st) {
  if (a.M <= 64) {
    if (p.cols == 64) launch_rows<DT, 2, 2, 2, 2, 3, 4, false>(a, p.splits, st);
    else launch_rows<DT, 1, 4, 4, 2, 6, 4, false>(a, p.splits, st);
  } else {
    if (p.cols == 192) launch_rows<DT, 2, 4, 2, 6, 2, 3, false>(a, p.splits, st);
    else launch_rows<DT, 1, 8, 4, 2, 3, 4, false>(a, p.splits, st);
  }
}

// Gate/up: 64 inter columns (128 W rows) a block; up to 64 rows, 32 columns (two blocks a CU) when
// there are more than 256 blocks of 64 (Qwen2.5-7B, 64 rows: 60.7 vs 70.6 us).
template <int DT>
void launch_glu(const RowsArgs &a, hipStream_t st) {
  if (a.M > 64) launch_rows<DT, 1, 8, 4, 2, 3, 4, true>(a, 1, st);
  else if (ceil_div(a.inter, 64) > 256) launch_rows<DT, 2, 2, 2, 2, 3, 4, true>(a, 1, st);
  else launch_rows<DT, 1, 4, 4, 2, 6, 4, true>(a, 1, st);
}

// The checks both entry points share; `rows` is the number of W rows.
int check_rows(const char *who, const void *x, int64_t ldx, const void *w, int64_t ldw, int M, int64_t rows, int K,
               int dtype) {
  if (!x || !w) return set_error(DELTA_ERR_INVALID, "%s: null pointer", who);
  if (M > 128) return set_error(DELTA_ERR_INVALID, "%s: M (%d) must be <= 128", who, M);
  if (dtype != DELTA_BF16 && dtype != DELTA_FP16) return set_error(DELTA_ERR_INVALID, "%s: dtype must be bf16 or fp16", who);
  if (K <= 0 || K % 64) return set_error(DELTA_ERR_INVALID, "%s: K (%d) must be a positive multiple of 64", who, K);
  if (ldx < K || ldw < K) return set_error(DELTA_ERR_INVALID, "%s: leading dimensions too small", who);
  if ((ldx % 8) || (ldw % 8) || (((uintptr_t)x | (uintptr_t)w) & 15u))
    return set_error(DELTA_ERR_INVALID, "%s: x and W rows must be 16-byte aligned", who);
  // 32-bit byte offsets from x and from a block's first W row
  if (ldx > ((int64_t)1 << 23) || rows > ((int64_t)1 << 31) / ldw)
    return set_error(DELTA_ERR_INVALID, "%s: leading dimensions too large", who);
  return DELTA_OK;
}

}  // namespace
}  // namespace delta

extern "C" DELTA_EXPORT int delta_gemm_rows128_splits(int M, int N, int K) {
  if (M <= 0 || M > 128 || N <= 0 || N % 16 || K <= 0 || K % 64) return 0;
  return delta::rows_plan(M, N, K).splits;
}

extern "C" DELTA_EXPORT int delta_gemm_rows128(const void *x, int64_t ldx, const void *w, int64_t ldw,
                                               const void *bias, void *out, int64_t ldo, float *partials, int M,
                                               int N, int K, int dtype, delta_stream_t stream) {
  using namespace delta;
  clear_error();
  const char *who = "delta_gemm_rows128";
  if (M <= 0 || N <= 0) return DELTA_OK;
  int rc = check_rows(who, x, ldx, w, ldw, M, 192, K, dtype);
  if (rc) return rc;
  if (N % 16) return set_error(DELTA_ERR_INVALID, "%s: N (%d) must be a multiple of 16", who, N);
  const RowsPlan p = rows_plan(M, N, K);
  if (p.splits == 1) {
    if (!out || ldo < N || (ldo % 4) || ((uintptr_t)out & 7u))
      return set_error(DELTA_ERR_INVALID, "%s: out must be [M, >= N] with 8-byte aligned rows", who);
  } else if (!partials || ((uintptr_t)partials & 15u)) {
    return set_error(DELTA_ERR_INVALID, "%s: this shape needs fp32 partials [%d][M][N] (16-byte aligned)", who, p.splits);
  }
  RowsArgs a;
  a.x = (const uint16_t *)x;
  a.ldx = ldx;
  a.w = (const uint16_t *)w;
  a.ldw = ldw;
  a.bias = (const uint16_t *)bias;
  a.out = (uint16_t *)out;
  a.ldo = ldo;
  a.part = partials;
  a.M = M;
  a.N = N;
  a.K = K;
  a.inter = 0;
  if (dtype == DELTA_BF16) launch_plain<DELTA_BF16>(a, p, (hipStream_t)stream);
  else launch_plain<DELTA_FP16>(a, p, (hipStream_t)stream);
  return check_launch(who);
}

extern "C" DELTA_EXPORT int delta_gemm_rows128_silu(const void *x, int64_t ldx, const void *w13, int64_t ldw, void *out,
                                                    int64_t ldo, int M, int inter, int K, int dtype,
                                                    delta_stream_t stream) {
  using namespace delta;
  clear_error();
  const char *who = "delta_gemm_rows128_silu";
  if (M <= 0 || inter <= 0) return DELTA_OK;
  if (inter % 16) return set_error(DELTA_ERR_INVALID, "%s: inter (%d) must be a multiple of 16", who, inter);
  int rc = check_rows(who, x, ldx, w13, ldw, M, (int64_t)inter + 64, K, dtype);
  if (rc) return rc;
  if (!out || ldo < inter || (ldo % 4) || ((uintptr_t)out & 7u))
    return set_error(DELTA_ERR_INVALID, "%s: out must be [M, >= inter] with 8-byte aligned rows", who);
  RowsArgs a;
  a.x = (const uint16_t *)x;
  a.ldx = ldx;
  a.w = (const uint16_t *)w13;
  a.ldw = ldw;
  a.bias = nullptr;
  a.out = (uint16_t *)out;
  a.ldo = ldo;
  a.part = nullptr;
  a.M = M;
  a.N = 2 * inter;
  a.K = K;
  a.inter = inter;
  if (dtype == DELTA_BF16) launch_glu<DELTA_BF16>(a, (hipStream_t)stream);
  else launch_glu<DELTA_FP16>(a, (hipStream_t)stream);
  return check_launch(who);
}
