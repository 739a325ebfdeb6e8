// Causal paged prefill attention for gfx950 (several query tokens per row, GQA).
//
// Replaces FlashInfer's BatchPrefillWithPagedKVCacheWrapper.run with causal=True for rows
// with qo_len > 1 (hoenza/DELTA backend.py:1091-1105, the prompt steps of the engine).  The
// cache already holds the row's new tokens (update_kv runs before attention, model.py:413-418),
// so query i of row b sits at position kv_len_b - qo_len_b + i and attends tokens 0..position.
//
// Work decomposition (flash-attention style, on 32x32 MFMA tiles): a block is PW waves of one
// (row, kv head) and a run of consecutive query tokens; each wave owns 32 query rows, the
// (token, q head) pairs of TW = 32 / G tokens (rows past TW * G idle when G does not divide
// 32), with its q in registers.  The block sweeps the row's kv tokens 64 at a time (four pages,
// two 32-token sub-tiles) up to its last token's position: each step's K and V (16 KiB each for
// one head) go from global memory straight to LDS (global_load_lds: no registers, no LDS store
// instructions) and are read by every wave.
//   PW = 8 (long prompts, see wide_blocks): one block per CU, four step buffers.  Waves 0-3 run each
//     step whole; waves 4-7, the second wave of each SIMD, run half a step behind (P.V of the
//     previous step, then S and softmax of this one), so the two waves of a SIMD are not both in
//     their softmax at once.  Steps are loaded two ahead.
//   PW = 4: two blocks per CU, two step buffers each, the next step's loads issued under this step's
//     MFMAs.  Half the tile: less idle time at the ends of short prompts, and one block's start runs
//     under the other's steps.
// What bounds it: MFMA and VALU issue of two waves per SIMD that overlap in part (without the MFMAs an
// 8192-token prompt takes 390-410 us of 500-520, without the exponentials 475, without the loads 500),
// under a clock that MFMA-heavy kernels pull down (a 16384^3 bf16 product reaches 1.57 PFLOP/s on this
// card; this kernel 1.06).  Llama-3-8B shape, graph-free launches, us (registers-staged 8-wave kernel
// before / PW 8 / PW 4): 8192 tokens 545 / 500 / 534, 2048 tokens 66 / 59 / 55, 300 tokens - / 15.5 /
// 13.1, 8 prompts of 128-1024 - / 54 / 52.6, 32 prompts of 64-256 - / 42 / 35.  Of that, the fences
// that keep fragment reads ahead of their MFMAs took 595 -> 571 (8192 tokens, with RoPE + append), the
// scalar work of the loads (one check for invalid pages per block instead of one per step) 2048 tokens
// 63 -> 58.  Prefetching a step's first K and V fragments in the step before: no gain (522 vs 516).
// Per wave and sub-tile:
//   S^T = K Q^T : 8 v_mfma_f32_32x32x16 over d, A = the tile's K rows from LDS
//         (lane%32 = kv token, d in 16 ks + 8 (lane / 32) + [0, 8)), B = the wave's q (same d
//         split, n = lane%32 = query row); D leaves lane l with its row n = l%32 and the 16 kv
//         tokens m_i = 8 (i / 4) + 4 (l / 32) + i % 4;
//   softmax: online per row in the log2 domain over the step's 32 scores of the lane, one
//         exchange with lane l ^ 32 (the row's other half) for the maximum; the row sum stays
//         per half until the end.  The reference maximum moves only when a score passes it by
//         more than 8 (log2), so the accumulators are rescaled on few steps; causal and kv_len
//         masks only on steps that need them;
//   O^T += V^T P^T : 8 v_mfma_f32_32x32x16 (4 d tiles x 2 kv chunks), B = the lane's own P in
//         its D order (chunk c = values 8c..8c+7, i.e. kv tokens 16c + 4 (l/32) + {0..3, 8..11}),
//         packed by v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32, A = V^T read from the padded tile
//         with ds_read_b64_tr_b16 in that same kv order; lane l accumulates
//         O[row l%32][d = 32 dt + 8 (i / 4) + 4 (l / 32) + i % 4].
// LDS tiles: 64 rows of 256 bytes, 16-byte chunks swizzled by row so that the fragment reads cover
// the banks once (see the step loads).  Page ids come by scalar loads, a step ahead.
// Blocks run heaviest first (the last query tiles attend the most tokens; see BlockOrder), the kv head
// fastest, so with 8 kv heads the blocks of one head land on the same XCD (blocks go to the XCDs round
// robin) and share its L2 for that head's K/V.  No merge.
#include "delta_common.h"

namespace delta {

int run_decode_rows(const void *q, int64_t q_stride_t, int64_t q_stride_h, const void *kv_cache, int64_t num_pages,
                    const int32_t *qo_indptr, const int32_t *kv_indptr, const int32_t *kv_indices,
                    int64_t kv_indices_len, const int32_t *kv_last_page_len, void *o, int64_t o_stride_t,
                    int64_t o_stride_h, float *lse, int batch, int hq, int hkv, int dtype, float sm_scale,
                    int64_t pages, int64_t max_pages, void *workspace, hipStream_t stream, const char *who);
size_t decode_rows_workspace_bytes(int batch, int hq, int64_t kv_indices_len);

namespace {

constexpr int kSub = 2;         // 32-token sub-tiles per step
constexpr int kKvStep = 32 * kSub;  // kv tokens per step
constexpr int kPgStep = kKvStep / 16;  // pages per step
constexpr int kTileB = kKvStep * 256;  // bytes of a step's K (or V) tile: 64 rows of 256 bytes

// Order of a kv head's blocks (find_tile).  A slot of the grid without a tile costs a launched block that
// holds LDS for a microsecond, and many of them among the others hold those back (prompts of 4096 and
// 1500 tokens, the shorter one's missing tiles launched between the longer one's: 232 us, packed 165;
// prompts of 300 beside 100 decoding rows, a row's slots together: 103, packed 77), so the blocks that
// exist come first:
//   kByTile, few rows: the last tiles of all rows first (they attend the most tokens), down to the rows'
//     first ones.  A row at a time leaves the last rows' heavy tiles to the end of the launch (us by tile / by
//     row: 8 prompts of 37-1500, 2 kv heads 42.6 / 55.7, 8 kv heads 99.6 / 102; 4 of 2048, 2 kv heads
//     71.7 / 88.4; 12 of 1000, 2 kv heads 63.7 / 68.1).
//   kByRow, more rows: a row's last tile first, then the next row.  What runs together shares few rows' K
//     and V in the L2 (16 prompts of 512, 8 kv heads 79.6 / 71.5; 32 of 64-256 40.8 / 36.4; 64 of 128
//     66.0 / 52.3).
//   kBySlot, one row or a CU for every slot: nothing to order, no search in front (100 prompts of 30, 2 kv
//     heads 11.8 / 12.2 by row).  With a second block on some CUs the order matters for rows of many tiles (4
//     prompts of 331 at 1331 tokens, 4 kv heads, 336 slots: 44.9 / 40.0 by tile), not for few (20 of 60, 320
//     slots: 11.1 / 11.9 by row).
enum BlockOrder { kBySlot = 0, kByRow = 1, kByTile = 2 };
constexpr int kByTileRows = 12;

struct PrefillArgs {
  const uint16_t *q;
  int64_t q_stride_t, q_stride_h;
  const uint16_t *kv;
  int64_t num_pages;
  const int32_t *qo_indptr;
  const int32_t *kv_indptr;
  const int32_t *kv_indices;
  int64_t kv_indices_len;
  const int32_t *last_page_len;
  uint16_t *o;
  int64_t o_stride_t, o_stride_h;
  float *lse;
  int batch, hq, hkv;
  int64_t num_tokens;     // query tokens of all rows, -1: not known
  int decode_rows;        // rows of one query token, their pages (for the choice of the blocks only)
  int64_t decode_pages;
  int skip_single;  // rows of one query token are run_decode_rows'
  int row_tiles;    // the most tiles a row has (of max_qo_len tokens)
  int order;        // of the blocks: kBySlot, kByRow, kByTile
  float sm_scale;
};

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short ps4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) ps4_t lds_ps4_t;

template <int DT>
struct Mfma32;
template <>
struct Mfma32<DELTA_BF16> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  __device__ __forceinline__ static f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
};
template <>
struct Mfma32<DELTA_FP16> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  __device__ __forceinline__ static f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
};

// Two floats -> two packed 16-bit values, round to nearest even (one v_cvt_pk_* on gfx950).
template <int DT>
__device__ __forceinline__ uint32_t pack2(float x, float y);
template <>
__device__ __forceinline__ uint32_t pack2<DELTA_BF16>(float x, float y) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{x, y}), b2));
}
template <>
__device__ __forceinline__ uint32_t pack2<DELTA_FP16>(float x, float y) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{x, y}), h2));
}

// max / sum of a value and its copy in lane l ^ 32
__device__ __forceinline__ float halves_max(float v) {
  auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1]));
}
__device__ __forceinline__ float halves_sum(float v) {
  auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(x[0]) + __uint_as_float(x[1]);
}

// A row's CSR bounds and last page length.
struct RowBounds {
  int q0, q1, kv0, kv1, last;
};
__device__ __forceinline__ RowBounds row_bounds(const PrefillArgs &a, int r) {
  if (r >= a.batch) return RowBounds{0, 0, 0, 0, 0};
  return RowBounds{a.qo_indptr[r], a.qo_indptr[r + 1], a.kv_indptr[r], a.kv_indptr[r + 1], a.last_page_len[r]};
}
__device__ __forceinline__ RowBounds bounds_of_lane(const RowBounds &x, int l) {
  return RowBounds{__builtin_amdgcn_readlane(x.q0, l), __builtin_amdgcn_readlane(x.q1, l),
                   __builtin_amdgcn_readlane(x.kv0, l), __builtin_amdgcn_readlane(x.kv1, l),
                   __builtin_amdgcn_readlane(x.last, l)};
}

// Row, with its bounds, and tile (BT query tokens) of block u of a kv head; false past the last one.  Only the
// device knows the rows' lengths, so the grid has batch * row_tiles slots.  Every lane loads a row's bounds, so
// that the row found costs no second round trip.
template <int BT>
__device__ __forceinline__ bool find_tile(const PrefillArgs &a, int u, int lane, RowBounds *row, int *tile) {
  auto tiles_of = [&](const RowBounds &x) {
    const int qn = x.q1 - x.q0;
    if (qn <= 0 || (a.skip_single && qn == 1)) return 0;
    const int n = (qn + BT - 1) / BT;
    return n < a.row_tiles ? n : a.row_tiles;
  };
  if (a.order == kBySlot) {
    const int r = u / a.row_tiles;
    *row = row_bounds(a, r);
    *tile = a.row_tiles - 1 - (u - r * a.row_tiles);
    return *tile < tiles_of(*row);
  }
  if (a.order == kByTile) {  // batch <= 64, row_tiles <= 32 * 64
    // Lane l counts the blocks from tile t_l on, sum over the rows of max(0, n_r - t_l), for 64 t at
    // once (more tiles: coarse, then fine).
    const RowBounds mine = row_bounds(a, lane);
    const int n = tiles_of(mine);
    auto blocks_from = [&](int t) {
      int s = 0;
      for (int r = 0; r < a.batch; ++r) {
        const int d = __builtin_amdgcn_readlane(n, r) - t;
        s += d > 0 ? d : 0;
      }
      return s;
    };
    const int step = (a.row_tiles + 63) / 64;
    int t0 = 0;
    if (step > 1) {
      const uint64_t m = __ballot(blocks_from(lane * step) > u);
      if (m == 0) return false;
      t0 = (__popcll(m) - 1) * step;
    }
    const int s = blocks_from(t0 + lane);
    const uint64_t m = __ballot(s > u);
    if (m == 0) return false;
    const int k = __popcll(m) - 1;  // 63 only if row_tiles = 64, whose tile 64 has no blocks
    const int above = k < 63 ? __builtin_amdgcn_readlane(s, k < 63 ? k + 1 : 63) : 0;
    const int t = t0 + k;
    // The rows rotate by tile: blocks go to the XCDs round robin, and with fewer than 8 kv heads a fixed
    // order would give an XCD all tiles of the same rows.
    const uint64_t has = __ballot(n > t);
    const int i = (u - above + t) % __popcll(has);
    const uint64_t it = __ballot(n > t && __popcll(has & ((1ull << lane) - 1)) == i);
    *row = bounds_of_lane(mine, __builtin_ctzll(it));
    *tile = t;
    return true;
  }
  int base = 0;
  for (int r0 = 0; r0 < a.batch; r0 += 64) {
    const RowBounds mine = row_bounds(a, r0 + lane);
    const int n = tiles_of(mine);
    int incl = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(incl, off, 64);
      if (lane >= off) incl += v;
    }
    const uint64_t m = __ballot(base + incl > u);
    if (m != 0) {
      const int l = __builtin_ctzll(m);
      *row = bounds_of_lane(mine, l);
      *tile = base + __builtin_amdgcn_readlane(incl, l) - 1 - u;
      return true;
    }
    base += __builtin_amdgcn_readlane(incl, 63);
  }
  return false;
}

template <int DT, int G, int PW>
__global__ void __launch_bounds__(PW * 64, 2) paged_prefill_kernel(PrefillArgs a) {
#pragma clang fp contract(off)
  using MF = Mfma32<DT>;
  constexpr int TW = 32 / G;                  // query tokens per wave
  constexpr int BT = PW * TW;                 // query tokens per block
  constexpr bool kLate = PW == 8;             // the second wave of each SIMD runs half a step behind
  // LDS step buffers: this step and the next, in flight; kLate also the late waves' step and one more
  // in flight.
  constexpr int kBufs = kLate ? 4 : 2;
  constexpr int kPgWave = 16 / PW;            // pages a wave loads rows of, per step
  // Step buffers, each the K tile, then the V tile (swizzled rows), shared by the block's waves.
  __shared__ __attribute__((aligned(1024))) char tiles[kBufs][2 * kTileB];

  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int hl = lane >> 5, n = lane & 31;
  const int h = blockIdx.x;
  RowBounds row;
  int tile;
  if (!find_tile<BT>(a, (int)(blockIdx.z * gridDim.y + blockIdx.y), lane, &row, &tile)) return;  // whole block
  const int64_t q0 = row.q0;
  const int qn = row.q1 - row.q0;
  const int btok0 = tile * BT;
  // The wave's first query token, read as a scalar: the compiler cannot see that wave (from the
  // thread index) is uniform, and with tok0 scalar the wave's step count and its diagonal test
  // (full / masked step) become scalar branches (8192-token prompt 594 -> 569-585 us in the kernel that
  // staged K and V through registers).
  const int tok0 = __builtin_amdgcn_readfirstlane(btok0 + wave * TW);

  // Row's pages and length (indptr entries clamped as in the decode kernels).
  const int64_t ilen = a.kv_indices_len;
  int64_t p0 = row.kv0, p1 = row.kv1;
  p0 = p0 < 0 ? 0 : (p0 > ilen ? ilen : p0);
  p1 = p1 < p0 ? p0 : (p1 > ilen ? ilen : p1);
  const int np = (int)(p1 - p0);
  int lp = row.last;
  lp = lp < 0 ? 0 : (lp > kPageSize ? kPageSize : lp);
  const int kv_len = np > 0 ? (np - 1) * kPageSize + lp : 0;

  // This lane's query row n = (token tt, head g).
  const int tt = n / G, g = n % G;
  const bool row_ok = n < TW * G && tok0 + tt < qn;
  const int qpos = kv_len - qn + tok0 + tt;  // attends tokens 0..qpos
  u32x4 qf[8];  // B operand of S^T = K Q^T: d = 16 ks + 8 hl + [0, 8)
  if (row_ok) {
    // With a negative scale q's signs are flipped (S of -q is exactly -S; the scale below is then
    // positive).  The xor also makes the loads complete here, before the kv loop.
    const uint32_t flip = a.sm_scale < 0.f ? 0x80008000u : 0u;
    const uint16_t *qp = a.q + (q0 + tok0 + tt) * a.q_stride_t + (int64_t)(h * G + g) * a.q_stride_h + 8 * hl;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = ld128(qp + 16 * ks) ^ u32x4{flip, flip, flip, flip};
  } else {
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = u32x4{0u, 0u, 0u, 0u};
  }

  // Steps the block sweeps (up to its last token's position) and the ones this wave needs.
  auto steps_upto = [&](int last_tok) {
    const int pos = kv_len - qn + last_tok;
    const int nt = pos >= 0 ? pos / kKvStep + 1 : 0;
    const int cap = (kv_len + kKvStep - 1) / kKvStep;
    return nt > cap ? cap : nt;
  };
  const int nsteps = steps_upto((btok0 + BT < qn ? btok0 + BT : qn) - 1);
  const int wsteps = tok0 < qn ? steps_upto((tok0 + TW < qn ? tok0 + TW : qn) - 1) : 0;
  // First query position of the wave: steps ending at or below it need no causal mask.
  const int wpos0 = kv_len - qn + tok0;

  // Step loads: K and V rows go straight to LDS, 1 KiB (4 rows of this head) per load, four loads
  // per wave: K rows 4 wave .. + 3 and 32 above, then the same V rows.  The rows of a load lie in
  // one page, so its base address is scalar and the lanes' offsets are fixed for the whole sweep.
  // 16-byte chunk ch of K row r sits at slot ch ^ (r % 16) and of V row r at ch ^ 4 (r % 4): the
  // K fragment reads (32 rows, one chunk) and the transposed V reads (4 rows x 64 bytes per 32
  // lanes) then cover the banks once.
  const uint32_t row_bytes = (uint32_t)a.hkv * kHeadDim * 2;
  const uint32_t page_bytes = 2 * kPageSize * row_bytes;
  const int wv = uniform((int)(threadIdx.x >> 6));
  const int lrow = lane >> 4, lch = lane & 15;
  const uint32_t koff = (4 * (wv & 3) + lrow) * row_bytes + 16 * (lch ^ (4 * (wv & 3) + lrow));
  const uint32_t voff = (kPageSize + 4 * (wv & 3) + lrow) * row_bytes + 16 * (lch ^ (4 * lrow));
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)&tiles[0][0] + wv * 1024;
  const char *const kvh = reinterpret_cast<const char *>(a.kv) + (int64_t)h * (kHeadDim * 2);
  // Page ids outside the cache (negative or past it) are looked for once, over all pages the block
  // sweeps: the steps of a row without any (the usual case) take its ids as they are.
  const int32_t *const row_ids = a.kv_indices + p0;
  auto page_bad = [&](int pid) { return pid < 0 || (int64_t)pid >= a.num_pages; };
  bool row_bad = false;
  for (int i = 0; i < nsteps * kPgStep && i < np; i += 64)
    row_bad |= __ballot(i + lane < np && page_bad(row_ids[i + lane < np ? i + lane : 0])) != 0;
  auto bad_of = [&](int j) {  // bit i: page i of step j lies outside the cache
    uint32_t r = 0;
#pragma unroll
    for (int i = 0; i < kPgStep; ++i) {
      const int pg = kPgStep * j + i;
      r |= (pg < np && page_bad(ld_scalar(row_ids, pg < np ? pg : np - 1)) ? 1u : 0u) << i;
    }
    return r;
  };
  // The pages the wave loads four rows of in step j: page (wave / 4) + i PW / 4 of its four; pages
  // past the row repeat its last one (masked later).
  const uint32_t last_pg = (uint32_t)(np - 1);
  uint32_t id[kPgWave];  // of the step issued next
  auto load_ids = [&](int j) {
#pragma unroll
    for (int i = 0; i < kPgWave; ++i) {
      const uint32_t pg = (uint32_t)(kPgStep * j + i * (PW / 4) + (wv >> 2));
      id[i] = (uint32_t)ld_scalar(row_ids, pg < last_pg ? pg : last_pg);
    }
  };
  auto issue = [&](int j, int i) {
    const uint32_t dst = lds0 + (uint32_t)(j % kBufs) * (2 * kTileB) + i * (PW / 4) * 4096;
    const uint32_t pid = row_bad && page_bad((int)id[i]) ? 0u : id[i];
    const char *pg = kvh + (uint64_t)pid * page_bytes;
    load_lds_1k(dst, pg, koff);
    load_lds_1k(dst + kTileB, pg, voff);
  };
  auto issue_step = [&](int j) {  // step j's loads, then the ids of step j + 1
#pragma unroll
    for (int i = 0; i < kPgWave; ++i) issue(j, i);
    load_ids(j + 1);
  };
  if (nsteps > 0) {
    load_ids(0);
    issue_step(0);
    if (kLate && nsteps > 1) issue_step(1);
  }
  uint32_t bad = 0;  // bad_of(j)

  float m = -INFINITY, l = 0.f;
  f32x16 acc[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;
  const float scale2 = fabsf(a.sm_scale) * kLog2e;
  // K fragment of k-slice ks: row 32 sb + n, chunk 2 ks + hl.
  uint32_t kfo[8];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) kfo[ks] = (uint32_t)(n * 256 + 16 * ((2 * ks + hl) ^ (n & 15)));
  // ds_read_b64_tr_b16 of V^T: 16-lane group q16 = lane / 16, t16 = lane % 16 reads rows
  // (kv) base + t16 / 4 at columns 32 dt + 16 (q16 % 2) + 4 (t16 % 4), and receives its column's four rows.
  const int q16 = lane >> 4, t16 = lane & 15;
  uint32_t vfo[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
    vfo[dt] = (uint32_t)(kTileB + (4 * hl + (t16 >> 2)) * 256 +
                         16 * ((4 * dt + 2 * (q16 & 1) + ((t16 & 3) >> 1)) ^ (4 * (t16 >> 2))) + 8 * (t16 & 1));

  // One step for the wave: S^T = K Q^T, the online softmax (accumulators rescaled when the
  // reference maximum moves) and P^T packed into pc.
  auto score_step = [&](int j, const char *tk, u32x4 (&pc)[2 * kSub]) {
    f32x16 S[kSub];
#pragma unroll
    for (int sb = 0; sb < kSub; ++sb)
#pragma unroll
      for (int i = 0; i < 16; ++i) S[sb][i] = 0.f;
    // K fragments three k-slices ahead of the MFMAs that use them; the fences keep the compiler from
    // sinking each read to its use, where every slice would wait out the LDS latency.
    auto kfrag = [&](int sb, int ks) { return *reinterpret_cast<const u32x4 *>(tk + kfo[ks] + sb * 8192); };
    u32x4 kq[4][kSub];
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
      for (int sb = 0; sb < kSub; ++sb) kq[s][sb] = kfrag(sb, s);
    __builtin_amdgcn_sched_barrier(0);
    // Raised wave priority over each MFMA run: of the SIMD's two waves, the one with MFMAs to issue goes
    // first, which pushes the other into its softmax meanwhile (8192 tokens 542 -> 512 us; 300 and 2048 tokens,
    // in 4-wave blocks, the same within 1-2 %).
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      if (ks + 3 < 8) {
#pragma unroll
        for (int sb = 0; sb < kSub; ++sb) kq[(ks + 3) % 4][sb] = kfrag(sb, ks + 3);
      }
#pragma unroll
      for (int sb = 0; sb < kSub; ++sb) S[sb] = MF::run(kq[ks % 4][sb], qf[ks], S[sb]);
      if (!kLate && ks < kPgWave && j + 1 < nsteps) issue(j + 1, ks);  // the next step's loads go out under the MFMAs
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!kLate && j + 1 < nsteps) load_ids(j + 2);
    __builtin_amdgcn_s_setprio(0);
    // Masks only where the step crosses the wave's first diagonal, kv_len, or a bad page.
    const int kv0 = j * kKvStep;
    const bool full = kv0 + kKvStep - 1 <= wpos0 && kv0 + kKvStep <= kv_len && bad == 0;
    // Row maxima on the raw scores (the scale is positive, so it commutes with max), then
    // x = S * scale - m as one fma.  m is the row's reference maximum: it moves only when a
    // score exceeds it by more than 8 (a factor of 2^8), so the exponentials stay <= 256 and the
    // accumulators are rescaled only on those steps.
    constexpr int NX = 16 * kSub;
    float x[NX];
    float pm = -INFINITY;
    if (full) {
#pragma unroll
      for (int i = 0; i < NX; ++i) {
        x[i] = S[i >> 4][i & 15];
        pm = fmaxf(pm, x[i]);
      }
    } else {
      bool pg_ok[kPgStep];
#pragma unroll
      for (int p = 0; p < kPgStep; ++p) pg_ok[p] = ((bad >> p) & 1u) == 0;
#pragma unroll
      for (int i = 0; i < NX; ++i) {
        const int mm = 32 * (i >> 4) + 8 * ((i & 15) >> 2) + 4 * hl + (i & 3);
        const int tk_i = kv0 + mm;
        x[i] = (row_ok && pg_ok[mm >> 4] && tk_i <= qpos && tk_i < kv_len) ? S[i >> 4][i & 15] : -INFINITY;
        pm = fmaxf(pm, x[i]);
      }
    }
    const float smax = halves_max(pm) * scale2;
    float alpha = 1.f;
    if (smax > m + 8.f) {  // also the first finite score of the row (m = -inf)
      alpha = fast_exp2(m - smax);
      m = smax;
    }
    const float nm = m == -INFINITY ? 0.f : -m;
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      x[i] = fast_exp2(fmaf(x[i], scale2, nm));
      ps += x[i];
    }
    l = l * alpha + ps;  // this half's tokens; the halves are summed once at the end
    if (__ballot(alpha != 1.f)) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[dt][i] *= alpha;
    }
    // P^T chunks: values 8c .. 8c + 7 of this lane, rounded to the KV dtype.
#pragma unroll
    for (int cc = 0; cc < 2 * kSub; ++cc)
#pragma unroll
      for (int w = 0; w < 4; ++w)
        pc[cc][w] = pack2<DT>(x[8 * cc + 2 * w], x[8 * cc + 2 * w + 1]);
  };
  // O^T += V^T P^T of a step whose P^T is in pc.
  auto pv_step = [&](const char *tk, const u32x4 (&pc)[2 * kSub]) {
    auto vfrag = [&](int i) {  // V^T fragment of chunk i / 4, d tile i % 4
      const char *rd = tk + vfo[i % 4] + (i / 4) * 4096;
      const ps4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ps4_t *)rd);
      const ps4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ps4_t *)(rd + 2048));
      u32x4 va;
      va[0] = (uint32_t)(uint16_t)v0[0] | ((uint32_t)(uint16_t)v0[1] << 16);
      va[1] = (uint32_t)(uint16_t)v0[2] | ((uint32_t)(uint16_t)v0[3] << 16);
      va[2] = (uint32_t)(uint16_t)v1[0] | ((uint32_t)(uint16_t)v1[1] << 16);
      va[3] = (uint32_t)(uint16_t)v1[2] | ((uint32_t)(uint16_t)v1[3] << 16);
      return va;
    };
    constexpr int kAhead = 4;  // fragments read ahead of their MFMAs
    u32x4 vq[kAhead + 1];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) vq[i] = vfrag(i);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < 8 * kSub; ++i) {
      if (i + kAhead < 8 * kSub) vq[(i + kAhead) % (kAhead + 1)] = vfrag(i + kAhead);
      acc[i % 4] = MF::run(vq[i % (kAhead + 1)], pc[i / 4], acc[i % 4]);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
  };

  // (PW = 8) Waves 0-3 (one per SIMD) run each step whole; waves 4-7, the SIMDs' second waves, run half
  // a step behind: P.V of the previous step first, then S and the softmax of this one.  So on
  // each SIMD one wave's softmax runs while the other wave's MFMAs do (P.V of one under the
  // other's softmax, S of one under the other's softmax), not both softmaxes at once.  A step's
  // tiles stay in LDS for one more step: the late waves read step j - 1 after the barrier of step j.
  const bool late = kLate && wave >= PW / 2;
  u32x4 pcar[2 * kSub];
  for (int j = 0; nsteps > 0 && j < nsteps + (kLate ? 1 : 0); ++j) {
    // Step j's loads have landed when at most the next step's (kLate: four) are pending.
    if (kLate && j + 1 < nsteps)
      wait_loads<2 * kPgWave>();
    else
      wait_loads<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (row_bad) bad = j < nsteps ? bad_of(j) : 0u;
    if (j < nsteps && ((j + 1) * kKvStep > kv_len || bad != 0)) {
      // V rows past kv_len and of pages outside the cache meet p = 0 but may hold NaN/Inf: zeros.
      constexpr int kTpr = PW;  // threads per row
      const int r = (int)threadIdx.x / kTpr;
      if (j * kKvStep + r >= kv_len || ((bad >> (r >> 4)) & 1u)) {
        char *vr = &tiles[j % kBufs][kTileB + r * 256 + 256 / kTpr * ((int)threadIdx.x % kTpr)];
#pragma unroll
        for (int i = 0; i < 16 / kTpr; ++i) st128(vr + 16 * i, u32x4{0u, 0u, 0u, 0u});
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    if (kLate ? j + 2 < nsteps : j >= wsteps && j + 1 < nsteps) issue_step(kLate ? j + 2 : j + 1);
    if (late) {
      if (j >= 1 && j - 1 < wsteps) pv_step(&tiles[(j - 1) % kBufs][0], pcar);
      if (j < wsteps) score_step(j, &tiles[j % kBufs][0], pcar);
    } else if (j < wsteps) {
      u32x4 pc[2 * kSub];
      score_step(j, &tiles[j % kBufs][0], pc);
      pv_step(&tiles[j % kBufs][0], pc);
    }
  }

  // Normalise and write: lane l holds O[row l%32][32 dt + 8 (i / 4) + 4 hl + i % 4].
  l = halves_sum(l);
  if (row_ok) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    uint16_t *op = a.o + (q0 + tok0 + tt) * a.o_stride_t + (int64_t)(h * G + g) * a.o_stride_h + 4 * hl;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        uint2 w;
        w.x = pack2<DT>(acc[dt][4 * q4] * inv, acc[dt][4 * q4 + 1] * inv);
        w.y = pack2<DT>(acc[dt][4 * q4 + 2] * inv, acc[dt][4 * q4 + 3] * inv);
        *reinterpret_cast<uint2 *>(op + 32 * dt + 8 * q4) = w;
      }
    if (a.lse && hl == 0) a.lse[(q0 + tok0 + tt) * a.hq + h * G + g] = l > 0.f ? (m + log2f(l)) * kLn2 : -INFINITY;
  }
}

// Whether blocks hold 8 waves instead of 4 (bt4 query tokens).  Where CUs would be left without a block, 4
// waves spread a prompt over twice as many; where the chip is full anyway, 8 waves run a step faster (loads
// two steps ahead, P.V of one wave under the softmax of the other).
bool wide_blocks(const PrefillArgs &a, int bt4, int max_qo) {
  // The longest prompt alone is 850 4-wave blocks, nearly two rounds over the chip's 512.  us for 8 / 4
  // waves, 8 kv heads of 4 q heads: 3000 tokens (752 blocks) 88.9 / 86.0, 3200 (800) 94.1 / 93.3, 3500 (880)
  // 103.5 / 111, 4000 (1000) 131 / 142, 8192 (2048) 513 / 541; 2 kv heads of 6: 4096 (410) 105.5 / 94.6,
  // 6500 (650) 172 / 165, 8192 (820) 231.5 / 230, 16384 (1640) 833 / 849.
  if (a.hkv * ceil_div(max_qo, bt4) >= 850) return true;
  // Prompts of one 8-wave block or two 4-wave ones, and the latter no longer fit one to a CU: 60 prompts
  // of 20, 4 kv heads of 7 (240 / 480 blocks) 10.2 / 12.6 us; 100 of 30, 2 of 6 (200 / 400) 10.9 / 11.8.
  const int64_t blocks = (int64_t)a.batch * a.hkv;
  if (max_qo > bt4 && max_qo <= 2 * bt4 && blocks <= 256 && 2 * blocks > 256) return true;
  // Prompts continued over at least 3.5 times as many cached tokens, whose blocks all sweep about as far, and
  // well more 4-wave blocks than one to a CU: 1500 tokens at 16 k (376 blocks) 426 / 464 us, 2048 at 8 k (512)
  // 284 / 298, 8 of 256 at 4 k (512) 139 / 149; but 1024 at 8 k (256) 222 / 195, 4 of 331 at 1 k (331, three
  // times; with RoPE + append) 49.4 / 47.5, 3000 at 8 k (2.7 times) 482 / 479, 2048 at 4 k (twice) 172 / 172.
  if (a.num_tokens < 0) return false;
  const int64_t tokens = a.num_tokens - a.decode_rows;
  const int64_t cached = (a.kv_indices_len - a.decode_pages) * kPageSize - tokens;
  return 2 * cached >= 7 * tokens && tokens * a.hkv >= 350 * (int64_t)bt4;
}

template <int DT, int G>
void launch_prefill_g(PrefillArgs a, int max_qo, hipStream_t stream) {
  const bool wide = wide_blocks(a, 32 / G * 4, max_qo);
  const int bt = 32 / G * (wide ? 8 : 4);
  a.row_tiles = (int)ceil_div(max_qo, bt);
  const int64_t slots = (int64_t)a.batch * a.row_tiles;
  a.order = a.batch == 1 || slots * a.hkv <= (a.row_tiles <= 4 ? 512 : 256) ? kBySlot
            : a.batch <= kByTileRows && a.row_tiles <= 32 * 64  ? kByTile
                                                                : kByRow;
  // Tiles of that many tokens over that many rows, at most: what is launched past the last one only exits, but
  // a row of 5000 tokens beside 20 of 100 has 1540 slots too many (242 us, with the bound 215).
  const int64_t most = a.num_tokens < 0 ? slots : (a.num_tokens + (int64_t)a.batch * (bt - 1)) / bt;
  const int64_t used = a.order == kBySlot || slots < most ? slots : most, y = used < 32768 ? used : 32768;
  const dim3 grid((unsigned)a.hkv, (unsigned)y, (unsigned)ceil_div(used, y));
  if (wide)
    hipLaunchKernelGGL((paged_prefill_kernel<DT, G, 8>), grid, dim3(512), 0, stream, a);
  else
    hipLaunchKernelGGL((paged_prefill_kernel<DT, G, 4>), grid, dim3(256), 0, stream, a);
}

template <int DT>
void launch_prefill(const PrefillArgs &a, int G, int max_qo, hipStream_t stream) {
  switch (G) {
    case 1: launch_prefill_g<DT, 1>(a, max_qo, stream); break;
    case 2: launch_prefill_g<DT, 2>(a, max_qo, stream); break;
    case 3: launch_prefill_g<DT, 3>(a, max_qo, stream); break;
    case 4: launch_prefill_g<DT, 4>(a, max_qo, stream); break;
    case 5: launch_prefill_g<DT, 5>(a, max_qo, stream); break;
    case 6: launch_prefill_g<DT, 6>(a, max_qo, stream); break;
    case 7: launch_prefill_g<DT, 7>(a, max_qo, stream); break;
    default: launch_prefill_g<DT, 8>(a, max_qo, stream); break;
  }
}

// With a workspace (of decode_rows_workspace_bytes) the rows of one query token go to run_decode_rows.
int run_prefill(const void *q, int64_t q_stride_t, int64_t q_stride_h, const void *kv_cache, int64_t num_pages,
                const int32_t *qo_indptr, const int32_t *kv_indptr, const int32_t *kv_indices, int64_t kv_indices_len,
                const int32_t *kv_last_page_len, void *o, int64_t o_stride_t, int64_t o_stride_h, float *lse, int batch,
                int num_qo_heads, int num_kv_heads, int head_dim, int dtype, float sm_scale, int max_qo_len,
                int64_t num_tokens, int decode_rows, int64_t decode_pages, int64_t decode_max_pages, void *workspace,
                size_t workspace_bytes, delta_stream_t stream, const char *who) {
  clear_error();
  if (batch <= 0 || max_qo_len <= 0) return DELTA_OK;
  if (head_dim != kHeadDim) return set_error(DELTA_ERR_INVALID, "%s: head_dim must be 128", who);
  if (num_kv_heads <= 0 || num_qo_heads <= 0 || num_qo_heads % num_kv_heads)
    return set_error(DELTA_ERR_INVALID, "%s: num_qo_heads must be a multiple of num_kv_heads", who);
  const int G = num_qo_heads / num_kv_heads;
  if (G > kMaxGroup) return set_error(DELTA_ERR_INVALID, "%s: group size %d > %d unsupported", who, G, kMaxGroup);
  if (dtype != DELTA_BF16 && dtype != DELTA_FP16) return set_error(DELTA_ERR_INVALID, "%s: bad dtype", who);
  if (!q || !kv_cache || !qo_indptr || !kv_indptr || !kv_indices || !kv_last_page_len || !o)
    return set_error(DELTA_ERR_INVALID, "%s: null pointer", who);
  if (((uintptr_t)q | (uintptr_t)kv_cache) & 15u || (q_stride_t % 8) || (q_stride_h % 8))
    return set_error(DELTA_ERR_INVALID, "%s: q and kv_cache 16-byte aligned, q strides multiples of 8", who);
  if (((uintptr_t)o & 7u) || (o_stride_t % 4) || (o_stride_h % 4))
    return set_error(DELTA_ERR_INVALID, "%s: o 8-byte aligned with strides in multiples of 4", who);
  if (num_pages <= 0 || kv_indices_len < 0) return set_error(DELTA_ERR_INVALID, "%s: empty cache", who);
  PrefillArgs a;
  a.q = (const uint16_t *)q;
  a.q_stride_t = q_stride_t;
  a.q_stride_h = q_stride_h;
  a.kv = (const uint16_t *)kv_cache;
  a.num_pages = num_pages;
  a.qo_indptr = qo_indptr;
  a.kv_indptr = kv_indptr;
  a.kv_indices = kv_indices;
  a.kv_indices_len = kv_indices_len;
  a.last_page_len = kv_last_page_len;
  a.o = (uint16_t *)o;
  a.o_stride_t = o_stride_t;
  a.o_stride_h = o_stride_h;
  a.lse = lse;
  a.batch = batch;
  a.hq = num_qo_heads;
  a.hkv = num_kv_heads;
  a.sm_scale = sm_scale;
  a.num_tokens = num_tokens;
  a.decode_rows = decode_rows;
  a.decode_pages = decode_pages;
  a.skip_single = workspace != nullptr;
  if (workspace) {
    const size_t need = decode_rows_workspace_bytes(batch, num_qo_heads, kv_indices_len);
    if (workspace_bytes < need)
      return set_error(DELTA_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", who, need, workspace_bytes);
    if ((uintptr_t)workspace & 255u) return set_error(DELTA_ERR_INVALID, "%s: workspace must be 256-byte aligned", who);
    const int rc = run_decode_rows(q, q_stride_t, q_stride_h, kv_cache, num_pages, qo_indptr, kv_indptr, kv_indices,
                                   kv_indices_len, kv_last_page_len, o, o_stride_t, o_stride_h, lse, batch, num_qo_heads,
                                   num_kv_heads, dtype, sm_scale, decode_pages, decode_max_pages, workspace,
                                   (hipStream_t)stream, who);
    if (rc || max_qo_len == 1) return rc;
  }
  if (dtype == DELTA_BF16)
    launch_prefill<DELTA_BF16>(a, G, max_qo_len, (hipStream_t)stream);
  else
    launch_prefill<DELTA_FP16>(a, G, max_qo_len, (hipStream_t)stream);
  return check_launch(who);
}
}  // namespace
}  // namespace delta

extern "C" DELTA_EXPORT int delta_paged_prefill(const void *q, int64_t q_stride_t, int64_t q_stride_h,
                                                const void *kv_cache, int64_t num_pages, const int32_t *qo_indptr,
                                                const int32_t *kv_indptr, const int32_t *kv_indices,
                                                int64_t kv_indices_len, const int32_t *kv_last_page_len, void *o,
                                                int64_t o_stride_t, int64_t o_stride_h, float *lse, int batch,
                                                int num_qo_heads, int num_kv_heads, int head_dim, int dtype,
                                                float sm_scale, int max_qo_len, delta_stream_t stream) {
  return delta::run_prefill(q, q_stride_t, q_stride_h, kv_cache, num_pages, qo_indptr, kv_indptr, kv_indices,
                            kv_indices_len, kv_last_page_len, o, o_stride_t, o_stride_h, lse, batch, num_qo_heads,
                            num_kv_heads, head_dim, dtype, sm_scale, max_qo_len, -1, 0, 0, 0, nullptr, 0, stream,
                            "delta_paged_prefill");
}

extern "C" DELTA_EXPORT size_t delta_paged_prefill_rows_workspace_bytes(int batch, int num_qo_heads, int num_kv_heads,
                                                                        int64_t kv_indices_len) {
  if (batch <= 0 || num_qo_heads <= 0 || num_kv_heads <= 0 || kv_indices_len < 0) return 0;
  return delta::decode_rows_workspace_bytes(batch, num_qo_heads, kv_indices_len);
}

extern "C" DELTA_EXPORT int delta_paged_prefill_rows(const void *q, int64_t q_stride_t, int64_t q_stride_h,
                                                     const void *kv_cache, int64_t num_pages, const int32_t *qo_indptr,
                                                     const int32_t *kv_indptr, const int32_t *kv_indices,
                                                     int64_t kv_indices_len, const int32_t *kv_last_page_len, void *o,
                                                     int64_t o_stride_t, int64_t o_stride_h, float *lse, int batch,
                                                     int num_qo_heads, int num_kv_heads, int head_dim, int dtype,
                                                     float sm_scale, int max_qo_len, int64_t num_tokens,
                                                     int decode_rows, int64_t decode_pages, int64_t decode_max_pages,
                                                     void *workspace, size_t workspace_bytes,
                                                     delta_stream_t stream) {
  const char *who = "delta_paged_prefill_rows";
  if (batch > 0 && max_qo_len > 0 &&
      (num_tokens < 0 || decode_rows < 0 || decode_rows > batch || decode_pages < 0 || decode_pages > kv_indices_len ||
       decode_max_pages < 0 || decode_max_pages > decode_pages)) {
    delta::clear_error();
    return delta::set_error(DELTA_ERR_INVALID,
                            "%s: num_tokens, decode_rows, decode_pages or decode_max_pages out of range", who);
  }
  return delta::run_prefill(q, q_stride_t, q_stride_h, kv_cache, num_pages, qo_indptr, kv_indptr, kv_indices,
                            kv_indices_len, kv_last_page_len, o, o_stride_t, o_stride_h, lse, batch, num_qo_heads,
                            num_kv_heads, head_dim, dtype, sm_scale, max_qo_len, num_tokens, decode_rows, decode_pages,
                            decode_max_pages, workspace, workspace_bytes, stream, who);
}
