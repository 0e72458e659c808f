// Affix importance for anchor selection (gfx950): for every request, the attention that its [MASK]
// queries pay to each cached affix key, soft-maxed over the affix keys only and summed over the mask
// queries and heads of one layer.
//
//   w[r, h, a]       = softmax_a( q[r, h] . rot(K[a, kv(h)], shift_b) * scale )     a in [0, A)
//   importance[b, a] += sum_{r in mask rows of b} sum_h w[r, h, a]
//
// Relocation is applied on the query side: q . rot(k, +s) = rot(q, -s) . k, so that every launch reads the cached
// affix keys as they lie in the cache: one copy, shared by all requests and resident in L2.  Scores come from the
// matrix core (S^T = K Q^T, keys as rows, one query column per lane).  No atomics anywhere: the result does not
// depend on scheduling.
//
// Head dims of 64 and 128 with affixes of up to 1280 keys: importance_fused_kernel, one pass over the scores, then
// importance_reduce_kernel, which adds the per-head partial sums to importance[b, :] in a fixed order.
//
// Everything else, two passes: a first launch writes each request's [MASK] queries, packed in mask-row order and
// (with relocation) rotated by minus the request's shift, into the workspace; then
//   1. statistics pass: the mask rows of a wave stay in registers, the affix keys stream by, and the wave
//      leaves log2 of each row's sum of 2^(score * c) in the workspace;
//   2. column pass: the affix keys of a wave stay in registers, the request's mask rows stream by, the scores
//      are recomputed, normalised with the stored row statistic (one subtraction in the exponent) and summed
//      per key; each wave is the only writer of its entries of the per-head partial sums in the workspace;
//   3. importance_reduce_kernel.
// Both passes exist twice: for head dims of 64, 128 and 256 the streamed operand is staged through LDS by the copy
// engine and shared by the four waves of a workgroup (importance_*_lds_kernel, further down); every other head dim
// loads its fragments straight from global memory in operand layout, 16 bytes per lane, without LDS or barriers
// (importance_stats_kernel, importance_colsum_kernel).
#include <mutex>
#include <type_traits>

#include "common.h"
#include "mma.h"
#include "attn_common.h"

namespace acache {

struct ImportanceParams {
  float *importance;
  const char *q;
  const char *k_cache;
  const int32_t *mask_rows;
  const int32_t *cu_mask;
  const int32_t *shifts;
  const float *cos_tab;
  const float *sin_tab;
  float *stats;            // per (mask row, head): log2 of the row's sum of 2^(score * c)
  float *partial;
  char *q_rot;            // [total_mask_rows, H, D] mask queries packed in mask-row order, counter-rotated
  int64_t total_q;        // rows of q; a mask row outside [0, total_q) is an absent query
  int64_t imp_stride;
  int64_t q_token_bytes, q_head_bytes;
  int64_t kv_slot_bytes, kv_head_bytes;
  int64_t affix_slot0;
  float scale_log2e;
  int32_t A;
  int32_t B;
  int32_t H;
  int32_t H_kv;
  int32_t rope_rows;
  int32_t max_row_tiles;
  int32_t D;  // head_dim
  int32_t total_mask_rows;  // entries of mask_rows, rows of the packed query copy and of stats
  int32_t max_mask_rows;    // the launch grids cover this many mask rows per request
};

// First mask row and number of mask rows of request b, held to what the workspace and the launch grids were
// sized for: the prefix sums live in device memory, where the host cannot check them, and a request that
// claims more rows than the caller declared is cut there instead of being read past the buffers.
__device__ __forceinline__ void request_rows(const ImportanceParams &p, int b, int &m0, int &n_rows) {
  m0 = p.cu_mask[b];
  m0 = m0 < 0 ? 0 : (m0 > p.total_mask_rows ? p.total_mask_rows : m0);
  int n = p.cu_mask[b + 1] - m0;
  const int room = p.total_mask_rows - m0;
  n = n > room ? room : n;
  n = n > p.max_mask_rows ? p.max_mask_rows : n;
  n_rows = n < 0 ? 0 : n;
}

// Operand fragments of 16 rows x D, KS = ceil(D / 32) slabs of 32 elements: lane (li, lg) takes elements
// 32*ks + 8*lg .. + 8 of row `row_ptr` (always a readable row: callers clamp indices instead of branching, so
// the loads of a tile issue back to back); chunks at or past D (a multiple of 16) read as zeros.
template <int D>
__device__ __forceinline__ void load_rows(vec16 (&f)[(D + 31) / 32], const char *row_ptr, int lg) {
  constexpr int KS = (D + 31) / 32;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    if (32 * ks + 32 <= D) {
      f[ks] = load16(row_ptr + (32 * ks + 8 * lg) * 2);
    } else {  // the half-filled last slab of D = 16 (mod 32): lane groups 2 and 3 hold zeros
      const vec16 v = load16(row_ptr + (32 * ks + 8 * (lg & 1)) * 2);
      f[ks] = lg < 2 ? v : vec16{{0, 0, 0, 0}};
    }
  }
}

// Counter-rotate the [MASK] queries once per call: q_rot[m0_b + r, h, :] = rot(q[mask_rows[m0_b + r], h, :], -shift_b).
// One row of D elements per D/16 lanes, the rotate-half partner in the same lane; fp32 products and sum rounded
// separately, one rounding to the query type (the query-side arithmetic of the attention kernel).  A mask row
// outside q is written as zeros (and counted as absent by the statistics kernel).
template <int DTYPE>
__global__ __launch_bounds__(256) void importance_rotate_kernel(ImportanceParams p) {
  const int D = p.D;
  const int half_bytes = D;  // D / 2 elements of 2 bytes
  const int lpr = half_bytes / 16;
  const int b = blockIdx.y;
  int m0, n_rows;
  request_rows(p, b, m0, n_rows);
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = g / lpr;
  const int lane = (int)(g - row * lpr);
  if (row >= (int64_t)n_rows * p.H) return;
  const int r = (int)(row / p.H);
  const int h = (int)(row - (int64_t)r * p.H);
  char *dst = p.q_rot + (((int64_t)(m0 + r) * p.H + h) * D) * 2 + lane * 16;
  const int64_t src_row = p.mask_rows[m0 + r];
  vec16 lo = {{0, 0, 0, 0}}, hi = {{0, 0, 0, 0}};
  if (src_row >= 0 && src_row < p.total_q) {
    const char *src = p.q + src_row * p.q_token_bytes + (int64_t)h * p.q_head_bytes + lane * 16;
    lo = load16(src);
    hi = load16(src + half_bytes);
    int shift = p.shifts ? p.shifts[b] : 0;
    if (shift < 0 || shift >= p.rope_rows) shift = 0;
    if (shift != 0)
      rotate_pair_half<DTYPE>(lo, hi, p.cos_tab + (int64_t)shift * D, p.sin_tab + (int64_t)shift * D, lane * 8, D / 2, -1.0f);
  }
  store16(dst, lo);
  store16(dst + half_bytes, hi);
}

// Row r of request b (first mask row m0), head h, in the packed copy the first launch wrote.  Always a readable
// address: r is clamped to the request's rows (callers discard what a clamped row contributes).  The copy is
// smaller than 4 GiB (checked at launch), so the offset is 32-bit arithmetic.
__device__ __forceinline__ const char *mask_query_row(const ImportanceParams &p, int m0, int n_rows, int r, int h) {
  r = r < n_rows ? r : n_rows - 1;
  return p.q_rot + ((uint32_t)(m0 + r) * (uint32_t)p.H + (uint32_t)h) * (uint32_t)(p.D * 2);
}

// Sum over the 16 lanes of a row (lanes sharing lane >> 4), left in every lane of the row: four rotate-and-add
// steps in the vector ALU's lane-permute path (no trip through LDS).
__device__ __forceinline__ float row_sum16(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xf, 0xf, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x124, 0xf, 0xf, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x122, 0xf, 0xf, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x121, 0xf, 0xf, false));
  return v;
}

constexpr int kKeysPerStep = 64;  // keys a colsum wave owns (four independent 16-key tiles in flight)
constexpr int kStatKeys = 32;     // keys a stats wave scores per loop step (two 16-key tiles x two row tiles in flight)

constexpr int kRowTilesPerWave = 4;  // 16-row tiles of mask queries a stats wave owns (keys are loaded once for all)

// One wave per (request, head, 64 mask rows): the rows stay in registers, the affix keys stream by, and the wave
// leaves log2(sum_a 2^(s[r, a] * c)) per row (running maximum + log2 of the running sum) in the workspace.
template <int DTYPE, int D>
__global__ __launch_bounds__(256) void importance_stats_kernel(ImportanceParams p) {
  constexpr int NQ = kRowTilesPerWave;
  constexpr int KS = (D + 31) / 32;
  using M = Mma<DTYPE>;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int groups = (p.max_row_tiles + NQ - 1) / NQ;
  const int b = blockIdx.x / groups, rg = blockIdx.x % groups;
  const int h = blockIdx.y * 4 + wave;
  int m0, n_rows;
  request_rows(p, b, m0, n_rows);
  const int row0 = rg * NQ * 16;
  if (h >= p.H || row0 >= n_rows) return;  // no barrier in this kernel: waves may leave early
  const int kvh = h / (p.H / p.H_kv);

  vec16 qf[NQ][KS];
#pragma unroll
  for (int qt = 0; qt < NQ; ++qt) load_rows<D>(qf[qt], mask_query_row(p, m0, n_rows, row0 + 16 * qt + li, h), lg);
  const char *k_base = p.k_cache + p.affix_slot0 * p.kv_slot_bytes + (int64_t)kvh * p.kv_head_bytes;
  const float c = p.scale_log2e;

  float m_run[NQ], l_run[NQ];  // per query column (lane li); l is this lane group's share
#pragma unroll
  for (int qt = 0; qt < NQ; ++qt) { m_run[qt] = -INFINITY; l_run[qt] = 0.0f; }
  constexpr int NT = kStatKeys / 16;
  // keys a0 + 16*nt + li of one step, clamped to the affix (a clamped key is masked out below)
  auto fetch = [&](int a0, vec16 (&kf)[NT][KS]) __attribute__((always_inline)) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int a = a0 + 16 * nt + li;
      load_rows<D>(kf[nt], k_base + (int64_t)(a < p.A ? a : p.A - 1) * p.kv_slot_bytes, lg);
    }
  };
  // one step on the keys in `kf`, with the next step's keys requested first (always: past the end the clamped
  // addresses are re-read and the result ignored, which keeps the loop free of a branch the loads would wait at)
  auto step = [&](int a0, vec16 (&kf)[NT][KS], vec16 (&kf_next)[NT][KS]) __attribute__((always_inline)) {
    fetch(a0 + kStatKeys, kf_next);
    const bool tail = a0 + kStatKeys > p.A;  // wave-uniform: only the last step holds keys past the affix
#pragma unroll
    for (int qp = 0; qp < NQ; qp += 2) {  // two row tiles at a time: four independent accumulator chains
      f32x4 sc[2][NT];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) sc[u][nt] = f32x4{0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) sc[u][nt] = M::run(kf[nt][ks], qf[qp + u][ks], sc[u][nt]);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int qt = qp + u;
        if (tail) {
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (a0 + 16 * nt + 4 * lg + i >= p.A) sc[u][nt][i] = -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sc[u][nt][i]);
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float m_new = fmaxf(m_run[qt], mx * c);  // finite: every step holds at least one existing key
        float add = 0.0f;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int i = 0; i < 4; ++i) add += __builtin_amdgcn_exp2f(__builtin_fmaf(sc[u][nt][i], c, -m_new));
        l_run[qt] = l_run[qt] * __builtin_amdgcn_exp2f(m_run[qt] - m_new) + add;
        m_run[qt] = m_new;
      }
    }
  };
  vec16 kf_a[NT][KS], kf_b[NT][KS];
  fetch(0, kf_a);
  for (int a0 = 0; a0 < p.A; a0 += 2 * kStatKeys) {
    step(a0, kf_a, kf_b);
    if (a0 + kStatKeys < p.A) step(a0 + kStatKeys, kf_b, kf_a);
  }
#pragma unroll
  for (int qt = 0; qt < NQ; ++qt) {
    float l = l_run[qt];
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    const int r = row0 + 16 * qt + li;
    if (lg == 0 && r < n_rows) {
      const int64_t src_row = p.mask_rows[m0 + r];
      const bool present = src_row >= 0 && src_row < p.total_q;  // an absent query gets 2^-inf = 0: it adds nothing
      p.stats[(int64_t)(m0 + r) * p.H + h] = present ? m_run[qt] + __builtin_amdgcn_logf(l) : INFINITY;
    }
  }
}

constexpr int kColRowTiles = 2;  // 16-row tiles of mask queries a colsum wave scores per loop step

// One wave per (request, head, 64 affix keys): the keys stay in registers, the request's mask rows stream by
// 32 at a time (the next 32 already on their way).  The wave is the only writer of partial[b, h, a0 .. a0 + 64).
template <int DTYPE, int D>
__global__ __launch_bounds__(256) void importance_colsum_kernel(ImportanceParams p) {
  constexpr int KS = (D + 31) / 32;
  constexpr int NR = kColRowTiles;
  using M = Mma<DTYPE>;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int b = blockIdx.z;
  const int h = blockIdx.y * 4 + wave;
  const int a0 = blockIdx.x * kKeysPerStep;
  int m0, n_rows;
  request_rows(p, b, m0, n_rows);
  if (h >= p.H) return;
  const float c = p.scale_log2e;
  const int kvh = h / (p.H / p.H_kv);
  const char *k_base = p.k_cache + p.affix_slot0 * p.kv_slot_bytes + (int64_t)kvh * p.kv_head_bytes;

  vec16 kf[4][KS];  // keys past the affix repeat the last one; their columns are not stored
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    const int a = a0 + 16 * nt + li;
    load_rows<D>(kf[nt], k_base + (int64_t)(a < p.A ? a : p.A - 1) * p.kv_slot_bytes, lg);
  }
  float col[4][4] = {};
  auto fetch = [&](int r0, vec16 (&qf)[NR][KS], float (&st)[NR]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NR; ++t) {
      const int r = r0 + 16 * t + li;
      load_rows<D>(qf[t], mask_query_row(p, m0, n_rows, r, h), lg);
      st[t] = p.stats[(int64_t)(m0 + (r < n_rows ? r : n_rows - 1)) * p.H + h];
    }
  };
  // one step on the 32 rows in `qf`, with the next 32 requested first (always: past the end the clamped rows are
  // re-read and ignored, which keeps the loop free of a branch the loads would wait at)
  auto step = [&](int r0, vec16 (&qf)[NR][KS], float (&st)[NR], vec16 (&qf_next)[NR][KS], float (&st_next)[NR])
      __attribute__((always_inline)) {
    fetch(r0 + 16 * NR, qf_next, st_next);
#pragma unroll
    for (int t = 0; t < NR; ++t) {
      // a row past the request's end was read from a clamped address: 2^-inf = 0 keeps it out of the sums (the
      // test sits here, not at the load, so that the prefetch is not waited for the moment it is issued)
      const float ref = r0 + 16 * t + li < n_rows ? st[t] : INFINITY;
      f32x4 sc[4];
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) sc[nt] = f32x4{0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)  // four independent accumulator chains between two steps of one chain
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) sc[nt] = M::run(kf[nt][ks], qf[t][ks], sc[nt]);
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) col[nt][i] += __builtin_amdgcn_exp2f(__builtin_fmaf(sc[nt][i], c, -ref));
    }
  };
  vec16 q_a[NR][KS], q_b[NR][KS];
  float st_a[NR], st_b[NR];
  if (n_rows > 0) fetch(0, q_a, st_a);
  for (int r0 = 0; r0 < n_rows; r0 += 32 * NR) {
    step(r0, q_a, st_a, q_b, st_b);
    if (r0 + 16 * NR < n_rows) step(r0 + 16 * NR, q_b, st_b, q_a, st_a);
  }
  // sum over the 16 query columns (lanes li) of every key row
  float *dst = p.partial + ((int64_t)b * p.H + h) * p.A;
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v = row_sum16(col[nt][i]);
      const int a = a0 + 16 * nt + 4 * lg + i;
      if (li == 0 && a < p.A) dst[a] = v;
    }
}

// ---------------------------------------------------------------------------------------------------
// The same two passes for head dims of 64, 128 and 256 with the streamed operand staged through LDS.
// In the kernels above every wave pulls the streamed rows (keys in the statistics pass, queries in the
// column pass) from L2 in operand layout, 64 bytes of a row per four lanes: the workgroup's four waves ask
// for the same or neighbouring rows four times over and the vector memory path, not the matrix core, sets
// the pace.  Here the four waves of a workgroup share one stream: the copy engine writes each 32-row tile
// into LDS once (whole rows, 16 bytes per lane, two buffers in turn) and all four waves read their
// fragments from there.  Rows are laid out with the 16-byte chunks of row r XOR-ed by r, so that the 16
// lanes reading one chunk column of 16 different rows hit 16 different bank groups.
constexpr int kStageRows = 32;  // query rows per LDS tile of the column pass
constexpr int kStageKeys = 64;  // keys per LDS tile of the statistics pass

template <int D, int ROWS>
struct StageGeometry {
  static constexpr int kChunks = D / 8;                   // 16-byte chunks per row (a power of two)
  static constexpr int kTileBytes = ROWS * D * 2;
  static constexpr int kCopiesPerWave = ROWS * D / 2048;  // 1 KiB wave copies per tile, split over four waves
  // chunk `c` of tile row `row` lives at this byte offset of the tile
  static __device__ __forceinline__ int offset(int row, int c) { return row * (D * 2) + ((c ^ (row & (kChunks - 1))) << 4); }
};

// Fragment of tile rows 16*t + li from LDS, in the layout load_rows() produces from global memory.
template <int D>
__device__ __forceinline__ void load_rows_lds(vec16 (&f)[D / 32], const char *tile, int t, int li, int lg) {
  using G = StageGeometry<D, 16>;  // the offset of a chunk does not depend on the tile height
#pragma unroll
  for (int ks = 0; ks < D / 32; ++ks) f[ks] = *(const vec16 *)(tile + G::offset(16 * t + li, 4 * ks + lg));
}

// One workgroup per (request, head, 256 mask rows): wave w keeps rows 64*w .. 64*w + 63 in registers, the
// affix keys stream through LDS 32 at a time.  Same arithmetic and the same statistic as importance_stats_kernel.
template <int DTYPE, int D>
__global__ __launch_bounds__(256) void importance_stats_lds_kernel(ImportanceParams p) {
  constexpr int NQ = kRowTilesPerWave, KS = D / 32, NT = 2;  // key tiles scored together (a 64-key LDS tile: two rounds)
  using M = Mma<DTYPE>;
  using G = StageGeometry<D, kStageKeys>;
  __shared__ __attribute__((aligned(1024))) char tiles[2][G::kTileBytes];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int groups = (p.max_row_tiles + 4 * NQ - 1) / (4 * NQ);
  const int b = blockIdx.x / groups, rg = blockIdx.x % groups;
  const int h = blockIdx.y;
  int m0, n_rows;
  request_rows(p, b, m0, n_rows);
  if (rg * 4 * NQ * 16 >= n_rows) return;  // the whole workgroup: nothing to score
  const int row0 = (rg * 4 + wave) * NQ * 16;
  const bool live = row0 < n_rows;  // a wave past the request's rows still copies and synchronises
  const int kvh = h / (p.H / p.H_kv);
  const float c = p.scale_log2e;

  vec16 qf[NQ][KS];
#pragma unroll
  for (int qt = 0; qt < NQ; ++qt) load_rows<D>(qf[qt], mask_query_row(p, m0, n_rows, row0 + 16 * qt + li, h), lg);
#pragma unroll
  for (int qt = 0; qt < NQ; ++qt)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) settle(qf[qt][ks]);

  // this lane's share of a tile copy: chunk slot `lane` of the 1 KiB piece (wave, j) holds which row and chunk?
  const char *k_base = p.k_cache + p.affix_slot0 * p.kv_slot_bytes + (int64_t)kvh * p.kv_head_bytes;
  int copy_row[G::kCopiesPerWave], copy_off[G::kCopiesPerWave];
#pragma unroll
  for (int j = 0; j < G::kCopiesPerWave; ++j) {
    const int slot = (wave * G::kCopiesPerWave + j) * 64 + lane;
    copy_row[j] = slot / G::kChunks;
    copy_off[j] = ((slot % G::kChunks) ^ (copy_row[j] & (G::kChunks - 1))) << 4;
  }
  auto issue = [&](int a0, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < G::kCopiesPerWave; ++j) {
      const int a = a0 + copy_row[j];
      lds_dma16(k_base + (int64_t)(a < p.A ? a : p.A - 1) * p.kv_slot_bytes + copy_off[j],
                tiles[buf] + (wave * G::kCopiesPerWave + j) * 1024);
    }
  };

  float m_run[NQ], l_run[NQ];
#pragma unroll
  for (int qt = 0; qt < NQ; ++qt) { m_run[qt] = -INFINITY; l_run[qt] = 0.0f; }
  issue(0, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int t0 = 0, it = 0; t0 < p.A; t0 += kStageKeys, ++it) {
    issue(t0 + kStageKeys, (it + 1) & 1);  // always: past the end the last key is re-read and ignored
    if (live) {
      const char *tile = tiles[it & 1];
#pragma unroll
     for (int half = 0; half < kStageKeys / (16 * NT); ++half) {
      const int a0 = t0 + 16 * NT * half;
      if (a0 >= p.A) break;  // wave-uniform
      const bool tail = a0 + 16 * NT > p.A;
      vec16 kf[NT][KS];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) load_rows_lds<D>(kf[nt], tile, NT * half + nt, li, lg);
#pragma unroll
      for (int qp = 0; qp < NQ; qp += 2) {
        f32x4 sc[2][NT];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) sc[u][nt] = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) sc[u][nt] = M::run(kf[nt][ks], qf[qp + u][ks], sc[u][nt]);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int qt = qp + u;
          if (tail) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (a0 + 16 * nt + 4 * lg + i >= p.A) sc[u][nt][i] = -INFINITY;
          }
          float mx = -INFINITY;
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sc[u][nt][i]);
          mx = fmaxf(mx, __shfl_xor(mx, 16));
          mx = fmaxf(mx, __shfl_xor(mx, 32));
          const float m_new = fmaxf(m_run[qt], mx * c);
          float add = 0.0f;
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) add += __builtin_amdgcn_exp2f(__builtin_fmaf(sc[u][nt][i], c, -m_new));
          l_run[qt] = l_run[qt] * __builtin_amdgcn_exp2f(m_run[qt] - m_new) + add;
          m_run[qt] = m_new;
        }
      }
     }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the next tile has landed ...
    __syncthreads();                                    // ... and everybody is done with this one
  }
  if (!live) return;
#pragma unroll
  for (int qt = 0; qt < NQ; ++qt) {
    float l = l_run[qt];
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    const int r = row0 + 16 * qt + li;
    if (lg == 0 && r < n_rows) {
      const int64_t src_row = p.mask_rows[m0 + r];
      const bool present = src_row >= 0 && src_row < p.total_q;
      p.stats[(int64_t)(m0 + r) * p.H + h] = present ? m_run[qt] + __builtin_amdgcn_logf(l) : INFINITY;
    }
  }
}

// One workgroup per (request, head, 256 affix keys): wave w keeps keys 64*w .. 64*w + 63 of the block in
// registers, the request's mask rows stream through LDS 32 at a time.  Same arithmetic as importance_colsum_kernel.
template <int DTYPE, int D>
__global__ __launch_bounds__(256) void importance_colsum_lds_kernel(ImportanceParams p) {
  constexpr int KS = D / 32, NR = kStageRows / 16;
  using M = Mma<DTYPE>;
  using G = StageGeometry<D, kStageRows>;
  __shared__ __attribute__((aligned(1024))) char tiles[2][G::kTileBytes];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int b = blockIdx.z;
  const int h = blockIdx.y;
  const int a0 = blockIdx.x * (4 * kKeysPerStep) + wave * kKeysPerStep;
  int m0, n_rows;
  request_rows(p, b, m0, n_rows);
  const bool live = a0 < p.A;  // a wave past the affix still copies and synchronises
  if (n_rows <= 0) {          // the whole workgroup: a request without mask rows has all-zero sums
    float *zero = p.partial + ((int64_t)b * p.H + h) * p.A;
    if (a0 + lane < p.A) zero[a0 + lane] = 0.0f;
    return;
  }
  const float c = p.scale_log2e;
  const int kvh = h / (p.H / p.H_kv);
  const char *k_base = p.k_cache + p.affix_slot0 * p.kv_slot_bytes + (int64_t)kvh * p.kv_head_bytes;

  vec16 kf[4][KS];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    const int a = a0 + 16 * nt + li;
    load_rows<D>(kf[nt], k_base + (int64_t)(a < p.A ? a : p.A - 1) * p.kv_slot_bytes, lg);
  }
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) settle(kf[nt][ks]);
  int copy_row[G::kCopiesPerWave], copy_off[G::kCopiesPerWave];
#pragma unroll
  for (int j = 0; j < G::kCopiesPerWave; ++j) {
    const int slot = (wave * G::kCopiesPerWave + j) * 64 + lane;
    copy_row[j] = slot / G::kChunks;
    copy_off[j] = ((slot % G::kChunks) ^ (copy_row[j] & (G::kChunks - 1))) << 4;
  }
  auto issue = [&](int r0, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < G::kCopiesPerWave; ++j)
      lds_dma16(mask_query_row(p, m0, n_rows, r0 + copy_row[j], h) + copy_off[j],
                tiles[buf] + (wave * G::kCopiesPerWave + j) * 1024);
  };
  auto statistic = [&](int r0, float (&st)[NR]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NR; ++t) {
      const int r = r0 + 16 * t + li;
      st[t] = p.stats[(int64_t)(m0 + (r < n_rows ? r : n_rows - 1)) * p.H + h];
    }
  };
  float col[4][4] = {};
  float st_cur[NR], st_next[NR];
  statistic(0, st_cur);
  issue(0, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int r0 = 0, it = 0; r0 < n_rows; r0 += kStageRows, ++it) {
    statistic(r0 + kStageRows, st_next);       // ordinary loads first, then the copies behind them
    issue(r0 + kStageRows, (it + 1) & 1);      // always: past the end the last row is re-read and ignored
    if (live) {
      const char *tile = tiles[it & 1];
#pragma unroll
      for (int t = 0; t < NR; ++t) {
        const float ref = r0 + 16 * t + li < n_rows ? st_cur[t] : INFINITY;  // 2^-inf = 0 for rows past the end
        vec16 qf[KS];
        load_rows_lds<D>(qf, tile, t, li, lg);
        f32x4 sc[4];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) sc[nt] = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int nt = 0; nt < 4; ++nt) sc[nt] = M::run(kf[nt][ks], qf[ks], sc[nt]);
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int i = 0; i < 4; ++i) col[nt][i] += __builtin_amdgcn_exp2f(__builtin_fmaf(sc[nt][i], c, -ref));
      }
    }
#pragma unroll
    for (int t = 0; t < NR; ++t) st_cur[t] = st_next[t];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the next tile has landed ...
    __syncthreads();                                    // ... and everybody is done with this one
  }
  if (!live) return;
  float *dst = p.partial + ((int64_t)b * p.H + h) * p.A;
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v = row_sum16(col[nt][i]);
      const int a = a0 + 16 * nt + 4 * lg + i;
      if (li == 0 && a < p.A) dst[a] = v;
    }
}

// ---------------------------------------------------------------------------------------------------
// Affixes of up to 1280 keys at head dims of 64 and 128: one pass over the scores.
//
// What bounds the two passes above is issue time per score (matrix product, multiply-add, exponential) and both
// spend it.  The column sums need every row's denominator first, so one pass has to keep a row's probabilities
// until the row is complete.  The register file of a CU can: the eight waves of a workgroup (two per SIMD, 256
// registers each) share a head's keys, each holds its 16 * NB of them as operands (NB * D / 8 registers) and the
// 4 * NB scores per lane of a 16-row query tile; the waves exchange (maximum, sum) per row through LDS, one barrier
// per tile, and add the normalised probabilities to per-lane column sums.  The keys are read once per workgroup,
// which takes the rows of several requests in turn (one workgroup per CU); the queries go straight from q to LDS by
// the copy engine while the item before is scored, and are counter-rotated there, so the packed copy in memory and
// its launch are gone too.  A wave with nine or ten key blocks keeps seven in registers and NBL of them, two or three, in
// LDS in fragment order, because operands, scores, column sums and the query fragment share the 256 registers.
//
// LLaDA heads, 256 rows a request, relocated, both launches of the call, two passes / this form: 16 requests with 300 /
// 600 / 1000 / 1100 / 1200 keys 68 / 90 / 120 / 134 / 139 -> 41 / 52 / 68 / 79 / 88 us; one request of 300 / 1000 keys
// 33 / 55 -> 13 / 20 us.  By the counters of the 1000-key launch a wave spends 512 matrix-pipe cycles and 325 vector
// instructions on a 16-row tile (rotation, stores and the keys' way into registers included), two waves per SIMD, the matrix
// pipe is busy 23 % of the time and 30 % of the wave cycles wait.  Sums of a
// whole chunk of up to 256 rows instead of 64 took 64 us at 1000 keys, but their order followed the batch.
// Measured and not taken: the two waves of a SIMD at different priorities (no change); scoring a wave's keys in two
// halves with references of their own, the first half's exponentials between the matrix instructions of the second
// (66.5 -> 68.5 us).
constexpr int kFusedWaves = 8;
constexpr int kFusedThreads = 64 * kFusedWaves;
// Query rows staged at a time: two buffers of them share the 160 KiB of LDS with the key blocks.
constexpr int fused_stage_rows(int head_dim, int lds_key_blocks) {
  return lds_key_blocks == 0 ? 256 : (lds_key_blocks == 2 || head_dim == 64 ? 128 : 64);
}
// Query rows of a request whose column sums are added up in registers before they are stored.  Rows are counted from the
// request's first one and the stored sums are added in order, so a request's importance does not depend on the batch it is
// scored in, whichever rows share a workgroup.
constexpr int kSumRows = 64;
// Sums 0 .. ceil(rows / kSumRows) - 1 of request b start at this one: a bound on what the requests in front of it need
// that every workgroup can compute, at most total_mask_rows / kSumRows + B sums in all.
__device__ __forceinline__ int first_sum(int m0, int b) { return m0 / kSumRows + b; }

// Column sums over the 16 lanes of a row, each lane left with the N / 16 sums N / 16 * (lane & 15) + j: every step adds one
// half of the values to the partner's and hands the other half over (partners differ in the step's bit and in all lower
// ones), 2.8 instructions a value instead of the five and a store of a few lanes that row_sum16 takes for each.
template <int HALF, int CTRL, int N>
__device__ __forceinline__ void spread_step(float (&v)[N], bool upper) {
#pragma unroll
  for (int j = 0; j < HALF; ++j) {
    const float keep = upper ? v[j + HALF] : v[j], give = upper ? v[j] : v[j + HALF];
    v[j] = keep + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, give), CTRL, 0xf, 0xf, true));
  }
}
template <int N>
__device__ __forceinline__ void spread_row_sums(float (&v)[N], int li) {
  static_assert(N % 16 == 0, "the halves stay whole");
  spread_step<N / 2, 0x140>(v, (li & 8) != 0);   // lane 15 - li of the row
  spread_step<N / 4, 0x141>(v, (li & 4) != 0);   // lane 7 - li of the half row
  spread_step<N / 8, 0x1b>(v, (li & 2) != 0);    // lane 3 - li of the quad
  spread_step<N / 16, 0xb1>(v, (li & 1) != 0);   // lane 1 - li of the pair
}

// Maximum / sum over the four lanes that share lane & 15 (the lane groups of one query column), in every lane.
template <class Op>
__device__ __forceinline__ float across_groups(float v, Op op) {
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  u32x2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = op(__uint_as_float(r.x), __uint_as_float(r.y));
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return op(__uint_as_float(r.x), __uint_as_float(r.y));
}

template <int DTYPE, int D, int NBR, int NBL>
__global__ __launch_bounds__(kFusedThreads) void importance_fused_kernel(ImportanceParams p, int chunk_rows, int chunks,
                                                                        int groups) {
  constexpr int NB = NBR + NBL, KS = D / 32;
  constexpr int TR = NB <= 5 ? 2 : 1;            // 16-row tiles per step: two where the registers allow
  constexpr bool AHEAD = NB <= 6;                // query fragments of the next step loaded during this one, likewise
  constexpr int STAGE_ROWS = fused_stage_rows(D, NBL);   // query rows staged at a time; chunk_rows is at most this
  static_assert(kSumRows % (16 * TR) == 0 && STAGE_ROWS % kSumRows == 0, "whole steps per sum, whole sums per item");
  constexpr int PAIRS = D / 16;                  // (d, d + D/2) chunk pairs per row
  constexpr int CHUNKS = D / 8;                  // 16-byte chunks per row
  constexpr int COPY_ROWS = 64 / CHUNKS;         // rows per wave copy
  constexpr int COPIES = STAGE_ROWS / COPY_ROWS / kFusedWaves;  // copies of a wave per item
  static_assert(COPIES * COPY_ROWS * kFusedWaves == STAGE_ROWS, "whole copies");
  using M = Mma<DTYPE>;
  using G = StageGeometry<D, 16>;
  __shared__ __attribute__((aligned(1024))) char q_stage[2][STAGE_ROWS * D * 2];
  __shared__ __attribute__((aligned(1024))) char k_rows[NBL ? kFusedWaves * NBL * KS * 1024 : 16];
  __shared__ __attribute__((aligned(16))) float row_max[2][16 * TR][kFusedWaves], row_sum[2][16 * TR][kFusedWaves];
  __shared__ float row_present[2][STAGE_ROWS];   // 1, or 0 for a row that is absent
  __shared__ __attribute__((aligned(16))) float rope[2][2 * D];  // cos and sin row of the request's shift

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const int h = blockIdx.x % p.H, group = blockIdx.x / p.H;
  const int kvh = h / (p.H / p.H_kv);
  // Keys dealt evenly: every wave's blocks are full except for the last one, whose absent rows start from -inf
  // (a masking step costs as much as the maximum, and the other waves would wait for the one that takes it).
  const int share = p.A / kFusedWaves, spare = p.A % kFusedWaves;
  const int a_wave = wave * share + (wave < spare ? wave : spare);
  const int n_keys = share + (wave < spare ? 1 : 0);   // 16 * (NB - 1) <= n_keys <= 16 * NB
  const float c = p.scale_log2e;

  // One item = (request, chunk of its mask rows).  Its rows go from q to LDS by the copy engine while the item before
  // is scored: indices first (fetch), the copies once those have arrived (issue), the rotation in LDS when the item's
  // turn has come.  Copy j of a wave covers COPY_ROWS rows; the swizzle is applied on the global side.
  struct Item { int m0, rows, shift, sum; };
  auto item_of = [&](int item) __attribute__((always_inline)) {
    Item it{0, 0, 0, 0};
    if (item < p.B * chunks) {
      const int b = item % p.B, first = item / p.B * chunk_rows;  // chunk by chunk: a request's last one is the short one
      request_rows(p, b, it.m0, it.rows);
      it.sum = first_sum(it.m0, b) + first / kSumRows;
      it.m0 += first;
      it.rows -= first;
      it.rows = it.rows > chunk_rows ? chunk_rows : (it.rows < 0 ? 0 : it.rows);
      it.shift = p.shifts ? p.shifts[b] : 0;
      if (it.shift < 0 || it.shift >= p.rope_rows) it.shift = 0;
    }
    return it;
  };
  int32_t src_row[COPIES];
  vec16 rope_part{{0, 0, 0, 0}};
  auto fetch = [&](const Item &it) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < COPIES; ++j) {
      const int r = (wave * COPIES + j) * COPY_ROWS + lane / CHUNKS;
      src_row[j] = r < it.rows ? p.mask_rows[it.m0 + r] : -1;
    }
    if (it.shift != 0 && tid < 2 * D / 4)
      rope_part = load16((tid < D / 4 ? p.cos_tab : p.sin_tab) + (int64_t)it.shift * D + (tid % (D / 4)) * 4);
  };
  auto issue = [&](const Item &it, int buf) __attribute__((always_inline)) {
    if (it.shift != 0 && tid < 2 * D / 4) store16(rope[buf] + tid * 4, rope_part);
#pragma unroll
    for (int j = 0; j < COPIES; ++j) {
      const int first = (wave * COPIES + j) * COPY_ROWS, r = first + lane / CHUNKS;
      const bool present = src_row[j] >= 0 && src_row[j] < p.total_q;
      const char *src = present ? p.q + src_row[j] * p.q_token_bytes + (int64_t)h * p.q_head_bytes +
                                      (((lane % CHUNKS) ^ (r & (CHUNKS - 1))) << 4)
                                : (const char *)kZeroRow + ((lane % CHUNKS) << 4);
      if (first < (it.rows + 16 * TR - 1) / (16 * TR) * (16 * TR)) {  // wave-uniform: rows that some tile reads
        lds_dma16(src, q_stage[buf] + first * D * 2);
        if (lane % CHUNKS == 0) row_present[buf][r] = present ? 1.0f : 0.0f;
      }
    }
  };
  Item next = item_of(group);
  fetch(next);

  // the wave's keys; past the affix they repeat the last one and their scores are masked
  const char *k_base = p.k_cache + p.affix_slot0 * p.kv_slot_bytes + (int64_t)kvh * p.kv_head_bytes;
  auto key_row = [&](int nt) __attribute__((always_inline)) {
    const int a = a_wave + 16 * nt + li;
    return k_base + (int64_t)(a < p.A ? a : p.A - 1) * p.kv_slot_bytes;
  };
  f32x4 absent;
#pragma unroll
  for (int i = 0; i < 4; ++i) absent[i] = 16 * (NB - 1) + 4 * lg + i < n_keys ? 0.0f : -INFINITY;
  vec16 kf[NBR][KS];
#pragma unroll
  for (int nt = 0; nt < NBR; ++nt) load_rows<D>(kf[nt], key_row(nt), lg);
  issue(next, 0);  // behind the key loads: the wait for the row indices does not hold those up
  char *const k_mine = k_rows + wave * NBL * KS * 1024 + lane * 16;
#pragma unroll
  for (int nt = 0; nt < NBL; ++nt) {
    vec16 f[KS];
    load_rows<D>(f, key_row(NBR + nt), lg);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) store16(k_mine + (nt * KS + ks) * 1024, f[ks]);
  }
#pragma unroll
  for (int nt = 0; nt < NBR; ++nt)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) settle(kf[nt][ks]);

  for (int item = group, turn = 0; item < p.B * chunks; item += groups, ++turn) {
    const int stage_buf = turn & 1;
    const Item now = next;
    next = item_of(item + groups);
    char *const q_rows = q_stage[stage_buf];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's copies of the item have landed ...
    __syncthreads();                                    // ... and everybody's; the other buffer is no longer read
    fetch(next);
    const int tiles = (now.rows + 16 * TR - 1) / (16 * TR) * TR;
    if (now.shift != 0) {
      const int ch = tid % PAIRS;
      float cs[16], sn[16];  // cos and sin of this thread's elements: first half of the row, second half
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        cs[j] = rope[stage_buf][ch * 8 + j];
        cs[8 + j] = rope[stage_buf][D / 2 + ch * 8 + j];
        sn[j] = rope[stage_buf][D + ch * 8 + j];
        sn[8 + j] = rope[stage_buf][D + D / 2 + ch * 8 + j];
      }
#pragma nounroll
      for (int r = tid / PAIRS; r < now.rows; r += kFusedThreads / PAIRS) {
        vec16 lo = load16(q_rows + G::offset(r, ch)), hi = load16(q_rows + G::offset(r, ch + PAIRS));
        rotate_pair_half_fast<DTYPE>(lo, hi, cs, sn, 0, 8, -1.0f);  // (188 -> 85 instructions a turn of this loop)
        store16(q_rows + G::offset(r, ch), lo);
        store16(q_rows + G::offset(r, ch + PAIRS), hi);
      }
      __syncthreads();
    }
    issue(next, stage_buf ^ 1);
    float *dst = p.partial + ((int64_t)now.sum * p.H + h) * p.A;

    vec16 qf[TR][KS];
    if (AHEAD) {
#pragma unroll
      for (int u = 0; u < TR; ++u) load_rows_lds<D>(qf[u], q_rows, u, li, lg);
    }
    for (int t0 = 0; t0 < tiles; t0 += kSumRows / 16) {
      const int t_stop = t0 + kSumRows / 16 < tiles ? t0 + kSumRows / 16 : tiles;
      float col[NB][4] = {};
      for (int t = t0; t < t_stop; t += TR) {
        const int buf = (t / TR) & 1;
        f32x4 sc[TR][NB];
        if (!AHEAD) {
#pragma unroll
          for (int u = 0; u < TR; ++u) load_rows_lds<D>(qf[u], q_rows, t + u, li, lg);
        }
#pragma unroll
        for (int u = 0; u < TR; ++u)
#pragma unroll
          for (int nt = 0; nt < NB; ++nt) sc[u][nt] = nt == NB - 1 ? absent : f32x4{0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int nt = 0; nt < NB; ++nt) {
            const vec16 k = nt < NBR ? kf[nt < NBR ? nt : 0][ks] : load16(k_mine + ((nt - NBR) * KS + ks) * 1024);
#pragma unroll
            for (int u = 0; u < TR; ++u) sc[u][nt] = M::run(k, qf[u][ks], sc[u][nt]);
          }
        if (AHEAD) {  // the next tiles' rows (past the last: rows that exist in LDS, never used)
#pragma unroll
          for (int u = 0; u < TR; ++u) load_rows_lds<D>(qf[u], q_rows, (t + TR + u) % (STAGE_ROWS / 16), li, lg);
        }
        float ref[TR];  // this wave's maximum per row; a wave without keys has -inf and probabilities of 0
#pragma unroll
        for (int u = 0; u < TR; ++u) {
          float mx = -INFINITY;
#pragma unroll
          for (int nt = 0; nt < NB; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sc[u][nt][i]);
          mx = across_groups(mx, [](float x, float y) { return fmaxf(x, y); }) * c;
          ref[u] = mx;
          mx = mx == -INFINITY ? 0.0f : mx;
          float add[4] = {};
#pragma unroll
          for (int nt = 0; nt < NB; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              sc[u][nt][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[u][nt][i], c, -mx));
              add[i] += sc[u][nt][i];
            }
          const float sum = across_groups((add[0] + add[1]) + (add[2] + add[3]), [](float x, float y) { return x + y; });
          if (lg == 0) { row_max[buf][16 * u + li][wave] = ref[u]; row_sum[buf][16 * u + li][wave] = sum; }
        }
        __syncthreads();  // the other buffer is free: everybody has read it before arriving here
        // lane group lg merges waves 2 lg and 2 lg + 1, the groups meet in registers
#pragma unroll
        for (int u = 0; u < TR; ++u) {
          const float2 m2 = *(const float2 *)&row_max[buf][16 * u + li][2 * lg];
          const float2 s2 = *(const float2 *)&row_sum[buf][16 * u + li][2 * lg];
          const float m = across_groups(fmaxf(m2.x, m2.y), [](float x, float y) { return fmaxf(x, y); });
          const float total = across_groups(s2.x * __builtin_amdgcn_exp2f(m2.x - m) + s2.y * __builtin_amdgcn_exp2f(m2.y - m),
                                            [](float x, float y) { return x + y; });
          float f = __builtin_amdgcn_exp2f(ref[u] - m) * __builtin_amdgcn_rcpf(total);
          // An absent row is a zero query: against an infinite key its scores are not numbers, and a factor of 0 would not
          // keep them out.
          const bool present = row_present[stage_buf][16 * (t + u) + li] != 0.0f;
          if (__builtin_amdgcn_ballot_w64(!present) != 0) {
            f = present ? f : 0.0f;
#pragma unroll
            for (int nt = 0; nt < NB; ++nt)
#pragma unroll
              for (int i = 0; i < 4; ++i) sc[u][nt][i] = present ? sc[u][nt][i] : 0.0f;
          }
#pragma unroll
          for (int nt = 0; nt < NB; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) col[nt][i] = __builtin_fmaf(sc[u][nt][i], f, col[nt][i]);
        }
      }
      constexpr int OWN = (NB + 3) / 4;  // sums a lane stores: key 16 * (n / 4) + 4 * lg + n % 4 for n = OWN * li + j
      float sums[16 * OWN];
#pragma unroll
      for (int n = 0; n < 16 * OWN; ++n) sums[n] = n < 4 * NB ? col[n < 4 * NB ? n / 4 : 0][n % 4] : 0.0f;
      int own = lane;  // opaque: what follows is computed here, not kept in registers across the tiles
      asm volatile("" : "+v"(own));
      spread_row_sums(sums, own & 15);
#pragma unroll
      for (int j = 0; j < OWN; ++j) {
        const int n = OWN * (own & 15) + j, a = 16 * (n / 4) + 4 * (own >> 4) + n % 4;
        if (a < n_keys) dst[a_wave + a] = sums[j];
      }
      dst += (int64_t)p.H * p.A;
    }
  }
}

// importance[b, a] += sum over the row sums of request b and the heads of partial[sum, h, a], in a fixed order: PARTS
// lanes take every PARTS-th partial row each (their loads all in flight together), then the shares are added in lane
// order.  ROW_SUMS: one sum per kSumRows rows (the one-pass form), otherwise one per request.  The chain of a lane's loads
// is what the launch takes: sixteen lanes in the one-pass form (four: 0.5 to 1 us more a call for one or two requests).
template <int PARTS, bool ROW_SUMS>
__global__ __launch_bounds__(64 * PARTS) void importance_reduce_kernel(ImportanceParams p) {
  __shared__ float share[PARTS][64];
  const int a = blockIdx.x * 64 + (threadIdx.x & 63);
  const int part = threadIdx.x >> 6;
  const int b = blockIdx.y;
  float acc = 0.0f;
  int first = b, sums = 1;
  if (ROW_SUMS) {
    int m0, n_rows;
    request_rows(p, b, m0, n_rows);
    first = first_sum(m0, b);
    sums = (n_rows + kSumRows - 1) / kSumRows;
  }
  const int rows = sums * p.H;
  if (a < p.A) {
    const float *src = p.partial + (int64_t)first * p.H * p.A + a;
#pragma unroll 8
    for (int r = part; r < rows; r += PARTS) acc += src[(int64_t)r * p.A];
  }
  share[part][threadIdx.x & 63] = acc;
  __syncthreads();
  if (part == 0 && a < p.A) {
    float *dst = p.importance + (int64_t)b * p.imp_stride + a;
    float total = share[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < PARTS; ++w) total += share[w][threadIdx.x];
    *dst += total;
  }
}

}  // namespace acache

using namespace acache;

static int64_t stats_bytes(int64_t total_mask_rows, int32_t H) {
  return (total_mask_rows * H * (int64_t)sizeof(float) + 15) / 16 * 16;
}

static int64_t partial_bytes(int32_t B, int32_t H, int32_t affix_len) {
  return ((int64_t)B * H * affix_len * (int64_t)sizeof(float) + 15) / 16 * 16;
}

extern "C" int64_t acache_affix_importance_workspace_bytes(int64_t total_mask_rows, int32_t B, int32_t H,
                                                           int32_t H_kv, int32_t D, int32_t affix_len,
                                                           int32_t relocated) {
  if (total_mask_rows < 0 || B < 0 || H < 0 || H_kv < 0 || D < 0 || affix_len < 0) return 0;
  (void)H_kv;
  (void)relocated;  // the two-pass form makes its packed copy of the mask queries (2-byte elements) either way
  // (one size for both forms: the one-pass form's partial sums take less than this)
  return stats_bytes(total_mask_rows, H) + partial_bytes(B, H, affix_len) + total_mask_rows * H * D * 2;
}

// Launches of the one-pass form, or kNotFused when the shape is not one of its shapes.
constexpr int kNotFused = -1000;
constexpr int kFusedWorkgroups = 256;  // one per CU: eight waves of 256 registers fill it

static int launch_fused(ImportanceParams p, int32_t dtype, int32_t D, dim3 reduce_grid, hipStream_t s) {
  if ((D != 128 && D != 64) || p.A > 1280) return kNotFused;
  // Work items are (request, chunk of its mask rows); `groups` workgroups per head take them in turn.  The chunk is
  // the multiple of the rows per sum with the shortest busiest workgroup, an item's own cost (staging, partial sums)
  // being worth about 16 rows.
  int groups = kFusedWorkgroups / p.H;
  groups = groups < 1 ? 1 : groups;
  const int blocks = ((p.A + kFusedWaves - 1) / kFusedWaves + 15) / 16;  // 16-key blocks of the waves with most keys
  const int stage_rows = fused_stage_rows(D, blocks > 8 ? blocks - 7 : 0);
  // The partial sums (total_mask_rows / kSumRows + B of them at most, per head) fit what the other form takes for its
  // statistics, partial sums and packed queries: a row's share of a sum is no more than its statistic and query.
  static_assert(1280 * 4 / kSumRows <= 4 + 2 * 64, "partial sums fit the workspace");
  int chunk_rows = 0, chunks = 0;
  int64_t best = INT64_MAX;
  for (int rows = kSumRows; rows <= stage_rows; rows += kSumRows) {
    const int64_t n = (p.max_mask_rows + (int64_t)rows - 1) / rows;
    const int64_t used = (p.max_mask_rows + 16 * n - 1) / (16 * n) * 16;  // on average: a request's last chunk is shorter
    const int64_t span = (n * p.B + groups - 1) / groups * (used + 16);
    if (span < best) { best = span; chunk_rows = rows; chunks = (int)n; }
  }
  if ((int64_t)chunks * p.B > 0x7fffffffLL / 2) return kNotFused;
  if ((int64_t)groups > (int64_t)chunks * p.B) groups = chunks * p.B;
  p.partial = (float *)p.stats;  // the whole workspace: this form needs neither row statistics nor packed queries
  const dim3 grid((unsigned)(p.H * groups));
#define ACACHE_FUSED(DT, HD, NBR, NBL)                                                                        \
  if (dtype == DT && D == HD && blocks == NBR + NBL) {                                                       \
    hipLaunchKernelGGL((importance_fused_kernel<DT, HD, NBR, NBL>), grid, dim3(kFusedThreads), 0, s, p, chunk_rows, chunks, groups); \
    const int rc = launch_status("importance_fused_kernel");                                                  \
    if (rc) return rc;                                                                                        \
    hipLaunchKernelGGL((importance_reduce_kernel<16, true>), reduce_grid, dim3(1024), 0, s, p);               \
    return launch_status("importance_reduce_kernel");                                                         \
  }
#define ACACHE_FUSED_SIZES(DT, HD) \
  ACACHE_FUSED(DT, HD, 1, 0) ACACHE_FUSED(DT, HD, 2, 0) ACACHE_FUSED(DT, HD, 3, 0) ACACHE_FUSED(DT, HD, 4, 0) \
  ACACHE_FUSED(DT, HD, 5, 0) ACACHE_FUSED(DT, HD, 6, 0) ACACHE_FUSED(DT, HD, 7, 0) ACACHE_FUSED(DT, HD, 8, 0) \
  ACACHE_FUSED(DT, HD, 7, 2) ACACHE_FUSED(DT, HD, 7, 3)
  ACACHE_FUSED_SIZES(ACACHE_BF16, 128)
  ACACHE_FUSED_SIZES(ACACHE_BF16, 64)
  ACACHE_FUSED_SIZES(ACACHE_F16, 128)
  ACACHE_FUSED_SIZES(ACACHE_F16, 64)
#undef ACACHE_FUSED_SIZES
#undef ACACHE_FUSED
  return kNotFused;
}

// Argument checks and the launches; `workspace` is caller memory or this library's file-scope scratch.
static int importance_launch(
    float *importance, const void *q, const void *k_cache, const int32_t *mask_rows, const int32_t *cu_mask,
    const int32_t *affix_shifts, const float *rope_cos, const float *rope_sin, int32_t rope_rows, float scale,
    int32_t affix_len, int64_t affix_slot0, int32_t B, int64_t total_q, int64_t total_mask_rows, int32_t max_mask_rows,
    int32_t H,
    int32_t H_kv, int32_t D, int32_t dtype, int64_t num_slots, int64_t importance_stride, int64_t q_token_stride,
    int64_t q_head_stride, int64_t kv_slot_stride, int64_t kv_head_stride, void *workspace, int64_t workspace_bytes,
    void *stream) {
  if (dtype != ACACHE_BF16 && dtype != ACACHE_F16)
    return fail(ACACHE_E_DTYPE, "affix_importance: dtype %d not supported (bf16 or f16)", dtype);
  if (D < 16 || D > 256 || D % 16 != 0)
    return fail(ACACHE_E_SHAPE, "affix_importance: head_dim %d not supported (a multiple of 16 up to 256)", D);
  if (B < 0 || affix_len < 0 || total_mask_rows < 0 || max_mask_rows < 0 || H <= 0 || H_kv <= 0 || H % H_kv)
    return fail(ACACHE_E_SHAPE, "affix_importance: bad sizes (B %d, A %d, H %d, H_kv %d)", B, affix_len, H, H_kv);
  if (B == 0 || affix_len == 0 || total_mask_rows == 0 || max_mask_rows == 0) return 0;
  if (total_q <= 0) return fail(ACACHE_E_SHAPE, "affix_importance: %lld mask rows but q has %lld rows",
                                (long long)total_mask_rows, (long long)total_q);
  if (!importance || !q || !k_cache || !mask_rows || !cu_mask || !workspace)
    return fail(ACACHE_E_NULL, "affix_importance: NULL pointer");
  if (affix_shifts && (!rope_cos || !rope_sin || rope_rows <= 0))
    return fail(ACACHE_E_MODE, "affix_importance: shifts given without RoPE tables");
  if (!(scale > 0.0f)) return fail(ACACHE_E_RANGE, "affix_importance: scale must be positive");
  if (affix_slot0 < 0 || affix_slot0 + affix_len > num_slots)
    return fail(ACACHE_E_RANGE, "affix_importance: affix slots [%lld, %lld) outside %lld slots", (long long)affix_slot0,
                (long long)(affix_slot0 + affix_len), (long long)num_slots);
  if (importance_stride < affix_len) return fail(ACACHE_E_SHAPE, "affix_importance: importance stride < affix_len");
  if (total_mask_rows * H * D * 2 >= ((int64_t)1 << 32))
    return fail(ACACHE_E_SHAPE, "affix_importance: %lld mask rows x %d heads x %d: the packed query copy must stay under 4 GiB",
                (long long)total_mask_rows, H, D);
  if (workspace_bytes < acache_affix_importance_workspace_bytes(total_mask_rows, B, H, H_kv, D, affix_len, affix_shifts != nullptr))
    return fail(ACACHE_E_SHAPE, "affix_importance: workspace of %lld bytes, %lld needed", (long long)workspace_bytes,
                (long long)acache_affix_importance_workspace_bytes(total_mask_rows, B, H, H_kv, D, affix_len, affix_shifts != nullptr));
  if (!aligned16(q) || !aligned16(k_cache) || !aligned16(workspace) || (rope_cos && !aligned16(rope_cos)) ||
      (rope_sin && !aligned16(rope_sin)) || (q_token_stride * 2) % 16 || (q_head_stride * 2) % 16 ||
      (kv_slot_stride * 2) % 16 || (kv_head_stride * 2) % 16)
    return fail(ACACHE_E_ALIGN, "affix_importance: pointers and strides must be 16-byte aligned");
  ImportanceParams p;
  p.importance = importance; p.q = (const char *)q; p.k_cache = (const char *)k_cache;
  p.mask_rows = mask_rows; p.cu_mask = cu_mask; p.shifts = affix_shifts;
  p.cos_tab = rope_cos; p.sin_tab = rope_sin; p.stats = (float *)workspace;
  p.partial = (float *)((char *)workspace + stats_bytes(total_mask_rows, H));
  p.q_rot = (char *)workspace + stats_bytes(total_mask_rows, H) + partial_bytes(B, H, affix_len);
  p.total_q = total_q;
  p.imp_stride = importance_stride;
  p.q_token_bytes = q_token_stride * 2; p.q_head_bytes = q_head_stride * 2;
  p.kv_slot_bytes = kv_slot_stride * 2; p.kv_head_bytes = kv_head_stride * 2;
  p.affix_slot0 = affix_slot0;
  p.scale_log2e = scale * 1.4426950408889634f;
  p.A = affix_len; p.B = B; p.H = H; p.H_kv = H_kv; p.rope_rows = rope_rows; p.D = D;
  p.max_row_tiles = (max_mask_rows + 15) / 16;
  p.total_mask_rows = (int32_t)total_mask_rows;
  p.max_mask_rows = max_mask_rows;
  hipStream_t s = (hipStream_t)stream;
  const int lanes_per_row = D * 2 / 32;
  const dim3 grid0((unsigned)(((int64_t)max_mask_rows * H * lanes_per_row + 255) / 256), (unsigned)B);
  const int row_groups = (p.max_row_tiles + kRowTilesPerWave - 1) / kRowTilesPerWave;
  const dim3 grid1((unsigned)((int64_t)B * row_groups), (unsigned)((H + 3) / 4));
  const dim3 grid2((unsigned)((affix_len + kKeysPerStep - 1) / kKeysPerStep), (unsigned)((H + 3) / 4), (unsigned)B);
  const dim3 grid3((unsigned)((affix_len + 63) / 64), (unsigned)B);
  // the LDS-staged pair: a workgroup per (request, head, 256 mask rows) and per (request, head, 256 affix keys)
  const int row_groups_staged = (p.max_row_tiles + 4 * kRowTilesPerWave - 1) / (4 * kRowTilesPerWave);
  const dim3 grid1s((unsigned)((int64_t)B * row_groups_staged), (unsigned)H);
  const dim3 grid2s((unsigned)((affix_len + 4 * kKeysPerStep - 1) / (4 * kKeysPerStep)), (unsigned)H, (unsigned)B);
  // One pass where a head's keys fit the registers (and LDS) of one workgroup.
  const int fused_rc = launch_fused(p, dtype, D, grid3, s);
  if (fused_rc != kNotFused) return fused_rc;
#define ACACHE_CASE(DT, HD)                                                                       \
  if (dtype == DT && D == HD) {                                                                   \
    hipLaunchKernelGGL((importance_rotate_kernel<DT>), grid0, dim3(256), 0, s, p);                \
    const int rc0 = launch_status("importance_rotate_kernel");                                    \
    if (rc0) return rc0;                                                                          \
    if constexpr (HD == 64 || HD == 128 || HD == 256) {                                           \
      hipLaunchKernelGGL((importance_stats_lds_kernel<DT, HD>), grid1s, dim3(256), 0, s, p);      \
      const int rc = launch_status("importance_stats_lds_kernel");                                \
      if (rc) return rc;                                                                          \
      hipLaunchKernelGGL((importance_colsum_lds_kernel<DT, HD>), grid2s, dim3(256), 0, s, p);     \
      const int rc2 = launch_status("importance_colsum_lds_kernel");                              \
      if (rc2) return rc2;                                                                        \
    } else {                                                                                      \
      hipLaunchKernelGGL((importance_stats_kernel<DT, HD>), grid1, dim3(256), 0, s, p);           \
      const int rc = launch_status("importance_stats_kernel");                                    \
      if (rc) return rc;                                                                          \
      hipLaunchKernelGGL((importance_colsum_kernel<DT, HD>), grid2, dim3(256), 0, s, p);          \
      const int rc2 = launch_status("importance_colsum_kernel");                                  \
      if (rc2) return rc2;                                                                        \
    }                                                                                             \
    hipLaunchKernelGGL((importance_reduce_kernel<4, false>), grid3, dim3(256), 0, s, p);          \
    return launch_status("importance_reduce_kernel");                                             \
  }
#define ACACHE_DIMS(DT)                                                                             \
  ACACHE_CASE(DT, 128) ACACHE_CASE(DT, 64) ACACHE_CASE(DT, 16) ACACHE_CASE(DT, 32) ACACHE_CASE(DT, 48)   \
  ACACHE_CASE(DT, 80) ACACHE_CASE(DT, 96) ACACHE_CASE(DT, 112) ACACHE_CASE(DT, 144) ACACHE_CASE(DT, 160) \
  ACACHE_CASE(DT, 176) ACACHE_CASE(DT, 192) ACACHE_CASE(DT, 208) ACACHE_CASE(DT, 224) ACACHE_CASE(DT, 240) \
  ACACHE_CASE(DT, 256)
  ACACHE_DIMS(ACACHE_BF16)
  ACACHE_DIMS(ACACHE_F16)
#undef ACACHE_DIMS
#undef ACACHE_CASE
  return fail(ACACHE_E_SHAPE, "affix_importance: unsupported dtype / head_dim");
}

extern "C" int acache_affix_importance(
    float *importance, const void *q, const void *k_cache, const int32_t *mask_rows, const int32_t *cu_mask,
    const int32_t *affix_shifts, const float *rope_cos, const float *rope_sin, int32_t rope_rows, float scale,
    int32_t affix_len, int64_t affix_slot0, int32_t B, int64_t total_q, int64_t total_mask_rows, int32_t max_mask_rows,
    int32_t H,
    int32_t H_kv, int32_t D, int32_t dtype, int64_t num_slots, int64_t importance_stride, int64_t q_token_stride,
    int64_t q_head_stride, int64_t kv_slot_stride, int64_t kv_head_stride, void *workspace, int64_t workspace_bytes,
    void *stream) {
  return importance_launch(importance, q, k_cache, mask_rows, cu_mask, affix_shifts, rope_cos, rope_sin, rope_rows, scale,
                           affix_len, affix_slot0, B, total_q, total_mask_rows, max_mask_rows, H, H_kv, D, dtype, num_slots,
                           importance_stride, q_token_stride, q_head_stride, kv_slot_stride, kv_head_stride, workspace,
                           workspace_bytes, stream);
}

// ---------------------------------------------------------------------------------------------------
// The same call for callers that cannot allocate device memory (code under HIP graph capture, serving
// loops, harnesses that forbid hipMalloc): the row statistics, per-head partial sums and counter-rotated queries
// live in a file-scope device array instead of a caller workspace.  Every GPU the library runs on holds
// its own copy of the array at its own address until the process ends; the address is looked up once per
// device and only that pointer is ever handed to kernels.  Nothing in the array has to start at zero:
// every word a launch reads was written by an earlier launch of the same call.
static __device__ __align__(256) unsigned char scratch[ACACHE_IMPORTANCE_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices] = {};

int scratch_of_current_device(void **out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail((int)e, "affix_importance_noalloc: hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices)
    return fail(ACACHE_E_RANGE, "affix_importance_noalloc: device %d outside the %d devices supported", dev, kMaxDevices);
  std::lock_guard<std::mutex> guard(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void *ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return fail(e != hipSuccess ? (int)e : ACACHE_E_NULL, "affix_importance_noalloc: hipGetSymbolAddress: %s",
                  hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}
}  // namespace

extern "C" int64_t acache_affix_importance_noalloc_max_bytes(void) { return ACACHE_IMPORTANCE_SCRATCH_BYTES; }

extern "C" int acache_affix_importance_noalloc(
    float *importance, const void *q, const void *k_cache, const int32_t *mask_rows, const int32_t *cu_mask,
    const int32_t *affix_shifts, const float *rope_cos, const float *rope_sin, int32_t rope_rows, float scale,
    int32_t affix_len, int64_t affix_slot0, int32_t B, int64_t total_q, int64_t total_mask_rows, int32_t max_mask_rows,
    int32_t H,
    int32_t H_kv, int32_t D, int32_t dtype, int64_t num_slots, int64_t importance_stride, int64_t q_token_stride,
    int64_t q_head_stride, int64_t kv_slot_stride, int64_t kv_head_stride, void *stream) {
  const int64_t need =
      acache_affix_importance_workspace_bytes(total_mask_rows, B, H, H_kv, D, affix_len, affix_shifts != nullptr);
  if (need > (int64_t)ACACHE_IMPORTANCE_SCRATCH_BYTES)
    return fail(ACACHE_E_SHAPE,
                "affix_importance_noalloc: this call needs %lld bytes of scratch, the built-in buffer holds %lld; "
                "use acache_affix_importance with a caller workspace",
                (long long)need, (long long)ACACHE_IMPORTANCE_SCRATCH_BYTES);
  void *ws = nullptr;
  const int rc = scratch_of_current_device(&ws);
  if (rc) return rc;
  return importance_launch(importance, q, k_cache, mask_rows, cu_mask, affix_shifts, rope_cos, rope_sin, rope_rows, scale,
                           affix_len, affix_slot0, B, total_q, total_mask_rows, max_mask_rows, H, H_kv, D, dtype, num_slots,
                           importance_stride, q_token_stride, q_head_stride, kv_slot_stride, kv_head_stride, ws,
                           ACACHE_IMPORTANCE_SCRATCH_BYTES, stream);
}
