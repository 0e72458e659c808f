// Varlen attention for batches of short query blocks (refinement steps: the 32 tokens of a generation block against
// a thousand cached keys), head dims 64 and 128, all three relocation modes and block tables.
//
// What bounds it: 32 query rows are so little matrix work per key that a workgroup whose waves share every key tile
// spends its time in the chain copy -> barrier -> LDS read -> scores -> softmax -> LDS read -> output, one tile after
// the other (about 0.9 us per 64 keys, nearly all of it latency).  So the waves do not share tiles: a unit is the 32
// query rows of one (request, head), every wave holds all of them and walks its own 32-key chunks (wave w takes chunks
// w, w + NW, ...) through its own two LDS buffers.  There is no barrier until the waves' partial results are merged at
// the end, the chains of the waves overlap, and each key is read from LDS once for all 32 rows.  A buffer is free as
// soon as its fragments are in registers, so the next chunk's keys are on their way while this one's scores are
// computed, and likewise the values.
//
// The copies are waited for by count (s_waitcnt vmcnt(n), they retire in order), so no other vector load may run in
// the loop: the slots of a wave's next sixteen chunks stay in registers.  (A ring of nine half tiles shared by four
// waves, one barrier per half: 25 us for one request.  Four such waves and two workgroups per CU, for more units than
// CUs: 16 LLaDA requests 51 us, against 48 of the two-deep ring in attn.hip.)
//
// The set-up is three dependent round trips (lengths; slots, queries, table rows; keys), as in attn_group.hip: the queries
// go through LDS once per unit and are relocated there once.  With every wave reading the 32 rows for itself behind a
// lookup of one request at a time it was 5.0 us of one request's 14.9.
//
// Measured (bf16, D = 128, 32 query rows and about 1 300 keys per request, three quarters of them shared in the relocation
// modes, microseconds per call, varlen_attn_unit_kernel / this kernel with a set-up per wave / whole units / now, in parts
// where units are few):
//   32 / 32 heads, plain 1 request 18.4 / 16.3 / 14.7 / 12.2, 4: 22.6 / 23.0 / 20.2 / 20.1; query side 1: 23.6 / 19.0 / 15.5 /
//   13.0, 4: 30.8 / 23.6 / 19.3 / 15.8, 8: 33.5 / 26.1 / 21.1 / 20.6; key side 1: 29.4 / 24.5 / 21.1 / 18.7.  28 / 4 heads,
//   plain 1: 18.6 / 16.7 / 14.9 / 12.5, 8: 19.5 / 19.5 / 16.9 / 16.6; query side 8: 25.6 / 22.1 / 17.7 / 17.1; key side 8: 31.1 /
//   28.8 / 23.6 / 23.6.  In whole units one request of 32 heads and 1 150 keys is 32 CUs with 590 KB of keys and values each,
//   which take 5.4 us by copies alone (110 GB/s into one CU); in four parts 128 CUs with 370 KB each.
#include "attn_common.h"

namespace acache {

static constexpr int NW = 8;  // waves per unit

template <int N> __device__ __forceinline__ void wait_copies() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// this wave's LDS reads have returned: their buffer may be filled again
__device__ __forceinline__ void wait_lds_reads() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// One unit: 32 query rows (query tile `tile_in_request` of request b) of one head, or its part `part` of FS: all scores, and
// D / FS features of the values and of the output.
template <int DTYPE, int D, int MODE, int FS>
__device__ __forceinline__ void short_attn_unit(const AttnParams &p, char *lds, char *lds_q, float *stats, float *lds_rope,
                                                int kvh, int head, int part, const ShortUnit &u) {
  constexpr int QROWS = 32, NQ16 = 2;         // query rows of a unit
  constexpr int BN = 32;                      // keys per chunk
  constexpr int KS = D / 32, DT = D / FS / 16;
  constexpr int ROW_BYTES = D * 2;
  constexpr int CH = ROW_BYTES / 16;          // 16-byte pieces per row
  constexpr int RW = 256 / ROW_BYTES;         // rows per 256-byte bank window
  constexpr int RPI = 64 / CH;                // rows per copy instruction
  constexpr int NI = BN / RPI;                // copy instructions per chunk and tensor
  constexpr int BUF_BYTES = BN * ROW_BYTES;
  // the same of this part's values: D / FS features of a row
  constexpr int V_ROW_BYTES = ROW_BYTES / FS, V_CH = CH / FS, V_RW = 256 / V_ROW_BYTES, V_RPI = 64 / V_CH, V_NI = BN / V_RPI;
  static_assert(V_NI >= 1 && V_CH >= 4, "whole copy instructions");
  constexpr int WAVE_BYTES = BUF_BYTES + BN * V_ROW_BYTES;  // a wave's K buffer, then its V buffer
  using M = Mma<DTYPE>;
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

  const int tid = opaque_tid(), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const int kv_begin = u.kv_begin, kv_len = u.kv_len, shared_len = u.shared_len, shift = u.shift;
  const int q_row0 = u.q_begin + u.tile * QROWS;
  const int rows = u.q_len - u.tile * QROWS < QROWS ? u.q_len - u.tile * QROWS : QROWS;
  char *const out_base = p.out + (int64_t)q_row0 * p.o_token_bytes + (int64_t)head * p.o_head_bytes + part * V_ROW_BYTES;

  if (kv_len <= 0) {  // no keys: defined output (zeros)
    for (int r = tid / V_CH; r < rows; r += 64 * NW / V_CH)
      store16(out_base + (int64_t)r * p.o_token_bytes + (tid % V_CH) * 16, vec16{{0, 0, 0, 0}});
    return;
  }

  // chunks: the shared range first (query-side mode), then the rest
  const int chunks_a = (shared_len + BN - 1) / BN;
  const int n_chunks = chunks_a + (kv_len - shared_len + BN - 1) / BN;

  // ---- copies -------------------------------------------------------------------------------------------------
  // Lane l of slots[j] holds the slot of row l % 32 of the wave's chunk 2 j + l / 32, counted from the last refill.
  constexpr int SLOT_REGS = 8;
  int slots[SLOT_REGS];
  auto load_slots = [&](int turn) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < SLOT_REGS; ++j) {
      const TileRange r = tile_range_of(wave + (turn + 2 * j + (lane >> 5)) * NW, chunks_a, shared_len, kv_len, BN);
      if (MODE == MODE_PAGED) {               // one table entry for the chunk; take_slots makes the slots of it
        slots[j] = r.n0 < r.n_end ? table_entry(p, u.b, r.n0) : -1;
        continue;
      }
      const int n = r.n0 + (lane & 31);
      const int s = p.slot_map[kv_begin + (n < kv_len ? n : kv_len - 1)];
      slots[j] = n < r.n_end ? s : -1;
    }
  };
  auto settle_slots = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < SLOT_REGS; ++j) asm volatile("" ::"v"(slots[j]));
  };
  const int dma_row = lane / CH, dma_piece = lane % CH;
  const char *const kc_base = uniform_ptr(p.k_cache + (int64_t)kvh * p.kv_head_bytes);
  const char *const vc_base = uniform_ptr(p.v_cache + (int64_t)kvh * p.kv_head_bytes + part * V_ROW_BYTES);
  // byte offset of this lane's (swizzled) piece inside its row of copy i: the layouts of attn_dma_part
  auto k_piece = [&](int i) __attribute__((always_inline)) {
    return (uint32_t)((dma_piece ^ (((i * RPI + dma_row) / RW) % CH)) << 4);
  };
  const int v_dma_row = lane / V_CH, v_dma_piece = lane % V_CH;
  auto v_piece = [&](int i) __attribute__((always_inline)) {
    return (uint32_t)((v_dma_piece ^ (2 * (((i * V_RPI + v_dma_row) / V_RW) % (V_CH / 2)))) << 4);
  };
  const uint32_t slot_limit = p.num_slots > 0x7fffffffLL ? 0x7fffffffu : (uint32_t)p.num_slots;
  const uint32_t slot_pitch = (uint32_t)p.kv_slot_bytes;
  const uint32_t k_dst = __builtin_amdgcn_readfirstlane(lds_offset_of(lds) + (uint32_t)(wave * WAVE_BYTES));
  int slot[NI], v_slot[V_NI];                 // this lane's slots in the chunk being copied; -1: absent
  bool all_present = false;
  int rot_slot = -1;                          // key-side mode: slot of row lane / 2 of that chunk
  auto take_slots = [&](int turn) __attribute__((always_inline)) {
    if (turn % (2 * SLOT_REGS) == 0) {
      if (turn > 0) load_slots(turn);
      settle_slots();
    } else if (turn % 2 == 0) {
#pragma unroll
      for (int j = 0; j + 1 < SLOT_REGS; ++j) slots[j] = slots[j + 1];
    }
    bool ok = true;
    auto slot_of_row = [&](int row) __attribute__((always_inline)) {
      int s = __shfl(slots[0], (turn % 2) * 32 + row);
      if (MODE == MODE_PAGED) {
        const int n = (wave + turn * NW) * BN + row;
        s = n < kv_len ? slot_of_entry(p, s, n) : -1;
      }
      return s;
    };
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      slot[i] = slot_of_row(i * RPI + dma_row);
      ok &= (uint32_t)slot[i] < slot_limit;
    }
#pragma unroll
    for (int i = 0; i < V_NI; ++i) v_slot[i] = FS == 1 ? slot[FS == 1 ? i : 0] : slot_of_row(i * V_RPI + v_dma_row);
    if (MODE == MODE_KEY_SIDE) rot_slot = __shfl(slots[0], (turn % 2) * 32 + lane / 2);
    all_present = p.small_cache && __builtin_amdgcn_ballot_w64(!ok) == 0;
  };
  auto copy_rows = [&]<int N>(const char *base, const int (&rows_slot)[N], int first, auto piece,
                              uint32_t dst) __attribute__((always_inline)) {
    if (all_present) {  // wave-uniform base + 32-bit offsets
#pragma unroll
      for (int i = 0; i < N; ++i)
        lds_dma16_off(base, __umul24((uint32_t)rows_slot[i], slot_pitch) + piece(i), dst + i * 1024);
    } else {            // absent rows come from the zero row
      const char *zero = reinterpret_cast<const char *>(kZeroRow) + (first << 4);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const char *src = base + ((uint64_t)(uint32_t)rows_slot[i] * slot_pitch + piece(i));
        lds_dma16_at((uint32_t)rows_slot[i] < slot_limit ? src : zero, dst + i * 1024);
      }
    }
  };
  auto copy_keys = [&]() __attribute__((always_inline)) { copy_rows(kc_base, slot, dma_piece, k_piece, k_dst); };
  auto copy_values = [&]() __attribute__((always_inline)) {
    copy_rows(vc_base, v_slot, v_dma_piece, v_piece, k_dst + BUF_BYTES);
  };

  typedef __attribute__((address_space(3))) const char *LdsBytes;
  // Key-side relocation: the shared rows of a chunk are rotated in LDS once they have landed, with the arithmetic of
  // the stand-alone relocation kernel.  Lane -> row lane / 2, half of its (d, d + D/2) pairs.
  auto rotate_shared_rows = [&](int chunk, int sl) __attribute__((always_inline)) {
    constexpr int PAIRS = CH / 2;
    const int lane = opaque_tid() & 63, row = lane / 2;
    const int delta = chunk * BN + row - sl, ad = delta < 0 ? -delta : delta;
    if (sl >= 0 && sl < p.shared_prefix_len && delta != 0 && ad < p.rope_rows) {
      char *bytes = lds + wave * WAVE_BYTES + row * ROW_BYTES;
      const int f = (row / RW) % CH;
      auto rotate_with = [&](const float *cr, const float *sr, float sign) __attribute__((always_inline)) {
#pragma nounroll
        for (int c = lane % 2; c < PAIRS; c += 2) {
          char *lo_p = bytes + ((c ^ f) << 4), *hi_p = bytes + (((c + PAIRS) ^ f) << 4);
          vec16 lo = load16(lo_p), hi = load16(hi_p);
          rotate_pair_half_fast<DTYPE>(lo, hi, cr, sr, c * 8, D / 2, sign);
          store16(lo_p, lo);
          store16(hi_p, hi);
        }
      };
      if (delta == shift) rotate_with(lds_rope, lds_rope + D, 1.0f);
      else rotate_with(p.cos_tab + (int64_t)ad * D, p.sin_tab + (int64_t)ad * D, delta < 0 ? -1.0f : 1.0f);
    }
  };

  float m_run[NQ16];
  f32x4 o_acc[NQ16][DT], l_acc[NQ16];
  const float c = p.scale_log2e;
#pragma unroll
  for (int qt = 0; qt < NQ16; ++qt) {
    m_run[qt] = -INFINITY;
    l_acc[qt] = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o_acc[qt][dt] = f32x4{0, 0, 0, 0};
  }
  const uint32_t one2 = M::pack2(1.0f, 1.0f);
  const vec16 ones{{one2, one2, one2, one2}};

  // ---- set-up: slots, queries and cos / sin rows in one round trip, the first chunks in the next ---------------------
  // The query rows lie in LDS like a chunk of keys, next to the counter-rotated q' in query-side mode, which scores the
  // shared keys against q' and the others against q: a wave holds one of the two and reads q when its shared chunks are done.
  // (Plain mode at head dim 64: half as many bytes and no rotation, so every wave reads the rows for itself, 0.4 us less of a
  // call of 8 us.)
  constexpr bool STAGE_Q = D == 128 || relocates(MODE);
  vec16 qf[NQ16][KS];
  load_slots(0);
  if (!STAGE_Q) {
#pragma unroll
    for (int qt = 0; qt < NQ16; ++qt) {
      const int row = qt * 16 + li < rows ? qt * 16 + li : rows - 1;
      const char *src = p.q + (int64_t)(q_row0 + row) * p.q_token_bytes + (int64_t)head * p.q_head_bytes;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[qt][ks] = load16(src + (32 * ks + 8 * lg) * 2);
    }
  } else if (wave < QROWS / RPI) {
    // (rows past the end repeat the last one and are not stored)
    const int row = wave * RPI + dma_row;
    const char *src = p.q + (int64_t)(q_row0 + (row < rows ? row : rows - 1)) * p.q_token_bytes + (int64_t)head * p.q_head_bytes +
                      ((dma_piece ^ ((row / RW) % CH)) << 4);
    lds_dma16_at(src, __builtin_amdgcn_readfirstlane(lds_offset_of(lds_q) + (uint32_t)(wave * RPI * ROW_BYTES)));
  }
  if (relocates(MODE)) copy_rope_rows<D>(p, shift, wave, lane, lds_rope);
  take_slots(0);
  copy_keys();                              // (a wave without a chunk copies zero rows)
  copy_values();
  if (STAGE_Q) {
    wait_copies<NI + V_NI>();               // queries and table rows have landed
    __syncthreads();
  }
  auto read_q = [&](const char *from) __attribute__((always_inline)) {
    const int swz = (li / RW) % CH;
#pragma unroll
    for (int qt = 0; qt < NQ16; ++qt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const u32x4 raw = *(__attribute__((address_space(3))) const u32x4 *)((LdsBytes)from + ((qt * 16 + li) * ROW_BYTES + (((4 * ks + lg) ^ swz) << 4)));
        qf[qt][ks] = vec16{{raw.x, raw.y, raw.z, raw.w}};
      }
  };
  if (MODE == MODE_QUERY_SIDE && shift != 0) {
    constexpr int PAIRS = CH / 2;
    if (tid < QROWS * PAIRS) {
      const int row = tid / PAIRS, pair = tid % PAIRS, f = (row / RW) % CH;
      const char *src = lds_q + row * ROW_BYTES;
      char *dst = lds_q + QROWS * ROW_BYTES + row * ROW_BYTES;
      vec16 lo = load16(src + ((pair ^ f) << 4)), hi = load16(src + (((pair + PAIRS) ^ f) << 4));
      rotate_pair_half_fast<DTYPE>(lo, hi, lds_rope, lds_rope + D, pair * 8, D / 2, -1.0f);
      store16(dst + ((pair ^ f) << 4), lo);
      store16(dst + (((pair + PAIRS) ^ f) << 4), hi);
    }
    __syncthreads();
  }
  if (STAGE_Q) {
    read_q(MODE == MODE_QUERY_SIDE && shift != 0 && wave < chunks_a ? lds_q + QROWS * ROW_BYTES : lds_q);
  } else {
#pragma unroll
    for (int qt = 0; qt < NQ16; ++qt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) settle(qf[qt][ks]);  // (waited for here, not inside the loop)
  }

  // ---- fragment addresses ---------------------------------------------------------------------------------------
  LdsBytes k_frag[KS], v_frag[DT];
  {
    const int lane = opaque_tid() & 63, li = lane & 15, lg = lane >> 4;
    const LdsBytes mine = (LdsBytes)lds + wave * WAVE_BYTES;
    const int k_swz = (li / RW) % CH;
    const int v_row = 4 * lg + (li >> 2), v_swz = (v_row / V_RW) % (V_CH / 2);
    const int v_off = v_row * V_ROW_BYTES + (((li & 3) >> 1) << 4) + ((li & 1) << 3);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) k_frag[ks] = mine + (li * ROW_BYTES + (((4 * ks + lg) ^ k_swz) << 4));
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) v_frag[dt] = mine + (BUF_BYTES + v_off + (((dt ^ v_swz) & (V_CH / 2 - 1)) << 5));
  }

  int turn = 0;
  for (int chunk = wave; chunk < n_chunks; chunk += NW) {
    const TileRange r = tile_range_of(chunk, chunks_a, shared_len, kv_len, BN);
    const bool more = chunk + NW < n_chunks;
    if (MODE == MODE_QUERY_SIDE && chunk >= chunks_a && chunk - NW < chunks_a && turn > 0) read_q(lds_q);
    const int rot_now = rot_slot;
    if (more) take_slots(++turn);

    wait_copies<V_NI>();                      // the keys have landed (the values, issued behind them, may not have)
    if (MODE == MODE_KEY_SIDE) {
      rotate_shared_rows(chunk, rot_now);
      wait_lds_reads();
    }
    vec16 kf[2][KS];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const u32x4 raw = *(__attribute__((address_space(3))) const u32x4 *)(k_frag[ks] + 16 * nt * ROW_BYTES);
        kf[nt][ks] = vec16{{raw.x, raw.y, raw.z, raw.w}};
      }
    wait_lds_reads();
    if (more) copy_keys();
    f32x4 s_acc[NQ16][2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int qt = 0; qt < NQ16; ++qt) s_acc[qt][nt] = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int qt = 0; qt < NQ16; ++qt) s_acc[qt][nt] = M::run(kf[nt][ks], qf[qt][ks], s_acc[qt][nt]);
    vec16 pf[NQ16][1];
    softmax_reference<NQ16, NQ16, 2, DT, true>(s_acc, m_run, l_acc, o_acc, c, r.n_end - r.n0, lg);
    softmax_probs_slab<M, 0, NQ16>(s_acc, m_run, l_acc, pf, ones, c);

    if (more) wait_copies<NI>();              // the values have landed
    else wait_copies<0>();
    vec16 vf[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)v_frag[dt]));
      const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)(v_frag[dt] + 16 * V_ROW_BYTES)));
      vf[dt] = vec16{{lo.x, lo.y, hi.x, hi.y}};
    }
    wait_lds_reads();
    if (more) copy_values();
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int qt = 0; qt < NQ16; ++qt) o_acc[qt][dt] = M::run(vf[dt], pf[qt][0], o_acc[qt][dt]);
  }

  // ---- merge: every wave parks its O (fp32, register order) in its own buffers; wave w then sums (query tile, 16
  // features) pairs w, w + NW, ... over the waves in wave order.  A wave without keys has reference -inf and adds 0.
  static_assert(NQ16 * DT * 64 * 16 <= WAVE_BYTES, "a wave's partial O must fit its buffers");
  {
    f32x4 *xo = reinterpret_cast<f32x4 *>(lds + wave * WAVE_BYTES);
#pragma unroll
    for (int qt = 0; qt < NQ16; ++qt) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) xo[(qt * DT + dt) * 64 + lane] = o_acc[qt][dt];
      if (lg == 0) {
        stats[((wave * NQ16 + qt) * 2) * 16 + li] = m_run[qt];
        stats[((wave * NQ16 + qt) * 2 + 1) * 16 + li] = l_acc[qt][0];
      }
    }
  }
  __syncthreads();
  if (NQ16 * DT < NW && wave >= NQ16 * DT) return;
#pragma unroll
  for (int k = 0; k < (NQ16 * DT + NW - 1) / NW; ++k) {
    static_assert(NQ16 * DT % NW == 0 || NQ16 * DT < NW, "the pairs are dealt evenly");
    const int job = wave + k * NW, qt = job / DT, dt = job % DT;
    float m[NW], top = -INFINITY, l = 0.0f;
    f32x4 o{0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      m[w] = stats[((w * NQ16 + qt) * 2) * 16 + li];
      top = fmaxf(top, m[w]);
    }
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float a = __builtin_amdgcn_exp2f(m[w] - top);
      l += stats[((w * NQ16 + qt) * 2 + 1) * 16 + li] * a;
      o += reinterpret_cast<const f32x4 *>(lds + w * WAVE_BYTES)[job * 64 + lane] * a;
    }
    const float inv = l > 0.0f ? 1.0f / l : 1.0f;
    const int qr = qt * 16 + li;
    if (qr < rows) {
      uint2 val;
      val.x = M::pack2(o[0] * inv, o[1] * inv);
      val.y = M::pack2(o[2] * inv, o[3] * inv);
      *reinterpret_cast<uint2 *>(out_base + (int64_t)qr * p.o_token_bytes + (16 * dt + 4 * lg) * 2) = val;
    }
  }
}

// The units of this workgroup: `tiles` query tiles of the batch are dealt in one turn, and what is behind them in others.
template <int DTYPE, int D, int MODE, int FS>
__device__ __forceinline__ void short_attn_units(const AttnParams &p, char *lds, char *lds_q, float *stats, float *lds_rope,
                                                 ShortBatch t, int tiles) {
  int rank, kvh, slice;
  if (!block_to_tile_slice<true>(p, tiles, p.H / p.H_kv * FS, rank, kvh, slice)) return;
  ShortUnit u;
  const int live = t.live;
  while (locate_short_unit<MODE>(p, t, 32, rank, u)) {
    short_attn_unit<DTYPE, D, MODE, FS>(p, lds, lds_q, stats, lds_rope, kvh, kvh * (p.H / p.H_kv) + slice / FS, slice % FS, u);
    rank += tiles;
    if (rank >= live) return;
    __syncthreads();
    t = load_short_batch<MODE>(p, 32);
  }
}

template <int DTYPE, int D, int MODE, int FS>
__global__ __launch_bounds__(64 * NW, 1) void short_attn_kernel(AttnParams p) {
  // the waves' buffers, the queries (and q'), the waves' (reference, denominator) pairs, the cos / sin rows of the shift
  constexpr int FEWER = FS > 1 && MODE != MODE_PAGED ? FS / 2 : FS;
  __shared__ __attribute__((aligned(1024))) char lds[NW * 32 * (D + D / FEWER) * 2];
  __shared__ __attribute__((aligned(1024))) char lds_q[(MODE == MODE_QUERY_SIDE ? 2 : 1) * 32 * D * 2];
  __shared__ float stats[NW * 2 * 2 * 16];
  __shared__ __attribute__((aligned(16))) float lds_rope[relocates(MODE) ? 2 * D : 4];
  const ShortBatch t = load_short_batch<MODE>(p, 32);
  // The grid holds num_tiles units per head, of which the live ones are dealt.  More than those (parts are counted for blocks
  // of one length, other lengths make up to twice the tiles) run in half as many parts, which the grid holds: one turn of the
  // CUs instead of two.  4 requests of 33 and 31 rows, 28 / 4 heads, 1 100 keys: plain 24.1 -> 15.3 us, key side 36.9 -> 21.9;
  // 2 of 32 / 32 heads: 22.6 -> 14.7, 33.7 -> 20.5.  (The common body comes first: behind the other it took 2 to 5 % longer.)
  if (FEWER == FS || __builtin_expect(p.B > 64 || t.live <= p.num_tiles, true))
    short_attn_units<DTYPE, D, MODE, FS>(p, lds, lds_q, stats, lds_rope, t, t.live < p.num_tiles ? t.live : p.num_tiles);
  else
    short_attn_units<DTYPE, D, MODE, FEWER>(p, lds, lds_q, stats, lds_rope, t,
                                            t.live < 2 * p.num_tiles ? t.live : 2 * p.num_tiles);
}

template <int DTYPE, int D, int MODE, int FS>
static int launch_short(AttnParams p, hipStream_t stream) {
  p.small_cache = small_cache(p);
  const int64_t blocks = attn_grid_blocks(p, p.H / p.H_kv * FS);
  if (blocks > 0x7fffffffLL) return fail(ACACHE_E_SHAPE, "varlen_attn: grid too large");
  hipLaunchKernelGGL((short_attn_kernel<DTYPE, D, MODE, FS>), dim3((unsigned)blocks), dim3(64 * NW), 0, stream, p);
  return launch_status("short_attn_kernel");
}

template <int DTYPE, int D, int MODE>
static int launch_parts(const AttnParams &p, int parts, hipStream_t stream) {
  if (D == 128 && parts == 4) return launch_short<DTYPE, D, MODE, D == 128 ? 4 : 1>(p, stream);
  if (D == 128 && parts == 2) return launch_short<DTYPE, D, MODE, D == 128 ? 2 : 1>(p, stream);
  return launch_short<DTYPE, D, MODE, 1>(p, stream);
}

int short_attention(const AttnParams &p, int parts, int mode, int dtype, hipStream_t stream) {
#define ACACHE_SHORT_MODE(DT, DD, MM) \
  if (dtype == DT && p.head_dim == DD && mode == MM) return launch_parts<DT, DD, MM>(p, parts, stream);
#define ACACHE_SHORT_ALL(DT, DD)            \
  ACACHE_SHORT_MODE(DT, DD, MODE_PLAIN)     \
  ACACHE_SHORT_MODE(DT, DD, MODE_KEY_SIDE)  \
  ACACHE_SHORT_MODE(DT, DD, MODE_QUERY_SIDE) \
  ACACHE_SHORT_MODE(DT, DD, MODE_PAGED)
  ACACHE_SHORT_ALL(ACACHE_BF16, 128)
  ACACHE_SHORT_ALL(ACACHE_BF16, 64)
  ACACHE_SHORT_ALL(ACACHE_F16, 128)
  ACACHE_SHORT_ALL(ACACHE_F16, 64)
#undef ACACHE_SHORT_ALL
#undef ACACHE_SHORT_MODE
  return fail(ACACHE_E_SHAPE, "varlen_attn: no short-query kernel for head_dim %d", p.head_dim);
}

}  // namespace acache
