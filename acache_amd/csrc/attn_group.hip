// Varlen attention for grouped-query batches of short query blocks: head dim 128, all three relocation modes and block
// tables.
//
// What bounds it: with a unit per query head (varlen_attn_unit_kernel) the heads of a group copy every key tile into LDS
// once each, and 32 rows are so little work per key that a unit spends its time in the chain copy -> scores -> softmax ->
// output.  Here a unit is the 32-row query tile of HU heads of a group, one unit per CU.  Its eight waves are 8 / HU streams
// of HU waves; in a round every stream takes 32 keys, which its waves copy together (32 / HU rows each) while the round
// before is computed, and each wave scores them for its own head.  The waves of a stream wait for one another only, so that
// streams drift apart and the matrix work of one runs beside the softmax of another; partial results of the streams are
// merged through LDS at the end.  Two heads: four streams, 128 KB of LDS; four heads: two streams, half the copies per score.
//
// The set-up is three dependent round trips (lengths; slots, queries, table rows; keys), and it counts: of 16 requests' 28
// us, 7 were set-up before the queries went through LDS once per unit and the lookup took all lengths in one trip.
//
// Measured (bf16, 28 / 4 heads, 32 query rows and about 1 100 keys per request, three quarters of them shared, microseconds
// per call, the kernels of attn.hip / this one): 2 heads, 16 requests: plain 23.6 / 21.1, key side 38.5 / 28.0, query side
// 28.5 / 22.0; 4 heads, query side, 24 requests 34.9 / 33.1, 32: 36.7 / 34.1, 64: 76.0 / 65.6; key side, 32: 44.0 / 37.5.
// A round takes 1.25 to 1.5 us.  Bounds of a round per SIMD: 68 matrix instructions (0.5 us), about 330 vector ones of
// which 32 transcendental (0.5); per CU 64 KB of copies (0.5) and 192 KB of LDS traffic (0.7).  With one barrier of the
// whole unit per round 1.7; copies spread over the matrix instructions instead of in one burst: the same.
#include "attn_common.h"

namespace acache {

static constexpr int GROUP_WAVES = 8;

template <int DTYPE, int D, int MODE, int HU>
__device__ __forceinline__ void group_attn_unit(const AttnParams &p, char *lds, char *lds_q, float *stats, float *lds_rope, int *landed,
                                                int kvh, int first_head, int heads, const ShortUnit &u) {
  constexpr int NW = GROUP_WAVES, W = NW / HU;  // streams
  constexpr int QROWS = 32, NQ16 = 2;
  constexpr int BN = 32;                        // keys per chunk
  constexpr int KS = D / 32, DT = D / 16;
  constexpr int ROW_BYTES = D * 2;
  constexpr int CH = ROW_BYTES / 16;            // 16-byte pieces per row
  constexpr int RW = 256 / ROW_BYTES;           // rows per 256-byte bank window
  constexpr int RPI = 64 / CH;                  // rows per copy instruction
  constexpr int RPW = BN / HU;                  // rows of its stream's chunk that a wave copies
  constexpr int NI = RPW / RPI;                 // copy instructions per round and tensor
  static_assert(NI >= 1 && RPW % RPI == 0, "whole copy instructions");
  constexpr int BUF_BYTES = BN * ROW_BYTES;
  constexpr int STREAM_BYTES = 4 * BUF_BYTES;   // K, V of even rounds, K, V of odd rounds
  using M = Mma<DTYPE>;
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

  const int tid = opaque_tid(), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int stream = wave / HU, which = wave % HU;
  const int li = lane & 15, lg = lane >> 4;
  const int kv_begin = u.kv_begin, kv_len = u.kv_len, shared_len = u.shared_len, shift = u.shift;
  const int q_row0 = u.q_begin + u.tile * QROWS;
  const int rows = u.q_len - u.tile * QROWS < QROWS ? u.q_len - u.tile * QROWS : QROWS;
  char *const out_base = p.out + (int64_t)q_row0 * p.o_token_bytes;

  if (kv_len <= 0) {  // no keys: defined output (zeros)
    for (int r = tid / CH; r < rows * heads; r += 64 * NW / CH)
      store16(out_base + (int64_t)(r % rows) * p.o_token_bytes + (int64_t)(first_head + r / rows) * p.o_head_bytes +
                  (tid % CH) * 16, vec16{{0, 0, 0, 0}});
    return;
  }

  // chunks: the shared range first (query-side mode), then the rest
  const int chunks_a = (shared_len + BN - 1) / BN;
  const int n_chunks = chunks_a + (kv_len - shared_len + BN - 1) / BN;
  const int rounds = (n_chunks + W - 1) / W;

  // ---- copies: rows which * RPW .. + RPW of the stream's chunk ---------------------------------------------------
  const int dma_row = which * RPW + lane / CH, dma_piece = lane % CH;   // + i * RPI
  const char *const kc_base = uniform_ptr(p.k_cache + (int64_t)kvh * p.kv_head_bytes);
  const char *const vc_base = uniform_ptr(p.v_cache + (int64_t)kvh * p.kv_head_bytes);
  const uint32_t slot_limit = p.num_slots > 0x7fffffffLL ? 0x7fffffffu : (uint32_t)p.num_slots;
  const uint32_t slot_pitch = (uint32_t)p.kv_slot_bytes;
  const uint32_t my_dst = __builtin_amdgcn_readfirstlane(lds_offset_of(lds) + (uint32_t)(stream * STREAM_BYTES + which * RPW * ROW_BYTES));
  int slot_next[NI], slot[NI];                // slots of the round after the one being copied, and of that one
  int rot_next = -1, rot_slot = -1;           // key-side mode: slot of row which * RPW + lane / (64 / RPW)
  const char *const slot_base = reinterpret_cast<const char *>(p.slot_map + kv_begin);
  auto load_slots = [&](int round) __attribute__((always_inline)) {
    const TileRange r = tile_range_of(round * W + stream, chunks_a, shared_len, kv_len, BN);
    if (MODE == MODE_PAGED) {                 // one table entry for the chunk; take_slots makes the slots of it
      slot_next[0] = r.n0 < r.n_end ? table_entry(p, u.b, r.n0) : -1;
      return;
    }
    const int rot_row = which * RPW + lane / (64 / RPW);
    if (r.n0 + BN <= r.n_end) {               // (wave-uniform) a scalar base, one offset per lane, immediates
      const char *const base = slot_base + (int64_t)r.n0 * 4;
#pragma unroll
      for (int i = 0; i < NI; ++i) slot_next[i] = *reinterpret_cast<const int *>(base + (uint32_t)(dma_row * 4) + i * RPI * 4);
      if (MODE == MODE_KEY_SIDE) rot_next = *reinterpret_cast<const int *>(base + (uint32_t)(rot_row * 4));
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int n = r.n0 + dma_row + i * RPI;
        const int s = *reinterpret_cast<const int *>(slot_base + (int64_t)(n < kv_len ? n : kv_len - 1) * 4);
        slot_next[i] = n < r.n_end ? s : -1;
      }
      if (MODE == MODE_KEY_SIDE) {
        const int n = r.n0 + rot_row;
        const int s = *reinterpret_cast<const int *>(slot_base + (int64_t)(n < kv_len ? n : kv_len - 1) * 4);
        rot_next = n < r.n_end ? s : -1;
      }
    }
  };
  bool all_present = false;
  auto take_slots = [&](int round) __attribute__((always_inline)) {
    bool ok = true;
    const int first = (round * W + stream) * BN + dma_row;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if (MODE == MODE_PAGED) slot[i] = first + i * RPI < kv_len ? slot_of_entry(p, slot_next[0], first + i * RPI) : -1;
      else slot[i] = slot_next[i];
      asm volatile("" : "+v"(slot[i]));       // (waited for here, in front of the next copies)
      ok &= (uint32_t)slot[i] < slot_limit;
    }
    if (MODE == MODE_KEY_SIDE) {
      rot_slot = rot_next;
      asm volatile("" : "+v"(rot_slot));
    }
    all_present = p.small_cache && __builtin_amdgcn_ballot_w64(!ok) == 0;
  };
  auto piece = [&](int i, bool value) __attribute__((always_inline)) {
    const int r = (dma_row + i * RPI) / RW;
    return (uint32_t)((dma_piece ^ (value ? 2 * (r % (CH / 2)) : r % CH)) << 4);
  };
  auto copy_round = [&](uint32_t dst) __attribute__((always_inline)) {
    if (all_present) {  // wave-uniform base + 32-bit offsets
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const uint32_t row = __umul24((uint32_t)slot[i], slot_pitch);
        lds_dma16_off(kc_base, row + piece(i, false), dst + i * RPI * ROW_BYTES);
        lds_dma16_off(vc_base, row + piece(i, true), dst + BUF_BYTES + i * RPI * ROW_BYTES);
      }
    } else {            // absent rows come from the zero row
      const char *zero = reinterpret_cast<const char *>(kZeroRow) + (dma_piece << 4);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const bool present = (uint32_t)slot[i] < slot_limit;
        const uint64_t row = (uint64_t)(uint32_t)slot[i] * slot_pitch;
        lds_dma16_at(present ? kc_base + (row + piece(i, false)) : zero, dst + i * RPI * ROW_BYTES);
        lds_dma16_at(present ? vc_base + (row + piece(i, true)) : zero, dst + BUF_BYTES + i * RPI * ROW_BYTES);
      }
    }
  };

  typedef __attribute__((address_space(3))) const char *LdsBytes;
  // Key-side relocation: a wave rotates the shared rows that it copied, in LDS, before the barrier publishes them, with
  // the arithmetic of the stand-alone relocation kernel.
  auto rotate_shared_rows = [&](int round, char *kbuf) __attribute__((always_inline)) {
    constexpr int PAIRS = CH / 2, LPR = 64 / RPW;  // lanes per row
    const int row = which * RPW + lane / LPR;
    const int chunk = round * W + stream;
    const int delta = chunk * BN + row - rot_slot, ad = delta < 0 ? -delta : delta;
    if (rot_slot >= 0 && rot_slot < p.shared_prefix_len && delta != 0 && ad < p.rope_rows) {
      char *bytes = kbuf + row * ROW_BYTES;
      const int f = (row / RW) % CH;
      auto rotate_with = [&](const float *cr, const float *sr, float sign) __attribute__((always_inline)) {
#pragma nounroll
        for (int c = lane % LPR; c < PAIRS; c += LPR) {
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

  // ---- set-up: slots, queries and cos / sin rows in one round trip, the first round's copies in the next -----------
  // The query rows of the unit's heads lie in LDS like chunks of keys.  Query-side mode scores the shared keys against
  // the counter-rotated q', which is made once for the unit in the buffers of the odd rounds, and the others against q.
  constexpr int QCOPIES = HU * QROWS / RPI / NW;  // copy instructions per wave for the queries
  load_slots(0);
#pragma unroll
  for (int i = 0; i < QCOPIES; ++i) {
    const int r = (wave * QCOPIES + i) * RPI + lane / CH, h = r / QROWS, row = r % QROWS;
    // (rows past the end repeat the last one, absent heads the first; neither is stored)
    const char *src = p.q + (int64_t)(q_row0 + (row < rows ? row : rows - 1)) * p.q_token_bytes +
                      (int64_t)(first_head + (h < heads ? h : 0)) * p.q_head_bytes + ((dma_piece ^ ((row / RW) % CH)) << 4);
    lds_dma16_at(src, __builtin_amdgcn_readfirstlane(lds_offset_of(lds_q) + (uint32_t)((wave * QCOPIES + i) * RPI * ROW_BYTES)));
  }
  if (lane == 0) landed[wave] = 0;
  if (relocates(MODE)) copy_rope_rows<D>(p, shift, wave, lane, lds_rope);
  take_slots(0);
  copy_round(my_dst);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NI) : "memory");  // queries and table rows have landed
  __syncthreads();
  const LdsBytes q_mine = (LdsBytes)lds_q + which * (QROWS * ROW_BYTES);
  // (q' of heads 2 s and 2 s + 1 in the odd rounds' buffers of stream s)
  static_assert(QROWS == BN && HU <= 2 * W, "a head's query rows are one buffer");
  auto q_rot_at = [](int h) __attribute__((always_inline)) { return (h / 2) * STREAM_BYTES + (2 + h % 2) * BUF_BYTES; };
  vec16 qf[NQ16][KS];
  auto read_q = [&](LdsBytes from) __attribute__((always_inline)) {
    const int swz = (li / RW) % CH;
#pragma unroll
    for (int qt = 0; qt < NQ16; ++qt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const u32x4 raw = *(__attribute__((address_space(3))) const u32x4 *)(from + ((qt * 16 + li) * ROW_BYTES + (((4 * ks + lg) ^ swz) << 4)));
        qf[qt][ks] = vec16{{raw.x, raw.y, raw.z, raw.w}};
      }
  };
  if (MODE == MODE_QUERY_SIDE && shift != 0) {
    constexpr int PAIRS = CH / 2;
#pragma unroll
    for (int job = 0; job < HU * QROWS * PAIRS / (64 * NW); ++job) {
      const int at = job * 64 * NW + tid, row = at / PAIRS, pair = at % PAIRS, f = (row / RW) % CH;
      const char *src = lds_q + row * ROW_BYTES;
      char *dst = lds + q_rot_at(row / QROWS) + (row % QROWS) * ROW_BYTES;
      vec16 lo = load16(src + ((pair ^ f) << 4)), hi = load16(src + (((pair + PAIRS) ^ f) << 4));
      rotate_pair_half_fast<DTYPE>(lo, hi, lds_rope, lds_rope + D, pair * 8, D / 2, -1.0f);
      store16(dst + ((pair ^ f) << 4), lo);
      store16(dst + (((pair + PAIRS) ^ f) << 4), hi);
    }
    __syncthreads();
    read_q(stream < chunks_a ? (LdsBytes)lds + q_rot_at(which) : q_mine);
    __syncthreads();                          // before a stream's first copies into those buffers
  } else {
    read_q(q_mine);
  }
  if (rounds > 1) load_slots(1);

  // ---- fragment addresses -----------------------------------------------------------------------------------------
  LdsBytes k_frag[KS], v_frag[DT];
  {
    const int lane = opaque_tid() & 63, li = lane & 15, lg = lane >> 4;
    const LdsBytes mine = (LdsBytes)lds + stream * STREAM_BYTES;
    const int k_swz = (li / RW) % CH;
    const int v_row = 4 * lg + (li >> 2), v_swz = (v_row / RW) % (CH / 2);
    const int v_off = v_row * ROW_BYTES + (((li & 3) >> 1) << 4) + ((li & 1) << 3);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) k_frag[ks] = mine + (li * ROW_BYTES + (((4 * ks + lg) ^ k_swz) << 4));
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) v_frag[dt] = mine + (BUF_BYTES + v_off + (((dt ^ v_swz) & (CH / 2 - 1)) << 5));
  }

  // A stream's waves wait for one another only: `landed` of a wave is the number of rounds whose rows it has copied, and
  // what it read of earlier rounds is in its registers by then.  All of them go through every round, so every wait ends.
  auto stream_barrier = [&](int count) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) volatile int *LdsFlag;
    const LdsFlag flags = (LdsFlag)landed + stream * HU;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    flags[which] = count;                       // (every lane the same value)
    while (__builtin_amdgcn_ballot_w64(flags[lane % HU] < count) != 0) {}
    asm volatile("" ::: "memory");
  };
  for (int round = 0; round < rounds; ++round) {
    const int HERE = (round & 1) * 2 * BUF_BYTES, THERE = 2 * BUF_BYTES - HERE;
    const int chunk = round * W + stream;
    const bool more = round + 1 < rounds;
    if (MODE == MODE_KEY_SIDE) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      rotate_shared_rows(round, lds + stream * STREAM_BYTES + HERE);
    }
    stream_barrier(round + 1);
    vec16 kf[2][KS];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const u32x4 raw = *(__attribute__((address_space(3))) const u32x4 *)(k_frag[ks] + (HERE + 16 * nt * ROW_BYTES));
        kf[nt][ks] = vec16{{raw.x, raw.y, raw.z, raw.w}};
      }
    if (more) {
      take_slots(round + 1);
      if (round + 2 < rounds) load_slots(round + 2);
      copy_round(my_dst + THERE);
    }
    if (chunk < n_chunks && which < heads) {
      const TileRange r = tile_range_of(chunk, chunks_a, shared_len, kv_len, BN);
      f32x4 s_acc[NQ16][2];
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int qt = 0; qt < NQ16; ++qt) s_acc[qt][nt] = f32x4{0, 0, 0, 0};
      if (MODE == MODE_QUERY_SIDE && chunk >= chunks_a && chunk - W < chunks_a && round > 0) read_q(q_mine);
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int qt = 0; qt < NQ16; ++qt) s_acc[qt][nt] = M::run(kf[nt][ks], qf[qt][ks], s_acc[qt][nt]);
      vec16 vf[DT];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)(v_frag[dt] + HERE)));
        const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)(v_frag[dt] + (HERE + 16 * ROW_BYTES))));
        vf[dt] = vec16{{lo.x, lo.y, hi.x, hi.y}};
      }
      vec16 pf[NQ16][1];
      softmax_reference<NQ16, NQ16, 2, DT, true>(s_acc, m_run, l_acc, o_acc, c, r.n_end - r.n0, lg);
      softmax_probs_slab<M, 0, NQ16>(s_acc, m_run, l_acc, pf, ones, c);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int qt = 0; qt < NQ16; ++qt) o_acc[qt][dt] = M::run(vf[dt], pf[qt][0], o_acc[qt][dt]);
    }
  }
  __syncthreads();  // every wave is done with the buffers

  // ---- merge: every wave parks its O (fp32, register order); the waves of a head take a share of its features each
  // and sum over the streams in order.  A stream without keys has reference -inf and adds 0.
  constexpr int PARK_BYTES = NQ16 * DT * 64 * 16;
  {
    f32x4 *xo = reinterpret_cast<f32x4 *>(lds + wave * PARK_BYTES);
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
  if (which >= heads) return;
  static_assert(DT % W == 0, "features of a query tile are dealt evenly");
#pragma unroll
  for (int qt = 0; qt < NQ16; ++qt) {
    float a[W], top = -INFINITY, l = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      a[w] = stats[(((w * HU + which) * NQ16 + qt) * 2) * 16 + li];
      top = fmaxf(top, a[w]);
    }
#pragma unroll
    for (int w = 0; w < W; ++w) {
      a[w] = __builtin_amdgcn_exp2f(a[w] - top);
      l += stats[(((w * HU + which) * NQ16 + qt) * 2 + 1) * 16 + li] * a[w];
    }
    const float inv = l > 0.0f ? 1.0f / l : 1.0f;
    const int qr = qt * 16 + li;
    char *const out_row = out_base + (int64_t)qr * p.o_token_bytes + (int64_t)(first_head + which) * p.o_head_bytes + 8 * lg;
#pragma unroll
    for (int k = 0; k < DT / W; ++k) {
      const int dt = k * W + stream;
      f32x4 o{0, 0, 0, 0};
#pragma unroll
      for (int w = 0; w < W; ++w)
        o += reinterpret_cast<const f32x4 *>(lds + (w * HU + which) * PARK_BYTES)[(qt * DT + dt) * 64 + lane] * a[w];
      if (qr < rows) {
        uint2 val;
        val.x = M::pack2(o[0] * inv, o[1] * inv);
        val.y = M::pack2(o[2] * inv, o[3] * inv);
        *reinterpret_cast<uint2 *>(out_row + 32 * dt) = val;
      }
    }
  }
}

// The units of this workgroup: `tiles` query tiles of the batch are dealt in one turn, and what is behind them in others.
template <int DTYPE, int D, int MODE, int HU>
__device__ __forceinline__ void group_attn_units(const AttnParams &p, char *lds, char *lds_q, float *stats, float *lds_rope, int *landed,
                                                 ShortBatch t, int tiles) {
  const int group = p.H / p.H_kv;
  int rank, kvh, slice;
  if (!block_to_tile_slice<true>(p, tiles, (group + HU - 1) / HU, rank, kvh, slice)) return;
  const int first = slice * HU, heads = group - first < HU ? group - first : HU;
  ShortUnit u;
  const int live = t.live;
  while (locate_short_unit<MODE>(p, t, 32, rank, u)) {
    group_attn_unit<DTYPE, D, MODE, HU>(p, lds, lds_q, stats, lds_rope, landed, kvh, kvh * group + first, heads, u);
    rank += tiles;
    if (rank >= live) return;
    __syncthreads();
    t = load_short_batch<MODE>(p, 32);
  }
}

template <int DTYPE, int D, int MODE, int HU>
__global__ __launch_bounds__(64 * GROUP_WAVES, 1) void group_attn_kernel(AttnParams p) {
  // two rounds of chunks and the queries (a unit of four heads needs less), later the parked partial sums; the (reference,
  // denominator) pairs; the cos / sin rows of the shift
  constexpr int RING = GROUP_WAVES / HU * 4 * 32 * D * 2, Q = HU * 32 * D * 2, PARK = GROUP_WAVES * 32 * D * 4;
  __shared__ __attribute__((aligned(1024))) char lds[RING + Q > PARK ? RING + Q : PARK];
  __shared__ int landed[GROUP_WAVES];
  __shared__ float stats[GROUP_WAVES * 2 * 2 * 16];
  __shared__ __attribute__((aligned(16))) float lds_rope[relocates(MODE) ? 2 * D : 4];
  const ShortBatch t = load_short_batch<MODE>(p, 32);
  // The grid holds num_tiles units per slice, of which the live ones are dealt.  More than those (units are counted for blocks
  // of one length) are units of four heads where the grid holds those: one longer turn of the CUs instead of two.  16 requests
  // of 33 and 31 rows, 28 / 4 heads, 1 100 keys: plain 36.4 -> 31.9 us, key side 47.5 -> 37.4, query side 37.5 -> 33.6.
  constexpr int RING4 = GROUP_WAVES / 4 * 4 * 32 * D * 2;
  static_assert(RING4 + 4 * 32 * D * 2 <= sizeof(lds) && PARK <= sizeof(lds), "units of four heads fit");
  if (HU == 4 || MODE == MODE_PAGED || __builtin_expect(p.B > 64 || t.live <= p.num_tiles ||
                                                        t.live > tiles_in_grid(p, (p.H / p.H_kv + 3) / 4, gridDim.x), true))
    group_attn_units<DTYPE, D, MODE, HU>(p, lds, lds + RING, stats, lds_rope, landed, t, t.live < p.num_tiles ? t.live : p.num_tiles);
  else
    group_attn_units<DTYPE, D, MODE, 4>(p, lds, lds + RING4, stats, lds_rope, landed, t, t.live);
}

template <int DTYPE, int D, int MODE, int HU>
static int launch_group(AttnParams p, hipStream_t stream) {
  p.small_cache = small_cache(p);
  const int64_t blocks = attn_grid_blocks(p, (p.H / p.H_kv + HU - 1) / HU);
  if (blocks > 0x7fffffffLL) return fail(ACACHE_E_SHAPE, "varlen_attn: grid too large");
  hipLaunchKernelGGL((group_attn_kernel<DTYPE, D, MODE, HU>), dim3((unsigned)blocks), dim3(64 * GROUP_WAVES), 0, stream, p);
  return launch_status("group_attn_kernel");
}

int group_attention(const AttnParams &p, int heads_per_unit, int mode, int dtype, hipStream_t stream) {
#define ACACHE_GROUP_MODE(DT, HU, MM) \
  if (dtype == DT && heads_per_unit == HU && mode == MM) return launch_group<DT, 128, MM, HU>(p, stream);
#define ACACHE_GROUP_ALL(DT, HU)            \
  ACACHE_GROUP_MODE(DT, HU, MODE_PLAIN)     \
  ACACHE_GROUP_MODE(DT, HU, MODE_KEY_SIDE)  \
  ACACHE_GROUP_MODE(DT, HU, MODE_QUERY_SIDE) \
  ACACHE_GROUP_MODE(DT, HU, MODE_PAGED)
  ACACHE_GROUP_ALL(ACACHE_BF16, 2)
  ACACHE_GROUP_ALL(ACACHE_F16, 2)
  ACACHE_GROUP_ALL(ACACHE_BF16, 4)
  ACACHE_GROUP_ALL(ACACHE_F16, 4)
#undef ACACHE_GROUP_ALL
#undef ACACHE_GROUP_MODE
  return fail(ACACHE_E_SHAPE, "varlen_attn: no grouped kernel for %d heads per unit", heads_per_unit);
}

}  // namespace acache
