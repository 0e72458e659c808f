// Varlen attention for batches of short query blocks (refinement steps: the 32 tokens of a generation block against
// a thousand cached keys), head dims 64 and 128, all three relocation modes.
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
// Measured (bf16, D = 128, 32 query rows and about 1 300 keys per request, three quarters of them shared, microseconds per
// call, varlen_attn_unit_kernel / this kernel):
//   LLaDA heads, plain 1 request 18.4 / 16.0, 4: 22.6 / 19.1; query side 1: 23.6 / 19.0, 4: 30.8 / 21.6, 8: 33.5 / 24.3;
//   key side 1: 29.4 / 24.0.  Dream heads, plain 1: 18.6 / 16.3, 8: 19.5 / 17.5; query side 8: 25.6 / 20.6; key side 8:
//   31.1 / 27.0.  One LLaDA request keeps 32 CUs busy with 590 KB of keys and values each, which takes 5.4 us by copies
//   alone (110 GB/s into one CU).
#include "attn_common.h"

namespace acache {

static constexpr int NW = 8;  // waves per unit

template <int N> __device__ __forceinline__ void wait_copies() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// this wave's LDS reads have returned: their buffer may be filled again
__device__ __forceinline__ void wait_lds_reads() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// One unit: 32 query rows (query tile `tile_in_request` of request b) of one head.
template <int DTYPE, int D, int MODE>
__device__ __forceinline__ void short_attn_unit(const AttnParams &p, char *lds, float *stats, float *lds_rope, int kvh,
                                                int hg, int b, int q_begin, int q_len, int tile_in_request,
                                                int kv_begin, int kv_len) {
  constexpr int QROWS = 32, NQ16 = 2;         // query rows of a unit
  constexpr int BN = 32;                      // keys per chunk
  constexpr int KS = D / 32, DT = D / 16;
  constexpr int ROW_BYTES = D * 2;
  constexpr int CH = ROW_BYTES / 16;          // 16-byte pieces per row
  constexpr int RW = 256 / ROW_BYTES;         // rows per 256-byte bank window
  constexpr int RPI = 64 / CH;                // rows per copy instruction
  constexpr int NI = BN / RPI;                // copy instructions per chunk and tensor
  constexpr int BUF_BYTES = BN * ROW_BYTES;
  constexpr int WAVE_BYTES = 2 * BUF_BYTES;   // a wave's K buffer, then its V buffer
  using M = Mma<DTYPE>;
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

  const int group = p.H / p.H_kv;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const int head = kvh * group + hg;
  const int q_row0 = tile_in_request * QROWS;
  char *const out_base = p.out + (int64_t)q_begin * p.o_token_bytes + (int64_t)head * p.o_head_bytes;

  if (kv_len <= 0) {  // no keys: defined output (zeros)
    for (int r = tid / CH; r < QROWS; r += 64 * NW / CH)
      if (q_row0 + r < q_len)
        store16(out_base + (int64_t)(q_row0 + r) * p.o_token_bytes + (tid % CH) * 16, vec16{{0, 0, 0, 0}});
    return;
  }

  int shared_len = 0, shift = 0;
  if (MODE == MODE_QUERY_SIDE) {
    shared_len = p.shared_kv_lens[b];
    shared_len = __builtin_amdgcn_readfirstlane(shared_len < 0 ? 0 : (shared_len > kv_len ? kv_len : shared_len));
  }
  if (MODE != MODE_PLAIN) {
    shift = p.affix_shifts[b];
    if (shift < 0 || shift >= p.rope_rows) shift = 0;
  }
  // chunks: the shared range first (query-side mode), then the rest
  const int chunks_a = (shared_len + BN - 1) / BN;
  const int n_chunks = chunks_a + (kv_len - shared_len + BN - 1) / BN;

  // Query fragments.  Query-side mode scores the shared keys against the counter-rotated q', the others against q; a
  // wave holds one of the two and reads q again when its shared chunks are done.
  vec16 qf[NQ16][KS];
  const char *const q_base = p.q + (int64_t)q_begin * p.q_token_bytes + (int64_t)head * p.q_head_bytes;
  auto load_q = [&](bool rotated) __attribute__((always_inline)) {
#pragma unroll
    for (int qt = 0; qt < NQ16; ++qt) {
      // (rows past the end repeat the last one and are not stored: a load under a lane mask is a block of its own)
      const int qr = q_row0 + qt * 16 + li < q_len ? q_row0 + qt * 16 + li : q_len - 1;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        qf[qt][ks] = load16(q_base + (int64_t)qr * p.q_token_bytes + (32 * ks + 8 * lg) * 2);
      if (MODE == MODE_QUERY_SIDE && rotated && shift != 0) {
        const float *cr = p.cos_tab + (int64_t)shift * D, *sr = p.sin_tab + (int64_t)shift * D;
#pragma unroll
        for (int ks = 0; ks < KS / 2; ++ks)
          rotate_pair<DTYPE, D>(qf[qt][ks], qf[qt][ks + KS / 2], cr, sr, 32 * ks + 8 * lg, -1.0f);
      }
    }
  };
  auto settle_q = [&]() __attribute__((always_inline)) {  // (waited for here, not inside the loop)
#pragma unroll
    for (int qt = 0; qt < NQ16; ++qt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) settle(qf[qt][ks]);
  };

  // ---- copies -------------------------------------------------------------------------------------------------
  // Lane l of slots[j] holds the slot of row l % 32 of the wave's chunk 2 j + l / 32, counted from the last refill.
  constexpr int SLOT_REGS = 8;
  int slots[SLOT_REGS];
  auto load_slots = [&](int turn) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < SLOT_REGS; ++j) {
      const TileRange r = tile_range_of(wave + (turn + 2 * j + (lane >> 5)) * NW, chunks_a, shared_len, kv_len, BN);
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
  const char *const vc_base = uniform_ptr(p.v_cache + (int64_t)kvh * p.kv_head_bytes);
  // byte offset of this lane's (swizzled) piece inside its row of copy i: the layouts of attn_dma_part
  auto k_piece = [&](int i) __attribute__((always_inline)) {
    return (uint32_t)((dma_piece ^ (((i * RPI + dma_row) / RW) % CH)) << 4);
  };
  auto v_piece = [&](int i) __attribute__((always_inline)) {
    return (uint32_t)((dma_piece ^ (2 * (((i * RPI + dma_row) / RW) % (CH / 2)))) << 4);
  };
  const uint32_t slot_limit = p.num_slots > 0x7fffffffLL ? 0x7fffffffu : (uint32_t)p.num_slots;
  const uint32_t slot_pitch = (uint32_t)p.kv_slot_bytes;
  const uint32_t k_dst = __builtin_amdgcn_readfirstlane(lds_offset_of(lds) + (uint32_t)(wave * WAVE_BYTES));
  int slot[NI];                               // this lane's slots in the chunk being copied; -1: absent
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
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      slot[i] = __shfl(slots[0], (turn % 2) * 32 + i * RPI + dma_row);
      ok &= (uint32_t)slot[i] < slot_limit;
    }
    if (MODE == MODE_KEY_SIDE) rot_slot = __shfl(slots[0], (turn % 2) * 32 + lane / 2);
    all_present = p.small_cache && __builtin_amdgcn_ballot_w64(!ok) == 0;
  };
  auto copy_chunk = [&](const char *base, auto piece, uint32_t dst) __attribute__((always_inline)) {
    if (all_present) {  // wave-uniform base + 32-bit offsets
#pragma unroll
      for (int i = 0; i < NI; ++i)
        lds_dma16_off(base, __umul24((uint32_t)slot[i], slot_pitch) + piece(i), dst + i * RPI * ROW_BYTES);
    } else {            // absent rows come from the zero row
      const char *zero = reinterpret_cast<const char *>(kZeroRow) + (dma_piece << 4);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const char *src = base + ((uint64_t)(uint32_t)slot[i] * slot_pitch + piece(i));
        lds_dma16_at((uint32_t)slot[i] < slot_limit ? src : zero, dst + i * RPI * ROW_BYTES);
      }
    }
  };

  // ---- fragment addresses ---------------------------------------------------------------------------------------
  typedef __attribute__((address_space(3))) const char *LdsBytes;
  LdsBytes k_frag[KS], v_frag[DT];
  {
    const LdsBytes mine = (LdsBytes)lds + wave * WAVE_BYTES;
    const int k_swz = (li / RW) % CH;
    const int v_row = 4 * lg + (li >> 2), v_swz = (v_row / RW) % (CH / 2);
    const int v_off = v_row * ROW_BYTES + (((li & 3) >> 1) << 4) + ((li & 1) << 3);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) k_frag[ks] = mine + (li * ROW_BYTES + (((4 * ks + lg) ^ k_swz) << 4));
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) v_frag[dt] = mine + (BUF_BYTES + v_off + (((dt ^ v_swz) & (CH / 2 - 1)) << 5));
  }

  // Key-side relocation: the shared rows of a chunk are rotated in LDS once they have landed, with the arithmetic of
  // the stand-alone relocation kernel.  Lane -> row lane / 2, half of its (d, d + D/2) pairs.
  if (MODE == MODE_KEY_SIDE) {
    if (tid < 2 * D / 4) {
      const float *src = (tid < D / 4 ? p.cos_tab : p.sin_tab) + (int64_t)shift * D + (tid % (D / 4)) * 4;
      store16(lds_rope + tid * 4, load16(src));
    }
    __syncthreads();
  }
  auto rotate_shared_rows = [&](int chunk, int sl) __attribute__((always_inline)) {
    constexpr int PAIRS = CH / 2;
    const int row = lane / 2;
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

  if (wave < n_chunks) {
    load_slots(0);                            // slots, queries and then the first chunk: two memory round trips
    load_q(MODE == MODE_QUERY_SIDE && wave < chunks_a);
    take_slots(0);
    copy_chunk(kc_base, k_piece, k_dst);
    copy_chunk(vc_base, v_piece, k_dst + BUF_BYTES);
    settle_q();
  }
  int turn = 0;
  for (int chunk = wave; chunk < n_chunks; chunk += NW) {
    const TileRange r = tile_range_of(chunk, chunks_a, shared_len, kv_len, BN);
    const bool more = chunk + NW < n_chunks;
    if (MODE == MODE_QUERY_SIDE && chunk >= chunks_a && chunk - NW < chunks_a && turn > 0) {
      load_q(false);
      settle_q();
    }
    const int rot_now = rot_slot;
    if (more) take_slots(++turn);

    wait_copies<NI>();                        // the keys have landed (the values, issued behind them, may not have)
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
    if (more) copy_chunk(kc_base, k_piece, k_dst);
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
      const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)(v_frag[dt] + 16 * ROW_BYTES)));
      vf[dt] = vec16{{lo.x, lo.y, hi.x, hi.y}};
    }
    wait_lds_reads();
    if (more) copy_chunk(vc_base, v_piece, k_dst + BUF_BYTES);
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
  for (int job = wave; job < NQ16 * DT; job += NW) {
    const int qt = job / DT, dt = job % DT;
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
    const int qr = q_row0 + qt * 16 + li;
    if (qr < q_len) {
      uint2 val;
      val.x = M::pack2(o[0] * inv, o[1] * inv);
      val.y = M::pack2(o[2] * inv, o[3] * inv);
      *reinterpret_cast<uint2 *>(out_base + (int64_t)qr * p.o_token_bytes + (16 * dt + 4 * lg) * 2) = val;
    }
  }
}

template <int DTYPE, int D, int MODE>
__global__ __launch_bounds__(64 * NW, 1) void short_attn_kernel(AttnParams p) {
  // the waves' buffers, their (reference, denominator) pairs, and in key-side mode the cos / sin rows of the shift
  __shared__ __attribute__((aligned(1024))) char lds[NW * 2 * 32 * D * 2];
  __shared__ float stats[NW * 2 * 2 * 16];
  __shared__ __attribute__((aligned(16))) float lds_rope[MODE == MODE_KEY_SIDE ? 2 * D : 4];
  int rank, kvh, hg, b = 0, q_begin = 0, q_len = 0, tile_in_request = 0, kv_begin = 0, kv_len = 0;
  if (!block_to_tile_head(p, rank, kvh, hg)) return;
  // The grid holds num_tiles units per head: all of them, or one per request, and the others follow in a second turn.
  if (p.B <= 64) {
    int live = rank + 1;
    for (; rank < live; rank += p.num_tiles) {
      if (!locate_query_tile_lpt(p.cu_q, p.cu_k, p.B, 32, rank, b, q_begin, q_len, tile_in_request, kv_begin, kv_len, &live)) return;
      short_attn_unit<DTYPE, D, MODE>(p, lds, stats, lds_rope, kvh, hg, b, q_begin, q_len, tile_in_request, kv_begin, kv_len);
      __syncthreads();
    }
  } else {
    for (; locate_query_tile(p.cu_q, p.B, 32, rank, b, q_begin, q_len, tile_in_request); rank += p.num_tiles) {
      b = __builtin_amdgcn_readfirstlane(b);
      kv_begin = p.cu_k[b];
      short_attn_unit<DTYPE, D, MODE>(p, lds, stats, lds_rope, kvh, hg, b, __builtin_amdgcn_readfirstlane(q_begin),
                                          __builtin_amdgcn_readfirstlane(q_len),
                                          __builtin_amdgcn_readfirstlane(tile_in_request), kv_begin,
                                          p.cu_k[b + 1] - kv_begin);
      __syncthreads();
    }
  }
}

template <int DTYPE, int D, int MODE>
static int launch_short(AttnParams p, hipStream_t stream) {
  p.small_cache = small_cache(p);
  const int64_t blocks = attn_grid_blocks(p);
  if (blocks > 0x7fffffffLL) return fail(ACACHE_E_SHAPE, "varlen_attn: grid too large");
  hipLaunchKernelGGL((short_attn_kernel<DTYPE, D, MODE>), dim3((unsigned)blocks), dim3(64 * NW), 0, stream, p);
  return launch_status("short_attn_kernel");
}

int short_attention(const AttnParams &p, int mode, int dtype, hipStream_t stream) {
#define ACACHE_SHORT_MODE(DT, DD, MM) \
  if (dtype == DT && p.head_dim == DD && mode == MM) return launch_short<DT, DD, MM>(p, stream);
#define ACACHE_SHORT_ALL(DT, DD)            \
  ACACHE_SHORT_MODE(DT, DD, MODE_PLAIN)     \
  ACACHE_SHORT_MODE(DT, DD, MODE_KEY_SIDE)  \
  ACACHE_SHORT_MODE(DT, DD, MODE_QUERY_SIDE)
  ACACHE_SHORT_ALL(ACACHE_BF16, 128)
  ACACHE_SHORT_ALL(ACACHE_BF16, 64)
  ACACHE_SHORT_ALL(ACACHE_F16, 128)
  ACACHE_SHORT_ALL(ACACHE_F16, 64)
#undef ACACHE_SHORT_ALL
#undef ACACHE_SHORT_MODE
  return fail(ACACHE_E_SHAPE, "varlen_attn: no short-query kernel for head_dim %d", p.head_dim);
}

}  // namespace acache
