// Causal chunked-prefill paged attention for chunks that fill the chip (gfx950 MFMA fp16).
//
// Same operation as paged_prefill_wide.hip (docs/architecture.md:246; contiguous semantics
// src/infurnace/executor/tinygrad/model.py:116-132: query row i sits at start_position + i and sees
// keys with key_pos <= query_pos), for calls with enough query rows to fill the chip without sharing
// key ranges out to workgroups (prefill_block_groups).
//
//  * Rows.  A workgroup of 4 waves serves 128 query rows of one kv head: 128 / G queries x the G
//    query heads.  Wave w holds 32 of them (32 / G consecutive queries), so two workgroups
//    share a CU: two waves per SIMD, one's MFMAs beside the other's softmax.  With too few workgroups
//    for that, a workgroup has two such key groups of 4 waves (KS = 2), which take alternate tiles and
//    merge through LDS (fp32) at the end.
//  * Keys.  All waves walk the same 64-key tiles, staged once per workgroup in LDS (two buffers):
//    wave w brings page w of the tile, K and V, through registers.  A key tile is read from L2 once
//    per 128 rows and written to LDS once, where a kernel whose waves are key groups moves it once
//    per wave.
//  * S^T = K Q^T and O^T += V^T P^T with v_mfma_f32_32x32x16_f16: a lane owns one query row, its 16
//    scores of a 32-key half are the B operands of two K = 16 steps of the second product.
//  * Fused append (kAppend, query_start a multiple of the page): pages at or past query_start are
//    read from new_k / new_v, and the workgroup that holds a page's queries stores its head of that
//    page to the pool from the registers that carry it to LDS.
//
// What bounds it: power, then issue.  2048 queries at 6144, 32 / 8 heads x 128 (240 GFLOP): 275 us,
// 875 TFLOP/s, against 334 us on the wide kernel (same run).  The matrix cores are busy 46% of the cycles;
// the clock is 1.87 GHz in the first launches of a burst and falls from there (263 -> 323 us over 12
// launches in a row; an 8192^3 fp16 product goes from 1355 to 1172 TFLOP/s).  8192 queries at 0, 16 / 8
// heads: 391 -> 308 us.
#include "ifn_common.hpp"

namespace ifn {

constexpr int kBPage = 16;               // tokens per page compiled in
constexpr int kBTile = 64;               // keys per tile
constexpr int kBPages = kBTile / kBPage;
constexpr int kBWaves = 4;
constexpr int kBThreads = kBWaves * kWave;
constexpr int kBXcdCus = 32;             // CUs per XCD, 8 XCDs

typedef __attribute__((address_space(3))) u32x4 lds_u32x4;

template <int D, int G>
struct BlockCfg {
  static constexpr int kQw = 32 * kBWaves / G;   // queries per workgroup
  static constexpr int kQwave = 32 / G;          // queries per wave
  static constexpr int kKS = D / 16;             // MFMA K-steps over the head dims
  static constexpr int kDT = D / 32;             // 32-dim output tiles
  static constexpr int kCh = D / 8;              // 16-byte chunks per key row
  static constexpr int kRowsI = kWave / kCh;     // key rows per 16-byte load instruction
  static constexpr int kInstr = kBPage / kRowsI; // instructions per page (of K, of V)
  // LDS rows are padded so that the 16 lanes of a 16-byte access, or the 32 of an 8-byte one, cover the
  // 64 banks once: K rows by one chunk (a fragment read takes one chunk of 16 rows), V rows by 64
  // bytes (a transposing read takes 64 bytes of 4 rows).
  static constexpr int kKRowB = 2 * D + 16;
  static constexpr int kVRowB = 2 * D + 64;
  static constexpr int kKTileB = kBTile * kKRowB;
  static constexpr int kVTileB = kBTile * kVRowB;
  static constexpr int kBufB = kKTileB + kVTileB;
  static constexpr int kLdsB = 2 * kBufB;
  static_assert(kQw % kBPage == 0, "a workgroup's queries are whole pages of the chunk");
};

// No instruction: the values must exist at this point.
__device__ __forceinline__ void blk_pin(f16x8& a, f16x8& b) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(a), "+v"(b));
#endif
}
// Workgroup barrier for LDS traffic alone: this wave's LDS writes are done, its loads may be in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int D, int G, int KS, bool kAppend>
__global__ __launch_bounds__(KS * kBThreads, 2) void prefill_block_kernel(
    f16* out, const f16* q, const f16* __restrict__ pool, int64_t num_pages, const int32_t* __restrict__ table,
    int32_t query_start, int32_t T, int32_t num_kv_heads, int32_t n_qb, float scale_log2, PrefillAppend ap) {
  using C = BlockCfg<D, G>;
  constexpr int kKS = C::kKS, kDT = C::kDT, kI = C::kInstr;
  constexpr int kMergeB = KS > 1 ? kBThreads * KS * (16 * kDT / KS + 2) * 4 : 0;
  constexpr int kLds = KS * C::kLdsB > kMergeB ? KS * C::kLdsB : kMergeB;
  __shared__ __attribute__((aligned(16))) unsigned char smem[kLds];
  // kv head = workgroup mod Hkv (for Hkv = 8 each XCD keeps one head's K/V in its L2); query blocks
  // go longest key range first.
  int bid = int(blockIdx.x);
  if constexpr (KS == 1) {
    // Two workgroups per CU: workgroups 32 apart on an XCD meet on one CU, so every other full round of
    // the chip runs in reverse and the long ranges meet the short ones (16 q heads, 4096 queries at 0:
    // 107.6 -> 101.6 us).
    const int per = 8 * kBXcdCus, r = bid % per;
    if ((bid / per) % 2 == 1 && bid - r + per <= int(gridDim.x)) bid += 8 * (kBXcdCus - 1 - 2 * (r / 8));
  }
  const int kvh = bid % num_kv_heads;
  const int qb = n_qb - 1 - bid / num_kv_heads;
  const int tid = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wave = wv % kBWaves, grp = wv / kBWaves;  // row block of the workgroup, key group
  const int lane = tid % kWave;
  const int col = lane % 32, half = lane / 32;
  const int hq = num_kv_heads * G;
  const int q0 = qb * C::kQw;
  const int total = query_start + T;
  const int key_end = min(total, query_start + q0 + C::kQw);  // keys some row sees
  const int n_tiles = int(ceil_div(key_end, kBTile));
  const int wq0 = q0 + wave * C::kQwave;                      // the wave's first query
  const int wave_first = query_start + wq0;                   // ... and its position: every row sees up to it
  const int wave_last = wave_first + C::kQwave - 1;
  const int my_q = wq0 + col % C::kQwave;
  const int my_head = kvh * G + col / C::kQwave;
  const int my_pos = query_start + my_q;

  const int64_t tok_stride = int64_t(num_kv_heads) * D;
  const int tok_bytes = int(tok_stride) * 2;
  const int64_t v_off = num_pages * kBPage * tok_stride;
  const int64_t page_elems = int64_t(kBPage) * tok_stride;
  const f16* head_pool = pool + int64_t(kvh) * D;

  // Page ids, 64 per window (16 tiles), one per lane; the next window is requested one window ahead.
  const int seq_pages = int(ceil_div(total, kBPage));
  auto load_window = [&](int w) __attribute__((always_inline)) {
    const int pg = 64 * w + lane;
    const int id = table[min(pg, seq_pages - 1)];
    return pg < seq_pages ? id : -1;
  };
  int win = 0, ids = load_window(0), ids_next = load_window(1);

  // This lane's query row: K-step s takes dims 16 s + 8 half .. + 7 (rows past the chunk: zeros).
  f16x8 qreg[kKS];
  {
    const f16* qp = q + (int64_t(min(my_q, T - 1)) * hq + my_head) * D + 8 * half;
#pragma unroll
    for (int s = 0; s < kKS; ++s) {
      const u32x4 v = ld16(qp + 16 * s);
      qreg[s] = as_h8(my_q < T ? v : u32x4{0u, 0u, 0u, 0u});
    }
  }

  // Staging of a tile: lane l of load n holds chunk l % kCh of the page's row kRowsI n + l / kCh.
  uint32_t goff[kI];  // byte offset of load n in its page's rows (the descriptor's bound applies to it)
#pragma unroll
  for (int n = 0; n < kI; ++n) goff[n] = uint32_t((n * C::kRowsI + lane / C::kCh) * tok_bytes + (lane % C::kCh) * 16);
  lds_u8* const lds = (lds_u8*)(smem) + grp * C::kLdsB;
  uint32_t kwr, vwr;  // LDS byte offsets of load 0
  {
    const int r = kBPage * wave + lane / C::kCh, c = lane % C::kCh;
    kwr = uint32_t(r * C::kKRowB + c * 16);
    vwr = uint32_t(C::kKTileB + r * C::kVRowB + c * 16);
  }
  // K runs one tile ahead of V: step i reads K of tile i + 1 and V of tile i.
  u32x4 kst[kI], vst[kI];
  struct Tile {
    int kt, fl;      // first key; page flags (bit p: page p is in the pool)
    int page, rows;  // this wave's page of the tile and its keys (0: none)
  };
  auto tile_at = [&](int i) __attribute__((always_inline)) -> Tile {
    const int t = KS * i + grp;
    if ((t >> 4) != win) {  // (uniform)
      win = t >> 4;
      ids = ids_next;
      ids_next = load_window(win + 1);
    }
    const uint64_t valid = __builtin_amdgcn_ballot_w64(ids >= 0 && int64_t(ids) < num_pages);
    const int fl = int(valid >> (4 * (t & 15))) & 15;
    const bool ok = ((fl >> wave) & 1) != 0;
    // (page and row count are uniform; readfirstlane keeps the descriptors in scalar registers)
    return Tile{kBTile * t, fl,
                __builtin_amdgcn_readfirstlane(ok ? __builtin_amdgcn_readlane(ids, (kBPages * t + wave) & 63) : 0),
                __builtin_amdgcn_readfirstlane(ok ? min(max(total - kBTile * t - kBPage * wave, 0), kBPage) : 0)};
  };
  // The rows of this wave's page of a tile: in the pool or, kAppend, among the chunk's own.
  auto page_rsrc = [&](const Tile& t, int64_t kv, const f16* own) __attribute__((always_inline)) {
    const f16* p = head_pool + int64_t(t.page) * page_elems + kv;
    if constexpr (kAppend) {
      const int t0 = t.kt + kBPage * wave - query_start;  // the page's first token within the chunk
      if (t0 >= 0) p = own + int64_t(min(t0, T - 1)) * tok_stride + int64_t(kvh) * D;
    }
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<f16*>(p), 0, t.rows * tok_bytes, 0x00020000);
  };
  auto load = [&](u32x4 (&st)[kI], __amdgpu_buffer_rsrc_t r) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < kI; ++n)
      st[n] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, goff[n], 0, 0));
  };
  // kAppend: a page of the workgroup's own tokens (this head) goes to the pool as well.
  auto put = [&](const u32x4 (&st)[kI], const Tile& t, int64_t kv) __attribute__((always_inline)) {
    if constexpr (kAppend) {
      const int t0 = t.kt + kBPage * wave - query_start;
      if (t0 >= q0 && t0 < q0 + C::kQw && t.rows > 0) {  // (uniform)
        f16* d = ap.pool + int64_t(t.page) * page_elems + int64_t(kvh) * D + kv;
        const __amdgpu_buffer_rsrc_t w = __builtin_amdgcn_make_buffer_rsrc(d, 0, t.rows * tok_bytes, 0x00020000);
#pragma unroll
        for (int n = 0; n < kI; ++n)
          __builtin_amdgcn_raw_buffer_store_b128(st[n], w, goff[n], 0, 0);
      }
    }
  };
  auto load_k = [&](const Tile& t) __attribute__((always_inline)) { load(kst, page_rsrc(t, 0, ap.new_k)); };
  auto load_v = [&](const Tile& t) __attribute__((always_inline)) { load(vst, page_rsrc(t, v_off, ap.new_v)); };
  auto store_k = [&](const Tile& t, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < kI; ++n)
      *reinterpret_cast<lds_u32x4*>(lds + buf * C::kBufB + kwr + n * C::kRowsI * C::kKRowB) = kst[n];
    put(kst, t, 0);
  };
  auto store_v = [&](const Tile& t, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < kI; ++n)
      *reinterpret_cast<lds_u32x4*>(lds + buf * C::kBufB + vwr + n * C::kRowsI * C::kVRowB) = vst[n];
    put(vst, t, v_off);
  };

  // Fragment reads.  K: key row 32 j + col, chunk 2 s + half.  V: lane = 16 g + 4 rr + q4 reads row
  // 4 (lane / 32) + rr of a page half, dims 32 dt + 16 (g % 2) + 4 q4 .. + 3.
  const uint32_t kfrag = uint32_t(col * C::kKRowB + half * 16);
  const uint32_t vfrag = uint32_t(C::kKTileB + (4 * half + (lane % 16) / 4) * C::kVRowB + 32 * ((lane / 16) % 2) + 8 * (lane % 4));

  float m = kNegBig, lsum = 0.f;
  f32x16 acc[kDT];
#pragma unroll
  for (int dt = 0; dt < kDT; ++dt) acc[dt] = f32x16{};

  float cand;  // the row maximum of the tile scored last (log2 units)
  // Scores of a tile, K in buffer b.
  auto score = [&](f32x16 (&st)[2], const lds_u8* b) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int s = 0; s < kKS; ++s) {
        const f16x8 kf = as_h8(*reinterpret_cast<const lds_u32x4*>(b + kfrag + 32 * s + 32 * C::kKRowB * j));
        st[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qreg[s], s == 0 ? f32x16{} : st[j], 0, 0, 0);
      }
  };
  // Causal limit, end of the sequence, invalid pages: score r of half j is key
  // 32 j + 8 (r / 4) + 4 half + r % 4 of the tile.
  auto mask = [&](f32x16 (&st)[2], const Tile& ti) __attribute__((always_inline)) {
    if (!((ti.fl == 15) & (ti.kt + kBTile <= total) & (ti.kt + kBTile - 1 <= wave_first))) {
      const int lim = min(my_pos, total - 1) - ti.kt;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int c = 32 * j + 8 * (r / 4) + r % 4;
          const int lp = ((ti.fl >> (2 * j + r / 8)) & 1) ? lim - 4 * half : -1;
          st[j][r] = c <= lp ? st[j][r] : -INFINITY;
        }
    }
  };
  auto row_max = [&](const f32x16 (&st)[2]) __attribute__((always_inline)) {
    float mx[8];
#pragma unroll
    for (int a = 0; a < 8; ++a) {
      const f32x16& x = st[a / 4];
      const int o = 4 * (a % 4);
      mx[a] = fmaxf(fmaxf(x[o], x[o + 1]), fmaxf(x[o + 2], x[o + 3]));
    }
    cand = max_lane32(fmaxf(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3])),
                                fmaxf(fmaxf(mx[4], mx[5]), fmaxf(mx[6], mx[7])))) * scale_log2;
  };
  // Lazy rescale: the reference maximum moves only when a score exceeds it by more than 8 (log2
  // units), so P < 2^8.
  auto rescale = [&]() __attribute__((always_inline)) {
    const bool grow = cand > m + 8.f;
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
      const float mn = grow ? cand : m;
      const float alpha = exp2_fast(m - mn);
      lsum *= alpha;
#pragma unroll
      for (int dt = 0; dt < kDT; ++dt) acc[dt] *= alpha;
      m = mn;
    }
  };
  // Probabilities of keys 16 u .. 16 u + 15, in fp16 (what the second product multiplies and lsum adds).
  auto prob = [&](const f32x16 (&st)[2], int u) __attribute__((always_inline)) -> f16x8 {
    float e[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) e[r] = exp2_fast(fmaf(st[u / 2][8 * (u % 2) + r], scale_log2, -m));
    return f16x8{f16(e[0]), f16(e[1]), f16(e[2]), f16(e[3]), f16(e[4]), f16(e[5]), f16(e[6]), f16(e[7])};
  };
  auto add_row_sum = [&](const f16x8& p) __attribute__((always_inline)) {
    const f16x2 one = f16x2{f16(1.f), f16(1.f)};
#pragma unroll
    for (int e = 0; e < 4; ++e) lsum = __builtin_amdgcn_fdot2(f16x2{p[2 * e], p[2 * e + 1]}, one, lsum, false);
  };
  // O^T += V^T P^T for keys 16 u .. 16 u + 15, V in buffer b.
  auto pv = [&](const lds_u8* b, const f16x8& p, int u) __attribute__((always_inline)) {
#pragma unroll
    for (int dt = 0; dt < kDT; ++dt) {
      const lds_u8* a = b + vfrag + u * kBPage * C::kVRowB + 64 * dt;
      const f16x4 lo = __builtin_bit_cast(f16x4, ds_read_tr16(a));
      const f16x4 hi = __builtin_bit_cast(f16x4, ds_read_tr16(a + 8 * C::kVRowB));
      const f16x8 vf = f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, p, acc[dt], 0, 0, 0);
    }
  };

  // Step i: tile i + 1's scores beside tile i's probabilities, then tile i's second product beside
  // tile i + 1's maxima.  K of tile i + 2 and V of tile i + 1 go to the buffers that K of tile i and V
  // of tile i - 1 left at the barrier before; the loads of the next ones are issued.
  // (A wave's rows see nothing of its last tiles when other waves' rows end later: it only stages.)
  const int steps = int(ceil_div(n_tiles, KS));
  const int wave_tiles = min(n_tiles, int(ceil_div(wave_last + 1, kBTile)));
  const int wave_steps = wave_tiles > grp ? int(ceil_div(wave_tiles - grp, KS)) : 0;
  Tile t1, t2;  // tiles i + 1 and i + 2
  auto step = [&](f32x16 (&sc)[2], f32x16 (&sn)[2], int i) __attribute__((always_inline)) {
    store_k(t2, i & 1);
    store_v(t1, (i + 1) & 1);
    const Tile t3 = tile_at(i + 3);
    load_k(t3);
    load_v(t2);
    if (i < wave_steps) {
      rescale();
      // Half of the probabilities go beside the score MFMAs, half beside the second product, so that
      // neither runs matrix or vector work alone (2048 queries at 6144, 32 q heads: 286 -> 275 us).
      __builtin_amdgcn_sched_barrier(0);
      score(sn, lds + ((i + 1) & 1) * C::kBufB);
      f16x8 p[4];
      p[0] = prob(sc, 0);
      p[1] = prob(sc, 1);
      add_row_sum(p[0]);
      add_row_sum(p[1]);
      blk_pin(p[0], p[1]);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // K fragment reads, two ahead
#pragma unroll
      for (int x = 0; x < 2 * kKS; ++x) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // K fragment read
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // VALU
        __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);  // exp2
      }
      __builtin_amdgcn_sched_barrier(0);
      mask(sn, t1);
      const lds_u8* const vb = lds + (i & 1) * C::kBufB;
      pv(vb, p[0], 0);
      pv(vb, p[1], 1);
      p[2] = prob(sc, 2);
      p[3] = prob(sc, 3);
      pv(vb, p[2], 2);
      pv(vb, p[3], 3);
      add_row_sum(p[2]);
      add_row_sum(p[3]);
      row_max(sn);
    }
    t1 = t2;
    t2 = t3;
    lds_barrier();
  };
  f32x16 sa[2], sb[2];
  {
    const Tile t0 = tile_at(0);
    t1 = tile_at(1);
    t2 = tile_at(2);
    load_k(t0);
    load_v(t0);
    store_k(t0, 0);
    load_k(t1);
    store_v(t0, 0);
    load_v(t1);
    store_k(t1, 1);
    load_k(t2);
    lds_barrier();
    score(sa, lds);
    mask(sa, t0);
    row_max(sa);
    lds_barrier();  // every wave has left K of tile 0
  }
  for (int i = 0; i < steps; i += 2) {
    step(sa, sb, i);
    step(sb, sa, i + 1);
  }

  float l = lsum + __shfl_xor(lsum, 32);
  constexpr int kOwn = kDT / KS;  // output tiles this wave finishes: kOwn grp .. + kOwn - 1
  f32x16 o[kOwn];
  if constexpr (KS == 1) {
#pragma unroll
    for (int d = 0; d < kOwn; ++d) o[d] = acc[d];
  } else {
    // The two key groups of a row block merge through LDS (free: the last barrier has passed): each wave
    // hands over the output tiles its partner finishes, with (m, l).
    float* const mb = reinterpret_cast<float*>(smem);
    auto slot = [&](int g) __attribute__((always_inline)) { return mb + ((g * kBWaves + wave) * (16 * kOwn + 2)) * kWave + lane; };
    float* const mine = slot(grp);
    mine[0] = m;
    mine[kWave] = l;
#pragma unroll
    for (int d = 0; d < kOwn; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) mine[(2 + 16 * d + r) * kWave] = grp == 0 ? acc[kOwn + d][r] : acc[d][r];
    __syncthreads();
    const float* const other = slot(1 - grp);
    const float mo = other[0], lo = other[kWave];
    const float mm = fmaxf(m, mo), a = exp2_fast(m - mm), b = exp2_fast(mo - mm);
    l = fmaf(b, lo, a * l);
#pragma unroll
    for (int d = 0; d < kOwn; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        o[d][r] = fmaf(b, other[(2 + 16 * d + r) * kWave], a * (grp == 0 ? acc[d][r] : acc[kOwn + d][r]));
  }
  if (my_q >= T) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  f16* orow = out + (int64_t(my_q) * hq + my_head) * D + 32 * kOwn * grp;
#pragma unroll
  for (int d = 0; d < kOwn; ++d)
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4)
      *reinterpret_cast<f16x4*>(orow + 32 * d + 8 * r4 + 4 * half) = f16x4{
          f16(o[d][4 * r4] * inv), f16(o[d][4 * r4 + 1] * inv), f16(o[d][4 * r4 + 2] * inv), f16(o[d][4 * r4 + 3] * inv)};
}

typedef void (*BlockKernel)(f16*, const f16*, const f16*, int64_t, const int32_t*, int32_t, int32_t, int32_t, int32_t,
                            float, PrefillAppend);

static BlockKernel pick_block(int d, int g, int ks, bool append) {
#define IFN_BLOCK_CASE(DD, GG) \
  if (d == DD && g == GG)                                                                               \
    return ks == 2 ? (append ? prefill_block_kernel<DD, GG, 2, true> : prefill_block_kernel<DD, GG, 2, false>) \
                   : (append ? prefill_block_kernel<DD, GG, 1, true> : prefill_block_kernel<DD, GG, 1, false>);
  IFN_BLOCK_CASE(128, 1) IFN_BLOCK_CASE(128, 2) IFN_BLOCK_CASE(128, 4) IFN_BLOCK_CASE(128, 8)
#undef IFN_BLOCK_CASE
  return nullptr;
}

// Which chunks take this kernel, and on how many key groups, by n = its workgroups (128 rows of a kv
// head each) against the CUs (us, fused append unless noted, 8 kv heads x 128: wide kernel / one group /
// two groups):
//  * n > CUs: always.  n >= 2 CUs: one group, two workgroups per CU (32 q heads, 2048 queries at 0: 80.6 /
//    58.6 / 66.6).  Below: two groups where the causal limit leaves the blocks uneven (1280 queries at
//    0: 43.6 / 35.8 / 31.0), one where the blocks are about equal (at 2048: 117.4 / 92.2 / 96.4).
//  * CUs / 2 < n <= CUs, query_start >= T: two groups, one workgroup per CU (768 queries at 2048: 68.0 /
//    60.6 / 52.3; 600 at 2048, plain: 56.2 / 53.1 / 45.0).  With the chunk's own keys the larger part
//    the longest block would set the time (16 q heads, 1536 at 0, plain: 24.7 / 33.8 / 29.4).
//  * n <= CUs / 2: the wide kernel, which splits the rows finer (512 at 2048: 38.9 / 55.7 / 44.7).
// Head dim 64 gains nothing here (16 q heads, 8192 at 0, plain: 197 wide, 198 on one group).
int prefill_block_groups(int32_t T, int32_t query_start, int32_t hq, int32_t hkv, int32_t d, int cus) {
  if (pick_block(d, hq / hkv, 1, false) == nullptr) return 0;
  const int64_t n = ceil_div(int64_t(T) * (hq / hkv), 32 * kBWaves) * hkv;
  if (n > cus) return n >= 2 * cus || query_start >= T ? 1 : 2;
  return 2 * n > cus && query_start >= T ? 2 : 0;
}

int prefill_block_launch(f16* out, const f16* q, const f16* pool, int64_t num_pages, const int32_t* table,
                         int32_t query_start, int32_t T, int32_t hq, int32_t hkv, int32_t d, float scale_log2,
                         int groups, const PrefillAppend& ap, hipStream_t stream) {
  BlockKernel k = pick_block(d, hq / hkv, groups, ap.pool != nullptr);
  if (k == nullptr || (ap.pool != nullptr && query_start % kBPage != 0)) return IFN_ERR_UNSUPPORTED;
  const int64_t n_qb = ceil_div(int64_t(T) * (hq / hkv), 32 * kBWaves);
  if (n_qb * hkv >= int64_t(1) << 31) return IFN_ERR_UNSUPPORTED;
  k<<<dim3(unsigned(n_qb * hkv)), dim3(unsigned(groups * kBThreads)), 0, stream>>>(out, q, pool, num_pages, table, query_start, T, hkv,
                                                              int(n_qb), scale_log2, ap);
  return ifn_launch_status();
}

}  // namespace ifn
