// Block-sparse causal attention at head_dim 128, one query tile per workgroup: the
// semantics and the arithmetic of attn.hip (same results bit for bit on ascending lists),
// split finer.
//
// attn.hip gives a CU one workgroup of eight waves with two adjacent query tiles; this
// kernel gives it two independent workgroups of four waves with one tile each, dealt by
// the hardware as slots come free:
//   * what a workgroup spends outside the block loop (its lists, the wait for Q and for
//     the first K / V tile, the diagonal block, the tail's staging, the output) runs
//     beside the other workgroup's products instead of leaving the CU idle;
//   * a tile walks its own list only, not the union with its neighbour's;
//   * items are half as long, so short launches spread over the CUs.
// Against that, K and V are copied into LDS once per tile instead of once per two.
//
// LDS per workgroup must stay under 80 KB, so blocks stream in 64-key halves (16 KB of K
// rows, 16 KB of V^T) through two buffer pairs, half h of a block always in pair h; the
// software pipeline over 32-key sub-blocks (attn.hip) carries on across the halves.
// A half's V is 128 contiguous bytes of each 256-byte dim row of the value tile: the
// swizzle c ^ (d & 15) keeps the 8 chunks of a half together, in the half h ^ (d >> 3 & 1)
// of the row, so a copy instruction reads whole cache lines and LDS row d holds chunk c of
// the half at (c & 7) ^ (d & 7).
#include <type_traits>

#include "attn_solo.h"

namespace spx {

constexpr int kSoloThreads = 256;                       // four waves of 32 query rows
constexpr int kSoloLoads = kMaxBlocksAttn / kSoloThreads;   // list positions per thread
constexpr int kHalfKeys = 64;
constexpr int kHalfElems = kHalfKeys * kHeadDim;
constexpr uint32_t kHalfBytes = kHalfElems * 2;         // K rows or V^T of one half

// Byte addresses in LDS of this lane's operand rows, buffer pair 0: k[c] chunk pair c of
// key row col; v[x] chunk 2 x + half of dim row col.
struct SoloTables {
  uint32_t k[8];
  uint32_t v[4];
};

__device__ __forceinline__ int solo_value_base(int col, int chunk) {
  return col * kHalfKeys + ((chunk ^ (col & 7)) << 3);
}

__device__ __forceinline__ SoloTables solo_tables(const uint16_t* k0, const uint16_t* v0) {
  SoloTables t;
  const int lane = thread_x() & 63;
  const int col = lane & 31, half = lane >> 5;
  const int e0 = operand_base(col);
  const uint32_t kb = lds_address(k0), vb = lds_address(v0);
#pragma unroll
  for (int c = 0; c < 8; ++c) t.k[c] = (uint32_t)opaque((int)(kb + (uint32_t)(e0 ^ (c << 4)) * 2u));
#pragma unroll
  for (int x = 0; x < 4; ++x)
    t.v[x] = (uint32_t)opaque((int)(vb + (uint32_t)solo_value_base(col, 2 * x + half) * 2u));
  return t;
}

template <int BUF>
__device__ __forceinline__ void solo_keys(const SoloTables& tb, int mb, bf16x8 (&r)[8]) {
#pragma unroll
  for (int dc = 0; dc < 8; ++dc) r[dc] = lds_at(tb.k[dc] + BUF * kHalfBytes + mb * 32 * kHeadDim * 2);
}

template <int BUF>
__device__ __forceinline__ void solo_values(const SoloTables& tb, int j, bf16x8 (&r)[8]) {
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int db = 0; db < 4; ++db)
      r[h * 4 + db] = lds_at(tb.v[2 * j + h] + BUF * kHalfBytes + db * 32 * kHalfKeys * 2);
}

// One unmasked half block in buffer pair BUF: two sub-blocks of attn.hip's full_block.
template <int BUF>
__device__ __forceinline__ void full_half(const SoloTables& tb, WaveState& ws, float scale,
                                          bf16x8 (&rv)[8], bf16x8 (&pend)[2]) {
  f32x16 s[2];
  bf16x8 p[2];
  bf16x8 rk[8];
  solo_keys<BUF>(tb, 0, rk);
  fence();
  sub_pv(rv, pend, ws);
  sub_scores(rk, ws, s[0]);
  fence();
  solo_keys<BUF>(tb, 1, rk);
  fence();
  shift_and_check(s[0], ws, scale);
  fence();
  solo_values<BUF>(tb, 0, rv);
  fence();
  sub_scores(rk, ws, s[1]);
  sub_exp(s[0], ws, p);
  fence();
  sub_pv(rv, p, ws);
  shift_and_check(s[1], ws, scale);
  fence();
  solo_values<BUF>(tb, 1, rv);
  fence();
  sub_exp(s[1], ws, pend);
}

// O^T += V^T P^T over NKC 16-key chunks; chunks 4.. in buffer pair 1.
template <int NKC>
__device__ __forceinline__ void solo_pv(const uint16_t* v0, WaveState& ws, const bf16x8 (&pb)[8]) {
  const int lane = thread_x() & 63;
  const int col = lane & 31, half = lane >> 5;
#pragma unroll
  for (int kc = 0; kc < NKC; ++kc) {
    const uint16_t* v = v0 + (kc >> 2) * kHalfElems + solo_value_base(col, 2 * (kc & 3) + half);
    bf16x8 r[4];
#pragma unroll
    for (int db = 0; db < 4; ++db) r[db] = lds_read16(v, db * 32 * kHalfKeys);
#pragma unroll
    for (int db = 0; db < 4; ++db) ws.o[db] = mfma32(r[db], pb[kc], ws.o[db]);
    fence();
  }
}

template <int NMB>
__device__ __forceinline__ void solo_diagonal(const uint16_t* k0, const uint16_t* v0, WaveState& ws,
                                              float scale, int q_pos) {
  f32x16 s[4];
  bf16x8 pb[8];
  scores<NMB, false>(k0, ws, 0, s);
  softmax<NMB, true, false>(s, ws, scale, q_pos, nullptr, 0, pb);
  solo_pv<2 * NMB>(v0, ws, pb);
}

// 16 KB into LDS, 16 bytes per thread and instruction: `src` uniform, `voff` this
// lane's byte offset, `step` elements per instruction.
__device__ __forceinline__ void dma_half(const uint16_t* src, uint32_t voff, int step,
                                         uint16_t* lds, int w) {
  const uint32_t base = lds_address(lds) + (uint32_t)w * 1024u;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t m0 = __builtin_amdgcn_readfirstlane(base + (uint32_t)i * 4096u);
    const uint16_t* s = src + i * step;
    uint32_t saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %2, %3\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved)
        : "s"(m0), "v"(voff), "s"(s)
        : "memory");
  }
}

// ---- tail staging: 64 entries, keys as bf16 hi / lo rows in the two K buffers, values
// in V buffer 0, logit bias. The first two waves make keys, the others values, each
// thread 8 entries x one 8-dim chunk with all its loads in flight; a value thread's
// entries are those of one 8-slot chunk, so it writes whole 16-byte chunks.
constexpr int kTailEntries = 8;

__device__ __forceinline__ int tail_entry(bool value, int sc, int m) {
  return value ? 16 * (sc >> 1) + 4 * (sc & 1) + (m & 3) + 8 * (m >> 2) : 8 * sc + m;
}

__device__ __forceinline__ void write_tail(bool value, uint16_t* kb, uint16_t* vb, int sc, int c,
                                           const float (&x)[kTailEntries][8]) {
  if (value) {
#pragma unroll
    for (int y = 0; y < 8; ++y) {
      u32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = pack_bf16x2(x[2 * e][y], x[2 * e + 1][y]);
      *reinterpret_cast<u32x4*>(vb + (c * 8 + y) * kHalfKeys + ((sc ^ y) << 3)) = w;
    }
  } else {
#pragma unroll
    for (int m = 0; m < kTailEntries; ++m) {
      u32x4 hi, lo;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t h2 = pack_bf16x2(x[m][2 * e], x[m][2 * e + 1]);
        hi[e] = h2;
        lo[e] = pack_bf16x2(x[m][2 * e] - bf16_lo(h2), x[m][2 * e + 1] - bf16_hi(h2));
      }
      *reinterpret_cast<u32x4*>(kb + swz(8 * sc + m, c)) = hi;
      *reinterpret_cast<u32x4*>(kb + swz(kTailTile + 8 * sc + m, c)) = lo;
    }
  }
}

// Block means (attn.hip: stage_tail): key mean K, value mean V, bias ln n_j.
__device__ __forceinline__ void solo_stage_means(const AttnArgs& a, const int16_t* ids, int ntail,
                                                 int t0, int64_t desc_base, uint16_t* kb,
                                                 uint16_t* vb, float* bias, int tid) {
  const bool value = tid >= 128;
  const int c = tid & 15, sc = (tid >> 4) & 7;
  const float* src = value ? a.mean_v : a.mean_k;
  float x[kTailEntries][8];
#pragma unroll
  for (int m = 0; m < kTailEntries; ++m) {
    const int j = ids[min(t0 + tail_entry(value, sc, m), ntail - 1)];   // past the end: zeroed below
    load8(src + (desc_base + (int64_t)j * a.kv_heads) * kHeadDim + c * 8, x[m]);
  }
  if (tid < kTailTile)
    bias[tid] = t0 + tid < ntail ? logf((float)a.bcounts[ids[t0 + tid]]) * kLog2e : -INFINITY;
#pragma unroll
  for (int m = 0; m < kTailEntries; ++m) {
    const bool past = t0 + tail_entry(value, sc, m) >= ntail;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[m][e] = past ? 0.0f : x[m][e];
  }
  write_tail(value, kb, vb, sc, c, x);
}

// Rescue tokens (attn.hip: stage_rescue), epb entries per block.
__device__ __forceinline__ void solo_stage_rescue(const AttnArgs& a, const int16_t* ids, int ntail,
                                                  int t0, int epb, int b, int g, int h, int t,
                                                  uint16_t* kb, uint16_t* vb, float* bias, int tid) {
  const int64_t tile_elems = (int64_t)kBlock * kHeadDim;
  const bool value = tid >= 128;
  const int c = tid & 15, sc = (tid >> 4) & 7;
  const uint8_t* choice = a.choice + ((int64_t)b * a.blocks + t) * a.blocks * a.q_heads + h;
  const uint16_t* kt = a.kt + ((int64_t)b * a.kv_heads + g) * a.blocks * tile_elems;
  const uint16_t* vg = a.v + b * a.vs_b + g * a.vs_h + c * 8;
  const float* mean = value ? a.mean_v : a.mean_k;
  int id[kTailEntries], tok[kTailEntries];
  u32x4 raw[kTailEntries];
#pragma unroll
  for (int m = 0; m < kTailEntries; ++m)
    id[m] = ids[min(t0 + tail_entry(value, sc, m) / epb, ntail - 1)];
#pragma unroll
  for (int m = 0; m < kTailEntries; ++m) tok[m] = choice[(int64_t)id[m] * a.q_heads];
#pragma unroll
  for (int m = 0; m < kTailEntries; ++m) {
    const uint16_t* p = value ? vg + ((int64_t)id[m] * kBlock + tok[m]) * a.vs_s
                              : kt + id[m] * tile_elems + tok[m] * kHeadDim + ((c ^ (tok[m] & 15)) << 3);
    raw[m] = *reinterpret_cast<const u32x4*>(p);
  }
  float x[kTailEntries][8];
#pragma unroll
  for (int m = 0; m < kTailEntries; ++m) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[m][2 * e] = bf16_lo(raw[m][e]);
      x[m][2 * e + 1] = bf16_hi(raw[m][e]);
    }
    const int i = tail_entry(value, sc, m);
    if (epb == 2 && (i & 1)) {
      float mean8[8];
      load8(mean + (((int64_t)b * a.blocks + id[m]) * a.kv_heads + g) * kHeadDim + c * 8, mean8);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        x[m][e] = (mean8[e] * (float)kBlock - x[m][e]) / (float)(kBlock - 1);
    }
    const bool past = t0 + i / epb >= ntail;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[m][e] = past ? 0.0f : x[m][e];
  }
  if (tid < kTailTile)
    bias[tid] = t0 + tid / epb >= ntail ? -INFINITY
                : epb == 2 && (tid & 1) ? logf((float)(kBlock - 1)) * kLog2e
                                        : 0.0f;
  write_tail(value, kb, vb, sc, c, x);
}

// Workgroup i runs on XCD i % 8. A unit is the q heads of one (tile, batch, kv group),
// consecutive on one XCD so that they share K and V in its L2; units go heaviest tile
// first and the kv group rotates with the tile, so that every XCD serves every stream
// (lists differ in length between heads).
template <bool TAIL>
__global__ __launch_bounds__(kSoloThreads, 2) void attn_solo_kernel(AttnArgs a) {
  const int bg = a.batch * a.kv_heads;
  const int local = (int)(blockIdx.x >> 3);
  const int unit = (local / a.group) * 8 + (int)(blockIdx.x & 7);
  if (unit >= a.blocks * bg) return;
  const int hg = local % a.group;
  const int rank = unit / bg;
  const int s = (unit + (bg < 8 ? rank * bg / 8 : rank)) % bg;
  const int t = a.blocks - 1 - rank;
  const int b = s / a.kv_heads, g = s % a.kv_heads, h = g * a.group + hg;

  __shared__ __align__(16) uint16_t kbuf[2][kHalfElems];
  __shared__ __align__(16) uint16_t vbuf[2][kHalfElems];
  __shared__ int16_t list[kMaxBlocksAttn + 1];        // listed blocks but t, then t
  __shared__ int16_t tlist[TAIL ? kMaxBlocksAttn : 1];
  __shared__ uint32_t listed[TAIL ? kMaxBlocksAttn / 32 : 1];
  __shared__ float tail_bias[TAIL ? kTailTile : 1];
  __shared__ int wave_full[kSoloLoads][4], wave_diag[4];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int q_pos = w * 32 + col;
  const float scale = a.scale_log2;

  // Q as whole 256-byte rows into buffer pair 1: rows 0-63 in K, 64-127 in V, 16-byte
  // chunk c of row r at c ^ (r & 15)
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int e = i * kSoloThreads + tid, r = e >> 4, cs = e & 15;
    const int64_t row = min((int64_t)t * kBlock + r, (int64_t)a.seq - 1);   // past the end: not stored
    const uint16_t* src = a.q + b * a.qs_b + row * a.qs_s + h * a.qs_h + ((cs ^ (r & 15)) << 3);
    dma_gather16(src, lds_address(i < 4 ? kbuf[1] : vbuf[1]) +
                          (uint32_t)(((i & 3) * kSoloThreads + w * 64) * 16));
  }
  // the list, in its order: blocks other than t (attended unmasked), and how often t
  int count = t + 1;
  int64_t entry[kSoloLoads];
  if (a.idx) {
    count = max(0, min(a.cnt[b * a.cs_b + t * a.cs_t + h * a.cs_h], a.blocks));
    const int64_t* src = a.idx + b * a.is_b + t * a.is_t + h * a.is_h;
#pragma unroll
    for (int r = 0; r < kSoloLoads; ++r)
      entry[r] = src[min(tid + r * kSoloThreads, max(count, 1) - 1) * a.is_p];
  } else {
#pragma unroll
    for (int r = 0; r < kSoloLoads; ++r) entry[r] = tid + r * kSoloThreads;
  }
  if (TAIL && tid < kMaxBlocksAttn / 32) listed[tid] = 0u;
  uint64_t full[kSoloLoads];
  int diag = 0;
#pragma unroll
  for (int r = 0; r < kSoloLoads; ++r) {
    const int64_t j = entry[r];
    const bool ok = tid + r * kSoloThreads < count && j >= 0 && j < a.blocks;
    full[r] = __ballot(ok && j != t);
    diag += __popcll(__ballot(ok && j == t));
    if (lane == 0) wave_full[r][w] = __popcll(full[r]);
  }
  if (lane == 0) wave_diag[w] = diag;
  block_sync();
  int n_full = 0;
#pragma unroll
  for (int r = 0; r < kSoloLoads; ++r) {
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      if (x == w && ((full[r] >> lane) & 1ull)) {
        const int j = (int)entry[r];
        list[n_full + __popcll(full[r] & ((1ull << lane) - 1ull))] = (int16_t)j;
        if (TAIL) atomicOr(&listed[j >> 5], 1u << (j & 31));
      }
      n_full += wave_full[r][x];
    }
  }
  n_full = __builtin_amdgcn_readfirstlane(n_full);
  const int n_diag = __builtin_amdgcn_readfirstlane(wave_diag[0] + wave_diag[1] + wave_diag[2] +
                                                    wave_diag[3]);
  if (tid == 0) list[n_full] = (int16_t)t;
  wait_tiles();   // this wave's share of the Q copy (visible to all after the barrier)
  block_sync();

  const int64_t tile_elems = (int64_t)kBlock * kHeadDim;
  const int64_t kv0 = ((int64_t)b * a.kv_heads + g) * a.blocks;
  const uint16_t* kbase = a.kt + kv0 * tile_elems;
  const uint16_t* vbase = a.vt + kv0 * tile_elems + (w & 1) * kHalfKeys;
  const uint32_t koff = (uint32_t)tid * 16u;
  const uint32_t voff = (uint32_t)((tid >> 3) * 256 + (tid & 7) * 16);
  // half H of block j into buffer pair H (dim rows 8 .. 15 mod 16, the odd waves' rows,
  // have their halves exchanged)
  auto copy_half = [&](int j, auto hh) {
    constexpr int H = decltype(hh)::value;
    const int64_t off = (int64_t)j * tile_elems;
    dma_half(kbase + off + H * kHalfElems, koff, kSoloThreads * 8, kbuf[H], w);
    dma_half(H ? vbase + off + ((w & 1) ? -kHalfKeys : kHalfKeys) : vbase + off, voff,
             32 * kBlock, vbuf[H], w);
  };
  using H0 = std::integral_constant<int, 0>;
  using H1 = std::integral_constant<int, 1>;
  if (n_full + n_diag > 0) copy_half(__builtin_amdgcn_readfirstlane(list[0]), H0{});

  WaveState ws;
  {
    const uint16_t* qs = w < 2 ? kbuf[1] : vbuf[1];
    const int r = q_pos & 63;
#pragma unroll
    for (int dc = 0; dc < 8; ++dc)
      ws.qb[dc] = as_bf16x8(
          *reinterpret_cast<const u32x4*>(qs + (r * 16 + ((2 * dc + half) ^ (r & 15))) * 8));
    ws.m = -INFINITY;
    ws.l = 0.0f;
    ws.neg_m = 0.0f;
    ws.thr = -INFINITY;
#pragma unroll
    for (int db = 0; db < 4; ++db) ws.o[db] = f32x16{};
  }
  const SoloTables tables = solo_tables(kbuf[0], vbuf[0]);
  bf16x8 rv[8], pend[2];   // the pending P V product of the last half (zeros: adds nothing)
#pragma unroll
  for (int i = 0; i < 8; ++i) rv[i] = bf16x8{};
  pend[0] = pend[1] = bf16x8{};
  for (int e = 0; e < n_full; ++e) {
    const int j = __builtin_amdgcn_readfirstlane(list[e]);
    const int jn = __builtin_amdgcn_readfirstlane(list[e + 1]);
    const bool more = e + 1 < n_full || n_diag > 0;
    wait_tiles();
    block_sync();   // half 0 of block e visible; every wave is done with pair 1
    copy_half(j, H1{});
    full_half<0>(tables, ws, scale, rv, pend);
    wait_tiles();
    block_sync();
    if (more) copy_half(jn, H0{});
    full_half<1>(tables, ws, scale, rv, pend);
  }
  sub_pv(rv, pend, ws);
  if (ws.thr != -INFINITY) ws.m = -ws.neg_m;   // the max the unmasked blocks settled on
  block_sync();     // every wave is done with pair 1
  if (n_diag > 0) {
    copy_half(t, H1{});
    wait_tiles();
    block_sync();
#pragma unroll 1
    for (int k = 0; k < n_diag; ++k) {
      switch (w) {   // wave w reaches key sub-blocks 0 .. w of the diagonal block
        case 0: solo_diagonal<1>(kbuf[0], vbuf[0], ws, scale, q_pos); break;
        case 1: solo_diagonal<2>(kbuf[0], vbuf[0], ws, scale, q_pos); break;
        case 2: solo_diagonal<3>(kbuf[0], vbuf[0], ws, scale, q_pos); break;
        default: solo_diagonal<4>(kbuf[0], vbuf[0], ws, scale, q_pos); break;
      }
    }
    block_sync();   // every wave is done with the diagonal block
  }

  if constexpr (TAIL) {
    // the tail: history blocks j < t not listed, ascending
    int ntail = 0;
    for (int j0 = 0; j0 < t; j0 += kSoloThreads) {
      const int j = j0 + tid;
      const bool in = j < t && !((listed[(j & (kMaxBlocksAttn - 1)) >> 5] >> (j & 31)) & 1u);
      const uint64_t m = __ballot(in);
      if (lane == 0) wave_diag[w] = __popcll(m);
      block_sync();
      int offset = ntail;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        if (x < w) offset += wave_diag[x];
        ntail += wave_diag[x];
      }
      if (in) tlist[offset + __popcll(m & ((1ull << lane) - 1ull))] = (int16_t)j;
      block_sync();
    }
    ntail = __builtin_amdgcn_readfirstlane(ntail);
    const int epb = a.tail_kind == 2 ? 2 : 1;   // tail entries per unselected block
    for (int t0 = 0; t0 < ntail; t0 += kTailTile / epb) {
      if (t0 > 0) block_sync();   // every wave is done with the previous tail tile
      const int tx = thread_x();
      if (a.tail_kind == 0)
        solo_stage_means(a, tlist, ntail, t0, (int64_t)b * a.blocks * a.kv_heads + g, kbuf[0],
                         vbuf[0], tail_bias, tx);
      else
        solo_stage_rescue(a, tlist, ntail, t0, epb, b, g, h, t, kbuf[0], vbuf[0], tail_bias, tx);
      block_sync();
      f32x16 sc[4];
      bf16x8 pb[8];
      scores<2, true>(kbuf[0], ws, 0, sc);
      softmax<2, false, true>(sc, ws, scale, q_pos, tail_bias, 0, pb);
      solo_pv<4>(vbuf[0], ws, pb);
    }
    block_sync();   // every wave is done with the buffers
  }

  // ---- epilogue: as attn.hip, each wave's 32 x 128 rows through 8 KB of the K buffers
  const float l = ws.l + xor32(ws.l);
  const bool any = l > 0.0f;
  const float inv = any ? 1.0f / l : 0.0f;
  const int tx = thread_x();
  const int wq = tx >> 6, half_e = (tx >> 5) & 1, col_e = tx & 31, lane_e = tx & 63;
  uint16_t* stage = &kbuf[0][0] + __builtin_amdgcn_readfirstlane(wq) * (32 * kBlock);
#pragma unroll
  for (int db = 0; db < 4; ++db) {
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      u32x2 v2;
      v2[0] = pack_bf16x2(ws.o[db][4 * rr] * inv, ws.o[db][4 * rr + 1] * inv);
      v2[1] = pack_bf16x2(ws.o[db][4 * rr + 2] * inv, ws.o[db][4 * rr + 3] * inv);
      const int c = db * 4 + rr;
      *reinterpret_cast<u32x2*>(stage + col_e * kBlock + ((c ^ (col_e & 15)) << 3) + 4 * half_e) = v2;
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int r = 4 * i + (lane_e >> 4), c = lane_e & 15;
    const u32x4 v4 = *reinterpret_cast<const u32x4*>(stage + r * kBlock + ((c ^ (r & 15)) << 3));
    const int64_t row = (int64_t)t * kBlock + wq * 32 + r;
    if (row < a.seq)   // non-temporal, as attn.hip
      __builtin_nontemporal_store(
          v4, reinterpret_cast<u32x4*>(static_cast<uint16_t*>(a.out) + b * a.os_b + row * a.os_s +
                                       h * a.os_h + c * 8));
  }
  const int64_t qrow = (int64_t)t * kBlock + wq * 32 + col_e;
  if (a.lse && qrow < a.seq && half_e == 0)
    a.lse[b * a.ls_b + qrow * a.ls_s + h * a.ls_h] = any ? natural_lse(ws.m, l) : -INFINITY;
}

void launch_attn_solo(const AttnArgs& a, bool tail, hipStream_t st) {
  const int units = a.blocks * a.batch * a.kv_heads;
  const unsigned grid = (unsigned)((units + 7) / 8) * 8u * (unsigned)a.group;
  if (tail) attn_solo_kernel<true><<<grid, kSoloThreads, 0, st>>>(a);
  else attn_solo_kernel<false><<<grid, kSoloThreads, 0, st>>>(a);
}

}  // namespace spx
