// Device code shared by the d = 128 attention kernels (attn.hip: tile pairs,
// attn_solo.hip: single tiles): launch arguments, a wave's online-softmax state and the
// steps on it, direct global->LDS loads and their waits.
#pragma once

#include "common.h"

namespace spx {

constexpr int kMaxBlocksAttn = 1024;
constexpr int kTailTile = 64;        // mean keys per tail tile (hi and lo rows fill K LDS)
// log2 headroom before a column's running max moves. P is bf16 and O, l are fp32, all
// with an 8-bit exponent, so probabilities up to 2^64 lose nothing; O then keeps
// 2^128 / (2^64 * 2^17 keys at the 131072-token limit) = 2^47 of headroom for |v|.
// Sharp score profiles (routed sparse layers) move a column's maximum by tens of
// log2 units from block to block: at a headroom of 2^8 the rescale branch ran in
// about half of a sparse layer's sub-blocks, at 2^64 in under 3 %.
constexpr float kLazyRescale = 64.0f;


struct AttnArgs {
  const uint16_t* q;
  int64_t qs_b, qs_s, qs_h;
  const uint16_t* kt;  // key tiles   [B, Hkv, NB, 128, D]  (LDS order, from the pool pass)
  const uint16_t* vt;  // value tiles [B, Hkv, NB, D, 128]
  const int64_t* idx;  // nullable: all causal blocks
  int64_t is_b, is_t, is_p, is_h;
  const int32_t* cnt;
  int64_t cs_b, cs_t, cs_h;
  const float* mean_k;  // [B, NB, Hkv, D]
  const float* mean_v;
  const int32_t* bcounts;  // [NB]
  const uint8_t* choice;   // rescue token per (b, t, j, h): [B, NB, NB, Hq]
  const uint16_t* v;       // V [B, S, Hkv, D] (strided): rescue tokens' value rows
  int64_t vs_b, vs_s, vs_h;
  int tail_kind;           // 0 block means, 1 rescue token, 2 rescue token + remainder mean
  void* out;
  int64_t os_b, os_s, os_h;
  float* lse;  // nullable
  int64_t ls_b, ls_s, ls_h;
  int batch, seq, q_heads, kv_heads, blocks, group, num_pairs;
  int xcds_per_stream;   // XCDs sharing one (batch, kv group) stream; 1: pair p on XCD p % 8
  float scale_log2;
  // Persistent grid (a caller queue): one workgroup per CU takes items until none
  // are left (draw_item). Tile pairs [0, static_tp) are dealt to XCDs as in the static
  // grid and taken in order through XCD x's counter queue[1 + x]; the rest (the
  // lightest) go through the tail counters in heaviest-first order.
  int* queue;        // SPX_WORK_QUEUE_INTS zeroed int32 (null: one workgroup per item)
  int static_tp;     // tile pairs on the per-XCD deal (all of them without a queue)
  int steal;         // workgroups also take items of other XCDs' static shares
  int share_items;   // xcds_per_stream > 1: items of each XCD's static share
  int dyn_items;     // items behind each tail counter: (tile pair, head) of one stream
                     // (xcds_per_stream > 1), else (tile pair, stream, head)
};

__device__ __forceinline__ int swz(int row, int chunk) {
  return row * kBlock + ((chunk ^ (row & 15)) << 3);
}

__device__ __forceinline__ bf16x8 lds_read16(const uint16_t* lds, int off) {
  return as_bf16x8(*reinterpret_cast<const u32x4*>(lds + off));
}

__device__ __forceinline__ bf16x8 pack8(const f32x16& v, int base) {
  u32x4 w;
  w[0] = pack_bf16x2(v[base + 0], v[base + 1]);
  w[1] = pack_bf16x2(v[base + 2], v[base + 3]);
  w[2] = pack_bf16x2(v[base + 4], v[base + 5]);
  w[3] = pack_bf16x2(v[base + 6], v[base + 7]);
  return as_bf16x8(w);
}

// The running-max rescale multiplies the O accumulators in place from inline
// assembly (tied operands keep O in its registers across the rarely taken
// branch). The compiler's hazard recognizer does not look inside asm statements,
// so the wait states an MFMA that wrote O needs before VALU access to O are issued
// here, at the top of that branch: the products into O are issued before the
// branch (their results are live on both of its paths), so these wait states sit
// between the last product and the first multiply. 19 >= the 16-pass XDL write ->
// VALU read / write requirement of the gfx940 family (the 8-pass products here
// need fewer). Not tied to O: tying it changes how the loop is scheduled.
__device__ __forceinline__ void o_settle() { asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 2"); }

// Per-wave online-softmax state for its 32 query columns.
struct WaveState {
  bf16x8 qb[8];   // Q^T B operands, dim chunk dc
  f32x16 o[4];    // O^T accumulators, dim block db
  float m;        // running max (base-2, scaled), lazily moved
  float l;        // running sum over this lane half's keys
  float neg_m;    // full blocks: -m once set (0 before)
  float thr;      // full blocks: lazy-move threshold on shifted scores (-inf before m is set)
};

// Per-lane gather into LDS: 16 bytes from this lane's own address land at
// lds_wave + 16 x lane, lds_wave being the same for the whole wave. Issued from
// assembly like dma_part, and awaited explicitly.
__device__ __forceinline__ void dma_gather16(const void* src, uint32_t lds_wave) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds_wave);
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %2, off\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "s"(m0), "v"(src)
      : "memory");
}

// threadIdx.x behind an opaque copy: values derived from it are recomputed for
// every work item of a persistent workgroup instead of being held across items.
__device__ __forceinline__ int thread_x() { return opaque((int)threadIdx.x); }

__device__ __forceinline__ void wait_tiles() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// LDS element offset of this lane's MFMA operand row (row & 15 == col & 15 for
// every operand row it reads) with 16-byte chunk 2 x + half, for x = 0: the chunk
// for any other x is base ^ (x << 4) (XOR swizzle c ^ (row & 15), c = 2 x + half).
__device__ __forceinline__ int operand_base(int row) {
  const int lane = thread_x() & 63;
  const int col = lane & 31, half = lane >> 5;
  const int cx = (col >> 1) & 7, hb = half ^ (col & 1);
  return row * kBlock + (cx << 4) + (hb << 3);
}

// Compiler fence: nothing is scheduled across it. Keeps operand reads issued a
// step ahead of the MFMAs that consume them.
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

// S^T for NMB 32-key sub-blocks at K rows row0 + 32 mb + col (for hi/lo mean
// keys, also rows + kTailTile). The NMB (x2) operand reads of a dim chunk are
// issued one chunk ahead of their MFMAs.
template <int NMB, bool HILO>
__device__ __forceinline__ void scores(const uint16_t* kb, const WaveState& ws, int row0,
                                       f32x16 (&s)[4]) {
  constexpr int P = NMB * (HILO ? 2 : 1);
  const int col = thread_x() & 31;
  const int e0 = opaque(operand_base(row0 + col));
  auto row_off = [](int part) {
    return HILO ? ((part & 1) ? kTailTile * kBlock : 0) + (part >> 1) * 32 * kBlock
                : part * 32 * kBlock;
  };
  bf16x8 ring[2][P];
#pragma unroll
  for (int mb = 0; mb < NMB; ++mb) s[mb] = f32x16{};
#pragma unroll
  for (int p = 0; p < P; ++p) ring[0][p] = lds_read16(kb, e0 + row_off(p));
  fence();
#pragma unroll
  for (int dc = 0; dc < 8; ++dc) {
    if (dc + 1 < 8) {
      const int e = e0 ^ ((dc + 1) << 4);
#pragma unroll
      for (int p = 0; p < P; ++p) ring[(dc + 1) & 1][p] = lds_read16(kb, e + row_off(p));
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int mb = HILO ? (p >> 1) : p;
      s[mb] = mfma32(ring[dc & 1][p], ws.qb[dc], s[mb]);
    }
    fence();
  }
}

// Softmax of one tile: masks (DIAG) / per-key biases (BIAS, already scaled),
// lazily moved running max, probabilities packed to bf16 B operands pb[2 mb + h],
// running sum, O rescale when any lane moved its max.
template <int NMB, bool DIAG, bool BIAS>
__device__ __forceinline__ void softmax(f32x16 (&s)[4], WaveState& ws, float scale, int q_pos,
                                        const float* bias, int bias_row0, bf16x8 (&pb)[8]) {
  const int lane = thread_x() & 63;
  float mx = -INFINITY;
#pragma unroll
  for (int mb = 0; mb < NMB; ++mb) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float x = s[mb][r];
      if (BIAS) x = fmaf(x, scale, bias[bias_row0 + mb * 32 + mfma32_row(r, lane)]);
      if (DIAG && mb * 32 + mfma32_row(r, lane) > q_pos) x = -INFINITY;
      s[mb][r] = x;
      mx = fmaxf(mx, x);
    }
  }
  mx = fmaxf(mx, xor32(mx));
  const float mxs = BIAS ? mx : mx * scale;
  const float m_new = (mxs > ws.m + kLazyRescale) ? mxs : ws.m;
  if (__any(m_new != ws.m)) {
    const float corr = (m_new == ws.m) ? 1.0f : exp2_fast(ws.m - m_new);
    // in place (tied operands): O keeps its registers across the rarely taken
    // branch instead of being copied into a second set on every block
    o_settle();
#pragma unroll
    for (int db = 0; db < 4; ++db) {
#pragma unroll
      for (int r = 0; r < 16; ++r) asm volatile("v_mul_f32 %0, %0, %1" : "+v"(ws.o[db][r]) : "v"(corr));
    }
    ws.l *= corr;
    ws.m = m_new;
  }
  const float neg_m = (ws.m == -INFINITY) ? 0.0f : -ws.m;
  float sum = 0.0f;
#pragma unroll
  for (int mb = 0; mb < NMB; ++mb) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float p = BIAS ? exp2_fast(s[mb][r] + neg_m) : exp2_fast(fmaf(s[mb][r], scale, neg_m));
      s[mb][r] = p;
      sum += p;
    }
    pb[2 * mb] = pack8(s[mb], 0);
    pb[2 * mb + 1] = pack8(s[mb], 8);
  }
  ws.l += sum;
}

__device__ __forceinline__ uint32_t lds_address(const uint16_t* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint16_t*)p;
}

__device__ __forceinline__ bf16x8 lds_at(uint32_t byte_address) {
  const u32x4 v =
      *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>((uintptr_t)byte_address);
  return as_bf16x8(v);
}

// scores of one sub-block: S^T = K_mb Q^T (8 chained MFMAs over the dim chunks)
__device__ __forceinline__ void sub_scores(const bf16x8 (&r)[8], const WaveState& ws, f32x16& acc) {
  acc = f32x16{};
#pragma unroll
  for (int dc = 0; dc < 8; ++dc) acc = mfma32(r[dc], ws.qb[dc], acc);
}

__device__ __forceinline__ void sub_pv(const bf16x8 (&r)[8], const bf16x8 (&p)[2], WaveState& ws) {
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int db = 0; db < 4; ++db) ws.o[db] = mfma32(r[h * 4 + db], p[h], ws.o[db]);
}

// Shift one sub-block's scores in place to x = s * scale + ws.neg_m (this lane's
// 16 keys of its column) and check them against the running max. The max runs
// over the shifted values: results of arithmetic, which the compiler's max takes
// without quieting them first. The running max moves lazily: only when a
// column's x exceeds ws.thr (2^64 once set); then (rarely) O and l are rescaled
// and x shifted by the same amount. Before the first move neg_m is 0 and thr
// -inf, so the first sub-block sets the max from its own scores. The common path
// checks each lane half's own max; the column max over both halves is formed
// only in the rare branch.
__device__ __forceinline__ void shift_and_check(f32x16& sv, WaveState& ws, float scale) {
#pragma unroll
  for (int r = 0; r < 16; ++r) sv[r] = fmaf(sv[r], scale, ws.neg_m);
  // each lane half checks its own 8 + 8 keys; only when some lane exceeds the
  // threshold is the column max of both halves formed
  float mx = fmaxf(fmaxf(sv[0], sv[1]), sv[2]);
#pragma unroll
  for (int r = 3; r < 15; r += 2) mx = fmaxf(fmaxf(mx, sv[r]), sv[r + 1]);
  mx = fmaxf(mx, sv[15]);
  if (__any(mx > ws.thr)) {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx),
                                                     false, false);
    mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    const bool move = mx > ws.thr;
    const float d = move ? mx : 0.0f;
    // nothing is accumulated before the first move (thr -inf): O and l stay 0
    const float corr = ws.thr == -INFINITY ? 0.0f : exp2_fast(-d);
    // in place (tied operands): O keeps its registers across the rarely taken branch
    o_settle();
#pragma unroll
    for (int db = 0; db < 4; ++db) {
#pragma unroll
      for (int r = 0; r < 16; ++r) asm volatile("v_mul_f32 %0, %0, %1" : "+v"(ws.o[db][r]) : "v"(corr));
    }
    ws.l *= corr;
    ws.neg_m -= d;
    if (move) ws.thr = kLazyRescale;
#pragma unroll
    for (int r = 0; r < 16; ++r) sv[r] -= d;
  }
}

// probabilities of one sub-block (shifted scores x) as bf16 B operands; the
// running sum adds the fp32 probabilities, as upstream/flashprefill_native_forward.py
// :332-338 does (sum before the cast for the P V product), pairwise so that the
// chain into l is short. (Summing the packed bf16 pairs with v_dot2_f32_bf16 instead
// took issue cycles from the matrix products beside it: four per product halved
// their rate in a microbenchmark, while plain adds there were nearly free.)
__device__ __forceinline__ void sub_exp(const f32x16& xv, WaveState& ws, bf16x8 (&p)[2]) {
  float pair_sum[8];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    u32x4 w;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a = exp2_fast(xv[8 * h + 2 * i]);
      const float b = exp2_fast(xv[8 * h + 2 * i + 1]);
      w[i] = pack_bf16x2(a, b);
      pair_sum[4 * h + i] = a + b;
    }
    p[h] = as_bf16x8(w);
  }
  const float sum = ((pair_sum[0] + pair_sum[1]) + (pair_sum[2] + pair_sum[3])) +
                    ((pair_sum[4] + pair_sum[5]) + (pair_sum[6] + pair_sum[7]));
  ws.l += sum;
}

// Natural-log LSE of a row with base-2 maximum m and probability sum l (contracted by
// hand: left to the compiler, the kernels differed in its last bit).
__device__ __forceinline__ float natural_lse(float m, float l) { return fmaf(m, kLn2, logf(l)); }

}  // namespace spx
