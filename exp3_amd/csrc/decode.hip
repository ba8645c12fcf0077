// One decode step: attention of a single query row per head over a KV cache (bf16
// inputs and output, fp32 softmax and accumulation), the non-prefill branch of
// attention.py:179-189.
//
// Bound: HBM. A step reads K and V once (67 MB behind a 32K prompt at 28/4 heads,
// D = 128) and does 4 FLOP per byte or less, so what matters is enough bytes in flight
// on all CUs and a short chain.
//   * The keys are split over workgroups (four waves) as well as over (batch, KV head)
//     streams, all q heads of a KV head together, so K and V are read once. Each wave
//     takes 8192 / D keys per step, with all K and V loads of a step (32 KB) issued
//     before the first use; at 32K a wave runs one step and a CU has eight waves.
//   * Scores: S^T = K Q^T with v_mfma_f32_16x16x32_bf16, K rows straight from global
//     memory in the A operand layout (no LDS), up to 16 q heads of a group as columns.
//   * P V in fp32: v_mfma_f32_16x16x4_f32 takes one fp32 value per lane, and register r
//     of the scores (key 4 (lane / 16) + r, query lane % 16) is its A operand as it is.
//     B operand: the lane's bf16 values of that key widened, each V load reading whole
//     rows (16 bytes per lane; product i covers dims 8 c + i). No transposes, no
//     shuffles, no rounding of P; the fp32 rate is enough (0.5 GFLOP at 32K).
//   * The four waves' (max, sum, O) merge in LDS; with more than one split a second
//     kernel merges the splits' fp32 partials.
// Measured (28/4 heads, one sequence; SDPA, which runs one workgroup per head, before; in
// brackets the bytes at the 6.2 TB/s of a pass over 1 GB that only reads; a device copy
// moves 5.0): 32641 keys 1156 -> 19 us for both kernels, 15.9 + 4.0 (10.8), 131072 keys
// 4580 -> 53 us (43), 4096 keys 150 -> 11 us in a graph (1.4); 8 x 16000 keys at 32/8 heads
// 630 -> 104 us (85); D = 256, 16/4 heads, 32641 keys 1660 -> 32 us (21.6).
#include <algorithm>

#include "common.h"

namespace spx {

constexpr int kDecodeThreads = 256;
constexpr int kDecodeWaves = kDecodeThreads / 64;
constexpr int kDecodeHeads = 16;         // q heads per workgroup (MFMA columns)
constexpr int kDecodeMaxSplits = 256;

template <int D>
struct DecodeShape {
  static constexpr int kTiles = 512 / D;                  // 16-key tiles per wave and step
  static constexpr int kWaveKeys = 16 * kTiles;
  static constexpr int kStepKeys = kWaveKeys * kDecodeWaves;
};

struct DecodeArgs {
  const uint16_t* q;
  int64_t qs_b, qs_h;
  const uint16_t* k;
  int64_t ks_b, ks_h, ks_s;
  const uint16_t* v;
  int64_t vs_b, vs_h, vs_s;
  uint16_t* out;             // [B, Hq, D] contiguous
  float* part_o;             // [B Hq, splits, D]
  float* part_ml;            // [B Hq, splits, 2]
  int batch, seq, q_heads, kv_heads, group, head_tiles;
  int splits, steps;         // key ranges of `steps` steps each
  float scale_log2;
};

__device__ __forceinline__ f32x4 mfma16(const bf16x8& a, const bf16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Weight of a partial with maximum m in a merge with maximum top: an empty partial
// (m = -inf) counts nothing, also where every partial is empty.
__device__ __forceinline__ float merge_weight(float m, float top) {
  return m == -INFINITY ? 0.0f : exp2_fast(m - top);
}

template <int D>
__global__ __launch_bounds__(kDecodeThreads, 2) void decode_split_kernel(DecodeArgs a) {
  using Shape = DecodeShape<D>;
  constexpr int T = Shape::kTiles;
  constexpr int KK = D / 32;      // score products per tile
  constexpr int H = D / 128;      // 128-dim halves of a V row
  __shared__ float part_m[kDecodeWaves][kDecodeHeads], part_l[kDecodeWaves][kDecodeHeads];
  __shared__ __align__(16) float part_o[kDecodeWaves][kDecodeHeads][D];

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int split = blockIdx.x;
  const int stream = blockIdx.y / a.head_tiles;
  const int h0 = (blockIdx.y % a.head_tiles) * kDecodeHeads;   // first q head of the group
  const int b = stream / a.kv_heads, kvh = stream % a.kv_heads;
  const int heads = min(kDecodeHeads, a.group - h0);
  const uint16_t* kb = a.k + b * a.ks_b + kvh * a.ks_h;
  const uint16_t* vb = a.v + b * a.vs_b + kvh * a.vs_h;

  // Q^T as B operand: column = q head (columns past the group repeat the last head;
  // they are not stored)
  bf16x8 qf[KK];
  {
    const int h = kvh * a.group + h0 + min(c, heads - 1);
    const uint16_t* qr = a.q + b * a.qs_b + h * a.qs_h + 8 * g;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
      qf[kk] = as_bf16x8(*reinterpret_cast<const u32x4*>(qr + 32 * kk));
  }
  f32x4 o[8 * H];
#pragma unroll
  for (int i = 0; i < 8 * H; ++i) o[i] = f32x4{};
  float m = -INFINITY, l = 0.0f;   // of query column c; l over this lane's keys

  const int first = split * a.steps * Shape::kStepKeys + w * Shape::kWaveKeys;
  for (int it = 0; it < a.steps; ++it) {
    const int key0 = first + it * Shape::kStepKeys;
    if (key0 >= a.seq) break;
    u32x4 kr[T][KK], vr[T][4][H];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int64_t row = min(key0 + 16 * t + c, a.seq - 1);   // rows past the end are masked
      const uint16_t* p = kb + row * a.ks_s + 8 * g;
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) kr[t][kk] = *reinterpret_cast<const u32x4*>(p + 32 * kk);
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = min(key0 + 16 * t + 4 * g + r, a.seq - 1);
        const uint16_t* p = vb + row * a.vs_s + 8 * c;
#pragma unroll
        for (int hv = 0; hv < H; ++hv)
          vr[t][r][hv] = *reinterpret_cast<const u32x4*>(p + 128 * hv);
      }
    }
    __builtin_amdgcn_sched_barrier(0);   // every load of the step is issued by now
    f32x4 s[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      s[t] = f32x4{};
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) s[t] = mfma16(as_bf16x8(kr[t][kk]), qf[kk], s[t]);
    }
    float mx = -INFINITY;
    if (key0 + Shape::kWaveKeys <= a.seq) {
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[t][r] *= a.scale_log2;
          mx = fmaxf(mx, s[t][r]);
        }
    } else {
      // the last keys: masked scores are -inf, and their (repeated) value rows zero, so
      // that an infinite value there does not meet a probability of 0
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool valid = key0 + 16 * t + 4 * g + r < a.seq;
          s[t][r] = valid ? s[t][r] * a.scale_log2 : -INFINITY;
          mx = fmaxf(mx, s[t][r]);
#pragma unroll
          for (int hv = 0; hv < H; ++hv)
            if (!valid) vr[t][r][hv] = u32x4{};
        }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m, mx);
    const float shift = m_new == -INFINITY ? 0.0f : m_new;   // no key of a finite score yet
    if (it > 0) {
      const float corr = merge_weight(m, shift);
      l *= corr;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float cr = __shfl(corr, 4 * g + r);   // of O's query row 4 g + r
#pragma unroll
        for (int i = 0; i < 8 * H; ++i) o[i][r] *= cr;
      }
    }
    m = m_new;
#pragma unroll
    for (int t = 0; t < T; ++t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = exp2_fast(s[t][r] - shift);
        l += p;
#pragma unroll
        for (int hv = 0; hv < H; ++hv) {
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const uint32_t v2 = vr[t][r][hv][x];
            o[8 * hv + 2 * x] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(p, bf16_lo(v2), o[8 * hv + 2 * x], 0, 0, 0);
            o[8 * hv + 2 * x + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                p, bf16_hi(v2), o[8 * hv + 2 * x + 1], 0, 0, 0);
          }
        }
      }
    }
  }
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);

  if (g == 0) {
    part_m[w][c] = m;
    part_l[w][c] = l;
  }
#pragma unroll
  for (int hv = 0; hv < H; ++hv)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int x = 0; x < 2; ++x)   // O[query 4 g + r][dim 128 hv + 8 c + i], i = 4 x ..
        *reinterpret_cast<f32x4*>(&part_o[w][4 * g + r][128 * hv + 8 * c + 4 * x]) =
            f32x4{o[8 * hv + 4 * x][r], o[8 * hv + 4 * x + 1][r], o[8 * hv + 4 * x + 2][r],
                  o[8 * hv + 4 * x + 3][r]};
  block_sync();
  for (int e = threadIdx.x; e < heads * (D / 4); e += kDecodeThreads) {
    const int qi = e / (D / 4), d = (e % (D / 4)) * 4;
    float top = part_m[0][qi];
#pragma unroll
    for (int x = 1; x < kDecodeWaves; ++x) top = fmaxf(top, part_m[x][qi]);
    float sum = 0.0f;
    f32x4 acc{};
#pragma unroll
    for (int x = 0; x < kDecodeWaves; ++x) {
      const float wt = merge_weight(part_m[x][qi], top);
      const f32x4 po = *reinterpret_cast<const f32x4*>(&part_o[x][qi][d]);
      sum += wt * part_l[x][qi];
#pragma unroll
      for (int y = 0; y < 4; ++y) acc[y] += wt * po[y];
    }
    const int64_t row = (int64_t)b * a.q_heads + kvh * a.group + h0 + qi;
    if (a.splits == 1) {
      const float inv = 1.0f / sum;
      u32x2 v2;
      v2[0] = pack_bf16x2(acc[0] * inv, acc[1] * inv);
      v2[1] = pack_bf16x2(acc[2] * inv, acc[3] * inv);
      *reinterpret_cast<u32x2*>(a.out + row * D + d) = v2;
    } else {
      *reinterpret_cast<f32x4*>(a.part_o + (row * a.splits + split) * D + d) = acc;
      if (d == 0) {
        a.part_ml[(row * a.splits + split) * 2] = top;
        a.part_ml[(row * a.splits + split) * 2 + 1] = sum;
      }
    }
  }
}

// Merge of the splits: one workgroup per (batch, q head) row. 256 threads = D / 4 groups
// of four dims x the splits in turn, then a reduction over the thread rows in LDS.
template <int D>
__global__ __launch_bounds__(kDecodeThreads) void decode_merge_kernel(DecodeArgs a) {
  constexpr int kCols = D / 4, kRows = kDecodeThreads / kCols;
  __shared__ float weight[kDecodeMaxSplits];
  __shared__ float red[2][kDecodeWaves];
  __shared__ __align__(16) float acc_s[kRows][D];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, w = tid >> 6;
  float m = -INFINITY, l = 0.0f;
  if (tid < a.splits) {
    const float* ml = a.part_ml + (row * a.splits + tid) * 2;
    m = ml[0];
    l = ml[1];
  }
  float top = m;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) top = fmaxf(top, __shfl_xor(top, o));
  if ((tid & 63) == 0) red[0][w] = top;
  block_sync();
  top = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
  const float wt = merge_weight(m, top);
  weight[tid] = wt;
  const float sum = wave_sum(tid < a.splits ? wt * l : 0.0f);
  if ((tid & 63) == 0) red[1][w] = sum;
  block_sync();
  const int col = tid % kCols, r0 = tid / kCols;
  f32x4 acc{};
  const float* src = a.part_o + row * a.splits * D + col * 4;
#pragma unroll 8
  for (int s = r0; s < a.splits; s += kRows) {
    const f32x4 po = *reinterpret_cast<const f32x4*>(src + (int64_t)s * D);
#pragma unroll
    for (int y = 0; y < 4; ++y) acc[y] += weight[s] * po[y];
  }
  *reinterpret_cast<f32x4*>(&acc_s[r0][col * 4]) = acc;
  block_sync();
  if (tid < D / 2) {
    const float inv = 1.0f / ((red[1][0] + red[1][1]) + (red[1][2] + red[1][3]));
    float x = 0.0f, y = 0.0f;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      x += acc_s[r][2 * tid];
      y += acc_s[r][2 * tid + 1];
    }
    *reinterpret_cast<uint32_t*>(a.out + row * D + 2 * tid) = pack_bf16x2(x * inv, y * inv);
  }
}

// Key ranges of a launch: `steps` steps of kStepKeys keys each. One step per range as
// long as there are at most 1024 workgroups (four per CU; two are resident) and 256
// ranges to merge, so that short caches still use many CUs. Up to two steps run as one
// workgroup per stream without the merge launch: 512 keys (28/4 heads) 13.0 us against
// 10.7 us plus the second launch's 3.5 us of host time (eager 13.1 against 16.3 us), the
// host being the bound there. So do three steps where only two ranges per stream fit, and
// four from three workgroups for each two residents on: cut in two, the ranges are uneven
// and in two rounds (8/8 heads, 64 sequences: 520 keys 43 us in two ranges, 31 in one, 800
// keys 47 and 40; SDPA 30 and 40. 48 sequences: 600 keys 34 and 31; 1024 keys 47 and 49).
template <int D>
void decode_ranges(int batch, int seq, int q_heads, int kv_heads, int& splits, int& steps) {
  const int64_t units = (seq + DecodeShape<D>::kStepKeys - 1) / DecodeShape<D>::kStepKeys;
  const int tiles = (q_heads / kv_heads + kDecodeHeads - 1) / kDecodeHeads;
  const int64_t streams = (int64_t)batch * kv_heads * tiles;
  const int64_t most = std::min<int64_t>(kDecodeMaxSplits, std::max<int64_t>(1, 1024 / streams));
  const int whole = most == 2 ? (streams > 384 ? 4 : 3) : 2;   // steps run as one range
  steps = (int)std::max<int64_t>((units + most - 1) / most, units <= whole ? units : 1);
  splits = (int)((units + steps - 1) / steps);
}

template <int D>
int launch_decode(DecodeArgs a, void* workspace, hipStream_t st) {
  decode_ranges<D>(a.batch, a.seq, a.q_heads, a.kv_heads, a.splits, a.steps);
  const int64_t rows = (int64_t)a.batch * a.q_heads;
  if (a.splits > 1) {
    SPX_REQUIRE(workspace != nullptr && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0,
                SPX_EINVAL, "decode: workspace null or not 16-byte aligned");
    a.part_o = static_cast<float*>(workspace);
    a.part_ml = a.part_o + rows * a.splits * D;
  }
  const dim3 grid(a.splits, (unsigned)(a.batch * a.kv_heads * a.head_tiles));
  decode_split_kernel<D><<<grid, kDecodeThreads, 0, st>>>(a);
  if (a.splits > 1) decode_merge_kernel<D><<<(unsigned)rows, kDecodeThreads, 0, st>>>(a);
  return launch_status("decode_attention");
}

}  // namespace spx

using namespace spx;

static bool decode_shape_ok(int batch, int seq, int q_heads, int kv_heads, int head_dim) {
  return batch > 0 && seq > 0 && q_heads > 0 && kv_heads > 0 && q_heads % kv_heads == 0 &&
         (head_dim == 128 || head_dim == 256) && seq <= (1 << 30) &&
         (int64_t)batch * q_heads <= 65535;
}

extern "C" int64_t spx_decode_workspace_bytes(int batch, int seq, int q_heads, int kv_heads,
                                              int head_dim) {
  if (!decode_shape_ok(batch, seq, q_heads, kv_heads, head_dim)) return -1;
  int splits, steps;
  if (head_dim == 128) decode_ranges<128>(batch, seq, q_heads, kv_heads, splits, steps);
  else decode_ranges<256>(batch, seq, q_heads, kv_heads, splits, steps);
  return splits > 1 ? (int64_t)batch * q_heads * splits * (head_dim + 2) * 4 : 0;
}

extern "C" int spx_decode_attention(const void* q, const int64_t* q_strides, const void* k,
                                    const int64_t* k_strides, const void* v,
                                    const int64_t* v_strides, int batch, int seq, int q_heads,
                                    int kv_heads, int head_dim, float scale, void* workspace,
                                    void* out, void* stream) {
  SPX_REQUIRE(head_dim == 128 || head_dim == 256, SPX_EUNSUPPORTED,
              "head_dim %d unsupported (128 or 256)", head_dim);
  SPX_REQUIRE(decode_shape_ok(batch, seq, q_heads, kv_heads, head_dim), SPX_EINVAL,
              "bad shape: batch %d seq %d q_heads %d kv_heads %d", batch, seq, q_heads, kv_heads);
  SPX_REQUIRE(q && k && v && out && q_strides && k_strides && v_strides, SPX_EINVAL,
              "null pointer");
  SPX_REQUIRE(q_strides[3] == 1 && k_strides[3] == 1 && v_strides[3] == 1, SPX_EINVAL,
              "innermost (dim) stride must be 1");
  const void* base[4] = {q, k, v, out};
  for (const void* p : base)
    SPX_REQUIRE((reinterpret_cast<uintptr_t>(p) & 15) == 0, SPX_EINVAL,
                "base pointers must be 16-byte aligned");
  for (int i = 0; i < 3; ++i)
    SPX_REQUIRE(q_strides[i] % 8 == 0 && k_strides[i] % 8 == 0 && v_strides[i] % 8 == 0,
                SPX_EINVAL, "batch / head / sequence strides must be multiples of 8 elements");
  DecodeArgs a{};
  a.q = static_cast<const uint16_t*>(q);
  a.qs_b = q_strides[0]; a.qs_h = q_strides[1];
  a.k = static_cast<const uint16_t*>(k);
  a.ks_b = k_strides[0]; a.ks_h = k_strides[1]; a.ks_s = k_strides[2];
  a.v = static_cast<const uint16_t*>(v);
  a.vs_b = v_strides[0]; a.vs_h = v_strides[1]; a.vs_s = v_strides[2];
  a.out = static_cast<uint16_t*>(out);
  a.batch = batch; a.seq = seq; a.q_heads = q_heads; a.kv_heads = kv_heads;
  a.group = q_heads / kv_heads;
  a.head_tiles = (a.group + kDecodeHeads - 1) / kDecodeHeads;
  a.scale_log2 = (float)((double)scale * 1.4426950408889634);
  hipStream_t st = static_cast<hipStream_t>(stream);
  return head_dim == 128 ? launch_decode<128>(a, workspace, st)
                         : launch_decode<256>(a, workspace, st);
}
