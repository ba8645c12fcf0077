// Block pooling: one HBM pass over K and V per (key block, kv head).
//
// Produces any subset of
//   * bf16 block-mean K (upstream/flashprefill_native_forward.py:27-69, 420-442):
//     fp32 sum over the valid rows / valid count, rounded to bf16;
//   * fp32 descriptors (kernels.py:22-46): mean_k, var_k = max(0, E[k^2] - mean^2),
//     mean_v, sigma_v = sqrt(sum_d max(0, E[v^2] - mean_v^2)), block counts;
//   * attention tiles: the block's K rows and its V transposed to [dim][128 key
//     slots] (key permutation of value_slot_of_key), rows / keys past the sequence
//     end zero, each 128 x 128 bf16 tile stored with 16-byte chunk c of row r at
//     position c ^ (r & 15). The attention kernel copies a tile into LDS verbatim
//     (direct global->LDS loads) and reads MFMA operands bank-conflict free.
//
// Bandwidth-bound at 32K tokens (134 MB with the tiles), latency-bound below (nine
// blocks at 1089 tokens: 36 workgroups). Half of a workgroup's waves take the K rows,
// the other half the V rows. Thread = 8 dims x the 16 rows of one value-slot chunk: all
// 16 of its 16-byte loads are in flight at once, and V is transposed in its registers
// (the 16 rows are exactly two 8-slot chunks of each of its dims); the finished value
// tile passes through LDS in 16-byte pieces so that it leaves in whole cache lines
// (stored from the registers, 16 bytes of each of 64 line parts per instruction: 34.5 us
// at 32K). Against the form before it, which ran K and V in the same threads and
// transposed V through LDS in 2-byte reads, same bits (tiles and descriptors, 4 KV
// heads): 1089 tokens 8.5 -> 5.0 us, 4096 9.1 -> 5.7, 32640 24.2 -> 21.8 (6.2 TB/s),
// 131072 111 -> 108; 4 x 2113, 8 heads, 16.5 -> 13.7; D = 256, 12001 tokens, 22.3 -> 18.7;
// descriptors alone at 32640 tokens 14.8 -> 12.6.
//
// Head dim 256 (Qwen3.5 full-attention layers): the same pass; key tiles keep the
// [128 keys][256 dims] layout (chunk c of row r at c ^ (r & 15), c < 32), value tiles
// are four 32-key sub-blocks [256 dims][32 slots] (16 KB each, the d = 256 attention
// kernel's LDS image) with 16-byte chunk c of dim row d at c ^ ((d >> 2) & 3).
#include "common.h"

namespace spx {

struct PoolArgs {
  const uint16_t* k;
  int64_t ks_b, ks_s, ks_h;
  const uint16_t* v;
  int64_t vs_b, vs_s, vs_h;
  int batch, seq, kv_heads, blocks;
  uint16_t* mean_k_bf16;  // [B, NB, Hkv, D]
  float* mean_k;          // [B, NB, Hkv, D]
  float* mean_v;
  float* var_k;
  float* sigma_v;  // [B, NB, Hkv]
  int32_t* counts;  // [NB]
  uint16_t* key_tiles;    // [B, Hkv, NB, 128, D]
  uint16_t* value_tiles;  // [B, Hkv, NB, D, 128]
};

__device__ __forceinline__ void accumulate8(const u32x4& raw, float* sum, float* sq) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = bf16_lo(raw[e]);
    const float b = bf16_hi(raw[e]);
    sum[2 * e] += a;
    sq[2 * e] = fmaf(a, a, sq[2 * e]);
    sum[2 * e + 1] += b;
    sq[2 * e + 1] = fmaf(b, b, sq[2 * e + 1]);
  }
}

// Value-tile words: the low / high halves of a (low word) and b.
__device__ __forceinline__ uint32_t low_halves(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x05040100u);
}
__device__ __forceinline__ uint32_t high_halves(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

constexpr int kPoolRows = 16;                        // rows per thread

// Columns sums of one operand over the block: part[0] / part[1] hold four row-quarter
// sums of x and x^2 per dim. The order of additions: within a quarter (32 rows) the two
// 16-row groups' sums, each a chain over its rows (two 8-row chains added at D = 128).
template <int D>
__device__ __forceinline__ void column_sums(const u32x4 (&raw)[kPoolRows], int c, int rg, int lane,
                                            float (&part)[2][4][D]) {
  constexpr int kChains = D == 128 ? 2 : 1;
  float sum[8], sq[8];
#pragma unroll
  for (int h = 0; h < kChains; ++h) {
    float s[8] = {}, q[8] = {};
#pragma unroll
    for (int i = 0; i < kPoolRows / kChains; ++i) accumulate8(raw[h * (kPoolRows / kChains) + i], s, q);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      sum[e] = h ? sum[e] + s[e] : s[e];
      sq[e] = h ? sq[e] + q[e] : q[e];
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    sum[e] += __shfl_xor(sum[e], 8);
    sq[e] += __shfl_xor(sq[e], 8);
  }
  if (!(rg & 1)) {
#pragma unroll
    for (int e = 0; e < 8; e += 4) {
      *reinterpret_cast<f32x4*>(&part[0][rg >> 1][c * 8 + e]) =
          f32x4{sum[e], sum[e + 1], sum[e + 2], sum[e + 3]};
      *reinterpret_cast<f32x4*>(&part[1][rg >> 1][c * 8 + e]) =
          f32x4{sq[e], sq[e + 1], sq[e + 2], sq[e + 3]};
    }
  }
}

// D threads per operand: K first (if DO_K or DO_TILES), then V (if DO_V or DO_TILES).
template <int D, bool DO_K, bool DO_V, bool DO_TILES>
__global__ __launch_bounds__(2 * D, 512 / D) void pool_kernel(PoolArgs a) {
  constexpr bool kReadK = DO_K || DO_TILES, kReadV = DO_V || DO_TILES;
  const int j = blockIdx.x;
  const int b = blockIdx.y / a.kv_heads;
  const int g = blockIdx.y % a.kv_heads;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  // which operand this wave takes, and its thread index there
  const bool is_v = kReadV && (!kReadK || __builtin_amdgcn_readfirstlane(tid) >= D);
  const int tx = kReadK && is_v ? tid - D : tid;
  const int c = (tx >> 6) * 8 + (lane & 7);   // 8-dim chunk
  const int rg = lane >> 3;                   // row group: rows rg * 16 + i
  const int n = min(kBlock, a.seq - j * kBlock);

  __shared__ __align__(16) float part_s[2][2][4][D];   // [K, V][x, x^2][quarter][dim]
  __shared__ __align__(16) uint16_t vtile[DO_TILES ? kBlock * D : 8];   // the value tile
  // (40 KB at D = 128: four workgroups per CU; the V wave's sigma goes where its own
  // first thread's column sum was)
  auto& part = part_s[is_v && kReadK];

  const int64_t tile_off = ((((int64_t)b * a.kv_heads + g) * a.blocks + j) * kBlock) * D;
  u32x4 raw[kPoolRows];
  if (kReadK || kReadV) {
    const uint16_t* base = is_v ? a.v + b * a.vs_b + g * a.vs_h : a.k + b * a.ks_b + g * a.ks_h;
    const int64_t stride = is_v ? a.vs_s : a.ks_s;
    base += (int64_t)j * kBlock * stride + c * 8;
#pragma unroll
    for (int i = 0; i < kPoolRows; ++i)   // rows past the end: the last row, zeroed below
      raw[i] = *reinterpret_cast<const u32x4*>(base + min(rg * kPoolRows + i, n - 1) * stride);
    if (n < kBlock) {
#pragma unroll
      for (int i = 0; i < kPoolRows; ++i)
        if (rg * kPoolRows + i >= n) raw[i] = u32x4{0u, 0u, 0u, 0u};
    }
  }

  if (DO_TILES) {
    if (!is_v) {
#pragma unroll
      for (int i = 0; i < kPoolRows; ++i) {
        const int row = rg * kPoolRows + i;
        *reinterpret_cast<u32x4*>(a.key_tiles + tile_off + row * D + ((c ^ i) << 3)) = raw[i];
      }
    } else {
      // slot -> key inside the 16 rows: 4 * half + (m % 4) + 8 * (m / 4) for slot
      // 8 * half + m; 16-byte chunk `chunk` of dim row d at the swizzled position
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int chunk = rg * 2 + half;
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          const int d = c * 8 + x;
          u32x4 w;
#pragma unroll
          for (int m = 0; m < 4; ++m) {
            const int key = 4 * half + 2 * (m & 1) + 8 * (m >> 1);
            const uint32_t lo = raw[key][x >> 1], hi = raw[key + 1][x >> 1];
            w[m] = (x & 1) ? high_halves(lo, hi) : low_halves(lo, hi);
          }
          uint16_t* dst =
              D == 128 ? vtile + d * kBlock + ((chunk ^ (d & 15)) << 3)
                       : vtile + (chunk >> 2) * (D * 32) + d * 32 + (((chunk & 3) ^ ((d >> 2) & 3)) << 3);
          *reinterpret_cast<u32x4*>(dst) = w;
        }
      }
    }
  }
  if ((DO_K && !is_v) || (DO_V && is_v)) column_sums<D>(raw, c, rg, lane, part);
  if (a.counts && blockIdx.y == 0 && tid == 0) a.counts[j] = n;
  block_sync();
  if (DO_TILES) {   // all waves: whole lines of the value tile
#pragma unroll
    for (int i = 0; i < kBlock * D / 8 / (2 * D); ++i) {
      const int e = (i * 2 * D + tid) * 8;
      *reinterpret_cast<u32x4*>(a.value_tiles + tile_off + e) =
          *reinterpret_cast<const u32x4*>(vtile + e);
    }
  }
  if (!DO_K && !DO_V) return;

  const float count = (float)n;
  const int64_t o = (((int64_t)b * a.blocks + j) * a.kv_heads + g) * D + tx;
  if (DO_K && !is_v) {
    const float s = part[0][0][tx] + part[0][1][tx] + part[0][2][tx] + part[0][3][tx];
    const float s2 = part[1][0][tx] + part[1][1][tx] + part[1][2][tx] + part[1][3][tx];
    const float mean = s / count;
    if (a.mean_k_bf16) a.mean_k_bf16[o] = to_bf16_bits(mean);
    if (a.mean_k) a.mean_k[o] = mean;
    if (a.var_k) a.var_k[o] = fmaxf(s2 / count - mean * mean, 0.0f);
  }
  if (DO_V && is_v) {
    const float s = part[0][0][tx] + part[0][1][tx] + part[0][2][tx] + part[0][3][tx];
    const float s2 = part[1][0][tx] + part[1][1][tx] + part[1][2][tx] + part[1][3][tx];
    const float mean = s / count;
    const float var = fmaxf(s2 / count - mean * mean, 0.0f);
    if (a.mean_v) a.mean_v[o] = mean;
    if (a.sigma_v) {
      const float total = wave_sum(var);
      if (lane == 0) part[0][0][tx] = total;
    }
  }
  if (DO_V && a.sigma_v) {
    block_sync();
    if (tid == 0) {
      float total = 0.0f;
#pragma unroll
      for (int x = 0; x < D / 64; ++x) total += part_s[kReadK][0][0][64 * x];
      a.sigma_v[((int64_t)b * a.blocks + j) * a.kv_heads + g] = sqrtf(total);
    }
  }
}

}  // namespace spx

using namespace spx;

template <int D>
static void launch_pool(int variant, dim3 grid, hipStream_t st, const PoolArgs& a) {
  switch (variant) {
    case 0: pool_kernel<D, false, false, false><<<grid, D, 0, st>>>(a); break;
    case 1: pool_kernel<D, false, false, true><<<grid, 2 * D, 0, st>>>(a); break;
    case 2: pool_kernel<D, false, true, false><<<grid, D, 0, st>>>(a); break;
    case 3: pool_kernel<D, false, true, true><<<grid, 2 * D, 0, st>>>(a); break;
    case 4: pool_kernel<D, true, false, false><<<grid, D, 0, st>>>(a); break;
    case 5: pool_kernel<D, true, false, true><<<grid, 2 * D, 0, st>>>(a); break;
    case 6: pool_kernel<D, true, true, false><<<grid, 2 * D, 0, st>>>(a); break;
    default: pool_kernel<D, true, true, true><<<grid, 2 * D, 0, st>>>(a); break;
  }
}

static int check_tensor4(const char* name, const void* p, const int64_t* st) {
  SPX_REQUIRE(p != nullptr && st != nullptr, SPX_EINVAL, "%s: null pointer", name);
  SPX_REQUIRE(st[3] == 1, SPX_EINVAL, "%s: innermost (dim) stride must be 1", name);
  SPX_REQUIRE((reinterpret_cast<uintptr_t>(p) & 15) == 0, SPX_EINVAL,
              "%s: base pointer must be 16-byte aligned", name);
  SPX_REQUIRE(st[0] % 8 == 0 && st[1] % 8 == 0 && st[2] % 8 == 0, SPX_EINVAL,
              "%s: batch / sequence / head strides must be multiples of 8 elements", name);
  return SPX_OK;
}

extern "C" int spx_block_pool(const void* k, const int64_t* k_strides, const void* v,
                              const int64_t* v_strides, int batch, int seq, int kv_heads,
                              int head_dim, int block_size, void* mean_k_bf16, float* mean_k,
                              float* mean_v, float* var_k, float* sigma_v, int32_t* counts,
                              void* key_tiles, void* value_tiles, void* stream) {
  SPX_REQUIRE(head_dim == 128 || head_dim == 256, SPX_EUNSUPPORTED,
              "head_dim %d unsupported (128 or 256)", head_dim);
  SPX_REQUIRE(block_size == kBlock, SPX_EUNSUPPORTED, "block_size %d unsupported (only 128)", block_size);
  SPX_REQUIRE(batch > 0 && seq > 0 && kv_heads > 0, SPX_EINVAL,
              "batch, seq and kv_heads must be positive (got %d, %d, %d)", batch, seq, kv_heads);
  SPX_REQUIRE((key_tiles == nullptr) == (value_tiles == nullptr), SPX_EINVAL,
              "key_tiles and value_tiles are produced together");
  const bool do_k = mean_k_bf16 || mean_k || var_k;
  const bool do_v = mean_v || sigma_v;
  const bool do_tiles = value_tiles != nullptr;
  if (do_k || do_tiles) { int e = check_tensor4("k", k, k_strides); if (e) return e; }
  if (do_v || do_tiles) { int e = check_tensor4("v", v, v_strides); if (e) return e; }
  if (do_tiles) {
    SPX_REQUIRE((reinterpret_cast<uintptr_t>(key_tiles) & 15) == 0 &&
                    (reinterpret_cast<uintptr_t>(value_tiles) & 15) == 0,
                SPX_EINVAL, "key_tiles / value_tiles must be 16-byte aligned");
  }
  if (!do_k && !do_v && !do_tiles && !counts) return SPX_OK;
  PoolArgs a{};
  a.k = static_cast<const uint16_t*>(k);
  if (do_k || do_tiles) { a.ks_b = k_strides[0]; a.ks_s = k_strides[1]; a.ks_h = k_strides[2]; }
  a.v = static_cast<const uint16_t*>(v);
  if (do_v || do_tiles) { a.vs_b = v_strides[0]; a.vs_s = v_strides[1]; a.vs_h = v_strides[2]; }
  a.batch = batch; a.seq = seq; a.kv_heads = kv_heads; a.blocks = num_blocks(seq);
  a.mean_k_bf16 = static_cast<uint16_t*>(mean_k_bf16);
  a.mean_k = mean_k; a.mean_v = mean_v; a.var_k = var_k; a.sigma_v = sigma_v;
  a.counts = counts;
  a.key_tiles = static_cast<uint16_t*>(key_tiles);
  a.value_tiles = static_cast<uint16_t*>(value_tiles);
  dim3 grid(a.blocks, batch * kv_heads);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int variant = (do_k ? 4 : 0) | (do_v ? 2 : 0) | (do_tiles ? 1 : 0);
  if (head_dim == 128) launch_pool<128>(variant, grid, st, a);
  else launch_pool<256>(variant, grid, st, a);
  return launch_status("block_pool");
}

extern "C" int spx_block_mean_k(const void* k, const int64_t* k_strides, int batch, int seq,
                                int kv_heads, int head_dim, int block_size, void* mean_k,
                                void* stream) {
  SPX_REQUIRE(mean_k != nullptr, SPX_EINVAL, "mean_k: null pointer");
  return spx_block_pool(k, k_strides, nullptr, nullptr, batch, seq, kv_heads, head_dim,
                        block_size, mean_k, nullptr, nullptr, nullptr, nullptr, nullptr,
                        nullptr, nullptr, stream);
}

extern "C" int spx_block_descriptors(const void* k, const int64_t* k_strides, const void* v,
                                     const int64_t* v_strides, int batch, int seq, int kv_heads,
                                     int head_dim, int block_size, float* mean_k, float* mean_v,
                                     float* var_k, float* sigma_v, int32_t* counts, void* stream) {
  SPX_REQUIRE(mean_k && mean_v && var_k && sigma_v && counts, SPX_EINVAL,
              "block_descriptors: every output must be given");
  return spx_block_pool(k, k_strides, v, v_strides, batch, seq, kv_heads, head_dim, block_size,
                        nullptr, mean_k, mean_v, var_k, sigma_v, counts, nullptr, nullptr, stream);
}
