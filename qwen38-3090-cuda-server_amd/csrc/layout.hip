// Load-time side of the library: weight allocation, the repack from the three
// accepted source layouts into the tile-major layout (w4a16_common.h), the
// bf16 dequant of repacked rows, status strings and the synthetic generator.
#include <hip/hip_runtime.h>

#include <type_traits>

#include <algorithm>
#include <cstdio>
#include <cstring>

#include "../../include/qwen_w4a16.h"
#include "w4a16_common.h"

namespace qw4 {

static thread_local int g_last_hip_error = 0;
void set_hip_error(int e) { g_last_hip_error = e; }

namespace {

// Nibble slot of element e in the AWQ order {0,2,4,6,1,3,5,7}: slot i holds
// element AWQ_ORDER[i], so element e sits at slot (e % 2) * 4 + e / 2 -- the same
// slot order as the repacked layout, which is why AWQ words along K move as is.
__device__ __forceinline__ int awq_slot(int e) { return slot_of_elem(e); }

// ------------------------------------------------------------------ repack
// Source layouts:
//   0 = compressed-tensors [N][K/8] (element e at slot e; w4a16_unpack.h:25-29)
//   1 = AWQ packed along K [K/8][N], 2 = AWQ packed along N [K][N/8].
// Nibbles of a compressed-tensors word (element e at nibble e) in slot order:
// the even elements in the low half, the odd ones in the high half.
__device__ __forceinline__ uint32_t ct_to_slots(uint32_t s) {
  uint32_t ev = s & 0x0F0F0F0Fu, od = (s >> 4) & 0x0F0F0F0Fu;
  ev = (ev | (ev >> 4)) & 0x00FF00FFu;
  od = (od | (od >> 4)) & 0x00FF00FFu;
  return ((ev | (ev >> 8)) & 0xFFFFu) | ((od | (od >> 8)) << 16);
}

// One wave per (tile, two groups), lane p at storage position p (row
// 4 (p % 16) + p / 16): whole 1 KiB of a block per store, and for source 0 the
// 128 contiguous bytes of a row that one lane needs. The scale records and
// zero points of the same groups go with them (lane r at row r), so a repack
// is one launch. Bound by memory: 5120x5120 compressed-tensors, 27 MB
// moved, 23 us in two launches with one thread per word, 10.2 us so.
// Source 2 spreads the 8 k of a word over 8 source rows, 32 loads for a lane's 16
// bytes: there a wave takes one chunk of one group (5120x512 / 5120x17408 7.6 / 39.4
// us with two whole groups a wave, 6.2 / 24.2 so).
template <int SRC>
struct RepackItem {
  static constexpr int kGroups = SRC == 2 ? 1 : 2;   // groups of a wave
  static constexpr int kChunks = SRC == 2 ? 1 : 4;   // of the block's four 1 KiB chunks
};

template <int SRC>
__global__ __launch_bounds__(256) void k_repack(uint32_t* __restrict__ dst,
                                                uint16_t* __restrict__ dscale,
                                                uint16_t* __restrict__ dzero,
                                                const uint32_t* __restrict__ src,
                                                const uint16_t* __restrict__ sscale,
                                                const uint32_t* __restrict__ szero, int n_src,
                                                int K, int G, int tile0) {
  const int lane = threadIdx.x & 63;
  constexpr int kGr = RepackItem<SRC>::kGroups, kCh = RepackItem<SRC>::kChunks;
  const int per_tile = (G + kGr - 1) / kGr;
  int item = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int j0 = item % (4 / kCh) * kCh;   // the item's first chunk
  item /= 4 / kCh;
  if (item >= (n_src / kTileN) * per_tile) return;
  const int bl = item / per_tile, g0 = (item % per_tile) * kGr;
  const int ns = bl * kTileN + tile_row_of_pos(lane);   // source row of position `lane`
  u32x4 q[kGr][kCh];
#pragma unroll
  for (int i = 0; i < kGr; ++i) {
    const int g = min(g0 + i, G - 1);
#pragma unroll
    for (int j = 0; j < kCh; ++j) {
      const int r = g * 16 + 4 * (j0 + j);   // words r .. r + 3 of the row: k = 8 r .. 8 r + 31
      if (SRC == 0) {
        const uint32_t* s = src + (size_t)ns * (K / 8) + r;
#pragma unroll
        for (int w = 0; w < 4; ++w) q[i][j][w] = s[w];
      } else if (SRC == 1) {   // the AWQ slot order is the repacked one
#pragma unroll
        for (int w = 0; w < 4; ++w) q[i][j][w] = src[(size_t)(r + w) * n_src + ns];
      } else {
        const int sh = 4 * awq_slot(ns & 7);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          uint32_t o = 0;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const uint32_t s = src[(size_t)(8 * (r + w) + e) * (n_src / 8) + (ns >> 3)];
            o |= ((s >> sh) & 0xFu) << (4 * slot_of_elem(e));
          }
          q[i][j][w] = o;
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kGr; ++i) {
    const int g = g0 + i;
    if (g >= G) break;
    const size_t blk = (size_t)(tile0 + bl) * G + g;
#pragma unroll
    for (int j = 0; j < kCh; ++j) {
      u32x4 o = q[i][j];
      if (SRC == 0)
#pragma unroll
        for (int w = 0; w < 4; ++w) o[w] = ct_to_slots(o[w]);
      *reinterpret_cast<u32x4*>(dst + blk * kWordsPerBlock + (j0 + j) * 256 + lane * 4) = o;
    }
    if (kCh < 4 && j0 != 0) continue;   // the record goes with the first chunk
    const int rn = bl * kTileN + lane;   // source row of the record's lane
    uint16_t sc;
    uint32_t z;
    if (SRC == 0) {
      sc = sscale[(size_t)rn * G + g];
      z = (szero[(size_t)(rn >> 3) * G + g] >> (4 * (rn & 7))) & 0xFu;  // w4a16_unpack.h:38-42
    } else {
      sc = sscale[(size_t)g * n_src + rn];
      z = (szero[(size_t)g * (n_src / 8) + (rn >> 3)] >> (4 * awq_slot(rn & 7))) & 0xFu;
    }
    dscale[blk * kMetaU16 + lane] = sc;
    // four rows' zero points to a u16
    z <<= 4 * (lane & 3);
    z |= __shfl_xor(z, 1, 64);
    z |= __shfl_xor(z, 2, 64);
    if ((lane & 3) == 0) {
      dzero[blk * 16 + (lane >> 2)] = (uint16_t)z;
      dscale[blk * kMetaU16 + 64 + (lane >> 2)] = (uint16_t)z;
    }
  }
}

// ----------------------------------------------------------------- dequant
// dst [nrows][K] = RNE(float(q - z) * s). One workgroup per (tile, kDeqGroups
// groups, IT rounds of 8 rows), so that every 16 lanes write 256 bytes of a row;
// one thread per 8 consecutive k. Bound by the bf16 store: 7168x5120, 73 MB: 25.8
// us with one thread per word along a row, 23.3 with a workgroup per whole tile, 20.3 so.
constexpr int kDeqGroups = 2;
constexpr int kDeqRows = 256 / (16 * kDeqGroups);   // rows a workgroup does at once
constexpr int kDeqIters = kTileN / kDeqRows;        // rounds over a tile's rows

// IT of a tile's rounds per workgroup.
template <int IT>
__global__ __launch_bounds__(256) void k_dequant_rows(uint16_t* __restrict__ dst,
                                                      const uint32_t* __restrict__ qw,
                                                      const uint16_t* __restrict__ sc,
                                                      const uint16_t* __restrict__ zr, int row0,
                                                      int nrows, int K, int G) {
  constexpr int kParts = kDeqIters / IT;
  const int per_tile = (G + kDeqGroups - 1) / kDeqGroups;
  const int part = (int)blockIdx.x % kParts, item = (int)blockIdx.x / kParts;
  const int b = (row0 >> 6) + item / per_tile;   // tile
  const int g0 = (item % per_tile) * kDeqGroups;
  // thread: word wi of its group (of kDeqGroups), row `rs` of every kDeqRows rows
  const int wi = threadIdx.x % (16 * kDeqGroups), rs = threadIdx.x / (16 * kDeqGroups);
  const int g = g0 + wi / 16, j = (wi >> 2) & 3, w = wi & 3;
  if (g >= G) return;
  const size_t blk = (size_t)b * G + g;
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int rr = rs + kDeqRows * (part * IT + it), n = b * kTileN + rr;   // row of the tile, of the tensor
    if (n < row0 || n >= row0 + nrows) continue;
    const uint32_t word = qw[blk * kWordsPerBlock + j * 256 + tile_pos_of_row(rr) * 4 + w];
    const float s = bf16_bits_to_f32(sc[blk * kMetaU16 + rr]);
    const int z = (zr[blk * 16 + (rr >> 2)] >> (4 * (rr & 3))) & 0xF;
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const float a = (float)((int)((word >> (4 * slot_of_elem(e))) & 0xFu) - z) * s;
      const float c = (float)((int)((word >> (4 * slot_of_elem(e + 1))) & 0xFu) - z) * s;
      o[e / 2] = pack_bf16x2(a, c);
    }
    *reinterpret_cast<u32x4*>(dst + (size_t)(n - row0) * K + (size_t)g * kGroup + 8 * (4 * j + w)) =
        u32x4{o[0], o[1], o[2], o[3]};
  }
}

// ------------------------------------------------------- INT4 quantizer
// The reference's k_quant_i4 (src/model/model.cu:140-172), the INT4 g128
// asymmetric lm_head quantizer, writing the repacked layout directly: one
// thread per (tile, group, row quad c); for each of its 4 rows and the group:
// lo / hi = min / max (fp32 of the bf16 values), s = (hi - lo) / 15 (1e-8 if
// not > 0), z = clamp(rint(-lo / s), 0, 15), stored scale bf16(s); each value
// q = clamp(rint(v * (1 / s)) + z, 0, 15) with the unrounded fp32 s. IEEE
// division and round-half-even as the reference's CUDA arithmetic.
__global__ void k_quant_i4(uint32_t* __restrict__ qw, uint16_t* __restrict__ sc,
                           uint16_t* __restrict__ zr, const uint16_t* __restrict__ src, int N,
                           int K, int G) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)(N / 4) * G) return;
  const int g = (int)(t % G), quad = (int)(t / G);
  const int b = quad >> 4, c = quad & 15;
  const size_t blk = (size_t)b * G + g;
  uint32_t zbits = 0;
  for (int i = 0; i < 4; ++i) {
    const int rr = 4 * c + i, n = b * kTileN + rr;
    const uint16_t* row = src + (size_t)n * K + (size_t)g * kGroup;
    float lo = 1e30f, hi = -1e30f;
    for (int e = 0; e < kGroup; ++e) {
      const float v = bf16_bits_to_f32(row[e]);
      lo = fminf(lo, v);
      hi = fmaxf(hi, v);
    }
    float s = (hi - lo) / 15.0f;
    if (!(s > 0.f)) s = 1e-8f;
    const int z = max(0, min(15, __float2int_rn(-lo / s)));
    sc[blk * kMetaU16 + rr] = to_bf16(s);
    zbits |= (uint32_t)z << (4 * i);
    const float inv = 1.0f / s;
    const int p = tile_pos_of_row(rr);
    for (int k8 = 0; k8 < kGroup / 8; ++k8) {   // word w of chunk j: k = 32 j + 8 w + e
      uint32_t word = 0;
      for (int e = 0; e < 8; ++e) {
        const int q = max(0, min(15, __float2int_rn(bf16_bits_to_f32(row[8 * k8 + e]) * inv) + z));
        word |= (uint32_t)q << (4 * slot_of_elem(e));
      }
      qw[blk * kWordsPerBlock + (k8 >> 2) * 256 + p * 4 + (k8 & 3)] = word;
    }
  }
  zr[blk * 16 + c] = (uint16_t)zbits;
  sc[blk * kMetaU16 + 64 + c] = (uint16_t)zbits;
}

// ------------------------------------------------------------ 8-bit weights
// W8A16 quantizer, the reference's k_quant_w8 (src/kernels/gemv_w4a16.cu:478-495)
// writing the 8-bit block layout directly: one thread per (row n, group g);
// mx = max |w|, s = bf16(mx / 127), q = clamp(rint(w * (127 / mx)), +-127),
// stored as u = q + 128 at [tile][g][j][position][32 B], j = k / 32 in the group.
__global__ void k_w8_quantize(uint8_t* __restrict__ qw, uint16_t* __restrict__ sc,
                              const uint16_t* __restrict__ src, int N, int K, int G) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)N * G) return;
  const int n = (int)(t / G), g = (int)(t % G);
  const u32x4* row = reinterpret_cast<const u32x4*>(src + (size_t)n * K + (size_t)g * kGroup);
  float mx = 0.f;
#pragma unroll 4
  for (int i = 0; i < 16; ++i) {
    const u32x4 v = row[i];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      mx = fmaxf(mx, fabsf(bf16_bits_to_f32(v[e] & 0xffffu)));
      mx = fmaxf(mx, fabsf(bf16_bits_to_f32(v[e] >> 16)));
    }
  }
  const float inv = mx > 0.f ? 127.0f / mx : 0.f;
  const int b = n >> 6, rr = n & 63;
  const size_t blk = (size_t)b * G + g;
  sc[blk * 64 + rr] = to_bf16(mx / 127.0f);
  uint8_t* dst = qw + blk * 8192 + tile_pos_of_row(rr) * 32;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t o[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32x4 v = row[4 * j + i];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t pair = 0;
#pragma unroll
        for (int hlf = 0; hlf < 2; ++hlf) {
          const float w = bf16_bits_to_f32(hlf ? (v[e] >> 16) : (v[e] & 0xffffu));
          int q = (int)__builtin_rintf(w * inv);
          q = q < -127 ? -127 : (q > 127 ? 127 : q);
          pair |= (uint32_t)(q + 128) << (8 * hlf);
        }
        // bytes 8i + 2e, 8i + 2e + 1 of the 32-byte chunk
        const int byte = 8 * i + 2 * e;
        if ((byte & 3) == 0)
          o[byte >> 2] = pair;
        else
          o[byte >> 2] |= pair << 16;
      }
    }
    u32x4* d = reinterpret_cast<u32x4*>(dst + (size_t)j * 2048);
    d[0] = u32x4{o[0], o[1], o[2], o[3]};
    d[1] = u32x4{o[4], o[5], o[6], o[7]};
  }
}

// dst [nrows][K] = RNE(q * s) of 8-bit weights, one thread per 8 consecutive k.
__global__ void k_w8_dequant_rows(uint16_t* __restrict__ dst, const uint8_t* __restrict__ qw,
                                  const uint16_t* __restrict__ sc, int row0, int nrows, int K,
                                  int G) {
  const int cpr = K / 8;
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)nrows * cpr) return;
  const int r = (int)(t / cpr), ci = (int)(t % cpr);
  const int n = row0 + r, b = n >> 6, rr = n & 63;
  const int g = ci >> 4, j = (ci >> 2) & 3, e8 = ci & 3;
  const size_t blk = (size_t)b * G + g;
  const u32x2 v = *reinterpret_cast<const u32x2*>(qw + blk * 8192 + (size_t)j * 2048 +
                                                  tile_pos_of_row(rr) * 32 + e8 * 8);
  const float s = bf16_bits_to_f32(sc[blk * 64 + rr]);
  uint32_t o[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t w = v[k >> 1] >> (16 * (k & 1));
    o[k] = pack_bf16x2((float)((int)(w & 0xffu) - 128) * s, (float)((int)((w >> 8) & 0xffu) - 128) * s);
  }
  *reinterpret_cast<u32x4*>(dst + (size_t)r * K + 8 * ci) = u32x4{o[0], o[1], o[2], o[3]};
}

// --------------------------------------------------------------- generator
// Counter-based synthetic inputs (identical spec in the CPU test oracle):
//   key = mix64(seed * 0xD1B54A32D192ED03 + stream_id)
//   draw(i) = mix64(key + (i + 1) * 0x9E3779B97F4A7C15), mix64 = SplitMix64 finalizer
//   u4(i) = draw(i) >> 60
//   normal(i) = Irwin-Hall(12) of the 16-bit fields of draw(3i..3i+2):
//               (S + 6) / 65536 - 6, exact in fp32
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ uint64_t gkey(uint64_t seed, uint64_t stream) {
  return mix64(seed * 0xD1B54A32D192ED03ull + stream);
}
__device__ __forceinline__ uint64_t gdraw(uint64_t key, uint64_t i) {
  return mix64(key + (i + 1) * 0x9E3779B97F4A7C15ull);
}
__device__ __forceinline__ float gnormal(uint64_t key, uint64_t i) {
  uint32_t s = 0;
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    const uint64_t r = gdraw(key, 3 * i + t);
    s += (uint32_t)(r & 0xffff) + (uint32_t)((r >> 16) & 0xffff) +
         (uint32_t)((r >> 32) & 0xffff) + (uint32_t)(r >> 48);
  }
  return __fsub_rn(__fmul_rn(__fadd_rn((float)s, 6.0f), 1.0f / 65536.0f), 6.0f);
}
__device__ __forceinline__ uint16_t rne_bf16(float f) {
  const uint32_t u = __float_as_uint(f);
  return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}
__device__ __forceinline__ uint16_t gen_value(uint64_t key, uint64_t i, int kind) {
  const float v = gnormal(key, i);
  return kind == 0 ? rne_bf16(v) : rne_bf16(__fadd_rn(fabsf(__fmul_rn(v, 0.02f)), 1e-4f));
}

__global__ void k_gen_bf16(uint16_t* out, size_t count, uint64_t seed, uint64_t stream,
                           uint64_t offset, int kind) {
  const uint64_t key = gkey(seed, stream);
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
       i += (size_t)gridDim.x * blockDim.x)
    out[i] = gen_value(key, offset + i, kind);
}

// qweight [K/8][N]: slot i of word [r][n] <- q[n][8r + AWQ_ORDER[i]], q[n][k] = u4(n*K + k)
__global__ void k_gen_awq_k_q(uint32_t* qw, int N, int K, uint64_t seed, uint64_t tensor) {
  const uint64_t key = gkey(seed, tensor * 8 + 0);
  const size_t total = (size_t)(K / 8) * N;
  for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < total;
       t += (size_t)gridDim.x * blockDim.x) {
    const size_t r = t / N, n = t % N;
    uint32_t w = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t q = (uint32_t)(gdraw(key, n * (size_t)K + 8 * r + e) >> 60);
      w |= q << (4 * awq_slot(e));
    }
    qw[t] = w;
  }
}

// scales [G][N] bf16 (s[n][g] = scale(n*G + g)); zeros [G][N/8] (zp[n][g] = u4(n*G + g))
__global__ void k_gen_awq_k_meta(uint16_t* sc, uint32_t* zr, int N, int G, uint64_t seed,
                                 uint64_t tensor) {
  const uint64_t kz = gkey(seed, tensor * 8 + 1), ks = gkey(seed, tensor * 8 + 2);
  const size_t total = (size_t)G * (N / 8);
  for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < total;
       t += (size_t)gridDim.x * blockDim.x) {
    const size_t g = t / (N / 8), c = t % (N / 8);
    uint32_t w = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const size_t n = 8 * c + e;
      w |= (uint32_t)(gdraw(kz, n * G + g) >> 60) << (4 * awq_slot(e));
      sc[g * N + n] = gen_value(ks, n * G + g, 1);
    }
    zr[t] = w;
  }
}

// Streaming read: grid-stride 16-byte loads, XOR-folded so nothing is dead code.
__global__ __launch_bounds__(256) void k_stream_read(const u32x4* __restrict__ src, size_t n16,
                                                     uint32_t* sink) {
  u32x4 acc = {0, 0, 0, 0};
  const size_t stride = (size_t)gridDim.x * 256;
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  for (; i + 3 * stride < n16; i += 4 * stride) {
    const u32x4 a = __builtin_nontemporal_load(src + i);
    const u32x4 b = __builtin_nontemporal_load(src + i + stride);
    const u32x4 c = __builtin_nontemporal_load(src + i + 2 * stride);
    const u32x4 d = __builtin_nontemporal_load(src + i + 3 * stride);
    acc ^= a ^ b ^ c ^ d;
  }
  for (; i < n16; i += stride) acc ^= __builtin_nontemporal_load(src + i);
  uint32_t v = acc[0] ^ acc[1] ^ acc[2] ^ acc[3];
  for (int off = 32; off > 0; off >>= 1) v ^= __shfl_xor(v, off, 64);
  __shared__ uint32_t part[4];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) sink[blockIdx.x] = part[0] ^ part[1] ^ part[2] ^ part[3];
}

int check_weights(const qw4_weights* w) {
  if (!w || !w->qweight || !w->scale || !w->zeros) return QW4_ERR_NULL;
  if (w->group_size != kGroup) return QW4_ERR_GROUP;
  if (w->out_f <= 0 || w->out_f % kTileN || w->in_f <= 0 || w->in_f % kGroup ||
      w->num_groups != w->in_f / kGroup)
    return QW4_ERR_SHAPE;
  return QW4_OK;
}

unsigned blocks_for(size_t n, unsigned tpb) { return (unsigned)((n + tpb - 1) / tpb); }

}  // namespace

int check_weights_public(const qw4_weights* w) { return check_weights(w); }

}  // namespace qw4

using namespace qw4;

// MFMA peak microbenchmark: every wave runs `iters` rounds of 8 independent
// v_mfma_f32_32x32x16_bf16 chains on operands hashed from the lane id (random
// bits keep the matrix cores at their realistic power draw) and folds the
// accumulators into sink[block] so nothing is dead code.
__global__ __launch_bounds__(256) void k_mfma_peak(uint32_t* sink, int iters) {
  typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
  const uint32_t l = threadIdx.x + 977u * blockIdx.x;
  u32x4 ra, rb;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    // bf16 pairs in [1, 2): exponent fixed, mantissas hashed
    ra[i] = 0x3F803F80u | ((l * 2654435761u + 40503u * i) & 0x007F007Fu);
    rb[i] = 0x3F803F80u | ((l * 2246822519u + 91711u * i) & 0x007F007Fu);
  }
  const bf16x8v A = __builtin_bit_cast(bf16x8v, ra), B = __builtin_bit_cast(bf16x8v, rb);
  f32x16 acc[8];
#pragma unroll
  for (int k = 0; k < 8; ++k)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[k][e] = 0.f;
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, B, acc[k], 0, 0, 0);
  }
  float v = 0.f;
#pragma unroll
  for (int k = 0; k < 8; ++k)
#pragma unroll
    for (int e = 0; e < 16; ++e) v += acc[k][e];
  if (threadIdx.x == 0) sink[blockIdx.x] = __float_as_uint(v);
}

extern "C" {

const char* qw4_status_string(int st) {
  switch (st) {
    case QW4_OK: return "ok";
    case QW4_ERR_NULL: return "null pointer";
    case QW4_ERR_SHAPE: return "unsupported shape (out_f % 64, in_f % 128, row offset or size)";
    case QW4_ERR_GROUP: return "unsupported group size (only 128)";
    case QW4_ERR_M: return "M out of range for this entry point";
    case QW4_ERR_SCRATCH: return "scratch or workspace too small";
    case QW4_ERR_ALIGN: return "pointer not aligned (16 bytes for activations)";
    case QW4_ERR_HIP: return "HIP runtime error";
    case QW4_ERR_NOMEM: return "device allocation failed";
    case QW4_ERR_LAYOUT: return "unknown source layout";
    case QW4_ERR_IO: return "checkpoint file cannot be opened, mapped or parsed";
    case QW4_ERR_NOTFOUND: return "tensor not found in the checkpoint";
    default: return "unknown status";
  }
}

int qw4_last_hip_error(void) { return g_last_hip_error; }
int qw4_version(void) { return 1; }

size_t qw4_weights_bytes(const qw4_weights* w) {
  if (!w) return 0;
  const size_t n = (size_t)w->out_f, k = (size_t)w->in_f, g = (size_t)w->num_groups;
  return n * k / 2 + n * g * kMetaBytes / kTileN + n * g / 2;
}

int qw4_weights_alloc(qw4_weights* w, int out_f, int in_f, int group_size, void* stream) {
  (void)stream;
  if (!w) return QW4_ERR_NULL;
  if (group_size != kGroup) return QW4_ERR_GROUP;
  if (out_f <= 0 || out_f % kTileN || in_f <= 0 || in_f % kGroup) return QW4_ERR_SHAPE;
  std::memset(w, 0, sizeof(*w));
  w->out_f = out_f;
  w->in_f = in_f;
  w->group_size = group_size;
  w->num_groups = in_f / group_size;
  const size_t n = (size_t)out_f, g = (size_t)w->num_groups;
  hipError_t e = hipMalloc((void**)&w->qweight, n * in_f / 2);
  if (e == hipSuccess) e = hipMalloc((void**)&w->scale, n * g * kMetaBytes / kTileN);
  if (e == hipSuccess) e = hipMalloc((void**)&w->zeros, n * g / 2);
  if (e != hipSuccess) {
    set_hip_error((int)e);
    (void)hipGetLastError();
    qw4_weights_free(w);
    return QW4_ERR_NOMEM;
  }
  return QW4_OK;
}

int qw4_weights_free(qw4_weights* w) {
  if (!w) return QW4_ERR_NULL;
  if (w->qweight) (void)hipFree(w->qweight);
  if (w->scale) (void)hipFree(w->scale);
  if (w->zeros) (void)hipFree(w->zeros);
  std::memset(w, 0, sizeof(*w));
  return QW4_OK;
}

static int repack_into(qw4_weights* w, int row_offset, const uint32_t* q, const uint16_t* s,
                       const uint32_t* z, int out_f, int src, void* stream) {
  int st = check_weights(w);
  if (st) return st;
  if (!q || !s || !z) return QW4_ERR_NULL;
  if (out_f <= 0 || out_f % kTileN || row_offset < 0 || row_offset % kTileN ||
      row_offset + out_f > w->out_f)
    return QW4_ERR_SHAPE;
  hipStream_t hs = (hipStream_t)stream;
  const int G = w->num_groups, tile0 = row_offset / kTileN;
  const size_t tiles = (size_t)(out_f / kTileN);
  const unsigned nb = blocks_for(tiles * ((G + 1) / 2), 4);   // waves of RepackItem<0>, <1>
  switch (src) {
    case 0:
      k_repack<0><<<nb, 256, 0, hs>>>(w->qweight, w->scale, w->zeros, q, s, z, out_f, w->in_f, G, tile0);
      break;
    case QW4_LAYOUT_AWQ_K:
      k_repack<1><<<nb, 256, 0, hs>>>(w->qweight, w->scale, w->zeros, q, s, z, out_f, w->in_f, G, tile0);
      break;
    case QW4_LAYOUT_AWQ_N:
      k_repack<2><<<blocks_for(tiles * G * 4, 4), 256, 0, hs>>>(w->qweight, w->scale, w->zeros, q, s, z, out_f, w->in_f, G, tile0);
      break;
    default:
      return QW4_ERR_LAYOUT;
  }
  QW4_LAUNCH_CHECK();
  return QW4_OK;
}

int qw4_repack_ct_into(qw4_weights* w, int row_offset, const uint32_t* packed,
                       const uint16_t* scale, const uint32_t* zp, int out_f, void* stream) {
  return repack_into(w, row_offset, packed, scale, zp, out_f, 0, stream);
}

int qw4_repack_ct(qw4_weights* w, const uint32_t* packed, const uint16_t* scale,
                  const uint32_t* zp, int out_f, int in_f, int group_size, void* stream) {
  int st = qw4_weights_alloc(w, out_f, in_f, group_size, stream);
  if (st) return st;
  return repack_into(w, 0, packed, scale, zp, out_f, 0, stream);
}

int qw4_repack_awq_into(qw4_weights* w, int row_offset, const uint32_t* qweight,
                        const uint16_t* scales, const uint32_t* zeros, int out_f, int layout,
                        void* stream) {
  if (layout != QW4_LAYOUT_AWQ_K && layout != QW4_LAYOUT_AWQ_N) return QW4_ERR_LAYOUT;
  return repack_into(w, row_offset, qweight, scales, zeros, out_f, layout, stream);
}

int qw4_dequant_rows(uint16_t* dst, const qw4_weights* w, int row0, int nrows, void* stream) {
  int st = check_weights(w);
  if (st) return st;
  if (!dst) return QW4_ERR_NULL;
  if (row0 < 0 || nrows < 0 || row0 + nrows > w->out_f) return QW4_ERR_SHAPE;
  if (((uintptr_t)dst & 15) != 0) return QW4_ERR_ALIGN;
  if (nrows == 0) return QW4_OK;
  const int tiles = ((row0 + nrows - 1) >> 6) - (row0 >> 6) + 1;
  const unsigned items = (unsigned)tiles * ((w->num_groups + kDeqGroups - 1) / kDeqGroups);
  // As many rounds of rows per workgroup as leave the CUs enough of them (us with
  // one / two / four / eight: 64 rows of K = 4096 2.8 / 2.9 / 3.3 / 4.2, 512 rows of K =
  // 5120 3.9 / 3.7 / 4.0 / 4.8, 2048 8.5 / 7.7 / 6.9 / 7.8, 7168 25.5 / 21.7 / 20.3 / 23.5;
  // 7168 just repacked, three repacks included, 42.9 / 38.6 / 35.9 / 37.2)
  const auto launch = [&](auto it) {
    constexpr int kIt = decltype(it)::value;
    k_dequant_rows<kIt><<<items * (kDeqIters / kIt), 256, 0, (hipStream_t)stream>>>(
        dst, w->qweight, w->scale, w->zeros, row0, nrows, w->in_f, w->num_groups);
  };
  if (items <= 160)
    launch(std::integral_constant<int, 1>{});
  else if (items <= 512)
    launch(std::integral_constant<int, 2>{});
  else
    launch(std::integral_constant<int, 4>{});
  QW4_LAUNCH_CHECK();
  return QW4_OK;
}

int qw4_quantize_w4a16(qw4_weights* w, const uint16_t* src, int out_f, int in_f, int group_size,
                       void* stream) {
  if (!w || !src) return QW4_ERR_NULL;
  std::memset(w, 0, sizeof(*w));
  if (group_size != kGroup) return QW4_ERR_GROUP;
  if (out_f <= 0 || out_f % kTileN || in_f <= 0 || in_f % kGroup) return QW4_ERR_SHAPE;
  const int st = qw4_weights_alloc(w, out_f, in_f, group_size, stream);
  if (st) return st;
  const size_t n = (size_t)(out_f / 4) * w->num_groups;
  k_quant_i4<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(w->qweight, w->scale, w->zeros,
                                                                  src, out_f, in_f, w->num_groups);
  QW4_LAUNCH_CHECK();
  return QW4_OK;
}

int qw4_w8_quantize(qw4_w8_weights* w, const uint16_t* src, int out_f, int in_f,
                    int group_size, void* stream) {
  if (!w || !src) return QW4_ERR_NULL;
  std::memset(w, 0, sizeof(*w));
  if (group_size != kGroup) return QW4_ERR_GROUP;
  if (out_f <= 0 || out_f % kTileN || in_f <= 0 || in_f % kGroup) return QW4_ERR_SHAPE;
  if ((size_t)out_f * in_f >= (1ull << 32)) return QW4_ERR_SHAPE;
  if ((uintptr_t)src & 15) return QW4_ERR_ALIGN;
  const int G = in_f / kGroup;
  hipError_t e = hipMalloc((void**)&w->qweight, (size_t)out_f * in_f);
  if (e == hipSuccess) e = hipMalloc((void**)&w->scale, (size_t)out_f * G * 2);
  if (e != hipSuccess) {
    set_hip_error((int)e);
    (void)hipGetLastError();
    if (w->qweight) (void)hipFree(w->qweight);
    if (w->scale) (void)hipFree(w->scale);
    std::memset(w, 0, sizeof(*w));
    return QW4_ERR_NOMEM;
  }
  w->out_f = out_f;
  w->in_f = in_f;
  w->group_size = group_size;
  w->num_groups = G;
  const size_t n = (size_t)out_f * G;
  k_w8_quantize<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(w->qweight, w->scale, src,
                                                                    out_f, in_f, G);
  QW4_LAUNCH_CHECK();
  return QW4_OK;
}

int qw4_w8_free(qw4_w8_weights* w) {
  if (!w) return QW4_ERR_NULL;
  if (w->qweight) (void)hipFree(w->qweight);
  if (w->scale) (void)hipFree(w->scale);
  std::memset(w, 0, sizeof(*w));
  return QW4_OK;
}

size_t qw4_w8_bytes(const qw4_w8_weights* w) {
  if (!w) return 0;
  return (size_t)w->out_f * w->in_f + (size_t)w->out_f * w->num_groups * 2;
}

int qw4_w8_dequant_rows(uint16_t* dst, const qw4_w8_weights* w, int row0, int nrows,
                        void* stream) {
  if (!dst || !w || !w->qweight || !w->scale) return QW4_ERR_NULL;
  if (w->group_size != kGroup || w->out_f % kTileN || w->in_f % kGroup ||
      w->num_groups != w->in_f / kGroup)
    return QW4_ERR_SHAPE;
  if (row0 < 0 || nrows < 0 || row0 + nrows > w->out_f) return QW4_ERR_SHAPE;
  if (((uintptr_t)dst & 15) != 0) return QW4_ERR_ALIGN;
  if (nrows == 0) return QW4_OK;
  const size_t n = (size_t)nrows * (w->in_f / 8);
  k_w8_dequant_rows<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(
      dst, w->qweight, w->scale, row0, nrows, w->in_f, w->num_groups);
  QW4_LAUNCH_CHECK();
  return QW4_OK;
}

int qw4_gen_bf16(uint16_t* out, size_t count, uint64_t seed, uint64_t stream_id,
                 uint64_t offset, int kind, void* stream) {
  if (!out) return QW4_ERR_NULL;
  if (count == 0) return QW4_OK;
  const unsigned nb = (unsigned)std::min<size_t>(blocks_for(count, 256), 65536);
  k_gen_bf16<<<nb, 256, 0, (hipStream_t)stream>>>(out, count, seed, stream_id, offset, kind);
  QW4_LAUNCH_CHECK();
  return QW4_OK;
}

int qw4_gen_awq_k(uint32_t* qweight, uint16_t* scales, uint32_t* zeros, int out_f, int in_f,
                  uint64_t seed, uint64_t tensor, void* stream) {
  if (!qweight || !scales || !zeros) return QW4_ERR_NULL;
  if (out_f <= 0 || out_f % 8 || in_f <= 0 || in_f % kGroup) return QW4_ERR_SHAPE;
  hipStream_t hs = (hipStream_t)stream;
  const size_t nq = (size_t)(in_f / 8) * out_f;
  k_gen_awq_k_q<<<(unsigned)std::min<size_t>(blocks_for(nq, 256), 65536), 256, 0, hs>>>(
      qweight, out_f, in_f, seed, tensor);
  const size_t nm = (size_t)(in_f / kGroup) * (out_f / 8);
  k_gen_awq_k_meta<<<(unsigned)std::min<size_t>(blocks_for(nm, 256), 65536), 256, 0, hs>>>(
      scales, zeros, out_f, in_f / kGroup, seed, tensor);
  QW4_LAUNCH_CHECK();
  return QW4_OK;
}

int qw4_mfma_peak(uint32_t* sink, int blocks, int iters, void* stream) {
  if (!sink) return QW4_ERR_NULL;
  if (blocks <= 0 || iters <= 0) return QW4_ERR_SHAPE;
  k_mfma_peak<<<blocks, 256, 0, (hipStream_t)stream>>>(sink, iters);
  QW4_LAUNCH_CHECK();
  return QW4_OK;
}

int qw4_stream_read(const void* src, size_t bytes, uint32_t* sink, int blocks, void* stream) {
  if (!src || !sink) return QW4_ERR_NULL;
  if (bytes % 16 || blocks <= 0) return QW4_ERR_SHAPE;
  if ((uintptr_t)src & 15) return QW4_ERR_ALIGN;
  k_stream_read<<<blocks, 256, 0, (hipStream_t)stream>>>(static_cast<const u32x4*>(src),
                                                         bytes / 16, sink);
  QW4_LAUNCH_CHECK();
  return QW4_OK;
}

}  // extern "C"
