// Shared by the skinny GEMV / GEMM translation units: kernel arguments, buffer
// resources, item loads into LDS slots, the bf16-MFMA math of one item and the
// epilogues.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <mutex>
#include <type_traits>

#include "../../include/qwen_w4a16.h"
#include "w4a16_common.h"

namespace qw4 {
// Cache policy of the decode kernels' weight loads: nontemporal (each byte is
// read once per call; measured 3-6% faster than the default policy).
constexpr int kWeightAux = 2;

// Epilogues of the skinny kernels:
//   OUT_BF16   y = bf16(acc)
//   OUT_F32    y = acc
//   OUT_ARGMAX the row argmax of acc (no logits written)
//   OUT_RES    y = bf16(res + bf16(acc)): linear then residual_add
//              (src/model/model.cu:781-783; y may be res)
//   OUT_SWIGLU y = bf16(silu(bf16(acc_gate)) * bf16(acc_up)) over a fused
//              [gate | up] weight: linear then swiglu (model.cu:776-778)
//   OUT_NORM   bf16 y of rmsnorm(x): rmsnorm then linear (model.cu:773-777)
enum { OUT_BF16 = 0, OUT_F32 = 1, OUT_ARGMAX = 2, OUT_RES = 3, OUT_SWIGLU = 4, OUT_NORM = 5 };

// Memory-side atomics on one cache line serialize; each counter gets its own line.
constexpr int kCounterStride = 32;
constexpr int kKeyGroups = 64;

struct SkinnyArgs {
  const uint32_t* qw;
  const uint16_t* sc;
  const uint16_t* zr;
  const uint16_t* x;
  void* y;
  uint32_t* counters;   // argmax arrival counters, one per 128-byte line
                        // (kCounterStride words): [0, 64) per key group,
                        // [64] of key groups
  uint64_t* keys;       // argmax keys [64 groups][16 rows], one line per group
  int M, N, K, G, tiles, P, U;
  uint32_t weight_bytes;   // packed weights (4- or 8-bit blocks)
  const uint16_t* res;     // OUT_RES: residual [M][N] (may be y)
  const uint16_t* nw;      // OUT_NORM: rmsnorm weight [K] (applied as 1 + w)
  float eps;               // OUT_NORM: rmsnorm epsilon
  int ld;                  // row stride of y (N; the intermediate size for OUT_SWIGLU)
};

// Monotonic key: larger value first, then lower index (elementwise.cu:103-104).
__device__ __forceinline__ uint64_t argmax_key(float v, int n) {
  uint32_t u = __float_as_uint(v);
  u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  return ((uint64_t)u << 32) | (uint64_t)(~(uint32_t)n);
}

// Arrival: release this workgroup's key updates, and acquire those of the
// workgroups counted before it (the last arriver then reads every key).
__device__ __forceinline__ uint32_t arrive_dev(uint32_t* p) {
  return __hip_atomic_fetch_add(p, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void clear_dev(uint32_t* p) {
  __hip_atomic_store(p, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Wait until every memory operation this wave issued has completed.
__device__ __forceinline__ void wait_all_mem() { __builtin_amdgcn_s_waitcnt(0); }

// Workgroup p owns units [start(p), start(p + 1)).
__device__ __forceinline__ int range_start(const SkinnyArgs& a, int p) {
  return (int)((long long)p * a.U / a.P);
}

// Buffer-resource loads: a loop-invariant per-lane offset plus a wave-uniform
// scalar offset per block. Activation rows past M lie outside the x resource
// (M rows of K) and read as zeros without touching memory: for M = 1, 60 of
// the 64 lanes issue no activation traffic.
struct SkinnyRsrc {
  __amdgpu_buffer_rsrc_t qw, sc, zr, x;
};

__device__ __forceinline__ SkinnyRsrc skinny_rsrc(const SkinnyArgs& a) {
  SkinnyRsrc r;
  r.qw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(a.qw), 0, (int)a.weight_bytes,
                                           0x00020000);
  // 4-bit: 160-byte (scale, zero-point) records per block; 8-bit: 128 bytes of scales
  r.sc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.sc), 0,
      (int)((uint32_t)a.N / kTileN * (uint32_t)a.G * (a.zr ? (uint32_t)kMetaBytes : 128u)),
      0x00020000);
  r.zr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.zr), 0,
                                           a.zr ? (int)((uint32_t)a.N * (uint32_t)a.G / 2u) : 0,
                                           0x00020000);
  r.x = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.x), 0,
                                          (int)((uint32_t)a.M * (uint32_t)a.K * 2u), 0x00020000);
  return r;
}

// ------------------------------------------------------- 8-bit weights
// W8A16 (the reference's lm_head format, gemv_w4a16.cuh:141-166): per (row,
// 128-group) a bf16 scale and int8 q in [-127, 127], stored as the byte
// u = q + 128. Block = (64-row tile, group), 8 KiB: [4 j][64 p][32 B], position
// p holding row 4 (p % 16) + p / 16 as in the 4-bit layout, chunk j covering
// k = 128 g + 32 j + [0, 32) in natural byte order. A byte is an exact bf16
// (u <= 255 needs 8 significant bits); the offset is removed like the 4-bit
// zero point: acc += s (C - 128 S_m), with S_m from the ones operand.
// Eight bytes -> eight bf16 values (exact).
__device__ __forceinline__ bf16x8 bytes8_bf16(uint32_t lo, uint32_t hi) {
  u32x4 o;
  o[0] = pack_bf16x2((float)(lo & 0xffu), (float)((lo >> 8) & 0xffu));
  o[1] = pack_bf16x2((float)((lo >> 16) & 0xffu), (float)(lo >> 24));
  o[2] = pack_bf16x2((float)(hi & 0xffu), (float)((hi >> 8) & 0xffu));
  o[3] = pack_bf16x2((float)((hi >> 16) & 0xffu), (float)(hi >> 24));
  return __builtin_bit_cast(bf16x8, o);
}

// Lane offset of its 16-byte chunk inside a block, per weight format: chunk
// q of position c (4-bit: 1 KiB per chunk; 8-bit: 2 KiB, two 16-byte halves).
template <int FMT>
struct Fmt {
  __device__ static uint32_t woff(int q, int c) {
    return FMT == 8 ? (uint32_t)(q * 2048 + c * 32) : (uint32_t)(q * 1024 + c * 16);
  }
};

// ------------------------------------------------------------- epilogues
// Running argmax of one workgroup: per lane, the best (value, column) of rows
// m = 4q + jj over the elements this workgroup finished.
struct Best {
  float v[4];
  int n[4];
};

__device__ __forceinline__ void best_init(Best& bs) {
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) {
    bs.v[jj] = -__builtin_inff();
    bs.n[jj] = 0x7fffffff;
  }
}

__device__ __forceinline__ void best_fold(Best& bs, int jj, float v, int n) {
  if (v > bs.v[jj] || (v == bs.v[jj] && n < bs.n[jj])) {
    bs.v[jj] = v;
    bs.n[jj] = n;
  }
}

// Wave 0 at the end of an argmax workgroup: fold the workgroup's best per row
// into key group p % 64 (one cache line per group); the last workgroup of a
// group bumps the group counter, and the last group to finish folds the 64
// groups, writes the indices and clears the state for the next call.
__device__ __forceinline__ void argmax_arrive(const SkinnyArgs& a, int p, Best& bs, int lane) {
  const int c = lane & 15, q = lane >> 4;
  const int grp = p % kKeyGroups;
  uint64_t* gkeys = a.keys + grp * 16;
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) {
    float v = bs.v[jj];
    int n = bs.n[jj];
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
      const float v2 = __shfl_xor(v, off, 64);
      const int n2 = __shfl_xor(n, off, 64);
      if (v2 > v || (v2 == v && n2 < n)) { v = v2; n = n2; }
    }
    const int m = 4 * q + jj;
    if (c == 0 && m < a.M)
      __hip_atomic_fetch_max(&gkeys[m], argmax_key(v, n), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
  }
  wait_all_mem();   // key updates complete before this workgroup is counted
  const int ngroups = a.P < kKeyGroups ? a.P : kKeyGroups;
  bool last = false;
  if (lane == 0) {
    const uint32_t in_grp = (uint32_t)((a.P - 1 - grp) / kKeyGroups + 1);
    uint32_t* gcnt = a.counters + (size_t)grp * kCounterStride;
    uint32_t* done = a.counters + (size_t)kKeyGroups * kCounterStride;
    // memory order: each workgroup's key updates happen before its release
    // increment of its group counter; the group's last arriver acquires them
    // and releases them on `done`, whose last arriver acquires all of them
    last = arrive_dev(gcnt) == in_grp - 1 && arrive_dev(done) == (uint32_t)(ngroups - 1);
  }
  if (!__builtin_amdgcn_readfirstlane((int)last)) return;
  // The last workgroup folds the groups: lane 16 h + m takes row m of groups
  // 16 h .. 16 h + 15, its loads in flight together, then the four quarters
  // meet. One lane reading every key one after another cost 8 us a row (INT4
  // head of 248320 rows, M = 9: 201 -> 129 us).
  static_assert(kKeyGroups == 64, "16 groups per quarter of the wave");
  uint64_t* const rkeys = a.keys + (size_t)q * 256 + c;   // row c, group 16 q
  uint64_t key[16], best = 0;
#pragma unroll
  for (int g2 = 0; g2 < 16; ++g2)   // zero for groups and rows that have none
    key[g2] = __hip_atomic_load(&rkeys[16 * g2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
  for (int g2 = 0; g2 < 16; ++g2) {
    best = key[g2] > best ? key[g2] : best;
    __hip_atomic_store(&rkeys[16 * g2], (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
#pragma unroll
  for (int off = 16; off < 64; off <<= 1) {
    const uint64_t o = (uint64_t)__shfl_xor((unsigned long long)best, off, 64);
    best = o > best ? o : best;
  }
  if (lane < 16 && lane < a.M)
    static_cast<int32_t*>(a.y)[lane] = (int32_t)(~(uint32_t)(best & 0xffffffffu));
  if (lane < ngroups) clear_dev(a.counters + (size_t)lane * kCounterStride);
  if (lane == 0) clear_dev(a.counters + (size_t)kKeyGroups * kCounterStride);
}

constexpr int kLdsBytes = 160 * 1024;   // LDS per CU on gfx950

template <int FMT, int S, bool XL>
struct RowsData {
  u32x4 w[S][FMT == 8 ? 2 : 1];
  u32x4 x[XL ? 1 : 4];       // activations (registers) unless they sit in LDS
  uint32_t s[(S + 1) / 2];   // bf16 scales of rows 4c + st0 + i, two per word
  uint32_t z;                // zero points of rows 4c .. 4c + 3 (4-bit)
};

template <int FMT, int S, bool XL>
__device__ __forceinline__ void rows_load(RowsData<FMT, S, XL>& d, const SkinnyRsrc& r, uint32_t blk,
                                          int g, uint32_t woff, uint32_t soff, uint32_t zoff,
                                          uint32_t xoff) {
  constexpr uint32_t kBlk = FMT == 8 ? 8192u : 4096u;
  constexpr uint32_t kQuad = FMT == 8 ? 512u : 256u;   // bytes of one row quad in a chunk
  constexpr uint32_t kScB = FMT == 8 ? 128u : (uint32_t)kMetaBytes;   // scale bytes per block
#pragma unroll
  for (int i = 0; i < S; ++i)
#pragma unroll
    for (int h = 0; h < (FMT == 8 ? 2 : 1); ++h)
      d.w[i][h] = __builtin_amdgcn_raw_buffer_load_b128(r.qw, woff + i * kQuad + h * 16,
                                                        blk * kBlk, kWeightAux);
  if (!XL) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
      d.x[t & (XL ? 0 : 3)] =
          __builtin_amdgcn_raw_buffer_load_b128(r.x, xoff + t * 16, (uint32_t)g * 256u, 0);
  }
  if (S == 4) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r.sc, soff, blk * kScB, 0);
    d.s[0] = v[0];
    d.s[(S + 1) / 2 - 1] = v[1];
  } else if (S == 2) {
    d.s[0] = __builtin_amdgcn_raw_buffer_load_b32(r.sc, soff, blk * kScB, 0);
  } else {
    // the aligned word holding this row's scale (half st0 & 1)
    d.s[0] = __builtin_amdgcn_raw_buffer_load_b32(r.sc, soff & ~3u, blk * kScB, 0);
  }
  // 32-bit loads only: a 16-bit load result gets masked right after the load,
  // which makes the compiler wait for it there (zoff: the aligned word holding
  // this lane's 16 bits)
  if (FMT == 4) d.z = __builtin_amdgcn_raw_buffer_load_b32(r.zr, zoff, blk * 32u, 0);
}

// ---- LDS-DMA items (k_rows with DMA): the weight, scale and zero-point
// loads of an item go straight into an LDS slot of the wave (buffer_load ...
// lds, lane i's bytes at slot + i * size), so the number of items in flight is
// bounded by LDS, not by registers. The compiler does not order LDS reads
// after these loads: each item waits with an explicit vmcnt (the loads issued
// after it, which complete after it) before reading its slot.
// Slot layout (16-byte units): NQ x 64 weight chunks, then a 256-byte area
// for the block's metadata, one 4-byte load per lane: 4-bit, the 160-byte
// (scale, zero-point) record (lane l < 40: word l; the others repeat word 0);
// 8-bit, the 128 bytes of scales (lane l: word l & 31). One metadata load per
// item instead of a scale and a zero-point load: every LDS-DMA instruction
// holds the CU's address unit ~16 cycles whatever its size.
template <int FMT, int S>
struct DmaSlot {
  static constexpr int kH = FMT == 8 ? 2 : 1;          // 16-byte chunks per row quad
  static constexpr int kNQ = S * kH;                     // weight loads per item
  static constexpr int kLoads = kNQ + 1;                 // loads per item
  static constexpr int kUnits = kNQ * 64 + 16;
};

// k_rows item slot with LDS-DMA items (16-byte units): DmaSlot's weights and
// metadata, then -- when the activations are not staged for the whole
// workgroup (!XL: M > 1 rows of a long K) -- the item's group of all 16
// activation rows (rows past M read as zeros), 16 chunks per row, chunk j of
// row r at unit 16 r + (j ^ r): the 16 lanes reading one k-chunk of rows
// 0..15 hit 16 different 16-byte bank groups.
template <int FMT, int S, bool XL>
constexpr int rows_slot_units() {
  return DmaSlot<FMT, S>::kUnits + (XL ? 0 : 256);
}

// 16 bytes per lane, nontemporal (weights); 4 bytes per lane (metadata)
__device__ __forceinline__ void dma_load16(__amdgpu_buffer_rsrc_t r, u32x4* dst, uint32_t voff,
                                           uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16,
                                           voff, soff, 0, kWeightAux);
}
// 16 bytes per lane, default cache policy (activations: every workgroup
// reads them, mostly from L2)
__device__ __forceinline__ void dma_load16c(__amdgpu_buffer_rsrc_t r, u32x4* dst, uint32_t voff,
                                            uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16,
                                           voff, soff, 0, 0);
}
__device__ __forceinline__ void dma_load4(__amdgpu_buffer_rsrc_t r, u32x4* dst, uint32_t voff,
                                          uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 4,
                                           voff, soff, 0, 0);
}

// Wait until at most N vector-memory operations of this wave are outstanding.
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N <= 63, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Workgroup barrier for LDS data written by ds_write. With LDS-DMA loads in
// flight __syncthreads() would also wait for all of them (its fence counts
// them as LDS writes); the unit sums only need this wave's LDS writes done.
template <bool DMA>
__device__ __forceinline__ void lds_barrier() {
  if constexpr (DMA)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  else
    __syncthreads();
}

template <int J, int D, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (J < D) {
    f(std::integral_constant<int, J>{});
    static_for<J + 1, D>(f);
  }
}

// Wait until at most n items' loads (kL each) of this wave are outstanding,
// n in [0, D) known only at run time (the immediate needs a switch).
template <int kL, int D>
__device__ __forceinline__ void wait_items(int n) {
  static_for<0, D>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    if (n == i) wait_vm<i * kL>();
  });
}


template <int FMT, int S>
__device__ __forceinline__ void dma_issue(u32x4* slot, const SkinnyRsrc& r, uint32_t blk,
                                          uint32_t woff, int lane) {
  using L = DmaSlot<FMT, S>;
  constexpr uint32_t kBlk = FMT == 8 ? 8192u : 4096u;
  constexpr uint32_t kQuad = FMT == 8 ? 512u : 256u;
#pragma unroll
  for (int i = 0; i < S; ++i)
#pragma unroll
    for (int h = 0; h < L::kH; ++h)
      dma_load16(r.qw, slot + (i * L::kH + h) * 64, woff + i * kQuad + h * 16, blk * kBlk);
  if (FMT == 4)
    dma_load4(r.sc, slot + L::kNQ * 64, lane < 40 ? (uint32_t)lane * 4u : 0u,
              blk * (uint32_t)kMetaBytes);
  else
    dma_load4(r.sc, slot + L::kNQ * 64, (uint32_t)(lane & 31) * 4u, blk * 128u);
}

template <int FMT, int S, bool XL>
__device__ __forceinline__ void dma_read(RowsData<FMT, S, XL>& d, const u32x4* slot, int lane,
                                         int st0) {
  using L = DmaSlot<FMT, S>;
  const int c = lane & 15;
#pragma unroll
  for (int i = 0; i < S; ++i)
#pragma unroll
    for (int h = 0; h < L::kH; ++h) d.w[i][h] = slot[(i * L::kH + h) * 64 + lane];
  const uint32_t* sm = reinterpret_cast<const uint32_t*>(slot + L::kNQ * 64);
  if (S == 4) {
    d.s[0] = sm[2 * c];
    d.s[(S + 1) / 2 - 1] = sm[2 * c + 1];
  } else {
    d.s[0] = sm[(4 * c + st0) >> 1];
  }
  if (FMT == 4) d.z = sm[32 + (c >> 1)];   // the record's copy of the zero-point words
}

// XL: activations come from LDS (xl: this lane's row, k chunk q, group g);
// otherwise from the registers rows_load filled. JJ: the output rows
// m = 4q + jj, jj < JJ, that are accumulated (M = 1: only jj = 0 is read).
template <int FMT, int S, bool XL, int JJ = 4>
__device__ __forceinline__ void rows_mma(f32x4 (&acc)[S], const RowsData<FMT, S, XL>& d, NibConst k,
                                         int st0, int zsh, const u32x4* xl) {
  const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{0x3F803F80u, 0x3F803F80u,
                                                       0x3F803F80u, 0x3F803F80u});
  f32x4 C[S], Cs;
  u32x4 xr[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) xr[t] = XL ? xl[t] : d.x[t & (XL ? 0 : 3)];
  // Scale and zero point first, pinned here: the loaded words must be dead
  // before the caller reloads this buffer, or the compiler keeps both copies
  // and moves them at the loop's back edge (waiting for the newest loads).
  float sf[S], zf[S];
#pragma unroll
  for (int i = 0; i < S; ++i) {
    const uint32_t sbits = (d.s[i >> 1] >> (16 * (S == 1 ? (st0 & 1) : (i & 1)))) & 0xffffu;
    sf[i] = bf16_bits_to_f32(sbits);
    zf[i] = FMT == 4 ? 128.0f + (float)((d.z >> (zsh + 4 * (st0 + i))) & 0xFu) : 128.0f;
    // staged activations (M = 1): pinned here, so the loaded words are dead
    // before the caller reloads the buffer (measured 1% faster; with
    // activations in registers the extra live values would spill)
    if (XL) asm volatile("" : "+v"(sf[i]), "+v"(zf[i])::"memory");
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const bf16x8 A = __builtin_bit_cast(bf16x8, xr[t]);
#pragma unroll
    for (int i = 0; i < S; ++i) {
      bf16x8 B;
      if (FMT == 4) {
        B = nib8(d.w[i][0][t], k);
      } else {
        const u32x4 v = d.w[i][(t >> 1) & (FMT == 8 ? 1 : 0)];
        B = bytes8_bf16(v[(t & 1) * 2], v[(t & 1) * 2 + 1]);
      }
      C[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          A, B, t == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : C[i], 0, 0, 0);
    }
    Cs = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, ones,
                                                 t == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : Cs,
                                                 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < S; ++i)
#pragma unroll
    for (int jj = 0; jj < JJ; ++jj) acc[i][jj] += sf[i] * (C[i][jj] - zf[i] * Cs[jj]);
}

// Final values of one unit (wave 0): rows m = 4q + jj, columns b*64 + 4c + st0 + i.
template <int OUT, int S>
__device__ __forceinline__ void emit_rows(const SkinnyArgs& a, int b, int st0,
                                          const f32x4 (&acc)[S], int lane, Best& bs) {
  const int c = lane & 15, q = lane >> 4;
  const int n0 = b * kTileN + 4 * c + st0;
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) {
    const int m = 4 * q + jj;
    if (OUT == OUT_ARGMAX) {
#pragma unroll
      for (int i = 0; i < S; ++i) best_fold(bs, jj, acc[i][jj], n0 + i);
      continue;
    }
    if (m >= a.M) continue;
    if (OUT == OUT_RES) {
      // bf16(res + bf16(acc)), the reference's linear then residual_add
      uint16_t* y = static_cast<uint16_t*>(a.y) + (size_t)m * a.ld + n0;
      const uint16_t* r = a.res + (size_t)m * a.ld + n0;
#pragma unroll
      for (int i = 0; i < S; ++i)
        y[i] = to_bf16(bf16_bits_to_f32(r[i]) + bf16_bits_to_f32(to_bf16(acc[i][jj])));
    } else if (OUT == OUT_BF16 || OUT == OUT_NORM) {
      uint16_t* y = static_cast<uint16_t*>(a.y) + (size_t)m * a.ld + n0;
      if (S == 4)
        *reinterpret_cast<u32x2*>(y) = u32x2{pack_bf16x2(acc[0][jj], acc[1 % S][jj]),
                                             pack_bf16x2(acc[2 % S][jj], acc[3 % S][jj])};
      else if (S == 2)
        *reinterpret_cast<uint32_t*>(y) = pack_bf16x2(acc[0][jj], acc[1 % S][jj]);
      else
        *y = to_bf16(acc[0][jj]);
    } else {
      float* y = static_cast<float*>(a.y) + (size_t)m * a.ld + n0;
#pragma unroll
      for (int i = 0; i < S; ++i) y[i] = acc[i][jj];
    }
  }
}


// OUT_SWIGLU (wave 0): gate rows of tile b (the intermediate index), their up
// rows' sums in u.
template <int S>
__device__ __forceinline__ void emit_swiglu(const SkinnyArgs& a, int b, int st0,
                                            const f32x4 (&g)[S], const f32x4 (&u)[S], int lane) {
  const int c = lane & 15, q = lane >> 4;
  const int n0 = b * kTileN + 4 * c + st0;
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) {
    const int m = 4 * q + jj;
    if (m >= a.M) continue;
    uint16_t* y = static_cast<uint16_t*>(a.y) + (size_t)m * a.ld + n0;
#pragma unroll
    for (int i = 0; i < S; ++i) y[i] = swiglu_bf16_bits(to_bf16(g[i][jj]), to_bf16(u[i][jj]));
  }
}

// ------------------------------------------------------------- host side
constexpr int kMaxDevices = 64;

inline int current_device() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) dev = 0;
  return dev;
}

// Dynamic LDS above the default limit is allowed per kernel, once per device:
// qw4_scratch_alloc raises every LDS-DMA kernel to its maximum, so no launch --
// captured into a graph or not -- has to. A launch that needs more than a
// kernel was raised to (no scratch allocated on this device yet) raises it
// under a lock.
inline std::mutex g_lds_mutex;

template <auto Kern>
void allow_lds(int bytes) {
  static std::atomic<int> set[kMaxDevices];
  std::atomic<int>& v = set[current_device()];
  if (bytes <= v.load(std::memory_order_acquire)) return;
  std::lock_guard<std::mutex> lock(g_lds_mutex);
  if (bytes <= v.load(std::memory_order_relaxed)) return;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(Kern),
                          hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess)
    v.store(bytes, std::memory_order_release);
  else
    (void)hipGetLastError();   // not sticky: the launch reports what matters
}

// k_rows_xr (rows_xr.hip): launches it for these arguments (P and U filled in)
// and returns true, or returns false where it does not apply.
bool rows_xr_launch(int out, int fmt, SkinnyArgs& a, int cus, hipStream_t st);
bool rows_xr2_launch(SkinnyArgs& a, int cus, hipStream_t st);   // 17 to 32 rows
// qw4_linear's 17 to 32 rows over one reading of the weights, each bitwise a
// 16-row pass's (skinny.hip); *taken false where that form does not apply.
int skinny_rows32(uint16_t* y, const qw4_weights* w, const uint16_t* x, int M, qw4_scratch* s,
                  void* stream, bool* taken);
void rows_xr_prepare();   // raises its kernels' dynamic LDS limits on this device

}  // namespace qw4
