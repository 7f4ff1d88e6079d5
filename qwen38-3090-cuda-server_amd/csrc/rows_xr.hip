// k_rows_xr: verify GEMM and heads (M = 2..16) with the activations held in
// registers, for K up to 8 x kXrMaxGroups groups; for K up to 5120 also two
// 16-row blocks of qw4_linear's small row counts (MB = 2).
//
// The work split and the sums are k_rows's (skinny.hip): workgroup p owns whole
// units (S row quads of a tile over all of K), wave w takes the groups w, w + 8,
// ..., the units are summed over the waves in wave order -- so the results are
// bitwise those of k_rows. There, every item (one group of one unit) brings its
// 16 activation rows through LDS: 4 KiB read (and, unstaged, written) for each
// 2 KiB of weights, and four MFMAs with a ones operand for the rows' sums. But a
// wave meets the same NG groups in every unit: here it reads their activation
// operands once into registers (16 NG of them, plus 4 NG for the sums S_m),
// and an item is its weights alone -- half the LDS traffic, two thirds of the
// MFMAs, no activation loads, and the LDS they took holds weights in flight.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/qwen_w4a16.h"
#include "skinny.h"
#include "w4a16_common.h"

namespace qw4 {
namespace {

constexpr int kXrW = 8;           // waves
constexpr int kXrMaxGroups = 8;   // groups a wave can hold: 160 of its 256 registers

// One row m = 4 q + m0 of a unit (lane = c + 16 q): columns 64 b + 4 c + st0 + i.
template <int OUT, int S>
__device__ __forceinline__ void xr_emit(const SkinnyArgs& a, int b, int st0, int m0,
                                        const float (&v)[S], const float (&g)[S], int lane,
                                        float& bv, int& bn) {
  const int c = lane & 15, m = 4 * (lane >> 4) + m0;
  const int n0 = b * kTileN + 4 * c + st0;
  if (OUT == OUT_ARGMAX) {
#pragma unroll
    for (int i = 0; i < S; ++i)
      if (v[i] > bv || (v[i] == bv && n0 + i < bn)) {
        bv = v[i];
        bn = n0 + i;
      }
    return;
  }
  if (m >= a.M) return;
  uint16_t* y = static_cast<uint16_t*>(a.y) + (size_t)m * a.ld + n0;
  uint32_t o[S];
#pragma unroll
  for (int i = 0; i < S; ++i) {
    o[i] = to_bf16(v[i]);
    if (OUT == OUT_RES)
      o[i] = to_bf16(bf16_bits_to_f32(a.res[(size_t)m * a.ld + n0 + i]) + bf16_bits_to_f32(o[i]));
    if (OUT == OUT_SWIGLU) o[i] = swiglu_bf16_bits(to_bf16(g[i]), o[i]);
  }
  if (S == 1)
    y[0] = (uint16_t)o[0];
  else
#pragma unroll
    for (int i = 0; i < S / 2; ++i)
      reinterpret_cast<uint32_t*>(y)[i] = o[2 * i] | (o[2 * i + 1] << 16);
}

template <int OUT, int FMT, int S, int NG, int D, int MB>
__global__ __launch_bounds__(64 * kXrW) void k_rows_xr(SkinnyArgs a) {
  using L = DmaSlot<FMT, S>;
  constexpr int W = kXrW;
  constexpr int kL = L::kLoads;
  constexpr uint32_t kPer = 4 / S;
  constexpr uint32_t kQuad = FMT == 8 ? 512u : 256u;
  // a wave's own area: first the rows of one group and row block on their way
  // into registers (4 KiB), then its partial sums of a unit, two buffers
  constexpr int kArea = 2 * MB * S * 64 > 256 ? 2 * MB * S * 64 : 256;
  __shared__ f32x4 red[W][kArea];
  __shared__ f32x4 csum[MB == 1 ? 1 : W][NG][MB][4];   // MB > 1: the row sums (no registers left)
  extern __shared__ u32x4 xr_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 15, q = lane >> 4;
  const SkinnyRsrc rs = skinny_rsrc(a);
  const int zsh = 16 * (c & 1);
  const uint32_t wbase = Fmt<FMT>::woff(q, c);
  const int p = blockIdx.x;
  // OUT_SWIGLU: units 2v (gate v) and 2v + 1 (its up unit), never split
  const int u0 = OUT == OUT_SWIGLU ? 2 * (int)((long long)p * (a.U / 2) / a.P) : range_start(a, p);
  const int u1 =
      OUT == OUT_SWIGLU ? 2 * (int)((long long)(p + 1) * (a.U / 2) / a.P) : range_start(a, p + 1);
  auto real_unit = [&](int v) {
    return OUT == OUT_SWIGLU ? ((v & 1) ? (v >> 1) + (int)((uint32_t)a.U / 2u) : (v >> 1)) : v;
  };
  const NibConst k = nib_const();
  const int nw = wave < a.G ? (a.G - 1 - wave) / W + 1 : 0;   // groups of this wave (<= NG)
  const int T = nw * (u1 - u0);                                // its items

  // Activation rows of this wave's groups: load t of a row block covers rows 4 t
  // .. 4 t + 3 whole (1 KiB; rows past M are zeros without traffic, whole loads
  // of them are not issued).
  u32x4 x[NG][MB][4];
  const int xrow = lane >> 4, xch = lane & 15;
#pragma unroll
  for (int i = 0; i < NG; ++i)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        x[i][mb][t] = u32x4{0u, 0u, 0u, 0u};
        if (i < nw && 16 * mb + 4 * t < a.M)
          x[i][mb][t] = __builtin_amdgcn_raw_buffer_load_b128(
              rs.x, (uint32_t)(16 * mb + 4 * t + xrow) * (uint32_t)a.K * 2u + (uint32_t)xch * 16u,
              (uint32_t)(wave + W * i) * 256u, 0);
      }
  __builtin_amdgcn_sched_barrier(0);

  // The first D items behind them.
  u32x4* const ring = xr_lds + wave * D * L::kUnits;
  const uint32_t oob_blk = (uint32_t)a.tiles * (uint32_t)a.G;
  int lu = u0, lg = wave;   // load cursor (wave-uniform)
  auto load_slot = [&](int j) __attribute__((always_inline)) {
    const bool in = lu < u1;
    const int ru = real_unit(lu);
    const int st0 = in ? (int)((uint32_t)ru % kPer) * S : 0;
    dma_issue<FMT, S>(ring + j * L::kUnits, rs,
                      in ? (uint32_t)((uint32_t)ru / kPer) * (uint32_t)a.G + (uint32_t)lg : oob_blk,
                      wbase + (uint32_t)st0 * kQuad, lane);
    lg += W;
    if (lg >= a.G) {
      lg = wave;
      ++lu;
    }
  };
#pragma unroll
  for (int j = 0; j < D; ++j) load_slot(j);

  // Each group through the wave's area into MFMA operand order (row c, chunk
  // 4 q + t; chunk j of row r at unit 16 r + (j ^ r): no bank conflicts); the
  // row sums with a ones operand, once per group instead of once per item.
  const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{0x3F803F80u, 0x3F803F80u,
                                                       0x3F803F80u, 0x3F803F80u});
  f32x4 Cs[MB == 1 ? NG : 1];
  {
    u32x4* const area = reinterpret_cast<u32x4*>(red[wave]);
#pragma unroll
    for (int i = 0; i < NG; ++i)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
        for (int t = 0; t < 4; ++t) area[(4 * t + xrow) * 16 + (xch ^ (4 * t + xrow))] = x[i][mb][t];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int t = 0; t < 4; ++t) x[i][mb][t] = area[16 * c + ((4 * q + t) ^ c)];
        __builtin_amdgcn_wave_barrier();
        f32x4 cs;
#pragma unroll
        for (int t = 0; t < 4; ++t)
          cs = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, x[i][mb][t]), ones,
              t == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : cs, 0, 0, 0);
        if (MB == 1)
          Cs[MB == 1 ? i : 0] = cs;
        else if (c == 0)   // the same for all 16 columns
          csum[MB == 1 ? 0 : wave][i][mb][q] = cs;
      }
  }

  f32x4 acc[MB][S];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int i = 0; i < S; ++i) acc[mb][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float bv = -__builtin_inff();   // OUT_ARGMAX: this thread's best of row m
  int bn = 0x7fffffff;
  float gate[S];                  // OUT_SWIGLU: the gate unit's sums
#pragma unroll
  for (int i = 0; i < S; ++i) gate[i] = 0.f;

  int j = 0, left = T;   // slot of the next item, items not yet done
  for (int u = u0; u < u1; ++u) {
    const int ru = real_unit(u);
    const int st0 = (int)((uint32_t)ru % kPer) * S;
    static_for<0, NG>([&](auto ic) __attribute__((always_inline)) {
      constexpr int gi = decltype(ic)::value;
      if (gi >= nw) return;   // wave-uniform
      // this item has landed; the min(D - 1, left - 1) behind it may be in flight
      if (left >= D)
        wait_vm<(D - 1) * kL>();
      else
        wait_items<kL, D>(left - 1);
      RowsData<FMT, S, true> d;
      dma_read<FMT, S, true>(d, ring + j * L::kUnits, lane, st0);
      f32x4 C[MB][S];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < S; ++i) {
          bf16x8 B;
          if (FMT == 4) {
            B = nib8(d.w[i][0][t], k);
          } else {
            const u32x4 v = d.w[i][(t >> 1) & (FMT == 8 ? 1 : 0)];
            B = bytes8_bf16(v[(t & 1) * 2], v[(t & 1) * 2 + 1]);
          }
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
            C[mb][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8, x[gi][mb][t]), B,
                t == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : C[mb][i], 0, 0, 0);
        }
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const f32x4 cs = MB == 1 ? Cs[MB == 1 ? gi : 0] : csum[MB == 1 ? 0 : wave][gi][mb][q];
#pragma unroll
        for (int i = 0; i < S; ++i) {
          const uint32_t sbits = (d.s[i >> 1] >> (16 * (S == 1 ? (st0 & 1) : (i & 1)))) & 0xffffu;
          const float sf = bf16_bits_to_f32(sbits);
          const float zf = FMT == 4 ? 128.0f + (float)((d.z >> (zsh + 4 * (st0 + i))) & 0xFu) : 128.0f;
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) acc[mb][i][jj] += sf * (C[mb][i][jj] - zf * cs[jj]);
        }
      }
      // the slot's reads have returned: load the item D ahead into it
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (left > D) load_slot(j);
      j = j + 1 == D ? 0 : j + 1;
      --left;
    });
    // Unit sums in wave order; row 4 q + jj by wave jj (mod 4) of one half of
    // the workgroup, the halves taking turns. Two buffers, one barrier a unit:
    // a buffer is written again two barriers after it was read.
    const int n = u - u0, par = n & 1;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int i = 0; i < S; ++i) {
        red[wave][((par * MB + mb) * S + i) * 64 + lane] = acc[mb][i];
        acc[mb][i] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    lds_barrier<true>();
    // one row block: the halves of the workgroup take turns; two: a half each
    if (MB == 2 || (wave >> 2) == ((OUT == OUT_SWIGLU ? n >> 1 : n) & 1)) {
      const int jj = wave & 3, mb = MB == 2 ? wave >> 2 : 0;
      float v[S];
#pragma unroll
      for (int i = 0; i < S; ++i) {
        const int at = (((par * MB + mb) * S + i) * 64 + lane) * 4 + jj;
        v[i] = reinterpret_cast<const float*>(red[0])[at];
#pragma unroll
        for (int w = 1; w < W; ++w) v[i] += reinterpret_cast<const float*>(red[w])[at];
      }
      if (OUT == OUT_SWIGLU && (n & 1) == 0) {
#pragma unroll
        for (int i = 0; i < S; ++i) gate[i] = v[i];
      } else {
        const uint32_t ou = OUT == OUT_SWIGLU ? (uint32_t)u >> 1 : (uint32_t)u;   // output unit
        xr_emit<OUT, S>(a, (int)(ou / kPer), (int)(ou % kPer) * S, 16 * mb + jj, v, gate, lane, bv, bn);
      }
    }
  }
  wait_vm<0>();   // no load lands in LDS after the workgroup released it
  if (OUT == OUT_ARGMAX) {
    // the 16 columns of a row, then the two halves' bests, as wave 0's Best
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
      const float v2 = __shfl_xor(bv, off, 64);
      const int n2 = __shfl_xor(bn, off, 64);
      if (v2 > bv || (v2 == bv && n2 < bn)) { bv = v2; bn = n2; }
    }
    lds_barrier<true>();   // every unit's sums have been read
    float* fv = reinterpret_cast<float*>(red[0]);
    int* fn = reinterpret_cast<int*>(red[0]) + 64;
    if (c == 0) {
      fv[wave * 4 + q] = bv;
      fn[wave * 4 + q] = bn;
    }
    lds_barrier<true>();
    if (wave == 0) {
      Best bs;
      best_init(bs);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        best_fold(bs, jj, fv[jj * 4 + q], fn[jj * 4 + q]);
        best_fold(bs, jj, fv[(jj + 4) * 4 + q], fn[(jj + 4) * 4 + q]);
      }
      argmax_arrive(a, p, bs, lane);
    }
  }
}

template <int OUT, int FMT, int S, int NG, int D, int MB = 1>
void launch(const SkinnyArgs& a, bool prepare, hipStream_t st) {
  constexpr auto kern = &k_rows_xr<OUT, FMT, S, NG, D, MB>;
  constexpr int lds = kXrW * D * DmaSlot<FMT, S>::kUnits * 16;
  static_assert(lds + kXrW * (MB * 4096 + NG * MB * 64) <= kLdsBytes, "ring and areas fit the CU's LDS");
  allow_lds<kern>(lds);
  if (!prepare) kern<<<a.P, 64 * kXrW, lds, st>>>(a);
}

// Registers for 3, 5 or 8 groups a wave (K up to 3072, 5120, 8192): 110 to 210
// of the 256, no spills. D3: items in flight where a wave has at most 3 groups.
template <int OUT, int FMT, int S, int D, int D3 = D>
void launch_ng(const SkinnyArgs& a, bool prepare, hipStream_t st) {
  const int ng = (a.G + kXrW - 1) / kXrW;
  if (prepare || ng <= 3) launch<OUT, FMT, S, 3, D3>(a, prepare, st);
  if (prepare || (ng > 3 && ng <= 5)) launch<OUT, FMT, S, 5, D>(a, prepare, st);
  if (prepare || ng > 5) launch<OUT, FMT, S, kXrMaxGroups, D>(a, prepare, st);
}

// Items in flight a wave: 4-bit 32-row units 3 (gate|up at M = 9: 2 19.9, 3
// 19.3, 4 20.1 us; 6 was 7% slower), 16-row units 4; 8-bit 16-row units 2 (the
// 248320-row head at M = 9: 2 214, 4 216, 6 217 us; 32-row units 222), but 4 for a
// short K, whose units end sooner (151936x1024 / 151936x2560 / 32064x2560 at M = 9: 2
// 34.9 / 71.8 / 18.9, 4 31.2 / 68.4 / 18.4, 6 32.5 / 70.8 / 19.4, k_rows 34.0 / 70.8 / 19.3).
template <int OUT, int FMT>
void launch_out(const SkinnyArgs& a, int S, bool prepare, hipStream_t st) {
  if constexpr (FMT == 4) {
    if (prepare || S == 1) launch_ng<OUT, FMT, 1, 4>(a, prepare, st);
    if (prepare || S == 2) launch_ng<OUT, FMT, 2, 3>(a, prepare, st);
  } else {
    launch_ng<OUT, FMT, 1, 2, 4>(a, prepare, st);
  }
}

void dispatch(int out, int fmt, const SkinnyArgs& a, int S, bool prepare, hipStream_t st) {
  if (fmt == 8) {
    if (prepare || out == OUT_BF16) launch_out<OUT_BF16, 8>(a, S, prepare, st);
    if (prepare || out == OUT_ARGMAX) launch_out<OUT_ARGMAX, 8>(a, S, prepare, st);
  } else {
    if (prepare || out == OUT_BF16) launch_out<OUT_BF16, 4>(a, S, prepare, st);
    if (prepare || out == OUT_ARGMAX) launch_out<OUT_ARGMAX, 4>(a, S, prepare, st);
    if (prepare || out == OUT_RES) launch_out<OUT_RES, 4>(a, S, prepare, st);
    if (prepare || out == OUT_SWIGLU) launch_out<OUT_SWIGLU, 4>(a, S, prepare, st);
  }
}

}  // namespace

// Where it is the faster one, measured on MI355X against k_rows (policy) in
// one process:
//  * workgroups own more than one 32-row unit on average (2 tiles > CUs): the
//    rows are loaded once for all of them. gate|up 34816x5120 at M = 2 / 9 / 16
//    21.0 / 21.9 / 22.8 -> 18.8 / 19.3 / 20.3 us, 16384x5120 at M = 9 / 16 11.8 /
//    13.1 -> 10.6 / 11.2, the 248320x5120 INT4 head with argmax at M = 9 / 16 129 /
//    163 -> 110 / 111, the 8-bit one at M = 9 257 -> 217. With one unit each the
//    rows cost as much either way (7168x5120 at M = 9 7.2 against 7.1) and the
//    passage through the areas comes before the first item (5120x6144 8.2
//    against 7.6), so k_rows keeps those;
//  * 16-row units (fewer than CUs / 4 tiles) with 8 rows or more, where k_rows
//    loads the rows into registers item by item: 896x5120 at M = 9 / 16 6.6 / 8.6 ->
//    6.0 / 6.3 us, but at M = 2 4.9 against 5.5.
bool rows_xr_launch(int out, int fmt, SkinnyArgs& a, int cus, hipStream_t st) {
  if (a.M < 2 || a.G > kXrW * kXrMaxGroups) return false;
  if (out != OUT_BF16 && out != OUT_ARGMAX && (fmt == 8 || (out != OUT_RES && out != OUT_SWIGLU)))
    return false;
  const bool small = out != OUT_SWIGLU && 4 * a.tiles < cus;   // 16-row units in k_rows
  if (!(2 * a.tiles > cus || (small && a.M >= 8))) return false;
  const int S = fmt == 8 || small ? 1 : 2;
  a.U = a.tiles * 4 / S;
  // as few workgroups as give none of them another unit: each brings all rows of
  // x (M = 2 / 9 / 16, against a workgroup per CU: 34816x5120 18.8 / 20.2 / 20.6 us, 19.2 /
  // 20.0 / 20.7; 28672x4096 13.7 / 14.3 / 14.9, 13.9 / 14.7 / 15.4; 34816x8192 28.7 / 29.9 /
  // 31.3, 29.2 / 31.7 / 31.7; 9472x5120 9.7 / 10.0 / 10.4, 9.3 / 9.9 / 10.6); the 8-bit heads own tens of units each, and with a short K every
  // workgroup streams for longer than it loads rows (151936x2560 at M = 9: 69.9 us
  // with 250 workgroups, 68.4 with 256)
  const int n = out == OUT_SWIGLU ? a.U / 2 : a.U, most = (n + cus - 1) / cus;
  a.P = fmt == 8 && a.G <= 3 * kXrW ? std::min(n, cus) : (n + most - 1) / most;
  dispatch(out, fmt, a, S, false, st);
  return true;
}

// Two row blocks (17 to 32 rows of qw4_linear) in one pass, each bitwise what a
// pass of its own gives, for K up to 5120 (32 registers a group: 230 in all, no
// spills). Faster than two passes at every size measured (32 rows): gate|up
// 34816x5120 40.0 -> 27.5 us, 7168x5120 15.5 -> 11.4, 5120x4096 12.9 -> 10.3,
// 896x5120 12.3 -> 10.8, 5120x512 7.9 -> 6.0.
bool rows_xr2_launch(SkinnyArgs& a, int cus, hipStream_t st) {
  const int ng = (a.G + kXrW - 1) / kXrW;
  if (a.M < 17 || a.M > 32 || ng > 5) return false;
  a.U = a.tiles * 2;
  const int most = (a.U + cus - 1) / cus;
  a.P = (a.U + most - 1) / most;
  if (ng <= 3)
    launch<OUT_BF16, 4, 2, 3, 3, 2>(a, false, st);
  else
    launch<OUT_BF16, 4, 2, 5, 3, 2>(a, false, st);
  return true;
}

void rows_xr_prepare() {
  SkinnyArgs a{};
  launch<OUT_BF16, 4, 2, 3, 3, 2>(a, true, nullptr);
  launch<OUT_BF16, 4, 2, 5, 3, 2>(a, true, nullptr);
  dispatch(0, 4, a, 0, true, nullptr);
  dispatch(0, 8, a, 0, true, nullptr);
}

}  // namespace qw4
