// Row argmax over bf16 logits, lowest index on ties -- the call-compatible
// counterparts of argmax / argmax_rows (src/kernels/elementwise.cu:96-158,
// :184-194). The lm_head path itself uses the fused fp32 argmax of the skinny
// kernel; these serve callers that already hold bf16 logits.
#include <hip/hip_runtime.h>

#include <cfloat>

#include "../../include/qwen_w4a16.h"
#include "w4a16_common.h"

namespace qw4 {
namespace {

__device__ __forceinline__ void better(float& v, int& i, float v2, int i2) {
  if (v2 > v || (v2 == v && i2 < i)) { v = v2; i = i2; }
}

// Block-wide (64 W threads) reduction of (value, index) pairs; thread 0's result.
template <int W>
__device__ __forceinline__ void block_best(float& v, int& i) {
  __shared__ float sv[W];
  __shared__ int si[W];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) better(v, i, __shfl_xor(v, off, 64), __shfl_xor(i, off, 64));
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { sv[wave] = v; si[wave] = i; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < W; ++w) better(v, i, sv[w], si[w]);
  }
}

__device__ __forceinline__ float ldbf(const uint16_t* p) { return bf16_bits_to_f32(*p); }

// Same semantics as the reference's kernels: each thread starts from
// (-FLT_MAX, 0) and takes a value only if strictly greater, so the lowest index
// wins ties and values never above -FLT_MAX (or NaN) leave index 0.
//
// One workgroup of T threads per row (the entry point has no scratch to combine
// several), so a row is bound by what one workgroup keeps in flight: kRowChunks
// 16-byte loads a thread. A chunk of 8 values costs a max tree and one compare;
// the place inside the chunk is looked up once, for the thread's best chunk.
constexpr int kRowChunks = 8;
constexpr int kShortRow = 128;

template <int T>
__global__ __launch_bounds__(T) void k_argmax_rows(int32_t* out, const uint16_t* x, int n) {
  const uint16_t* row = x + (size_t)blockIdx.x * n;
  float v = -FLT_MAX;
  int i = 0;
  auto take = [&](int k) {
    const float f = ldbf(row + k);
    if (f > v) { v = f; i = k; }
  };
  // values before the row's first 16-byte boundary, whole chunks, the rest;
  // a thread's indices only grow, so a strict compare keeps the lowest
  // up to two values a thread: no chunks, whose best needs a second look (2 rows of 65
  // 2.5 us with them, 2.3 so; 129 to 700 values, few rows: 2.5 to 2.75 with chunks, no
  // better value by value, also in four waves)
  const bool few = T == 64 && n <= kShortRow;
  if (few)
    for (int k = threadIdx.x; k < n; k += T) take(k);
  const int head = few ? 0 : min(n, (int)((16 - ((uintptr_t)row & 15)) & 15) / 2);
  const int chunks = few ? 0 : (n - head) / 8;
  if ((int)threadIdx.x < head) take(threadIdx.x);
  const u32x4* body = reinterpret_cast<const u32x4*>(row + head);
  int best = -1;   // the chunk that holds this thread's best value
  for (int k = threadIdx.x; k < chunks; k += kRowChunks * T) {
    const int left = chunks - (k - (int)threadIdx.x);   // chunks of the row from this round on
    u32x4 d[kRowChunks];
#pragma unroll
    for (int j = 0; j < kRowChunks; ++j) {
      const int kj = k + j * T;
      if (T == 1024 || j * T < left) d[j] = body[kj < chunks ? kj : k];   // past the end: chunk k again, never greater
    }
#pragma unroll
    for (int j = 0; j < kRowChunks; ++j) {
      if (T < 1024 && j * T >= left) break;   // uniform: a short row has fewer rounds of loads
      float m = -FLT_MAX;   // fmaxf passes over NaN
#pragma unroll
      for (int e = 0; e < 4; ++e)
        m = fmaxf(m, fmaxf(__uint_as_float(d[j][e] << 16), __uint_as_float(d[j][e] & 0xffff0000u)));
      if (m > v) { v = m; best = k + j * T; }
    }
  }
  if (best >= 0) {
    const int k = head + 8 * best;
#pragma unroll
    for (int e = 7; e >= 0; --e)
      if (ldbf(row + k + e) == v) i = k + e;
  }
  const int tail = head + 8 * chunks + (int)threadIdx.x;
  if (!few && tail < n) take(tail);
  block_best<T / 64>(v, i);
  if (threadIdx.x == 0) out[blockIdx.x] = i;
}

__global__ __launch_bounds__(256) void k_argmax_partial(int32_t* idx, float* val,
                                                        const uint16_t* x, int n) {
  float v = -FLT_MAX;
  int i = 0;
  for (int k = blockIdx.x * 256 + threadIdx.x; k < n; k += gridDim.x * 256) {
    const float f = ldbf(x + k);
    if (f > v) { v = f; i = k; }
  }
  block_best<4>(v, i);
  if (threadIdx.x == 0) { idx[blockIdx.x] = i; val[blockIdx.x] = v; }
}

__global__ __launch_bounds__(256) void k_argmax_final(int32_t* out, const int32_t* idx,
                                                      const float* val, int chunks) {
  float v = -FLT_MAX;
  int i = 0;
  for (int k = threadIdx.x; k < chunks; k += 256) better(v, i, val[k], idx[k]);
  block_best<4>(v, i);
  if (threadIdx.x == 0) out[0] = i;
}

}  // namespace
}  // namespace qw4

using namespace qw4;

extern "C" {

int qw4_argmax(int32_t* out, const uint16_t* x, int n, int32_t* scratch, void* stream) {
  if (!out || !x || !scratch) return QW4_ERR_NULL;
  if (n <= 0) return QW4_ERR_SHAPE;
  const int chunks = 256;
  int32_t* idx = scratch;
  float* val = reinterpret_cast<float*>(scratch + chunks);
  hipStream_t hs = (hipStream_t)stream;
  k_argmax_partial<<<chunks, 256, 0, hs>>>(idx, val, x, n);
  k_argmax_final<<<1, 256, 0, hs>>>(out, idx, val, chunks);
  QW4_LAUNCH_CHECK();
  return QW4_OK;
}

int qw4_argmax_rows(int32_t* out, const uint16_t* x, int rows, int n, void* stream) {
  if (!out || !x) return QW4_ERR_NULL;
  if (rows < 0 || n <= 0) return QW4_ERR_SHAPE;
  if (rows == 0) return QW4_OK;
  // Few long rows: 16 waves a row, for what one CU can keep in flight (5 rows of
  // 248320: 116 us with 256 threads and 2-byte loads, 25 with 256 threads and
  // 16-byte loads, 14 so; at 24000 values 256 and 1024 threads meet). Short rows:
  // the waves of a workgroup are the cost (16384 rows of 64: 1024 threads 80 us, 256
  // 17, 64 8; of 1000: 83, 20, 10; from 4096 values on 256 beat 64). More rows than
  // two a CU need no 16 waves each to fill it (1000 rows of 64000: 31 us, 256
  // threads 25).
  hipStream_t hs = (hipStream_t)stream;
  if (n > 24576 && rows <= 512)
    k_argmax_rows<1024><<<rows, 1024, 0, hs>>>(out, x, n);
  else if (n > 2048)
    k_argmax_rows<256><<<rows, 256, 0, hs>>>(out, x, n);
  else
    k_argmax_rows<64><<<rows, 64, 0, hs>>>(out, x, n);
  QW4_LAUNCH_CHECK();
  return QW4_OK;
}

}  // extern "C"
