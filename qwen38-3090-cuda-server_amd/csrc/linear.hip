// The reference's linear() path choice (src/model/model.cu:522-565,
// :643-658) over this library's kernels: the GEMV for one row, the skinny
// kernel in chunks of 16 or 32 rows while it reads the weights fewer times
// than the prefill GEMM would cost, the prefill GEMM beyond. Host code only.
#include <atomic>

#include "../../include/qwen_w4a16.h"
#include "skinny.h"

namespace {

std::atomic<int> g_lin_max_t{0};   // qw4_tune_linear override (0: the rule below)

// Rows up to which skinny passes run instead of the prefill GEMM: they use the
// weights exactly where the GEMM rounds them to bf16, so this line is not moved
// with every change of either's speed. 16 whole passes under the ratio that
// 16-row passes (0.245 us per MB of weights + 5.8 us) and the GEMM (60 us + 0.4
// us per MB) had on MI355X when it was set: 48 rows for gate|up (93 MB), 64 for
// down (46 MB), 96 for qkv (19 MB), 112 for o_proj (11 MB).
int lin_max_t(const qw4_weights* w) {
  const int v = g_lin_max_t.load(std::memory_order_relaxed);
  if (v > 0) return v;
  const double mb = (double)w->out_f * w->in_f * (0.5 + 2.5 / 128) / 1e6;
  const int chunks = (int)((60.0 + 0.4 * mb) / (0.245 * mb + 5.8));
  return 16 * (chunks < 1 ? 1 : chunks);
}

}  // namespace

extern "C" {

int qw4_tune_linear(int max_t) {
  if (max_t < 0) return QW4_ERR_SHAPE;
  g_lin_max_t.store(max_t, std::memory_order_relaxed);
  return 0;
}

int qw4_linear_max_t(const qw4_weights* w) {
  if (!w || w->out_f <= 0 || w->in_f <= 0) return QW4_ERR_NULL;
  return lin_max_t(w);
}

int qw4_linear(uint16_t* y, const qw4_weights* w, const uint16_t* x, int T, qw4_scratch* s,
               qw4_workspace* ws, void* stream) {
  if (!y || !w || !x) return QW4_ERR_NULL;
  if (T < 1) return QW4_ERR_M;
  if (T == 1) return qw4_gemv(y, w, x, s, stream);
  if (T <= lin_max_t(w) && s) {
    const int chunk = s->max_m < 16 ? s->max_m : 16;
    if (chunk < 1) return QW4_ERR_SCRATCH;
    for (int i = 0, n; i < T; i += n) {
      // two 16-row passes in one where it pays; a last single row stays a pass
      // of its own (the GEMV's sums)
      const int left = T - i;
      n = left < 32 ? left : 32;
      if (n % 16 == 1) --n;
      if (chunk == 16 && n > 16) {
        bool taken = false;
        const int st = qw4::skinny_rows32(y + (size_t)i * w->out_f, w, x + (size_t)i * w->in_f, n, s,
                                          stream, &taken);
        if (st) return st;
        if (taken) continue;
      }
      n = left < chunk ? left : chunk;
      const int st = qw4_gemm_small(y + (size_t)i * w->out_f, w, x + (size_t)i * w->in_f, n, s,
                                    stream);
      if (st) return st;
    }
    return QW4_OK;
  }
  return qw4_gemm(y, w, x, T, ws, stream);
}

}  // extern "C"
