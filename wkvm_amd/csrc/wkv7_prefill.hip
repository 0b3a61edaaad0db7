// Varlen WKV7 prefill over slot states: the whole-head kernel (one workgroup
// per (sequence, head)) and the C entry points. The algorithm, schedule and
// layouts are described in wkv7_prefill_core.h.
#include <atomic>

#include "wkv7_prefill_core.h"

namespace wkv7 {
namespace {

struct WholeHead {
  static constexpr int kStateWaves = 4;
  static constexpr bool kEarlyB = true;
  // One state wave per SIMD; beside it on SIMD 0 and 1 the two parities'
  // operand waves of a channel half, on SIMD 2 score 0 and the inverse, on
  // SIMD 3 score 1 and io (one operand wave per SIMD instead: 4 % slower).
  static constexpr uint64_t kRoles = 0x4311'2211'0000ull, kParts = 0x0032'1010'3210ull;
};

}  // namespace
}  // namespace wkv7

using namespace wkv7;

namespace {
// Compute units of the current device (cached per device; 256 on MI355X; 0
// when the runtime cannot say, which keeps one workgroup per (sequence, head)).
int device_cus() {
  static std::atomic<int> cus[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  int n = cus[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      return 0;
    cus[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// p: every field but layers.
int prefill_launch(PrefillPlan& p, int32_t layers, const wkv7_layer_io* io, int32_t y_dtype,
                   void* stream) {
  const int64_t items = int64_t(p.nseq) * p.H * layers, cus = device_cus();
  // A launch that leaves half or more of the compute units idle splits each
  // (sequence, head) over two or four workgroups by value columns (same
  // arithmetic per column, so the same bits). A tick is the shorter the fewer
  // state waves share the unit, and the preparation is repeated by each
  // workgroup, which costs nothing while a unit stays free for it: 4 x 1500
  // tokens x 32 heads 77.7 us whole, 73.5 in halves, 134.8 in quarters (which
  // no longer run side by side). It costs power, though: where a launch is long
  // enough to run into the limit, quarters on more than three quarters of the
  // units are slower than halves on half as many. us for 2000 tokens, halves /
  // quarters: 48 heads 82 / 78, 56 82 / 85, 64 83 / 87; 64 heads x 512 tokens 25.5 /
  // 24.9, x 900 40.1 / 42.2.
  const bool hot = p.total_tokens > 768 * int64_t(p.nseq);
  const int split = 4 * items <= (hot ? cus * 3 / 4 : cus) ? 4 : 2 * items <= cus ? 2 : 1;
  const int64_t blocks = items * split;
  if (blocks > int64_t(0x7fffffff)) return WKV7_ERR_ARG;
  p.layers = layers;
  hipStream_t s = as_stream(stream);
  const bool f32 = y_dtype == WKV7_Y_F32, scaled = p.scale != 1.0f;
  if (split > 1) return prefill_split_launch(split, unsigned(blocks), s, f32, scaled, p, io);
  return launch_form<WholeHead>(unsigned(blocks), s, f32, scaled, p, io);
}

// y rows are stored as 8-byte (bf16) or 16-byte (fp32) vectors
bool y_aligned(const void* y, int32_t y_dtype) {
  return (reinterpret_cast<uintptr_t>(y) & (y_dtype == WKV7_Y_F32 ? 15u : 7u)) == 0;
}

bool inputs_aligned(const uint16_t* r, const uint16_t* w, const uint16_t* k, const uint16_t* v,
                    const uint16_t* a, const uint16_t* b) {
  // inputs are read as 16-byte vectors
  const uintptr_t align = reinterpret_cast<uintptr_t>(r) | reinterpret_cast<uintptr_t>(w) |
                          reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
                          reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b);
  return (align & 15u) == 0;
}
}  // namespace

extern "C" int wkv7_prefill_varlen(float* wkv_layer, int64_t num_rows, int32_t H,
                                   const int32_t* slot_ids, const int32_t* cu_seqlens,
                                   const int32_t* seq_order, int32_t nseq, int64_t total_tokens,
                                   const uint16_t* r,
                                   const uint16_t* w, const uint16_t* k, const uint16_t* v,
                                   const uint16_t* a, const uint16_t* b, void* y, int32_t y_dtype,
                                   int32_t zero_init, float scale, void* stream) {
  if (nseq < 0 || H < 1 || num_rows < 1 || total_tokens < 0) return WKV7_ERR_ARG;
  if (y_dtype != WKV7_Y_BF16 && y_dtype != WKV7_Y_F32) return WKV7_ERR_ARG;
  if (nseq == 0) return WKV7_OK;
  if (!wkv_layer || !slot_ids || !cu_seqlens) return WKV7_ERR_ARG;
  if (total_tokens > 0 && (!r || !w || !k || !v || !a || !b || !y)) return WKV7_ERR_ARG;
  if (!inputs_aligned(r, w, k, v, a, b) || !y_aligned(y, y_dtype)) return WKV7_ERR_SHAPE;
  const Runs runs{nullptr, nullptr, nseq, nullptr, 0, nullptr, nullptr, nullptr, 0};
  PrefillPlan p{wkv_layer, num_rows,     H,         slot_ids, cu_seqlens, seq_order,
                nseq,      total_tokens, zero_init, scale,    runs};
  const wkv7_layer_io io{r, w, k, v, a, b, y};
  return prefill_launch(p, 1, &io, y_dtype, stream);
}

extern "C" int wkv7_prefill_layers(float* wkv, int64_t layer_stride, int32_t layers,
                                   int64_t num_rows, int32_t H, const int32_t* slot_ids,
                                   const int32_t* cu_seqlens, const int32_t* seq_order,
                                   int32_t nseq, int64_t total_tokens, const wkv7_layer_io* io,
                                   int32_t y_dtype, int32_t zero_init, float scale,
                                   void* stream) {
  if (layers < 0 || nseq < 0 || H < 1 || num_rows < 1 || total_tokens < 0) return WKV7_ERR_ARG;
  if (y_dtype != WKV7_Y_BF16 && y_dtype != WKV7_Y_F32) return WKV7_ERR_ARG;
  if (layers == 0 || nseq == 0) return WKV7_OK;
  if (!wkv || !slot_ids || !cu_seqlens || !io) return WKV7_ERR_ARG;
  if (layers > 1 && layer_stride < num_rows * int64_t(H) * kHead * kHead) return WKV7_ERR_SHAPE;
  for (int32_t l = 0; l < layers; ++l) {
    const wkv7_layer_io& x = io[l];
    if (total_tokens > 0 && (!x.r || !x.w || !x.k || !x.v || !x.a || !x.b || !x.y))
      return WKV7_ERR_ARG;
    if (!inputs_aligned(x.r, x.w, x.k, x.v, x.a, x.b) || !y_aligned(x.y, y_dtype))
      return WKV7_ERR_SHAPE;
  }
  const Runs runs{nullptr, nullptr, nseq, nullptr, 0, nullptr, nullptr, nullptr, 0};
  // as many layers per launch as its argument table holds and its work items
  // fit into 32 bits
  const int64_t fit = int64_t(UINT32_MAX) / (int64_t(nseq) * H * kWaves * kWave);
  const int32_t step = fit < 1 ? 1 : fit < kMaxLayers ? int32_t(fit) : kMaxLayers;
  for (int32_t l = 0; l < layers; l += step) {
    const int32_t n = layers - l < step ? layers - l : step;
    PrefillPlan p{wkv + l * layer_stride, num_rows,     H,         slot_ids, cu_seqlens, seq_order,
                  nseq,                   total_tokens, zero_init, scale,    runs};
    p.layer_stride = layer_stride;
    const int rc = prefill_launch(p, n, io + l, y_dtype, stream);
    if (rc != WKV7_OK) return rc;
  }
  return WKV7_OK;
}

extern "C" int wkv7_prefill_runs(float* wkv_layer, int64_t num_rows, int32_t H,
                                 const int32_t* slot_ids, const int32_t* cu_seqlens,
                                 const int32_t* seq_order, int32_t nseq, int64_t total_tokens,
                                 const uint16_t* r, const uint16_t* w, const uint16_t* k,
                                 const uint16_t* v, const uint16_t* a, const uint16_t* b, void* y,
                                 int32_t y_dtype, int32_t zero_init, float scale,
                                 const int32_t* run_flags, const int32_t* cu_alt,
                                 int32_t n_primary, float* state_alt, int64_t alt_rows,
                                 void* y_alt, const float* state_in, int64_t in_rows,
                                 const int32_t* in_ids, void* stream) {
  if (nseq < 0 || H < 1 || num_rows < 1 || total_tokens < 0 || alt_rows < 0) return WKV7_ERR_ARG;
  if (in_rows < 0 || (state_in && in_rows < 1) || (in_ids && !state_in)) return WKV7_ERR_ARG;
  if (state_in && !in_ids && in_rows < nseq) return WKV7_ERR_SHAPE;
  if (n_primary < 0 || n_primary > nseq) return WKV7_ERR_ARG;
  if (y_dtype != WKV7_Y_BF16 && y_dtype != WKV7_Y_F32) return WKV7_ERR_ARG;
  if (nseq == 0) return WKV7_OK;
  if (!wkv_layer || !slot_ids || (n_primary > 0 && !cu_seqlens)) return WKV7_ERR_ARG;
  if (n_primary < nseq && !cu_alt) return WKV7_ERR_ARG;
  if (alt_rows > 0 && !state_alt) return WKV7_ERR_ARG;
  if (total_tokens > 0 && (!r || !w || !k || !v || !a || !b || !y)) return WKV7_ERR_ARG;
  if (!inputs_aligned(r, w, k, v, a, b) || !y_aligned(y, y_dtype) ||
      (y_alt && !y_aligned(y_alt, y_dtype)))
    return WKV7_ERR_SHAPE;
  const Runs runs{run_flags, cu_alt,   n_primary, state_alt, alt_rows,
                  y_alt ? y_alt : y, state_in, in_ids,    in_rows};
  PrefillPlan p{wkv_layer, num_rows,     H,         slot_ids, cu_seqlens, seq_order,
                nseq,      total_tokens, zero_init, scale,    runs};
  const wkv7_layer_io io{r, w, k, v, a, b, y};
  return prefill_launch(p, 1, &io, y_dtype, stream);
}

extern "C" int wkv7_prefill_into(const float* state_in, int64_t in_rows, const int32_t* in_ids,
                                 float* state_out, int64_t out_rows, const int32_t* out_ids,
                                 int32_t H, const int32_t* cu_seqlens, const int32_t* seq_order,
                                 int32_t nseq, int64_t total_tokens, const uint16_t* r,
                                 const uint16_t* w, const uint16_t* k, const uint16_t* v,
                                 const uint16_t* a, const uint16_t* b, void* y, int32_t y_dtype,
                                 float scale, void* stream) {
  if (nseq < 0 || H < 1 || total_tokens < 0 || in_rows < 0 || out_rows < 0) return WKV7_ERR_ARG;
  if (y_dtype != WKV7_Y_BF16 && y_dtype != WKV7_Y_F32) return WKV7_ERR_ARG;
  if ((in_ids && !state_in) || (out_ids && !state_out)) return WKV7_ERR_ARG;
  if (nseq == 0) return WKV7_OK;
  if (!cu_seqlens) return WKV7_ERR_ARG;
  if (total_tokens > 0 && (!r || !w || !k || !v || !a || !b || !y)) return WKV7_ERR_ARG;
  if ((state_in && !in_ids && in_rows < nseq) || (state_out && !out_ids && out_rows < nseq))
    return WKV7_ERR_SHAPE;
  if (!inputs_aligned(r, w, k, v, a, b) || !y_aligned(y, y_dtype)) return WKV7_ERR_SHAPE;
  // no state_in: zero initial state; no state_out: no final state written
  const Runs runs{nullptr, nullptr, nseq, nullptr, 0, nullptr, state_in, in_ids, in_rows};
  PrefillPlan p{state_out, state_out ? out_rows : 0, H,                out_ids, cu_seqlens, seq_order,
                nseq,      total_tokens,             state_in ? 0 : 1, scale,   runs};
  const wkv7_layer_io io{r, w, k, v, a, b, y};
  return prefill_launch(p, 1, &io, y_dtype, stream);
}
