// Combination step of the segmented prefill (wkv7_prefill_runs + these two).
//
// The WKV7 scan is linear in its initial state. A sequence cut into segments
// runs segment 0 from its slot state and every later segment g twice, side by
// side: from zero state with the real inputs (y0_g, final state H0_g) and from
// the identity with k = v = 0, which gives the segment's transition Phi_g as
// the final state and q_g = (scale r)^T Phi_t as y. With H_in the state
// entering segment g:
//   H_out = H0_g + Phi_g H_in          (wkv7_segment_chain, in segment order)
//   y_g   = y0_g + q_g H_in            (wkv7_segment_correct, all tokens at once)
// Both in fp32; state matrices use the pool layout [j][i] (key j, value i),
// on which Phi acts from the left.
#include "wkv7_mfma.h"

namespace wkv7 {
namespace {

constexpr int kCombThreads = 256;
constexpr int kMat = kHead * kHead;  // floats per 64 x 64 head matrix

// A quarter (16 value columns) of one (sequence, head) per workgroup; thread t
// owns row j = t / 4 and the columns 16 q + 4 (t % 4) .. + 3 of the products.
// The columns are independent, and one workgroup per head left most units
// idle: three segments of 32 heads 20 us whole, 8 us in quarters.
constexpr int kChainSplit = 4;
__global__ __launch_bounds__(kCombThreads) void segment_chain_kernel(
    float* __restrict__ wkv, int64_t num_rows, int H, const float* __restrict__ alt,
    int64_t alt_rows, const int32_t* __restrict__ seq_tab, int nseq,
    const int32_t* __restrict__ seg_tab, int nsegs, float* __restrict__ hin) {
  __shared__ float4 cur[kHead][4];  // H_in, these columns
  const int64_t item = blockIdx.x / kChainSplit;
  const int64_t s = item / H;
  const int64_t head = item - s * H;
  if (s >= nseq) return;
  const int64_t slot = seq_tab[3 * s];
  const int first = seq_tab[3 * s + 1], count = seq_tab[3 * s + 2];
  if (slot < 0 || slot >= num_rows || first < 0 || count < 0 || first + count > nsegs) return;
  const int j = threadIdx.x >> 2, c = threadIdx.x & 3;
  const int at = j * 16 + 4 * int(blockIdx.x % kChainSplit) + c;  // this thread's float4
  float4* state = reinterpret_cast<float4*>(wkv + (slot * H + head) * kMat) + at;
  float4 h = *state;
  for (int n = 0; n < count; ++n) {
    const int seg = first + n;
    const int64_t row_main = seg_tab[2 * seg], row_phi = seg_tab[2 * seg + 1];
    reinterpret_cast<float4*>(hin + (int64_t(seg) * H + head) * kMat)[at] = h;
    const bool ok = row_main >= 0 && row_main < alt_rows && row_phi >= 0 && row_phi < alt_rows;
    if (!ok) continue;  // uniform
    cur[j][c] = h;
    __syncthreads();
    const float4* phi = reinterpret_cast<const float4*>(alt + (row_phi * H + head) * kMat);
    h = reinterpret_cast<const float4*>(alt + (row_main * H + head) * kMat)[at];
    for (int m4 = 0; m4 < 16; ++m4) {
      const float4 p = phi[j * 16 + m4];
      const float pv[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float4 hv = cur[4 * m4 + e][c];
        h.x = fmaf(pv[e], hv.x, h.x);
        h.y = fmaf(pv[e], hv.y, h.y);
        h.z = fmaf(pv[e], hv.z, h.z);
        h.w = fmaf(pv[e], hv.w, h.w);
      }
    }
    __syncthreads();  // every thread has read cur
  }
  *state = h;
}

// One block of at most 64 tokens of one head per workgroup, 16 tokens per
// wave: y^T = y0^T + H_in^T q^T on the matrix cores, in fp32 throughout (fp32
// operands and accumulators, y0 as the first term), so that a value column's y
// depends on that column of H_in alone and rounds as fp32 multiply-adds do.
// v_mfma_f32_16x16x4_f32, lane l, li = l % 16, lg = l / 16: A lane holds A[li][lg],
// B lane holds B[lg][li], the accumulator D[4lg .. 4lg+3][li]. k label lg of a
// step is key 32 kb + 8 lg + e, so that q goes from memory straight to the B
// operand and H_in comes from LDS in rows of kHinPitch floats: the four rows
// of a read lie 8 apart, 16 banks from each other. The 564 bytes per token-head
// bound it: 16384 tokens x 32 heads 67 us (4.4 TB/s); as
// scalar multiply-adds out of LDS 88 us, as three bf16 products of hi + lo
// parts 65 us, at 2^-16 and with a column's non-finite value in its neighbour.
constexpr int kHinPitch = kHead + 2;
template <bool kF32Out>
__global__ __launch_bounds__(kCombThreads) void segment_correct_kernel(
    int64_t total_tokens, int H, const float* __restrict__ y0, const float* __restrict__ q,
    const int32_t* __restrict__ blk_tab, int nblk, const float* __restrict__ hin, int nsegs,
    void* __restrict__ y) {
  __shared__ __align__(16) float hs[kHead * kHinPitch];  // H_in: [key][value column]
  const int64_t blk = blockIdx.x / H;
  const int64_t head = blockIdx.x - blk * H;
  if (blk >= nblk) return;
  const int64_t tok0 = blk_tab[3 * blk];
  const int cnt = blk_tab[3 * blk + 1], seg = blk_tab[3 * blk + 2];
  const bool corr = seg >= 0 && seg < nsegs;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int ti = 16 * int(threadIdx.x >> 6) + li;
  const int64_t tok = tok0 + ti;
  const bool mine = ti < cnt && tok >= 0 && tok < total_tokens;
  const int64_t base = (tok * H + head) * kHead;
  // lane: token li, value columns 16 ct + 4 lg .. + 3 of every tile ct
  f32x4 acc[4] = {}, qv[2][2] = {};
  if (mine) {
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
      acc[ct] = __builtin_nontemporal_load(
          reinterpret_cast<const f32x4*>(y0 + base + 16 * ct + 4 * lg));
    if (corr) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          qv[kb][i] = __builtin_nontemporal_load(
              reinterpret_cast<const f32x4*>(q + base + 32 * kb + 8 * lg + 4 * i));
    }
  }
  if (corr) {  // uniform
    const f32x4* src = reinterpret_cast<const f32x4*>(hin + (int64_t(seg) * H + head) * kMat);
#pragma unroll
    for (int i = 0; i < kMat / 4 / kCombThreads; ++i) {
      const int at = kCombThreads * i + threadIdx.x;
      const f32x4 h = src[at];
      float* row = &hs[(at >> 4) * kHinPitch + 4 * (at & 15)];  // 8-byte aligned
      *reinterpret_cast<float2*>(row) = make_float2(h[0], h[1]);
      *reinterpret_cast<float2*>(row + 2) = make_float2(h[2], h[3]);
    }
    __syncthreads();
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
          acc[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(
              hs[(32 * kb + 8 * lg + e) * kHinPitch + 16 * ct + li], qv[kb][e >> 2][e & 3],
              acc[ct], 0, 0, 0);
    // past the last product's 8 passes before a vector instruction reads it (the
    // accumulators as "a": with "v" they would be read back ahead of the wait)
    asm volatile("s_nop 15" : "+a"(acc[0]), "+a"(acc[1]), "+a"(acc[2]), "+a"(acc[3]));
  }
  if (!mine) return;
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    const int64_t o = base + 16 * ct + 4 * lg;
    if constexpr (kF32Out)
      *reinterpret_cast<f32x4*>(static_cast<float*>(y) + o) = acc[ct];
    else
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(y) + o) =
          make_uint2(pack_bf16(acc[ct][0], acc[ct][1]), pack_bf16(acc[ct][2], acc[ct][3]));
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace wkv7

using namespace wkv7;

extern "C" int wkv7_segment_chain(float* wkv_layer, int64_t num_rows, int32_t H,
                                  const float* state_alt, int64_t alt_rows,
                                  const int32_t* seq_tab, int32_t nseq, const int32_t* seg_tab,
                                  int32_t nsegs, float* hin, void* stream) {
  if (num_rows < 1 || H < 1 || alt_rows < 0 || nseq < 0 || nsegs < 0) return WKV7_ERR_ARG;
  if (nseq == 0) return WKV7_OK;
  if (!wkv_layer || !seq_tab || (nsegs > 0 && (!seg_tab || !state_alt || !hin)))
    return WKV7_ERR_ARG;
  if (!aligned16(wkv_layer) || (nsegs > 0 && (!aligned16(state_alt) || !aligned16(hin))))
    return WKV7_ERR_SHAPE;
  const int64_t blocks = int64_t(nseq) * H * kChainSplit;
  if (blocks > int64_t(0x7fffffff)) return WKV7_ERR_ARG;
  segment_chain_kernel<<<unsigned(blocks), kCombThreads, 0, as_stream(stream)>>>(
      wkv_layer, num_rows, H, state_alt, alt_rows, seq_tab, nseq, seg_tab, nsegs, hin);
  return launch_status();
}

extern "C" int wkv7_segment_correct(int64_t total_tokens, int32_t H, const float* y0,
                                    const float* q, const int32_t* blk_tab, int32_t nblk,
                                    const float* hin, int32_t nsegs, void* y, int32_t y_dtype,
                                    void* stream) {
  if (total_tokens < 0 || H < 1 || nblk < 0 || nsegs < 0) return WKV7_ERR_ARG;
  if (y_dtype != WKV7_Y_BF16 && y_dtype != WKV7_Y_F32) return WKV7_ERR_ARG;
  if (nblk == 0 || total_tokens == 0) return WKV7_OK;
  if (!y0 || !blk_tab || !y || (nsegs > 0 && (!q || !hin))) return WKV7_ERR_ARG;
  if (!aligned16(y0) || (nsegs > 0 && (!aligned16(q) || !aligned16(hin))) ||
      (y_dtype == WKV7_Y_F32 ? !aligned16(y) : (reinterpret_cast<uintptr_t>(y) & 7u)))
    return WKV7_ERR_SHAPE;
  const int64_t blocks = int64_t(nblk) * H;
  if (blocks > int64_t(0x7fffffff)) return WKV7_ERR_ARG;
  hipStream_t s = as_stream(stream);
  if (y_dtype == WKV7_Y_F32)
    segment_correct_kernel<true><<<unsigned(blocks), kCombThreads, 0, s>>>(
        total_tokens, H, y0, q, blk_tab, nblk, hin, nsegs, y);
  else
    segment_correct_kernel<false><<<unsigned(blocks), kCombThreads, 0, s>>>(
        total_tokens, H, y0, q, blk_tab, nblk, hin, nsegs, y);
  return launch_status();
}
