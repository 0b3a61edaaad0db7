// Device code of the WKV7 chunked prefill, included by one translation unit
// per group of workgroup forms (wkv7_prefill.hip: whole heads and the entry
// points; wkv7_prefill_split.hip: heads split over workgroups), so that no
// form changes the other's code.
//
// One workgroup of 12 wavefronts walks one (sequence, head), or the 16 or 32
// value columns of one that it owns. Its state columns stay in MFMA
// accumulator registers for the whole sequence (16 columns per state wave) and
// touch HBM only to load the initial state and store the final one.
//
// The sequence is solved in 16-token sub-chunks. With G_t the inclusive
// cumulative log-decay inside a sub-chunk (G_{-1} = 0):
//   A^_t = a_t e^{G_{t-1}}   R^_t = scale r_t e^{G_t}   B~_s = b_s e^{-G_s}   K~_s = k_s e^{-G_s}
//   L_ab = tril(A^ B~^T, -1)  L_ak = tril(A^ K~^T, -1)  M_rb = tril(R^ B~^T)  M_rk = tril(R^ K~^T)
//   P  = (I - L_ab)^{-1} (A^ h + L_ak V)            (row t: p_t = a_t^T h_{t-1})
//   Y  = R^ h + M_rb P + M_rk V
//   h' = diag(e^{G_15}) (h + B~^T P + K~^T V)
// Sub-chunk referencing keeps every decay factor within e^{+-16 |w|}, far from
// fp32/bf16 range limits for RWKV-7's decays (|w| < 0.61 per token). Padding
// tokens past the end of a sequence enter as w = 0 (decay 1) and zero
// vectors, i.e. identity steps.
//
// Schedule: a software pipeline over sub-chunks, one workgroup barrier per
// tick. In tick k
//   state     (4, 2 or 1 waves) runs sub-chunk k's state step (the products
//             above) on operands read in the tick before
//   inverse   (1) sub-chunk k+1: T = (I - L_ab)^{-1}
//   scores    (2) sub-chunk k+2: L_ab and M_rb in one wave, L_ak and M_rk in
//             the other (each pair shares its B~ / K~ reads); the second also
//             stores sub-chunk k-1's y as whole rows
//   operands  (4) decays and operand matrices, 32 key channels per wave, the
//             even and the odd sub-chunks in waves of their own: k+4 in its
//             first, k+3 in its second tick
//   io        (1) asks for sub-chunk k+7's input rows, whole 128-byte rows
//             straight into LDS, two sub-chunks in flight beyond the next
// Sub-chunk j's operands live in ring slot j % 4 from tick j-3 to tick j.
//
// What bounds it: with every compute unit busy the power limit (8 x 4096
// tokens x 32 heads: 203 us and 2.41 GHz for a launch by itself, 231 us at
// about 2.1 GHz in a row of them), then the products' and the vector units'
// work, no longer LDS or issue slots alone: 95 M instructions, 57 M LDS cycles
// and 10.5 M bank-conflict cycles per such launch, where one wave per role and
// SIMD (16 waves, every wave's operands read at the start of its tick, each
// split by an unpack and a subtraction) took 124 M, 77 M and 21 M, 219 us by
// itself and 254 us in a row. With few heads the state wave's dependent chain
// (about 0.43 us per tick by itself) and the operand waves beside it.
// A sequence of one sub-chunk is nearly all fill, one tick longer here than in
// that kernel, so no role works past the sub-chunk after the end and a
// workgroup finds its work in 32-bit arithmetic: 64 x 8 tokens x 32 heads
// 37.8 us (44.7 with the pipeline running on over zero rows and 64-bit
// divisions; 39.8 there), 32 x 40 tokens 28.2 (31.5, 32.0).
//
// Precision: MFMA operands that are not exact bf16 inputs are split into bf16
// hi + lo parts, a product formed as hi*hi + hi*lo + lo*hi with fp32
// accumulation (~2^-16 relative per product), except two that enter as one
// bf16 each: A^ and T (solved in fp32, then rounded). Those cost ~2^-9
// relative on P only. h enters the A^ h product split as well: as one bf16
// it left a 4096-token run with no decay on half the key channels at 8e-4
// relative L2 on y and state (1.5e-4 split). Products with the exact bf16 v
// need one MFMA per term pair. Operand layouts below
// (v_mfma_f32_16x16x32_bf16, lane l, li = l%16, lg = l/16): A lane holds
// A[li][8lg..8lg+7] of a 32-wide k block, B lane holds B[8lg..8lg+7][li], the
// accumulator holds D[4lg..4lg+3][li]; the same registers are A or, for the
// transposed product, B. Contractions over 16 tokens put k = 4lg..4lg+3 in
// elements 0..3 of both operands and a second term of the sum in 4..7; with
// that labelling a 16x16 accumulator is already the B operand of the next
// 16-token product, straight from registers, and an LDS transpose read of
// token rows 4lg..4lg+3 is the A operand B~^T / K~^T or the B operand v.
// Contractions over the 64 key rows take the k labels of a 32-row block in
// the order the state tiles hold them (key_row below), so the state is a B
// operand straight from registers as well.
#pragma once

#include <type_traits>

#include "wkv7_mfma.h"

namespace wkv7 {
namespace {

constexpr int kSub = 16;   // tokens per sub-chunk
constexpr int kRing = 4;   // operand ring slots
constexpr int kIn = 4;     // input row slots (tick j - 7, where they are asked for, to tick j - 4)
constexpr int kVRing = 8;  // v rows live from tick j - 7 to tick j - 1

// Key row held by row m of state tile jb. A lane of the B operand of key block
// kb holds the rows 4lg .. 4lg+3 of the tiles 2kb and 2kb+1; as its k labels
// 8lg .. 8lg+7 are the channels 32kb + 8lg .. + 7 in order, those rows are
// 32kb + 8lg + {0..3} and 32kb + 8lg + {4..7}.
__device__ __forceinline__ int key_row(int jb, int m) {
  return 32 * (jb >> 1) + 8 * (m >> 2) + 4 * (jb & 1) + (m & 3);
}

// One sub-chunk's operands, every array row-major [token][channel].
struct __align__(16) Slot {
  uint16_t A[kSub * kPR];       // A^ as one bf16 [t][channel]
  uint16_t R[2][kSub * kPR];    // R^ hi/lo [t][channel]
  uint16_t B[2][kSub * kPR];    // B~ hi/lo [s][channel]
  uint16_t K[2][kSub * kPR];    // K~ hi/lo [s][channel]
  uint4 M[4][kWave];            // T, L_ak, M_rb, M_rk as {hi, lo} in A-operand lane order
  float gam[kHead];             // e^{G_15}, the sub-chunk's decay
};

// y of a sub-chunk staged for the row stores: [token][64 values] rows padded by
// 16 bytes (both pitches keep 16-byte reads aligned and spread the state
// waves' row writes over the banks).
constexpr int kYRowB = kHead * 2 + 16;  // bf16 row pitch in bytes
constexpr int kYRowF = kHead * 4 + 16;  // fp32 row pitch in bytes

struct __align__(16) Shared {
  Slot slot[kRing];
  float4 Lf[2][kWave];                 // L_ab in fp32, A-operand lane order
  unsigned char ys[2][kSub * kYRowF];  // y of sub-chunks k (state waves) and k-1 (its stores)
  uint4 inb[kIn][5][kSub][8];          // input rows r, w, k, a, b, 128 B each
  uint4 v[kVRing][kSub][8];            // v rows, the layout of rk_off
};

typedef __attribute__((address_space(3))) uint4 lds_uint4;
__device__ __forceinline__ uint32_t lds_addr(const uint4* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const lds_uint4*)p));
}
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// Value of the lane one to the left in the DPP row; the first lane gets `first`.
__device__ __forceinline__ float row_prev(float x, float first) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(__float_as_int(first), __float_as_int(x), 0x111, 0xf, 0xf, false));
}

// Ends a pipeline tick. The scheduling fence keeps the compiler from moving
// the next tick's arithmetic above the barrier.
__device__ __forceinline__ void end_tick() {
  __syncthreads();
  __builtin_amdgcn_sched_barrier(0);
}

}  // namespace

// (External linkage: prefill_split_launch takes them to the other translation
// unit.)
struct Inputs {
  const uint16_t *r, *w, *k, *v, *a, *b;
};

// Per-run options of wkv7_prefill_runs and wkv7_prefill_into (all absent for
// wkv7_prefill_varlen). Runs [0, n_primary) take their token range from
// cu_seqlens; run n_primary + i takes [ranges[2i], ranges[2i+1]). Flags select
// the initial state (slot row, zero or identity), zero k and v, and redirect y
// and the final state. With state_in set, a run that starts from a stored
// state reads it from state_in (row in_ids[run], or row `run` when in_ids is
// null) instead of its slot row.
struct Runs {
  const int32_t* flags;   // [nseq] or null
  const int32_t* cu_alt;  // [2 (nseq - n_primary)] begin/end pairs, or null
  int32_t n_primary;
  float* state_alt;       // [alt_rows, H, 64, 64]
  int64_t alt_rows;
  void* y_alt;            // like y
  const float* state_in;  // [in_rows, H, 64, 64] or null
  const int32_t* in_ids;  // [nseq] or null
  int64_t in_rows;
};

// `layers` layers share the plan: layer l's states are at wkv + l *
// layer_stride, its vectors io[l] (one launch instead of a layer's launch
// after the other's tail).
struct PrefillPlan {
  float* wkv;  // final states, and initial ones unless runs.state_in or zero_init; null: none
  int64_t num_rows;
  int H;
  const int32_t *slot_ids, *cu_seqlens, *seq_order;  // slot_ids null: run s is row s
  int nseq;
  int64_t total_tokens;
  int zero_init;
  float scale;
  Runs runs;
  int layers;
  int64_t layer_stride;
};

// A launch's arguments: one layer's vectors, or the table of kMaxLayers (1.75
// KiB, of which a launch of one layer would copy 56 bytes for its own).
template <int N>
struct PrefillArgs : PrefillPlan {
  wkv7_layer_io io[N];
};

// Launches the forms of wkv7_prefill_split.hip: `split` (2 or 4) workgroups
// per (sequence, head).
int prefill_split_launch(int split, unsigned blocks, hipStream_t s, bool f32_out, bool scaled,
                         const PrefillPlan& p, const wkv7_layer_io* io);

namespace {

struct SeqGeom {
  int64_t t_beg, t_end;  // token range of the sequence
  int64_t tstride;       // elements between consecutive tokens (H * 64)
  int64_t hoff;          // element offset of this head inside a token row
};

// ---- operands -------------------------------------------------------------------------

// One lane's view of a sub-chunk's inputs: channels c0 .. c0+7, c0 = 32 part +
// 8 (lane / 16), of token lane % 16 (r, k, a, b: one 16-byte chunk each), and
// w transposed: w[m] holds channel 32 part + 8 (t / 4) + 4m + t % 4, t = lane %
// 16, at tokens 4 (lane / 16) .. + 3.
struct SubIn {
  uint4 r, k, a, b;
  uint2 w[2];
};

__device__ __forceinline__ void read_inputs(const Shared& sm, SubIn& d, int slot, int lane,
                                            int part) {
  const int t = lane & 15, cg = lane >> 4;
  auto rows = [&](int input) {
    return reinterpret_cast<const uint16_t*>(&sm.inb[slot][input][0][0]);
  };
#pragma unroll
  for (int m = 0; m < 2; ++m)
    d.w[m] = ld_tr(rows(1) + rk_off(4 * cg + (t >> 2), 32 * part + 8 * (t & 3) + 4 * m));
  const int off = rk_off(t, 32 * part + 8 * cg);
  d.k = ld16(rows(2) + off);
  d.b = ld16(rows(4) + off);
  d.a = ld16(rows(3) + off);
  d.r = ld16(rows(0) + off);
}

// Operands of a sub-chunk for key channels [32 part, 32 part + 32), over two
// ticks: this chain (row reads, decay sums, exponentials, products, splits,
// stores) is the longest of a sub-chunk's preparation, longer than a tick, so
// the even and the odd sub-chunks have waves of their own. The first tick ends
// with K~ (and with kEarlyB B~) in registers, the second makes the rest and
// stores. kEarlyB is the better balance beside four state waves (0.89 against
// 0.92 us per tick), the other beside one or two (0.52 against 0.57).
// Padding tokens are zeros already (the row loads stop at the sequence end).
// kScaled: scale != 1 (fla's default is 1, where R^ = r e^G needs no multiply
// by it).
template <bool kScaled, bool kEarlyB>
struct Operands {
  uint4 r, a, b, kh, kl, bh, bl;
  float eh[8], ie[8];  // e^G and e^-G of this lane's token and channels

  // The compiler would move the first tick's work past the barrier, next to
  // its use.
  static __device__ __forceinline__ void keep(uint4& x) {
    asm volatile("" : "+v"(x.x), "+v"(x.y), "+v"(x.z), "+v"(x.w));
  }

  __device__ __forceinline__ void make_b(const Neg& n) {
    float x[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) x[m] = elem(b, m) * ie[m];
    split8(x, bh, bl, n);
  }

  __device__ __forceinline__ void first(const SubIn& in, int lane, const Neg& n) {
    const int t = lane & 15, cg = lane >> 4;
    constexpr float kLog2e = 1.4426950408889634f;
    // wsum[m][e] = sum_{s <= t} w[s][c0 + 4m + e] for this lane's token t, as the
    // product (W^T L^T)[c][t]: A = W^T and the constant B[s][t] = [s <= t]. The
    // matrix cores take the sum off the vector ALUs. On the 16x16x32
    // instruction with zero upper halves: results of the legacy 16x16x16 one,
    // read back by VALU, have come out wrong now and then on gfx950 with this
    // toolchain's wait-state insertion.
    const int s0 = 4 * cg;
    const uint32_t one = 0x3f80u;  // bf16 1.0
    const uint4 lt =
        make_uint4((s0 <= t ? one : 0u) | (s0 + 1 <= t ? one << 16 : 0u),
                   (s0 + 2 <= t ? one : 0u) | (s0 + 3 <= t ? one << 16 : 0u), 0u, 0u);
    f32x4 wsum[2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
      wsum[m] = mma32(make_uint4(in.w[m].x, in.w[m].y, 0u, 0u), lt, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const float G = wsum[m >> 2][m & 3] * kLog2e;  // log2 decay through token t
      eh[m] = __builtin_amdgcn_exp2f(G);
      ie[m] = __builtin_amdgcn_exp2f(-G);
    }
    float x[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) x[m] = elem(in.k, m) * ie[m];
    split8(x, kh, kl, n);
    keep(kh);
    keep(kl);
    r = in.r;
    a = in.a;
    b = in.b;
    if constexpr (kEarlyB) {
      make_b(n);
      keep(bh);
      keep(bl);
    } else {
#pragma unroll
      for (int m = 0; m < 8; ++m) asm volatile("" : "+v"(ie[m]));
    }
  }

  __device__ __forceinline__ void second(Slot& S, int lane, int part, float scale, const Neg& n) {
    const int t = lane & 15, c0 = 32 * part + 8 * (lane >> 4), ro = rk_off(t, c0);
    st16(&S.K[0][ro], kh);
    st16(&S.K[1][ro], kl);
    if constexpr (!kEarlyB) make_b(n);
    st16(&S.B[0][ro], bh);
    st16(&S.B[1][ro], bl);
    float x[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) x[m] = elem(a, m) * row_prev(eh[m], 1.f);  // through token t-1
    st16(&S.A[ro], make_uint4(pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3]),
                              pack_bf16(x[4], x[5]), pack_bf16(x[6], x[7])));
#pragma unroll
    for (int m = 0; m < 8; ++m)
      x[m] = kScaled ? elem(r, m) * scale * eh[m] : elem(r, m) * eh[m];
    uint4 hi, lo;
    split8(x, hi, lo, n);
    st16(&S.R[0][ro], hi);
    st16(&S.R[1][ro], lo);
    if (t == kSub - 1) {
      *reinterpret_cast<f32x4*>(&S.gam[c0]) = f32x4{eh[0], eh[1], eh[2], eh[3]};
      *reinterpret_cast<f32x4*>(&S.gam[c0 + 4]) = f32x4{eh[4], eh[5], eh[6], eh[7]};
    }
  }
};

// part: bit 0 the channel half, bit 1 the parity of its sub-chunks.
template <bool kScaled, bool kEarlyB>
__device__ __forceinline__ void operand_role(Shared& sm, int64_t n_sub, int lane, int part,
                                             float scale) {
  const Neg n = neg_consts();
  const int odd = part >> 1;
  part &= 1;
  end_tick();  // the first rows' fill tick
  if (odd) end_tick();
  // Sub-chunk j takes ticks j-4 and j-3; the last tick is n_sub - 1. (The
  // sub-chunk past the end, of zero rows, is the last one: its K~ is read.)
  int64_t j = odd;
  for (; j <= n_sub; j += 2) {
    Operands<kScaled, kEarlyB> op;
    {
      SubIn d;
      read_inputs(sm, d, int(j & (kIn - 1)), lane, part);
      op.first(d, lane, n);
    }
    end_tick();
    op.second(sm.slot[j & (kRing - 1)], lane, part, scale, n);
    end_tick();
  }
  for (; j < n_sub + 4; ++j) end_tick();
}

// ---- scores ---------------------------------------------------------------------------

// Two score matrices of sub-chunk j: pair 0 is L_ab and M_rb (against B~),
// pair 1 L_ak and M_rk (against K~), each as the transposed product Y X^T,
// whose accumulator is the matrix in A-operand lane order. X is A^ (one bf16)
// for the L matrix and the split R^ for M.
template <int pair>
__device__ __forceinline__ void stage_scores(Shared& sm, int64_t j, int lane, const Neg& n) {
  Slot& S = sm.slot[j & (kRing - 1)];
  const int li = lane & 15, lg = lane >> 4;
  const uint16_t* Y = pair ? &S.K[0][0] : &S.B[0][0];
  constexpr int kLo = kSub * kPR;  // hi -> lo array distance
  f32x4 l = {0.f, 0.f, 0.f, 0.f}, m = l;
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
    const int off = rk_off(li, 32 * kb + 8 * lg);
    const uint4 yh = ld16(Y + off), yl = ld16(Y + kLo + off), a = ld16(&S.A[off]);
    l = mma32(yl, a, l);  // (yh + yl) A^
    l = mma32(yh, a, l);
    m = mma32x3(yh, yl, ld16(&S.R[0][off]), ld16(&S.R[1][off]), m);
  }
  // d[r] = D[t = li][s = 4lg + r]; L keeps s < t, M keeps s <= t
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    l[r] = (4 * lg + r < li) ? l[r] : 0.f;
    m[r] = (4 * lg + r <= li) ? m[r] : 0.f;
  }
  uint2 hi, lo;
  if constexpr (pair == 0) {
    *reinterpret_cast<f32x4*>(&sm.Lf[j & 1][lane]) = l;  // T is solved from it in fp32
  } else {
    pack_split(l, hi, lo, n);
    S.M[1][lane] = make_uint4(hi.x, hi.y, lo.x, lo.y);
  }
  pack_split(m, hi, lo, n);
  S.M[2 + pair][lane] = make_uint4(hi.x, hi.y, lo.x, lo.y);
}

// ---- inverse --------------------------------------------------------------------------

// Forward substitution of four columns, one step per row Q: every lane of a
// 16-lane DPP row adds L[tq][Q] times lane Q's value (row_newbcast), T[Q][c].
// A DPP read of a register that a vector instruction just wrote needs two
// wait states: the three other columns' steps stand in between, and the first
// step starts with them.
#define WKV7_SUBST(Q, L)                                                    \
  "v_fmac_f32_dpp %0, %0, " L " row_newbcast:" Q " row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %1, %1, " L " row_newbcast:" Q " row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %2, %2, " L " row_newbcast:" Q " row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %3, %3, " L " row_newbcast:" Q " row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ void substitute(float (&c)[4], const float (&L)[kSub]) {
  asm volatile(
      "s_nop 1\n\t" WKV7_SUBST("0", "%4") WKV7_SUBST("1", "%5") WKV7_SUBST("2", "%6")
      WKV7_SUBST("3", "%7") WKV7_SUBST("4", "%8") WKV7_SUBST("5", "%9") WKV7_SUBST("6", "%10")
      WKV7_SUBST("7", "%11") WKV7_SUBST("8", "%12") WKV7_SUBST("9", "%13")
      WKV7_SUBST("10", "%14") WKV7_SUBST("11", "%15") WKV7_SUBST("12", "%16")
      WKV7_SUBST("13", "%17") WKV7_SUBST("14", "%18")
      : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3])
      : "v"(L[0]), "v"(L[1]), "v"(L[2]), "v"(L[3]), "v"(L[4]), "v"(L[5]), "v"(L[6]), "v"(L[7]),
        "v"(L[8]), "v"(L[9]), "v"(L[10]), "v"(L[11]), "v"(L[12]), "v"(L[13]), "v"(L[14]));
}
#undef WKV7_SUBST

// T = (I - L_ab)^{-1} of sub-chunk j by forward substitution in fp32: lane
// (row tq, column group cg) accumulates T[tq][c] = [tq == c] +
// sum_{q < tq} L[tq][q] T[q][c] for its columns 4 cg .. 4 cg + 3 (L[tq][q] = 0
// for q >= tq); the lanes of one column group form one DPP row. The four
// columns of a lane are then its elements of the A operand.
__device__ __forceinline__ void stage_inverse(Shared& sm, int64_t j, int lane) {
  const int tq = lane & 15, cg = lane >> 4;
  const float4* L = sm.Lf[j & 1];
  float Lr[kSub];  // row tq of L_ab
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const float4 v4 = L[tq + 16 * g];
    Lr[4 * g] = v4.x;
    Lr[4 * g + 1] = v4.y;
    Lr[4 * g + 2] = v4.z;
    Lr[4 * g + 3] = v4.w;
  }
  float acc[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = (tq == 4 * cg + e) ? 1.f : 0.f;
  substitute(acc, Lr);
  // once in each half: P = T X takes X's hi and lo halves in one product
  const uint32_t lo = pack_bf16(acc[0], acc[1]), hi = pack_bf16(acc[2], acc[3]);
  sm.slot[j & (kRing - 1)].M[0][lane] = make_uint4(lo, hi, lo, hi);
}

__device__ __forceinline__ void inverse_role(Shared& sm, int64_t n_sub, int lane) {
  for (int i = 0; i < 4; ++i) end_tick();
  for (int64_t j = 0; j < n_sub; ++j) {
    stage_inverse(sm, j, lane);
    end_tick();
  }
  end_tick();
}

// ---- io -------------------------------------------------------------------------------

// Input loads: whole 128-byte rows straight into LDS. Each input has one
// buffer resource, based at the sequence's first token and sized to the
// sequence, so rows past the sequence end arrive as zeros (the padding
// tokens; with k = v = 0 runs the k and v resources have an empty range). A
// sub-chunk is 12 loads of 8 tokens x 128 B (6 inputs x 2 halves): lane l
// fetches token 8 half + l / 8, 16-byte chunk (l % 8) ^ (token % 8) of the
// row, so the chunks sit XOR-swizzled by the token (the layout of rk_off).
// Every row is read once: with the non-temporal hint the loads alone of
// 8 x 4096 tokens x 32 heads (805 MB) take 134 us, 6.0 TB/s, without it 155.
__device__ __forceinline__ void buf_load_lds16(__amdgpu_buffer_rsrc_t rs, uint32_t voff,
                                               uint32_t soff, uint32_t lds_base) {
  // 16 bytes per lane into LDS at lds_base + 16 lane (M0)
  asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
               : : "{m0}"(lds_base), "v"(voff), "s"(rs), "s"(soff) : "memory");
}

constexpr int kLoads = 12;  // row loads per sub-chunk
// Offsets inside a resource stay below this (plus one sub-chunk); a longer
// sequence moves its resources' base forward.
constexpr uint32_t kRebase = 1u << 30;

struct RowSrc {
  const uint16_t* base[6];  // r, w, k, v, a, b at the resources' first token
  int64_t left;             // bytes of the sequence from there on
  uint32_t soff;            // next sub-chunk's byte offset
  uint32_t step;            // bytes per sub-chunk
  uint32_t voff[2];         // this lane's byte offset of each half
  bool kvz;
  __amdgpu_buffer_rsrc_t rs[6];

  __device__ __forceinline__ void make() {
    const int64_t most = int64_t(kRebase) * 2 - 1;
    const uint32_t bytes = left < 0 ? 0u : static_cast<uint32_t>(left < most ? left : most);
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      // an empty range makes every load return zero (runs with k = v = 0)
      const uint32_t n = kvz && (i == 2 || i == 3) ? 0u : bytes;
      rs[i] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base[i]),
                                                static_cast<short>(0), static_cast<int>(n),
                                                0x00020000);
    }
  }

  __device__ __forceinline__ RowSrc(const Inputs& in, const SeqGeom& g, int lane, bool kvz_) {
    const uint16_t* p[6] = {in.r, in.w, in.k, in.v, in.a, in.b};
#pragma unroll
    for (int i = 0; i < 6; ++i) base[i] = p[i] + g.t_beg * g.tstride + g.hoff;
    left = (g.t_end - g.t_beg) * g.tstride * 2;
    soff = 0;
    step = 2u * uint32_t(kSub) * uint32_t(g.tstride);
    const uint32_t row = uint32_t(lane >> 3), c = uint32_t(lane & 7) ^ row;
    voff[0] = 2u * (row * uint32_t(g.tstride) + 8u * c);
    voff[1] = voff[0] + step / 2;
    kvz = kvz_;
    make();
  }

  // Asks for sub-chunk j's rows; called for j = 0, 1, 2, ...
  __device__ __forceinline__ void issue(Shared& sm, int64_t j) {
    if (soff >= kRebase) {  // (uniform, once per GiB)
#pragma unroll
      for (int i = 0; i < 6; ++i) base[i] += soff / 2;
      left -= soff;
      soff = 0;
      make();
    }
    const uint32_t in = lds_addr(&sm.inb[j & (kIn - 1)][0][0][0]);
    const uint32_t v = lds_addr(&sm.v[j & (kVRing - 1)][0][0]);
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const uint32_t dst = i == 3 ? v : in + (i < 3 ? i : i - 1) * (kSub * 128);
      buf_load_lds16(rs[i], voff[0], soff, dst);
      buf_load_lds16(rs[i], voff[1], soff, dst + 1024);
    }
    soff += step;
  }
};

// y rows of one sub-chunk between LDS and memory, kCols value columns from
// col0 on: 16-byte pieces, piece p of token p / kPer.
template <bool kF32Out, int kCols>
struct YRows {
  static constexpr int kEsz = kF32Out ? 4 : 2;
  static constexpr int kPer = kCols * kEsz / 16;  // pieces per token
  static constexpr int kN = (kSub * kPer + kWave - 1) / kWave;
  typedef unsigned piece __attribute__((ext_vector_type(4)));
  typedef unsigned out_piece __attribute__((ext_vector_type(4), aligned(8)));  // (bf16 y: 8-byte aligned)
  piece d[kN];

  __device__ __forceinline__ void read(const Shared& sm, int64_t j, int lane, int col0) {
    const unsigned char* ys = sm.ys[j & 1] + col0 * kEsz;
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const int p = kWave * i + lane, t = (p / kPer) & (kSub - 1), c = p % kPer;
      d[i] = *reinterpret_cast<const piece*>(ys + t * (kF32Out ? kYRowF : kYRowB) + 16 * c);
    }
  }
  __device__ __forceinline__ void write(void* y, int64_t j, const SeqGeom& g, int lane,
                                        int col0) const {
    unsigned char* yb = static_cast<unsigned char*>(y) +
                        ((g.t_beg + kSub * j) * g.tstride + g.hoff + col0) * kEsz;
    const int left = int(min(g.t_end - g.t_beg - kSub * j, int64_t(kSub)));
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const int p = kWave * i + lane, t = p / kPer, c = p % kPer;
      if (t < left) *reinterpret_cast<out_piece*>(yb + t * g.tstride * kEsz + 16 * c) = d[i];
    }
  }
};

// At the end of tick k sub-chunk k+5's rows must have landed (the operand
// waves read them in the next tick): everything but the two sub-chunks' loads
// asked for after it. The last sub-chunk asked for is the one past the end.
__device__ __forceinline__ void io_role(Shared& sm, const Inputs& in, const SeqGeom& g,
                                        int64_t n_sub, int lane, bool kvz) {
  RowSrc src(in, g, lane, kvz);
  src.issue(sm, 0);
  src.issue(sm, 1);
  for (int64_t j = 2; j <= n_sub; ++j) {  // tick j - 7
    src.issue(sm, j);
    wait_vm<2 * kLoads>();
    end_tick();
  }
  wait_vm<kLoads>();
  end_tick();
  wait_vm<0>();
  for (int i = 0; i < 5; ++i) end_tick();
}

// Pair 1's wave also stores the y rows of the sub-chunk before the state
// step's.
template <int pair, bool kF32Out, int kCols>
__device__ __forceinline__ void score_role(Shared& sm, const SeqGeom& g, int64_t n_sub, int lane,
                                           void* y, int col0) {
  const Neg n = neg_consts();
  for (int i = 0; i < 3; ++i) end_tick();
  for (int i = 0; i < 3; ++i) {  // ticks -2 .. 0
    if (i < n_sub) stage_scores<pair>(sm, i, lane, n);
    end_tick();
  }
  YRows<kF32Out, kCols> rows;
  for (int64_t k = 1; k < n_sub; ++k) {
    if constexpr (pair == 1) {
      rows.read(sm, k - 1, lane, col0);
      rows.write(y, k - 1, g, lane, col0);
    }
    if (k + 2 < n_sub) stage_scores<pair>(sm, k + 2, lane, n);
    end_tick();
  }
  if constexpr (pair == 1) {
    rows.read(sm, n_sub - 1, lane, col0);
    rows.write(y, n_sub - 1, g, lane, col0);
  }
}

// ---- state ----------------------------------------------------------------------------

// What a state wave reads of a sub-chunk one tick before its state step (all
// of it but T is there by then), so that the LDS latency is off the step's
// chain.
struct Ahead {
  uint4 ah[2], rh[2], rl[2], lak, mrk, vv;  // vv: {v, v}

  __device__ __forceinline__ void read(const Shared& sm, int64_t j, int lane, int col0) {
    const Slot& S = sm.slot[j & (kRing - 1)];
    const int li = lane & 15, lg = lane >> 4;
    const uint16_t* V = reinterpret_cast<const uint16_t*>(&sm.v[j & (kVRing - 1)][0][0]);
    const uint2 v = ld_tr(V + rk_off(4 * lg + (li >> 2), col0 + 4 * (li & 3)));
    vv = make_uint4(v.x, v.y, v.x, v.y);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      const int off = rk_off(li, 32 * kb + 8 * lg);
      ah[kb] = ld16(&S.A[off]);
      rh[kb] = ld16(&S.R[0][off]);
      rl[kb] = ld16(&S.R[1][off]);
    }
    lak = S.M[1][lane];
    mrk = S.M[3][lane];
  }
};

// Transposed 16-token operand B~^T or K~^T of key block jb, {hi, lo}: this
// lane reads token row 4 lg + li / 4 at channel 4 (li % 4) of the block and
// receives the block's channel li at tokens 4 lg .. 4 lg + 3.
__device__ __forceinline__ uint4 ld_split_tr(const uint16_t (&x)[2][kSub * kPR], int jb, int lane) {
  const int li = lane & 15, lg = lane >> 4;
  const int off = rk_off(4 * lg + (li >> 2), key_row(jb, 4 * (li & 3)));
  const uint2 hi = ld_tr(&x[0][off]), lo = ld_tr(&x[1][off]);
  return make_uint4(hi.x, hi.y, lo.x, lo.y);
}

// One wave's 16 state columns as the chain carries them from tick to tick:
// split, as the B operand of key blocks kb (tiles 2kb and 2kb+1); in fp32 with
// the next sub-chunk's K~^T V added; and that sub-chunk's L_ak V and
// (M_rk V)^T.
struct State {
  uint4 hi[2], lo[2];
  f32x4 hk[4], X, Z;

  // From the state h before the sub-chunk of kt and in. K~^T V is added first,
  // so that h itself dies in the split (its difference is formed in place).
  __device__ __forceinline__ void take(const f32x4 (&h)[4], const uint4 (&kt)[4], const Ahead& in,
                                       const Neg& n) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int jb = 0; jb < 4; ++jb) hk[jb] = mma32(kt[jb], in.vv, h[jb]);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      uint2 h0h, h0l, h1h, h1l;
      pack_split(h[2 * kb], h0h, h0l, n);
      pack_split(h[2 * kb + 1], h1h, h1l, n);
      hi[kb] = make_uint4(h0h.x, h0h.y, h1h.x, h1h.y);
      lo[kb] = make_uint4(h0l.x, h0l.y, h1l.x, h1l.y);
    }
    X = mma32(in.lak, in.vv, zero);
    Z = mma32(in.vv, in.mrk, zero);
  }
};

// The state wave's y of sub-chunk j (token lane % 16, four value columns)
// into the staging rows, rounded as the output dtype.
template <bool kF32Out>
__device__ __forceinline__ void stage_y(Shared& sm, const f32x4& Z, int64_t j, int lane, int col) {
  unsigned char* row = sm.ys[j & 1] + (lane & 15) * (kF32Out ? kYRowF : kYRowB);
  if constexpr (kF32Out)
    *reinterpret_cast<f32x4*>(row + 4 * col) = Z;
  else
    *reinterpret_cast<uint2*>(row + 2 * col) =
        make_uint2(pack_bf16(Z[0], Z[1]), pack_bf16(Z[2], Z[3]));
}

// State step of sub-chunk j. 16-token products use both halves of the 32-wide
// instruction for two terms of one sum: {mh, ml}.{v, v} = M V for an exact v,
// and {mh, ml}.{ph, 0} + {mh, ml}.{pl, ph} = mh ph + mh pl + ml ph for a split
// P. y is computed transposed (value columns by tokens), so that a lane holds
// four neighbouring columns of one token. The compiler's own order of the
// step is kept: fences that put each tile's vector work beside the next
// tile's products made the chain 15 % longer.
template <bool kF32Out>
__device__ __forceinline__ void stage_state(Shared& sm, State& st, Ahead& in, int64_t j, int lane,
                                            int col0, const Neg& n) {
  const Slot& S = sm.slot[j & (kRing - 1)];
  const int lg = lane >> 4;
  const uint4 tm = S.M[0][lane];
  uint4 bt[4], kt[4];
  f32x4 gm[4];
#pragma unroll
  for (int jb = 0; jb < 4; ++jb) bt[jb] = ld_split_tr(S.B, jb, lane);
  const uint4 mrb = S.M[2][lane];
#pragma unroll
  for (int jb = 0; jb < 4; ++jb)
    gm[jb] = *reinterpret_cast<const f32x4*>(&S.gam[key_row(jb, 4 * lg)]);
  f32x4 X = st.X, Z = st.Z;
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {  // X: + A^ h (A^ as one bf16, h split)
    X = mma32(in.ah[kb], st.lo[kb], X);
    X = mma32(in.ah[kb], st.hi[kb], X);
  }
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {  // Z: + (R^ h)^T
    Z = mma32(st.hi[kb], in.rl[kb], Z);
    Z = mma32(st.lo[kb], in.rh[kb], Z);
    Z = mma32(st.hi[kb], in.rh[kb], Z);
  }
  uint2 xh, xl, ph, pl;
  pack_split(X, xh, xl, n);
  // P = T xh + T xl
  const f32x4 P = mma32(tm, make_uint4(xh.x, xh.y, xl.x, xl.y), f32x4{0.f, 0.f, 0.f, 0.f});
  in.read(sm, j + 1, lane, col0);
#pragma unroll
  for (int jb = 0; jb < 4; ++jb) kt[jb] = ld_split_tr(sm.slot[(j + 1) & (kRing - 1)].K, jb, lane);
  pack_split(P, ph, pl, n);
  const uint4 pp = make_uint4(pl.x, pl.y, ph.x, ph.y);  // {pl, ph}
  const uint4 p0 = make_uint4(ph.x, ph.y, 0u, 0u);      // {ph, 0}
  f32x4 h[4];
#pragma unroll
  for (int jb = 0; jb < 4; ++jb) {
    h[jb] = mma32(bt[jb], p0, st.hk[jb]);
    h[jb] = mma32(bt[jb], pp, h[jb]);
    h[jb] *= gm[jb];
  }
  Z = mma32(p0, mrb, Z);  // (M_rb P)^T: mh ph
  Z = mma32(pp, mrb, Z);  // + mh pl + ml ph
  st.take(h, kt, in, n);
  stage_y<kF32Out>(sm, Z, j, lane, col0 + 4 * lg);
}

// Value columns col0 .. col0 + 15. hsrc / hdst: this head's [64 keys][64
// values] tile (hsrc null: zero start, or the identity with `eye`; hdst null:
// the final state is not written).
template <bool kF32Out>
__device__ __forceinline__ void state_role(Shared& sm, const float* hsrc, float* hdst, bool eye,
                                           int64_t n_sub, int lane, int col0) {
  const int li = lane & 15, lg = lane >> 4;
  const Neg n = neg_consts();
  // State columns of this wave as 16x16 accumulator tiles.
  f32x4 h[4];
  if (hsrc) {
#pragma unroll
    for (int jb = 0; jb < 4; ++jb)
#pragma unroll
      for (int r = 0; r < 4; ++r) h[jb][r] = hsrc[key_row(jb, 4 * lg + r) * kHead + col0 + li];
  } else {
#pragma unroll
    for (int jb = 0; jb < 4; ++jb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        h[jb][r] = eye && key_row(jb, 4 * lg + r) == col0 + li ? 1.f : 0.f;
  }
  if (n_sub > 0) {
    for (int i = 0; i < 4; ++i) end_tick();  // fill ticks
    Ahead in;
    in.read(sm, 0, lane, col0);
    uint4 kt[4];
#pragma unroll
    for (int jb = 0; jb < 4; ++jb) kt[jb] = ld_split_tr(sm.slot[0].K, jb, lane);
    State st;
    st.take(h, kt, in, n);
    end_tick();
    for (int64_t k = 0; k < n_sub; ++k) {
      stage_state<kF32Out>(sm, st, in, k, lane, col0, n);
      end_tick();
    }
    // the sub-chunk past the end has k = v = 0: hk is the final state (of its
    // other operands nothing is made, and nothing of what they give is used)
#pragma unroll
    for (int jb = 0; jb < 4; ++jb) h[jb] = st.hk[jb];
  }
  if (hdst) {
#pragma unroll
    for (int jb = 0; jb < 4; ++jb)
#pragma unroll
      for (int r = 0; r < 4; ++r) hdst[key_row(jb, 4 * lg + r) * kHead + col0 + li] = h[jb][r];
  }
}

// ---- the kernel -----------------------------------------------------------------------

// y = 0 for every token of a run whose state rows were rejected (as the decode
// step does for a rejected row): 16 lanes per 128-byte (bf16) or 256-byte
// (fp32) row.
template <bool kF32Out>
__device__ __forceinline__ void zero_y(void* y, const SeqGeom& g) {
  const int col = threadIdx.x & 15;
  for (int64_t t = g.t_beg + (threadIdx.x >> 4); t < g.t_end; t += blockDim.x / 16) {
    const int64_t o = t * g.tstride + g.hoff;
    if constexpr (kF32Out)
      reinterpret_cast<float4*>(static_cast<float*>(y) + o)[col] = make_float4(0.f, 0.f, 0.f, 0.f);
    else
      reinterpret_cast<uint2*>(static_cast<uint16_t*>(y) + o)[col] = make_uint2(0u, 0u);
  }
}

enum Role : int { kState, kOperand, kScore, kInverse, kIo, kNone };

// A workgroup form: kStateWaves value-column blocks of 16 per workgroup, and
// the role and part of each of its 12 waves, 4 bits per wave from wave 0 up
// (wave w runs on SIMD w % 4).
constexpr int kWaves = 12;

template <class Form, bool kF32Out, bool kScaled, int N>
__global__ __launch_bounds__(kWaves * kWave) void prefill_kernel(const PrefillArgs<N> p) {
  constexpr int kCols = Form::kStateWaves * 16;  // value columns per workgroup
  constexpr int kSplit = kHead / kCols;                     // workgroups per (sequence, head)
  __shared__ Shared sm;

  const int lane = threadIdx.x & 63;
  // wave-uniform by construction; through readfirstlane the compiler knows it,
  // so the role branches are scalar branches
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  // sequences outermost: the longest ones of every layer start first (a
  // launch's workgroups fit 32 bits)
  const uint32_t item = blockIdx.x / kSplit, heads = uint32_t(p.H);
  const uint32_t per_seq = N == 1 ? heads : uint32_t(p.layers) * heads;
  const uint32_t at = item / per_seq, rest = item - at * per_seq;
  const uint32_t layer_at = N == 1 ? 0 : rest / heads;
  const int64_t pos = at, layer = layer_at, head = rest - layer_at * heads;
  const wkv7_layer_io& io = p.io[layer_at];
  const int64_t seq = p.seq_order ? int64_t(p.seq_order[pos]) : pos;
  if (seq < 0 || seq >= p.nseq) return;  // uniform: the whole block leaves
  const Runs& runs = p.runs;
  const int fl = runs.flags ? runs.flags[seq] : 0;
  const int32_t* cu = p.cu_seqlens;
  int64_t ci = seq;
  if (seq >= runs.n_primary) {  // only with cu_alt (n_primary = nseq otherwise)
    cu = runs.cu_alt;
    ci = 2 * (seq - runs.n_primary);
  }
  SeqGeom g;
  g.t_end = min(max(int64_t(cu[ci + 1]), int64_t(0)), p.total_tokens);
  g.t_beg = min(max(int64_t(cu[ci]), int64_t(0)), g.t_end);
  g.tstride = int64_t(p.H) * kHead;
  g.hoff = head * kHead;
  const int64_t n_sub = (g.t_end - g.t_beg + kSub - 1) / kSub;
  void* yb = (fl & WKV7_RUN_Y_ALT) ? runs.y_alt : io.y;

  // State rows of this run: checked before any state access (uniform).
  const bool state_alt = fl & WKV7_RUN_STATE_ALT;
  float* out_base = state_alt ? runs.state_alt : p.wkv ? p.wkv + layer * p.layer_stride : nullptr;
  const int64_t out_rows = state_alt ? runs.alt_rows : p.num_rows;
  const int64_t slot = p.slot_ids ? int64_t(p.slot_ids[seq]) : seq;
  const bool from_eye = fl & WKV7_RUN_INIT_IDENTITY;
  const bool from_zero = !from_eye && (p.zero_init || (fl & WKV7_RUN_INIT_ZERO));
  const bool from_in = !from_eye && !from_zero && runs.state_in;
  const int64_t in_row = from_in ? (runs.in_ids ? int64_t(runs.in_ids[seq]) : seq) : 0;
  const bool rows_ok = (!out_base || (slot >= 0 && slot < out_rows)) &&
                       (!from_in || (in_row >= 0 && in_row < runs.in_rows)) &&
                       (from_eye || from_zero || from_in || out_base);
  if (!rows_ok) {
    zero_y<kF32Out>(yb, g);
    return;  // uniform: the whole block leaves
  }
  const int wg_col = kSplit > 1 ? int(blockIdx.x % kSplit) * kCols : 0;
  const int role = int((Form::kRoles >> (4 * wave)) & 15);
  const int part = int((Form::kParts >> (4 * wave)) & 15);
  if (role == kState) {
    const int64_t tile = kHead * kHead;
    const float* hsrc = from_eye || from_zero ? nullptr
                        : from_in ? runs.state_in + (in_row * p.H + head) * tile
                                  : out_base + (slot * p.H + head) * tile;
    float* hdst = out_base ? out_base + (slot * p.H + head) * tile : nullptr;
    state_role<kF32Out>(sm, hsrc, hdst, from_eye, n_sub, lane, wg_col + 16 * part);
  } else if (n_sub > 0) {
    if (role == kOperand)
      operand_role<kScaled, Form::kEarlyB>(sm, n_sub, lane, part, p.scale);
    else if (role == kScore && part == 0)
      score_role<0, kF32Out, kCols>(sm, g, n_sub, lane, yb, wg_col);
    else if (role == kScore)
      score_role<1, kF32Out, kCols>(sm, g, n_sub, lane, yb, wg_col);
    else if (role == kInverse)
      inverse_role(sm, n_sub, lane);
    else if (role == kIo)
      io_role(sm, Inputs{io.r, io.w, io.k, io.v, io.a, io.b}, g, n_sub, lane, fl & WKV7_RUN_KV_ZERO);
    else
      for (int64_t k = 0; k < n_sub + 5; ++k) end_tick();  // no work: every tick's barrier
  }
}

template <class Form, int N>
int launch_layers(unsigned blocks, hipStream_t s, bool f32_out, bool scaled, const PrefillPlan& p,
                  const wkv7_layer_io* io) {
  PrefillArgs<N> a{p, {}};
  for (int l = 0; l < p.layers; ++l) a.io[l] = io[l];
  const dim3 grid(blocks), threads(kWaves * kWave);
  if (f32_out) {
    if (scaled) prefill_kernel<Form, true, true, N><<<grid, threads, 0, s>>>(a);
    else prefill_kernel<Form, true, false, N><<<grid, threads, 0, s>>>(a);
  } else {
    if (scaled) prefill_kernel<Form, false, true, N><<<grid, threads, 0, s>>>(a);
    else prefill_kernel<Form, false, false, N><<<grid, threads, 0, s>>>(a);
  }
  return launch_status();
}

template <class Form>
int launch_form(unsigned blocks, hipStream_t s, bool f32_out, bool scaled, const PrefillPlan& p,
                const wkv7_layer_io* io) {
  return p.layers == 1 ? launch_layers<Form, 1>(blocks, s, f32_out, scaled, p, io)
                       : launch_layers<Form, kMaxLayers>(blocks, s, f32_out, scaled, p, io);
}

}  // namespace
}  // namespace wkv7
