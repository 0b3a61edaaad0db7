// The prefill kernels for launches that would leave compute units idle: each
// (sequence, head) runs on two or four workgroups, each owning 32 or 16 of the
// head's 64 value columns and repeating the preparation, which does not depend
// on them. The per-column arithmetic is the whole-head kernel's
// (wkv7_prefill_core.h), so the results are the same bits.
#include "wkv7_prefill_core.h"

namespace wkv7 {
namespace {

struct HalfHead {
  static constexpr int kStateWaves = 2;
  static constexpr bool kEarlyB = false;
  // SIMD 0: state 0, score 0, inverse; 1: state 1, score 1, io; 2 and 3: the
  // two parities' operand waves of a channel half
  static constexpr uint64_t kRoles = 0x5543'1122'1100ull, kParts = 0x0000'3210'1010ull;
};

struct QuarterHead {
  static constexpr int kStateWaves = 1;
  static constexpr bool kEarlyB = false;
  // SIMD 0: state, io; 1 and 2: the operand waves of a channel half; 3: both
  // scores and the inverse (io elsewhere and the state wave by itself: 5 %
  // slower)
  static constexpr uint64_t kRoles = 0x3555'2114'2110ull, kParts = 0x0000'1320'0100ull;
};

}  // namespace

int prefill_split_launch(int split, unsigned blocks, hipStream_t s, bool f32_out, bool scaled,
                         const PrefillPlan& p, const wkv7_layer_io* io) {
  if (split == 2) return launch_form<HalfHead>(blocks, s, f32_out, scaled, p, io);
  return launch_form<QuarterHead>(blocks, s, f32_out, scaled, p, io);
}

}  // namespace wkv7
