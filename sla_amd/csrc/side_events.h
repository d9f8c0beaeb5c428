// Ordering of a caller's second stream against its main one (module_fwd.hip, sage.hip).
#pragma once
#include "common.h"

#include <mutex>

namespace sla {

// One set per device, made on first use and kept.  A call records and waits on them while it holds the lock: calls from
// several host threads take turns enqueueing.
struct SideEvents {
  hipEvent_t fork = nullptr, first = nullptr, second = nullptr, third = nullptr;
};
std::mutex& side_events_mutex();
int side_events_for_current_device(SideEvents** out);      // (with the lock held)

// A call uses the second stream only from this size of one of q, k, v on, or from this many operations of one product over the
// selected tiles on (few heads with long sequences, whose short kernels are few workgroups with long chains).  Handing work to
// it and back costs 25 us of host time in the forward, 30 in the quantised one and 80 in the backward, which the GPU has to
// be busy for: the line is where the pass on one stream takes as long as the host needs to enqueue it on two.
// Measured, two streams against one, over 2 to 40 heads, both head dims, 4 to 64 MiB (forward + backward in us):
//   by size, rows of 64 values: 24 heads x 4096 (12 MiB) 314 / 202, x 5461 (16 MiB) 320 / 269, x 8192 (24 MiB) 329 / 337;
//     40 heads x 2457 329 / 243, x 3276 337 / 330, x 6553 398 / 424; rows of 128: 8 heads x 6144 (12 MiB) 296 / 206, x 8192
//     294 / 245, x 12288 337 / 352; 40 heads x 1228 246 / 223, x 1638 (16 MiB) 248 / 271; 24 heads x 2730 274 / 294.  The forward
//     and the quantised forward gain 2 to 11 % from 16 MiB on (24 heads x 5461 x 64: 72 / 76 and 100.6 / 101.4).
//   by operations, below 16 MiB: 2 heads x 40000 x 64, 62 blocks per row (41 GFLOP) 633 / 722, forward 171 / 180, quantised 191 /
//     198; 16 heads x 4096 x 64, 32 blocks (17 GFLOP) 301 / 302, 86 / 89, 90 / 95; 4 heads x 16000 x 64, 25 blocks (13 GFLOP) 288 /
//     317, 85 / 89, 109 / 99; 24 heads x 2700 x 64, 21 blocks (11 GFLOP) 342 / 302, 87 / 89, 98 / 107.
constexpr int64_t SIDE_MIN_BYTES = 16ll << 20;
constexpr int64_t SIDE_MIN_OPS = 16000000000ll;
static inline bool side_stream_pays(int B, int H, int L, int D, int topk) {
  const int64_t elems = (int64_t)B * H * L * D;
  return elems * 2 >= SIDE_MIN_BYTES || elems * 2 * 64 * topk >= SIDE_MIN_OPS;
}

#define SLA_HIP_OK(call) SLA_REQUIRE((call) == hipSuccess, SLA_ERR_LAUNCH, #call " failed")

}  // namespace sla
