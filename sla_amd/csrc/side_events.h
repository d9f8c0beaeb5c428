// Ordering of a caller's second stream against its main one (module_fwd.hip, module_bwd.hip).
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

// A call uses the second stream only from this size of one of q, k, v on.  Handing work to it and back costs 25 us of host
// time in the forward and 80 us in the backward, which the overlap has to win back.  Measured (forward + backward, 12 heads
// of 128, two streams against one, in us): 4096 rows (12.6 MB) 301 / 239, 8192 rows (25 MB) 402 / 432, 32760 rows (101 MB)
// 1928 / 1997; the forward alone 78 / 84, 120 / 133, 478 / 502, with 25 us more of host time per call.
constexpr int64_t SIDE_MIN_BYTES = 16ll << 20;
static inline bool side_stream_pays(int B, int H, int L, int D) { return (int64_t)B * H * L * D * 2 >= SIDE_MIN_BYTES; }

#define SLA_HIP_OK(call) SLA_REQUIRE((call) == hipSuccess, SLA_ERR_LAUNCH, #call " failed")

}  // namespace sla
