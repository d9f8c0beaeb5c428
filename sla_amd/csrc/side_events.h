// Ordering of a caller's second stream against its main one (module_fwd.hip, sage.hip).
#pragma once
#include "common.h"

#include <mutex>

namespace sla {

// One set per device, made on first use and kept.  A call records and waits on them while it holds the lock: calls from
// several host threads take turns enqueueing.
struct SideEvents {
  hipEvent_t fork = nullptr, join = nullptr;
};
std::mutex& side_events_mutex();
int side_events_for_current_device(SideEvents** out);      // (with the lock held)

// The module's forward uses the second stream from this size of one of q, k, v on.  Handing work to it and back costs 15 to 40 us
// where a call is waited for, and on one stream the independent launches are merged anyway.  Measured, two streams / one, us per
// call among others (and waited for): 12 heads x 6500 x 128 (19 MiB) 103 / 103 (137 / 124), 40 x 6500 x 64 (32 MiB) 122 / 126 (156 / 147),
// 12 x 16000 x 128 (47 MiB) 265 / 263 (302 / 286), 8 x 32000 x 128 (63 MiB) 548 / 546 (581 / 566), 2 x 75600 x 128 (37 MiB) 751 / 760
// (800 / 782); 12 x 32760 x 128 (96 MiB) 484 / 500.
constexpr int64_t SIDE_MIN_BYTES_FWD = 64ll << 20;
static inline bool side_stream_pays_fwd(int B, int H, int L, int D) { return (int64_t)B * H * L * D * 2 >= SIDE_MIN_BYTES_FWD; }

// The quantised forward, whose preparation is mostly passes over memory, from this size on, or from this many operations of one
// product over the selected tiles on (few heads with long sequences).  Two / one: 12 heads x 6500 x 128 (19 MiB) 122 / 128 (164 /
// 157), 24 x 6500 x 64 106 / 104 (153 / 135), 16 x 8000 x 128 (31 MiB) 155 / 154 (196 / 184), 40 x 6500 x 64 (32 MiB) 145 / 161 (192 /
// 191), 12 x 16000 x 128 257 / 282, 4 x 40000 x 128 359 / 390.
constexpr int64_t SIDE_MIN_BYTES = 16ll << 20;
constexpr int64_t SIDE_MIN_OPS = 16000000000ll;
static inline bool side_stream_pays(int B, int H, int L, int D, int topk) {
  const int64_t elems = (int64_t)B * H * L * D;
  return elems * 2 >= SIDE_MIN_BYTES || elems * 2 * 64 * topk >= SIDE_MIN_OPS;
}

#define SLA_HIP_OK(call) SLA_REQUIRE((call) == hipSuccess, SLA_ERR_LAUNCH, #call " failed")

}  // namespace sla
