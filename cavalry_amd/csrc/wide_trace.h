// Traces over the wide tree; see wide_trace.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "launch.h"
#include "lbvh.h"

namespace cav {

// Launched through ls after the dispensers and pass counters are cleared;
// coop's buffers and a wide tree are required. counters as in lbvh.h.
void wide_closest(const TraceBvh& bvh, const float* rays, int64_t nrays, const uint32_t* nrays_dev, int32_t* prim,
                  float* t, float* u, float* v, uint32_t* counters, const TraceLaunch& L, const TraceCoop& coop,
                  LaunchSink& ls);
void wide_occluded(const TraceBvh& bvh, const float* rays, int64_t nrays, const uint32_t* nrays_dev,
                   const float* limit, const int32_t* src, const int32_t* dst, uint8_t* visible, uint32_t* counters,
                   const TraceLaunch& L, const TraceCoop& coop, LaunchSink& ls);

}  // namespace cav
