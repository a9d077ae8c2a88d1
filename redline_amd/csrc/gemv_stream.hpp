// The streaming weight-only GEMV (gemv_stream.hip): entry points for the
// launch policies in gemv_w4.hip.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstdint>

namespace rlk {

struct StreamCall {
  const uint16_t* x;
  const uint8_t* w;
  const uint16_t* scales;
  const uint16_t* offsets;  // null: INT8 weight, one scale per row
  const uint16_t* bias;
  void* y;
  int m, n, k, group_size, mode, y_ld;
};

// Launches the streaming kernel; kNoFit when the shape is not one it takes (K
// a multiple of 128; INT4: groups of 32, 64 or a multiple of 128).
int launch_gemv_stream(const StreamCall& c, hipStream_t stream);

}  // namespace rlk
