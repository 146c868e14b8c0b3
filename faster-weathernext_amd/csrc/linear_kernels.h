// Launch arguments of the linear weight gradient (linear.hip), formed by linear_api.cpp.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fwn {

struct WgradArgs {
  const void* g;      // [rows, outs] bf16
  const void* x;      // [rows, ins] bf16
  float* part;        // [splits, outs, ins], then [splits, outs] where db is given
  void* dw;           // [outs, ins] bf16
  void* db;           // [outs] bf16 or null
  int64_t rows;
  int32_t outs, ins;
  int32_t splits;     // row ranges, each `chunk` rows (the last may be shorter)
  int32_t chunk;      // a multiple of 32
};

hipError_t launch_wgrad(const WgradArgs& a, hipStream_t stream);

}  // namespace fwn
