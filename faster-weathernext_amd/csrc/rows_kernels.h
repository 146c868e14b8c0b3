// Interface between the row-pass launchers (rows_api.cpp) and their kernels (rows.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fwn_rows.h"

namespace fwn {

struct RowArgs {
  const void* x;
  const int64_t* perm;
  void* x_out;       // gather: permuted copy of x
  void* norm_out;    // gather: its layer norm, or null
  const float* mul;  // scatter: [batch, channels] or null
  const float* add;  // scatter: [batch, channels] or null
  void* out;         // scatter: output
  const void* addend;  // scatter: added to x before the norm (the sum goes to x_out, required then), or null
  int32_t batch, n, channels;
  float eps;
  bool stream;  // set by launch_rows: the kernel whose stores are non-temporal
};

enum class RowPass { kGatherNorm, kNormScatter };

// Launches one pass; dtype is FWN_F32 or FWN_BF16 and channels a validated multiple of 8.
hipError_t launch_rows(RowPass pass, int dtype, const RowArgs& a, hipStream_t stream);

struct CondArgs {
  const void* weight[FWN_COND_MAX];  // [2 * channels, cond_size] of each norm
  const void* bias[FWN_COND_MAX];    // [2 * channels]
  const void* cond;                  // [batch, cond_size]
  float* mul;                        // [count, batch, channels]
  float* add;
  int32_t count, batch, channels, cond_size;
};

hipError_t launch_cond(int dtype, const CondArgs& a, hipStream_t stream);

struct RowBwdArgs {
  const void* x;
  const int64_t* perm_grad;  // row i's g_norm is row perm_grad[i], or null
  const int64_t* perm_out;   // row i's gradient goes to row perm_out[i], or null
  const void* g_norm;        // or null
  const void* g_res;         // or null
  const float* mul;          // [batch, channels] or null
  void* gx;
  float* part;   // [batch][blocks][2][channels] partial sums (g_mul's, g_add's), or null: no sums
  float* g_mul;  // [batch, channels], with part
  float* g_add;
  int32_t batch, n, channels, blocks;  // blocks: workgroups per batch member
  float eps;
  bool stream;  // set by launch_rows_bwd: the kernel whose stores are non-temporal
};

// Workgroups per batch member of the backward pass.
int32_t rows_bwd_blocks(int32_t batch, int32_t n, bool sums);

// The backward pass and, with a.part, the reduction of its partial sums.
hipError_t launch_rows_bwd(int dtype, const RowBwdArgs& a, hipStream_t stream);

}  // namespace fwn
