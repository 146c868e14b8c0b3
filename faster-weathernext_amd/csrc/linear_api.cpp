// C ABI of the linear weight gradient (fwn_rows.h): host-side validation and the split of the rows.
#include <algorithm>
#include <cstdint>

#include <hip/hip_runtime.h>

#include "fwn_internal.h"
#include "fwn_rows.h"
#include "linear_kernels.h"

namespace fwn {
namespace {

constexpr int64_t kCus = 256;
constexpr int64_t kTile = 256;        // output tile of a workgroup
constexpr int64_t kRows = 32;         // rows of one pipeline stage
constexpr int64_t kLeast = 8 * kRows;  // rows below which another split costs more than it gives
constexpr int64_t kBytes = INT64_C(1) << 31;

// One workgroup a CU and as many row ranges as that allows; ranges whose bytes fit the 32-bit offsets.
int plan(int64_t rows, int32_t outs, int32_t ins, WgradArgs* a, const char* what) {
  if (rows < 1) return fail(FWN_ERR_INVALID_ARG, "%s: %lld rows", what, (long long)rows);
  if (outs < 1 || ins < 1 || outs % FWN_LINEAR_UNIT || ins % FWN_LINEAR_UNIT || outs > FWN_LINEAR_MAX ||
      ins > FWN_LINEAR_MAX)
    return fail(FWN_ERR_INVALID_ARG, "%s: outs %d and ins %d must be multiples of %d up to %d", what, outs, ins,
                FWN_LINEAR_UNIT, FWN_LINEAR_MAX);
  const int64_t tiles = (int64_t)((outs + kTile - 1) / kTile) * ((ins + kTile - 1) / kTile);
  // Offsets reach three stages and a tile's columns past a range's end.
  const int64_t most = kBytes / (2 * std::max(outs, ins)) / kRows * kRows - 16 * kRows;
  int64_t splits = std::min(std::max<int64_t>(1, kCus / tiles), std::max<int64_t>(1, rows / kLeast));
  int64_t chunk = ((rows + splits - 1) / splits + kRows - 1) / kRows * kRows;
  chunk = std::min(chunk, most);
  splits = (rows + chunk - 1) / chunk;
  if (splits * tiles > INT32_MAX / 2) return fail(FWN_ERR_INVALID_ARG, "%s: too many rows", what);
  a->rows = rows;
  a->outs = outs;
  a->ins = ins;
  a->splits = (int32_t)splits;
  a->chunk = (int32_t)chunk;
  return FWN_OK;
}

uint64_t part_bytes(const WgradArgs& a) {
  return (uint64_t)a.splits * a.outs * ((uint64_t)a.ins + 1) * sizeof(float);
}

bool misaligned(const void* p) { return ((uintptr_t)p & 15u) != 0; }

}  // namespace
}  // namespace fwn

extern "C" {

int fwn_linear_wgrad_workspace_size(int64_t rows, int32_t outs, int32_t ins, uint64_t* bytes) {
  using namespace fwn;
  clear_error();
  const char* what = "fwn_linear_wgrad_workspace_size";
  if (!bytes) return fail(FWN_ERR_INVALID_ARG, "%s: null argument", what);
  WgradArgs a{};
  const int rc = plan(rows, outs, ins, &a, what);
  if (rc != FWN_OK) return rc;
  *bytes = part_bytes(a);
  return FWN_OK;
}

int fwn_linear_wgrad_launch(int64_t rows, int32_t outs, int32_t ins, const void* g, const void* x, void* dw, void* db,
                            void* workspace, uint64_t workspace_bytes, void* stream) {
  using namespace fwn;
  clear_error();
  const char* what = "fwn_linear_wgrad_launch";
  WgradArgs a{};
  const int rc = plan(rows, outs, ins, &a, what);
  if (rc != FWN_OK) return rc;
  if (!g || !x || !dw || !workspace) return fail(FWN_ERR_INVALID_ARG, "%s: null argument", what);
  if (misaligned(g) || misaligned(x) || misaligned(dw) || misaligned(db) || misaligned(workspace))
    return fail(FWN_ERR_INVALID_ARG, "%s: tensors and workspace must be 16-byte aligned", what);
  if (workspace_bytes < part_bytes(a))
    return fail(FWN_ERR_INVALID_ARG, "%s: workspace of %llu bytes, %llu needed", what, (unsigned long long)workspace_bytes,
                (unsigned long long)part_bytes(a));
  a.g = g;
  a.x = x;
  a.part = (float*)workspace;
  a.dw = dw;
  a.db = db;
  const hipError_t e = launch_wgrad(a, (hipStream_t)stream);
  if (e != hipSuccess) return fail(FWN_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
  return FWN_OK;
}

}  // extern "C"
