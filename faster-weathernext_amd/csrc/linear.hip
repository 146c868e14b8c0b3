// Weight gradient of a linear layer over very many rows: dw = g^T x, db = column sums of g.
//
// The product's output is small (768 x 768 to 3072 x 768: 9 to 36 tiles of 256 x 256 for 256 CUs) and
// its inner dimension long (40,962 nodes), so the rows are split over enough workgroups to fill the
// chip, each writing a float32 partial tile that a second pass sums in a fixed order.
// Measured (db included), us, this kernel against a GEMM and a column sum in sequence, which leave
// most of the chip idle: 40,962 rows of 768 x 2304 162 / 414, 768 x 768 67 / 255, 768 x 3072 194 / 405
// (982 TFLOP/s), 256 x 256 31 / 152; 10,242 rows of 768 x 768 34 / 89; 2,562 rows 25 / 40. Of the large
// ones about three quarters is the matrix units' time, the rest the partials' trip through memory
// (66 MB), the pipeline's fill and the LDS reads.
//
// A workgroup is 8 waves on one 256 x 256 tile, a wave 128 x 64 of it (8 accumulators of 32x32, 128
// registers): per 16 rows it reads 6 KB of LDS for 8 MFMAs, so the CU reads 48 KB (about 250 clocks at
// the 198 bytes a clock that transpose reads reach) in 512 of its matrix clocks, where 128 x 128 over 4
// waves would leave one wave a SIMD and 64 x 64 over 16 would read 64 KB for 512. Both operands are row-major in the contracted dimension, so both are transpose reads
// (ds_read_b64_tr_b16) of [32 rows][128 columns] tiles in the swizzled layout of the attention
// kernels. Four 32 KB stages of 32 rows (128 KB of the 160): the copies of two stages are in flight
// while one stage is read and the next has landed.
#include "attn_bf16_tiles.h"
#include "linear_kernels.h"

namespace fwn {
namespace {

constexpr int TILE = 256, ROWS = 32;           // output tile, rows of a stage
constexpr int SUB = ROWS * 128 * 2;            // one [32][128] bf16 sub-tile
constexpr int STAGE = 4 * SUB;                 // g columns 0-127, 128-255, x columns 0-127, 128-255
constexpr int STAGES = 4;

// All but the newest `vm` of this wave's copies have landed and its LDS reads have returned.
template <int vm>
__device__ __forceinline__ void stage_barrier() {
  __builtin_amdgcn_s_waitcnt(0x0070 | vm);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__global__ void __launch_bounds__(512, 2) wgrad_kernel(WgradArgs a) {
  // One array a stage: the compiler waits for the copies into the array a read names, and for those
  // alone (with one array it waits for the newest copy before every read).
  __shared__ __align__(16) char lds0[STAGE], lds1[STAGE], lds2[STAGE], lds3[STAGE];
  lds_char *const s0 = (lds_char*)lds0, *const s1 = (lds_char*)lds1, *const s2 = (lds_char*)lds2,
           *const s3 = (lds_char*)lds3;
  const int lane = (int)threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // Workgroups go to the 8 XCDs in turn: each takes a contiguous range of (row range, tile), so the
  // tiles that read the same rows share an L2.
  const int total = (int)gridDim.x, xcd = (int)blockIdx.x & 7, q = total >> 3, rem = total & 7;
  const int id = xcd * q + (xcd < rem ? xcd : rem) + ((int)blockIdx.x >> 3);
  const int ti = (a.ins + TILE - 1) / TILE, tiles = (a.outs + TILE - 1) / TILE * ti;
  const int split = id / tiles, tile = id - split * tiles, to = tile / ti;
  const int o0 = to * TILE, i0 = (tile - to * ti) * TILE;
  const int64_t r0 = (int64_t)split * a.chunk;
  const int rows = (int)(a.rows - r0 < a.chunk ? a.rows - r0 : a.chunk);
  const uint32_t sg = (uint32_t)a.outs * 2, sx = (uint32_t)a.ins * 2;
  // Rows past the range lie past the buffer's end: their copies are zeros.
  const rsrc_t rg = make_rsrc((const uint16_t*)a.g + r0 * a.outs, (uint32_t)rows * sg);
  const rsrc_t rx = make_rsrc((const uint16_t*)a.x + r0 * a.ins, (uint32_t)rows * sx);

  // One instruction of wave w: rows 4w .. 4w + 3 of a sub-tile.
  const int row = 4 * w + lane / 16;
  const uint32_t chunk = (uint32_t)((lane % 16) ^ swz<16>(row)) << 4;
  uint32_t vg = (uint32_t)row * sg + (uint32_t)o0 * 2 + chunk, vx = (uint32_t)row * sx + (uint32_t)i0 * 2 + chunk;
  const auto copy = [&](lds_char* stage) {  // the next 32 rows
    lds_char* base = stage + w * 1024;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rg, (__attribute__((address_space(3))) void*)(base + h * SUB), 16,
                                               (int)(vg + h * 256), 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (__attribute__((address_space(3))) void*)(base + (2 + h) * SUB), 16,
                                               (int)(vx + h * 256), 0, 0, 0);
    }
    vg += ROWS * sg;
    vx += ROWS * sx;
  };

  const int wo = w >> 2, wi = w & 3;  // this wave's output rows 128 wo .. and columns 64 wi ..
  Off<128> off;
  off.init(lane);
  uint32_t offx[2][2];
#pragma unroll
  for (int n = 0; n < 2; ++n)
#pragma unroll
    for (int h = 0; h < 2; ++h) offx[n][h] = (2 + (wi >> 1)) * SUB + ((wi & 1) ? off.tr[2 + n][h] : off.tr[n][h]);
  // The operands of rows 16c .. 16c + 15 of a stage.
  const auto read = [&](const lds_char* stage, int c, u32x4(&fa)[4], u32x4(&fb)[2]) {
    const lds_char* base = stage + c * (16 * 256);
#pragma unroll
    for (int m = 0; m < 4; ++m) fa[m] = tr_operand<128>(base + wo * SUB, off, m, 0, 0);
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const u32x2 lo = tr_read(base, offx[n][0]), hi = tr_read(base, offx[n][1]);
      fb[n] = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  };
  f32x16 acc[4][2];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int n = 0; n < 2; ++n) acc[m][n] = zero16();
  const auto multiply = [&](const u32x4(&fa)[4], const u32x4(&fb)[2]) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int n = 0; n < 2; ++n) acc[m][n] = mfma_bf16(fa[m], fb[n], acc[m][n]);
  };
  // db: in the workgroups of the first column tile wave wi sums the wi-th 32 of its 128 columns of g.
  const bool sums = a.db != nullptr && i0 == 0;
  float sum = 0.f;
  uint32_t offs[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    offs[h] = wo * SUB + (wi < 2 ? (wi == 0 ? off.tr[0][h] : off.tr[1][h]) : (wi == 2 ? off.tr[2][h] : off.tr[3][h]));
  const auto add = [&](const lds_char* stage) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {  // 16 rows: two reads of 4 rows a lane half
      const u32x2 v = tr_read(stage + (k >> 1) * (16 * 256), offs[k & 1]);
      sum += (__builtin_bit_cast(float, v[0] << 16) + __builtin_bit_cast(float, v[0] & 0xffff0000u)) +
             (__builtin_bit_cast(float, v[1] << 16) + __builtin_bit_cast(float, v[1] & 0xffff0000u));
    }
  };

  const int steps = (rows + ROWS - 1) / ROWS;
  u32x4 a0[4], b0[2], a1[4], b1[2];
  copy(s0);
  copy(s1);
  copy(s2);
  stage_barrier<8>();  // s0
  read(s0, 0, a0, b0);
  const auto step = [&](lds_char* now, lds_char* next, lds_char* last) {
    // The next stage has landed for every wave, and every wave has read all of the last one, whose
    // place the stage after the two in flight takes.
    stage_barrier<4>();
    copy(last);
    read(now, 1, a1, b1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(a0, b0);
    if (sums) add(now);
    read(next, 0, a0, b0);
    __builtin_amdgcn_sched_barrier(0);
    multiply(a1, b1);
  };
  for (int t = 0;; t += STAGES) {
    step(s0, s1, s3);
    if (t + 1 >= steps) break;
    step(s1, s2, s0);
    if (t + 2 >= steps) break;
    step(s2, s3, s1);
    if (t + 3 >= steps) break;
    step(s3, s0, s2);
    if (t + 4 >= steps) break;
  }
  wait_vmem();  // no copy outlives the workgroup's LDS

  // Columns of a tile past outs or ins hold the next rows' entries: computed, not stored.
  const int j = lane & 31, half = lane >> 5;
  float* part = a.part + ((int64_t)split * a.outs + o0 + 128 * wo) * a.ins + i0 + 64 * wi + j;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    if (o0 + 128 * wo + 32 * m >= a.outs || i0 + 64 * wi >= a.ins) break;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float* p = part + (int64_t)(32 * m + 8 * (r >> 2) + 4 * half + (r & 3)) * a.ins;
      p[0] = acc[m][0][r];
      p[32] = acc[m][1][r];
    }
  }
  if (sums) {
    sum += __shfl_xor(sum, 32);
    if (half == 0 && o0 + 128 * wo + 32 * wi < a.outs)
      a.part[((int64_t)a.splits * a.ins + split) * a.outs + o0 + 128 * wo + 32 * wi + j] = sum;
  }
}

// Sums the partials in the order of the splits: 4 entries a thread, dw's first, then db's.
__global__ void __launch_bounds__(256) wgrad_sum_kernel(WgradArgs a) {
  const int64_t dw4 = (int64_t)a.outs * a.ins / 4;
  int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const float* p = a.part;
  uint16_t* out = (uint16_t*)a.dw;
  int64_t n4 = dw4;
  if (e >= dw4) {
    e -= dw4;
    n4 = a.outs / 4;
    if (a.db == nullptr || e >= n4) return;
    p += (int64_t)a.splits * a.outs * a.ins;
    out = (uint16_t*)a.db;
  }
  f32x4 sum = ((const f32x4*)p)[e];
#pragma unroll 4
  for (int s = 1; s < a.splits; ++s) sum += ((const f32x4*)p)[(int64_t)s * n4 + e];
  uint16_t r[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) r[k] = __builtin_bit_cast(uint16_t, (__bf16)sum[k]);
  ((u32x2*)out)[e] = u32x2{(uint32_t)r[0] | (uint32_t)r[1] << 16, (uint32_t)r[2] | (uint32_t)r[3] << 16};
}

}  // namespace

hipError_t launch_wgrad(const WgradArgs& a, hipStream_t stream) {
  const unsigned tiles = (unsigned)((a.outs + TILE - 1) / TILE) * (unsigned)((a.ins + TILE - 1) / TILE);
  hipLaunchKernelGGL(wgrad_kernel, dim3(tiles * (unsigned)a.splits), dim3(512), 0, stream, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t quads = (int64_t)a.outs * a.ins / 4 + (a.db ? a.outs / 4 : 0);
  hipLaunchKernelGGL(wgrad_sum_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

}  // namespace fwn
