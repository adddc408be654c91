// Register butterflies of the transform passes (exact FP64 modular products of
// ck_arith.h, lazy values) and the lane transpose between them.
#pragma once

#include "ck_arith.h"

namespace ck {

// forward radix-16 (4 CT stages), element index bits high to low; twiddle
// slot (1 << s) - 1 + blk for sub-stage s
__device__ __forceinline__ void ct16(double x[16], const uint32_t tw[15],
                                     double q, double qr) {
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const int half = 8 >> s;
#pragma unroll
    for (int blk = 0; blk < (1 << s); blk++) {
      const double w = (double)tw[(1 << s) - 1 + blk];
#pragma unroll
      for (int j = 0; j < half; j++) {
        double &a = x[blk * 2 * half + j];
        double &b = x[blk * 2 * half + j + half];
        const double r = mulmod_fq(b, w, q, qr);
        b = a - r;
        a = a + r;
      }
    }
  }
}

// inverse radix-16 (4 GS stages), element index bits low to high; twiddle
// slot 16 - (16 >> u) + blk for sub-stage u
__device__ __forceinline__ void gs16(double x[16], const uint32_t tw[15],
                                     double q, double qr) {
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int half = 1 << u;
#pragma unroll
    for (int blk = 0; blk < (8 >> u); blk++) {
      const double w = (double)tw[16 - (16 >> u) + blk];
#pragma unroll
      for (int j = 0; j < half; j++) {
        double &a = x[blk * 2 * half + j];
        double &b = x[blk * 2 * half + j + half];
        const double d = a - b;
        a = a + b;
        b = mulmod_fq(d, w, q, qr);
      }
    }
  }
}

// Orders a wave's LDS writes before its later reads of other lanes' words: the
// hardware runs one wave's LDS accesses in order, the compiler has to as well.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Keeps the scheduler from moving global loads and stores across this point
// (it sinks prefetches to their use to save registers).
__device__ __forceinline__ void keep_loads() { __builtin_amdgcn_sched_barrier(0x38F); }

// 4 x 4 transpose between the lane groups g = 0..3 and four registers: lane
// group g of register h holds element (g, h) before and (h, g) after.
__device__ __forceinline__ void swap_lanes(int &a, int &b, bool wide) {
  typedef unsigned v2u __attribute__((ext_vector_type(2)));
  const v2u r = wide ? __builtin_amdgcn_permlane32_swap((unsigned)a, (unsigned)b, false, false)
                     : __builtin_amdgcn_permlane16_swap((unsigned)a, (unsigned)b, false, false);
  a = (int)r[0];
  b = (int)r[1];
}
__device__ __forceinline__ void transpose_groups(int &r0, int &r1, int &r2, int &r3) {
  swap_lanes(r0, r2, true);
  swap_lanes(r1, r3, true);
  swap_lanes(r0, r1, false);
  swap_lanes(r2, r3, false);
}
__device__ __forceinline__ void transpose_groups(double x[4]) {
  int lo[4], hi[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    lo[i] = __double2loint(x[i]);
    hi[i] = __double2hiint(x[i]);
  }
  transpose_groups(lo[0], lo[1], lo[2], lo[3]);
  transpose_groups(hi[0], hi[1], hi[2], hi[3]);
#pragma unroll
  for (int i = 0; i < 4; i++) x[i] = __hiloint2double(hi[i], lo[i]);
}

// forward radix-4 (two CT stages, element index bits high to low): twiddles
// wa for the first stage, wb[0..1] for the second
__device__ __forceinline__ void ct4(double x[4], uint32_t wa, const uint32_t wb[2], double q,
                                    double qr) {
  const double a = (double)wa, b0 = (double)wb[0], b1 = (double)wb[1];
  const double r2 = mulmod_fq(x[2], a, q, qr), r3 = mulmod_fq(x[3], a, q, qr);
  const double y0 = x[0] + r2, y2 = x[0] - r2, y1 = x[1] + r3, y3 = x[1] - r3;
  const double s1 = mulmod_fq(y1, b0, q, qr), s3 = mulmod_fq(y3, b1, q, qr);
  x[0] = y0 + s1;
  x[1] = y0 - s1;
  x[2] = y2 + s3;
  x[3] = y2 - s3;
}
// inverse radix-4 (two GS stages, element index bits low to high): twiddles
// wa[0..1] for the first stage, wb for the second
__device__ __forceinline__ void gs4(double x[4], const uint32_t wa[2], uint32_t wb, double q,
                                    double qr) {
  const double a0 = (double)wa[0], a1 = (double)wa[1], b = (double)wb;
  const double y0 = x[0] + x[1], y1 = mulmod_fq(x[0] - x[1], a0, q, qr);
  const double y2 = x[2] + x[3], y3 = mulmod_fq(x[2] - x[3], a1, q, qr);
  x[0] = y0 + y2;
  x[2] = mulmod_fq(y0 - y2, b, q, qr);
  x[1] = y1 + y3;
  x[3] = mulmod_fq(y1 - y3, b, q, qr);
}

}  // namespace ck
