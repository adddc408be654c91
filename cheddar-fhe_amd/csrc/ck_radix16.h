// Radix-16 register butterflies of the transform passes (exact FP64 modular
// products of ck_arith.h, lazy values).
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

}  // namespace ck
