// One to three consecutive batched Winograd levels of an FP64 product in single
// passes (fused_f64.hip).  With L levels a matrix has 4^L sub-blocks of q
// elements, numbered by their quadrants from the outermost level on ((a, b) at
// (4 a + b) * q, (a, b, c) at (16 a + 4 b + c) * q), and 7^L operands a side,
// numbered (i, j(, k)) in the same way.  An operand is plain, a sub-block
// itself, iff all its level operands are (bb_plain).
#pragma once
#include "fused2.h"

namespace caps {

// pre-additions for both operands of one sub-problem
struct FusedPre {
  const double *in[2];  // A (side 0) and B (side 1)
  double *out[2];       // the operands that are not plain (bs != 0: all), in order
  long long step;       // elements from one operand to the next
  int m, bs;            // bs != 0: sub-blocks of m x m leaves in bs x bs blocks, operands
                        // with column-major leaves
};

// post-combinations of one sub-problem
struct FusedPost {
  const double *q;  // product t at t * step
  long long step;
  double *c;
  int m, bs;        // as in FusedPre: products column-major, C blocked
};

constexpr int fused_products(int levels) { return levels == 1 ? 7 : (levels == 2 ? 49 : 343); }
constexpr int fused_written(int levels, bool all) {
  return fused_products(levels) - (all ? 0 : (levels == 1 ? 3 : (levels == 2 ? 9 : 27)));
}

// operands and products lie on whole 128-byte lines (none has two writers), an
// odd number of them apart (a power of two puts a position of all 343 on a few
// memory channels)
inline long long fused_step(long long q) { return ((q + 15) / 16 | 1) * 16; }
// 32-bit offsets within an operand
inline bool fused_fits(long long q) { return q > 0 && q < (1LL << 28); }
hipError_t launch_fused_pre(const FusedPre *d_P, int levels, long long q, bool blocked,
                            hipStream_t s);
hipError_t launch_fused_post(const FusedPost *d_P, int levels, long long q, bool blocked,
                             hipStream_t s);

}  // namespace caps
