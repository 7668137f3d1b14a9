// Three consecutive batched Winograd levels of an FP64 product in single
// passes (fused3.hip).  Sub-block (a, b, c) of a matrix, a, b, c quadrants of
// the three levels, lies at element (16 a + 4 b + c) * q; operand (i, j, k) is
// plain iff i, j and k are (bb_plain).
#pragma once
#include "fused2.h"

namespace caps {

// pre-additions of three 'b' levels for both operands of one sub-problem
struct B3Pre {
  const double *in[2];  // A (side 0) and B (side 1): 64 sub-blocks of q elements
  double *out[2];       // the 316 operands that are not plain, in (i, j, k) order
  long long step;       // elements from one operand to the next
};

// post-combinations of three 'b' levels of one sub-problem
struct B3Post {
  const double *q;  // product (i, j, k) at (49 i + 7 j + k) * step
  long long step;
  double *c;        // C's 64 sub-blocks
};

constexpr int B3_WRITTEN = 343 - 27;

// operands and products lie on whole 128-byte lines (none has two writers), an
// odd number of them apart (a power of two puts a position of all 343 on a few
// memory channels)
inline long long b3_step(long long q) { return ((q + 15) / 16 | 1) * 16; }
// 32-bit offsets within an operand
inline bool b3_fits(long long q) { return q > 0 && q < (1LL << 28); }
hipError_t launch_b3_pre(const B3Pre *d_P, long long q, hipStream_t s);
hipError_t launch_b3_post(const B3Post *d_P, long long q, hipStream_t s);

}  // namespace caps
