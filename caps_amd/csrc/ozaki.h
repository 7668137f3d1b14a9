// Split-precision leaf product (Ozaki scheme II: integer modular emulation of
// an FP64 GEMM; K. Ozaki, Y. Uchino, T. Imamura, "Ozaki Scheme II: A
// GEMM-oriented emulation of floating-point matrix multiplication using an
// integer modular technique", 2025).  No counterpart in the reference, whose
// leaf is a BLAS dgemm (dgemm-blas.cpp:4-13).
//
// For a leaf product C = A * B (m x m, column-major FP64):
//  1. scale: row i of A by 2^sa_i, column j of B by 2^sb_j, powers of two
//     chosen from deterministic 2-norm upper bounds so that
//        sum_k |A'_ik| |B'_kj| <= ||A'_i.|| ||B'_.j|| <= L^2 < M / 2,
//     with A' = trunc(2^sa A), B' = trunc(2^sb B) (exact FP64 integers) and
//     M the product of the moduli;
//  2. split: A' mod m_l and B' mod m_l as symmetric residues (INT8 planes),
//     A-side planes row-major (k contiguous), B-side column-major;
//  3. product: C'_l = A'_l B'_l on the INT8 matrix cores with exact INT32
//     accumulation, reduced mod m_l in the epilogue (INT8 output plane);
//  4. reconstruct: X = sum_l C'_l W_l  (mod M) by the Chinese remainder
//     theorem in FP64 with the weights W_l split into 37-bit pieces, so every
//     partial sum is exact; X = A'B' exactly (assembled in 128 bits), returned
//     correctly rounded to FP64, then C = 2^-(sa_i + sb_j) X.
// Integer-valued leaves whose products fit 53 bits come out exact.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"

namespace caps {

constexpr int OZ_MAX_MODULI = 16;  // M <= 2^128: X fits 128 bits
constexpr int OZ_MAX_PIECES = 4;
constexpr int OZ_PIECE_BITS = 37;
constexpr int OZ_DEFAULT_MODULI = 14;
// row / column chunks of the deterministic sum-of-squares reduction
constexpr int OZ_CHUNKS = 8;

struct OzakiConsts {
  int nmod;
  int npieces;
  int m[OZ_MAX_MODULI];
  unsigned dot16[OZ_MAX_MODULI];           // 1 | (2^16 mod m_l) << 16: halves of a sum (residue_of_sum)
  int bias[OZ_MAX_MODULI];                 // least multiple of m_l >= 2^28: keeps sums positive
  int c22[OZ_MAX_MODULI];                  // round(2^22 / m_l): quotients of small sums (mod_k)
  double inv_m[OZ_MAX_MODULI];
  double w[OZ_MAX_MODULI][OZ_MAX_PIECES];  // CRT weight W_l in base 2^37 digits
  double Mp[OZ_MAX_PIECES];                // M in base 2^37 digits
  double invM;                             // 1 / M (rounded)
  double L;                                // per-side norm bound, L^2 < M/2
  double log2M;
};

// Residue planes store a leaf of order m0 with rows (A side) or columns (B and
// C side) at a pitch of residue_pitch(m0) bytes, of which the first
// residue_k(m0) hold residues, zero past m0: 16-byte chunks are aligned and
// wholly inside or outside for every leaf size, so no kernel reads residues
// byte by byte, and zero k positions add nothing to a product.  Bytes past
// residue_k, and past the rows in residue_area, are never part of a result.
//
// The pitch is the largest of the multiples of 128, 64, 32 and 16 that adds at
// most 1/32, and a leaf fills whole 128-byte lines where that adds at most
// 1/32: rows and planes that straddle lines cost the leaf GEMM and the passes
// more than the padding.  Leaves of 750 (n = 3000, r = 2) at a pitch of 752:
// 0.53 ms in the GEMM, 0.22 in B's split.
__host__ __device__ constexpr int residue_k(int m0) { return (m0 + 15) & ~15; }
__host__ __device__ constexpr int residue_pitch(int m0) {
  for (int a = 128; a > 16; a /= 2) {
    const int p = (m0 + a - 1) / a * a;
    if (32LL * p <= 33LL * m0) return p;
  }
  return residue_k(m0);
}
__host__ __device__ constexpr long long residue_area(int m0) {
  const long long a = (long long)m0 * residue_pitch(m0);
  return a >= 4096 ? (a + 127) / 128 * 128 : a;
}

struct OzLeaf {
  const double *A;  // m x m column-major
  const double *B;
  double *C;
  int *ea;          // m row exponents of A
  int *eb;          // m column exponents of B
  int8_t *ra;       // nmod planes of residue_area(m), row-major leaf
  int8_t *rb;       // nmod planes, column-major
  int8_t *rc;       // nmod planes, column-major (product residues)
  double *pa;       // OZ_CHUNKS x m partial row sums of squares (A)
  double *pb;       // m column sums of squares (B)
};

// One leaf product of the INT8 GEMM step: nmod residue planes per operand,
// plane l of an operand at base + l * stride (bytes).  a: row-major leaves
// (k contiguous), b and c: column-major, all of residue_pitch.  Element e of C's plane l sits
// at c + l * sc + (e >> 7) * cseg + (e & 127): cseg = 128 is the plain plane;
// a larger cseg interleaves the 128-byte segments of several products (the
// 256-tile kernels only: residue_gemm_segmented says which launches take them).
struct RGemm {
  const int8_t *a;
  const int8_t *b;
  int8_t *c;
  long long sa, sb, sc;
  long long cseg;
};

// Host: moduli and CRT constants for nmod moduli (2..OZ_MAX_MODULI).
// Returns false if nmod is out of range.
bool ozaki_make_consts(int nmod, OzakiConsts &k);

// The moduli used (greedy pairwise-coprime, descending from 256).
const int *ozaki_moduli_table();

// Number of 37-bit pieces of M for nmod moduli.
int ozaki_npieces(int nmod);

// step: 0 = scale, 1 = split, 3 = reconstruct (OzLeaf tables)
hipError_t launch_ozaki_step(int step, const OzLeaf *d_tab, int count, int m, int nmod,
                             const OzakiConsts *d_consts, hipStream_t s);

// C_l = A_l B_l (mod m_l) for every leaf of the table and every modulus, one
// persistent launch.  Operands are m x m quadtrees of `levels` quadrant levels
// over leaves of size m >> levels (A leaves row-major, B and C column-major);
// levels > 0 needs leaves that are multiples of 128.
// the same products on BF16 MFMA with FP32 accumulation (bit-identical results)
hipError_t launch_residue_gemm_bf16(const RGemm *d_tab, int count, int m, int levels, int nmod,
                                    const OzakiConsts *d_consts, hipStream_t s);
// The block tile of `problems` INT8 products (leaves x moduli) of order m: 256
// (the large-tile kernel) or 64..192, by residue_tile_cost's estimate of a
// launch of `tiles` tiles over K.
int residue_block_tile(int m, int levels, int tile, long long problems);
double residue_tile_cost(int bt, double tiles, int K);
// launch_residue_gemm (INT8) / launch_residue_gemm_bf16 (bf16) runs these
// leaves on the 256-tile kernel for whole tiles, which honours RGemm::cseg
bool residue_gemm_segmented(int m, int levels, int tile, bool bf16, long long problems);
// INT8 products over segments of different sizes in one persistent launch
// (kernels.h VSeg: args are RGemm tables, n = order, gx = tiles per dimension,
// gy = leaves x moduli, aux = quadtree levels), block tile bt < 256
hipError_t launch_residue_gemm_multi(int bt, const char *d_tables, const VSeg *d_segs, int nseg,
                                     int total_tiles, int nmod, const OzakiConsts *d_consts,
                                     hipStream_t s);
// tile: 0 = the block tile of residue_block_tile, 1 = the same below 256
hipError_t launch_residue_gemm(const RGemm *d_tab, int count, int m, int levels, int nmod,
                               const OzakiConsts *d_consts, hipStream_t s, int tile = 0);

}  // namespace caps
