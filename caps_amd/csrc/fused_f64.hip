// One to three Winograd levels of an FP64 product per pass (fused_f64.h): the
// operands of a level are never written for the next one to read.  Per element
// of A or B a pass over three levels moves 1 + 316/64 elements where passes over
// two and one move 3.5 + 6.1, and back 343/64 + 1 where those move 8.4 + 4.1.
// Bound by HBM: n = 5000 (leaves of 625) 489 us at 4.9 TB/s and 230 us at 5.5
// TB/s, where the two and one took 891 and 534 us; n = 1024 27 us, 47 before.
// The sums are those of ew_ops.h, level by level: the same bits.
//
// Leaves in bs x bs blocks are made column-major on the way (the pre pass writes
// all operands then) and C is put back into blocks: the passes work position by
// position, so a thread takes one column-major position and moves the blocked
// side at its permuted place.
#include "ew_ops.h"
#include "fused_f64.h"
#include "ozaki_dev.h"

namespace caps {

namespace {

// global-memory views (accesses through them are global_*, not flat_*)
typedef __attribute__((address_space(1))) double gdouble;
typedef const __attribute__((address_space(1))) double gcdouble;

// element of a thread at byte offset u (32 bits: scalar base, no 64-bit vector
// arithmetic)
__device__ __forceinline__ gcdouble *at(gcdouble *p, unsigned u) {
  return (gcdouble *)((const __attribute__((address_space(1))) char *)p + u);
}
__device__ __forceinline__ gdouble *at(gdouble *p, unsigned u) {
  return (gdouble *)((__attribute__((address_space(1))) char *)p + u);
}

// operand I of a level from its four quadrants (11, 21, 12, 22): T1..T7 for
// SIDE 0, S1..S7 for SIDE 1, the expression trees of Ew<EW_BFS_PRE>.  A shared
// sub-expression (T3, S3) is formed again for each operand: the passes have
// additions to spare and no registers.
template <int SIDE, int I>
__device__ __forceinline__ double operand(double q0, double q1, double q2, double q3) {
  if constexpr (SIDE == 0) {
    if constexpr (I == 0) return q0;
    if constexpr (I == 1) return q2;
    if constexpr (I == 2) return q1 + q3;
    if constexpr (I == 3) return (q1 + q3) - q0;
    if constexpr (I == 4) return q0 - q1;
    if constexpr (I == 5) return q2 - ((q1 + q3) - q0);
    return q3;
  } else {
    if constexpr (I == 0) return q0;
    if constexpr (I == 1) return q1;
    if constexpr (I == 2) return q2 - q0;
    if constexpr (I == 3) return q3 - (q2 - q0);
    if constexpr (I == 4) return q3 - q2;
    if constexpr (I == 5) return q3;
    return (q3 - (q2 - q0)) - q1;
  }
}

// The operands (J, K) of two levels from the values v at sub-positions (b, c),
// on from o; without the plain ones if PLAIN (the levels above are plain and
// nothing is permuted).
template <int SIDE, bool PLAIN, int J, int K>
__device__ __forceinline__ void store_k(const double (&w)[4], gdouble *&o, long long step,
                                        unsigned u) {
  if constexpr (!(PLAIN && bb_plain(SIDE, J) && bb_plain(SIDE, K))) {
    *at(o, u) = operand<SIDE, K>(w[0], w[1], w[2], w[3]);
    o += step;
  }
  if constexpr (K < 6) store_k<SIDE, PLAIN, J, K + 1>(w, o, step, u);
}

template <int SIDE, bool PLAIN, int J>
__device__ __forceinline__ void store_jk(const double (&v)[4][4], gdouble *&o, long long step,
                                         unsigned u) {
  double w[4];
#pragma unroll
  for (int c = 0; c < 4; c++) w[c] = operand<SIDE, J>(v[0][c], v[1][c], v[2][c], v[3][c]);
  store_k<SIDE, PLAIN, J, 0>(w, o, step, u);
  if constexpr (J < 6) store_jk<SIDE, PLAIN, J + 1>(v, o, step, u);
}

// operands (I, j, k) written before (I, 0, 0)
__host__ __device__ constexpr int written_before(int side, int i, bool all) {
  int w = 0;
  for (int t = 0; t < i; t++) w += !all && bb_plain(side, t) ? 40 : 49;
  return w;
}

// three levels: level-1 operand I of the position and everything below it
template <int SIDE, int I, bool ALL>
__device__ __forceinline__ void store_i(const double (&x)[4][4][4], gdouble *out, long long step,
                                        unsigned u) {
  double v[4][4];
#pragma unroll
  for (int b = 0; b < 4; b++)
#pragma unroll
    for (int c = 0; c < 4; c++)
      v[b][c] = operand<SIDE, I>(x[0][b][c], x[1][b][c], x[2][b][c], x[3][b][c]);
  gdouble *o = out + written_before(SIDE, I, ALL) * step;
  store_jk<SIDE, !ALL && bb_plain(SIDE, I), 0>(v, o, step, u);
}

__device__ __forceinline__ void load_quad(gcdouble *in, int a, long long q, unsigned u,
                                          double (&x)[4][4]) {
#pragma unroll
  for (int b = 0; b < 4; b++)
#pragma unroll
    for (int c = 0; c < 4; c++) x[b][c] = *at(in + (16 * a + 4 * b + c) * q, u);
}

// byte offset of column-major position p (of leaves m x m) in blocked leaves
__device__ __forceinline__ unsigned blocked_offset(unsigned p, int m, int bs) {
  const unsigned mm = (unsigned)m * m, leaf = p / mm, e = p - leaf * mm;
  const unsigned j = e / m, i = e - j * m;
  return 8 * (leaf * mm + (unsigned)leaf_elem_offset(m, bs, (int)i, (int)j));
}

// thread: one position (read at u0, written at u), all of one side
template <int SIDE, int LEVELS, bool ALL>
__device__ __forceinline__ void pre_all(gcdouble *in, gdouble *out, long long q, long long step,
                                        unsigned u0, unsigned u) {
  if constexpr (LEVELS == 1) {
    double x[4];
#pragma unroll
    for (int a = 0; a < 4; a++) x[a] = *at(in + a * q, u0);
    store_k<SIDE, !ALL, 0, 0>(x, out, step, u);
  } else if constexpr (LEVELS == 2) {
    double x[4][4];
    load_quad(in, 0, q, u0, x);
    store_jk<SIDE, !ALL, 0>(x, out, step, u);
  } else {
    double x[4][4][4];
#pragma unroll
    for (int a = 0; a < 4; a++) load_quad(in, a, q, u0, x[a]);
    store_i<SIDE, 0, ALL>(x, out, step, u);
    store_i<SIDE, 1, ALL>(x, out, step, u);
    store_i<SIDE, 2, ALL>(x, out, step, u);
    store_i<SIDE, 3, ALL>(x, out, step, u);
    store_i<SIDE, 4, ALL>(x, out, step, u);
    store_i<SIDE, 5, ALL>(x, out, step, u);
    store_i<SIDE, 6, ALL>(x, out, step, u);
  }
}

// three levels, thread: one position, level-1 operand I of one side (quadrants
// it does not need are not loaded: their loads are dead)
template <int SIDE, int I, bool ALL>
__device__ __forceinline__ void pre_one(gcdouble *in, gdouble *out, long long q, long long step,
                                        unsigned u0, unsigned u) {
  double x[4][4][4];
#pragma unroll
  for (int a = 0; a < 4; a++) load_quad(in, a, q, u0, x[a]);
  store_i<SIDE, I, ALL>(x, out, step, u);
}

template <int SIDE, bool ALL>
__device__ __forceinline__ void pre_split(gcdouble *in, gdouble *out, long long q,
                                          long long step, unsigned u0, unsigned u, int i) {
  switch (i) {
    case 0: pre_one<SIDE, 0, ALL>(in, out, q, step, u0, u); break;
    case 1: pre_one<SIDE, 1, ALL>(in, out, q, step, u0, u); break;
    case 2: pre_one<SIDE, 2, ALL>(in, out, q, step, u0, u); break;
    case 3: pre_one<SIDE, 3, ALL>(in, out, q, step, u0, u); break;
    case 4: pre_one<SIDE, 4, ALL>(in, out, q, step, u0, u); break;
    case 5: pre_one<SIDE, 5, ALL>(in, out, q, step, u0, u); break;
    default: pre_one<SIDE, 6, ALL>(in, out, q, step, u0, u); break;
  }
}

// grid.y: side.  ALL: blocked leaves, all operands written
template <int T, int LEVELS, bool ALL>
__global__ __launch_bounds__(T, 2) void fused_pre_kernel(const FusedPre *__restrict__ P,
                                                         long long q) {
  const unsigned p = blockIdx.x * T + threadIdx.x;
  if (p >= q) return;
  const unsigned u = 8 * p, u0 = ALL ? blocked_offset(p, P->m, P->bs) : u;
  const int side = blockIdx.y;
  gcdouble *in = (gcdouble *)P->in[side];
  gdouble *out = (gdouble *)P->out[side];
  if (side)
    pre_all<1, LEVELS, ALL>(in, out, q, P->step, u0, u);
  else
    pre_all<0, LEVELS, ALL>(in, out, q, P->step, u0, u);
}

// three levels, grid.y: side and level-1 operand
template <int T, bool ALL>
__global__ __launch_bounds__(T) void fused_pre_split_kernel(const FusedPre *__restrict__ P,
                                                            long long q) {
  const unsigned p = blockIdx.x * T + threadIdx.x;
  if (p >= q) return;
  const unsigned u = 8 * p, u0 = ALL ? blocked_offset(p, P->m, P->bs) : u;
  const int i = blockIdx.y >> 1;
  if (blockIdx.y & 1)
    pre_split<1, ALL>((gcdouble *)P->in[1], (gdouble *)P->out[1], q, P->step, u0, u, i);
  else
    pre_split<0, ALL>((gcdouble *)P->in[0], (gdouble *)P->out[0], q, P->step, u0, u, i);
}

// the four quadrants (11, 21, 12, 22) of a level from its seven products
__device__ __forceinline__ void combine(const double (&p)[7], double (&c)[4]) {
  Ew<EW_BFS_POST>::apply(p, c);
}

// the 16 sub-positions of two levels from their 49 products (49 i on: those of
// level-1 product i)
__device__ __forceinline__ void product(gcdouble *in, int i, long long step, unsigned u,
                                        double (&y)[4][4]) {
  double v[7][7], l2[7][4];
  gcdouble *p = in + 49 * i * step;
  // all loads before the first use: the scheduler would wait after every few
  // (n = 1024: 24.8 -> 11 us)
#pragma unroll
  for (int t = 0; t < 49; t++) v[t / 7][t % 7] = __builtin_nontemporal_load(at(p + t * step, u));
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < 7; j++) combine(v[j], l2[j]);
#pragma unroll
  for (int c = 0; c < 4; c++) {
    double p2[7], o[4];
#pragma unroll
    for (int j = 0; j < 7; j++) p2[j] = l2[j][c];
    combine(p2, o);
#pragma unroll
    for (int b = 0; b < 4; b++) y[b][c] = o[b];
  }
}

__device__ __forceinline__ void store_quad(gdouble *out, int a, long long q, unsigned u,
                                           const double (&y)[4][4]) {
#pragma unroll
  for (int b = 0; b < 4; b++)
#pragma unroll
    for (int c = 0; c < 4; c++) *at(out + (16 * a + 4 * b + c) * q, u) = y[b][c];
}

// z = x + y, z = x - y over the 16 sub-positions
__device__ __forceinline__ void add16(const double (&x)[4][4], const double (&y)[4][4],
                                      double (&z)[4][4], bool minus = false) {
#pragma unroll
  for (int b = 0; b < 4; b++)
#pragma unroll
    for (int c = 0; c < 4; c++) z[b][c] = minus ? x[b][c] - y[b][c] : x[b][c] + y[b][c];
}

// thread: one position (read at u, written at u0); three levels: level-1
// products in the order that needs the fewest of them at a time (C11 = Q1 + Q2,
// U1 = Q1 + Q4, U2 = U1 + Q5, C21 = U2 - Q7, C22 = U2 + Q3, C12 = (U1 + Q3) +
// Q6)
template <int T, int LEVELS, bool BLOCKED>
__global__ __launch_bounds__(T, 2) void fused_post_kernel(const FusedPost *__restrict__ P,
                                                          long long q) {
  const unsigned p = blockIdx.x * T + threadIdx.x;
  if (p >= q) return;
  const unsigned u = 8 * p, u0 = BLOCKED ? blocked_offset(p, P->m, P->bs) : u;
  gcdouble *in = (gcdouble *)P->q;
  gdouble *out = (gdouble *)P->c;
  const long long step = P->step;
  if constexpr (LEVELS == 1) {
    double v[7], c[4];
#pragma unroll
    for (int k = 0; k < 7; k++) v[k] = __builtin_nontemporal_load(at(in + k * step, u));
    combine(v, c);
#pragma unroll
    for (int a = 0; a < 4; a++) *at(out + a * q, u0) = c[a];
    return;
  }
  double w[4][4], y[4][4], z[4][4], r[4][4];
  product(in, 0, step, u, w);
  if constexpr (LEVELS == 2) {
    store_quad(out, 0, q, u0, w);
    return;
  }
  product(in, 1, step, u, y);
  add16(w, y, r);
  store_quad(out, 0, q, u0, r);  // C11
  product(in, 3, step, u, y);
  add16(w, y, w);  // U1
  product(in, 4, step, u, y);
  add16(w, y, z);  // U2
  product(in, 6, step, u, y);
  add16(z, y, r, true);
  store_quad(out, 1, q, u0, r);  // C21
  product(in, 2, step, u, y);
  add16(z, y, r);
  store_quad(out, 3, q, u0, r);  // C22
  add16(w, y, w);                // U3
  product(in, 5, step, u, y);
  add16(w, y, r);
  store_quad(out, 2, q, u0, r);  // C12
}

// the seven products' sum for quadrant a (0 = 11, 1 = 21, 2 = 12, 3 = 22), term
// by term: quadrant a has terms(a) products, the t-th is term(a, t)
__device__ __forceinline__ int terms(int a) { return a == 0 ? 2 : 4; }
__device__ __forceinline__ int term(int a, int t) {
  if (t == 0) return 0;
  if (t == 1) return a == 0 ? 1 : 3;
  if (t == 2) return a == 2 ? 2 : 4;
  return a == 1 ? 6 : (a == 2 ? 5 : 2);
}

// the sub-positions c of quadrant b of level-1 product i
__device__ __forceinline__ void product_quad(gcdouble *in, int i, int b, long long step,
                                             unsigned u, double (&y)[4]) {
  for (int t = 0; t < terms(b); t++) {
    gcdouble *p = in + (49 * i + 7 * term(b, t)) * step;
    double v[7], c[4];
#pragma unroll
    for (int k = 0; k < 7; k++) v[k] = *at(p + k * step, u);
    combine(v, c);
    const bool minus = b == 1 && t == 3;
#pragma unroll
    for (int h = 0; h < 4; h++) y[h] = t == 0 ? c[h] : (minus ? y[h] - c[h] : y[h] + c[h]);
  }
}

// three levels, grid.y: quadrants a, b of C
template <int T, bool BLOCKED>
__global__ __launch_bounds__(T) void fused_post_split_kernel(const FusedPost *__restrict__ P,
                                                             long long q) {
  const unsigned p = blockIdx.x * T + threadIdx.x;
  if (p >= q) return;
  const unsigned u = 8 * p, u0 = BLOCKED ? blocked_offset(p, P->m, P->bs) : u;
  const int a = blockIdx.y >> 2, b = blockIdx.y & 3;
  gcdouble *in = (gcdouble *)P->q;
  gdouble *out = (gdouble *)P->c;
  double w[4];
  for (int t = 0; t < terms(a); t++) {
    double y[4];
    product_quad(in, term(a, t), b, P->step, u, y);
    const bool minus = a == 1 && t == 3;
#pragma unroll
    for (int h = 0; h < 4; h++) w[h] = t == 0 ? y[h] : (minus ? w[h] - y[h] : w[h] + y[h]);
  }
#pragma unroll
  for (int h = 0; h < 4; h++) *at(out + (16 * a + 4 * b + h) * q, u0) = w[h];
}

// The launch shape by the blocks that the positions make.  Blocks of 256 keep
// 2 KB of each of the 380 streams together (n = 5000: 857 us for both passes,
// 1011 with blocks of 64).  Where those leave CUs without a block, blocks of 64
// do not (n = 1536: 64 us against 95 split); below one of them per CU, each
// level-1 operand gets blocks of its own, and each pair of quadrants of C, which
// read 14/4 of the operands and four times the products (n = 392: 14 us, where
// two fused levels and a single one took 26).
template <int LEVELS, bool ALL>
hipError_t launch_pre(const FusedPre *P, long long q, hipStream_t s) {
  const long long cus = device_cu_count();
  const unsigned b256 = (unsigned)((q + 255) / 256), b64 = (unsigned)((q + 63) / 64);
  if (b256 >= cus)
    hipLaunchKernelGGL((fused_pre_kernel<256, LEVELS, ALL>), dim3(b256, 2), dim3(256), 0, s, P, q);
  else if (LEVELS < 3 || b64 >= cus)
    hipLaunchKernelGGL((fused_pre_kernel<64, LEVELS, ALL>), dim3(b64, 2), dim3(64), 0, s, P, q);
  else
    hipLaunchKernelGGL((fused_pre_split_kernel<64, ALL>), dim3(b64, 14), dim3(64), 0, s, P, q);
  return hipGetLastError();
}

template <int LEVELS, bool BLOCKED>
hipError_t launch_post(const FusedPost *P, long long q, hipStream_t s) {
  const long long cus = device_cu_count();
  const unsigned b256 = (unsigned)((q + 255) / 256), b64 = (unsigned)((q + 63) / 64);
  if (b256 >= cus)
    hipLaunchKernelGGL((fused_post_kernel<256, LEVELS, BLOCKED>), dim3(b256), dim3(256), 0, s, P,
                       q);
  else if (LEVELS < 3 || b64 >= cus)
    hipLaunchKernelGGL((fused_post_kernel<64, LEVELS, BLOCKED>), dim3(b64), dim3(64), 0, s, P, q);
  else
    hipLaunchKernelGGL((fused_post_split_kernel<64, BLOCKED>), dim3(b64, 16), dim3(64), 0, s, P,
                       q);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_fused_pre(const FusedPre *P, int levels, long long q, bool blocked,
                            hipStream_t s) {
  if (!fused_fits(q) || levels < 1 || levels > 3) return hipErrorInvalidValue;
  if (levels == 1) return blocked ? launch_pre<1, true>(P, q, s) : launch_pre<1, false>(P, q, s);
  if (levels == 2) return blocked ? launch_pre<2, true>(P, q, s) : launch_pre<2, false>(P, q, s);
  return blocked ? launch_pre<3, true>(P, q, s) : launch_pre<3, false>(P, q, s);
}

hipError_t launch_fused_post(const FusedPost *P, int levels, long long q, bool blocked,
                             hipStream_t s) {
  if (!fused_fits(q) || levels < 1 || levels > 3) return hipErrorInvalidValue;
  if (levels == 1) return blocked ? launch_post<1, true>(P, q, s) : launch_post<1, false>(P, q, s);
  if (levels == 2) return blocked ? launch_post<2, true>(P, q, s) : launch_post<2, false>(P, q, s);
  return blocked ? launch_post<3, true>(P, q, s) : launch_post<3, false>(P, q, s);
}

}  // namespace caps
