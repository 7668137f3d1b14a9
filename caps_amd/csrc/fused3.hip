// Three Winograd levels of an FP64 product per pass (fused3.h): the operands
// of a level are never written for the next one to read.  Per element of A or
// B the pre pass moves 1 + 316/64 elements where two fused levels and a single
// one move 3.5 + 6.1, the post pass 343/64 + 1 where they move 8.4 + 4.1.
// Bound by HBM: n = 5000 (leaves of 625) 489 us at 4.9 TB/s and 230 us at 5.5
// TB/s, where the two and one took 891 and 534 us; n = 1024 27 us, 47 before.
// The sums are those of ew_ops.h, level by level: the same bits.
#include "ew_ops.h"
#include "fused3.h"

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

// operands (I, j, k) written before (I, 0, 0)
__host__ __device__ constexpr int written_before(int side, int i) {
  int w = 0;
  for (int t = 0; t < i; t++) w += bb_plain(side, t) ? 40 : 49;
  return w;
}

template <int SIDE, int I, int J, int K>
__device__ __forceinline__ void store_k(const double (&w)[4], gdouble *&o, long long step,
                                        unsigned u) {
  if constexpr (!(bb_plain(SIDE, I) && bb_plain(SIDE, J) && bb_plain(SIDE, K))) {
    *at(o, u) = operand<SIDE, K>(w[0], w[1], w[2], w[3]);
    o += step;
  }
  if constexpr (K < 6) store_k<SIDE, I, J, K + 1>(w, o, step, u);
}

template <int SIDE, int I, int J>
__device__ __forceinline__ void store_jk(const double (&v)[4][4], gdouble *&o, long long step,
                                         unsigned u) {
  double w[4];
#pragma unroll
  for (int c = 0; c < 4; c++) w[c] = operand<SIDE, J>(v[0][c], v[1][c], v[2][c], v[3][c]);
  store_k<SIDE, I, J, 0>(w, o, step, u);
  if constexpr (J < 6) store_jk<SIDE, I, J + 1>(v, o, step, u);
}

// level-1 operand I of the position and everything below it
template <int SIDE, int I>
__device__ __forceinline__ void store_i(const double (&x)[4][4][4], gdouble *out, long long step,
                                        unsigned u) {
  double v[4][4];
#pragma unroll
  for (int b = 0; b < 4; b++)
#pragma unroll
    for (int c = 0; c < 4; c++)
      v[b][c] = operand<SIDE, I>(x[0][b][c], x[1][b][c], x[2][b][c], x[3][b][c]);
  gdouble *o = out + written_before(SIDE, I) * step;
  store_jk<SIDE, I, 0>(v, o, step, u);
}

__device__ __forceinline__ void load_quad(gcdouble *in, int a, long long q, unsigned u,
                                          double (&x)[4][4][4]) {
#pragma unroll
  for (int b = 0; b < 4; b++)
#pragma unroll
    for (int c = 0; c < 4; c++) x[a][b][c] = *at(in + (16 * a + 4 * b + c) * q, u);
}

// thread: one position, all of one side
template <int SIDE>
__device__ __forceinline__ void pre_all(gcdouble *in, gdouble *out, long long q, long long step,
                                        unsigned u) {
  double x[4][4][4];
#pragma unroll
  for (int a = 0; a < 4; a++) load_quad(in, a, q, u, x);
  store_i<SIDE, 0>(x, out, step, u);
  store_i<SIDE, 1>(x, out, step, u);
  store_i<SIDE, 2>(x, out, step, u);
  store_i<SIDE, 3>(x, out, step, u);
  store_i<SIDE, 4>(x, out, step, u);
  store_i<SIDE, 5>(x, out, step, u);
  store_i<SIDE, 6>(x, out, step, u);
}

// thread: one position, level-1 operand I of one side (unused quadrants are
// not loaded: their loads are dead)
template <int SIDE, int I>
__device__ __forceinline__ void pre_one(gcdouble *in, gdouble *out, long long q, long long step,
                                        unsigned u) {
  double x[4][4][4];
#pragma unroll
  for (int a = 0; a < 4; a++) load_quad(in, a, q, u, x);
  store_i<SIDE, I>(x, out, step, u);
}

template <int SIDE>
__device__ __forceinline__ void pre_split(gcdouble *in, gdouble *out, long long q,
                                          long long step, unsigned u, int i) {
  switch (i) {
    case 0: pre_one<SIDE, 0>(in, out, q, step, u); break;
    case 1: pre_one<SIDE, 1>(in, out, q, step, u); break;
    case 2: pre_one<SIDE, 2>(in, out, q, step, u); break;
    case 3: pre_one<SIDE, 3>(in, out, q, step, u); break;
    case 4: pre_one<SIDE, 4>(in, out, q, step, u); break;
    case 5: pre_one<SIDE, 5>(in, out, q, step, u); break;
    default: pre_one<SIDE, 6>(in, out, q, step, u); break;
  }
}

// grid.y: side
template <int T>
__global__ __launch_bounds__(T, 2) void b3_pre_kernel(const B3Pre *__restrict__ P, long long q) {
  const unsigned u = 8 * (blockIdx.x * T + threadIdx.x);
  if (u >= 8 * q) return;
  const int side = blockIdx.y;
  gcdouble *in = (gcdouble *)P->in[side];
  gdouble *out = (gdouble *)P->out[side];
  if (side)
    pre_all<1>(in, out, q, P->step, u);
  else
    pre_all<0>(in, out, q, P->step, u);
}

// grid.y: side and level-1 operand
template <int T>
__global__ __launch_bounds__(T) void b3_pre_split_kernel(const B3Pre *__restrict__ P, long long q) {
  const unsigned u = 8 * (blockIdx.x * T + threadIdx.x);
  if (u >= 8 * q) return;
  const int i = blockIdx.y >> 1;
  if (blockIdx.y & 1)
    pre_split<1>((gcdouble *)P->in[1], (gdouble *)P->out[1], q, P->step, u, i);
  else
    pre_split<0>((gcdouble *)P->in[0], (gdouble *)P->out[0], q, P->step, u, i);
}

// the four quadrants (11, 21, 12, 22) of a level from its seven products
__device__ __forceinline__ void combine(const double (&p)[7], double (&c)[4]) {
  Ew<EW_BFS_POST>::apply(p, c);
}

// level-1 product i from the 49 below it
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

// thread: one position; level-1 products in the order that needs the fewest
// of them at a time (C11 = Q1 + Q2, U1 = Q1 + Q4, U2 = U1 + Q5, C21 = U2 - Q7,
// C22 = U2 + Q3, C12 = (U1 + Q3) + Q6)
template <int T>
__global__ __launch_bounds__(T, 2) void b3_post_kernel(const B3Post *__restrict__ P, long long q) {
  const unsigned u = 8 * (blockIdx.x * T + threadIdx.x);
  if (u >= 8 * q) return;
  gcdouble *in = (gcdouble *)P->q;
  gdouble *out = (gdouble *)P->c;
  const long long step = P->step;
  double w[4][4], y[4][4], z[4][4], r[4][4];
  product(in, 0, step, u, w);
  product(in, 1, step, u, y);
  add16(w, y, r);
  store_quad(out, 0, q, u, r);  // C11
  product(in, 3, step, u, y);
  add16(w, y, w);  // U1
  product(in, 4, step, u, y);
  add16(w, y, z);  // U2
  product(in, 6, step, u, y);
  add16(z, y, r, true);
  store_quad(out, 1, q, u, r);  // C21
  product(in, 2, step, u, y);
  add16(z, y, r);
  store_quad(out, 3, q, u, r);  // C22
  add16(w, y, w);               // U3
  product(in, 5, step, u, y);
  add16(w, y, r);
  store_quad(out, 2, q, u, r);  // C12
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

// grid.y: quadrants a, b of C
template <int T>
__global__ __launch_bounds__(T) void b3_post_split_kernel(const B3Post *__restrict__ P,
                                                          long long q) {
  const unsigned u = 8 * (blockIdx.x * T + threadIdx.x);
  if (u >= 8 * q) return;
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
  for (int h = 0; h < 4; h++) *at(out + (16 * a + 4 * b + h) * q, u) = w[h];
}

// The launch shape by the blocks that the positions make.  Blocks of 256 keep
// 2 KB of each of the 380 streams together (n = 5000: 857 us for both passes,
// 1011 with blocks of 64).  Where those leave CUs without a block, blocks of 64
// do not (n = 1536: 64 us against 95 split); below one of them per CU, each
// level-1 operand gets blocks of its own, and each pair of quadrants of C, which
// read 14/4 of the operands and four times the products (n = 392: 14 us, where
// two fused levels and a single one took 26).
template <typename F>
hipError_t by_positions(long long q, F &&launch) {
  if (!b3_fits(q)) return hipErrorInvalidValue;
  const long long cus = device_cu_count();
  const unsigned b256 = (unsigned)((q + 255) / 256), b64 = (unsigned)((q + 63) / 64);
  if (b256 >= cus)
    launch(b256, 256, false);
  else
    launch(b64, 64, b64 < cus);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_b3_pre(const B3Pre *P, long long q, hipStream_t s) {
  return by_positions(q, [&](unsigned gx, int t, bool split) {
    if (split)
      hipLaunchKernelGGL((b3_pre_split_kernel<64>), dim3(gx, 14), dim3(64), 0, s, P, q);
    else if (t == 64)
      hipLaunchKernelGGL((b3_pre_kernel<64>), dim3(gx, 2), dim3(64), 0, s, P, q);
    else
      hipLaunchKernelGGL((b3_pre_kernel<256>), dim3(gx, 2), dim3(256), 0, s, P, q);
  });
}

hipError_t launch_b3_post(const B3Post *P, long long q, hipStream_t s) {
  return by_positions(q, [&](unsigned gx, int t, bool split) {
    if (split)
      hipLaunchKernelGGL((b3_post_split_kernel<64>), dim3(gx, 16), dim3(64), 0, s, P, q);
    else if (t == 64)
      hipLaunchKernelGGL((b3_post_kernel<64>), dim3(gx), dim3(64), 0, s, P, q);
    else
      hipLaunchKernelGGL((b3_post_kernel<256>), dim3(gx), dim3(256), 0, s, P, q);
  });
}

}  // namespace caps
