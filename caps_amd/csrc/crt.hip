// Kernels of the residue-domain Strassen (crt.h): scale, split, residue
// Winograd steps and the final CRT reconstruction.  All HBM-bound.
#include "crt.h"
#include "ew_ops.h"
#include "kernels.h"
#include "ozaki_dev.h"

namespace caps {

namespace {

constexpr int T = 256;

// ------------------------------------------------------------------ scale
// partials (e, s) of 64 rows of A over chunk by of a leaf column block: lane =
// row, each of the 4 waves takes a quarter of the chunk's columns, wave 0
// merges them (in wave order).  Bound by the read of A where the blocks fill
// the device (n = 8192: 5.8 TB/s with the columns of B); a thread per row made
// 20 blocks at n = 1280, each a chain of 40 loads: 37 -> 8.8 us (n = 3000:
// 75 -> 36) for the rows of A and the columns of B together.
// PLAIN: column-major leaves (bs == 1 or bs == m), 8 columns per step.
typedef double2 RowLds[T / 64][64];

template <bool PLAIN>
__device__ __forceinline__ void rowpart_body(const CrtMats *__restrict__ M, int bx, int by,
                                             RowLds &P) {
  const int n = M->n, m = M->m, nrec = M->nrec, bs = M->bs, ch = M->chunks;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int row = bx * 64 + lane, i = min(row, n - 1);
  const int c = by;  // bj * chunks + k
  const int bj = c / ch, k = (c - bj * ch) * (T / 64) + wv;
  const int per = (m + ch * (T / 64) - 1) / (ch * (T / 64));
  const int lj0 = min(m, k * per), lj1 = min(m, lj0 + per);
  int e = NOSCALE;
  double s = 0.0;
  if (PLAIN) {
    const double *base = M->A + caps_elem_offset(n, nrec, bs, i, bj * m);  // (i, bj m)
    int lj = lj0;
    for (; lj + 8 <= lj1; lj += 8) {
      double v[8];
#pragma unroll
      for (int t = 0; t < 8; t++) v[t] = base[(long long)(lj + t) * m];
      int e8;
      double s8;
      sq_block8(v, e8, s8);
      sq_merge(e, s, e8, s8);
    }
    for (; lj < lj1; lj++) sq_acc(base[(long long)lj * m], e, s);
  } else {
    for (int lj = lj0; lj < lj1; lj++)
      sq_acc(M->A[caps_elem_offset(n, nrec, bs, i, bj * m + lj)], e, s);
  }
  P[wv][lane] = make_double2(s, (double)e);
  __syncthreads();
  if (wv == 0 && row < n) {
#pragma unroll
    for (int w = 1; w < T / 64; w++) sq_merge(e, s, (int)P[w][lane].y, P[w][lane].x);
    reinterpret_cast<double2 *>(M->pa)[(long long)c * n + i] = make_double2(s, (double)e);
  }
}

// partial of column j of B over leaf row block bi: one wave, fixed butterfly.
// PLAIN: column-major leaves, each lane takes 8 rows (stride 64) per step.
template <bool PLAIN>
__device__ __forceinline__ void colpart_body(const CrtMats *__restrict__ M, int bx) {
  const int n = M->n, m = M->m, nrec = M->nrec, bs = M->bs;
  const long long w = (long long)bx * (T / 64) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int nblk = 1 << nrec;
  if (w >= (long long)n * nblk) return;
  const int j = (int)(w % n), bi = (int)(w / n);
  int e = NOSCALE;
  double s = 0.0;
  if (PLAIN) {
    const double *col = M->B + caps_elem_offset(n, nrec, bs, bi * m, j);  // (bi m, j)
    int li = lane;
    for (; li + 7 * 64 < m; li += 8 * 64) {
      double v[8];
#pragma unroll
      for (int t = 0; t < 8; t++) v[t] = col[li + 64 * t];
      int e8;
      double s8;
      sq_block8(v, e8, s8);
      sq_merge(e, s, e8, s8);
    }
    for (; li < m; li += 64) sq_acc(col[li], e, s);
  } else {
    for (int li = lane; li < m; li += 64)
      sq_acc(M->B[caps_elem_offset(n, nrec, bs, bi * m + li, j)], e, s);
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    int e2 = __shfl_down(e, off, 64);
    double s2 = __shfl_down(s, off, 64);
    if (lane < off) sq_merge(e, s, e2, s2);
  }
  if (lane == 0) reinterpret_cast<double2 *>(M->pb)[(long long)bi * n + j] = make_double2(s, (double)e);
}

// row partials of A (the first blocks: x over the rows, then the chunks) and
// column partials of B in one launch: together they fill the device sooner
template <bool PLAIN>
__device__ __forceinline__ void partials_body(const CrtMats *__restrict__ M, int bx, RowLds &P) {
  const int gx = (M->n + 63) / 64, rows = gx * (M->chunks << M->nrec);
  if (bx < rows)
    rowpart_body<PLAIN>(M, bx % gx, bx / gx, P);
  else
    colpart_body<PLAIN>(M, bx - rows);
}

template <bool PLAIN>
__global__ __launch_bounds__(T) void crt_partials_kernel(const CrtMats *__restrict__ M) {
  __shared__ RowLds P;
  partials_body<PLAIN>(M, blockIdx.x, P);
}

// merges `count` partials, one every n; 4 loads in flight
__device__ __forceinline__ int merged_exponent(const double2 *p, int count, int n, double L) {
  int e = NOSCALE;
  double s = 0.0;
  int c = 0;
  for (; c + 4 <= count; c += 4) {
    double2 v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = p[(long long)(c + k) * n];
#pragma unroll
    for (int k = 0; k < 4; k++) sq_merge(e, s, (int)v[k].y, v[k].x);
  }
  for (; c < count; c++) {
    const double2 v = p[(long long)c * n];
    sq_merge(e, s, (int)v.y, v.x);
  }
  return scale_exponent(e, s, L);
}

__device__ __forceinline__ void finalize_body(const CrtMats *__restrict__ M,
                                              const OzakiConsts *__restrict__ kc, int bx) {
  const int n = M->n;
  const int i = bx * T + threadIdx.x;
  if (i >= n) return;
  const int nblk = 1 << M->nrec;
  M->sa[i] = merged_exponent(reinterpret_cast<const double2 *>(M->pa) + i, nblk * M->chunks, n,
                             kc->L);
  M->sb[i] = merged_exponent(reinterpret_cast<const double2 *>(M->pb) + i, nblk, n, kc->L);
}

__global__ __launch_bounds__(T) void crt_finalize_kernel(const CrtMats *__restrict__ M,
                                                         const OzakiConsts *__restrict__ kc) {
  finalize_body(M, kc, blockIdx.x);
}

// ------------------------------------------------------------------ split
// A leaf L -> row-major residue leaves, transposed through LDS: tiles of 32
// rows x 128 k.  PLAIN (the leaf column-major, bs == 1 or bs == m): the
// column-major side moves as 256-byte column pieces; the row-major side moves
// as 128-byte row pieces (8 lanes x 16 residues).  Elements past m are zero,
// 16-byte chunks past residue_k skipped.  Column c of the tile in T2[c], row r
// at slot r ^ tswz(c); the transposed read has lanes on 8 rows and 8 column
// groups, the swizzle puts 4 of the groups 8 slots apart (the other 4 pairs
// share a slot: a 64-lane 8-byte read spans at least two 256-byte passes
// anyway).
constexpr int SPLIT_R = 32, SPLIT_K = 128;
__device__ __forceinline__ int tswz(int c) { return ((c >> 4) & 3) << 3; }

template <bool PLAIN>
__device__ __forceinline__ void split_a_body(const CrtMats *__restrict__ M,
                                             const OzakiConsts *__restrict__ kc, int bx, int by,
                                             double (&T2)[SPLIT_K][SPLIT_R]) {
  const int m = M->m, nmod = M->nmod, bs = M->bs;
  const int L = by;
  int bi, bj;
  leaf_coords(L, M->nrec, bi, bj);
  const double *A = M->A + (long long)L * m * m;
  const long long plane = M->plane;
  const int tk = (m + SPLIT_K - 1) / SPLIT_K;
  const int r0 = (bx / tk) * SPLIT_R, k0 = (bx % tk) * SPLIT_K;
  // a thread's 16 elements: one row, every 8th column.  Elements outside are
  // read at the leaf's first one and dropped, so that all loads go out before a
  // wait (a branch around each: 13.6 against 9.3 us at n = 640, 57 against 50 at
  // n = 3000)
  constexpr int NV = SPLIT_R * SPLIT_K / T, DC = T / SPLIT_R;
  const int tr = threadIdx.x % SPLIT_R, tc = threadIdx.x / SPLIT_R;
  double v[NV];
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int ti = r0 + tr, tj = k0 + tc + DC * i;
    const bool in = ti < m && tj < m;
    v[i] = A[!in ? 0 : (PLAIN ? ti + (long long)tj * m : leaf_elem_offset(m, bs, ti, tj))];
    v[i] = in ? v[i] : 0.0;
  }
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int c = tc + DC * i;
    T2[c][tr ^ tswz(c)] = v[i];
  }
  __syncthreads();
  const int r = threadIdx.x >> 3, kq = (threadIdx.x & 7) * 16;
  const int li = r0 + r;
  if (li >= m || k0 + kq >= m) return;
  const int sa = M->sa[bi * m + li];
  double x[16];
#pragma unroll
  for (int c = 0; c < 16; c++) x[c] = trunc(ldexp(T2[kq + c][r ^ tswz(kq)], sa));
  int8_t *dst = M->ra + L * residue_area(m) + (long long)li * residue_pitch(m) + k0 + kq;
  for (int l = 0; l < nmod; l++) {
    const int mi = kc->m[l];
    const double inv = kc->inv_m[l];
    const int c22 = kc->c22[l];
    unsigned w[4];
#pragma unroll
    for (int q = 0; q < 4; q++)
      w[q] = pack4_lo(sym_residue(x[4 * q], mi, inv, c22),
                      sym_residue(x[4 * q + 1], mi, inv, c22),
                      sym_residue(x[4 * q + 2], mi, inv, c22),
                      sym_residue(x[4 * q + 3], mi, inv, c22));
    *reinterpret_cast<uint4 *>(dst + l * plane) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

template <bool PLAIN>
__global__ __launch_bounds__(T) void crt_split_a_kernel(const CrtMats *__restrict__ M,
                                                        const OzakiConsts *__restrict__ kc) {
  __shared__ double Ts[SPLIT_K][SPLIT_R];  // [col][swizzled row]
  split_a_body<PLAIN>(M, kc, blockIdx.x, blockIdx.y, Ts);
}

// B leaf L -> column-major residue leaves; thread per 16 consecutive rows of a
// column (rows past m are zero).  PLAIN: the leaf is column-major.
template <bool PLAIN>
__device__ __forceinline__ void split_b_body(const CrtMats *__restrict__ M,
                                             const OzakiConsts *__restrict__ kc, int bx, int by,
                                             int gx) {
  const int m = M->m, nmod = M->nmod, bs = M->bs;
  const int L = by;
  int bi, bj;
  leaf_coords(L, M->nrec, bi, bj);
  const double *B = M->B + (long long)L * m * m;
  int8_t *rb = M->rb + L * residue_area(m);
  const long long plane = M->plane;
  const int ld = residue_pitch(m), c16 = residue_k(m) / 16;
  const long long units = (long long)m * c16;
  for (long long u = (long long)bx * T + threadIdx.x; u < units; u += (long long)gx * T) {
    const int lj = (int)(u / c16), li = (int)(u - (long long)lj * c16) * 16;
    const int s = M->sb[bj * m + lj];
    double x[16];
    if (PLAIN) {
      load_rows16(B + (long long)lj * m + li, m - li, x);
    } else {
#pragma unroll
      for (int c = 0; c < 16; c++)
        x[c] = li + c < m ? B[leaf_elem_offset(m, bs, li + c, lj)] : 0.0;
    }
#pragma unroll
    for (int c = 0; c < 16; c++) x[c] = trunc(ldexp(x[c], s));
    for (int l = 0; l < nmod; l++) {
      const int mi = kc->m[l];
      const double inv = kc->inv_m[l];
      const int c22 = kc->c22[l];
      unsigned w[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        unsigned v = 0;
#pragma unroll
        for (int b = 0; b < 4; b++)
          v |= (unsigned)(sym_residue(x[4 * q + b], mi, inv, c22) & 0xff) << (8 * b);
        w[q] = v;
      }
      *reinterpret_cast<uint4 *>(rb + l * plane + (long long)lj * ld + li) =
          make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
}

template <bool PLAIN>
__global__ __launch_bounds__(T) void crt_split_b_kernel(const CrtMats *__restrict__ M,
                                                        const OzakiConsts *__restrict__ kc) {
  split_b_body<PLAIN>(M, kc, blockIdx.x, blockIdx.y, gridDim.x);
}

// ------------------------------------------------------------------ reconstruct
// C' residues (column-major leaves) -> C (CAPS layout, bs blocks); thread: 4
// consecutive rows of a column.  PLAIN: the leaf of C is column-major.
template <int NP, bool PLAIN>
__device__ __forceinline__ void recon_body(const CrtMats *__restrict__ M,
                                           const OzakiConsts *__restrict__ kc, int bx, int by,
                                           int gx) {
  const int m = M->m, nmod = M->nmod, bs = M->bs;
  const int L = by;
  int bi, bj;
  leaf_coords(L, M->nrec, bi, bj);
  double *C = M->C + (long long)L * m * m;
  const int8_t *rc = M->rc + L * residue_area(m);
  const long long plane = M->plane;
  const int ld = residue_pitch(m), w4 = (m + 3) / 4;  // words of a column with rows below m
  const long long units = (long long)m * w4;
  for (long long u = (long long)bx * T + threadIdx.x; u < units; u += (long long)gx * T) {
    const int lj = (int)(u / w4), li = (int)(u - (long long)lj * w4) * 4;
    const int sb = M->sb[bj * m + lj];
    const int *sa = M->sa + bi * m + li;
    double S[4][NP];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int p = 0; p < NP; p++) S[q][p] = 0.0;
    for (int l = 0; l < nmod; l++) {
      const unsigned w =
          *reinterpret_cast<const unsigned *>(rc + l * plane + (long long)lj * ld + li);
#pragma unroll
      for (int q = 0; q < 4; q++) crt_acc<NP>(S[q], (int)(int8_t)((w >> (8 * q)) & 0xff), l, kc);
    }
    if (PLAIN && m % 4 == 0) {
      double out[4];
#pragma unroll
      for (int q = 0; q < 4; q++) out[q] = ldexp(crt_finish<NP>(S[q], kc), -(sa[q] + sb));
      double2 *dst = reinterpret_cast<double2 *>(C + (long long)lj * m + li);
      dst[0] = make_double2(out[0], out[1]);
      dst[1] = make_double2(out[2], out[3]);
    } else {
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (li + q < m)
          C[PLAIN ? (long long)lj * m + li + q : leaf_elem_offset(m, bs, li + q, lj)] =
              ldexp(crt_finish<NP>(S[q], kc), -(sa[q] + sb));
    }
  }
}

template <int NP, bool PLAIN>
__global__ __launch_bounds__(T) void crt_recon_kernel(const CrtMats *__restrict__ M,
                                                      const OzakiConsts *__restrict__ kc) {
  recon_body<NP, PLAIN>(M, kc, blockIdx.x, blockIdx.y, gridDim.x);
}

// ------------------------------------------------------------------ segmented CRT steps
// One launch per kernel over the items of an uneven batch: segment args are
// CrtMats descriptions (crt_grid gives each item the grid it has alone).
template <int K, bool F, int NP>
__global__ __launch_bounds__(T) void crt_multi_kernel(const char *__restrict__ base,
                                                      const VSeg *__restrict__ segs, int nseg,
                                                      const OzakiConsts *__restrict__ kc) {
  __shared__ double Ts[K == CRT_SPLIT_A ? SPLIT_K : 1][K == CRT_SPLIT_A ? SPLIT_R : 1];
  __shared__ double2 P[K == CRT_PARTIALS ? T / 64 : 1][K == CRT_PARTIALS ? 64 : 1];
  const VSeg &S = segs[vseg_find(segs, nseg, blockIdx.x)];
  const int l = blockIdx.x - S.blk0;
  const int bx = l % S.gx, by = l / S.gx;
  const CrtMats *M = reinterpret_cast<const CrtMats *>(base + S.arg);
  if constexpr (K == CRT_PARTIALS) partials_body<F>(M, l, P);
  if constexpr (K == CRT_FINALIZE) finalize_body(M, kc, bx);
  if constexpr (K == CRT_SPLIT_A) split_a_body<F>(M, kc, bx, by, Ts);
  if constexpr (K == CRT_SPLIT_B) split_b_body<F>(M, kc, bx, by, S.gx);
  if constexpr (K == CRT_RECON) recon_body<NP, F>(M, kc, bx, by, S.gx);
}

// ------------------------------------------------------------------ residue Winograd steps
template <int OP, bool VEC4>
__device__ __forceinline__ void rew_body(const RPtrs &P, long long n, int l, int bx, int gx,
                                         const OzakiConsts *__restrict__ kc) {
  using Op = Ew<OP>;
  const int mi = kc->m[l], c22 = kc->c22[l];  // sums of at most 4 residues: |y| <= 512
  const int8_t *in[Op::NIN];
  int8_t *out[Op::NOUT];
#pragma unroll
  for (int k = 0; k < Op::NIN; k++) in[k] = P.in[k] + l * P.sin[k];
#pragma unroll
  for (int k = 0; k < Op::NOUT; k++) out[k] = P.out[k] + l * P.sout[k];
  const long long stride = (long long)gx * T;
  if (VEC4) {
    const long long n4 = n >> 2;
    for (long long i = (long long)bx * T + threadIdx.x; i < n4; i += stride) {
      unsigned w[Op::NIN];
#pragma unroll
      for (int k = 0; k < Op::NIN; k++) w[k] = reinterpret_cast<const unsigned *>(in[k])[i];
      unsigned o[Op::NOUT];
#pragma unroll
      for (int k = 0; k < Op::NOUT; k++) o[k] = 0;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        int x[Op::NIN], y[Op::NOUT];
#pragma unroll
        for (int k = 0; k < Op::NIN; k++) x[k] = (int)(int8_t)((w[k] >> (8 * b)) & 0xff);
        Op::apply(x, y);
#pragma unroll
        for (int k = 0; k < Op::NOUT; k++)
          o[k] |= (unsigned)(mod_k(y[k], c22, mi) & 0xff) << (8 * b);
      }
#pragma unroll
      for (int k = 0; k < Op::NOUT; k++) reinterpret_cast<unsigned *>(out[k])[i] = o[k];
    }
  } else {
    for (long long i = (long long)bx * T + threadIdx.x; i < n; i += stride) {
      int x[Op::NIN], y[Op::NOUT];
#pragma unroll
      for (int k = 0; k < Op::NIN; k++) x[k] = (int)in[k][i];
      Op::apply(x, y);
#pragma unroll
      for (int k = 0; k < Op::NOUT; k++) out[k][i] = (int8_t)mod_k(y[k], c22, mi);
    }
  }
}

// grid (blocks, entries, moduli)
template <int OP, bool VEC4>
__global__ __launch_bounds__(T) void rew_kernel(const RPtrs *__restrict__ tab, long long n,
                                                const OzakiConsts *__restrict__ kc) {
  rew_body<OP, VEC4>(tab[blockIdx.y], n, blockIdx.z, blockIdx.x, gridDim.x, kc);
}

// segments: gx blocks x (entries * moduli), aux = moduli
template <int OP, bool VEC4>
__global__ __launch_bounds__(T) void rew_multi_kernel(const char *__restrict__ base,
                                                      const VSeg *__restrict__ segs, int nseg,
                                                      const OzakiConsts *__restrict__ kc) {
  const VSeg &S = segs[vseg_find(segs, nseg, blockIdx.x)];
  const int l = blockIdx.x - S.blk0;
  const int by = l / S.gx;
  const RPtrs *tab = reinterpret_cast<const RPtrs *>(base + S.arg);
  rew_body<OP, VEC4>(tab[by / S.aux], S.n, by % S.aux, l % S.gx, S.gx, kc);
}

template <int OP>
hipError_t launch_rew_op(const RPtrs *tab, int count, long long n, int nmod, bool vec4,
                         const OzakiConsts *kc, hipStream_t s) {
  int gx, gy;
  rew_grid(count, n, nmod, vec4, gx, gy);
  dim3 grid((unsigned)gx, (unsigned)count, (unsigned)nmod);
  if (vec4)
    hipLaunchKernelGGL((rew_kernel<OP, true>), grid, dim3(T), 0, s, tab, n, kc);
  else
    hipLaunchKernelGGL((rew_kernel<OP, false>), grid, dim3(T), 0, s, tab, n, kc);
  return hipGetLastError();
}

template <int OP>
hipError_t launch_rew_op_multi(const char *base, const VSeg *segs, int nseg, int blocks,
                               bool vec4, const OzakiConsts *kc, hipStream_t s) {
  if (vec4)
    hipLaunchKernelGGL((rew_multi_kernel<OP, true>), dim3(blocks), dim3(T), 0, s, base, segs,
                       nseg, kc);
  else
    hipLaunchKernelGGL((rew_multi_kernel<OP, false>), dim3(blocks), dim3(T), 0, s, base, segs,
                       nseg, kc);
  return hipGetLastError();
}

template <int K, bool F>
hipError_t launch_crt_multi_k(int np, const char *base, const VSeg *segs, int nseg, int blocks,
                              const OzakiConsts *kc, hipStream_t s) {
  if (K != CRT_RECON || np <= 2)
    hipLaunchKernelGGL((crt_multi_kernel<K, F, 2>), dim3(blocks), dim3(T), 0, s, base, segs, nseg,
                       kc);
  else if (np == 3)
    hipLaunchKernelGGL((crt_multi_kernel<K, F, 3>), dim3(blocks), dim3(T), 0, s, base, segs, nseg,
                       kc);
  else
    hipLaunchKernelGGL((crt_multi_kernel<K, F, 4>), dim3(blocks), dim3(T), 0, s, base, segs, nseg,
                       kc);
  return hipGetLastError();
}

template <int K>
hipError_t launch_crt_multi_f(bool flag, int np, const char *base, const VSeg *segs, int nseg,
                              int blocks, const OzakiConsts *kc, hipStream_t s) {
  return flag ? launch_crt_multi_k<K, true>(np, base, segs, nseg, blocks, kc, s)
              : launch_crt_multi_k<K, false>(np, base, segs, nseg, blocks, kc, s);
}

unsigned capped_blocks(long long units, long long per_grid) {
  long long b = (units + T - 1) / T;
  long long cap = (long long)device_cu_count() * 8 / (per_grid > 0 ? per_grid : 1);
  if (cap < 1) cap = 1;
  if (b > cap) b = cap;
  return (unsigned)(b < 1 ? 1 : b);
}

template <int NP>
hipError_t launch_recon(const CrtMats *M, const CrtMats &h, const OzakiConsts *kc, hipStream_t s) {
  int gx, gy;
  const bool fast = crt_grid(CRT_RECON, h, gx, gy);
  dim3 grid((unsigned)gx, (unsigned)gy);
  if (fast)
    hipLaunchKernelGGL((crt_recon_kernel<NP, true>), grid, dim3(T), 0, s, M, kc);
  else
    hipLaunchKernelGGL((crt_recon_kernel<NP, false>), grid, dim3(T), 0, s, M, kc);
  return hipGetLastError();
}

}  // namespace

void rew_grid(int count, long long n, int nmod, bool vec4, int &gx, int &gy) {
  const long long units = vec4 ? (n >> 2) : n;
  long long blocks = (units + T - 1) / T;
  long long cap = (long long)device_cu_count() * 8 / ((long long)count * nmod);
  if (cap < 1) cap = 1;
  if (blocks > cap) blocks = cap;
  if (blocks < 1) blocks = 1;
  gx = (int)blocks;
  gy = count * nmod;
}

bool crt_grid(int k, const CrtMats &h, int &gx, int &gy) {
  const int leaves = 1 << (2 * h.nrec);
  const int nblk = 1 << h.nrec;
  const bool plain = (h.bs == 1 || h.bs == h.m);
  gy = 1;
  switch (k) {
    case CRT_PARTIALS:
      gx = (h.n + 63) / 64 * nblk * h.chunks + (int)(((long long)h.n * nblk + 3) / 4);
      return plain;
    case CRT_FINALIZE:
      gx = (h.n + T - 1) / T;
      return false;
    case CRT_SPLIT_A:
      gx = ((h.m + SPLIT_R - 1) / SPLIT_R) * ((h.m + SPLIT_K - 1) / SPLIT_K);
      gy = leaves;
      return plain;
    case CRT_SPLIT_B:
      gx = (int)capped_blocks((long long)h.m * residue_k(h.m) / 16, leaves);
      gy = leaves;
      return plain;
    case CRT_RECON:
      gx = (int)capped_blocks((long long)h.m * ((h.m + 3) / 4), leaves);
      gy = leaves;
      return plain;
  }
  gx = 0;
  return false;
}

hipError_t launch_crt_multi(int k, bool flag, int np, const char *base, const VSeg *segs,
                            int nseg, int blocks, const OzakiConsts *kc, hipStream_t s) {
  if (nseg <= 0 || blocks <= 0) return hipSuccess;
  switch (k) {
    case CRT_PARTIALS: return launch_crt_multi_f<CRT_PARTIALS>(flag, np, base, segs, nseg, blocks, kc, s);
    case CRT_FINALIZE: return launch_crt_multi_f<CRT_FINALIZE>(false, np, base, segs, nseg, blocks, kc, s);
    case CRT_SPLIT_A: return launch_crt_multi_f<CRT_SPLIT_A>(flag, np, base, segs, nseg, blocks, kc, s);
    case CRT_SPLIT_B: return launch_crt_multi_f<CRT_SPLIT_B>(flag, np, base, segs, nseg, blocks, kc, s);
    case CRT_RECON: return launch_crt_multi_f<CRT_RECON>(flag, np, base, segs, nseg, blocks, kc, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_residue_ew_multi(int op, const char *base, const VSeg *segs, int nseg,
                                   int blocks, bool vec4, const OzakiConsts *kc, hipStream_t s) {
  if (nseg <= 0 || blocks <= 0) return hipSuccess;
  switch (op) {
    case EW_BFS_PRE: return launch_rew_op_multi<EW_BFS_PRE>(base, segs, nseg, blocks, vec4, kc, s);
    case EW_BFS_POST: return launch_rew_op_multi<EW_BFS_POST>(base, segs, nseg, blocks, vec4, kc, s);
    case EW_DFS_PRE1: return launch_rew_op_multi<EW_DFS_PRE1>(base, segs, nseg, blocks, vec4, kc, s);
    case EW_DFS_PRE2: return launch_rew_op_multi<EW_DFS_PRE2>(base, segs, nseg, blocks, vec4, kc, s);
    case EW_DFS_PRE3: return launch_rew_op_multi<EW_DFS_PRE3>(base, segs, nseg, blocks, vec4, kc, s);
    case EW_DFS_POST1: return launch_rew_op_multi<EW_DFS_POST1>(base, segs, nseg, blocks, vec4, kc, s);
    case EW_DFS_POST2: return launch_rew_op_multi<EW_DFS_POST2>(base, segs, nseg, blocks, vec4, kc, s);
    case EW_DFS_POST3: return launch_rew_op_multi<EW_DFS_POST3>(base, segs, nseg, blocks, vec4, kc, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_crt_step(int step, const CrtMats *M, const CrtMats &h, const OzakiConsts *kc,
                           hipStream_t s) {
  const int leaves = 1 << (2 * h.nrec);
  if (leaves > 65535) return hipErrorInvalidValue;
  int gx, gy;
  bool f;
  switch (step) {
    case 0: {
      f = crt_grid(CRT_PARTIALS, h, gx, gy);
      if (f)
        hipLaunchKernelGGL((crt_partials_kernel<true>), dim3(gx), dim3(T), 0, s, M);
      else
        hipLaunchKernelGGL((crt_partials_kernel<false>), dim3(gx), dim3(T), 0, s, M);
      crt_grid(CRT_FINALIZE, h, gx, gy);
      hipLaunchKernelGGL(crt_finalize_kernel, dim3(gx), dim3(T), 0, s, M, kc);
      return hipGetLastError();
    }
    case 1: {
      f = crt_grid(CRT_SPLIT_A, h, gx, gy);
      if (f)
        hipLaunchKernelGGL((crt_split_a_kernel<true>), dim3(gx, gy), dim3(T), 0, s, M, kc);
      else
        hipLaunchKernelGGL((crt_split_a_kernel<false>), dim3(gx, gy), dim3(T), 0, s, M, kc);
      if (h.fused_b) return hipGetLastError();
      f = crt_grid(CRT_SPLIT_B, h, gx, gy);
      if (f)
        hipLaunchKernelGGL((crt_split_b_kernel<true>), dim3(gx, gy), dim3(T), 0, s, M, kc);
      else
        hipLaunchKernelGGL((crt_split_b_kernel<false>), dim3(gx, gy), dim3(T), 0, s, M, kc);
      return hipGetLastError();
    }
    case 2: {
      switch (ozaki_npieces(h.nmod)) {
        case 1:
        case 2: return launch_recon<2>(M, h, kc, s);
        case 3: return launch_recon<3>(M, h, kc, s);
        default: return launch_recon<4>(M, h, kc, s);
      }
    }
  }
  return hipErrorInvalidValue;
}

hipError_t launch_residue_ew(int op, const RPtrs *tab, int count, long long n, int nmod,
                             bool vec4, const OzakiConsts *kc, hipStream_t s) {
  if (count <= 0 || n <= 0) return hipSuccess;
  if (nmod < 2 || nmod > OZ_MAX_MODULI) return hipErrorInvalidValue;
  for (int c0 = 0; c0 < count; c0 += 65535) {
    const RPtrs *t = tab + c0;
    const int c = count - c0 < 65535 ? count - c0 : 65535;
    hipError_t e = hipErrorInvalidValue;
    switch (op) {
      case EW_BFS_PRE: e = launch_rew_op<EW_BFS_PRE>(t, c, n, nmod, vec4, kc, s); break;
      case EW_BFS_POST: e = launch_rew_op<EW_BFS_POST>(t, c, n, nmod, vec4, kc, s); break;
      case EW_DFS_PRE1: e = launch_rew_op<EW_DFS_PRE1>(t, c, n, nmod, vec4, kc, s); break;
      case EW_DFS_PRE2: e = launch_rew_op<EW_DFS_PRE2>(t, c, n, nmod, vec4, kc, s); break;
      case EW_DFS_PRE3: e = launch_rew_op<EW_DFS_PRE3>(t, c, n, nmod, vec4, kc, s); break;
      case EW_DFS_POST1: e = launch_rew_op<EW_DFS_POST1>(t, c, n, nmod, vec4, kc, s); break;
      case EW_DFS_POST2: e = launch_rew_op<EW_DFS_POST2>(t, c, n, nmod, vec4, kc, s); break;
      case EW_DFS_POST3: e = launch_rew_op<EW_DFS_POST3>(t, c, n, nmod, vec4, kc, s); break;
    }
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace caps
