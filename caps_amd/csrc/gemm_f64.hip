// Batched FP64 leaf GEMM on the gfx950 matrix cores (replaces the BLAS call
// square_dgemm_zero, dgemm-blas.cpp:4-13: C = A*B, beta = 0, column-major).
//
// MFMA-bound: v_mfma_f64_16x16x4_f64 (2048 flop, 64 cycles of a SIMD's matrix
// core).  Block tile 128 x 128, 64 x 64 or 32 x 32 (dgemm_block_tile), 4
// waves in a 2 x 2 grid; a wave of the 128 tile holds 64 x 64 = 4 x 4 MFMA
// tiles.  Every tile size sums each element's products in the same K order,
// so the results do not depend on it.
//
// K goes through LDS in slices of 16, two stages, filled by buffer loads that
// write LDS directly (no registers and no LDS stores for the operands).  The
// block barrier of a slice sits before its last quarter: there every wave has
// its last fragments in registers, so the stage is free for the slice after
// next, and the first fragments of the next slice are read while the last
// quarter's MFMAs run; no wave starts a slice waiting for LDS.  Measured on
// 49 products of 2048^3: 13.9 ms (60 TFLOP/s, MFMA busy 0.78) with operands
// staged through registers and the barrier between slices, 12.0 ms with the
// direct loads, 11.75 ms (71.5 TFLOP/s, busy 0.93 at 2.38 GHz) with the
// barrier moved; without any operand load it takes 11.9 (barrier between
// slices), so what is left is the matrix cores' own rate.
//
// One persistent launch covers all tiles of all problems of the batch (the
// 7^b sub-products of the batched levels).  Consecutive tile ids stay on the
// same XCD (blocks are dispatched round-robin over the 8 XCDs) and sweep an
// 8 x 4 patch of tiles, so one XCD's L2 sees 8 A row panels and 4 B column
// panels of one problem at a time.
#include <math.h>

#include "kernels.h"
#include "tilemap.h"

namespace caps {

long long dgemm_full_tiles(int bt, long long total);

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void *lds_ptr;
typedef __attribute__((address_space(1))) double gdouble;

constexpr int NT = 256;
constexpr int BK = 16;  // K slice

// Block tile BT x BT (128, 64 or 32), 4 waves in a 2 x 2 grid of (BT / 2)^2
// wave tiles.
template <int BT>
struct Tile {
  static constexpr int WT = BT / 2;        // wave tile
  static constexpr int MT = WT / 16;       // MFMA tiles per wave dimension
  static constexpr int STAGE = BT * BK;    // doubles of one operand's stage
  static constexpr int OCC = BT == 128 ? 2 : (BT == 64 ? 4 : 8);  // blocks per CU
  static constexpr int IT = STAGE / 2 / NT;  // 16-byte chunks per thread and operand
};

// LDS stage of an operand, in 16-byte slots filled in lane order (slot s of
// the stage by lane s % 64 of one 1 KB load):
//   A: column k of the slice = BT / 2 slots; row pair c in slot c ^ 8 (k & 1)
//   B: column j of the tile = 8 slots of two k; pair c in slot c ^ ((j >> 1) & 7)
// The 32 lanes of a ds_read_b64 pass hold 16 rows (columns) and two
// neighbouring k: for A the two k fall into different halves of the 256 bytes
// of the 64 banks, for B the 8 columns of one parity take 8 distinct slots,
// so a pass touches every bank once.
template <int BT>
__device__ __forceinline__ void slot_a(int s, int &k, int &row) {
  k = s / (BT / 2);
  row = 2 * ((s % (BT / 2)) ^ (8 * (k & 1)));
}
__device__ __forceinline__ void slot_b(int s, int &k, int &col) {
  col = s >> 3;
  k = 2 * ((s & 7) ^ ((col >> 1) & 7));
}

// block barrier for stages filled by this wave's own loads: the caller has
// waited for them; the empty asm statements keep memory operations on their
// side (__syncthreads would add a fence that waits for everything)
__device__ __forceinline__ void stage_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// byte offset of a lane that must not access memory: beyond NUM_RECORDS, so
// the buffer range check returns zeros
constexpr int NUM_RECORDS = 0x40000000;
constexpr int OUT_OF_RANGE = 0x7fffff00;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t slice_rsrc(const double *p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(p), 0, NUM_RECORDS, 0x00020000);
}

// 64 lanes x 16 bytes from the slice at p (lane offset v) to 1 KB of LDS
__device__ __forceinline__ void dma_1k(__amdgpu_buffer_rsrc_t r, double *lds, int v) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr)lds, 16, v, 0, 0, 0);
}

// One block tile (ti, tj) of C = A * B.  Operands are m x m, stored as a
// quadtree of 2^d x 2^d column-major leaves of size m0 = m >> d in the CAPS
// quadrant order (d = 0: plain column-major); without EDGE m0 % BT == 0, so
// every tile and K slice lies in one leaf.  EDGE (d = 0): rows and columns
// beyond m read as zero and are not stored; a last K slice of m % 16 elements
// is staged through registers, element by element.
template <int BT, bool EDGE>
__device__ __forceinline__ void dgemm_tile(const double *__restrict__ A,
                                           const double *__restrict__ B, double *__restrict__ C,
                                           int m, int m0, int d, int ti, int tj, double *S) {
  using T = Tile<BT>;
  constexpr int WT = T::WT, MT = T::MT, IT = T::IT;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int l16 = lane & 15, lk = lane >> 4;
  const int nk = m / BK;  // whole slices
  const int row0 = ti * BT, col0 = tj * BT;
  const long long mm0 = (long long)m0 * m0;

  // byte offsets, in a slice, of the chunks this lane stages
  int va[IT], vb[IT];
#pragma unroll
  for (int it = 0; it < IT; it++) {
    const int s = (it * 4 + wave) * 64 + lane;
    int k, r, c;
    slot_a<BT>(s, k, r);
    va[it] = (EDGE && row0 + r >= m) ? OUT_OF_RANGE : (k * m0 + r) * 8;
    slot_b(s, k, c);
    vb[it] = (EDGE && col0 + c >= m) ? OUT_OF_RANGE : (c * m0 + k) * 8;
  }
  // first element of the next A slice (row0, k) and B slice (k, col0), moved
  // along K: 16 columns of A and 16 rows of B per slice, the next leaf of the
  // quadtree after m0
  auto a_at = [&](int k) {
    return A + quad_leaf(row0 / m0, k / m0, d) * mm0 + (row0 % m0);
  };
  auto b_at = [&](int k) {
    return B + quad_leaf(k / m0, col0 / m0, d) * mm0 + (long long)(col0 % m0) * m0;
  };
  const double *pa = d == 0 ? A + row0 : a_at(0);
  const double *pb = d == 0 ? B + (long long)col0 * m0 : b_at(0);
  int kleft = m0;  // k to the end of the leaf
  int knext = 0;
  auto stage = [&](double *As, double *Bs) {
    const __amdgpu_buffer_rsrc_t ra = slice_rsrc(pa), rb = slice_rsrc(pb);
#pragma unroll
    for (int it = 0; it < IT; it++) dma_1k(ra, As + (it * 4 + wave) * 128, va[it]);
#pragma unroll
    for (int it = 0; it < IT; it++) dma_1k(rb, Bs + (it * 4 + wave) * 128, vb[it]);
    pa += (long long)BK * m0;
    pb += BK;
    knext += BK;
    kleft -= BK;
    if (kleft == 0 && knext < m) {
      pa = a_at(knext);
      pb = b_at(knext);
      kleft = m0;
    }
  };
  // this lane's fragment offsets (doubles): A row wm WT + 16 r + l16, k = 4 kk
  // + lk; the slot XOR swaps the 16-row groups of odd k
  const int odd = lk & 1;
  const int fa = lk * BT + wm * WT + l16;
  const int fae = fa + 16 * odd, fao = fa - 16 * odd;  // even / odd group
  const int fa1 = lk * BT + ((wm ^ odd) * 16) + l16;   // MT == 1: the group is wm itself
  const int sb = (l16 >> 1) & 7;
  int fb[4];
#pragma unroll
  for (int kk = 0; kk < 4; kk++)
    fb[kk] = (wn * WT + l16) * BK + (((2 * kk + (lk >> 1)) ^ sb) << 1) + odd;
  auto frags = [&](const double *As, const double *Bs, int kk, double (&a)[MT], double (&b)[MT]) {
#pragma unroll
    for (int r = 0; r < MT; r++)
      a[r] = MT == 1 ? As[fa1 + 4 * kk * BT]
                     : As[((r & 1) ? fao : fae) + 4 * kk * BT + 16 * r];
#pragma unroll
    for (int c = 0; c < MT; c++) b[c] = Bs[fb[kk] + c * 16 * BK];
  };

  v4d acc[MT][MT];
#pragma unroll
  for (int r = 0; r < MT; r++)
#pragma unroll
    for (int c = 0; c < MT; c++) acc[r][c] = v4d{0.0, 0.0, 0.0, 0.0};
  double a[4][MT], b[4][MT];
  auto mfmas = [&](int kk) {
#pragma unroll
    for (int r = 0; r < MT; r++)
#pragma unroll
      for (int c = 0; c < MT; c++)
        acc[r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[kk][c], a[kk][r], acc[r][c], 0, 0, 0);
  };
  constexpr int ST = T::STAGE;
  if (nk > 0) stage(S, S + ST);
  if (nk > 1) stage(S + 2 * ST, S + 3 * ST);
  if (nk > 1)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * IT) : "memory");
  else
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  stage_barrier();
  if (nk > 0) frags(S, S + ST, 0, a[0], b[0]);
  // slice kt: the first fragments are in registers, the others are read two
  // LDS instructions per MT MFMAs; the barrier comes before the last quarter
  for (int kt = 0; kt < nk; kt++) {
    double *cur = S + 2 * (kt & 1) * ST, *oth = S + 2 * ((kt & 1) ^ 1) * ST;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 1; kk < 4; kk++) frags(cur, cur + ST, kk, a[kk], b[kk]);
#pragma unroll
    for (int kk = 0; kk < 3; kk++) mfmas(kk);
#pragma unroll
    for (int i = 0; i < 3 * MT; i++) {
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, MT, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    // this wave's part of slice kt + 1 has landed and its last fragments of
    // slice kt are read
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    stage_barrier();
    if (kt + 1 < nk) frags(oth, oth + ST, 0, a[0], b[0]);
    if (kt + 2 < nk) stage(cur, cur + ST);
    mfmas(3);
  }
  stage_barrier();
  if (EDGE && nk * BK < m) {
    const int k0 = nk * BK;
#pragma unroll
    for (int it = 0; it < IT; it++) {
      const int s = (it * 4 + wave) * 64 + lane;
      int k, r, c;
      v2d v;
      slot_a<BT>(s, k, r);
      const double *ta = A + (long long)(k0 + k) * m + row0 + r;
      v.x = (k0 + k < m && row0 + r < m) ? ta[0] : 0.0;
      v.y = (k0 + k < m && row0 + r + 1 < m) ? ta[1] : 0.0;
      *reinterpret_cast<v2d *>(S + 2 * s) = v;
      slot_b(s, k, c);
      const double *tb = B + (long long)(col0 + c) * m + k0 + k;
      v.x = (col0 + c < m && k0 + k < m) ? tb[0] : 0.0;
      v.y = (col0 + c < m && k0 + k + 1 < m) ? tb[1] : 0.0;
      *reinterpret_cast<v2d *>(S + ST + 2 * s) = v;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
      frags(S, S + ST, kk, a[kk], b[kk]);
      mfmas(kk);
    }
    __syncthreads();
  }

  // D of mfma(b, a): lane holds row (lane % 16) of the 16 x 16 tile and
  // columns (lane / 16) + 4 v in its four result registers, so a store writes
  // whole 128-byte column pieces
  gdouble *Ct = (gdouble *)(C + (d == 0 ? 0 : quad_leaf(row0 / m0, col0 / m0, d) * mm0));
  const int rt = (d == 0 ? row0 : row0 % m0) + wm * WT + l16;
  const int ct = (d == 0 ? col0 : col0 % m0) + wn * WT + lk;
#pragma unroll
  for (int c = 0; c < MT; c++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int col = ct + c * 16 + 4 * v;
      gdouble *dst = Ct + (long long)col * m0 + rt;
#pragma unroll
      for (int r = 0; r < MT; r++)
        if (!EDGE || (col < m && rt + 16 * r < m)) dst[16 * r] = acc[r][c][v];
    }
}

// One persistent launch over all tiles of all problems of one size: the first
// `full` whole, the others as four tiles of half the size (dgemm_full_tiles),
// starting with the blocks dispatched last.
template <int BT, bool CHECK>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(Tile<BT>::OCC, Tile<BT>::OCC))) void
dgemm_kernel(const GemmPtrs *__restrict__ tab, int m,
                                                   TileMap map, int full, int m0, int d) {
  constexpr int STAGE = Tile<BT>::STAGE;
  __shared__ __attribute__((aligned(1024))) double S[4 * STAGE];
  const int G = gridDim.x;
  for (int round = 0; round * G < full; round++) {
    const int tile = round_tile(round, blockIdx.x, G, full);
    if (tile >= full) break;
    int prob, ti, tj;
    tile_coords(map, tile, prob, ti, tj);
    const GemmPtrs &P = tab[prob];
    dgemm_tile<BT, CHECK>(P.A, P.B, P.C, m, m0, d, ti, tj, S);
  }
  if constexpr (BT > 32) {
    const int subs = 4 * (map.total - full);
    const int last = (G / NXCD - 1 - (int)blockIdx.x / NXCD) * NXCD + (int)blockIdx.x % NXCD;
    for (int round = 0; round * G < subs; round++) {
      const int sub = round_tile(round, last, G, subs);
      if (sub >= subs) break;
      int prob, ti, tj;
      tile_coords(map, full + (sub >> 2), prob, ti, tj);
      ti = 2 * ti + (sub & 1);
      tj = 2 * tj + ((sub >> 1) & 1);
      if (CHECK && (ti * (BT / 2) >= m || tj * (BT / 2) >= m)) continue;
      const GemmPtrs &P = tab[prob];
      dgemm_tile<BT / 2, CHECK>(P.A, P.B, P.C, m, m0, d, ti, tj, S);
    }
  }
}

// One persistent launch over the tiles of problems of several sizes (the
// leaf products of an uneven batch): segment s holds gy problems of order n
// with gx x gx tiles each, from global tile blk0 on, arg = its GemmPtrs
// table, aux = quadtree levels | edge checks << 8.
template <int BT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(Tile<BT>::OCC, Tile<BT>::OCC))) void
dgemm_multi_kernel(const char *__restrict__ base,
                                                         const VSeg *__restrict__ segs, int nseg,
                                                         int total) {
  constexpr int STAGE = Tile<BT>::STAGE;
  __shared__ __attribute__((aligned(1024))) double S[4 * STAGE];
  const int G = gridDim.x;
  for (int round = 0; round * G < total; round++) {
    const int tile = round_tile(round, blockIdx.x, G, total);
    if (tile >= total) break;
    const VSeg &V = segs[vseg_find(segs, nseg, tile)];
    const int m = (int)V.n, d = V.aux & 255;
    const int local = tile - V.blk0, per = V.gx * V.gx;
    const int prob = local / per, r = local - prob * per;
    const int ti = r % V.gx, tj = r / V.gx;
    const GemmPtrs &P = reinterpret_cast<const GemmPtrs *>(base + V.arg)[prob];
    if (V.aux >> 8)
      dgemm_tile<BT, true>(P.A, P.B, P.C, m, m >> d, d, ti, tj, S);
    else
      dgemm_tile<BT, false>(P.A, P.B, P.C, m, m >> d, d, ti, tj, S);
  }
}

template <int BT>
hipError_t launch_tile(const GemmPtrs *tab, int count, int m, int levels, hipStream_t s) {
  bool ok;
  TileMap map = make_tilemap(m, BT, count, ok);
  if (!ok) return hipErrorInvalidValue;
  const int m0 = m >> levels;
  const bool fast = (m0 % BT == 0);
  if (!fast && levels > 0) return hipErrorInvalidValue;  // quadtree operands need whole tiles
  // persistent grid: as many blocks per CU as registers and LDS allow, a
  // multiple of the XCD count
  const int full = (int)dgemm_full_tiles(BT, map.total);
  const long long items = full + 4LL * (map.total - full);
  const int G = persistent_grid(Tile<BT>::OCC, device_cu_count(),
                                (int)(items < 0x7ffffff0LL ? items : 0x7ffffff0LL));
  if (fast)
    hipLaunchKernelGGL((dgemm_kernel<BT, false>), dim3(G), dim3(NT), 0, s, tab, m, map, full, m0,
                       levels);
  else
    hipLaunchKernelGGL((dgemm_kernel<BT, true>), dim3(G), dim3(NT), 0, s, tab, m, map, full, m0,
                       levels);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_dgemm_batched(const GemmPtrs *tab, int count, int m, int levels, int tile,
                                hipStream_t s) {
  if (count <= 0 || m <= 0) return hipSuccess;
  const int m0 = m >> levels;
  if (levels < 0 || (m0 << levels) != m) return hipErrorInvalidValue;
  switch (dgemm_block_tile(m, levels, tile, count)) {
    case 32: return launch_tile<32>(tab, count, m, levels, s);
    case 64: return launch_tile<64>(tab, count, m, levels, s);
    default: return launch_tile<128>(tab, count, m, levels, s);
  }
}

// Cost of a launch in units of one CU's full rate: the busiest CU runs
// ceil(tiles / CUs) tiles of bt^2 outputs.  The smaller tiles move more
// operand bytes per product and run at 0.86 (64) and 0.6 (32) of the 128
// tile's rate (49 products of 2048^3: 71.5, 60 and 41-49 TFLOP/s), but leave
// less of the device idle.  Measured with 128 / 64 / 32 tiles, all whole (us): one product
// of 512^3 72 / 25 / 15, of 1024^3 142 / 50 / 55; 49 of 256^3 46 / 44 / 53,
// of 384^3 111 / 119 / 142, of 512^3 283 / 265 / 332, of 750^3 842 / 869 /
// 1114; 343 of 49^3 26 / 13 / 13.
static double tile_time(int bt) {
  return bt * bt / (bt == 128 ? 1.0 : (bt == 64 ? 0.86 : 0.6));
}

double dgemm_tile_cost(int bt, double tiles) {
  return ceil(tiles / device_cu_count()) * tile_time(bt);
}

// Tiles that run whole, of `total`: all, or as many as give each CU the same
// number where the remaining ones take less time as tiles of half the size on
// more CUs.  Measured with all tiles whole and with this rule (us, with the
// last round spread over the XCDs): 49 products of 256^3 47 and 42, of 320^3
// 97 and 67, of 512^3 261 and 239, of 750^3 858 and 786; 7 of 2048^3 2136 and
// 1932.
long long dgemm_full_tiles(int bt, long long total) {
  const long long cus = device_cu_count(), left = total % cus;
  if (bt == 32 || left == 0) return total;
  return dgemm_tile_cost(bt / 2, 4.0 * left) < tile_time(bt) ? total - left : total;
}

int dgemm_block_tile(int m, int levels, int tile, long long count) {
  const int m0 = m >> levels;
  // tile 1: 64 x 64 block tiles (quadtree operands only when the leaf is a
  // multiple)
  if (tile == 1 && (levels == 0 || m0 % 64 == 0)) return 64;
  int best = 128;
  double cost = INFINITY;
  for (int bt = 128; bt >= 32; bt /= 2) {
    if (levels > 0 && m0 % bt != 0) continue;
    const double t = (m + bt - 1) / bt;
    const double tiles = t * t * (double)count, full = (double)dgemm_full_tiles(bt, (long long)tiles);
    const double c = dgemm_tile_cost(bt, full) + dgemm_tile_cost(bt / 2, 4 * (tiles - full));
    if (c < cost) {
      best = bt;
      cost = c;
    }
  }
  return best;
}

hipError_t launch_dgemm_multi(int bt, const char *base, const VSeg *segs, int nseg, int total,
                              hipStream_t s) {
  if (nseg <= 0 || total <= 0) return hipSuccess;
  const auto grid = [&](int occ) { return dim3(persistent_grid(occ, device_cu_count(), total)); };
  switch (bt) {
    case 32:
      hipLaunchKernelGGL((dgemm_multi_kernel<32>), grid(Tile<32>::OCC), dim3(NT), 0, s, base, segs,
                         nseg, total);
      break;
    case 64:
      hipLaunchKernelGGL((dgemm_multi_kernel<64>), grid(Tile<64>::OCC), dim3(NT), 0, s, base, segs,
                         nseg, total);
      break;
    case 128:
      hipLaunchKernelGGL((dgemm_multi_kernel<128>), grid(Tile<128>::OCC), dim3(NT), 0, s, base,
                         segs, nseg, total);
      break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace caps
