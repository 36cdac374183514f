// direct.hip -- direct solve of the eliminated system: banded Cholesky (L L^T) per mesh.
//
// The reference's solve() has a direct branch, solve(algorithm="GaussJordan")
// (FEMSolverClass.f90:1795-1798) -> gauss_jordan_crs (FEMSolverClass.f90:2413-2460), whose body
// stops with "Under construction" after the first pivot test ("A is singular" on a zero pivot,
// :2455).  This file gives that branch a working direct method for the symmetric positive
// definite systems the elimination produces (FEMSolverClass.f90:1707-1756 keeps K symmetric:
// fixed rows and columns are zeroed with a unit diagonal).
//
// Per mesh (one mesh = the whole system, or every mesh of a block-diagonal batch):
//  * ordering (host, once per sparsity pattern): the node (DOF=3 block) or DOF graph is
//    renumbered by the candidate of smallest bandwidth among the natural order, reverse
//    Cuthill-McKee and lexicographic coordinate sorts along each axis;
//  * band storage (LAPACK dpbtrf 'L' layout): entry (r, c), 0 <= r - c <= b, of the permuted
//    matrix at band[c*ld + r - c], ld >= b + 1; the order is padded to a multiple of 32 with
//    unit diagonal rows;
//  * factorization: left-looking by blocks of 32 columns: the block's (b+32) x 32 rows are
//    updated by the previous b columns with FP64 MFMA 16x16x4 tiles, the two 16 x 16 diagonal
//    tiles are factored with cross-lane operations and the tiles below are multiplied by their
//    inverse transposes.  A persistent kernel takes (mesh, share) items from a largest-first
//    queue; a mesh that alone would decide the time is shared by several workgroups, which take
//    its blocks in turn: a workgroup updates its block with the columns that are complete while
//    the others finish the preceding blocks, and publishes its own block as the mesh's progress;
//  * triangular solves (k_band_solve, half bandwidths up to 1024): blocks of 32 rows; the
//    diagonal blocks' inverses, formed in parallel beforehand, turn the serial solve into a
//    32 x 32 product, the moving window of the right-hand side stays in LDS, and a second,
//    row-major copy of L (written by the factorization beside the band) makes the backward
//    update's loads contiguous too.  Wider bands, and systems whose second copy does not fit the
//    memory: band_solve (blocks of 16, the diagonal solve in one wave).
// Fixed-precision iterative refinement on the true residual b - A x (the CRS values, in
// FP64) follows as requested.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <numeric>
#include <thread>
#include <vector>

#include "pf_internal.hpp"

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int DBT = 512;   // threads per workgroup of the factor/solve kernel

struct DMesh {
  int64_t d0;    // first DOF of the mesh in the system
  int64_t boff;  // first band entry
  int64_t woff;  // first entry of the mesh's permutation and work vector
  int32_t n;     // DOFs
  int32_t npad;  // n rounded up to a multiple of 32
  int32_t b;     // half bandwidth of the permuted matrix (DOFs)
  int32_t ld;    // leading dimension of the band (>= b + 1, even)
};

// share g of G of a mesh's factorization: blocks g, g + G, g + 2 G, ...
struct DItem {
  int32_t m, g, G, pad;
};

struct DArgs {
  const DMesh *mesh;
  const int32_t *order;  // queue order (largest first)
  const DItem *item;     // factorization: queue of shares, those of a mesh adjacent
  int32_t nitem;
  int32_t *progress;     // per mesh: blocks of 32 columns complete (-1: not positive definite, -2: gave up)
  int32_t polls;         // of a share for the preceding block before it gives up
  int32_t *queue;
  int32_t nmesh;
  int32_t mode;          // 0: factor, then solve x = A^-1 rhs; 1: solve only, x += A^-1 rhs; 2: factor only
  double *band;
  double *rows;          // L row by row: entry (r, c) at rows[boff + r ld + (r - c)] (NULL: not kept)
  const double *dinv;    // inverses of the 32 x 32 diagonal blocks: block J row i at dinv[32 (woff + 32 J + i)]
  const int32_t *perm;   // band index q of mesh m -> local DOF (perm[woff + q], q < n)
  double *w;             // work vector (npad per mesh)
  const double *rhs;
  double *x;
  int32_t *status;       // per mesh
  int64_t *t_raw;        // per mesh: wall-clock start, end of the factor+solve
};

__device__ inline double shfl(double v, int src) { return __shfl(v, src, 64); }

// A value read from LDS that is the same in every lane, as a scalar.
__device__ inline int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// p[i]: scalar base, 32-bit lane offset (one address register per load instead of two)
__device__ inline double at(const double *__restrict__ p, uint32_t i) {
  return *(const double *)((const char *)p + (i * 8u));
}

// The wave index within the workgroup as a scalar: the compiler cannot tell that
// threadIdx.x / 64 is the same in every lane of a wave, and without this every tile index,
// chunk bound and loop counter derived from it would be kept per lane, with masked branches
// and full waits for outstanding loads where they join.
__device__ inline int wave_id() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// The lane index, re-read inside a loop so that the compiler rebuilds the lane masks derived
// from it there instead of hoisting hundreds of them out of the loop and spilling them.
__device__ inline int lane_id() {
  int l = (int)(threadIdx.x & 63);
  asm volatile("" : "+v"(l));
  return l;
}

// acc += A B for the 16x4 fragment A (lane l holds A[l%16][l/16]) and the 4x16 fragment B
// (lane l holds B[l/16][l%16]); accumulator layout (that of
// v_mfma_f64_16x16x4f64): lane l, element v: row 4 v + l/16, column l%16.  MF: the matrix core; else the
// same product from cross-lane reads and FMAs.
template <bool MF>
__device__ inline void tile_fma(d4 &acc, double af, double bf, int q, int jl) {
  if constexpr (MF) {
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(af, bf, acc, 0, 0, 0);
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double bk = shfl(bf, 16 * k + jl);
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[v] += shfl(af, 16 * k + 4 * v + q) * bk;
    }
  }
}

// Geometry of one block of 32 columns j0 .. j0+31 and of a wave's tiles in one pass: row
// tiles t (rows R = j0 + 16 t .. R+15, t < T) of the rows j0 .. j0+31+b, column tiles
// ct = 0 (columns j0 .. j0+15) and ct = 1 (j0+16 .. j0+31); the wave holds tiles
// tb, tb + W, ..., tb + (MAXT-1) W.  MAXT tiles of 16 rows x 32 columns per wave: 2, 4 or 6, the
// fewest that hold the whole block in one pass where 6 do.  A second pass would start its update
// only after the first one's diagonal tiles, which the shares of a mesh cannot overlap, and every
// B fragment feeds all of a wave's tiles.
struct BlockGeom {
  int j0, b, npad, T, tb, W;
  int64_t ld;
};

// Fragments of U consecutive 4-column chunks c0, c0+4, ... of the previous columns: A
// fragments L[R + l%16][c + l/16] of the wave's tiles and B fragments L[j0 + 16 ct + l%16]
// [c + l/16] of both column tiles.  This is the form for the first chunks of a tile (where
// some lanes' entries lie outside the band) and the last rows: every load has an index
// clamped into the band and chunks from cend on repeat the last one, so the loads are
// unconditional and stay in flight together (a load under a condition keeps the register's older
// value alive across the loop and spills it), and the entries outside the band are replaced by zero
// where they are used.
template <int U, int MAXT>
struct Frags {
  double b[U][2];
  double a[U][MAXT];
};

template <int U, int MAXT>
__device__ inline void load_frags(Frags<U, MAXT> &f, const double *__restrict__ band, const BlockGeom &g, int c0,
                                  int cend, int q, int jl) {
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int c = min(c0 + 4 * u, cend - 4);
    const double *col = band + (int64_t)c * g.ld;
    const uint32_t lq = (uint32_t)(q * (int)g.ld);
    const int ck = c + q;
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) f.b[u][ct] = at(col, lq + min(g.j0 + 16 * ct + jl - ck, g.b));  // j0 + jl > ck
#pragma unroll
    for (int i = 0; i < MAXT; ++i) {
      const int R = g.j0 + 16 * (g.tb + g.W * i);
      f.a[u][i] = at(col, lq + min(R + jl - ck, g.b));  // R + jl > ck
    }
  }
}

// acc[i][ct] += A (-B_ct) over the group's chunks (tile 0 has no column tile 1)
template <bool MF, int U, int MAXT>
__device__ inline void mfma_frags(const Frags<U, MAXT> &f, d4 (*acc)[2], const BlockGeom &g, int c0, int cend, int q,
                                  int jl) {
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int c = c0 + 4 * u;
    if (c >= cend) continue;  // wave-uniform
    const int ck = c + q;
    double bn[2];
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) bn[ct] = (g.j0 + 16 * ct + jl - ck <= g.b) ? -f.b[u][ct] : 0.0;
#pragma unroll
    for (int i = 0; i < MAXT; ++i) {
      const int t = g.tb + g.W * i;
      const int R = g.j0 + 16 * t;
      if (t < g.T && c + 3 >= R - g.b) {  // wave-uniform
        const int ra = R + jl;
        const double af = (ra < g.npad && ra - ck <= g.b) ? f.a[u][i] : 0.0;
        tile_fma<MF>(acc[i][0], af, bn[0], q, jl);
        if (t >= 1) tile_fma<MF>(acc[i][1], af, bn[1], q, jl);
      }
    }
  }
}

// The steady part of a pass: chunks cs <= c < ce, where every lane's entry of each of the
// wave's nt existing tiles and of both column tiles lies inside the band and the tiles' rows
// end before the padding.  Branch-free: scalar bases that advance by 4 (ld - 1)
// doubles per chunk, two groups of chunks in flight, each A fragment used by both column
// tiles.
template <bool MF, int U, int MAXT>
__device__ inline void steady_update(d4 (*acc)[2], const double *__restrict__ band, const BlockGeom &g, int cs,
                                     int ce, int nt, int q, int jl) {
  const int64_t step = g.ld - 1;
  const double *pb = band + (int64_t)cs * step + g.j0;
  const uint32_t lq = (uint32_t)(q * (int)step + jl);
  double a0[U][MAXT], a1[U][MAXT], b0[U][2], b1[U][2];
  auto load = [&](double (&a)[U][MAXT], double (&bb)[U][2], int c) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const double *col = pb + (int64_t)(min(c + 4 * u, ce - 4) - cs) * step;
#pragma unroll
      for (int i = 0; i < MAXT; ++i) a[u][i] = at(col + 16 * (g.tb + g.W * min(i, nt - 1)), lq);
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) bb[u][ct] = at(col + 16 * ct, lq);
    }
  };
  auto prod = [&](const double (&a)[U][MAXT], const double (&bb)[U][2], int c) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (c + 4 * u >= ce) continue;  // wave-uniform
      const double bn0 = -bb[u][0], bn1 = -bb[u][1];
#pragma unroll
      for (int i = 0; i < MAXT; ++i)
        if (i < nt) {
          tile_fma<MF>(acc[i][0], a[u][i], bn0, q, jl);
          if (g.tb + g.W * i >= 1) tile_fma<MF>(acc[i][1], a[u][i], bn1, q, jl);
        }
    }
  };
  load(a0, b0, cs);
  for (int c = cs; c < ce; c += 8 * U) {
    load(a1, b1, c + 4 * U);
    prod(a0, b0, c);
    load(a0, b0, c + 8 * U);
    prod(a1, b1, c + 4 * U);
  }
}

// LDS written by other lanes of the wave may be read after this.  (The hardware keeps a wave's LDS
// accesses in order; without the fence the compiler may hand a lane back what it wrote itself.)
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// v of one lane, as a scalar
__device__ inline double bcast(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

constexpr int LS = 17;  // row stride of 16 x 16 tiles in LDS: rows and columns both without bank conflicts

// Diagonal tile of column tile ct (held by the calling wave in accumulator layout): Cholesky
// factor L_d to the band (columns col0 .. col0+15), and L_d^-T to LDS sLi; *sflag on a non-positive
// pivot.  This is the serial chain of a block, so it is kept short: lane i < 16 holds row i of the
// tile and lane 16 + j column j of the identity, both in registers; step k scales entry k and
// subtracts the multiples L[j][k] (scalars, from lane j) of it from the entries j > k.  The same
// instructions turn the rows into L_d and the identity's columns into those of L_d^-1, without a
// branch.  (Before: the factor in the accumulator layout and the inverse after it, by cross-lane
// reads under masks, which were most of a block's 47 us.)
__device__ inline void diag_block(const d4 &a, double *__restrict__ band, double *__restrict__ lrow, int64_t ld,
                                  int b, int col0, double *sL, double *sLi, int32_t *sflag) {
  const int ln = lane_id();
  const int q = ln >> 4, jl = ln & 15;
#pragma unroll
  for (int v = 0; v < 4; ++v) sL[(4 * v + q) * LS + jl] = a[v];
  wave_sync();
  double r[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const double l = sL[jl * LS + j];
    r[j] = q == 0 ? l : (j == jl ? 1.0 : 0.0);
  }
  bool bad = false;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const double piv = bcast(r[k], k);
    bad = bad || !(piv > 0.0);
    const double s = sqrt(piv);
    const double rs = 1.0 / s;
    r[k] = ln == k ? s : r[k] * rs;
#pragma unroll
    for (int j = k + 1; j < 16; ++j) r[j] = fma(-r[k], bcast(r[k], j), r[j]);
  }
  // rows of L_d; column j of L_d^-1 is row j of L_d^-T
  double *out = (q == 0 ? sL : sLi) + jl * LS;
  if (q < 2) {
#pragma unroll
    for (int j = 0; j < 16; ++j) out[j] = r[j];
  }
  wave_sync();
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int i = 4 * v + q;
    const int d = i - jl;
    const double l = sL[i * LS + jl];
    if (d >= 0 && d <= b) {
      band[(int64_t)(col0 + jl) * ld + d] = l;
      if (lrow) lrow[(int64_t)(col0 + i) * ld + d] = l;
    }
  }
  if (bad && ln == 0) *sflag = 1;
}

// x = c m^T for 16 x 16 tiles: c in accumulator layout (through the wave's LDS tile myC into
// A fragments), m given by its B fragments mb[cq] = m[jl][4 cq + q]... i.e. B[kk][n] =
// m^T[4 cq + kk][n]; sign -1 subtracts the product from acc instead
template <bool MF>
__device__ inline void tile_times(d4 &acc, const d4 &c, const double *mb, double *myC) {
  const int ln = lane_id();
  const int q = ln >> 4, jl = ln & 15;
#pragma unroll
  for (int v = 0; v < 4; ++v) myC[(4 * v + q) * LS + jl] = c[v];
  wave_sync();
  double af[4];
#pragma unroll
  for (int cq = 0; cq < 4; ++cq) af[cq] = myC[jl * LS + 4 * cq + q];
  wave_sync();  // myC is free again
#pragma unroll
  for (int cq = 0; cq < 4; ++cq) tile_fma<MF>(acc, af[cq], mb[cq], q, jl);
}

// store a tile (accumulator layout) of column tile starting at col0 into the band
__device__ inline void store_tile(const d4 &x, double *__restrict__ band, double *__restrict__ lrow, int64_t ld,
                                  int b, int npad, int R, int col0) {
  const int ln = lane_id();
  const int q = ln >> 4, jl = ln & 15;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int r = R + 4 * v + q;
    const int d = r - (col0 + jl);
    if (r < npad && d >= 0 && d <= b) {
      band[(int64_t)(col0 + jl) * ld + d] = x[v];
      if (lrow) lrow[(int64_t)r * ld + d] = x[v];
    }
  }
}

// s_sleep(1) polls of a share for the preceding block before it gives up: seconds, against the
// microseconds that a block takes.  (The launch is cooperative and the shares are the first items of
// the queue, one per workgroup: all of them run.  Where they do not all the same, the mesh is factored
// again by one workgroup.)
constexpr int32_t SHARE_POLLS = 1 << 22;

// progress is only read, and only written, where a mesh has several shares
__device__ inline int publish_failure(int32_t *progress, int shares) {
  if (shares > 1 && threadIdx.x == 0)
    __hip_atomic_store(progress, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return PF_NOT_SPD;
}

// what another share's failure means for this one
__device__ inline int progress_failed(const int32_t *progress) {
  return __hip_atomic_load(progress, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == -1 ? PF_NOT_SPD : PF_ERR_HIP;
}

// Left-looking blocked band Cholesky of one mesh by blocks of 32 columns, a share of its blocks by
// the whole workgroup.
// Per block: every wave updates its tiles of rows j0 .. j0+31+b in both column tiles with the
// previous b columns (MFMA; each A fragment feeds both column tiles; loads of the next group
// of chunks overlap the products of the current one).  Then wave 0 factors the first
// diagonal tile (L00, and L00^-T); every wave forms its column-0 tiles L(t,0) = C L00^-T;
// the owner of tile 1 publishes L10; every wave subtracts L(t,0) L10^T from its column-1
// tiles; wave 1 factors the second diagonal tile (L11, L11^-T); every wave forms
// L(t,1) = C L11^-T.  Four barriers per block.
// Bound, one mesh in shares: the chain of a block, 20 us (24,640 equations, b = 350: 15.6 ms for
// 770 blocks; 84 ms with its two solves before, 26 now); many meshes: the largest one's chain and the
// stream of the previous b columns that every block rereads.
template <int BT, bool MF, int MAXT>
__device__ __forceinline__ int factor_mesh(const DMesh &M, double *band, double *__restrict__ lrow, int share,
                                           int shares, int32_t *progress, int32_t polls_max, double *sL,
                                           double *sLi, double *sC, int32_t *sflag) {
  constexpr int W = BT / 64;
  constexpr int U = MAXT <= 4 ? 4 : 2;  // chunks per group of the steady part, two groups in flight
  constexpr int UR = U;                 // chunks per group of the ramp
  const int wv = wave_id();
  const int b = M.b, npad = M.npad;
  const int64_t ld = M.ld;
  double *myC = sC + 16 * LS * wv;
  double *sLi0 = sLi, *sL10 = sLi + 16 * LS, *sLi1 = sLi + 32 * LS;
  if (threadIdx.x == 0) *sflag = 0;
  __syncthreads();
  int have = shares == 1 ? npad : 0;  // columns complete and visible to this workgroup
  // blocks until at least `want` columns are, false when the mesh has failed
  const auto columns = [&](int want) {
    if (have >= want) return true;
    __syncthreads();
    if (threadIdx.x == 0) {
      int p, polls = 0;
      while ((p = __hip_atomic_load(progress, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) >= 0 && 32 * p < want &&
             ++polls < polls_max)
        __builtin_amdgcn_s_sleep(1);
      if (p >= 0 && 32 * p < want) {  // the other shares never came: nobody may wait for this one
        p = -2;
        __hip_atomic_store(progress, -2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      sflag[1] = p;
    }
    __syncthreads();
    const int p = uniform(sflag[1]);
    have = 32 * p;
    return p >= 0;
  };
  for (int j0 = 32 * share; j0 < npad; j0 += 32 * shares) {
    const int lane = lane_id();
    const int q = lane >> 4, jl = lane & 15;
    const int rows = min(32 + b, npad - j0);  // rows j0 .. j0+rows-1 hold the block's nonzeros
    const int T = (rows + 15) >> 4;           // >= 2
    const int P = (T + W * MAXT - 1) / (W * MAXT);
    double mb0[4], mb10[4], mb1[4];  // B fragments of L00^-T, -L10^T, L11^-T (set in pass 0)
    for (int p = 0; p < P; ++p) {
      BlockGeom g{j0, b, npad, T, wv + W * MAXT * p, W, ld};
      d4 acc[MAXT][2];
#pragma unroll
      for (int i = 0; i < MAXT; ++i) {
        const int t = g.tb + W * i;
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
          const int64_t cc = j0 + 16 * ct + jl;
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int r = j0 + 16 * t + 4 * v + q;
            acc[i][ct][v] = band[cc * ld + min(max(r - (int)cc, 0), b)];  // clamped: inside the band
          }
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int r = j0 + 16 * t + 4 * v + q;
            const int d = r - (int)cc;
            if (!(t < T && r < npad && d >= 0 && d <= b)) acc[i][ct][v] = 0.0;
          }
        }
      }
      // the block's columns lo .. hi-1 so far: those complete at hand, then the others as they come
      const int c_first = max(0, j0 - b) & ~31;
      int lo = c_first;
      do {
        // wait for the next block only, and take what is there by then
        if (!columns(min(j0, max(lo + 32, have)))) return progress_failed(progress);
        const int hi = min(j0, have);
        if (g.tb < T) {
          // A[block rows, j0..j0+31] -= L[block rows, c] L[j0..j0+31, c]^T, c < j0: a ramp with
          // predicates up to cs, then the branch-free steady part
          const int clo = max(0, j0 + 16 * g.tb - b) & ~3;
          const int nt = min(MAXT, (T - 1 - g.tb) / W + 1);  // existing tiles of this wave
          const int Rl = j0 + 16 * (g.tb + W * (nt - 1));
          const int cs = Rl + 16 <= npad ? min(j0, max(clo, (max(Rl + 15, j0 + 31) - b + 3) & ~3)) : j0;
          const int re = min(cs, hi);
          const int rb = max(clo, lo);
          if (rb < re) {
            Frags<UR, MAXT> f0, f1;
            load_frags(f0, band, g, rb, re, q, jl);
            for (int c = rb; c < re; c += 8 * UR) {
              load_frags(f1, band, g, c + 4 * UR, re, q, jl);
              mfma_frags<MF>(f0, acc, g, c, re, q, jl);
              load_frags(f0, band, g, c + 8 * UR, re, q, jl);
              mfma_frags<MF>(f1, acc, g, c + 4 * UR, re, q, jl);
            }
          }
          if (hi > cs) steady_update<MF, U, MAXT>(acc, band, g, max(cs, lo), hi, nt, q, jl);
        }
        lo = hi;
      } while (lo < j0);
      if (p == 0) {
        if (wv == 0) diag_block(acc[0][0], band, lrow, ld, b, j0, sL, sLi0, sflag);
        __syncthreads();
        if (uniform(*sflag)) return publish_failure(progress, shares);
#pragma unroll
        for (int cq = 0; cq < 4; ++cq) mb0[cq] = sLi0[(4 * cq + q) * LS + jl];
      }
      // column tile 0 below the diagonal: L(t,0) = C L00^-T; tile 1 publishes L10
#pragma unroll
      for (int i = 0; i < MAXT; ++i) {
        const int t = g.tb + W * i;
        if (t >= 1 && t < T) {
          d4 x = {0.0, 0.0, 0.0, 0.0};
          tile_times<MF>(x, acc[i][0], mb0, myC);
          acc[i][0] = x;
          store_tile(x, band, lrow, ld, b, npad, j0 + 16 * t, j0);
          if (t == 1) {
#pragma unroll
            for (int v = 0; v < 4; ++v) sL10[(4 * v + q) * LS + jl] = x[v];
          }
        }
      }
      if (p == 0) {
        __syncthreads();
        // B fragment of -L10^T: B[kk][n] = -L10[n][4 cq + kk]
#pragma unroll
        for (int cq = 0; cq < 4; ++cq) mb10[cq] = -sL10[jl * LS + 4 * cq + q];
      }
      // column tile 1: C(t,1) -= L(t,0) L10^T
#pragma unroll
      for (int i = 0; i < MAXT; ++i) {
        const int t = g.tb + W * i;
        if (t >= 1 && t < T) tile_times<MF>(acc[i][1], acc[i][0], mb10, myC);
      }
      if (p == 0) {
        if (wv == 1) diag_block(acc[0][1], band, lrow, ld, b, j0 + 16, sL, sLi1, sflag);
        __syncthreads();
        if (uniform(*sflag)) return publish_failure(progress, shares);
#pragma unroll
        for (int cq = 0; cq < 4; ++cq) mb1[cq] = sLi1[(4 * cq + q) * LS + jl];
      }
      // column tile 1 below its diagonal: L(t,1) = C L11^-T
#pragma unroll
      for (int i = 0; i < MAXT; ++i) {
        const int t = g.tb + W * i;
        if (t >= 2 && t < T) {
          d4 x = {0.0, 0.0, 0.0, 0.0};
          tile_times<MF>(x, acc[i][1], mb1, myC);
          store_tile(x, band, lrow, ld, b, npad, j0 + 16 * t, j0 + 16);
        }
      }
    }
    if (shares > 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every wave's part of the block is out
    __syncthreads();
    if (shares > 1 && threadIdx.x == 0) {
      // the blocks complete in order, so the mesh stands at this one unless a share gave up meanwhile: that
      // stays (the next wait finds it), or the others would wait out their bounds one after the other
      int32_t at = j0 / 32;
      (void)__hip_atomic_compare_exchange_strong(progress, &at, j0 / 32 + 1, __ATOMIC_RELEASE, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  return PF_OK;
}

// L L^T z = w in place (w: npad entries of the mesh's work vector).  The 16 x 16 diagonal
// solves run in wave 0 with the block's L entries loaded before the serial steps.
template <int BT>
__device__ void band_solve(const DMesh &M, const double *__restrict__ band, double *__restrict__ w, double *sY) {
  const int wv = wave_id();
  const int b = M.b, npad = M.npad;
  const int64_t ld = M.ld;
  // forward: L y = w
  for (int j0 = 0; j0 < npad; j0 += 16) {
    if (wv == 0) {
      const int lane = lane_id();
      const int jr = lane & 15;
      double Lr[16];  // row jr of the diagonal block: L[j0+jr][j0+k]
#pragma unroll
      for (int k = 0; k < 16; ++k) Lr[k] = band[(int64_t)(j0 + k) * ld + min(max(jr - k, 0), b)];
#pragma unroll
      for (int k = 0; k < 16; ++k)
        if (!(k <= jr && jr - k <= b)) Lr[k] = 0.0;
      double acc = lane < 16 ? w[j0 + lane] : 0.0;
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        if (lane == k) acc /= Lr[k];
        const double yk = shfl(acc, k);
        if (lane > k && lane < 16) acc -= Lr[k] * yk;
      }
      if (lane < 16) {
        w[j0 + lane] = acc;
        sY[lane] = acc;
      }
    }
    __syncthreads();
    const int rend = min(npad, j0 + 16 + b);
    for (int r = j0 + 16 + (int)threadIdx.x; r < rend; r += BT) {
      double l[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) l[j] = band[(int64_t)(j0 + j) * ld + min(r - j0 - j, b)];  // d >= 1
      double s = 0.0;
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if (r - j0 - j <= b) s += l[j] * sY[j];
      w[r] -= s;
    }
    __syncthreads();
  }
  // backward: L^T z = y
  for (int j0 = npad - 16; j0 >= 0; j0 -= 16) {
    if (wv == 0) {
      const int lane = lane_id();
      const int jr = lane & 15;
      double Lc[16];  // column jr of the diagonal block: L[j0+k][j0+jr]
#pragma unroll
      for (int k = 0; k < 16; ++k) Lc[k] = band[(int64_t)(j0 + jr) * ld + min(max(k - jr, 0), b)];
#pragma unroll
      for (int k = 0; k < 16; ++k)
        if (!(k >= jr && k - jr <= b)) Lc[k] = 0.0;
      double acc = lane < 16 ? w[j0 + lane] : 0.0;
#pragma unroll
      for (int k = 15; k >= 0; --k) {
        if (lane == k) acc /= Lc[k];
        const double xk = shfl(acc, k);
        if (lane < k) acc -= Lc[k] * xk;
      }
      if (lane < 16) {
        w[j0 + lane] = acc;
        sY[lane] = acc;
      }
    }
    __syncthreads();
    const int ibeg = max(0, j0 - b);
    for (int i = ibeg + (int)threadIdx.x; i < j0; i += BT) {
      double l[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) l[j] = band[(int64_t)i * ld + min(j0 + j - i, b)];  // d >= 1
      double s = 0.0;
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if (j0 + j - i <= b) s += l[j] * sY[j];
      w[i] -= s;
    }
    __syncthreads();
  }
}

__global__ void k_direct_queue_reset(int32_t *q) {
  if (threadIdx.x == 0 && blockIdx.x == 0) q[0] = 0;
}

__global__ void k_direct_progress_reset(int32_t n, int32_t *__restrict__ progress, int32_t *__restrict__ status) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    progress[i] = 0;
    status[i] = PF_OK;
  }
}

__global__ void k_flag_clear(int32_t *f) {
  if (threadIdx.x == 0 && blockIdx.x == 0) f[0] = 0;
}

// mode 0: factor (the whole mesh per workgroup), then solve; 1: solve; 2: factor, in shares
template <int BT, bool MF, int MAXT>
__global__ void __launch_bounds__(BT) k_direct(DArgs a) {
  __shared__ double sL[16 * LS];
  __shared__ double sLi[48 * LS];
  __shared__ double sC[16 * LS * (BT / 64)];
  __shared__ double sY[16];
  __shared__ int32_t next, sflag[2];
  const int total = a.mode == 2 ? a.nitem : a.nmesh;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) next = atomicAdd(a.queue, 1);
    __syncthreads();
    const int32_t qi = uniform(next);
    if (qi >= total) break;
    const DItem it = a.mode == 2 ? a.item[qi] : DItem{a.order[qi], 0, 1, 0};
    const int32_t m = it.m;
    const DMesh M = a.mesh[m];
    const int64_t t0 = wall_clock64();
    double *band = a.band + M.boff;
    int st = a.mode != 1 ? factor_mesh<BT, MF, MAXT>(M, band, a.rows ? a.rows + M.boff : nullptr, it.g, it.G,
                                               a.progress + m, a.polls, sL, sLi, sC, sflag)
                         : a.status[m];
    if (a.mode == 2) {
      // the share of the last block reports for the mesh, the first one for its start
      if (threadIdx.x == 0) {
        if (st != PF_OK) a.status[m] = st;
        if (it.g == 0) a.t_raw[2 * m] = t0;
        if (it.g == (M.npad / 32 - 1) % it.G) a.t_raw[2 * m + 1] = wall_clock64();
      }
      continue;
    }
    double *w = a.w + M.woff;
    const int32_t *perm = a.perm + M.woff;
    if (st == PF_OK) {
      for (int q = threadIdx.x; q < M.npad; q += BT) w[q] = q < M.n ? a.rhs[M.d0 + perm[q]] : 0.0;
      __syncthreads();
      band_solve<BT>(M, band, w, sY);
      for (int q = threadIdx.x; q < M.n; q += BT) {
        const int64_t r = M.d0 + perm[q];
        a.x[r] = a.mode == 0 ? w[q] : a.x[r] + w[q];
      }
    } else if (a.mode == 0) {
      for (int q = threadIdx.x; q < M.n; q += BT) a.x[M.d0 + q] = 0.0;
    }
    if (threadIdx.x == 0 && a.mode == 0) {
      a.status[m] = st;
      a.t_raw[2 * m] = t0;
      a.t_raw[2 * m + 1] = wall_clock64();
    }
  }
}

// ---- triangular solves with the diagonal blocks' inverses -------------------------------
constexpr int SB = 32;      // rows per block
constexpr int SWS = 2048;   // window of the right-hand side in LDS (power of two >= SMAXB + 2 SB)
constexpr int SMAXB = 1024; // widest band

// inverse of the lower triangular diagonal blocks, one thread per column, four blocks per workgroup
__global__ void __launch_bounds__(4 * SB) k_diag_inverse(int32_t nmesh, const DMesh *__restrict__ mesh,
                                                         const int32_t *__restrict__ status,
                                                         const double *__restrict__ band, double *__restrict__ dinv) {
  __shared__ double sL[4][SB][SB + 1];
  const int32_t m = blockIdx.y;
  const DMesh M = mesh[m];
  if (status[m] != PF_OK) return;  // whole grid row
  const int blk = 4 * blockIdx.x + threadIdx.x / SB, j = threadIdx.x % SB;
  const bool live = SB * blk < M.npad;
  double(*L)[SB + 1] = sL[threadIdx.x / SB];
  if (live) {
    const double *col = band + M.boff + (int64_t)(SB * blk + j) * M.ld;
    for (int i = 0; i < SB; ++i) L[i][j] = i >= j && i - j <= M.b ? col[i - j] : 0.0;
  }
  __syncthreads();
  if (!live) return;
  double z[SB];
#pragma unroll
  for (int i = 0; i < SB; ++i) {
    double t = i == j ? 1.0 : 0.0;
#pragma unroll
    for (int k = 0; k < i; ++k) t = __builtin_fma(-L[i][k], z[k], t);
    z[i] = t / L[i][i];
  }
  double *out = dinv + (int64_t)SB * (M.woff + SB * blk);
#pragma unroll
  for (int i = 0; i < SB; ++i) out[SB * i + j] = z[i];
}

template <int CTRL>
__device__ inline double dpp_move(double x) {
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true),
                          __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true));
}

// One direction of L L^T z = w (FWD: L y = w, else L^T z = y), w in place.  Per block of 32 the
// workgroup multiplies the block of w by the inverse of the diagonal block, eight lanes per row, and
// then subtracts the block's columns (rows) from the b <= NR BT entries of w that follow (precede), NR
// per thread; their loads are issued DEPTH blocks ahead.
// Bound: what one CU streams (37 GB/s: b = 350, 90 KB per block, 2.4 us per block).  DEPTH: as many
// blocks as the registers hold (b <= 512: 3.73 ms per solve of 24,640 equations with 2, 4.08 with 1; the
// solves by blocks of 16: 11 ms).  b <= 1024: 1024 threads with one entry each (22.1 ms for 192 meshes up
// to b = 690) rather than 512 with two (24.8 ms).
template <int BT, int NR, int DEPTH, bool FWD>
__device__ __forceinline__ void band_sweep(const DMesh &M, const double *__restrict__ L,
                                           const double *__restrict__ dinv, double *__restrict__ w, double *sw,
                                           double *sY) {
  const int tid = threadIdx.x;
  const int b = M.b, npad = M.npad, nb = npad / SB;
  const int64_t ld = M.ld;
  // entry t = tid of the panel beside block j0: row j0 + SB + t (FWD) or column j0 - 1 - t; its L
  // values for the block's columns (rows) j lie at distance SB + t - j or j + 1 + t, contiguous over
  // t.  Those outside the band (distance > b) read a neighbouring entry, at most SB past the
  // mesh's last (the buffers end with as many), and are dropped.
  double l[DEPTH][NR][SB];
  const auto panel = [&](int j0, double (&to)[NR][SB]) {
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      uint32_t tc = (uint32_t)max(min(tid + k * BT, b - 1), 0);
      asm volatile("" : "+v"(tc));  // keeps the lane's part of the address apart from the scalar part
      const double *p = L + (int64_t)j0 * ld + (FWD ? SB : 1);
#pragma unroll
      for (int j = 0; j < SB; ++j, p += FWD ? ld - 1 : ld + 1) to[k][j] = at(p, tc);
    }
  };
  double di[4];
  const int mi = tid >> 3, ms = (tid & 7) * 4;  // row of the product, first of this lane's four terms
  const auto inverse = [&](int J) {
    if (mi < SB)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        di[k] = FWD ? dinv[(int64_t)SB * (SB * J + mi) + ms + k] : dinv[(int64_t)SB * (SB * J + ms + k) + mi];
  };
  const auto entry = [&](int J, int t) { return FWD ? SB * J + t : npad - 1 - (nb - 1 - J) * SB - t; };
  // the window: the first block and the b entries beside it; SB more enter with every block
  const int J0 = FWD ? 0 : nb - 1;
  for (int t = tid; t < SB + b; t += BT) {
    const int i = entry(J0, t);
    if (i >= 0 && i < npad) sw[i & (SWS - 1)] = w[i];
  }
#pragma unroll
  for (int k = 0; k < DEPTH; ++k) panel(SB * (FWD ? min(k, nb - 1) : max(nb - 1 - k, 0)), l[k]);
  inverse(J0);
  const auto block = [&](int step, double (&lb)[NR][SB]) {
    const int J = FWD ? step : nb - 1 - step;
    const int j0 = SB * J;
    const int in = entry(J, SB + b + tid);  // enters the window with the next block
    double win = 0.0;
    const bool enter = tid < SB && in >= 0 && in < npad;
    if (enter) win = w[in];
    __syncthreads();  // the block's entries of w are final
    if (mi < SB) {
      double p = 0.0;
#pragma unroll
      for (int k = 0; k < 4; ++k) p = __builtin_fma(di[k], sw[(j0 + ms + k) & (SWS - 1)], p);
      p += dpp_move<0xb1>(p);   // quad_perm 1,0,3,2
      p += dpp_move<0x4e>(p);   // quad_perm 2,3,0,1
      p += dpp_move<0x141>(p);  // row_half_mirror: the other four of the eight
      if ((tid & 7) == 0) {
        sY[mi] = p;
        w[j0 + mi] = p;
      }
    }
    if (step + 1 < nb) inverse(FWD ? J + 1 : J - 1);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      int t = tid + k * BT;
      asm volatile("" : "+v"(t));  // else the masks below are kept over the blocks, and spilled
      double s0 = 0.0, s1 = 0.0;
      if (64 * wave_id() + k * BT + 64 + SB <= b) {  // the whole wave inside the band
#pragma unroll
        for (int j = 0; j < SB; j += 2) {
          s0 = __builtin_fma(lb[k][j], sY[j], s0);
          s1 = __builtin_fma(lb[k][j + 1], sY[j + 1], s1);
        }
      } else {
#pragma unroll
        for (int j = 0; j < SB; j += 2) {
          s0 = __builtin_fma((FWD ? SB + t - j : j + 1 + t) <= b ? lb[k][j] : 0.0, sY[j], s0);
          s1 = __builtin_fma((FWD ? SB + t - j - 1 : j + 2 + t) <= b ? lb[k][j + 1] : 0.0, sY[j + 1], s1);
        }
      }
      const int i = entry(J, SB + t);
      if (t < b && i >= 0 && i < npad) sw[i & (SWS - 1)] -= s0 + s1;
    }
    if (enter) sw[in & (SWS - 1)] = win;
    panel(SB * (FWD ? min(J + DEPTH, nb - 1) : max(J - DEPTH, 0)), lb);  // past the end: the last once more
  };
  for (int step = 0; step < nb; step += DEPTH) {
#pragma unroll
    for (int k = 0; k < DEPTH; ++k)
      if (step + k < nb) block(step + k, l[k]);
  }
  __syncthreads();
}

template <int BT, int NR, int DEPTH>
__global__ void __launch_bounds__(BT) k_band_solve(DArgs a) {
  __shared__ double sw[SWS];
  __shared__ double sY[SB];
  __shared__ int32_t next;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) next = atomicAdd(a.queue, 1);
    __syncthreads();
    const int32_t qi = uniform(next);
    if (qi >= a.nmesh) break;
    const int32_t m = a.order[qi];
    const DMesh M = a.mesh[m];
    double *w = a.w + M.woff;
    const int32_t *perm = a.perm + M.woff;
    if (a.status[m] == PF_OK) {
      for (int q = threadIdx.x; q < M.npad; q += BT) w[q] = q < M.n ? a.rhs[M.d0 + perm[q]] : 0.0;
      __syncthreads();
      const double *dinv = a.dinv + (int64_t)SB * M.woff;
      band_sweep<BT, NR, DEPTH, true>(M, a.band + M.boff, dinv, w, sw, sY);
      band_sweep<BT, NR, DEPTH, false>(M, a.rows + M.boff, dinv, w, sw, sY);
      for (int q = threadIdx.x; q < M.n; q += BT) {
        const int64_t r = M.d0 + perm[q];
        a.x[r] = a.mode == 0 ? w[q] : a.x[r] + w[q];
      }
    } else if (a.mode == 0) {
      for (int q = threadIdx.x; q < M.n; q += BT) a.x[M.d0 + q] = 0.0;
    }
    if (threadIdx.x == 0 && a.mode == 0) a.t_raw[2 * m + 1] = wall_clock64();
  }
}

__global__ void k_band_zero(double *__restrict__ band, int64_t count) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count; i += stride) band[i] = 0.0;
}

// lower triangle of P A P^T into the band: one SUB-lane subgroup per row
template <int SUB>
__global__ void __launch_bounds__(256) k_band_scatter(int64_t n, const int64_t *__restrict__ row_ptr,
                                                      const int32_t *__restrict__ col_idx,
                                                      const double *__restrict__ val, const DMesh *__restrict__ mesh,
                                                      const int32_t *__restrict__ dmesh,
                                                      const int32_t *__restrict__ bidx, double *__restrict__ band,
                                                      int32_t *__restrict__ bad) {
  const int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t r = g / SUB;
  const int lane = (int)(g % SUB);
  if (r >= n) return;
  const int32_t m = dmesh[r];
  const DMesh M = mesh[m];
  const int64_t pr = bidx[r];
  const int64_t e = row_ptr[r + 1] - 1;
  for (int64_t k = row_ptr[r] - 1 + lane; k < e; k += SUB) {
    const int64_t c = col_idx[k] - 1;
    const int64_t pc = bidx[c];
    // an entry outside the mesh or the analysed band means a stale analysis: flag, never write
    if (dmesh[c] != m || pr - pc > M.b || pc - pr > M.b) {
      atomicOr(bad, 1);
    } else if (pr >= pc) {
      band[M.boff + pc * M.ld + (pr - pc)] = val[k];
    }
  }
}

// unit diagonal of the padding rows n .. npad-1 of every mesh
__global__ void k_band_pad(int32_t nmesh, const DMesh *__restrict__ mesh, double *__restrict__ band) {
  const int32_t m = blockIdx.x;
  if (m >= nmesh) return;
  const DMesh M = mesh[m];
  for (int q = M.n + (int)threadIdx.x; q < M.npad; q += blockDim.x) band[M.boff + (int64_t)q * M.ld] = 1.0;
}

// r = rhs - y over every mesh's rows, and per mesh (|r|^2, |rhs|^2); one workgroup per mesh
__global__ void __launch_bounds__(256) k_direct_resid(int32_t nmesh, const DMesh *__restrict__ mesh,
                                                      const double *__restrict__ rhs, const double *__restrict__ y,
                                                      double *__restrict__ r, double *__restrict__ norms) {
  __shared__ double sh[2][4];
  const int32_t m = blockIdx.x;
  if (m >= nmesh) return;
  const DMesh M = mesh[m];
  double t0 = 0.0, t1 = 0.0;
  for (int64_t i = M.d0 + threadIdx.x; i < M.d0 + M.n; i += 256) {
    const double bi = rhs[i];
    const double ri = bi - y[i];
    r[i] = ri;
    t0 += ri * ri;
    t1 += bi * bi;
  }
  for (int o = 32; o > 0; o >>= 1) {
    t0 += __shfl_xor(t0, o, 64);
    t1 += __shfl_xor(t1, o, 64);
  }
  const int wv = wave_id();
  if ((threadIdx.x & 63) == 0) {
    sh[0][wv] = t0;
    sh[1][wv] = t1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    norms[2 * m] = sh[0][0] + sh[0][1] + sh[0][2] + sh[0][3];
    norms[2 * m + 1] = sh[1][0] + sh[1][1] + sh[1][2] + sh[1][3];
  }
}

// node (DOF group) neighbours from a DOF=3 blocked CRS: every third column of row 3i
__global__ void k_group_cols(int64_t nn, const int64_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx,
                             const int64_t *__restrict__ goff, int32_t *__restrict__ gcol) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= nn) return;
  const int64_t r0 = row_ptr[3 * i] - 1;
  const int64_t m = goff[i + 1] - goff[i];
  for (int64_t t = 0; t < m; ++t) gcol[goff[i] + t] = (col_idx[r0 + 3 * t] - 1) / 3;
}

// ---------------------------------------------------------------------------------
// orderings (host)

struct LocalGraph {
  int64_t g0 = 0, ng = 0;                 // groups g0 .. g0+ng-1
  const int64_t *off = nullptr;           // global group adjacency offsets
  const int32_t *adj = nullptr;           // global group ids
};

int64_t bandwidth_of(const LocalGraph &G, const std::vector<int32_t> &pos) {
  int64_t bw = 0;
  for (int64_t i = 0; i < G.ng; ++i) {
    const int64_t pi = pos[i];
    for (int64_t k = G.off[G.g0 + i]; k < G.off[G.g0 + i + 1]; ++k) {
      const int64_t j = G.adj[k] - G.g0;
      if (j < 0 || j >= G.ng) continue;  // outside the mesh (not expected in a checked partition)
      const int64_t d = pi > pos[j] ? pi - pos[j] : pos[j] - pi;
      if (d > bw) bw = d;
    }
  }
  return bw;
}

// reverse Cuthill-McKee from a pseudo-peripheral start (George-Liu), components in turn
std::vector<int32_t> rcm_order(const LocalGraph &G) {
  const int64_t n = G.ng;
  std::vector<int32_t> deg(n);
  for (int64_t i = 0; i < n; ++i) deg[i] = (int32_t)(G.off[G.g0 + i + 1] - G.off[G.g0 + i]);
  std::vector<int32_t> order;
  order.reserve(n);
  std::vector<char> done(n, 0);
  std::vector<int32_t> level(n, -1), queue;
  queue.reserve(n);
  auto bfs_levels = [&](int32_t s, int32_t &last_first, int32_t &nlev) {
    queue.clear();
    queue.push_back(s);
    level[s] = 0;
    size_t h = 0;
    while (h < queue.size()) {
      const int32_t u = queue[h++];
      for (int64_t k = G.off[G.g0 + u]; k < G.off[G.g0 + u + 1]; ++k) {
        const int64_t v = G.adj[k] - G.g0;
        if (v < 0 || v >= n || done[v] || level[v] >= 0) continue;
        level[v] = level[u] + 1;
        queue.push_back((int32_t)v);
      }
    }
    nlev = level[queue.back()] + 1;
    last_first = queue.back();
    int32_t best = queue.back();
    for (size_t t = queue.size(); t-- > 0;) {
      const int32_t u = queue[t];
      if (level[u] != nlev - 1) break;
      if (deg[u] < deg[best]) best = u;
    }
    last_first = best;
    for (int32_t u : queue) level[u] = -1;
  };
  for (;;) {
    int32_t s = -1;
    for (int64_t i = 0; i < n; ++i)
      if (!done[i] && (s < 0 || deg[i] < deg[s])) s = (int32_t)i;
    if (s < 0) break;
    int32_t cand = s, nlev = 0, nlev2 = 0;
    bfs_levels(s, cand, nlev);
    for (int it = 0; it < 8; ++it) {
      int32_t c2 = cand;
      bfs_levels(cand, c2, nlev2);
      if (nlev2 <= nlev) break;
      s = cand;
      nlev = nlev2;
      cand = c2;
    }
    // Cuthill-McKee from s: neighbours by increasing degree
    const size_t first = order.size();
    order.push_back(s);
    done[s] = 1;
    std::vector<int32_t> nb;
    for (size_t h = first; h < order.size(); ++h) {
      const int32_t u = order[h];
      nb.clear();
      for (int64_t k = G.off[G.g0 + u]; k < G.off[G.g0 + u + 1]; ++k) {
        const int64_t v = G.adj[k] - G.g0;
        if (v < 0 || v >= n || done[v]) continue;
        done[v] = 1;
        nb.push_back((int32_t)v);
      }
      std::stable_sort(nb.begin(), nb.end(), [&](int32_t x, int32_t y) { return deg[x] < deg[y]; });
      order.insert(order.end(), nb.begin(), nb.end());
    }
  }
  std::reverse(order.begin(), order.end());
  return order;
}

struct MeshOrder {
  std::vector<int32_t> order;  // new position -> local group
  int64_t bw = 0;              // in groups
  int32_t kind = 0;            // 0 natural, 1 RCM, 2/3/4 coordinate sort with x/y/z primary
};

MeshOrder best_order(const LocalGraph &G, const double *coords, int64_t ncoord) {
  MeshOrder best;
  best.order.resize(G.ng);
  std::iota(best.order.begin(), best.order.end(), 0);
  std::vector<int32_t> pos(G.ng);
  auto eval = [&](const std::vector<int32_t> &ord) {
    for (int64_t k = 0; k < G.ng; ++k) pos[ord[k]] = (int32_t)k;
    return bandwidth_of(G, pos);
  };
  best.bw = eval(best.order);
  best.kind = 0;
  {
    std::vector<int32_t> o = rcm_order(G);
    const int64_t bw = eval(o);
    if (bw < best.bw) {
      best.bw = bw;
      best.order = std::move(o);
      best.kind = 1;
    }
  }
  if (coords) {
    double lo[3], hi[3];
    for (int d = 0; d < 3; ++d) {
      lo[d] = 1e300;
      hi[d] = -1e300;
      for (int64_t i = 0; i < G.ng; ++i) {
        const double v = coords[d * ncoord + G.g0 + i];
        lo[d] = std::min(lo[d], v);
        hi[d] = std::max(hi[d], v);
      }
    }
    for (int p = 0; p < 3; ++p) {
      int s = (p + 1) % 3, t = (p + 2) % 3;
      if (hi[t] - lo[t] > hi[s] - lo[s]) std::swap(s, t);
      std::vector<int32_t> o(G.ng);
      std::iota(o.begin(), o.end(), 0);
      auto key = [&](int32_t i, int d) { return coords[d * ncoord + G.g0 + i]; };
      std::stable_sort(o.begin(), o.end(), [&](int32_t x, int32_t y) {
        if (key(x, p) != key(y, p)) return key(x, p) < key(y, p);
        if (key(x, s) != key(y, s)) return key(x, s) < key(y, s);
        return key(x, t) < key(y, t);
      });
      const int64_t bw = eval(o);
      if (bw < best.bw) {
        best.bw = bw;
        best.order = std::move(o);
        best.kind = 2 + p;
      }
    }
  }
  return best;
}

}  // namespace

// ---------------------------------------------------------------------------------

struct DirectWork {
  // analysis (sparsity pattern and partition)
  uint64_t pattern_key = 0;
  std::vector<int64_t> dof_off;
  int32_t nmesh = 0;
  int32_t group = 1;
  int64_t n = 0;
  std::vector<DMesh> hmesh;
  std::vector<int32_t> kinds;
  std::vector<int32_t> hperm;  // band index -> local DOF, per mesh at woff
  DevBuf<DMesh> mesh;
  DevBuf<int32_t> perm, bidx, dmesh, order, queue, status, flag;
  DevBuf<int64_t> t_raw;
  DevBuf<double> band, w, r, y, norms;
  DevBuf<double> rows, dinv;   // L row by row and the diagonal blocks' inverses (fast solves)
  bool fast_solve = false;     // both are kept
  std::vector<DItem> hitem;    // shares of the factorizations, largest mesh first
  DevBuf<DItem> item;
  DevBuf<int32_t> progress;
  bool shared = false;         // some mesh has more than one
  int32_t maxb = 0, maxpad = 0;
  int64_t band_entries = 0, work_entries = 0;
  double analyse_ms = 0.0;
  // factor held in band: the matrix version it was computed from (0: none)
  uint64_t factor_version = 0;
  bool factor_ok = false;
};

void pf_direct_work_destroy(DirectWork *d) { delete d; }

void pf_direct_invalidate(DirectWork *d) {
  if (d) d->factor_version = 0;
}

int pf_direct_analyse(pf_ctx *ctx, DirectWork **pd, int64_t n, const int64_t *row_ptr, const int32_t *col_idx,
                      int32_t nmesh, const int64_t *dof_off, const double *coords_dev, int64_t ncoord,
                      uint64_t pattern_key) {
  if (nmesh < 1 || n < 1 || dof_off[0] != 0 || dof_off[nmesh] != n) {
    pf_set_error("direct: meshes must partition the %lld DOFs", (long long)n);
    return PF_INVALID;
  }
  for (int32_t m = 0; m < nmesh; ++m)
    if (dof_off[m + 1] <= dof_off[m]) {
      pf_set_error("direct: mesh %d is empty", m);
      return PF_INVALID;
    }
  if (!*pd) *pd = new DirectWork();
  DirectWork *D = *pd;
  if (D->pattern_key == pattern_key && D->nmesh == nmesh && D->n == n &&
      (int64_t)D->dof_off.size() == nmesh + 1 && std::equal(D->dof_off.begin(), D->dof_off.end(), dof_off))
    return PF_OK;
  const auto tstart = std::chrono::steady_clock::now();
  D->pattern_key = 0;
  D->factor_version = 0;
  D->nmesh = 0;
  PF_CHECK(D->flag.ensure(1));
  int blocked3 = 0;
  if (n % 3 == 0) PF_CHECK(pf_block_structure_check(ctx, n, row_ptr, col_idx, n / 3, D->flag.p, &blocked3));
  const int32_t g = blocked3 ? 3 : 1;
  for (int32_t m = 0; m <= nmesh; ++m)
    if (dof_off[m] % g != 0) {
      pf_set_error("direct: mesh offsets must be whole DOF=3 blocks");
      return PF_INVALID;
    }
  const int64_t ng = n / g;
  // group adjacency on the host
  std::vector<int64_t> hrp(n + 1);
  PF_HIP(hipMemcpyAsync(hrp.data(), row_ptr, sizeof(int64_t) * (n + 1), hipMemcpyDeviceToHost, ctx->stream));
  PF_HIP(hipStreamSynchronize(ctx->stream));
  std::vector<int64_t> goff(ng + 1, 0);
  std::vector<int32_t> gadj;
  if (g == 3) {
    for (int64_t i = 0; i < ng; ++i) goff[i + 1] = goff[i] + (hrp[3 * i + 1] - hrp[3 * i]) / 3;
    DevBuf<int64_t> doff;
    DevBuf<int32_t> dcol;
    PF_CHECK(doff.ensure(ng + 1));
    PF_CHECK(dcol.ensure(std::max<int64_t>(goff[ng], 1)));
    PF_HIP(hipMemcpyAsync(doff.p, goff.data(), sizeof(int64_t) * (ng + 1), hipMemcpyHostToDevice, ctx->stream));
    k_group_cols<<<pf_blocks(ng, 256, INT32_MAX), 256, 0, ctx->stream>>>(ng, row_ptr, col_idx, doff.p, dcol.p);
    PF_HIP(hipGetLastError());
    gadj.resize(goff[ng]);
    PF_HIP(hipMemcpyAsync(gadj.data(), dcol.p, sizeof(int32_t) * goff[ng], hipMemcpyDeviceToHost, ctx->stream));
    PF_HIP(hipStreamSynchronize(ctx->stream));
  } else {
    const int64_t nnz = hrp[n] - 1;
    gadj.resize(nnz);
    PF_HIP(hipMemcpyAsync(gadj.data(), col_idx, sizeof(int32_t) * nnz, hipMemcpyDeviceToHost, ctx->stream));
    PF_HIP(hipStreamSynchronize(ctx->stream));
    for (int64_t i = 0; i <= n; ++i) goff[i] = hrp[i] - 1;
    for (auto &c : gadj) c -= 1;
  }
  std::vector<double> coords;
  if (coords_dev && g == 3 && ncoord == ng) {
    coords.resize(3 * ncoord);
    PF_HIP(hipMemcpyAsync(coords.data(), coords_dev, sizeof(double) * 3 * ncoord, hipMemcpyDeviceToHost,
                          ctx->stream));
    PF_HIP(hipStreamSynchronize(ctx->stream));
  }
  // per-mesh orderings, meshes spread over host threads
  std::vector<MeshOrder> ord(nmesh);
  {
    unsigned nt = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
    nt = (unsigned)std::min<int64_t>(nt, nmesh);
    std::vector<std::thread> th;
    std::atomic<int32_t> next{0};
    for (unsigned t = 0; t < nt; ++t)
      th.emplace_back([&]() {
        for (;;) {
          const int32_t m = next.fetch_add(1);
          if (m >= nmesh) break;
          LocalGraph G;
          G.g0 = dof_off[m] / g;
          G.ng = (dof_off[m + 1] - dof_off[m]) / g;
          G.off = goff.data();
          G.adj = gadj.data();
          ord[m] = best_order(G, coords.empty() ? nullptr : coords.data(), ncoord);
        }
      });
    for (auto &t : th) t.join();
  }
  // band layout
  D->hmesh.assign(nmesh, DMesh{});
  D->kinds.assign(nmesh, 0);
  int64_t boff = 0, woff = 0;
  for (int32_t m = 0; m < nmesh; ++m) {
    DMesh &M = D->hmesh[m];
    const int64_t nm = dof_off[m + 1] - dof_off[m];
    if (nm > (int64_t)INT32_MAX - 16) {
      pf_set_error("direct: mesh %d has %lld DOFs, more than the band kernels index", m, (long long)nm);
      return PF_INVALID;
    }
    M.d0 = dof_off[m];
    M.n = (int32_t)nm;
    M.npad = (int32_t)((nm + 31) / 32 * 32);
    M.b = (int32_t)(g * ord[m].bw + g - 1);
    M.ld = (M.b + 2) & ~1;
    M.boff = boff;
    M.woff = woff;
    boff += (int64_t)M.npad * M.ld;
    woff += M.npad;
    D->kinds[m] = ord[m].kind;
  }
  size_t free_b = 0, total_b = 0;
  PF_HIP(hipMemGetInfo(&free_b, &total_b));
  const double need = 8.0 * (double)(boff + 2 * SB);
  const double have = (double)free_b + 8.0 * (double)D->band.n;
  if (need > have - 2.0e9) {
    pf_set_error("direct: the band factors need %.2f GB of device memory, %.2f GB are free", need * 1e-9,
                 have * 1e-9);
    return PF_ERR_NOMEM;
  }
  D->maxb = D->maxpad = 0;
  for (const DMesh &M : D->hmesh) {
    D->maxb = std::max(D->maxb, M.b);
    D->maxpad = std::max(D->maxpad, M.npad);
  }
  // the second copy of the factor and the inverses, where they fit beside the band
  D->fast_solve = D->maxb <= SMAXB && nmesh <= 65535 &&
                  need * 2.0 + 8.0 * SB * (double)woff <=
                      have + 8.0 * ((double)D->rows.n + (double)D->dinv.n) - 4.0e9;
  if (D->fast_solve) {
    PF_CHECK(D->rows.ensure(std::max<int64_t>(boff, 1) + 2 * SB));
    PF_CHECK(D->dinv.ensure(std::max<int64_t>(SB * woff, 1)));
  } else {
    D->rows.release();
    D->dinv.release();
  }
  D->hperm.assign(woff, 0);
  std::vector<int32_t> hbidx(n), hdm(n);
  for (int32_t m = 0; m < nmesh; ++m) {
    const DMesh &M = D->hmesh[m];
    const std::vector<int32_t> &o = ord[m].order;
    for (int64_t k = 0; k < (int64_t)o.size(); ++k)
      for (int d = 0; d < g; ++d) {
        const int32_t q = (int32_t)(g * k + d);
        const int32_t loc = g * o[k] + d;
        D->hperm[M.woff + q] = loc;
        hbidx[M.d0 + loc] = q;
        hdm[M.d0 + loc] = m;
      }
  }
  std::vector<int32_t> qorder(nmesh);
  std::iota(qorder.begin(), qorder.end(), 0);
  std::stable_sort(qorder.begin(), qorder.end(), [&](int32_t x, int32_t y) {
    const DMesh &a = D->hmesh[x], &b = D->hmesh[y];
    return (double)a.npad * a.b * a.b > (double)b.npad * b.b * b.b;
  });
  // shares: a mesh takes as many workgroups as keep it from outlasting the others (all the work over
  // all the CUs), up to what its blocks can use: the time of a block on one workgroup (measured:
  // 50 us at b = 350, 110 us at b = 690) over the time that passes between one block's columns and
  // the next's (the last update, two diagonal tiles, the exchange: 20 us measured with many shares),
  // and one.  More shares only take CUs from the other meshes: 24,640 equations of b = 350 took 38.8,
  // 20.5, 15.6 and 15.6 ms with 1, 2, 4 and 6; 192 meshes up to b = 690, whole passes, 339, 241, 182, 171
  // and 187 ms with up to 1, 2, 4, 6 and 10.
  D->hitem.clear();
  D->shared = false;
  {
    const auto block_us = [](const DMesh &M) { return 32.0 * M.b * (double)M.b / 190.0e3 + 29.0; };
    const auto work = [&](const DMesh &M) { return block_us(M) * (M.npad / 32); };
    double sum = 0.0;
    for (const DMesh &M : D->hmesh) sum += work(M);
    const double even = sum / ctx->num_cus;
    for (int32_t m : qorder) {
      const DMesh &M = D->hmesh[m];
      // all shares of a mesh among the items that the resident workgroups take first, so that no
      // share ever waits for one that is still in the queue
      const double room = std::max(1.0, (double)ctx->num_cus - (double)D->hitem.size());
      const double most = std::min(room, std::min(std::min(16.0, block_us(M) / 16.0 + 1.0), M.npad / 32.0));
      const int G = std::max(1, (int)std::min(std::ceil(work(M) / even), std::floor(most)));
      for (int g = 0; g < G; ++g) D->hitem.push_back(DItem{m, g, G, 0});
      D->shared = D->shared || G > 1;
    }
  }
  PF_CHECK(D->item.ensure(D->hitem.size()));
  PF_CHECK(D->progress.ensure(nmesh));
  PF_HIP(hipMemcpyAsync(D->item.p, D->hitem.data(), sizeof(DItem) * D->hitem.size(), hipMemcpyHostToDevice,
                        ctx->stream));
  PF_CHECK(D->band.ensure(std::max<int64_t>(boff, 1) + 2 * SB));
  PF_CHECK(D->mesh.ensure(nmesh));
  PF_CHECK(D->perm.ensure(std::max<int64_t>(woff, 1)));
  PF_CHECK(D->w.ensure(std::max<int64_t>(woff, 1)));
  PF_CHECK(D->bidx.ensure(n));
  PF_CHECK(D->dmesh.ensure(n));
  PF_CHECK(D->order.ensure(nmesh));
  PF_CHECK(D->queue.ensure(1));
  PF_CHECK(D->status.ensure(nmesh));
  PF_CHECK(D->t_raw.ensure(2 * (size_t)nmesh));
  PF_CHECK(D->norms.ensure(2 * (size_t)nmesh));
  PF_CHECK(D->r.ensure(n + 1));
  PF_CHECK(D->y.ensure(n + 1));
  PF_HIP(hipMemcpyAsync(D->mesh.p, D->hmesh.data(), sizeof(DMesh) * nmesh, hipMemcpyHostToDevice, ctx->stream));
  PF_HIP(hipMemcpyAsync(D->perm.p, D->hperm.data(), sizeof(int32_t) * woff, hipMemcpyHostToDevice, ctx->stream));
  PF_HIP(hipMemcpyAsync(D->bidx.p, hbidx.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, ctx->stream));
  PF_HIP(hipMemcpyAsync(D->dmesh.p, hdm.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, ctx->stream));
  PF_HIP(hipMemcpyAsync(D->order.p, qorder.data(), sizeof(int32_t) * nmesh, hipMemcpyHostToDevice, ctx->stream));
  PF_HIP(hipStreamSynchronize(ctx->stream));
  D->band_entries = boff;
  D->work_entries = woff;
  D->group = g;
  D->n = n;
  D->dof_off.assign(dof_off, dof_off + nmesh + 1);
  D->nmesh = nmesh;
  D->pattern_key = pattern_key;
  D->analyse_ms =
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - tstart).count();
  return PF_OK;
}

namespace {
// from now on (until the next analysis) every mesh is factored by one workgroup
int whole_meshes(pf_ctx *ctx, DirectWork *D) {
  std::vector<DItem> whole;
  for (const DItem &it : D->hitem)
    if (it.g == 0) whole.push_back(DItem{it.m, 0, 1, 0});
  D->hitem = whole;
  D->shared = false;
  PF_HIP(hipMemcpyAsync(D->item.p, D->hitem.data(), sizeof(DItem) * D->hitem.size(), hipMemcpyHostToDevice,
                        ctx->stream));
  return PF_OK;
}

int launch_direct(pf_ctx *ctx, DirectWork *D, int mode, const double *rhs, double *x, bool mfma) {
  DArgs a{};
  a.mesh = D->mesh.p;
  a.order = D->order.p;
  a.queue = D->queue.p;
  a.nmesh = D->nmesh;
  a.mode = mode;
  a.band = D->band.p;
  a.perm = D->perm.p;
  a.w = D->w.p;
  a.rhs = rhs;
  a.x = x;
  a.status = D->status.p;
  a.t_raw = D->t_raw.p;
  a.progress = D->progress.p;
  a.polls = ctx->polls > 0 ? ctx->polls : SHARE_POLLS;
  a.rows = D->fast_solve ? D->rows.p : nullptr;
  a.dinv = D->fast_solve ? D->dinv.p : nullptr;
  // two workgroups per CU at most; no more workgroups than meshes
  const int grid = std::max(1, std::min(D->nmesh, 2 * ctx->num_cus));
  const auto solve = [&]() -> int {
    k_direct_queue_reset<<<1, 64, 0, ctx->stream>>>(D->queue.p);
    if (D->maxb <= 256)
      k_band_solve<256, 1, 2><<<grid, 256, 0, ctx->stream>>>(a);
    else if (D->maxb <= 512)
      k_band_solve<512, 1, 2><<<grid, 512, 0, ctx->stream>>>(a);
    else
      k_band_solve<1024, 1, 1><<<grid, 1024, 0, ctx->stream>>>(a);
    PF_HIP(hipGetLastError());
    return PF_OK;
  };
  if (D->fast_solve && mode == 1) return solve();
  // tiles of the widest block over the waves
  const int tiles = (32 + D->maxb + 15) / 16;
  const void *kernel;
  if (!mfma) kernel = (const void *)k_direct<DBT, false, 2>;
  else if (tiles <= 2 * (DBT / 64)) kernel = (const void *)k_direct<DBT, true, 2>;
  else if (tiles <= 4 * (DBT / 64)) kernel = (const void *)k_direct<DBT, true, 4>;
  else kernel = (const void *)k_direct<DBT, true, 6>;
  k_direct_queue_reset<<<1, 64, 0, ctx->stream>>>(D->queue.p);
  PF_HIP(hipGetLastError());
  if (D->fast_solve) {
    a.mode = 2;
    a.item = D->item.p;
    a.nitem = (int32_t)D->hitem.size();
    k_direct_progress_reset<<<pf_blocks(D->nmesh, 256), 256, 0, ctx->stream>>>(D->nmesh, D->progress.p, D->status.p);
    PF_HIP(hipGetLastError());
    if (D->shared) {
      // the shares of a mesh wait for each other: all workgroups resident
      const int g2 = std::min((int)D->hitem.size(), ctx->num_cus);
      void *args[] = {&a};
      if (pf_launch_together(ctx, kernel, (unsigned)g2, DBT, args, 0) != hipSuccess) {
        (void)hipGetLastError();  // e.g. fewer CUs available to this process
        PF_CHECK(whole_meshes(ctx, D));
        a.nitem = (int32_t)D->hitem.size();
      }
    }
  }
  if (a.mode != 2 || !D->shared) {
    void *args[] = {&a};
    PF_HIP(hipLaunchKernel(kernel, dim3(grid), dim3(DBT), args, 0, ctx->stream));
  }
  ctx->forms.direct_shares = 1;
  if (D->fast_solve)
    for (const DItem &it : D->hitem) ctx->forms.direct_shares = std::max(ctx->forms.direct_shares, it.G);
  if (D->fast_solve) {
    const unsigned per = (unsigned)((D->maxpad / SB + 3) / 4);
    k_diag_inverse<<<dim3(per, (unsigned)D->nmesh), 4 * SB, 0, ctx->stream>>>(D->nmesh, D->mesh.p, D->status.p,
                                                                             D->band.p, D->dinv.p);
    a.mode = 0;
    PF_CHECK(solve());
  }
  return PF_OK;
}

// r = rhs - A x and the per-mesh norms
int residual(pf_ctx *ctx, DirectWork *D, int64_t n, const int64_t *row_ptr, const int32_t *col_idx,
             const double *val, double avg_row, const double *rhs, const double *x) {
  PF_CHECK(pf_spmv_crs_launch<double>(ctx, n, row_ptr, col_idx, val, x, D->y.p, avg_row));
  k_direct_resid<<<D->nmesh, 256, 0, ctx->stream>>>(D->nmesh, D->mesh.p, rhs, D->y.p, D->r.p, D->norms.p);
  PF_HIP(hipGetLastError());
  return PF_OK;
}
}  // namespace

int pf_direct_solve_device(pf_ctx *ctx, DirectWork *D, int64_t n, const int64_t *row_ptr, const int32_t *col_idx,
                           const double *val, int64_t nnz, const double *rhs, double *x, uint64_t mat_version,
                           int32_t refine, int32_t mfma, pf_batch_mesh_stats *mesh_stats, pf_stats *total) {
  if (!D || D->nmesh < 1 || D->n != n) {
    pf_set_error("direct: no analysis for this system");
    return PF_INVALID;
  }
  if (refine < 0 || refine > 100) {
    pf_set_error("direct: refinement steps must be in [0, 100]");
    return PF_INVALID;
  }
  const double avg_row = n > 0 ? (double)nnz / (double)n : 1.0;
  float setup_ms = 0.f, solve_ms = 0.f;
  const bool refactor = D->factor_version != mat_version || mat_version == 0;
  PF_HIP(hipEventRecord(ctx->ev0, ctx->stream));
  if (refactor) {
    D->factor_version = 0;
    k_band_zero<<<pf_blocks(D->band_entries, 256, 8 * 2048), 256, 0, ctx->stream>>>(D->band.p, D->band_entries);
    PF_HIP(hipGetLastError());
    k_flag_clear<<<1, 64, 0, ctx->stream>>>(D->flag.p);
    k_band_scatter<16><<<pf_blocks(n * 16, 256, INT32_MAX), 256, 0, ctx->stream>>>(
        n, row_ptr, col_idx, val, D->mesh.p, D->dmesh.p, D->bidx.p, D->band.p, D->flag.p);
    PF_HIP(hipGetLastError());
    int32_t bad = 0;
    PF_HIP(hipMemcpyAsync(&bad, D->flag.p, sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
    PF_HIP(hipStreamSynchronize(ctx->stream));
    if (bad) {
      pf_set_error("direct: the matrix has entries outside the analysed meshes or band (pattern changed?)");
      return PF_INVALID;
    }
    k_band_pad<<<D->nmesh, 64, 0, ctx->stream>>>(D->nmesh, D->mesh.p, D->band.p);
    PF_HIP(hipGetLastError());
  }
  PF_HIP(hipEventRecord(ctx->ev1, ctx->stream));
  PF_HIP(hipEventSynchronize(ctx->ev1));
  PF_HIP(hipEventElapsedTime(&setup_ms, ctx->ev0, ctx->ev1));
  PF_HIP(hipEventRecord(ctx->ev0, ctx->stream));
  if (refactor) {
    PF_CHECK(launch_direct(ctx, D, 0, rhs, x, mfma != 0));
  } else {
    // factor kept: solve only (x = 0 + A^-1 rhs)
    PF_HIP(hipMemsetAsync(x, 0, sizeof(double) * n, ctx->stream));
    PF_CHECK(launch_direct(ctx, D, 1, rhs, x, mfma != 0));
  }
  for (int32_t s = 0; s < refine; ++s) {
    PF_CHECK(residual(ctx, D, n, row_ptr, col_idx, val, avg_row, rhs, x));
    PF_CHECK(launch_direct(ctx, D, 1, D->r.p, x, mfma != 0));
  }
  PF_CHECK(residual(ctx, D, n, row_ptr, col_idx, val, avg_row, rhs, x));
  PF_HIP(hipEventRecord(ctx->ev1, ctx->stream));
  PF_HIP(hipEventSynchronize(ctx->ev1));
  PF_HIP(hipEventElapsedTime(&solve_ms, ctx->ev0, ctx->ev1));
  const int32_t nm = D->nmesh;
  std::vector<int32_t> st(nm);
  std::vector<int64_t> raw(2 * (size_t)nm);
  std::vector<double> nrm(2 * (size_t)nm);
  PF_HIP(hipMemcpyAsync(st.data(), D->status.p, sizeof(int32_t) * nm, hipMemcpyDeviceToHost, ctx->stream));
  PF_HIP(hipMemcpyAsync(raw.data(), D->t_raw.p, sizeof(int64_t) * 2 * nm, hipMemcpyDeviceToHost, ctx->stream));
  PF_HIP(hipMemcpyAsync(nrm.data(), D->norms.p, sizeof(double) * 2 * nm, hipMemcpyDeviceToHost, ctx->stream));
  PF_HIP(hipStreamSynchronize(ctx->stream));
  if (D->shared && std::find(st.begin(), st.end(), (int32_t)PF_ERR_HIP) != st.end()) {
    // a share waited in vain for another: again, without waits (the band holds a part of the factor)
    PF_CHECK(whole_meshes(ctx, D));
    D->factor_version = 0;
    return pf_direct_solve_device(ctx, D, n, row_ptr, col_idx, val, nnz, rhs, x, mat_version, refine, mfma, mesh_stats,
                                  total);
  }
  int rate_khz = 0;
  PF_HIP(hipDeviceGetAttribute(&rate_khz, hipDeviceAttributeWallClockRate, ctx->device));
  const double tick_ms = rate_khz > 0 ? 1.0 / (double)rate_khz : 0.0;
  int64_t tmin = raw[0];
  for (int32_t m = 0; m < nm; ++m) tmin = std::min(tmin, raw[2 * m]);
  int status = PF_OK;
  double worst = 0.0;
  bool all_ok = true;
  for (int32_t m = 0; m < nm; ++m) {
    const double relres = nrm[2 * m + 1] > 0.0 ? std::sqrt(nrm[2 * m] / nrm[2 * m + 1]) : std::sqrt(nrm[2 * m]);
    if (st[m] != PF_OK) all_ok = false;
    if (status == PF_OK && st[m] != PF_OK) status = st[m];
    if (st[m] == PF_OK) worst = std::max(worst, relres);
    if (mesh_stats) {
      pf_batch_mesh_stats &s = mesh_stats[m];
      std::memset(&s, 0, sizeof(s));
      s.status = st[m];
      s.iterations = st[m] == PF_OK ? 1 + refine : 0;
      s.replacements = st[m] == PF_OK ? refine : 0;
      s.workgroup = -1;
      s.true_relres = relres;
      s.start_ms = (double)(raw[2 * m] - tmin) * tick_ms;
      s.end_ms = (double)(raw[2 * m + 1] - tmin) * tick_ms;
    }
  }
  if (refactor && all_ok) D->factor_version = mat_version;
  if (total) {
    std::memset(total, 0, sizeof(*total));
    total->status = status;
    total->iterations = 1 + refine;
    total->outer_iterations = refine;
    total->true_relres = worst;
    total->solve_ms = solve_ms;
    total->setup_ms = setup_ms;
  }
  return status;
}

int pf_direct_info(DirectWork *D, int32_t mesh, int64_t *n, int32_t *bandwidth, int32_t *kind, int32_t *perm) {
  if (!D || D->nmesh < 1 || mesh < 0 || mesh >= D->nmesh) {
    pf_set_error("direct: no analysis, or mesh %d out of range", mesh);
    return PF_INVALID;
  }
  const DMesh &M = D->hmesh[mesh];
  if (n) *n = M.n;
  if (bandwidth) *bandwidth = M.b;
  if (kind) *kind = D->kinds[mesh];
  if (perm) std::memcpy(perm, D->hperm.data() + M.woff, sizeof(int32_t) * M.n);
  return PF_OK;
}

int pf_direct_factor_get(pf_ctx *ctx, DirectWork *D, int32_t mesh, double *ab) {
  if (!D || D->nmesh < 1 || mesh < 0 || mesh >= D->nmesh || D->factor_version == 0) {
    pf_set_error("direct: no factor held for mesh %d", mesh);
    return PF_INVALID;
  }
  const DMesh &M = D->hmesh[mesh];
  // LAPACK lower band layout with ldab = b + 1, columns 0 .. n-1
  PF_HIP(hipMemcpy2DAsync(ab, sizeof(double) * (M.b + 1), D->band.p + M.boff, sizeof(double) * M.ld,
                          sizeof(double) * (M.b + 1), M.n, hipMemcpyDeviceToHost, ctx->stream));
  PF_HIP(hipStreamSynchronize(ctx->stream));
  return PF_OK;
}
