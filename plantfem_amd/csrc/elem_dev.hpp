// elem_dev.hpp -- the stiffness product y = K x element by element, without the assembled matrix.
//
// K = sum_e Ke with Ke = sum_gp B^T D B detJ (the element matrices of assemble.hip).  For one
// element the product needs the 24 coordinates, 24 vector entries and two Lame constants and
// 460 (parallelepipeds) to 1250 FP64 operations; the assembled product streams 27 3x3 blocks per
// node (1.9 KB) for the same result.
//
// Layout: the elements are sorted into tiles of at most ET along a space-filling curve, one thread
// per element, one workgroup per tile.  A tile gathers its nodes' vector entries and coordinates
// once into LDS, every thread evaluates its element, the 24 results go back through LDS and each
// tile node ("slot") sums its at most 8 contributions in a fixed order (a node with more takes
// several slots).  A second kernel sums each node's slots (1.76 per element for bricks) in tile
// order.  No atomics: results are the same on every run.
//
// Element arithmetic.  With the modal coefficients c of the 8 nodal values (sums and
// differences, 23 additions per component), the reference gradients are
//   d/dxi = c_x + eta c_xy + zeta c_xz + eta zeta c_xyz  (and cyclic),
// unscaled (8 x the gradient).  The gradients of u and of X at the 2x2x2 Gauss points, the stress
// of B = (J^-T or J^-1) dN/dxi (jmode 0, 1) and the transposed gradient follow from these with the
// adjugate A of J and one reciprocal per Gauss point: G = A / detJ, so K u needs A^T D A / detJ.
// Where J is the same at all Gauss points (parallelepipeds: every Cube3D mesh) the functions 1,
// xi, eta, zeta, eta zeta, ... are orthogonal over the Gauss points, so each meets A^T D A once
// instead of eight times.
#pragma once
#include "pf_internal.hpp"

namespace pfelem {

constexpr int ET = 128;           // elements per tile = threads per workgroup
constexpr int NPT = 2;            // slots per thread whose tables are loaded ahead of the element work
constexpr int PLANE = 8 * ET + 8; // doubles per component of the exchange buffer; entry 8 * ET is 0
constexpr int EXCH = 3 * PLANE;
constexpr double GP = 0.57735026918962576;

// modal coefficients of nodal values v (hex8 node order): x, y, z, xy, xz, yz, xyz (the constant
// one has no gradient)
struct Modes {
  double x, y, z, xy, xz, yz, t;
};

__device__ inline Modes to_modes(const double (&v)[8]) {
  const double s01 = v[0] + v[1], d01 = v[1] - v[0], s32 = v[3] + v[2], d32 = v[2] - v[3];
  const double s45 = v[4] + v[5], d45 = v[5] - v[4], s76 = v[7] + v[6], d76 = v[6] - v[7];
  const double bss = s01 + s32, bsd = s32 - s01, bds = d01 + d32, bdd = d32 - d01;
  const double tss = s45 + s76, tsd = s76 - s45, tds = d45 + d76, tdd = d76 - d45;
  return Modes{bds + tds, bsd + tsd, tss - bss, bdd + tdd, tds - bds, tsd - bsd, tdd - bdd};
}

__device__ inline void from_modes(const Modes &q, double (&f)[8]) {
  // f_a = sum_m sign_m(a) q_m
  const double bx = q.x - q.xz, tx = q.x + q.xz, by = q.y - q.yz, ty = q.y + q.yz;
  const double bxy = q.xy - q.t, txy = q.xy + q.t;
  const double b0 = -q.z, t0 = q.z;
  const double bm = b0 - by, bp = b0 + by, tm = t0 - ty, tp = t0 + ty;  // eta = -1, +1
  const double bxm = bx - bxy, bxp = bx + bxy, txm = tx - txy, txp = tx + txy;
  f[0] = bm - bxm;
  f[1] = bm + bxm;
  f[2] = bp + bxp;
  f[3] = bp - bxp;
  f[4] = tm - txm;
  f[5] = tm + txm;
  f[6] = tp + txp;
  f[7] = tp - txp;
}

// 1/d by the hardware estimate and two Newton steps
__device__ inline double recip(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
  return __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
}

// T[i] (row i: transposed-gradient direction i, 3 components) of one Gauss point from the unscaled
// J (rows dX/dxi_i) and Du (rows du/dxi_i)
template <int JM>
__device__ inline void gauss_point(const double (&J)[3][3], const double (&Du)[3][3], double lam, double mu,
                                   double (&T)[3][3]) {
  double A[3][3];  // adjugate
  A[0][0] = J[1][1] * J[2][2] - J[1][2] * J[2][1];
  A[0][1] = J[0][2] * J[2][1] - J[0][1] * J[2][2];
  A[0][2] = J[0][1] * J[1][2] - J[0][2] * J[1][1];
  A[1][0] = J[1][2] * J[2][0] - J[1][0] * J[2][2];
  A[1][1] = J[0][0] * J[2][2] - J[0][2] * J[2][0];
  A[1][2] = J[0][2] * J[1][0] - J[0][0] * J[1][2];
  A[2][0] = J[1][0] * J[2][1] - J[1][1] * J[2][0];
  A[2][1] = J[0][1] * J[2][0] - J[0][0] * J[2][1];
  A[2][2] = J[0][0] * J[1][1] - J[0][1] * J[1][0];
  const double det = J[0][0] * A[0][0] + J[0][1] * A[1][0] + J[0][2] * A[2][0];
  const double w = recip(512.0 * det);
  const double lw = lam * w, mw = mu * w;
  double H[3][3];
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (JM == 0)
        H[p][d] = A[0][p] * Du[0][d] + A[1][p] * Du[1][d] + A[2][p] * Du[2][d];
      else
        H[p][d] = A[p][0] * Du[0][d] + A[p][1] * Du[1][d] + A[p][2] * Du[2][d];
    }
  const double tr = (H[0][0] + H[1][1] + H[2][2]) * lw, m2 = mw + mw;
  const double s00 = m2 * H[0][0] + tr, s11 = m2 * H[1][1] + tr, s22 = m2 * H[2][2] + tr;
  const double s01 = mw * (H[0][1] + H[1][0]), s02 = mw * (H[0][2] + H[2][0]), s12 = mw * (H[1][2] + H[2][1]);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const double a0 = JM == 0 ? A[i][0] : A[0][i], a1 = JM == 0 ? A[i][1] : A[1][i],
                 a2 = JM == 0 ? A[i][2] : A[2][i];
    T[i][0] = a0 * s00 + a1 * s01 + a2 * s02;
    T[i][1] = a0 * s01 + a1 * s11 + a2 * s12;
    T[i][2] = a0 * s02 + a1 * s12 + a2 * s22;
  }
}

// q[d] = modal forces of Ke u, component d, from the modes of X and u.  The loop over (eta, zeta)
// stays a loop and the two Gauss points of a turn stay apart: unrolled or interleaved, the
// eight Gauss points' intermediates spill.
template <int JM>
__device__ inline void element(const Modes (&X)[3], const Modes (&u)[3], double lam, double mu, Modes (&q)[3]) {
#pragma unroll
  for (int d = 0; d < 3; ++d) q[d] = Modes{0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
  for (int k = 0; k < 4; ++k) {
    const double oy = k & 1 ? 1.0 : -1.0, oz = k & 2 ? 1.0 : -1.0;
    const double gy = oy * GP, gz = oz * GP;
    double T[2][3][3];
#pragma unroll
    for (int sx = 0; sx < 2; ++sx) {
      const double gx = sx ? GP : -GP;
      double J[3][3], Du[3][3];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        J[0][d] = (X[d].x + gz * X[d].xz) + gy * (X[d].xy + gz * X[d].t);
        J[1][d] = (X[d].y + gz * X[d].yz) + gx * (X[d].xy + gz * X[d].t);
        J[2][d] = (X[d].z + gy * X[d].yz) + gx * (X[d].xz + gy * X[d].t);
        Du[0][d] = (u[d].x + gz * u[d].xz) + gy * (u[d].xy + gz * u[d].t);
        Du[1][d] = (u[d].y + gz * u[d].yz) + gx * (u[d].xy + gz * u[d].t);
        Du[2][d] = (u[d].z + gy * u[d].yz) + gx * (u[d].xz + gy * u[d].t);
      }
      gauss_point<JM>(J, Du, lam, mu, T[sx]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double a = T[0][0][d] + T[1][0][d];
      const double b = T[0][1][d] + T[1][1][d], bm = T[1][1][d] - T[0][1][d];
      const double c = T[0][2][d] + T[1][2][d], cm = T[1][2][d] - T[0][2][d];
      q[d].x += a;
      q[d].y += b;
      q[d].z += c;
      q[d].xy += oy * a + bm;
      q[d].xz += oz * a + cm;
      q[d].yz += oz * b + oy * c;
      q[d].t += oz * (oy * a + bm) + oy * cm;
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    q[d].xy *= GP;
    q[d].xz *= GP;
    q[d].yz *= GP;
    q[d].t *= GP * GP;
  }
}

// The same where J is constant over the element (rows J of the unscaled Jacobian).  The gradient of
// function f (one of 1, xi, eta, zeta, eta zeta, xi zeta, xi eta) has rows g_i for the modes whose
// derivative along i is f; summed over the Gauss points f^2 is 8, 8/3 or 8/9.
template <int JM>
__device__ inline void element_affine(const double (&J)[3][3], const Modes (&u)[3], double lam, double mu,
                                      Modes (&q)[3]) {
  double B[3][3];  // B[i] = A[i][.] (jmode 0) or A[.][i] (jmode 1): H = sum_i B[i] g_i^T / det
  {
    const double a00 = J[1][1] * J[2][2] - J[1][2] * J[2][1], a01 = J[0][2] * J[2][1] - J[0][1] * J[2][2],
                 a02 = J[0][1] * J[1][2] - J[0][2] * J[1][1];
    const double a10 = J[1][2] * J[2][0] - J[1][0] * J[2][2], a11 = J[0][0] * J[2][2] - J[0][2] * J[2][0],
                 a12 = J[0][2] * J[1][0] - J[0][0] * J[1][2];
    const double a20 = J[1][0] * J[2][1] - J[1][1] * J[2][0], a21 = J[0][1] * J[2][0] - J[0][0] * J[2][1],
                 a22 = J[0][0] * J[1][1] - J[0][1] * J[1][0];
    const double w = 8.0 * recip(512.0 * (J[0][0] * a00 + J[0][1] * a10 + J[0][2] * a20));
    lam *= w;
    mu *= w;
    B[0][0] = a00;
    B[1][1] = a11;
    B[2][2] = a22;
    B[0][1] = JM == 0 ? a01 : a10;
    B[1][0] = JM == 0 ? a10 : a01;
    B[0][2] = JM == 0 ? a02 : a20;
    B[2][0] = JM == 0 ? a20 : a02;
    B[1][2] = JM == 0 ? a12 : a21;
    B[2][1] = JM == 0 ? a21 : a12;
  }
  // T_i = B_i S with S the stress of H = sum_k B_k g_k^T over the rows k != skip (skip = 3: all)
  const auto stress = [&](const double (&g)[3][3], int skip, double (&T)[3][3]) {
    double H[3][3];
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        double h = 0.0;
#pragma unroll
        for (int k = 0; k < 3; ++k)
          if (k != skip) h = __builtin_fma(B[k][p], g[k][d], h);
        H[p][d] = h;
      }
    const double tr = (H[0][0] + H[1][1] + H[2][2]) * lam, m2 = mu + mu;
    const double s00 = m2 * H[0][0] + tr, s11 = m2 * H[1][1] + tr, s22 = m2 * H[2][2] + tr;
    const double s01 = mu * (H[0][1] + H[1][0]), s02 = mu * (H[0][2] + H[2][0]), s12 = mu * (H[1][2] + H[2][1]);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      if (i == skip) continue;
      T[i][0] = B[i][0] * s00 + B[i][1] * s01 + B[i][2] * s02;
      T[i][1] = B[i][0] * s01 + B[i][1] * s11 + B[i][2] * s12;
      T[i][2] = B[i][0] * s02 + B[i][1] * s12 + B[i][2] * s22;
    }
  };
  double g[3][3], T[3][3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    g[0][d] = u[d].x;
    g[1][d] = u[d].y;
    g[2][d] = u[d].z;
  }
  stress(g, 3, T);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    q[d].x = T[0][d];
    q[d].y = T[1][d];
    q[d].z = T[2][d];
    g[1][d] = u[d].xy;  // function xi
    g[2][d] = u[d].xz;
  }
  stress(g, 0, T);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    q[d].xy = T[1][d];
    q[d].xz = T[2][d];
    g[0][d] = u[d].xy;  // function eta
    g[2][d] = u[d].yz;
  }
  stress(g, 1, T);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    q[d].xy += T[0][d];
    q[d].yz = T[2][d];
    g[0][d] = u[d].xz;  // function zeta
    g[1][d] = u[d].yz;
  }
  stress(g, 2, T);
  // eta zeta, xi zeta, xi eta: one row each, T_i = (lam + mu) B_i (B_i.t) + mu |B_i|^2 t
  double tt[3] = {0.0, 0.0, 0.0}, dd = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const double bt = B[i][0] * u[0].t + B[i][1] * u[1].t + B[i][2] * u[2].t;
    dd += B[i][0] * B[i][0] + B[i][1] * B[i][1] + B[i][2] * B[i][2];
#pragma unroll
    for (int d = 0; d < 3; ++d) tt[d] += bt * B[i][d];
  }
  const double c1 = (lam + mu) * (1.0 / 9.0), c2 = mu * dd * (1.0 / 9.0);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    q[d].xy *= 1.0 / 3.0;
    q[d].xz = (q[d].xz + T[0][d]) * (1.0 / 3.0);
    q[d].yz = (q[d].yz + T[1][d]) * (1.0 / 3.0);
    q[d].t = c1 * tt[d] + c2 * u[d].t;
  }
}

// One tile: xf(j) = vector entry of DOF j (entries of fixed DOFs count as 0); part receives the
// tile's slot sums (3 doubles per slot).  Every thread of the ET-thread workgroup calls it; sh
// holds max(6 * umax, EXCH) doubles.  AFF: every element of the mesh is a parallelepiped.
template <int JM, bool AFF, typename XF>
__device__ inline void tile(const ElemView &p, int t, double *sh, XF xf, double *__restrict__ part) {
  const int tid = threadIdx.x;
  const int4 td = p.tdesc[t];
  const int e0 = td.x, cnt = td.y, s0 = td.z, ns = td.w;
  double *sx = sh, *sX = sh + 3 * ns;
  const bool live = tid < cnt;
  // all loads that depend on the tile's offsets only
  uint4 lc = {0u, 0u, 0u, 0u};
  double2 lm = {0.0, 0.0};
  int32_t node[NPT];
  uint4 tab[NPT];
#pragma unroll
  for (int k = 0; k < NPT; ++k) {
    const int j = tid + k * ET;
    node[k] = j < ns ? p.snode[s0 + j] : 0;
  }
  if (live) {
    lc = p.lconn[e0 + tid];
    lm = p.lamu[e0 + tid];
  }
  const auto tables = [&] {
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
      const int j = tid + k * ET;
      tab[k] = j < ns ? p.stab[s0 + j] : make_uint4(0u, 0u, 0u, 0u);
    }
  };
  if constexpr (AFF) tables();  // the general form has no registers to hold them
  const auto stage = [&](int j, int32_t nd) {  // top three bits of a slot's node: its fixed DOFs
    const int64_t i = 3 * (int64_t)(nd & 0x1fffffff);
    const double x0 = xf(i), x1 = xf(i + 1), x2 = xf(i + 2);
    sx[3 * j] = (nd & 0x20000000) ? 0.0 : x0;
    sx[3 * j + 1] = (nd & 0x40000000) ? 0.0 : x1;
    sx[3 * j + 2] = nd < 0 ? 0.0 : x2;
  };
  const double *xp = p.sxyz + 3 * (int64_t)s0;
  for (int k = tid; k < 3 * ns; k += ET) sX[k] = xp[k];
#pragma unroll
  for (int k = 0; k < NPT; ++k)
    if (tid + k * ET < ns) stage(tid + k * ET, node[k]);
  for (int j = tid + NPT * ET; j < ns; j += ET) stage(j, p.snode[s0 + j]);
  __syncthreads();
  Modes q[3];
  if (live) {
    const int l[8] = {(int)(lc.x & 0xffffu), (int)(lc.x >> 16), (int)(lc.y & 0xffffu), (int)(lc.y >> 16),
                      (int)(lc.z & 0xffffu), (int)(lc.z >> 16), (int)(lc.w & 0xffffu), (int)(lc.w >> 16)};
    Modes u[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      double v[8];
#pragma unroll
      for (int a = 0; a < 8; ++a) v[a] = sx[3 * l[a] + d];
      u[d] = to_modes(v);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (AFF) {
      double J[3][3];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double o = sX[3 * l[0] + d];
        J[0][d] = 4.0 * (sX[3 * l[1] + d] - o);
        J[1][d] = 4.0 * (sX[3 * l[3] + d] - o);
        J[2][d] = 4.0 * (sX[3 * l[4] + d] - o);
      }
      element_affine<JM>(J, u, lm.x, lm.y, q);
    } else {
      Modes X[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        double v[8];
#pragma unroll
        for (int a = 0; a < 8; ++a) v[a] = sX[3 * l[a] + d];
        X[d] = to_modes(v);
        __builtin_amdgcn_sched_barrier(0);
      }
      element<JM>(X, u, lm.x, lm.y, q);
    }
  }
  if constexpr (!AFF) tables();
  __syncthreads();  // the staged values are consumed
  if (live) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      double f[8];
      from_modes(q[d], f);
#pragma unroll
      for (int a = 0; a < 8; ++a) sh[d * PLANE + a * ET + tid] = f[a];
    }
  }
  if (tid < 3) sh[tid * PLANE + 8 * ET] = 0.0;  // what the unused entries of a slot's table name
  __syncthreads();
  const auto gather = [&](int j, const uint4 &w) {
    const int g[8] = {(int)(w.x & 0xffffu), (int)(w.x >> 16), (int)(w.y & 0xffffu), (int)(w.y >> 16),
                      (int)(w.z & 0xffffu), (int)(w.z >> 16), (int)(w.w & 0xffffu), (int)(w.w >> 16)};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      double s = sh[d * PLANE + g[0]];
#pragma unroll
      for (int k = 1; k < 8; ++k) s += sh[d * PLANE + g[k]];
      part[3 * (int64_t)(s0 + j) + d] = s;
    }
  };
#pragma unroll
  for (int k = 0; k < NPT; ++k)
    if (tid + k * ET < ns) gather(tid + k * ET, tab[k]);
  for (int j = tid + NPT * ET; j < ns; j += ET) gather(j, p.stab[s0 + j]);
  __syncthreads();  // the next tile rewrites sh
}

// tiles of workgroup b of G: consecutive tiles, which share nodes, go to one XCD (workgroups go
// round the 8 XCDs), so its L2 serves their gathers
__device__ inline int tile_of(int k, int ntile, int G) {
  if (G % 8 != 0) return k < ntile ? k : -1;
  const int per = (ntile + 7) / 8;
  const int t = (k % 8) * per + k / 8;
  return k / 8 < per && t < ntile ? t : -1;
}

// y of node i (3 rows) from its slots' sums: fixed rows are unit rows
template <typename XF>
__device__ inline void node_sum(const ElemView &p, int64_t i, const double *__restrict__ part, XF xf, double (&y)[3]) {
  const int2 r = p.nrec[i];  // slots: (slot, 1) or (offset into nslot, count); flags in the top bits
  const int cnt = r.y & 0x1fffffff;
  y[0] = y[1] = y[2] = 0.0;
  if (cnt == 1) {
    const double *q = part + 3 * (int64_t)r.x;
    y[0] = q[0];
    y[1] = q[1];
    y[2] = q[2];
  } else {
    for (int k = 0; k < cnt; ++k) {
      const double *q = part + 3 * (int64_t)p.nslot[r.x + k];
      y[0] += q[0];
      y[1] += q[1];
      y[2] += q[2];
    }
  }
  if (p.rscale) {
    y[0] *= p.rscale[3 * i];
    y[1] *= p.rscale[3 * i + 1];
    y[2] *= p.rscale[3 * i + 2];
  }
  if (cnt > 0 && (r.y & ~0x1fffffff)) {
    if (r.y & 0x20000000) y[0] = xf(3 * i);
    if (r.y & 0x40000000) y[1] = xf(3 * i + 1);
    if (r.y < 0) y[2] = xf(3 * i + 2);
  }
}

}  // namespace pfelem
