// elem.hip -- tiles of the element-by-element stiffness product (elem_dev.hpp): built once per
// mesh, on the device but for the packing of a few thousand cell counts.
//
// Elements are keyed by the cell of their centroid on a grid of the mesh's mean element extents
// per axis (a Cube3D mesh gets one element per cell, whatever its sides) in blocks of 4x4x4
// cells along a Z-order curve; the host packs consecutive blocks into tiles of at most ET = 128
// elements, starting a new tile where the pair of blocks at hand would not fit any more, so that a
// brick mesh's tiles are 8x4x4 elements (225 nodes; 1.76 per element).
#include <algorithm>
#include <cmath>
#include <vector>

#include "elem_dev.hpp"

namespace {

using pfelem::ET;

constexpr int32_t UMAX_LIMIT = 8 * ET;  // slots of a tile (48 KB of LDS)

// per block: min/max of the element nodes' coordinates (6), sum of the element extents (3)
__global__ void __launch_bounds__(256) k_el_extents(int64_t nn, int64_t ne, const double *__restrict__ xyz,
                                                    const int32_t *__restrict__ en, double *__restrict__ out) {
  double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY}, ex[3] = {0, 0, 0};
  for (int64_t e = blockIdx.x * (int64_t)256 + threadIdx.x; e < ne; e += (int64_t)gridDim.x * 256) {
    for (int d = 0; d < 3; ++d) {
      double a = INFINITY, b = -INFINITY;
      for (int k = 0; k < 8; ++k) {
        const double v = xyz[d * nn + en[(int64_t)k * ne + e] - 1];
        a = fmin(a, v);
        b = fmax(b, v);
      }
      lo[d] = fmin(lo[d], a);
      hi[d] = fmax(hi[d], b);
      ex[d] += b - a;
    }
  }
  __shared__ double sh[256];
  for (int k = 0; k < 9; ++k) {
    sh[threadIdx.x] = k < 3 ? lo[k] : (k < 6 ? hi[k - 3] : ex[k - 6]);
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
      if ((int)threadIdx.x < s) {
        const double a = sh[threadIdx.x], b = sh[threadIdx.x + s];
        sh[threadIdx.x] = k < 3 ? fmin(a, b) : (k < 6 ? fmax(a, b) : a + b);
      }
      __syncthreads();
    }
    if (threadIdx.x == 0) out[9 * (int64_t)blockIdx.x + k] = sh[0];
    __syncthreads();
  }
}

struct Grid {
  double lo[3], inv[3];
};

__device__ inline uint32_t spread10(uint32_t v) {  // 10 bits to every third position
  v = (v | (v << 16)) & 0x030000ffu;
  v = (v | (v << 8)) & 0x0300f00fu;
  v = (v | (v << 4)) & 0x030c30c3u;
  return (v | (v << 2)) & 0x09249249u;
}

// key: Z-order code of the element's 4x4x4 block of cells, then the element id
__global__ void k_el_keys(int64_t nn, int64_t ne, const double *__restrict__ xyz, const int32_t *__restrict__ en,
                          Grid g, uint64_t *__restrict__ keys) {
  const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e >= ne) return;
  uint32_t code = 0;
  for (int d = 0; d < 3; ++d) {
    double c = 0.0;
    for (int k = 0; k < 8; ++k) c += xyz[d * nn + en[(int64_t)k * ne + e] - 1];
    const double f = fmin(fmax((0.125 * c - g.lo[d]) * g.inv[d], 0.0), 4095.0);  // NaN: 0
    code |= spread10((uint32_t)f >> 2) << d;
  }
  keys[e] = ((uint64_t)code << 32) | (uint32_t)e;
}

__global__ void k_el_heads(int64_t ne, const uint64_t *__restrict__ keys, int32_t *__restrict__ head) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= ne) return;
  head[i] = i == 0 || (keys[i] >> 32) != (keys[i - 1] >> 32);
}

__global__ void k_el_runs(int64_t ne, const uint64_t *__restrict__ keys, const int32_t *__restrict__ head,
                          const int64_t *__restrict__ rank, int32_t *__restrict__ start,
                          int32_t *__restrict__ code, int32_t *__restrict__ eperm) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= ne) return;
  eperm[i] = (int32_t)(keys[i] & 0xffffffffu);
  if (head[i]) {
    start[rank[i]] = (int32_t)i;
    code[rank[i]] = (int32_t)(keys[i] >> 32);
  }
}

// Slots of tile blockIdx.x: its 8 x cnt (node, contribution) pairs sorted in LDS, a slot per node
// and started eight contributions.  FILL = false: ns[t] only.
template <bool FILL>
__global__ void __launch_bounds__(ET) k_el_tiles(int64_t nn, int64_t ne, const double *__restrict__ xyz,
                                                 const int32_t *__restrict__ en, const int32_t *__restrict__ eperm,
                                                 const int4 *__restrict__ tdesc, int32_t *__restrict__ ns,
                                                 int32_t *__restrict__ snode, double *__restrict__ sxyz,
                                                 uint4 *__restrict__ lconn, uint16_t *__restrict__ stab) {
  constexpr int N = 8 * ET;
  __shared__ uint64_t key[N];
  __shared__ int32_t scan[ET];
  __shared__ uint16_t lidx[FILL ? N : 1];
  const int t = blockIdx.x, tid = threadIdx.x;
  const int4 td = tdesc[t];
  const int e0 = td.x, cnt = td.y;
  const int64_t e = tid < cnt ? eperm[e0 + tid] : 0;
  for (int a = 0; a < 8; ++a) {
    const int q = a * ET + tid;
    key[q] = tid < cnt ? ((uint64_t)(uint32_t)(en[(int64_t)a * ne + e] - 1) << 32) | (uint32_t)q : ~(uint64_t)0;
  }
  for (int k = 2; k <= N; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      __syncthreads();
      for (int h = tid; h < N / 2; h += ET) {
        const int i = 2 * h - (h & (j - 1)), l = i + j;
        const uint64_t x = key[i], y = key[l];
        if ((x > y) == ((i & k) == 0)) {
          key[i] = y;
          key[l] = x;
        }
      }
    }
  __syncthreads();
  const int m = 8 * cnt;  // live pairs come first
  // place of pair i among its node's pairs, by walking back (few steps: a node has few elements)
  const auto place = [&](int i) {
    int b = 0;
    while (i - b > 0 && (key[i - b - 1] >> 32) == (key[i] >> 32)) ++b;
    return b;
  };
  int heads = 0;
  for (int k = 0; k < 8; ++k) {
    const int i = 8 * tid + k;
    if (i < m && place(i) % 8 == 0) ++heads;
  }
  scan[tid] = heads;
  __syncthreads();
  for (int off = 1; off < ET; off <<= 1) {
    const int32_t add = tid >= off ? scan[tid - off] : 0;
    __syncthreads();
    scan[tid] += add;
    __syncthreads();
  }
  if constexpr (!FILL) {
    if (tid == 0) ns[t] = scan[ET - 1];
    return;
  } else {
    const int64_t s0 = td.z;
    // relative to the tile's first node: only differences count, and these stay exact far from
    // the mesh's origin
    const int64_t node0 = (int64_t)(key[0] >> 32);
    int rank = scan[tid] - heads - 1;
    for (int k = 0; k < 8; ++k) {
      const int i = 8 * tid + k;
      if (i >= m) break;
      const int32_t node = (int32_t)(key[i] >> 32);
      const int q = (int)(key[i] & 0xffffffffu);
      const int at = place(i) % 8;
      if (at == 0) {
        ++rank;
        snode[s0 + rank] = node;
        for (int d = 0; d < 3; ++d) sxyz[3 * (s0 + rank) + d] = xyz[d * nn + node] - xyz[d * nn + node0];
      }
      stab[8 * (s0 + rank) + at] = (uint16_t)q;  // the others stay 8 * ET
      lidx[q] = (uint16_t)rank;
    }
    __syncthreads();
    if (tid < cnt) {
      uint32_t w[4];
      for (int k = 0; k < 4; ++k)
        w[k] = (uint32_t)lidx[(2 * k) * ET + tid] | ((uint32_t)lidx[(2 * k + 1) * ET + tid] << 16);
      lconn[e0 + tid] = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
}

__global__ void k_el_fill16(int64_t n, uint16_t v, uint16_t *__restrict__ a) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) a[i] = v;
}

// *bad = 1 when an element is no parallelepiped: a mixed mode of its coordinates beyond the
// rounding of the coordinates themselves (tol = 16 eps max |X|, a sum of eight of them)
__global__ void k_el_affine(int64_t nn, int64_t ne, const double *__restrict__ xyz, const int32_t *__restrict__ en,
                            double tol, int32_t *__restrict__ bad) {
  const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e >= ne) return;
  bool ok = true;
  for (int d = 0; d < 3; ++d) {
    double v[8];
    for (int a = 0; a < 8; ++a) v[a] = xyz[d * nn + en[(int64_t)a * ne + e] - 1];
    const pfelem::Modes c = pfelem::to_modes(v);
    ok = ok && fabs(c.xy) <= tol && fabs(c.xz) <= tol && fabs(c.yz) <= tol && fabs(c.t) <= tol;
  }
  if (!ok) *bad = 1;
}

__global__ void k_el_slot_keys(int64_t m, const int32_t *__restrict__ snode, uint64_t *__restrict__ keys,
                               int32_t *__restrict__ cnt) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= m) return;
  keys[k] = ((uint64_t)(uint32_t)snode[k] << 32) | (uint32_t)k;
  atomicAdd(&cnt[snode[k]], 1);
}

__global__ void k_el_slot_lists(int64_t m, int64_t nn, const uint64_t *__restrict__ keys,
                                const int64_t *__restrict__ off, int32_t *__restrict__ nslot,
                                int2 *__restrict__ nrec) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k < m) nslot[k] = (int32_t)(keys[k] & 0xffffffffu);
  if (k < nn) {
    const int32_t c = (int32_t)(off[k + 1] - off[k]);
    nrec[k] = make_int2(c == 1 ? (int32_t)(keys[off[k]] & 0xffffffffu) : (int32_t)off[k], c);
  }
}

__device__ inline int32_t fixed_bits(const uint8_t *__restrict__ fixed, int64_t node) {
  if (!fixed) return 0;
  const uint8_t *f = fixed + 3 * node;
  return (int32_t)((f[0] ? 0x20000000u : 0u) | (f[1] ? 0x40000000u : 0u) | (f[2] ? 0x80000000u : 0u));
}

// Lame constants as DMatrix forms them (FEMDomainClass.f90:11607-11636), fixed DOFs per slot and node
__global__ void k_el_state(int64_t ne, int64_t nn, int64_t nslots, const int32_t *__restrict__ eperm,
                           const double *__restrict__ E, const double *__restrict__ nu,
                           const uint8_t *__restrict__ fixed, double2 *__restrict__ lamu,
                           int32_t *__restrict__ snode, int2 *__restrict__ nrec) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < ne) {
    const double Ee = E[eperm[i]], v = nu[eperm[i]];
    lamu[i] = make_double2(v * Ee / (1.0 + v) / (1.0 - 2.0 * v), Ee / 2.0 / (1.0 + v));
  }
  if (i < nslots) {
    const int32_t node = snode[i] & 0x1fffffff;
    snode[i] = node | fixed_bits(fixed, node);
  }
  if (i < nn) nrec[i].y = (nrec[i].y & 0x1fffffff) | fixed_bits(fixed, i);
}

struct PlainV {
  const double *__restrict__ x;
  __device__ double operator()(int64_t j) const { return x[j]; }
};

template <int JM, bool AFF>
__global__ void __launch_bounds__(ET, AFF ? 3 : 2) k_el_product(ElemView v, const double *__restrict__ x,
                                                                double *__restrict__ part) {
  extern __shared__ double sh[];
  for (int t = blockIdx.x; t < v.ntile; t += gridDim.x) pfelem::tile<JM, AFF>(v, t, sh, PlainV{x}, part);
}

__global__ void __launch_bounds__(256) k_el_rows(ElemView v, const double *__restrict__ x,
                                                 const double *__restrict__ part, double *__restrict__ y) {
  const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (i >= v.nn) return;
  double s[3];
  pfelem::node_sum(v, i, part, PlainV{x}, s);
  for (int d = 0; d < 3; ++d) y[3 * i + d] = s[d];
}

// tile boundaries in the sorted element order from the blocks' runs
std::vector<int32_t> pack_tiles(const std::vector<int32_t> &start, const std::vector<int32_t> &code, int32_t ne) {
  std::vector<int32_t> toff;
  toff.push_back(0);
  const size_t nb = start.size();
  const auto end_of = [&](size_t b) { return b + 1 < nb ? start[b + 1] : ne; };
  size_t b = 0;
  while (b < nb) {
    size_t q = b;  // blocks of the same pair
    while (q < nb && (code[q] >> 1) == (code[b] >> 1)) ++q;
    const int32_t group = end_of(q - 1) - start[b];
    const int32_t fill = start[b] - toff.back();
    if (group <= ET && fill + group > ET && 2 * fill > ET) toff.push_back(start[b]);
    for (; b < q; ++b) {
      const int32_t e = end_of(b);
      if (e - toff.back() > ET && start[b] > toff.back()) toff.push_back(start[b]);
      while (e - toff.back() > ET) toff.push_back(toff.back() + ET);
    }
  }
  if (toff.back() < ne) toff.push_back(ne);
  return toff;
}

}  // namespace

int pf_elem_plan(pf_ctx *ctx, NodeGraph &g, bool *ok) {
  ElemPlan &p = g.elem;
  *ok = p.ok;
  if (p.tried) return PF_OK;
  p.ok = false;
  p.tried = true;
  if (g.nne != 8 || !g.has_coords || g.ne < 1 || g.ne >= ((int64_t)1 << 27) || g.nn >= ((int64_t)1 << 29))
    return PF_OK;
  hipStream_t st = ctx->stream;
  const int64_t ne = g.ne, nn = g.nn;
  // mean element extents per axis
  const unsigned nb = pf_blocks(ne, 256, 256);
  DevBuf<double> ext;
  PF_CHECK(ext.ensure((size_t)nb * 9));
  k_el_extents<<<nb, 256, 0, st>>>(nn, ne, g.nodcoord.p, g.elemnod.p, ext.p);
  PF_HIP(hipGetLastError());
  std::vector<double> h((size_t)nb * 9);
  PF_HIP(hipMemcpyAsync(h.data(), ext.p, sizeof(double) * h.size(), hipMemcpyDeviceToHost, st));
  PF_HIP(hipStreamSynchronize(st));
  Grid grid;
  double top = 0.0;  // largest coordinate
  for (int d = 0; d < 3; ++d) {
    double lo = INFINITY, ex = 0.0;
    for (unsigned b = 0; b < nb; ++b) {
      lo = std::fmin(lo, h[9 * b + d]);
      top = std::fmax(top, std::fmax(std::fabs(h[9 * b + d]), std::fabs(h[9 * b + 3 + d])));
      ex += h[9 * b + 6 + d];
    }
    ex /= (double)ne;
    grid.lo[d] = std::isfinite(lo) ? lo : 0.0;
    grid.inv[d] = ex > 0.0 && std::isfinite(ex) ? 1.0 / ex : 0.0;
  }
  // elements in Z-order of their blocks of cells
  DevBuf<uint64_t> ka, kb;
  DevBuf<int32_t> head, start, code;
  DevBuf<int64_t> rank, tmp;
  const size_t most = (size_t)std::max(ne, nn) + 1;
  PF_CHECK(ka.ensure(most));
  PF_CHECK(kb.ensure(most));
  PF_CHECK(head.ensure(most));
  PF_CHECK(rank.ensure(most));
  PF_CHECK(start.ensure((size_t)ne));
  PF_CHECK(code.ensure((size_t)ne));
  PF_CHECK(p.eperm.ensure((size_t)ne));
  const unsigned ge = pf_blocks(ne, 256, INT32_MAX);
  k_el_keys<<<ge, 256, 0, st>>>(nn, ne, g.nodcoord.p, g.elemnod.p, grid, ka.p);
  PF_HIP(hipGetLastError());
  bool in_tmp = false;
  PF_CHECK(pf_sort_u64(ctx, ka.p, kb.p, ne, 62, &in_tmp));
  const uint64_t *keys = in_tmp ? kb.p : ka.p;
  k_el_heads<<<ge, 256, 0, st>>>(ne, keys, head.p);
  PF_CHECK(pf_scan_i32_to_i64(ctx, head.p, ne, rank.p, tmp));
  k_el_runs<<<ge, 256, 0, st>>>(ne, keys, head.p, rank.p, start.p, code.p, p.eperm.p);
  PF_HIP(hipGetLastError());
  int64_t nrun = 0;
  PF_CHECK(pf_read_i64(ctx, rank.p + ne, &nrun));
  std::vector<int32_t> hs((size_t)nrun), hc((size_t)nrun);
  PF_HIP(hipMemcpyAsync(hs.data(), start.p, sizeof(int32_t) * nrun, hipMemcpyDeviceToHost, st));
  PF_HIP(hipMemcpyAsync(hc.data(), code.p, sizeof(int32_t) * nrun, hipMemcpyDeviceToHost, st));
  PF_HIP(hipStreamSynchronize(st));
  const std::vector<int32_t> toff = pack_tiles(hs, hc, (int32_t)ne);
  p.ntile = (int32_t)toff.size() - 1;
  std::vector<int4> desc((size_t)p.ntile);
  for (int32_t t = 0; t < p.ntile; ++t) desc[t] = make_int4(toff[t], toff[t + 1] - toff[t], 0, 0);
  PF_CHECK(p.tdesc.ensure(desc.size()));
  PF_HIP(hipMemcpyAsync(p.tdesc.p, desc.data(), sizeof(int4) * desc.size(), hipMemcpyHostToDevice, st));
  // slots
  k_el_tiles<false><<<p.ntile, ET, 0, st>>>(nn, ne, g.nodcoord.p, g.elemnod.p, p.eperm.p, p.tdesc.p, start.p, nullptr,
                                            nullptr, nullptr, nullptr);
  PF_HIP(hipMemsetAsync(code.p, 0, sizeof(int32_t), st));
  k_el_affine<<<ge, 256, 0, st>>>(nn, ne, g.nodcoord.p, g.elemnod.p, 16.0 * 2.220446049250313e-16 * top, code.p);
  PF_HIP(hipGetLastError());
  std::vector<int32_t> ns_of((size_t)p.ntile);
  int32_t bad = 0;
  PF_HIP(hipMemcpyAsync(ns_of.data(), start.p, sizeof(int32_t) * p.ntile, hipMemcpyDeviceToHost, st));
  PF_HIP(hipMemcpyAsync(&bad, code.p, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  PF_HIP(hipStreamSynchronize(st));
  p.affine = bad ? 0 : 1;
  p.umax = 0;
  p.nslots = 0;
  for (int32_t t = 0; t < p.ntile; ++t) {
    p.umax = std::max(p.umax, ns_of[t]);
    desc[t].z = (int32_t)p.nslots;
    desc[t].w = ns_of[t];
    p.nslots += ns_of[t];
  }
  // meshes whose tiles share few nodes (loose elements) stay with the assembled matrix
  if (p.umax > UMAX_LIMIT || p.nslots > 5 * ne + 4096) return PF_OK;
  PF_HIP(hipMemcpyAsync(p.tdesc.p, desc.data(), sizeof(int4) * desc.size(), hipMemcpyHostToDevice, st));
  const size_t ns = (size_t)p.nslots;
  PF_CHECK(p.snode.ensure(ns));
  PF_CHECK(p.stab.ensure(ns));
  PF_CHECK(p.sxyz.ensure(3 * ns));
  PF_CHECK(p.part.ensure(3 * ns));
  PF_CHECK(p.lconn.ensure((size_t)ne));
  PF_CHECK(p.lamu.ensure((size_t)ne));
  k_el_fill16<<<pf_blocks(8 * p.nslots, 256, INT32_MAX), 256, 0, st>>>(8 * p.nslots, (uint16_t)(8 * ET),
                                                                      reinterpret_cast<uint16_t *>(p.stab.p));
  k_el_tiles<true><<<p.ntile, ET, 0, st>>>(nn, ne, g.nodcoord.p, g.elemnod.p, p.eperm.p, p.tdesc.p, nullptr, p.snode.p,
                                           p.sxyz.p, p.lconn.p, reinterpret_cast<uint16_t *>(p.stab.p));
  PF_HIP(hipGetLastError());
  // node -> its slots, ascending
  PF_CHECK(ka.ensure(ns));
  PF_CHECK(kb.ensure(ns));
  PF_CHECK(p.nrec.ensure((size_t)nn + 1));
  PF_CHECK(p.nslot.ensure(ns));
  PF_HIP(hipMemsetAsync(head.p, 0, sizeof(int32_t) * (nn + 1), st));
  k_el_slot_keys<<<pf_blocks(p.nslots, 256, INT32_MAX), 256, 0, st>>>(p.nslots, p.snode.p, ka.p, head.p);
  PF_CHECK(pf_scan_i32_to_i64(ctx, head.p, nn, rank.p, tmp));
  int bits = 33;
  while (bits < 62 && ((int64_t)1 << (bits - 32)) < nn) ++bits;
  PF_CHECK(pf_sort_u64(ctx, ka.p, kb.p, p.nslots, bits, &in_tmp));
  k_el_slot_lists<<<pf_blocks(std::max<int64_t>(p.nslots, nn), 256, INT32_MAX), 256, 0, st>>>(
      p.nslots, nn, in_tmp ? kb.p : ka.p, rank.p, p.nslot.p, p.nrec.p);
  PF_HIP(hipGetLastError());
  PF_HIP(hipStreamSynchronize(st));  // host arrays and scratch end here
  p.ok = true;
  *ok = true;
  return PF_OK;
}

size_t pf_elem_lds(const ElemView &v) {
  return sizeof(double) * (size_t)std::max(6 * v.umax, (int32_t)pfelem::EXCH);
}

int pf_elem_view(pf_ctx *ctx, const ElemSource &src, ElemView *v) {
  const NodeGraph &g = *src.g;
  const ElemPlan &p = g.elem;
  if (!p.ok) {
    pf_set_error("internal: element product without a plan");
    return PF_INVALID;
  }
  k_el_state<<<pf_blocks(std::max(std::max(g.ne, g.nn), p.nslots), 256, INT32_MAX), 256, 0, ctx->stream>>>(
      g.ne, g.nn, p.nslots, p.eperm.p, src.E, src.nu, src.fixed, p.lamu.p, p.snode.p, p.nrec.p);
  PF_HIP(hipGetLastError());
  *v = ElemView{p.ntile, p.umax, p.affine, g.nn, p.tdesc.p, p.snode.p, p.sxyz.p, p.stab.p, p.lconn.p, p.lamu.p,
                p.nrec.p, p.nslot.p, src.rscale};
  return PF_OK;
}

int pf_elem_apply(pf_ctx *ctx, const ElemSource &src, const double *x, double *y) {
  ElemView v;
  PF_CHECK(pf_elem_view(ctx, src, &v));
  const unsigned grid = (unsigned)std::min<int64_t>(v.ntile, 2 * (int64_t)ctx->num_cus);
  double *part = src.g->elem.part.p;
  const size_t lds = pf_elem_lds(v);
  hipStream_t st = ctx->stream;
  if (src.jmode == 0 && v.affine) k_el_product<0, true><<<grid, ET, lds, st>>>(v, x, part);
  else if (src.jmode == 0) k_el_product<0, false><<<grid, ET, lds, st>>>(v, x, part);
  else if (v.affine) k_el_product<1, true><<<grid, ET, lds, st>>>(v, x, part);
  else k_el_product<1, false><<<grid, ET, lds, st>>>(v, x, part);
  k_el_rows<<<pf_blocks(v.nn, 256, INT32_MAX), 256, 0, st>>>(v, x, part, y);
  PF_HIP(hipGetLastError());
  return PF_OK;
}

namespace {
// scale = d, or scale * d when the rows were scaled before
__global__ void k_scale_update(int64_t n, const double *__restrict__ d, bool again, double *__restrict__ scale) {
  const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (i < n) scale[i] = again ? scale[i] * d[i] : d[i];
}
}  // namespace

int pf_scale_update(pf_ctx *ctx, int64_t n, const double *d, bool again, double *scale) {
  if (n > 0) k_scale_update<<<pf_blocks(n, 256, INT32_MAX), 256, 0, ctx->stream>>>(n, d, again, scale);
  PF_HIP(hipGetLastError());
  return PF_OK;
}
