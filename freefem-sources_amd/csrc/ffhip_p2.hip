// ffhip_p2.hip — vector P2 ([P2,P2,P2]) linear elasticity on tetrahedra:
// node numbering, matrix pattern, rows from the elements' vertex gradients,
// atomic-free row assembly, clamped boundary rows and body-force right-hand
// side.
//
// Replaces, for `varf va([u1,u2,u3],[v1,v2,v3]) = int3d(Th)(lambda*div(u)*div(v)
// + 2*mu*(epsilon(u)'*epsilon(v))) + int3d(Th)(f'*v) + on(4, u1=0,u2=0,u3=0)`
// on Vh(Th,[P2,P2,P2]):
//   node numbering   GenericMesh::BuildDFNumbering (GenericMesh.hpp:1880-1920)
//                    and FESpacen.cpp:403-428 (dof = 3*node + component)
//   element matrix   Element_Op (problem.cpp:6337-6437) with the P2 basis of
//                    TypeOfFE_P2Lagrange3d::FB (P012_3d.cpp:199-270), Tet_5
//   accumulation     HashMatrix::operator+= (HashMatrix.cpp:1294-1332)
//   Dirichlet        AssembleBC (problem.cpp:10120-10164), SetBC tgv
//   right-hand side  Element_rhs (problem.cpp:7940-7978)
//
// Design:
//   numbering  every (element, local node) item carries a key (vertex or
//              edge); a node's number is the rank of its first item, found
//              with atomicMin over vertices, a radix sort of the edge keys and
//              one scan over the items — equal to FreeFEM's sequential
//              first-appearance numbering.
//   pattern    node rows (sorted unique node columns, a wave per row, as
//              P1), expanded to scalar rows of 3 x 3 blocks.
//   element    the P2 gradients are linear in the barycentrics, so a tet leaves
//              only its vertex gradients (Lame: |K| and G, 13 doubles; scalar:
//              their products and the moments of kappa at the Tet_5 points, 25).
//   rows       one wave per node: the incident tets' blocks of the node's row
//              are formed from those, added in element order into the rows
//              staged in LDS, and written back contiguously.  No element
//              matrices in memory, no atomics, deterministic.
#include <hipcub/hipcub.hpp>

#include <climits>
#include <vector>

#include "ffhip_fem.hpp"

namespace ffhip {
void set_diag_rows(ffhip_ctx ctx, int64_t n, const uint8_t *onbc, const int64_t *diag, double tgv,
                   double *vals, int *missing);

// Tet::nvedge (local vertex pairs of the 6 edges)
static __constant__ int c_edge[6][2] = {{0, 1}, {0, 2}, {0, 3}, {1, 2}, {1, 3}, {2, 3}};

static unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

__device__ inline uint64_t edge_key(int32_t a, int32_t b) {
  if (a > b) { const int32_t t = a; a = b; b = t; }
  return ((uint64_t)(uint32_t)a << 32) | (uint32_t)b;
}

// ---------------------------------------------------------------- numbering
__global__ void k_fill_i32(int64_t n, int32_t v, int32_t *__restrict__ p) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// first item (10 k + i) of every vertex
__global__ void k_p2_vfirst(int64_t nt, const int32_t *__restrict__ tets, int32_t *__restrict__ firstv) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= 4 * nt) return;
  const int64_t k = m / 4;
  const int i = (int)(m % 4);
  atomicMin(&firstv[tets[m]], (int32_t)(10 * k + i));
}

// edge keys and their items, in item order (the radix sort is stable)
// sort keys of the edge items: min << vb | max (vb the bits of a vertex id,
// so the radix sort runs over 2 vb bits, not 64)
__global__ void k_p2_edge_keys(int64_t nt, const int32_t *__restrict__ tets, int vb,
                               uint64_t *__restrict__ keys, int32_t *__restrict__ items) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= 6 * nt) return;
  const int64_t k = m / 6;
  const int j = (int)(m % 6);
  const int32_t *t = tets + 4 * k;
  const int32_t a = t[c_edge[j][0]], b = t[c_edge[j][1]];
  keys[m] = ((uint64_t)(uint32_t)(a < b ? a : b) << vb) | (uint32_t)(a < b ? b : a);
  items[m] = (int32_t)(10 * k + 4 + j);
}

// head flags of the sorted edge keys; first-appearance marks of edge items
__global__ void k_p2_edge_heads(int64_t E, const uint64_t *__restrict__ skeys,
                                const int32_t *__restrict__ sitems, int64_t *__restrict__ head,
                                int64_t *__restrict__ mark) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= E) return;
  const int64_t h = (p == 0 || skeys[p] != skeys[p - 1]) ? 1 : 0;
  if (p == 0) head[E] = mark[E / 6 * 10] = 0;  // the scans' last inputs
  head[p] = h;
  mark[sitems[p]] = h;
}

// edge segment of every edge item; unique keys and their first items
__global__ void k_p2_edge_seg(int64_t E, const uint64_t *__restrict__ skeys, int vb,
                              const int32_t *__restrict__ sitems, const int64_t *__restrict__ hscan,
                              const int64_t *__restrict__ head, int32_t *__restrict__ item_seg,
                              uint64_t *__restrict__ ukeys, int32_t *__restrict__ segfirst) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= E) return;
  const int64_t seg = hscan[p] + head[p] - 1;  // inclusive scan - 1
  const int32_t item = sitems[p];
  item_seg[(item / 10) * 6 + (item % 10 - 4)] = (int32_t)seg;
  if (head[p]) {  // the unique keys in edge_key form (min << 32 | max)
    const uint64_t k = skeys[p];
    ukeys[seg] = ((k >> vb) << 32) | (k & ((uint64_t(1) << vb) - 1));
    segfirst[seg] = item;
  }
}

__global__ void k_p2_vmark(int64_t nt, const int32_t *__restrict__ tets,
                           const int32_t *__restrict__ firstv, int64_t *__restrict__ mark) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= 4 * nt) return;
  const int64_t k = m / 4;
  const int i = (int)(m % 4);
  const int32_t item = (int32_t)(10 * k + i);
  mark[10 * k + i] = firstv[tets[m]] == item ? 1 : 0;
}

__global__ void k_p2_assign(int64_t nt, const int32_t *__restrict__ tets,
                            const int32_t *__restrict__ firstv, const int32_t *__restrict__ item_seg,
                            const int32_t *__restrict__ segfirst, const int64_t *__restrict__ rank,
                            int32_t *__restrict__ elem_nodes) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= 10 * nt) return;
  const int64_t k = m / 10;
  const int i = (int)(m % 10);
  const int32_t first = i < 4 ? firstv[tets[4 * k + i]] : segfirst[item_seg[6 * k + i - 4]];
  elem_nodes[m] = (int32_t)rank[first];
}

__global__ void k_p2_vnode(int64_t nv, const int32_t *__restrict__ firstv,
                           const int64_t *__restrict__ rank, int32_t *__restrict__ vnode) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  const int32_t f = firstv[v];
  vnode[v] = f == INT_MAX ? -1 : (int32_t)rank[f];
}

__global__ void k_p2_enode(int64_t ne, const int32_t *__restrict__ segfirst,
                           const int64_t *__restrict__ rank, int32_t *__restrict__ enode) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s < ne) enode[s] = (int32_t)rank[segfirst[s]];
}

// ---------------------------------------------------------------- pattern
constexpr int kNodeCap = 96;   // node columns per node row
constexpr int kNodeHash = 256;  // LDS hash slots per node row

// One node row per wave: the 10 nodes of each of the row's elements, one after
// the other over the lanes (an edge node has about 5 elements: one pass of 64;
// a lane per element left nine lanes in ten idle), are placed in an
// open-addressing set in LDS, the lanes of a pass together: read, write where
// free, read back.  The set is compacted by ballots, the columns are ordered by
// a counting sort and written to the row's buffer (kNodeCap entries), with the
// row length, the relative diagonal position and the 10 slot bytes of every
// incidence (each lane kept its columns' slots in the set, which get their
// ranks).  A row with more than 64 incident elements, more than kNodeCap
// columns or a full set raises *ovf (the lane-per-row merge then builds the
// whole pattern).  133 -> 65 us on a 27 x 24 x 21 box, cube(32) 270 -> 137.
__global__ __launch_bounds__(256) void k_p2_pattern_wave(
    int64_t nn, const int32_t *__restrict__ elem_nodes, const int64_t *__restrict__ n2e_ptr,
    const int32_t *__restrict__ n2e, int64_t *__restrict__ nlen, int32_t *__restrict__ rowbuf,
    int8_t *__restrict__ dposr, uint8_t *__restrict__ slot8, int *__restrict__ ovf) {
  constexpr int NW = 256 / kWave, NP = 10, kFree = INT_MAX;  // passes of a row of 64 elements
  constexpr int kCols = (kNodeCap + 3) / 4 * 4;
  // every array below is one wave's: no block barrier
  __shared__ __align__(16) int32_t hk_[NW][kNodeHash];
  __shared__ __align__(16) int32_t ucol_[NW][kCols];
  __shared__ uint8_t uslot_[NW][kCols];        // the set slot of each column
  __shared__ uint8_t hrank_[NW][kNodeHash];    // the offset in the row of the column in each set slot
  const int lane = threadIdx.x % kWave, w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  int32_t *const hk = hk_[w], *const ucol = ucol_[w];
  uint8_t *const uslot = uslot_[w], *const hrank = hrank_[w];
  const int64_t a = (int64_t)blockIdx.x * NW + w;
  if (a >= nn) return;
  const int64_t k0 = n2e_ptr[a];
  const int64_t d0 = n2e_ptr[a + 1] - k0;
  bool ok = d0 <= kWave;
  const int items = ok ? 10 * (int)d0 : 0;
  *reinterpret_cast<int4 *>(&hk[4 * lane]) = make_int4(kFree, kFree, kFree, kFree);
  for (int i = lane; i < kCols; i += kWave) ucol[i] = kFree;
  uint32_t slot[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    slot[p] = 0;
    if (p * kWave >= items) break;
    const int t = p * kWave + lane, q = t / 10;
    bool open = t < items;
    int32_t c = kFree;
    if (open) c = elem_nodes[10 * (int64_t)(n2e[k0 + q] / 10) + (t - 10 * q)];
    slot[p] = ((uint32_t)c * 2654435761u) >> (32 - 8);
    for (int probe = 0;; ++probe) {  // ends: every slot looked at
      wave_lds_sync();
      const int32_t was = __hip_atomic_load(&hk[slot[p]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      wave_lds_sync();
      if (open && was == kFree)
        __hip_atomic_store(&hk[slot[p]], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      wave_lds_sync();
      const int32_t is = __hip_atomic_load(&hk[slot[p]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      open = open && is != c;
      if (__builtin_amdgcn_ballot_w64(open) == 0) break;
      if (probe == kNodeHash) { ok = false; break; }  // full
      if (open) slot[p] = (slot[p] + 1) & (kNodeHash - 1);
    }
  }
  wave_lds_sync();
  int len = 0;
  {
    const int4 h4 = *reinterpret_cast<const int4 *>(&hk[4 * lane]);
    const int32_t k4[4] = {h4.x, h4.y, h4.z, h4.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool full = k4[j] != kFree;
      const uint64_t m = __builtin_amdgcn_ballot_w64(full);
      const int at = len + __builtin_popcountll(m & ((1ull << lane) - 1));
      if (full && at < kNodeCap) {
        ucol[at] = k4[j];
        uslot[at] = (uint8_t)(4 * lane + j);
      }
      len += __builtin_popcountll(m);
    }
  }
  wave_lds_sync();
  if (len > kNodeCap) ok = false;
  if (!ok) {
    if (lane == 0) atomicOr(ovf, 1);
    return;
  }
  // the rank of a column is the number of smaller columns
  int dpos = 0;
  for (int j0 = 0; j0 < len; j0 += kWave) {
    const int j = j0 + lane;
    const bool on = j < len;
    const int32_t u = on ? ucol[j] : kFree;
    int rk = 0;
    for (int g = 0; g < len; g += 4) {  // past len: kFree
      const int4 c4 = *reinterpret_cast<const int4 *>(&ucol[g]);
      rk += (c4.x < u) + (c4.y < u) + (c4.z < u) + (c4.w < u);
    }
    dpos += __builtin_popcountll(__builtin_amdgcn_ballot_w64(on && (int64_t)u < a));
    if (on) {
      hrank[uslot[j]] = (uint8_t)rk;
      rowbuf[kNodeCap * a + rk] = u;
    }
  }
  wave_lds_sync();
  if (lane == 0) { nlen[a] = len; dposr[a] = (int8_t)(len ? dpos : -1); }
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    if (p * kWave >= items) break;
    const int t = p * kWave + lane;
    if (t < items) slot8[k0 * 10 + t] = hrank[slot[p]];
  }
}

// scalar rows 3a + c of node a: for every node column b, columns 3b, 3b+1, 3b+2
// (node columns from ncol at nodeptr, or from the row buffers when rowbuf != null).
// One wave per node: the node's 3 rows are one run of 9 L columns at 9 p0,
// written with consecutive lanes on consecutive entries (each column formed once
// for the three rows: cube(32) 149 -> 113 us).
__global__ __launch_bounds__(256) void k_p2v_expand(int64_t nn, const int64_t *__restrict__ nodeptr,
                                                    const int32_t *__restrict__ ncol,
                                                    const int64_t *__restrict__ ndiag,
                                                    const int32_t *__restrict__ rowbuf,
                                                    const int8_t *__restrict__ dposr,
                                                    int64_t *__restrict__ rowptr,
                                                    int32_t *__restrict__ colidx,
                                                    int64_t *__restrict__ diag) {
  const int lane = threadIdx.x % kWave;
  const int64_t a = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  if (a >= nn) return;  // uniform in the wave
  const int64_t p0 = nodeptr[a];
  const int L = (int)(nodeptr[a + 1] - p0);
  const int32_t *cols = rowbuf ? rowbuf + kNodeCap * a : ncol + p0;
  const int64_t base0 = 9 * p0;
  for (int j = lane; j < 3 * L; j += kWave) {
    const int q = j / 3;
    const int32_t col = 3 * cols[q] + (j - 3 * q);
    colidx[base0 + j] = col;
    colidx[base0 + 3 * L + j] = col;
    colidx[base0 + 6 * L + j] = col;
  }
  if (lane < 3) {
    const int c = lane;
    const int64_t r = 3 * a + c, base = base0 + c * 3 * L;
    rowptr[r] = base;
    if (r == 3 * nn - 1) rowptr[3 * nn] = 9 * nodeptr[nn];
    const int64_t d = rowbuf ? (dposr[a] < 0 ? -1 : dposr[a]) : (ndiag[a] < 0 ? -1 : ndiag[a] - p0);
    diag[r] = d < 0 ? -1 : base + 3 * d + c;
  }
}

// scalar P2: the node rows are the matrix rows (columns from ncol at nodeptr,
// or from the row buffers when rowbuf != null)
__global__ void k_p2_compact(int64_t nn, const int64_t *__restrict__ nodeptr,
                             const int32_t *__restrict__ ncol, const int64_t *__restrict__ ndiag,
                             const int32_t *__restrict__ rowbuf, const int8_t *__restrict__ dposr,
                             int64_t *__restrict__ rowptr, int32_t *__restrict__ colidx,
                             int64_t *__restrict__ diag) {
  // 16 lanes per row (a lane per row copied its run alone: 27 x 24 x 21 box 42 us, now 14)
  const int64_t a = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 16;
  if (a >= nn) return;
  const int lane = threadIdx.x % 16;
  const int64_t p0 = nodeptr[a], L = nodeptr[a + 1] - p0;
  if (rowbuf)
    for (int64_t q = lane; q < L; q += 16) colidx[p0 + q] = rowbuf[kNodeCap * a + q];
  if (lane != 0) return;
  rowptr[a] = p0;
  if (a == nn - 1) rowptr[nn] = nodeptr[nn];
  const int64_t d = rowbuf ? (dposr[a] < 0 ? -1 : dposr[a]) : (ndiag[a] < 0 ? -1 : ndiag[a] - p0);
  diag[a] = d < 0 ? -1 : p0 + d;
}

// ---------------------------------------------------------------- element integrals, row assembly
// A P2 gradient is linear in the barycentrics l_v:
//   vertex i:        4 G_i l_i - G_i
//   edge (i0, i1):   4 (G_i1 l_i0 + G_i0 l_i1)              (P012_3d.cpp:236-262)
// so the integral of d_c phi_i d_c' phi_j over a tet is a sum over at most
// 2 x 2 pairs of vertex gradients, each with a weight that depends on the pair's
// barycentric indices alone (the mean of l_v l_w is (1 + delta_vw) / 20), or,
// with a coefficient kappa, on the second moments of kappa.  Tet_5 is exact
// for these integrands (degree 2; with kappa the moments are taken at its
// points), so these are the values of Element_Op up to rounding.
//
// What the element pass leaves per tet (stride kLame / kLap doubles):
//   Lame:    G_0..G_3, |K|
//   Laplace: G_v . G_w (10), m_vw = int kappa l_v l_w (10, both packed by sym4),
//            M_v = sum_w m_vw (4), M = sum_v M_v
constexpr int kLame = 13, kLap = 25;

__global__ __launch_bounds__(256) void k_p2_elem_lame(int64_t nt, const double *__restrict__ xyz,
                                                      const int32_t *__restrict__ tets,
                                                      double *__restrict__ E) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nt) return;
  const int4 tv = reinterpret_cast<const int4 *>(tets)[e];
  const int32_t id[4] = {tv.x, tv.y, tv.z, tv.w};
  double v[4][3], G[4][3];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int k = 0; k < 3; ++k) v[i][k] = xyz[3 * (int64_t)id[i] + k];
  const double mes = tet_geom(v, G);
  double *o = E + kLame * e;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int k = 0; k < 3; ++k) o[3 * i + k] = G[i][k];
  o[12] = mes;
}

__global__ __launch_bounds__(256) void k_p2_elem_lap(int64_t nt, const double *__restrict__ xyz,
                                                     const int32_t *__restrict__ tets, int kind,
                                                     double c0, const double *__restrict__ kappa_e,
                                                     double *__restrict__ E) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nt) return;
  const int4 tv = reinterpret_cast<const int4 *>(tets)[e];
  const int32_t id[4] = {tv.x, tv.y, tv.z, tv.w};
  double v[4][3], G[4][3], u[4] = {0., 0., 0., 0.};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int k = 0; k < 3; ++k) v[i][k] = xyz[3 * (int64_t)id[i] + k];
    if (kind == FFHIP_COEF_P1) u[i] = kappa_e[id[i]];
  }
  const double mes = tet_geom(v, G);
  // kappa constant or linear: the integrals of l_i l_j l_k, |K| / 120 (2 and 6 times
  // that with two and three equal).  The rule's 14 points otherwise: a chain of
  // 7 us, unrolled so that the points' loads are not waited for one by one.
  double m[10] = {0., 0., 0., 0., 0., 0., 0., 0., 0., 0.};
  if (kind != FFHIP_COEF_SIN3 && kind != FFHIP_COEF_QP) {
    if (kind != FFHIP_COEF_P1) u[0] = u[1] = u[2] = u[3] = kind == FFHIP_COEF_P0 ? kappa_e[e] : c0;
    const double w = mes * (1. / 120.), S = (u[0] + u[1]) + (u[2] + u[3]);
    int o = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = i; j < 4; ++j) {
        const double t = S + u[i] + u[j];
        m[o++] = w * (i == j ? t + t : t);
      }
  } else {
#pragma unroll
    for (int q = 0; q < 14; ++q) {
      const double px = c_qf5_pts[q][0], py = c_qf5_pts[q][1], pz = c_qf5_pts[q][2];
      const double l[4] = {1. - (px + py + pz), px, py, pz};
      double kq;
      if (kind == FFHIP_COEF_QP) {
        kq = kappa_e[14 * e + q];
      } else {
        double P[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) P[k] = l[0] * v[0][k] + px * v[1][k] + py * v[2][k] + pz * v[3][k];
        kq = kappa_sin3(P[0], P[1], P[2]);
      }
      const double W = (mes * qf5_weight(q)) * kq;
      int o = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = i; j < 4; ++j) m[o++] += (W * l[i]) * l[j];
    }
  }
  double *o = E + kLap * e;
  double M = 0.;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    double Mi = 0.;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      Mi += m[sym4(i, j)];
      if (j >= i) {
        o[sym4(i, j)] = G[i][0] * G[j][0] + G[i][1] * G[j][1] + G[i][2] * G[j][2];
        o[10 + sym4(i, j)] = m[sym4(i, j)];
      }
    }
    o[20 + i] = Mi;
    M += Mi;
  }
  o[24] = M;
}

// the (at most two) terms of basis i: barycentric l[s] times the gradient of
// vertex x[s]; a vertex has one (and the constant -G_i, in the weights)
struct P2Terms {
  int vert, l[2], x[2];
};
__device__ inline P2Terms p2_terms(int i) {
  P2Terms t;
  t.vert = i < 4;
  const int ed = i < 4 ? 0 : i - 4;
  t.l[0] = i < 4 ? i : c_edge[ed][0];
  t.l[1] = i < 4 ? i : c_edge[ed][1];
  t.x[0] = t.l[1];
  t.x[1] = t.l[0];
  return t;
}

// A wave takes `nodes` consecutive node rows, six incidences (60 lanes, one
// per (incidence, local node j)) at a time: the six tets' integrals are staged
// in LDS, each lane forms its 3 x 3 block (Laplace: its entry) of the element's
// row, and the blocks are added to the row in LDS one incidence after the
// other, in element order.  The next six incidences' integrals and the items
// after those are loaded meanwhile: one row at a time the chain of dependent
// loads (list, items, integrals) took 728 us at cube(32) (69.1 M values), this
// way 352 us with 14 us for the element pass (391 us with a read, add and write
// per block instead of LDS additions; 4 or 16 nodes per wave within 3 %).  Bound by instruction issue: about
// 900 instructions per six incidences.  The element matrices formed on the matrix cores
// (M = D W D^T per tet, 7.2 KB each) and gathered from memory took 606 + 494 us.
template <bool LAP>
__global__ __launch_bounds__(64) void k_p2_rows(
    int64_t nn, int nodes, const int64_t *__restrict__ nodeptr, const int64_t *__restrict__ n2e_ptr,
    const int32_t *__restrict__ n2e, const uint8_t *__restrict__ slot8, const double *__restrict__ E,
    double lambda, double mu, double *__restrict__ vals) {
  constexpr int ED = LAP ? kLap : kLame, NB = LAP ? 1 : 9, NV = 10 * NB, GI = 6;
  constexpr int NE = (GI * ED + kWave - 1) / kWave;
  __shared__ double acc[NB * kNodeCap];
  __shared__ double el[NE * kWave];
  __shared__ double blk[GI * NV];
  __shared__ uint8_t so[kWave];
  const int lane = threadIdx.x;
  const int64_t a0 = (int64_t)xcd_block_id() * nodes;
  if (a0 >= nn) return;  // one wave per block
  const int cnt = (int)(nn - a0 < nodes ? nn - a0 : nodes);
  // this wave's row and list offsets: lane q holds those of node a0 + q
  const int64_t myp = nodeptr[a0 + (lane < cnt ? lane : cnt)];
  const int64_t myk = n2e_ptr[a0 + (lane < cnt ? lane : cnt)];
  auto bcast = [](int64_t v, int q) -> int64_t {
    const int lo = __builtin_amdgcn_readlane((int)(v & 0xffffffff), q);
    const int hi = __builtin_amdgcn_readlane((int)(v >> 32), q);
    return ((int64_t)hi << 32) | (uint32_t)lo;
  };
  const int u = lane / 10, j = lane - 10 * u;
  const P2Terms C = p2_terms(j);
  // a group: incidences [k, k + n) of node a0 + c (n <= 6; n = 0 past the end)
  struct Group {
    int c, n;
    int64_t k;
  };
  auto first = [&](int c) {
    Group g{c, 0, 0};
    if (c < cnt) {
      g.k = bcast(myk, c);
      const int64_t d = bcast(myk, c + 1) - g.k;
      g.n = (int)(d < GI ? d : GI);
    }
    return g;
  };
  auto next = [&](const Group &g) {
    if (g.c >= cnt) return g;
    const int64_t left = bcast(myk, g.c + 1) - (g.k + GI);
    if (left > 0) return Group{g.c, (int)(left < GI ? left : GI), g.k + GI};
    return first(g.c + 1);
  };
  auto load_items = [&](const Group &g, int32_t &item, int &sb) {
    item = 0;
    sb = 0;
    if (u < g.n) {
      item = n2e[g.k + u];
      sb = slot8[g.k * 10 + lane];
    }
  };
  auto load_integrals = [&](const Group &g, int32_t item, double (&r)[NE]) {
    const int32_t e = item / 10;
#pragma unroll
    for (int x0 = 0; x0 < NE; ++x0) {
      const int x = x0 * kWave + lane, uu = x / ED;
      const int32_t eu = __shfl(e, uu < GI ? 10 * uu : 0, kWave);
      r[x0] = uu < g.n ? E[(int64_t)eu * ED + (x - uu * ED)] : 0.;
    }
  };
  Group g0 = first(0), g1 = next(g0);
  int32_t item0, item1;
  int so0, so1;
  double r0[NE];
  load_items(g0, item0, so0);
  load_items(g1, item1, so1);
  load_integrals(g0, item0, r0);
  int64_t p0 = 0;
  int L = 0, tj[2] = {0, 0}, tdst[2] = {0, 0}, row = -1;
  while (g0.c < cnt) {
    if (g0.c != row) {  // the node's row starts
      row = g0.c;
      p0 = bcast(myp, row);
      L = (int)(bcast(myp, row + 1) - p0);
      for (int t = lane; t < NB * L; t += kWave) acc[t] = 0.;
      if (!LAP) {  // this lane's two entries of a 90-value block, [c][j][c'] of t = lane, lane + 64
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int t = lane + h * kWave, c = t / 30, r2 = t % 30;
          tj[h] = r2 / 3;
          tdst[h] = c * 3 * L + r2 % 3;  // + 3 * offset of node column j
        }
      }
    }
#pragma unroll
    for (int x0 = 0; x0 < NE; ++x0) el[x0 * kWave + lane] = r0[x0];
    so[lane] = (uint8_t)so0;
    const int i = item0 - 10 * (item0 / 10), ng = g0.n;
    const Group g2 = next(g1);
    int32_t item2;
    int so2;
    load_integrals(g1, item1, r0);
    load_items(g2, item2, so2);
    wave_lds_sync();
    if (u < ng) {
      const double *g = el + u * ED;
      const P2Terms R = p2_terms(i);
      if constexpr (LAP) {
        double k = 0.;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            if ((s && R.vert) || (t && C.vert)) continue;
            double w = 16. * g[10 + sym4(R.l[s], C.l[t])];
            if (R.vert) w -= 4. * g[20 + C.l[t]];
            if (C.vert) w -= 4. * g[20 + R.l[s]];
            if (R.vert && C.vert) w += g[24];
            k += w * g[sym4(R.x[s], C.x[t])];
          }
        blk[lane] = k;
      } else {
        // weights of a pair of terms, equal and different barycentrics:
        // 16 (1 + delta) / 20 for two edges, less 1 with a vertex among them
        const bool ee = !R.vert && !C.vert;
        const double hi = ee ? 1.6 : 0.6, lo = ee ? 0.8 : -0.2, mes = g[12];
        double X[2][3], Y[2][3];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const double w0 = R.l[s] == C.l[0] ? hi : lo;
          const double w1 = C.vert ? 0. : (R.l[s] == C.l[1] ? hi : lo);
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            X[s][c] = (s && R.vert) ? 0. : mes * g[3 * R.x[s] + c];
            Y[s][c] = w0 * g[3 * C.x[0] + c] + w1 * g[3 * C.x[1] + c];
          }
        }
        double B[3][3];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int d = 0; d < 3; ++d) B[c][d] = X[0][c] * Y[0][d] + X[1][c] * Y[1][d];
        const double tr = B[0][0] + B[1][1] + B[2][2];
        double *o = blk + u * NV + 3 * j;
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int d = 0; d < 3; ++d)
            o[30 * c + d] = lambda * B[c][d] + mu * B[d][c] + (c == d ? mu * tr : 0.);
      }
    }
    wave_lds_sync();
    // element order: a wave's LDS additions are carried out in the order they
    // are issued, and the lanes of one go to different slots
    auto add = [](double *p, double v) {
      (void)__hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    };
    if constexpr (LAP) {
      const double v = u < ng ? blk[lane] : 0.;
      for (int uu = 0; uu < ng; ++uu)
        if (u == uu) add(&acc[so0], v);
    } else {
      double v[GI][2];
      int o[GI][2];
#pragma unroll
      for (int uu = 0; uu < GI; ++uu)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int t = lane + h * kWave;
          v[uu][h] = t < NV ? blk[uu * NV + t] : 0.;
          o[uu][h] = tdst[h] + 3 * so[10 * uu + tj[h]];
        }
#pragma unroll
      for (int uu = 0; uu < GI; ++uu)
        if (uu < ng) {  // uniform
          add(&acc[o[uu][0]], v[uu][0]);
          if (lane < NV - kWave) add(&acc[o[uu][1]], v[uu][1]);
        }
    }
    wave_lds_sync();
    if (g1.c != row) {  // the row is complete
      double *out = vals + NB * p0;
      for (int t = lane; t < NB * L; t += kWave) out[t] = acc[t];
      wave_lds_sync();
    }
    g0 = g1; g1 = g2;
    item0 = item1; item1 = item2;
    so0 = so1; so1 = so2;
  }
}

// Nodes of a wave of k_p2_rows: 8, fewer where that leaves the chip without waves
// and a call waits for one wave's chain.  1 / 2 / 4 / 8, us per assembly, elasticity
// on cubes: 343 nodes 24.3 / 27.2 / 30.8 / 36.6, 9261 40.1 / 36.8 / 37.3 / 43.2, 35.9 k 89 /
// 72.3 / 67.5 / 72.4, 118 k 253 / 193 / 162 / 160, 275 k 588 / 465 / 374 / 364; scalar 343
// 27.1 / 29.3 / 32.4 / 37.7, 9261 33.4 / 33.4 / 36.4 / 42.5, 68.9 k 81.7 / 70.7 / 65.5 / 70.6.
static int nodes_per_wave(int64_t nn) { return nn <= 1 << 12 ? 1 : nn <= 1 << 14 ? 2 : nn <= 100000 ? 4 : 8; }

// ---------------------------------------------------------------- Dirichlet
__device__ inline int32_t find_edge_node(const uint64_t *__restrict__ ekeys,
                                         const int32_t *__restrict__ enode, int64_t ne, uint64_t key) {
  int64_t lo = 0, hi = ne - 1;
  while (lo <= hi) {
    const int64_t mid = (lo + hi) >> 1;
    const uint64_t k = ekeys[mid];
    if (k == key) return enode[mid];
    if (k < key) lo = mid + 1; else hi = mid - 1;
  }
  return -1;
}

// dofs of the labelled boundary triangles: 3 vertex nodes and 3 edge nodes,
// all components
__global__ void k_p2v_mark_bc(int64_t nbe, const int32_t *__restrict__ btri,
                              const int32_t *__restrict__ blab, Labels labels,
                              const int32_t *__restrict__ vnode,
                              const uint64_t *__restrict__ ekeys, const int32_t *__restrict__ enode,
                              int64_t ne, int ncomp, uint8_t *__restrict__ onbc,
                              int *__restrict__ missing) {
  // a lane per corner of a triangle: the vertex, and the edge to the next one (the
  // three searches of a triangle one after the other took 18 us for 9)
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, f = i / 3;
  if (f >= nbe || !labels.has(blab[f])) return;
  const int k = (int)(i - 3 * f);
  const int32_t v = btri[i], v1 = btri[3 * f + (k == 2 ? 0 : k + 1)];
  const int32_t nodes[2] = {vnode[v], find_edge_node(ekeys, enode, ne, edge_key(v, v1))};
  for (int q = 0; q < 2; ++q) {
    if (nodes[q] < 0) { *missing = 1; continue; }
    for (int c = 0; c < ncomp; ++c) onbc[ncomp * (int64_t)nodes[q] + c] = 1;
  }
}

// ---------------------------------------------------------------- right-hand side
// |K| of every tet
__global__ __launch_bounds__(256) void k_p2_mes(int64_t nt, const double *__restrict__ xyz,
                                                const int32_t *__restrict__ tets,
                                                double *__restrict__ mes) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nt) return;
  const int4 tv = reinterpret_cast<const int4 *>(tets)[e];
  const int32_t id[4] = {tv.x, tv.y, tv.z, tv.w};
  double v[4][3];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int k = 0; k < 3; ++k) v[i][k] = xyz[3 * (int64_t)id[i] + k];
  mes[e] = tet_mesure(v);
}

// b_(ncomp a + c) = f_c int phi_a, the integral of a P2 basis function over
// its tets: -|K| / 20 for a vertex, |K| / 5 for an edge (Element_rhs with Tet_5,
// exact here); the |K| added in element order; tgv * g_c on Dirichlet rows.  A
// wave takes 64 nodes, reads their incidence lists consecutively and stages the
// measures in LDS; each lane adds its own node's.  cube(32), 275 k nodes:
// 10 us and 5 us for the measures; a lane per node that walked its tets with the
// 14 points took 397 us.
__global__ __launch_bounds__(64) void k_p2v_rhs(int64_t nn, const double *__restrict__ mes,
                                                const int64_t *__restrict__ n2e_ptr,
                                                const int32_t *__restrict__ n2e, int ncomp, double f0,
                                                double f1, double f2,
                                                const uint8_t *__restrict__ onbc, double tgv, double g0,
                                                double g1, double g2, double *__restrict__ b) {
  constexpr int U = 8, CAP = kWave * U;
  __shared__ double st[CAP + CAP / 32];
  auto pos = [](int i) { return i + (i >> 5); };
  const int lane = threadIdx.x;
  const int64_t r0 = (int64_t)xcd_block_id() * kWave, a = r0 + lane;
  if (r0 >= nn) return;  // one wave per block
  const int64_t p0 = n2e_ptr[a < nn ? a : nn], p1 = n2e_ptr[a + 1 < nn ? a + 1 : nn];
  const int64_t seg0 = n2e_ptr[r0], seg1 = n2e_ptr[r0 + kWave < nn ? r0 + kWave : nn];
  const bool vert = p0 < p1 && n2e[p0] % 10 < 4;
  double s = 0.;
  for (int64_t c0 = seg0; c0 < seg1; c0 += CAP) {
    const int cnt = (int)(seg1 - c0 < CAP ? seg1 - c0 : CAP);
    int32_t e[U];
    double t[U];
#pragma unroll
    for (int u = 0; u < U; ++u) e[u] = lane + u * kWave < cnt ? n2e[c0 + lane + u * kWave] / 10 : 0;
#pragma unroll
    for (int u = 0; u < U; ++u) t[u] = mes[e[u]];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (lane + u * kWave < cnt) st[pos(lane + u * kWave)] = t[u];
    wave_lds_sync();
    const int b0 = (int)((p0 > c0 ? p0 : c0) - c0);
    const int b1 = (int)((p1 < c0 + cnt ? p1 : c0 + cnt) - c0);
    for (int k = b0; k < b1; ++k) s += st[pos(k)];
    wave_lds_sync();
  }
  if (a >= nn) return;
  const double w = vert ? -s / 20. : s / 5.;
  const double f[3] = {f0, f1, f2}, g[3] = {g0, g1, g2};
  for (int c = 0; c < ncomp; ++c)
    b[ncomp * a + c] = onbc[ncomp * a + c] ? tgv * g[c] : w * f[c];
}

// the two passes of a right-hand side
static void p2_rhs(ffhip_ctx ctx, ffhip_p2v sp, int ncomp, const double f[3], const uint8_t *onbc,
                   double tgv, const double g[3], double *b) {
  hipStream_t s = ctx->stream;
  ffhip_mesh m = sp->mesh;
  Arena ar(ctx, Arena::bytes(m->nt, 8));
  double *mes = ar.take<double>(m->nt);
  ctx->tic();
  k_p2_mes<<<nblk(m->nt, 256), 256, 0, s>>>(m->nt, m->xyz, m->elems, mes);
  k_p2v_rhs<<<(nblk(sp->nnodes, kWave) + 7) / 8 * 8, kWave, 0, s>>>(
      sp->nnodes, mes, sp->n2e_ptr, sp->n2e, ncomp, f[0], f[1], f[2], onbc, tgv, g[0], g[1], g[2], b);
  FFHIP_CHECK(hipGetLastError());
  ctx->toc();
}

// onbc (ncomp nnodes bytes) of the labelled boundary; *missing (host, read
// after the stream's wait) raised if a node was missing
static void p2v_mark(ffhip_ctx ctx, ffhip_p2v sp, const Labels &labels, int ncomp, uint8_t *onbc,
                     int *missing) {
  ffhip_mesh m = sp->mesh;
  clear(ctx, {{onbc, (size_t)(ncomp * sp->nnodes)}});
  if (m->nbe)
    k_p2v_mark_bc<<<nblk(3 * m->nbe, 256), 256, 0, ctx->stream>>>(m->nbe, m->belems, m->blab, labels, sp->vnode,
                                                              sp->ekeys, sp->enode, sp->ne, ncomp, onbc,
                                                              missing);
  FFHIP_CHECK(hipGetLastError());
}

static void p2v_release(ffhip_p2v sp) {
  dfree(sp->elem_nodes); dfree(sp->vnode); dfree(sp->ekeys); dfree(sp->enode);
  dfree(sp->n2e_ptr); dfree(sp->n2e);
  delete sp;
}

}  // namespace ffhip

using namespace ffhip;

extern "C" {

int ffhip_p2v_create(ffhip_ctx ctx, ffhip_mesh m, ffhip_p2v *out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && m && out, FFHIP_ERR_ARG, "ffhip_p2v_create: null argument");
    FFHIP_REQUIRE(m->dim == 3 && m->nloc == 4, FFHIP_ERR_UNSUPPORTED,
                  "ffhip_p2v_create: needs a tetrahedral mesh");
    FFHIP_REQUIRE(m->nt > 0 && 10 * m->nt < INT_MAX, FFHIP_ERR_UNSUPPORTED,
                  "ffhip_p2v_create: %lld elements (need 10 nt < 2^31)", (long long)m->nt);
    hipStream_t s = ctx->stream;
    const int64_t nt = m->nt, nv = m->nv, E = 6 * nt, NI = 10 * nt;
    int vb = 1;  // bits of a vertex id
    while (vb < 31 && (int64_t(1) << vb) < nv) ++vb;
    ffhip_p2v sp = new ffhip_p2v_s();
    sp->ctx = ctx; sp->mesh = m;
    try {
      size_t tb = 0;
      FFHIP_CHECK(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, (uint64_t *)nullptr, (uint64_t *)nullptr,
                                                     (int32_t *)nullptr, (int32_t *)nullptr, (int)E, 0,
                                                     2 * vb, s));
      Arena ar(ctx, Arena::bytes(nv, 4) + 2 * Arena::bytes(E, 8) + 4 * Arena::bytes(E, 4) +
                        Arena::bytes(tb, 1) + 2 * Arena::bytes(E + 1, 8) + 2 * Arena::bytes(NI + 1, 8));
      ctx->tic();
      int32_t *firstv = ar.take<int32_t>(nv);
      k_fill_i32<<<nblk(nv, 256), 256, 0, s>>>(nv, INT_MAX, firstv);
      k_p2_vfirst<<<nblk(4 * nt, 256), 256, 0, s>>>(nt, m->elems, firstv);
      uint64_t *keys = ar.take<uint64_t>(E), *skeys = ar.take<uint64_t>(E);
      int32_t *items = ar.take<int32_t>(E), *sitems = ar.take<int32_t>(E);
      k_p2_edge_keys<<<nblk(E, 256), 256, 0, s>>>(nt, m->elems, vb, keys, items);
      void *tmp = ar.take<char>(tb);
      FFHIP_CHECK(hipcub::DeviceRadixSort::SortPairs(tmp, tb, keys, skeys, items, sitems, (int)E, 0,
                                                     2 * vb, s));
      int64_t *head = ar.take<int64_t>(E + 1), *hscan = ar.take<int64_t>(E + 1);
      int64_t *mark = ar.take<int64_t>(NI + 1), *rank = ar.take<int64_t>(NI + 1);
      k_p2_edge_heads<<<nblk(E, 256), 256, 0, s>>>(E, skeys, sitems, head, mark);
      k_p2_vmark<<<nblk(4 * nt, 256), 256, 0, s>>>(nt, m->elems, firstv, mark);
      exclusive_scan_i64(ctx, head, hscan, E + 1);
      exclusive_scan_i64(ctx, mark, rank, NI + 1);
      fetch(ctx, {{&sp->ne, hscan + E, 8}, {&sp->nnodes, rank + NI, 8}});
      int32_t *item_seg = ar.take<int32_t>(E);
      int32_t *segfirst = ar.take<int32_t>(E);  // ne <= E
      sp->ekeys = dalloc<uint64_t>(sp->ne);
      k_p2_edge_seg<<<nblk(E, 256), 256, 0, s>>>(E, skeys, vb, sitems, hscan, head, item_seg, sp->ekeys,
                                                 segfirst);
      sp->elem_nodes = dalloc<int32_t>(NI);
      k_p2_assign<<<nblk(NI, 256), 256, 0, s>>>(nt, m->elems, firstv, item_seg, segfirst, rank,
                                                sp->elem_nodes);
      sp->vnode = dalloc<int32_t>(nv);
      k_p2_vnode<<<nblk(nv, 256), 256, 0, s>>>(nv, firstv, rank, sp->vnode);
      sp->enode = dalloc<int32_t>(sp->ne);
      k_p2_enode<<<nblk(sp->ne, 256), 256, 0, s>>>(sp->ne, segfirst, rank, sp->enode);
      FFHIP_CHECK(hipGetLastError());
      FFHIP_CHECK(hipStreamSynchronize(s));
      // the arena's temporaries are dead from here on (build_incidence reuses the work buffer)
      build_incidence(ctx, sp->elem_nodes, nt, 10, sp->nnodes, &sp->n2e_ptr, &sp->n2e, nullptr,
                      nullptr, nullptr);
      ctx->toc();
    } catch (...) {
      (void)hipStreamSynchronize(s);
      p2v_release(sp);
      throw;
    }
    *out = sp;
  });
}

int ffhip_p2v_info(ffhip_p2v sp, int64_t *nnodes, int64_t *ndof) {
  return guard([&] {
    FFHIP_REQUIRE(sp, FFHIP_ERR_ARG, "ffhip_p2v_info: null space");
    if (nnodes) *nnodes = sp->nnodes;
    if (ndof) *ndof = 3 * sp->nnodes;
  });
}

int ffhip_p2v_download(ffhip_p2v sp, int32_t *elem_nodes) {
  return guard([&] {
    FFHIP_REQUIRE(sp && elem_nodes, FFHIP_ERR_ARG, "ffhip_p2v_download: null argument");
    hipStream_t s = sp->ctx->stream;
    FFHIP_CHECK(hipMemcpyAsync(elem_nodes, sp->elem_nodes, 4 * 10 * sp->mesh->nt,
                               hipMemcpyDeviceToHost, s));
    FFHIP_CHECK(hipStreamSynchronize(s));
  });
}

int ffhip_p2v_free(ffhip_p2v sp) {
  return guard([&] {
    if (!sp) return;
    (void)hipStreamSynchronize(sp->ctx->stream);
    p2v_release(sp);
  });
}

}  // extern "C"

namespace ffhip {
// the node pattern of the P2 space (one wave per node row, the lane-per-row
// merge if a row does not fit), then the matrix rows: 3 x 3 blocks of the node
// columns (ncomp = 3) or the node rows themselves (ncomp = 1)
static void p2_pattern(ffhip_ctx ctx, ffhip_p2v sp, int ncomp, ffhip_mat *out) {
    hipStream_t s = ctx->stream;
    ffhip_mesh m = sp->mesh;
    const int64_t nn = sp->nnodes, n = ncomp * nn;
    FFHIP_REQUIRE(n < INT_MAX, FFHIP_ERR_UNSUPPORTED, "ffhip_pattern_p2: too many dofs");
    ffhip_mat A = new ffhip_mat_s();
    A->ctx = ctx; A->n = n; A->p2v = sp; A->ncomp = ncomp;
    try {
      Arena ar(ctx, Arena::bytes(nn + 1, 8) + Arena::bytes(1, 4) + Arena::bytes(nn, 8) +
                        Arena::bytes(kNodeCap * nn, 4) + Arena::bytes(nn, 1));
      ctx->tic();
      int64_t *len = ar.take<int64_t>(nn + 1);
      int *ovf = ar.take<int>(1);
      A->nodeptr = dalloc<int64_t>(nn + 1);
      int64_t *ndiag = ar.take<int64_t>(nn);
      int32_t *rowbuf = ar.take<int32_t>(kNodeCap * nn);
      int8_t *dposr = ar.take<int8_t>(nn);
      A->slot8 = dalloc<uint8_t>(m->nt * 100);
      clear(ctx, {{len, 8 * (size_t)(nn + 1)}, {ovf, sizeof(int)}});
      // one wave per node row (hash set in LDS); the lane-per-row merge if a
      // row does not fit
      k_p2_pattern_wave<<<nblk(nn * kWave, 256), 256, 0, s>>>(nn, sp->elem_nodes, sp->n2e_ptr, sp->n2e,
                                                              len, rowbuf, dposr, A->slot8, ovf);
      FFHIP_CHECK(hipGetLastError());
      exclusive_scan_i64(ctx, len, A->nodeptr, nn + 1);
      int over = 0;
      int64_t nnz_nodes = 0;
      fetch(ctx, {{&over, ovf, sizeof(over)}, {&nnz_nodes, A->nodeptr + nn, 8}});
      const bool wave_ok = over == 0;
      constexpr int B = 128, CAP = kNodeCap;
      if (!wave_ok) {
        clear(ctx, {{len, 8 * (size_t)(nn + 1)}, {ovf, sizeof(int)}});
        k_pattern_rows<B, CAP, false><<<nblk(nn, B), B, 0, s>>>(
            nn, 10, sp->elem_nodes, sp->n2e_ptr, sp->n2e, len, nullptr, nullptr, nullptr, nullptr,
            nullptr, ovf);
        FFHIP_CHECK(hipGetLastError());
        FFHIP_REQUIRE(read_flag(ctx, ovf) == 0, FFHIP_ERR_UNSUPPORTED,
                      "ffhip_pattern_p2v: a node couples to more than %d nodes", CAP);
        exclusive_scan_i64(ctx, len, A->nodeptr, nn + 1);
        nnz_nodes = read_i64(ctx, A->nodeptr + nn);
      }
      int32_t *ncol = nullptr;
      if (!wave_ok) {
        ncol = rowbuf;  // the row buffers are free: nnz_nodes <= kNodeCap * nn
        k_pattern_rows<B, CAP, true><<<nblk(nn, B), B, 0, s>>>(
            nn, 10, sp->elem_nodes, sp->n2e_ptr, sp->n2e, nullptr, A->nodeptr, ncol, ndiag, nullptr,
            A->slot8, ovf);
      }
      A->nnz = (int64_t)ncomp * ncomp * nnz_nodes;
      A->rowptr = dalloc<int64_t>(n + 1);
      A->colidx = dalloc<int32_t>(A->nnz);
      A->diag = dalloc<int64_t>(n);
      A->vals = dalloc<double>(A->nnz);
      if (ncomp == 3)
        k_p2v_expand<<<nblk(nn * kWave, 256), 256, 0, s>>>(nn, A->nodeptr, ncol, ndiag,
                                                  wave_ok ? rowbuf : nullptr, dposr, A->rowptr,
                                                  A->colidx, A->diag);
      else {
        if (!wave_ok)  // the merge wrote the columns at their CSR positions
          FFHIP_CHECK(hipMemcpyAsync(A->colidx, ncol, 4 * nnz_nodes, hipMemcpyDeviceToDevice, s));
        k_p2_compact<<<nblk(16 * nn, 256), 256, 0, s>>>(nn, A->nodeptr, ncol, ndiag,
                                                   wave_ok ? rowbuf : nullptr, dposr, A->rowptr,
                                                   A->colidx, A->diag);
      }
      FFHIP_CHECK(hipMemsetAsync(A->vals, 0, 8 * A->nnz, s));
      FFHIP_CHECK(hipGetLastError());
      ctx->toc();
      A->max_row = ncomp * CAP;
    } catch (...) {
      (void)hipStreamSynchronize(s);
      dfree(A->rowptr); dfree(A->colidx); dfree(A->vals); dfree(A->diag);
      dfree(A->nodeptr); dfree(A->slot8);
      delete A;
      throw;
    }
    *out = A;
}
}  // namespace ffhip

extern "C" {

int ffhip_pattern_p2v(ffhip_ctx ctx, ffhip_p2v sp, ffhip_mat *out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && sp && out, FFHIP_ERR_ARG, "ffhip_pattern_p2v: null argument");
    p2_pattern(ctx, sp, 3, out);
  });
}

int ffhip_pattern_p2(ffhip_ctx ctx, ffhip_p2v sp, ffhip_mat *out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && sp && out, FFHIP_ERR_ARG, "ffhip_pattern_p2: null argument");
    p2_pattern(ctx, sp, 1, out);
  });
}

int ffhip_assemble_p2v_elasticity(ffhip_ctx ctx, ffhip_p2v sp, ffhip_mat A, double lambda,
                                  double mu) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && sp && A && A->p2v == sp && A->slot8 && A->ncomp == 3, FFHIP_ERR_ARG,
                  "ffhip_assemble_p2v_elasticity: matrix pattern was not built from this space");
    hipStream_t s = ctx->stream;
    ffhip_mesh m = sp->mesh;
    Arena ar(ctx, Arena::bytes(kLame * m->nt, 8));
    double *E = ar.take<double>(kLame * m->nt);
    ctx->tic();
    k_p2_elem_lame<<<nblk(m->nt, 256), 256, 0, s>>>(m->nt, m->xyz, m->elems, E);
    const int nodes = nodes_per_wave(sp->nnodes);
    k_p2_rows<false><<<(nblk(sp->nnodes, nodes) + 7) / 8 * 8, kWave, 0, s>>>(
        sp->nnodes, nodes, A->nodeptr, sp->n2e_ptr, sp->n2e, A->slot8, E, lambda, mu, A->vals);
    FFHIP_CHECK(hipGetLastError());
    ctx->toc();
  });
}

int ffhip_set_bc_p2v(ffhip_ctx ctx, ffhip_p2v sp, ffhip_mat A, const int32_t *labels, int nlab,
                     double tgv, uint8_t *onbc_out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && sp && A && A->n == 3 * sp->nnodes, FFHIP_ERR_ARG,
                  "ffhip_set_bc_p2v: bad arguments");
    FFHIP_REQUIRE(nlab >= 0 && (nlab == 0 || labels), FFHIP_ERR_ARG, "ffhip_set_bc_p2v: labels");
    FFHIP_REQUIRE(tgv > 0, FFHIP_ERR_UNSUPPORTED, "ffhip_set_bc_p2v: only tgv > 0 is supported");
    uint8_t *onbc = dalloc<uint8_t>(A->n);
    const LabelArg labs(ctx, labels, nlab);
    const int *unknown = ctx->flag(0), *missing = ctx->flag(1);
    try {
      ctx->tic();
      p2v_mark(ctx, sp, labs.L, 3, onbc, ctx->flag(0));
      set_diag_rows(ctx, A->n, onbc, A->diag, tgv, A->vals, ctx->flag(1));
      ctx->toc();
      if (onbc_out) {
        FFHIP_CHECK(hipMemcpyAsync(onbc_out, onbc, A->n, hipMemcpyDeviceToHost, ctx->stream));
        FFHIP_CHECK(hipStreamSynchronize(ctx->stream));
      }
    } catch (...) {
      (void)hipStreamSynchronize(ctx->stream);
      dfree(onbc);
      throw;
    }
    const bool ok = !*unknown;
    const int miss = *missing;
    dfree(onbc);
    FFHIP_REQUIRE(ok, FFHIP_ERR_INTERNAL, "ffhip_set_bc_p2v: a boundary edge is no element edge");
    FFHIP_REQUIRE(miss == 0, FFHIP_ERR_INTERNAL, "ffhip_set_bc_p2v: a Dirichlet row has no diagonal");
  });
}

int ffhip_rhs_p2v(ffhip_ctx ctx, ffhip_p2v sp, const double f[3], const int32_t *labels, int nlab,
                  double tgv, const double g[3], double *b, int on_device) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && sp && f && b, FFHIP_ERR_ARG, "ffhip_rhs_p2v: null argument");
    FFHIP_REQUIRE(nlab >= 0 && (nlab == 0 || labels), FFHIP_ERR_ARG, "ffhip_rhs_p2v: labels");
    hipStream_t s = ctx->stream;
    const int64_t n = 3 * sp->nnodes;
    const double gz[3] = {0., 0., 0.};
    const double *gg = g ? g : gz;
    uint8_t *onbc = dalloc<uint8_t>(n);
    double *bd = on_device ? b : nullptr;
    const LabelArg labs(ctx, labels, nlab);
    const int *unknown = ctx->flag(0);
    try {
      p2v_mark(ctx, sp, labs.L, 3, onbc, ctx->flag(0));
      if (!on_device) bd = dalloc<double>(n);
      p2_rhs(ctx, sp, 3, f, onbc, tgv, gg, bd);
      if (!on_device) {
        FFHIP_CHECK(hipMemcpyAsync(b, bd, 8 * n, hipMemcpyDeviceToHost, s));
        FFHIP_CHECK(hipStreamSynchronize(s));
      }
    } catch (...) {
      (void)hipStreamSynchronize(s);
      dfree(onbc);
      if (!on_device) dfree(bd);
      throw;
    }
    dfree(onbc);
    if (!on_device) dfree(bd);
    FFHIP_REQUIRE(!*unknown, FFHIP_ERR_INTERNAL, "ffhip_rhs_p2v: a boundary edge is no element edge");
  });
}

// ---- scalar P2 (Vh(Th,P2), dof = node)
int ffhip_assemble_p2(ffhip_ctx ctx, ffhip_p2v sp, ffhip_mat A, int kind, double c0,
                      const double *kappa_e, int kappa_on_device) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && sp && A && A->p2v == sp && A->slot8 && A->ncomp == 1, FFHIP_ERR_ARG,
                  "ffhip_assemble_p2: matrix pattern was not built by ffhip_pattern_p2 from this space");
    FFHIP_REQUIRE(kind == FFHIP_COEF_CONST || kind == FFHIP_COEF_SIN3 || kind == FFHIP_COEF_P0 ||
                      kind == FFHIP_COEF_QP || kind == FFHIP_COEF_P1,
                  FFHIP_ERR_ARG, "ffhip_assemble_p2: coefficient kind %d", kind);
    const bool arr = kind == FFHIP_COEF_P0 || kind == FFHIP_COEF_QP || kind == FFHIP_COEF_P1;
    FFHIP_REQUIRE(!arr || kappa_e, FFHIP_ERR_ARG, "ffhip_assemble_p2: kappa_e");
    hipStream_t s = ctx->stream;
    ffhip_mesh m = sp->mesh;
    const int64_t cnt = kind == FFHIP_COEF_P1 ? m->nv : kind == FFHIP_COEF_P0 ? m->nt : 14 * m->nt;
    Arena ar(ctx, Arena::bytes(kLap * m->nt, 8) + (arr && !kappa_on_device ? Arena::bytes(cnt, 8) : 0));
    double *E = ar.take<double>(kLap * m->nt);
    const double *kd = kappa_e;
    if (arr && !kappa_on_device) {
      double *kb = ar.take<double>(cnt);
      FFHIP_CHECK(hipMemcpyAsync(kb, kappa_e, 8 * cnt, hipMemcpyHostToDevice, s));
      kd = kb;
    }
    ctx->tic();
    k_p2_elem_lap<<<nblk(m->nt, 256), 256, 0, s>>>(m->nt, m->xyz, m->elems, kind, c0, kd, E);
    const int nodes = nodes_per_wave(sp->nnodes);
    k_p2_rows<true><<<(nblk(sp->nnodes, nodes) + 7) / 8 * 8, kWave, 0, s>>>(
        sp->nnodes, nodes, A->nodeptr, sp->n2e_ptr, sp->n2e, A->slot8, E, 0., 0., A->vals);
    FFHIP_CHECK(hipGetLastError());
    ctx->toc();
  });
}

int ffhip_set_bc_p2(ffhip_ctx ctx, ffhip_p2v sp, ffhip_mat A, const int32_t *labels, int nlab,
                    double tgv, uint8_t *onbc_out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && sp && A && A->ncomp == 1 && A->n == sp->nnodes, FFHIP_ERR_ARG,
                  "ffhip_set_bc_p2: bad arguments");
    FFHIP_REQUIRE(nlab >= 0 && (nlab == 0 || labels), FFHIP_ERR_ARG, "ffhip_set_bc_p2: labels");
    FFHIP_REQUIRE(tgv > 0, FFHIP_ERR_UNSUPPORTED, "ffhip_set_bc_p2: only tgv > 0 is supported");
    uint8_t *onbc = dalloc<uint8_t>(A->n);
    const LabelArg labs(ctx, labels, nlab);
    const int *unknown = ctx->flag(0), *missing = ctx->flag(1);
    try {
      ctx->tic();
      p2v_mark(ctx, sp, labs.L, 1, onbc, ctx->flag(0));
      set_diag_rows(ctx, A->n, onbc, A->diag, tgv, A->vals, ctx->flag(1));
      ctx->toc();
      if (onbc_out) {
        FFHIP_CHECK(hipMemcpyAsync(onbc_out, onbc, A->n, hipMemcpyDeviceToHost, ctx->stream));
        FFHIP_CHECK(hipStreamSynchronize(ctx->stream));
      }
    } catch (...) {
      (void)hipStreamSynchronize(ctx->stream);
      dfree(onbc);
      throw;
    }
    const bool ok = !*unknown;
    const int miss = *missing;
    dfree(onbc);
    FFHIP_REQUIRE(ok, FFHIP_ERR_INTERNAL, "ffhip_set_bc_p2: a boundary edge is no element edge");
    FFHIP_REQUIRE(miss == 0, FFHIP_ERR_INTERNAL, "ffhip_set_bc_p2: a Dirichlet row has no diagonal");
  });
}

int ffhip_rhs_p2(ffhip_ctx ctx, ffhip_p2v sp, double f, const int32_t *labels, int nlab, double tgv,
                 double g, double *b, int on_device) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && sp && b, FFHIP_ERR_ARG, "ffhip_rhs_p2: null argument");
    FFHIP_REQUIRE(nlab >= 0 && (nlab == 0 || labels), FFHIP_ERR_ARG, "ffhip_rhs_p2: labels");
    hipStream_t s = ctx->stream;
    const int64_t n = sp->nnodes;
    uint8_t *onbc = dalloc<uint8_t>(n);
    double *bd = on_device ? b : nullptr;
    const LabelArg labs(ctx, labels, nlab);
    const int *unknown = ctx->flag(0);
    try {
      p2v_mark(ctx, sp, labs.L, 1, onbc, ctx->flag(0));
      if (!on_device) bd = dalloc<double>(n);
      const double fv[3] = {f, 0., 0.}, gv[3] = {g, 0., 0.};
      p2_rhs(ctx, sp, 1, fv, onbc, tgv, gv, bd);
      if (!on_device) {
        FFHIP_CHECK(hipMemcpyAsync(b, bd, 8 * n, hipMemcpyDeviceToHost, s));
        FFHIP_CHECK(hipStreamSynchronize(s));
      }
    } catch (...) {
      (void)hipStreamSynchronize(s);
      dfree(onbc);
      if (!on_device) dfree(bd);
      throw;
    }
    dfree(onbc);
    if (!on_device) dfree(bd);
    FFHIP_REQUIRE(!*unknown, FFHIP_ERR_INTERNAL, "ffhip_rhs_p2: a boundary edge is no element edge");
  });
}

}  // extern "C"
