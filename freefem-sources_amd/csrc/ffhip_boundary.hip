// ffhip_boundary.hip — boundary integrals of P1 varfs and linear forms:
//   int2d(Th3, labels)(alpha*u*v)  /  int1d(Th2, labels)(alpha*u*v)   (matrix)
//   int2d(Th3, labels)(g*v)        /  int1d(Th2, labels)(g*v)         (right-hand side)
// i.e. the Robin / Neumann terms of a FreeFEM problem.
//
// FreeFEM visits the boundary elements whose label is listed, in boundary-
// element order, and adds the face (edge) element matrix of the adjacent
// element (AssembleBilinearForm 3D, src/fflib/problem.cpp:1273-1327; the face
// branch of Element_Op, problem.cpp:6515-6561: coef = |N(ie)|/2 * w_q at the
// T_5 points of the face; 2D edges: problem.cpp:6223-6240, coef = |E| w_q at
// the QF_GaussLegendre3 points) and of the linear form (Element_rhs,
// problem.cpp:8517-8590).  On a face only the basis functions of its own
// vertices are non-zero, so the contribution is the boundary element's own
// P1 mass matrix weighted by the coefficient.
//
// GPU mapping: one lane per vertex row walks the vertex's boundary-element
// incidences in boundary-element order and adds that element's row into the
// CSR slots of the row (found by binary search in the sorted columns): every
// slot is owned by one lane and receives its contributions in FreeFEM's order,
// after the volume terms already in the matrix — deterministic, no atomics.
// The boundary is small next to the volume (a surface of the mesh), so the
// element rows are recomputed per incidence rather than stored.
#include <hip/hip_runtime.h>

#include <cmath>

#include "ffhip_fem.hpp"

namespace ffhip {


namespace {

unsigned nblocks(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

// Quadrature of a boundary element: T_5 (QuadratureFormular.cpp:172-186) on
// triangles, QF_GaussLegendre3 (QuadratureFormular.cpp:320-343) on edges.
// Point q of element e is x_q = (1 - s_q - t_q) B0 + s_q B1 + t_q B2
// (edges: (1 - s_q) B0 + s_q B1) for its vertices B in mesh order.
struct BndRule {
  int nq;
  double s[7], t[7], w[7];
};

BndRule rule(int dim) {
  BndRule R{};
  if (dim == 3) {
    const double sqrt15 = 3.87298334620741688517926539978;
    const double a = 1.E0 / 3.E0, A = 0.225E0;
    const double r = (6 - sqrt15) / 21, s = (9 + 2 * sqrt15) / 21, B = (155 - sqrt15) / 1200;
    const double u = (6 + sqrt15) / 21, v = (9 - 2 * sqrt15) / 21, C = (155 + sqrt15) / 1200;
    const double P[7][2] = {{a, a}, {r, r}, {r, s}, {s, r}, {u, u}, {u, v}, {v, u}};
    const double W[7] = {A, B, B, B, C, C, C};
    R.nq = 7;
    for (int q = 0; q < 7; ++q) { R.s[q] = P[q][0]; R.t[q] = P[q][1]; R.w[q] = W[q]; }
  } else {
    const double g1 = (1 - sqrt(3. / 5.)) / 2;
    R.nq = 3;
    R.s[0] = 0.5; R.s[1] = g1; R.s[2] = 1 - g1;
    R.w[0] = 8. / 18.; R.w[1] = 5. / 18.; R.w[2] = 5. / 18.;
  }
  return R;
}

__device__ inline double coef_at(int kind, double c0, const double *__restrict__ coef, int64_t e,
                                 int q, int nq, const double *P, int dim) {
  if (kind == FFHIP_COEF_SIN3) {
    double s = 0.5 * sin2pi(P[0]);
    s = s * sin2pi(P[1]);
    if (dim == 3) s = s * sin2pi(P[2]);
    return 1 + s;
  }
  if (kind == FFHIP_COEF_QP) return coef[e * nq + q];
  if (kind == FFHIP_COEF_P0) return coef[e];
  return c0;
}

// A wave takes ROWS vertices: their (boundary element, local vertex) items
// are one run of blist, a lane each, 64 at a time (the integral and the slots of
// the vertex's row), then the vertices' lanes add them in their order.  MAT: add
// the rows of alpha*u*v into vals (slots of row v); otherwise add g*v into b[v]
// (rows with skip[v] set are left alone: they are the Dirichlet rows that on(...)
// overwrites afterwards).  Bound by the chain of a lane (points, searches): a
// lane per vertex with all its items took 42 us (matrix) and 15 (right-hand side)
// on a 61 x 50 x 43 box, now 26 and 10.
// Most waves find no item, so what a mesh's inside costs is the number of blocks,
// and what its boundary costs is a wave's chain.  us, 64 threads and 16 vertices a
// wave / 256 and 16 / 256 and 32 / 256 and 64: right-hand side square(300) 6.3 / 6.2 /
// 6.2 / 6.9, square(1000) 18.4 / 9.1 / 7.6 / 7.1, square(2000) 58.6 / 25.0 / 15.5 / 10.1,
// cube(64) 12.1 / 12.0 / 12.4 / 18.2, cube(160) 64.9 / 49.9 / 45.0 / 45.6, cube(200) 117 /
// 79.0 / 65.3 / 63.6 (with a sine 131 / 138 / 119 / 121); matrix square(1000) 20.7 / 11.8 /
// 10.1 / 12.3, square(2000) 61.9 / 28.6 / 19.6 / 15.8, cube(30) 20.5 / 21.2 / 27.5 / 49.6,
// cube(200) 200 / 257 / 241 / 252.
template <int NB, bool MAT, int BLOCK, int ROWS>
__global__ __launch_bounds__(BLOCK) void k_p1_boundary(
    int64_t n, const double *__restrict__ xyz, const int32_t *__restrict__ belems,
    const int32_t *__restrict__ blab, Labels labels,
    const int64_t *__restrict__ bptr, const int32_t *__restrict__ blist, BndRule R, int kind,
    double c0, const double *__restrict__ coef, const int64_t *__restrict__ rowptr,
    const int32_t *__restrict__ colidx, double *__restrict__ vals, const uint8_t *__restrict__ skip,
    double *__restrict__ b, int *__restrict__ missing) {
  constexpr int D = NB;  // coordinates per vertex: 3 for faces of a 3D mesh, 2 for edges
  constexpr int NW = BLOCK / kWave;  // the waves run on their own: no block barrier
  __shared__ double sv_[NW][kWave][MAT ? NB : 1];   // an item's entries
  __shared__ int32_t so_[NW][kWave][MAT ? NB : 1];  // their slots in the row, -1: none
  const int lane = NW == 1 ? threadIdx.x : threadIdx.x % kWave;
  const int w = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  auto &sv = sv_[w];
  auto &so = so_[w];
  const int64_t v0 = ((int64_t)blockIdx.x * NW + w) * ROWS, v1 = v0 + ROWS < n ? v0 + ROWS : n;
  if (NW > 1 && v0 >= n) return;
  const int64_t kbeg = bptr[v0], kend = bptr[v1];
  if (kbeg == kend) return;
  // lane < ROWS: a vertex, its items [q0, q1)
  const int64_t own = v0 + lane;
  int64_t q0 = kend, q1 = kend, r0 = 0;
  double bv = 0.;
  if (lane < ROWS && own < n) {
    q0 = bptr[own];
    q1 = bptr[own + 1];
    if (q0 < q1) {
      if (MAT) r0 = rowptr[own];
      else if (skip && skip[own]) q1 = q0;
      else bv = b[own];
    }
  }
  for (int64_t kc = kbeg; kc < kend; kc += kWave) {
    const int64_t k = kc + lane;
    int32_t item = 0;
    int64_t e = 0;
    bool on = k < kend;
    if (on) {
      item = blist[k];
      e = item / NB;
      on = labels.has(blab[e]);
    }
#pragma unroll
    for (int m = 0; m < (MAT ? NB : 1); ++m) {
      so[lane][m] = -1;
      if (!MAT) sv[lane][m] = 0.;
    }
    if (on) {
      const int l = item - (int)e * NB;
      double B[NB][D];
      int32_t vid[NB];
#pragma unroll
      for (int m = 0; m < NB; ++m) {
        vid[m] = belems[NB * e + m];
#pragma unroll
        for (int c = 0; c < D; ++c) B[m][c] = xyz[(int64_t)D * vid[m] + c];
      }
      double meas;
      if constexpr (NB == 3) {  // |N| / 2 with N the cross product of two edges
        const double a0 = B[1][0] - B[0][0], a1 = B[1][1] - B[0][1], a2 = B[1][2] - B[0][2];
        const double c0_ = B[2][0] - B[0][0], c1 = B[2][1] - B[0][1], c2 = B[2][2] - B[0][2];
        const double N0 = a1 * c2 - a2 * c1, N1 = a2 * c0_ - a0 * c2, N2 = a0 * c1 - a1 * c0_;
        meas = 0.5 * sqrt(N0 * N0 + N1 * N1 + N2 * N2);
      } else {
        const double E0 = B[1][0] - B[0][0], E1 = B[1][1] - B[0][1];
        meas = sqrt(E0 * E0 + E1 * E1);
      }
      double row[NB];
#pragma unroll
      for (int m = 0; m < NB; ++m) row[m] = 0.;
      double r = 0.;
      for (int q = 0; q < R.nq; ++q) {
        double lam[NB];
        if constexpr (NB == 3) {
          lam[0] = 1. - R.s[q] - R.t[q]; lam[1] = R.s[q]; lam[2] = R.t[q];
        } else {
          lam[0] = 1. - R.s[q]; lam[1] = R.s[q];
        }
        double ll = lam[0];  // lam[l] without a dynamically indexed register array
#pragma unroll
        for (int m = 1; m < NB; ++m) ll = l == m ? lam[m] : ll;
        double P[3] = {0., 0., 0.};
#pragma unroll
        for (int c = 0; c < D; ++c) {
          double x = 0.;
#pragma unroll
          for (int m = 0; m < NB; ++m) x += lam[m] * B[m][c];
          P[c] = x;
        }
        const double W = meas * R.w[q] * coef_at(kind, c0, coef, e, q, R.nq, P, D);
        if (MAT) {
#pragma unroll
          for (int m = 0; m < NB; ++m) row[m] += W * ll * lam[m];
        } else {
          r += W * ll;
        }
      }
      if (MAT) {
        int32_t v = vid[0];  // the item's vertex
#pragma unroll
        for (int m = 1; m < NB; ++m) v = l == m ? vid[m] : v;
        const int64_t a0 = rowptr[v];
        const int L = (int)(rowptr[v + 1] - a0);
        int lo[NB], hi[NB];  // first column >= vid[m]: the searches step together
#pragma unroll
        for (int m = 0; m < NB; ++m) { lo[m] = 0; hi[m] = L; }
        for (int w = L; w > 0; w >>= 1) {
          int32_t c[NB];
#pragma unroll
          for (int m = 0; m < NB; ++m) c[m] = lo[m] < hi[m] ? colidx[a0 + ((lo[m] + hi[m]) >> 1)] : 0;
#pragma unroll
          for (int m = 0; m < NB; ++m) {
            const int mid = (lo[m] + hi[m]) >> 1;
            if (lo[m] < hi[m]) {
              if (c[m] < vid[m]) lo[m] = mid + 1; else hi[m] = mid;
            }
          }
        }
#pragma unroll
        for (int m = 0; m < NB; ++m) {
          const bool there = lo[m] < L && colidx[a0 + lo[m]] == vid[m];
          if (!there) *missing = 1;
          so[lane][m] = there ? lo[m] : -1;
          sv[lane][m] = row[m];
        }
      } else {
        so[lane][0] = 0;
        sv[lane][0] = r;
      }
    }
    wave_lds_sync();
    const int b0 = (int)((q0 > kc ? q0 : kc) - kc), b1 = (int)((q1 < kc + kWave ? q1 : kc + kWave) - kc);
    for (int i = b0; i < b1; ++i) {
      if (MAT) {
        double a[NB];
#pragma unroll
        for (int m = 0; m < NB; ++m)
          if (so[i][m] >= 0) a[m] = vals[r0 + so[i][m]];
#pragma unroll
        for (int m = 0; m < NB; ++m)
          if (so[i][m] >= 0) vals[r0 + so[i][m]] = a[m] + sv[i][m];
      } else if (so[i][0] >= 0) {
        bv += sv[i][0];
      }
    }
    wave_lds_sync();
  }
  if (!MAT && q0 < q1) b[own] = bv;
}

// vertex -> (boundary element * nbloc + local) lists, boundary-element order
void build_b2v(ffhip_mesh m) {
  if (m->b2e_ptr) return;
  build_incidence(m->ctx, m->belems, m->nbe, m->nbloc, m->nv, &m->b2e_ptr, &m->b2e, nullptr,
                  nullptr, nullptr);
}

// device copy of a coefficient array (nullptr when none is needed)
const double *coef_device(ffhip_mesh m, int kind, const double *coef, int on_device,
                          double **owned) {
  *owned = nullptr;
  if (kind != FFHIP_COEF_P0 && kind != FFHIP_COEF_QP) return nullptr;
  FFHIP_REQUIRE(coef, FFHIP_ERR_ARG, "boundary term: coefficient array missing");
  if (on_device) return coef;
  const int64_t cnt = kind == FFHIP_COEF_P0 ? m->nbe : m->nbe * (m->dim == 3 ? 7 : 3);
  *owned = dalloc<double>(cnt);
  FFHIP_CHECK(hipMemcpyAsync(*owned, coef, 8 * cnt, hipMemcpyHostToDevice, m->ctx->stream));
  return *owned;
}

bool valid_kind(int k) {
  return k == FFHIP_COEF_CONST || k == FFHIP_COEF_SIN3 || k == FFHIP_COEF_P0 || k == FFHIP_COEF_QP;
}

}  // namespace
}  // namespace ffhip

using namespace ffhip;

extern "C" {

int ffhip_assemble_p1_boundary(ffhip_ctx ctx, ffhip_mesh m, ffhip_mat A, const int32_t *labels,
                               int nlab, int kind, double c0, const double *coef, int on_device) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && m && A && A->n == m->nv && A->ncomp == 0 && A->vals, FFHIP_ERR_ARG,
                  "ffhip_assemble_p1_boundary: needs the P1 matrix of this mesh");
    FFHIP_REQUIRE(nlab > 0 && labels, FFHIP_ERR_ARG, "ffhip_assemble_p1_boundary: labels");
    FFHIP_REQUIRE(valid_kind(kind), FFHIP_ERR_ARG, "ffhip_assemble_p1_boundary: coefficient kind");
    if (m->nbe == 0) return;
    hipStream_t s = ctx->stream;
    build_b2v(m);
    double *owned;
    const double *cd = coef_device(m, kind, coef, on_device, &owned);
    const LabelArg labs(ctx, labels, nlab);
    int *missing = ctx->flag(0);
    const BndRule R = rule(m->dim);
    ctx->tic();
    auto run = [&](auto kernel, int block, int rows) {
      kernel<<<nblocks(m->nv, rows * (block / kWave)), block, 0, s>>>(
          m->nv, m->xyz, m->belems, m->blab, labs.L, m->b2e_ptr, m->b2e, R, kind, c0, cd, A->rowptr,
          A->colidx, A->vals, nullptr, nullptr, missing);
    };
    if (m->dim == 3) run(k_p1_boundary<3, true, 64, 16>, 64, 16);
    else if (m->nv <= 1 << 21) run(k_p1_boundary<2, true, 256, 32>, 256, 32);
    else run(k_p1_boundary<2, true, 256, 64>, 256, 64);
    FFHIP_CHECK(hipGetLastError());
    ctx->toc();
    const int miss = *missing;
    dfree(owned);
    FFHIP_REQUIRE(miss == 0, FFHIP_ERR_ARG,
                  "ffhip_assemble_p1_boundary: a boundary element is not a face of the mesh");
  });
}

int ffhip_rhs_p1_boundary(ffhip_ctx ctx, ffhip_mesh m, const int32_t *labels, int nlab, int kind,
                          double g0, const double *coef, const int32_t *dlabels, int ndlab,
                          double *b, int on_device) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && m && b, FFHIP_ERR_ARG, "ffhip_rhs_p1_boundary: bad arguments");
    FFHIP_REQUIRE(nlab > 0 && labels, FFHIP_ERR_ARG, "ffhip_rhs_p1_boundary: labels");
    FFHIP_REQUIRE(ndlab >= 0 && (ndlab == 0 || dlabels), FFHIP_ERR_ARG,
                  "ffhip_rhs_p1_boundary: Dirichlet labels");
    FFHIP_REQUIRE(valid_kind(kind), FFHIP_ERR_ARG, "ffhip_rhs_p1_boundary: coefficient kind");
    if (m->nbe == 0) return;
    hipStream_t s = ctx->stream;
    const int64_t n = m->nv;
    build_b2v(m);
    double *owned;
    const double *cd = coef_device(m, kind, coef, on_device, &owned);
    const LabelArg labs(ctx, labels, nlab), dlabs(ctx, dlabels, ndlab);
    uint8_t *skip = nullptr;
    if (ndlab) {
      skip = dalloc<uint8_t>(n);
      mark_bc(ctx, m, dlabs.L, skip);
    }
    double *bd = b;
    if (!on_device) {
      bd = dalloc<double>(n);
      FFHIP_CHECK(hipMemcpyAsync(bd, b, 8 * n, hipMemcpyHostToDevice, s));
    }
    const BndRule R = rule(m->dim);
    ctx->tic();
    auto run = [&](auto kernel, int block, int rows) {
      kernel<<<nblocks(n, rows * (block / kWave)), block, 0, s>>>(
          n, m->xyz, m->belems, m->blab, labs.L, m->b2e_ptr, m->b2e, R, kind, g0, cd, nullptr, nullptr,
          nullptr, skip, bd, nullptr);
    };
    if (m->dim == 2 && n <= 1 << 21) run(k_p1_boundary<2, false, 256, 32>, 256, 32);
    else if (m->dim == 2) run(k_p1_boundary<2, false, 256, 64>, 256, 64);
    else if (n <= 1 << 22) run(k_p1_boundary<3, false, 64, 16>, 64, 16);
    else run(k_p1_boundary<3, false, 256, 32>, 256, 32);
    FFHIP_CHECK(hipGetLastError());
    ctx->toc();
    if (!on_device) {
      FFHIP_CHECK(hipMemcpy(b, bd, 8 * n, hipMemcpyDeviceToHost));
      dfree(bd);
    }
    dfree(skip); dfree(owned);
  });
}

}  // extern "C"
