// ffhip_cg.hip — Jacobi-preconditioned conjugate gradient on one MI355X.
//
// Replaces SolverCG / HMatVirtPrecon / ConjugueGradient
// (src/femlib/VirtualSolverCG.hpp:13-192, src/femlib/CG.cpp:195-265).
//
// Layout: the solver streams the matrix in sliced ELL with 64-row slices
// (one wavefront per slice, one lane per row, column-major inside a slice),
// so every matrix load of a wave is one contiguous 256 B (int32) / 512 B
// (FP64) segment and no cross-lane reduction is needed per row.
//
// Iteration (same recurrences as ConjugueGradient):
//   K1: x += rho H_prev; H = gamma*H_prev - C g, partial sum of (g,H)
//   K2: AH = A H, partial sum of (H,AH)
//   K3: rho = -(g,H)/(H,AH); g += rho AH; (g, D^-1 g)
// Systems in the caches form H in K2, for every gathered column (k_pcg_dir_matvec,
// k_mix_dir_matvec); long solves of large box matrices read half of the values
// (k_pcg_matvec_sym); small systems are solved by one workgroup (k_pcg_small).
// Each kernel starts by re-reducing the previous kernel's per-block partial
// sums in a fixed order, so all blocks derive identical scalars with no
// cross-block atomics or fences, and the result is bitwise reproducible.
// Convergence is decided on the device (sticky done flag); the host only
// polls every few iterations.
//
// MIXED mode: the FP32 copy of D^-1/2 A D^-1/2 is streamed by an FP32 CG
// whose iterate is folded into the FP64 solution and whose residual is
// replaced by the FP64 residual b - A x at reliable-update points
// (iterative refinement that keeps the Krylov direction); dot products are
// accumulated in FP64 and convergence is only accepted on the FP64 residual.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <vector>

#include "ffhip_internal.hpp"

namespace ffhip {
void build_v2e(ffhip_mesh m);
bool transpose_map(ffhip_ctx ctx, ffhip_mat A, int64_t *tmap);

constexpr int kSlice = 64;
constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kSlice;

// Tuning of the streaming mat-vec kernels: unroll depth of a row (sliced ELL;
// 3x3-block rows with FP64 and with FP32 values), the waves per SIMD the
// register allocation targets, and resident blocks per CU.
#ifndef FFHIP_SELL_U
#define FFHIP_SELL_U 16
#endif
#ifndef FFHIP_WPE
#define FFHIP_WPE 3
#endif
#ifndef FFHIP_BSR_U
#define FFHIP_BSR_U 2
#endif
#ifndef FFHIP_BSR_U32
#define FFHIP_BSR_U32 8
#endif
#ifndef FFHIP_GRID_PER_CU
#define FFHIP_GRID_PER_CU (FFHIP_WPE)
#endif
#define FFHIP_MATVEC_ATTR __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(FFHIP_WPE, FFHIP_WPE)))
// A matrix of up to this many bytes per mat-vec is read with plain loads: it
// stays in the Infinity Cache (256 MiB).  Both sides measured, plain against
// non-temporal: cube(96) FP64 (134 MB) 25.4 / 32.4 us, cube(112) (214 MB) 40.6 /
// 49.0, cube(24) [P2,P2,P2] (250 MB) 46 / 61, cube(136) FP32 (229 MB) 41 / 46;
// beyond: cube(120) FP64 (264 MB) 61.8 / 60.6, cube(144) FP32 (272 MB) 56.7 / 53.9,
// cube(160) FP64 (644 MB) 150.5 / 139.6.
constexpr int64_t kCachedMatrix = 256000000;
constexpr int kU = FFHIP_SELL_U;

// matrix layouts of the mat-vec kernels (described at MatFmt below)
constexpr int kSell = 0;
constexpr int kCsrV = 1;
constexpr int kSell16 = 2;  // sliced ELL with 16-bit column deltas (col - row)
constexpr int kBsr3 = 3;    // 3x3 blocks of the [P2,P2,P2] node rows, a block's waves on a slice together
constexpr int kBsr3W = 4;   // the same layout, a wave per slice (a kernel of its own: never a solver's fmt)
// MIXED: the FP32 residual is replaced by the FP64 one once (r32, r32) fell by
// this factor since the last replacement (every two decades of the residual
// norm: FP32 recurrences of ill-conditioned systems, e.g. vector P2
// elasticity, drift if left longer; P1 Poisson is insensitive to it)
constexpr double kMixUpdate = 1e-2;
constexpr int kLanesPerRow = 16;

struct CgState {
  double gcg_prev[2];  // (g, Cg) at the start of the iteration, by parity
  double gcg0, eps2;
  double sigma;        // MIXED: scale of the FP32 residual
  double rho32;        // MIXED: (r32, r32) at the start of the last executed step
  int done;            // 0 run, 1 converged, 2 gcg0 < 1e-30, 3 itmax, 4 NaN
  int iters;
  int need_update;     // MIXED: reliable update requested
  int refinements;
  // iteration of the first launch of the current chunk (the kernels add their
  // position in the chunk; k_cg_advance moves it on), so one captured chunk
  // serves every chunk of a solve
  int it0;
  int itmax;
  double eps;
  // FP64 PCG: the stop decision of the direction kernel (published as done by
  // the next mat-vec launch, so every block of the deciding launch still runs)
  // and the step length of the last update, whose x += rho H the next
  // direction kernel applies
  int stop;
  double rho;
};

// ---------------------------------------------------------------- reductions
// Sum of P partials (stride `stride`, component `c`), identical in every block.
__device__ inline double reduce_partials(const double *__restrict__ p, int P, int stride, int c,
                                         double *lds) {
  double s = 0.;
  for (int i = threadIdx.x; i < P; i += kBlock) s += p[(int64_t)i * stride + c];
  return block_sum<kBlock>(s, lds);
}

// Loads of the streamed matrix: NT past every cache (a matrix that does not
// fit in the Infinity Cache would only push the vectors out of it), else
// plain, so that a matrix that fits stays there from one mat-vec to the next
// (MatFmt::nt).
template <bool NT, class T>
__device__ inline T mload(const T *p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}

// One row of a slice: sum_k a_k * X(j_k) over the L (wave-uniform) entries of
// this lane's row.  Unrolled by U: the U column and value loads of a round
// are all issued before any gather, so every wave keeps 2U streaming loads
// and U (or 2U) gathers in flight instead of one dependent chain per entry.
// IT = int32_t: absolute columns; IT = int16_t: deltas to the row (row0 + d).
template <bool NT, int U, class V, class ACC, class IT, class F>
__device__ inline ACC sell_row(const IT *__restrict__ colp, const V *__restrict__ valp, int L,
                               int32_t row0, F xval) {
  ACC acc = 0;
  for (int k = 0; k < L; k += U) {
    int32_t j[U];
    V a[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      j[u] = row0;  // past the row end: a valid column with a zero value
      a[u] = 0;
      if (k + u < L) {
        const IT c = mload<NT>(colp + (int64_t)(k + u) * kSlice);
        j[u] = sizeof(IT) == 2 ? row0 + (int32_t)c : (int32_t)c;
        a[u] = mload<NT>(valp + (int64_t)(k + u) * kSlice);
      }
    }
    ACC xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) xv[u] = xval(j[u]);  // all gathers issued together
#pragma unroll
    for (int u = 0; u < U; ++u) acc += (ACC)a[u] * xv[u];
  }
  return acc;
}

// 16-bit column deltas packed four per lane: the deltas of entries 4g..4g+3 of
// a lane's row are one 8-byte load (layout [g][lane][4] inside a slice), so a
// round of U entries issues U/4 index loads ahead of the U value loads.
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// FP64 values of a kSell16 slice of width L are stored in entry pairs: pair m
// (entries 2m, 2m+1) of lane l at 2 (64 m + l), so one 16-byte load per lane
// reads two entries of its row; for odd L the last entry follows the L/2 pair
// planes as one plane of single values.  Position of entry k of lane l,
// relative to the slice start:
__host__ __device__ inline int64_t pair_pos(int L, int k, int lane) {
  const int h = L >> 1;
  return (k >> 1) < h ? ((int64_t)(k >> 1) * kSlice + lane) * 2 + (k & 1) : (int64_t)h * 2 * kSlice + lane;
}

template <bool NT, int U, class V, class ACC, class F>
__device__ inline ACC sell_row16(const int16_t *__restrict__ colp, const V *__restrict__ valp,
                                 int L, int32_t row0, F xval) {
  static_assert(U % 4 == 0, "unroll by whole index groups");
  ACC acc = 0;
  for (int k = 0; k < L; k += U) {
    int32_t j[U];
    V a[U];
#pragma unroll
    for (int g = 0; g < U / 4; ++g) {
      u32x2 pk = {0u, 0u};  // past the row end: deltas 0 (the row itself)
      if (k + 4 * g < L)
        pk = mload<NT>(reinterpret_cast<const u32x2 *>(colp + (int64_t)((k >> 2) + g) * (4 * kSlice)));
      j[4 * g + 0] = row0 + (int32_t)(int16_t)(pk.x & 0xffffu);
      j[4 * g + 1] = row0 + (int32_t)(int16_t)(pk.x >> 16);
      j[4 * g + 2] = row0 + (int32_t)(int16_t)(pk.y & 0xffffu);
      j[4 * g + 3] = row0 + (int32_t)(int16_t)(pk.y >> 16);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      a[u] = 0;
      if (k + u < L) a[u] = mload<NT>(valp + (int64_t)(k + u) * kSlice);
    }
    ACC xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) xv[u] = xval(j[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) acc += (ACC)a[u] * xv[u];
  }
  return acc;
}

// wave-uniform slice index (kept in scalar registers)
__device__ inline int64_t uniform(int64_t v) {
  const int lo = __builtin_amdgcn_readfirstlane((int)(v & 0xffffffff));
  const int hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
  return ((int64_t)hi << 32) | (uint32_t)lo;
}
__device__ inline int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x / kSlice); }

// Slices of this wave in the streaming sliced-ELL kernels: each XCD's
// contiguous slice range is walked by all of its waves together, wave q taking
// slices q, q + Q, q + 2Q, ... (Q waves on the XCD), so the XCD streams one
// contiguous window of Q slices at a time and a column's x value, needed by
// rows up to one window-width apart (the plane neighbours of a 3D mesh), is
// re-read while still in that XCD's L2 (cube(160) P1: 8 % less HBM fetch, the
// FP32 mat-vec 6 % faster than with a contiguous chunk per block).  The
// [P2,P2,P2] block layout, whose node rows are sorted by length in windows, ran
// 1.8x slower this way and walks chunks.
__device__ inline void wave_slices(int64_t S, int64_t &first, int64_t &end, int64_t &stride) {
  const int G = gridDim.x, b = blockIdx.x;
  const int groups = (G % 8) ? 1 : 8;
  const int grp = b % groups, loc = b / groups, nloc = G / groups;
  first = (grp * S) / groups + (int64_t)loc * kWavesPerBlock + wave_id();
  end = ((grp + 1) * S) / groups;
  stride = (int64_t)nloc * kWavesPerBlock;
}

// the maximum over a wave, in every lane
__device__ inline int wave_max(int v) {
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off, kWave));
  return v;
}

// ---------------------------------------------------------------- SELL build
// What the solver set-up reads back to the host, in one copy: the tgv
// figures (k_tgv_reduce), the layout sizes (k_setup_sizes) and the columns' order
// (sample_order).
struct SetupRb {
  double ttgv, ntgv;      // the tgv value (0: none) and the count of rows holding it
  int64_t ents, ents16;   // entries of the sliced layout, of its packed 16-bit deltas
  int far;                // some column is more than 2^15 from its row
  // of sampled rows: entries, those whose place in the next row holds the next
  // column, and those where it holds one within kNear columns
  int entries, next, near_;
};

// How far apart the values lie that lanes on consecutive rows gather: 128 pairs of
// rows (r, r + 1) spread by the golden ratio (an even spread would meet the ends of
// a box's lines), 16 lanes on the first 16 entries of a pair, every load of the
// pairs in flight together.  n > 1.
constexpr int kNear = 64, kOrderBlock = 256;
__device__ inline void sample_order(int64_t n, const int64_t *__restrict__ rowptr,
                                    const int32_t *__restrict__ colidx, SetupRb *__restrict__ rb) {
  __shared__ double lds[kOrderBlock / kWave];
  constexpr int Q = 8;
  const int g = threadIdx.x / 16, k = threadIdx.x % 16;
  int64_t p0[Q], p1[Q], p2[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const uint32_t u = (uint32_t)(g * Q + q) * 2654435769u;
    const int64_t r = (int64_t)(((uint64_t)u * (uint64_t)(n - 1)) >> 32);
    p0[q] = rowptr[r];
    p1[q] = rowptr[r + 1];
    p2[q] = rowptr[r + 2];
  }
  int entries = 0, next = 0, near_ = 0;
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const bool in = p0[q] + k < p1[q], both = in && p1[q] + k < p2[q];
    const int d = both ? colidx[p1[q] + k] - colidx[p0[q] + k] : INT_MAX;
    entries += in;
    next += d == 1;
    near_ += d >= -kNear && d <= kNear;
  }
  const double e = block_sum<kOrderBlock>(entries, lds), a = block_sum<kOrderBlock>(next, lds),
               b = block_sum<kOrderBlock>(near_, lds);
  if (threadIdx.x != 0) return;
  rb->entries = (int)e;
  rb->next = (int)a;
  rb->near_ = (int)b;
}

// the widest row of each slice: a wave per slice (a lane per slice walked its 64
// rows: 13 us for P2 on a 27 x 24 x 21 box, square(200) 11); with colidx a block past
// the slices' samples the order of the columns meanwhile
__global__ __launch_bounds__(kOrderBlock) void k_sell_len(int64_t n, int64_t S, const int64_t *__restrict__ rowptr,
                                                          const int32_t *__restrict__ colidx, SetupRb *__restrict__ rb,
                                                          int32_t *__restrict__ len, int64_t *__restrict__ cnt) {
  if (colidx && blockIdx.x == gridDim.x - 1) {
    sample_order(n, rowptr, colidx, rb);
    return;
  }
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, s = r / kSlice;
  if (s >= S) return;
  const int m = wave_max(r < n ? (int)(rowptr[r + 1] - rowptr[r]) : 0);
  if (threadIdx.x % kSlice != 0) return;
  len[s] = m;
  cnt[s] = (int64_t)m * kSlice;
  if (s == 0) cnt[S] = 0;  // the scan's last input
}

// vals_src may be permuted through tmap (transposed values)
// One block per 64-row slice: the slice's CSR segment is read once, coalesced,
// into LDS (when it fits in kFillStage entries; otherwise the rows are read
// from memory where they lie), then the block writes the slice layout plane
// by plane, consecutive threads on consecutive rows, so every store is
// coalesced (FP64 entry pairs as one 16-byte store).  Entries past a row's
// end are zeros at the row's own column.
// 1280 entries (a P1 slice of 64 rows of 15 holds 960): 15 KB of LDS, 10
// blocks per CU (2048 entries, 6 blocks per CU: cube(160) 401 -> 330 us)
constexpr int kFillStage = 1280;
__global__ __launch_bounds__(256) void k_sell_fill(
    int64_t n, int64_t S, const int64_t *__restrict__ rowptr, const int32_t *__restrict__ colidx,
    const double *__restrict__ vals, const int64_t *__restrict__ tmap,
    const int64_t *__restrict__ sptr, const int32_t *__restrict__ len,
    const double *__restrict__ dsc, int32_t *__restrict__ scol,
    const int64_t *__restrict__ sptr16, int16_t *__restrict__ scol16, double *__restrict__ sval,
    float *__restrict__ sval32, bool pairs, const int64_t *__restrict__ diag,
    double *__restrict__ dout, uint8_t *__restrict__ hout, int *__restrict__ far) {
  __shared__ int32_t lc[kFillStage];
  __shared__ double lv[kFillStage];
  __shared__ int64_t rs[kSlice];  // row start (in the stage, or in the CSR)
  __shared__ int32_t rl[kSlice];  // row length
  const int t = threadIdx.x;
  const int64_t sl = blockIdx.x;
  const int64_t r0 = sl * kSlice;
  const int64_t rend = r0 + kSlice < n ? r0 + kSlice : n;
  const int64_t seg0 = r0 < n ? rowptr[r0] : 0, seg1 = r0 < n ? rowptr[rend] : 0;
  const bool staged = seg1 - seg0 <= kFillStage;
  if (t < kSlice) {
    const int64_t r = r0 + t;
    const int64_t p = r < n ? rowptr[r] : 0;
    rs[t] = staged ? p - seg0 : p;
    rl[t] = r < n ? (int32_t)(rowptr[r + 1] - p) : 0;
  }
  if (staged)
    for (int64_t i = t; i < seg1 - seg0; i += blockDim.x) {
      lc[i] = colidx[seg0 + i];
      lv[i] = tmap ? vals[tmap[seg0 + i]] : vals[seg0 + i];
    }
  __syncthreads();
  if (dout && t < kSlice && r0 + t < n) {  // the diagonal of the Jacobi set-up (as k_diag_vals)
    const int64_t r = r0 + t, q = diag[r];
    dout[r] = q < 0 ? 0. : (staged && !tmap && q >= seg0 && q < seg1 ? lv[q - seg0] : vals[q]);
    hout[r] = q >= 0;
  }
  const int L = len[sl];
  const int64_t base = sptr[sl];
  // entry k of lane li's row; past its end a zero at the row's own column
  auto col = [&](int li, int k) -> int32_t {
    if (k < rl[li]) return staged ? lc[rs[li] + k] : colidx[rs[li] + k];
    const int64_t r = r0 + li;
    return r < n ? (int32_t)r : 0;
  };
  auto val = [&](int li, int k) -> double {
    if (k >= rl[li]) return 0.;
    const int64_t q = rs[li] + k;
    return staged ? lv[q] : (tmap ? vals[tmap[q]] : vals[q]);
  };
  if (sval && pairs) {
    const int Lh = L >> 1;
    for (int it = t; it < (Lh + (L & 1)) * kSlice; it += blockDim.x) {
      const int li = it % kSlice, kp = it / kSlice;
      if (kp < Lh)
        *reinterpret_cast<double2 *>(sval + base + ((int64_t)kp * kSlice + li) * 2) =
            double2{val(li, 2 * kp), val(li, 2 * kp + 1)};
      else  // the odd last entry: its own plane after the pairs
        sval[base + pair_pos(L, L - 1, li)] = val(li, L - 1);
    }
  }
  for (int it = t; it < L * kSlice; it += blockDim.x) {
    const int li = it % kSlice, k = it / kSlice;
    const int64_t idx = base + it;  // entry k of lane li: k kSlice + li
    if (sval && !pairs) sval[idx] = val(li, k);
    if (scol || sval32) {
      const int32_t c = col(li, k);
      if (scol) scol[idx] = c;
      if (sval32)
        sval32[idx] = k < rl[li] ? (float)(val(li, k) * dsc[r0 + li] * dsc[c]) : 0.f;
    }
  }
  if (scol16) {  // [g][lane][4] packed deltas, the group tail padded with 0: one 8-byte store per group
    for (int it = t; it < ((L + 3) >> 2) * kSlice; it += blockDim.x) {
      const int li = it % kSlice, g = it / kSlice;
      const int64_t r = r0 + li;
      uint32_t h[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = 4 * g + q;
        const int64_t dl = k < rl[li] ? (int64_t)col(li, k) - r : 0;
        if (far && (dl < -32768 || dl > 32767)) atomicOr(far, 1);  // then refilled with int32 columns
        h[q] = (uint32_t)(uint16_t)(int16_t)dl;
      }
      const u32x2 pk = {h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
      *reinterpret_cast<u32x2 *>(scol16 + sptr16[sl] + (int64_t)it * 4) = pk;
    }
  }
}

// slice sizes of the packed 16-bit index array (widths rounded up to 4)
__global__ void k_sell_len4(int64_t S, const int32_t *__restrict__ len, int64_t *__restrict__ cnt) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s < S) cnt[s] = (int64_t)((len[s] + 3) & ~3) * kSlice;
  if (s == 0) cnt[S] = 0;
}

// node-row sort keys: window of 4096 rows in the high bits, longer rows first
__global__ void k_bsr_keys(int64_t nb, const int64_t *__restrict__ bptr, uint32_t *__restrict__ key,
                           int32_t *__restrict__ val) {
  const int64_t a = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= nb) return;
  const int64_t L = bptr[a + 1] - bptr[a];
  key[a] = ((uint32_t)(a >> 12) << 8) | (uint32_t)(255 - (L < 255 ? L : 255));
  val[a] = (int32_t)a;
}

// slice widths of the sorted node rows
__global__ void k_bsr_len(int64_t nb, int64_t S3, const int64_t *__restrict__ bptr,
                          const int32_t *__restrict__ perm, int32_t *__restrict__ len,
                          int64_t *__restrict__ cnt) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, s = i / kSlice;
  if (s >= S3) return;
  int m = 0;
  if (i < nb) {
    const int32_t a = perm[i];
    m = (int)(bptr[a + 1] - bptr[a]);
  }
  m = wave_max(m);
  if (threadIdx.x % kSlice != 0) return;
  len[s] = m;
  cnt[s] = (int64_t)m * kSlice;
  if (s == 0) cnt[S3] = 0;
}

// 3x3 blocks of a vector-P2 matrix from its scalar CSR: entry k of sorted node
// row i (node a = perm[i]) holds rows 3a..3a+2 at offsets 3k..3k+2 of those
// rows (values optionally through tmap; FP32 copy of D^-1/2 A D^-1/2).
// One block per 64-row slice: the slice's rows are read KC blocks at a time,
// each of its 3 x 64 scalar rows as one contiguous run of 3 KC values, into
// LDS (the next KC blocks' values already on their way while these are written),
// and written out entry-major, a thread per block entry (the 9 x 64 values of
// block entry k of the slice at 9 ptr[s] + 9 64 k, placed by bsr_pos, as
// 16-byte vectors); padding entries get value 0 and the row's own block column.
// Bound by HBM: 12 B read and 8 (+ 4) written per value.  cube(32) with both
// copies: 1175 us with one value per thread and step (two loads in flight, a
// scaling gather per value and side), now 512 us, 3.1 TB/s (KC = 4: 617 us,
// KC = 12: 534 us).
constexpr int kBsrKC = 8;
// Position of value q (3c + c') of lane li inside one slice entry of the
// 3x3-block values (9 x 64 values per entry): values 0..7 in vectors of W = 16
// bytes / sizeof(value) per lane (FP64 pairs, FP32 quads), [vector][lane][W],
// then value 8 of the 64 lanes.
template <class V>
__host__ __device__ constexpr int bsr_pos(int q, int li) {
  constexpr int W = 16 / (int)sizeof(V);
  return q < 8 ? ((q / W) * kSlice + li) * W + q % W : 8 * kSlice + li;
}
template <bool TMAP>
__global__ __launch_bounds__(256) void k_bsr_fill(
    int64_t nb, const int64_t *__restrict__ bptr, const int32_t *__restrict__ perm,
    const int64_t *__restrict__ sptr, const int32_t *__restrict__ slen,
    const int64_t *__restrict__ rowptr, const int32_t *__restrict__ colidx,
    const double *__restrict__ vals, const int64_t *__restrict__ tmap,
    const double *__restrict__ dsc, int32_t *__restrict__ bcol, double *__restrict__ bval,
    float *__restrict__ bval32) {
  constexpr int KC = kBsrKC, P = kSlice + 1;  // P: padded lane stride (LDS banks)
  constexpr int NL = kSlice * 9 * KC / 256, NE = KC * kSlice / 256;  // values, block entries per thread
  __shared__ double T[9 * KC * P];
  __shared__ int32_t An[kSlice], Ln[kSlice];
  __shared__ int64_t R0[3 * kSlice];
  __shared__ double Ds[3 * kSlice];  // the rows' scaling
  const int64_t s = blockIdx.x;
  const int t = threadIdx.x;
  if (t < kSlice) {
    const int64_t i = s * kSlice + t;
    const int32_t a = i < nb ? perm[i] : -1;
    An[t] = a;
    Ln[t] = a >= 0 ? (int32_t)(bptr[a + 1] - bptr[a]) : 0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      R0[3 * t + c] = a >= 0 ? rowptr[3 * (int64_t)a + c] : 0;
      Ds[3 * t + c] = bval32 && a >= 0 ? dsc[3 * (int64_t)a + c] : 0.;
    }
  }
  __syncthreads();
  const int W = slen[s];
  const int64_t base = sptr[s];
  // item u of thread t: t + 256 u = (li * 3 + c) * 3 KC + x, x = 3 kk + cp
  auto load = [&](int k0, double (&v)[NL], int32_t (&cb)[NE]) {
#pragma unroll
    for (int u = 0; u < NL; ++u) {
      const int it = t + 256 * u, x = it % (3 * KC), rc = it / (3 * KC);
      const int k = k0 + x / 3;
      v[u] = 0.;
      if (k < Ln[rc / 3]) {
        const int64_t src = R0[rc] + 3 * (int64_t)k0 + x;
        v[u] = TMAP ? vals[tmap[src]] : vals[src];
      }
    }
#pragma unroll
    for (int u = 0; u < NE; ++u) {
      const int li = (t + 256 * u) % kSlice, k = k0 + (t + 256 * u) / kSlice;
      cb[u] = k < Ln[li] ? colidx[R0[3 * li] + 3 * (int64_t)k] : -1;
    }
  };
  double v[NL];
  int32_t cb[NE];
  load(0, v, cb);
  for (int k0 = 0; k0 < W; k0 += KC) {
#pragma unroll
    for (int u = 0; u < NL; ++u) {
      const int it = t + 256 * u, x = it % (3 * KC), rc = it / (3 * KC);
      T[((3 * (rc % 3) + x % 3) * KC + x / 3) * P + rc / 3] = v[u];
    }
    int32_t col[NE];
#pragma unroll
    for (int u = 0; u < NE; ++u) col[u] = cb[u] < 0 ? -1 : cb[u] / 3;
    __syncthreads();
    if (k0 + KC < W) load(k0 + KC, v, cb);
#pragma unroll
    for (int u = 0; u < NE; ++u) {
      const int li = (t + 256 * u) % kSlice, kk = (t + 256 * u) / kSlice;
      if (k0 + kk >= W) continue;
      const int64_t e = base + (int64_t)(k0 + kk) * kSlice, eb = 9 * e;
      double w[9];
#pragma unroll
      for (int q = 0; q < 9; ++q) w[q] = T[(q * KC + kk) * P + li];
      if (bval) {
#pragma unroll
        for (int q = 0; q < 8; q += 2)
          *reinterpret_cast<double2 *>(bval + eb + bsr_pos<double>(q, li)) = double2{w[q], w[q + 1]};
        bval[eb + bsr_pos<double>(8, li)] = w[8];
      }
      if (bval32) {
        double dc[3] = {0., 0., 0.};
        if (col[u] >= 0) {
#pragma unroll
          for (int c = 0; c < 3; ++c) dc[c] = dsc[3 * (int64_t)col[u] + c];
        }
        float f[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) f[q] = col[u] < 0 ? 0.f : (float)(w[q] * Ds[3 * li + q / 3] * dc[q % 3]);
#pragma unroll
        for (int q = 0; q < 8; q += 4)
          *reinterpret_cast<float4 *>(bval32 + eb + bsr_pos<float>(q, li)) =
              float4{f[q], f[q + 1], f[q + 2], f[q + 3]};
        bval32[eb + bsr_pos<float>(8, li)] = f[8];
      }
      if (bcol) bcol[e + li] = col[u] >= 0 ? col[u] : (An[li] >= 0 ? An[li] : 0);
    }
    __syncthreads();
  }
}

// First slice of each of nw blocks (or waves) when the S3 slices are split over
// them by entries: w takes the slices that start in [w E / nw, (w+1) E / nw),
// E = sptr[S3].
__global__ void k_bsr_waves(int64_t S3, const int64_t *__restrict__ sptr, int nw,
                            int32_t *__restrict__ wstart) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w > nw) return;
  const int64_t e = w == nw ? sptr[S3] : (int64_t)w * sptr[S3] / nw;
  int64_t lo = 0, hi = S3;  // first slice s with sptr[s] >= e
  while (lo < hi) {
    const int64_t mid = (lo + hi) / 2;
    if (sptr[mid] < e) lo = mid + 1;
    else hi = mid;
  }
  wstart[w] = (int32_t)lo;
}

// CSR-layout values: A (optionally transposed through tmap) and/or the FP32
// copy of D^-1/2 A D^-1/2, one 16-lane group per row
__global__ void k_csr_fill(int64_t n, const int64_t *__restrict__ rowptr,
                           const int32_t *__restrict__ colidx, const double *__restrict__ vals,
                           const int64_t *__restrict__ tmap, const double *__restrict__ dsc,
                           double *__restrict__ dv, float *__restrict__ fv) {
  const int64_t r = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kLanesPerRow;
  const int lane = threadIdx.x % kLanesPerRow;
  if (r >= n) return;
  const int64_t k1 = rowptr[r + 1];
  for (int64_t k = rowptr[r] + lane; k < k1; k += kLanesPerRow) {
    const double a = tmap ? vals[tmap[k]] : vals[k];
    if (dv) dv[k] = a;
    if (fv) fv[k] = (float)(a * dsc[r] * dsc[colidx[k]]);
  }
}

// ---------------------------------------------------------------- Jacobi / tgv
__global__ void k_diag_vals(int64_t n, const int64_t *__restrict__ diag,
                            const double *__restrict__ vals, double *__restrict__ d,
                            uint8_t *__restrict__ has) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t s = diag[i];
  d[i] = s >= 0 ? vals[s] : 0.;
  has[i] = s >= 0;
}

// pass 1: max diagonal; pass 2: count of the max (*top), max of the rest
// (HashMatrix::gettgv, HashMatrix.cpp:1340-1371)
__global__ void k_tgv_pass(int64_t n, const double *__restrict__ d, const uint8_t *__restrict__ has,
                           const double *__restrict__ topp, int pass, double *__restrict__ out) {
  __shared__ double lds[kBlock / kWave];
  const double top = pass == 2 ? *topp : 0.;
  double m = 0., c = 0.;  // the reference starts from ttgv = max1 = 0
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
    if (!has[i]) continue;
    const double a = d[i];
    if (pass == 1) m = fmax(m, a);
    else if (a == top) c += 1.;
    else m = fmax(m, a);
  }
  // block max via shuffles
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, kWave));
  const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (lane == 0) lds[w] = m;
  __syncthreads();
  double bm = 0.;
  for (int i = 0; i < kBlock / kWave; ++i) bm = fmax(bm, lds[i]);
  const double bc = block_sum<kBlock>(c, lds);
  if (threadIdx.x == 0) { out[2 * blockIdx.x] = bm; out[2 * blockIdx.x + 1] = bc; }
}

// the partials of a k_tgv_pass, one block: pass 1 puts the max in rb->ttgv;
// pass 2 applies gettgv's rule (a max not 1e6 x above the next distinct
// value is no tgv) to that max, the count and the max of the rest.  Maxima
// and integral counts are exact in any order.
__global__ __launch_bounds__(kBlock) void k_tgv_reduce(int GB, const double *__restrict__ part,
                                                       int pass, SetupRb *__restrict__ rb) {
  __shared__ double lds[kBlock / kWave];
  double m = 0., c = 0.;
  for (int i = threadIdx.x; i < GB; i += kBlock) {
    m = fmax(m, part[2 * i]);
    c += part[2 * i + 1];
  }
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, kWave));
  const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (lane == 0) lds[w] = m;
  __syncthreads();
  double bm = 0.;
  for (int i = 0; i < kBlock / kWave; ++i) bm = fmax(bm, lds[i]);
  const double count = block_sum<kBlock>(c, lds);
  if (threadIdx.x != 0) return;
  if (pass == 1) {
    rb->ttgv = bm;
    return;
  }
  double ttgv = rb->ttgv, ntgv = count;
  if (bm * 1e6 > ttgv) { ttgv = 0.; ntgv = 0.; }
  rb->ttgv = ttgv;
  rb->ntgv = ntgv;
}

// the layout sizes for the host (entries of the sliced layout and of the
// packed deltas: the last slice offsets) and the far-column flag's start
__global__ void k_setup_sizes(SetupRb *__restrict__ rb, const int64_t *__restrict__ ents,
                              const int64_t *__restrict__ ents16, int far) {
  rb->ents = ents ? *ents : 0;
  rb->ents16 = ents16 ? *ents16 : 0;
  rb->far = far;
}

__global__ void k_jacobi(int64_t n, const double *__restrict__ d, const uint8_t *__restrict__ has,
                         const SetupRb *__restrict__ rb, double *__restrict__ dinv,
                         double *__restrict__ dsc, uint8_t *__restrict__ wcl) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double tgve = rb->ttgv <= 0 ? 1e200 : rb->ttgv;
  const bool with_wcl = rb->ntgv > 0;
  const double a = has[i] ? d[i] : 0.;  // a missing diagonal reads as 0 (then 1)
  dinv[i] = (a * a < 1e-60) ? 1. : 1. / a;
  dsc[i] = a > 0. ? 1. / sqrt(a) : 1.;
  wcl[i] = with_wcl ? (has[i] && d[i] == tgve) : 0;
}

// SetInitWithBC (VirtualSolverCG.hpp:93-99)
__global__ void k_init_bc(int64_t n, const uint8_t *__restrict__ wcl, const double *__restrict__ b,
                          double tgv, double *__restrict__ x) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && wcl[i]) x[i] = b[i] / tgv;
}

// ---------------------------------------------------------------- matrix formats
// Every mat-vec kernel streams the matrix through one of these layouts:
//   kSell:   sliced ELL, 64-row slices (one lane per row, no reduction) — for
//            matrices whose rows have nearly equal length (P1);
//   kSell16: the same with 16-bit column deltas packed four per lane;
//   kCsrV:   CSR with 16 lanes per row and a shuffle reduction — for rows of
//            very different lengths, where sliced ELL would pad;
//   kBsr3:   3x3 blocks of a vector-P2 matrix, sliced ELL over node rows:
//            the node rows are sorted by length inside windows of 4096 rows
//            (so a 64-row slice pads little), one lane per node row (3 scalar
//            rows), one int32 block column and 9 values per slice entry, the
//            values of a slice entry-major (9 x 64 per entry) — 76 B per 9
//            FP64 entries instead of 108, every load coalesced.
template <class V>
struct MatFmt {
  int64_t n, S;
  const int64_t *ptr;  // kSell*: slice offsets (S+1); kCsrV: row pointers (n+1)
  const int32_t *len;  // kSell*: slice widths
  const int32_t *col;  // kSell, kCsrV
  const int16_t *col16;  // kSell16: col - row, packed [group of 4][lane][4] per slice
  const int64_t *ptr16;  // kSell16: slice offsets of col16
  const V *val;          // kBsr3: 9 ents values, entry k of slice s at 9 ptr[s] + 9 64 k (bsr_pos)
  int64_t nb;            // kBsr3: node rows (ptr/len/col: slices, perm: rows)
  const int32_t *perm;   // kBsr3: node row of each sorted position
  const int32_t *wstart; // kBsr3: first slice of each block (kBsr3W: wave), and the end, split by entries
  bool nt;  // the matrix's loads bypass the caches
};

// Buffer resource over [p, p + bytes): a buffer load at a byte offset past
// `bytes` returns 0 and touches no memory (raw buffer, stride 0).
__device__ inline __amdgpu_buffer_rsrc_t slice_rsrc(const void *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}
constexpr int kBufNT = 2;  // cache policy of a non-temporal buffer load

// Entries k >= U of a kSell16 FP64 row (rows longer than U), summed into acc
// in entry order, four per round (one packed delta group).
template <bool NT, class ACC, class F>
__device__ inline ACC sell16_tail(const int16_t *__restrict__ col16, const double *__restrict__ val,
                                  int L, int lane, int32_t row0, F xval, ACC acc) {
  for (int k = kU; k < L; k += 4) {
    const u32x2 pk = mload<NT>(reinterpret_cast<const u32x2 *>(col16 + (int64_t)(k >> 2) * (4 * kSlice) + 4 * lane));
    const int32_t j[4] = {row0 + (int32_t)(int16_t)(pk.x & 0xffffu), row0 + (int32_t)(int16_t)(pk.x >> 16),
                          row0 + (int32_t)(int16_t)(pk.y & 0xffffu), row0 + (int32_t)(int16_t)(pk.y >> 16)};
    double a[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) a[t] = k + t < L ? mload<NT>(val + pair_pos(L, k + t, lane)) : 0.;
#pragma unroll
    for (int t = 0; t < 4; ++t) acc += (ACC)a[t] * xval(j[t]);
  }
  return acc;
}

// Row r32 (lane `lane` of slice s) of an FP64 kSell16 matrix times X.  A slice's
// values (entry pairs, 16-byte loads) and packed deltas are read through buffer
// resources that end at the slice's last entry, so the loads of a round are
// issued unconditionally: entries past the slice width read as value 0, delta 0
// (the row itself).  pre(r32) (the row's own epilogue operands, into pv) is
// issued with the gathers.  The products are summed in entry order.
template <bool NT, class ACC, class F, class P, class PV>
__device__ inline ACC sell16_slice_row(const MatFmt<double> &M, int64_t s, int lane, int32_t r32, F xval,
                                       P pre, PV &pv) {
  constexpr int U = kU, G4 = kU / 4, NP = kU / 2;
  static_assert(kU % 4 == 0, "unroll by whole index groups");
  const int64_t vb = uniform(M.ptr[s]), cb = uniform(M.ptr16[s]);
  const int L = __builtin_amdgcn_readfirstlane(M.len[s]);
  const int Lh = L >> 1;
  const auto rc = slice_rsrc(M.col16 + cb, (uint32_t)((L + 3) >> 2) * (4 * kSlice) * 2);
  const auto rp = slice_rsrc(M.val + vb, (uint32_t)Lh * (2 * kSlice) * 8);
  const auto r1 = slice_rsrc(M.val + vb + (int64_t)Lh * (2 * kSlice), (uint32_t)(L & 1) * kSlice * 8);
  u32x2 pk[G4];
#pragma unroll
  for (int g = 0; g < G4; ++g)
    pk[g] = __builtin_amdgcn_raw_buffer_load_b64(rc, (g * kSlice + lane) * 8, 0, NT ? kBufNT : 0);
  u32x4 q[NP];
#pragma unroll
  for (int m = 0; m < NP; ++m)
    q[m] = __builtin_amdgcn_raw_buffer_load_b128(rp, (m * kSlice + lane) * 16, 0, NT ? kBufNT : 0);
  const u32x2 odd = __builtin_amdgcn_raw_buffer_load_b64(r1, lane * 8, 0, NT ? kBufNT : 0);
  int32_t j[U];
#pragma unroll
  for (int g = 0; g < G4; ++g) {
    j[4 * g + 0] = r32 + (int32_t)(int16_t)(pk[g].x & 0xffffu);
    j[4 * g + 1] = r32 + (int32_t)(int16_t)(pk[g].x >> 16);
    j[4 * g + 2] = r32 + (int32_t)(int16_t)(pk[g].y & 0xffffu);
    j[4 * g + 3] = r32 + (int32_t)(int16_t)(pk[g].y >> 16);
  }
  double a[U];
#pragma unroll
  for (int m = 0; m < NP; ++m) {
    const u32x2 lo = m == Lh ? odd : u32x2{q[m].x, q[m].y};
    a[2 * m] = __builtin_bit_cast(double, lo);
    a[2 * m + 1] = __builtin_bit_cast(double, u32x2{q[m].z, q[m].w});
  }
  ACC xv[U];
#pragma unroll
  for (int u = 0; u < U; ++u) xv[u] = xval(j[u]);
  pv = pre(r32);
  ACC acc = 0;
#pragma unroll
  for (int u = 0; u < U; ++u) acc += (ACC)a[u] * xv[u];
  if (L > U) acc = sell16_tail<NT>(M.col16 + cb, M.val + vb, L, lane, r32, xval, acc);
  return acc;
}

// The FP64 kSell16 walk over this wave's slices.  epi(r, acc, pre(r), r < n) is
// called for every lane (rows past n only in the last slice, whose pre was
// given a clamped row).
template <bool NT, class ACC, class F, class P, class E>
__device__ inline void sell16_walk(const MatFmt<double> &M, F xval, P pre, E epi) {
  int64_t s, s1, ds;
  wave_slices(M.S, s, s1, ds);
  const int lane = threadIdx.x % kSlice;
  for (; s < s1; s += ds) {
    const int64_t r = s * kSlice + lane;
    // rows past n (last slice) have only padding: their column is clamped
    const int32_t r32 = (int32_t)(r < M.n ? r : M.n - 1);
    decltype(pre(r32)) pv;
    const ACC acc = sell16_slice_row<NT, ACC>(M, s, lane, r32, xval, pre, pv);
    epi(r, acc, pv, r < M.n);
  }
}

// One CSR row over the 16 lanes of a group, the sum in every lane.
template <bool NT, class V, class ACC, class F>
__device__ inline ACC csr_row_sum(const MatFmt<V> &M, int64_t r, bool in, int lane, F xval) {
  ACC acc = 0;
  if (in) {
    const int64_t k0 = M.ptr[r], k1 = M.ptr[r + 1];
    for (int64_t k = k0 + lane; k < k1; k += 4 * kLanesPerRow) {
      int32_t j[4];
      V a[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t kk = k + u * kLanesPerRow;
        j[u] = 0;
        a[u] = 0;
        if (kk < k1) { j[u] = mload<NT>(M.col + kk); a[u] = mload<NT>(M.val + kk); }
      }
      ACC xv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) xv[u] = xval(j[u]);
#pragma unroll
      for (int u = 0; u < 4; ++u) acc += (ACC)a[u] * xv[u];
    }
  }
#pragma unroll
  for (int off = kLanesPerRow / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, kWave);
  return acc;
}

// Calls epi(r, sum_k a_rk X(j_k)) once for every row r of this block's range;
// for kCsrV only the first lane of each 16-lane group calls it.
template <bool NT, int KIND, class V, class ACC, class F, class E>
__device__ inline void matvec_rows_as(const MatFmt<V> &M, F xval, E epi) {
  if constexpr (KIND == kSell16 && sizeof(V) == 8) {
    sell16_walk<NT, ACC>(M, xval, [](int32_t) { return 0; },
                     [&](int64_t r, ACC acc, int, bool row) { if (row) epi(r, acc); });
  } else if constexpr (KIND == kSell || KIND == kSell16) {
    int64_t s0, s1, ds;
    wave_slices(M.S, s0, s1, ds);
    const int lane = threadIdx.x % kSlice;
    for (int64_t s = s0; s < s1; s += ds) {
      const int64_t base = uniform(M.ptr[s]) + lane;
      const int L = __builtin_amdgcn_readfirstlane(M.len[s]);
      const int64_t r = s * kSlice + lane;
      // rows past n (last slice) have only padding: their column is clamped
      const int32_t r32 = (int32_t)(r < M.n ? r : M.n - 1);
      ACC acc;
      if constexpr (KIND == kSell16)
        acc = sell_row16<NT, kU, V, ACC>(M.col16 + uniform(M.ptr16[s]) + 4 * lane, M.val + base, L, r32,
                                     xval);
      else
        acc = sell_row<NT, kU, V, ACC, int32_t>(M.col + base, M.val + base, L, r32, xval);
      if (r < M.n) epi(r, acc);
    }
  } else if constexpr (KIND == kBsr3 || KIND == kBsr3W) {
    constexpr bool SHARE = KIND == kBsr3;
    // While there are fewer slices than waves or the matrix stays in the caches
    // (kBsr3), the block's four waves take each slice together, a quarter of its entries each (a wave per slice
    // left one serial chain of 14-32 rounds per SIMD at cube(20), 1077 slices: 50 us,
    // now 29 with the matrix kept in the caches, 41 without; cube(8) 18 -> 9.6 us);
    // their sums meet in LDS, added in entry order, and 192 threads finish the
    // slice's rows.  Else a wave per slice: no barrier, no wave without entries
    // (slices of 16 to 24 are two to three groups of 8).  Shared / a wave each, us
    // FP64 (at 2 / 3 blocks per CU): cube(28), 2894 slices, 102.8 / 105.2, cube(30),
    // 3547, 118.0 / 111.9, cube(34) 175.4 / 164.8; FP32 cube(28) 39.3 / 50.0 (in the
    // caches), cube(30) 54.2 / 52.0, cube(32) 68.5 / 64.0, cube(40) 136.1 / 125.6.
    // Groups of U block entries; the next group's block columns are loaded
    // with the current group's values, so the gathers of x need no second
    // round trip.  The slice's columns and values are read through buffer
    // resources bounded to the slice: past its width they read 0 without a
    // memory access, and those blocks' sums are dropped by a uniform select.
    constexpr int U = sizeof(V) == 8 ? FFHIP_BSR_U : FFHIP_BSR_U32;
    __shared__ ACC red[SHARE ? 2 : 1][SHARE ? kWavesPerBlock : 1][SHARE ? 3 * kSlice : 1];
    // slices split over the blocks or the waves by entries (rows of vertex and
    // of edge nodes differ in length by about 2.5x)
    const int wk = SHARE ? xcd_block_id() : xcd_block_id() * kWavesPerBlock + wave_id();
    const int64_t s0 = __builtin_amdgcn_readfirstlane(M.wstart[wk]);
    const int64_t s1 = __builtin_amdgcn_readfirstlane(M.wstart[wk + 1]);
    const int lane = threadIdx.x % kSlice, wv = wave_id();
    int buf = 0;
    for (int64_t s = s0; s < s1; ++s, buf ^= 1) {
      const int64_t sb = uniform(M.ptr[s]);
      const int L = __builtin_amdgcn_readfirstlane(M.len[s]);
      int k0 = 0, k1 = L;  // this wave's entries
      if constexpr (SHARE) {
        const int part = (L + kWavesPerBlock * U - 1) / (kWavesPerBlock * U) * U;
        k0 = wv * part < L ? wv * part : L;
        k1 = k0 + part < L ? k0 + part : L;
      }
      const auto rc = slice_rsrc(M.col + sb, (uint32_t)L * kSlice * 4);
      const auto rv = slice_rsrc(M.val + 9 * sb, (uint32_t)L * (9 * kSlice) * (uint32_t)sizeof(V));
      // shared: the row that this thread finishes is component t / 64 of the lane's node
      const int64_t i = s * kSlice + lane;
      const int32_t a = (wv < 3 || !SHARE) && i < M.nb ? M.perm[i] : -1;
      ACC s0v = 0, s1v = 0, s2v = 0;
      int32_t bn[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        bn[u] = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(rc, ((k0 + u) * kSlice + lane) * 4, 0, NT ? kBufNT : 0);
      for (int k = k0; k < k1; k += U) {
        int32_t b[U];
        ACC xv[U][3];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          b[u] = bn[u];
#pragma unroll
          for (int c = 0; c < 3; ++c) xv[u][c] = xval(3 * b[u] + c);
        }
        V wv9[U][9];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          constexpr int W = 16 / (int)sizeof(V), Z = (int)sizeof(V);
          const int eb = 9 * kSlice * (k + u);
#pragma unroll
          for (int g = 0; g < 8 / W; ++g) {
            const u32x4 r = __builtin_amdgcn_raw_buffer_load_b128(rv, (eb + bsr_pos<V>(g * W, lane)) * Z, 0, NT ? kBufNT : 0);
            if constexpr (sizeof(V) == 8) {
              wv9[u][2 * g] = __builtin_bit_cast(V, u32x2{r.x, r.y});
              wv9[u][2 * g + 1] = __builtin_bit_cast(V, u32x2{r.z, r.w});
            } else {
              // the whole vector is reinterpreted (a bit cast of one component
              // lvalue, r.y, reads the vector's first component)
              const f32x4 f = __builtin_bit_cast(f32x4, r);
              wv9[u][4 * g] = f.x;
              wv9[u][4 * g + 1] = f.y;
              wv9[u][4 * g + 2] = f.z;
              wv9[u][4 * g + 3] = f.w;
            }
          }
          const int o8 = (eb + bsr_pos<V>(8, lane)) * Z;
          if constexpr (sizeof(V) == 8)
            wv9[u][8] = __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(rv, o8, 0, NT ? kBufNT : 0));
          else
            wv9[u][8] = __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(rv, o8, 0, NT ? kBufNT : 0));
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
          bn[u] = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(rc, ((k + U + u) * kSlice + lane) * 4, 0, NT ? kBufNT : 0);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const ACC t0 = (ACC)wv9[u][0] * xv[u][0] + (ACC)wv9[u][1] * xv[u][1] + (ACC)wv9[u][2] * xv[u][2];
          const ACC t1 = (ACC)wv9[u][3] * xv[u][0] + (ACC)wv9[u][4] * xv[u][1] + (ACC)wv9[u][5] * xv[u][2];
          const ACC t2 = (ACC)wv9[u][6] * xv[u][0] + (ACC)wv9[u][7] * xv[u][1] + (ACC)wv9[u][8] * xv[u][2];
          const bool in = k + u < k1;
          s0v += in ? t0 : (ACC)0;
          s1v += in ? t1 : (ACC)0;
          s2v += in ? t2 : (ACC)0;
        }
        // keeps the next group's column loads in this iteration (the compiler
        // would otherwise load them again at the top of the next one and wait
        // for them there before the gathers)
#pragma unroll
        for (int u = 0; u < U; ++u) asm volatile("" : "+v"(bn[u]));
      }
      if constexpr (SHARE) {
        red[buf][wv][lane] = s0v;
        red[buf][wv][kSlice + lane] = s1v;
        red[buf][wv][2 * kSlice + lane] = s2v;
        // two buffers: the next slice's sums go to the other one, and the one
        // after that comes behind the next barrier
        __syncthreads();
        if (a >= 0) {
          ACC acc = red[buf][0][threadIdx.x];
#pragma unroll
          for (int w = 1; w < kWavesPerBlock; ++w) acc += red[buf][w][threadIdx.x];
          epi(3 * (int64_t)a + wv, acc);
        }
      } else if (a >= 0) {
        epi(3 * (int64_t)a, s0v);
        epi(3 * (int64_t)a + 1, s1v);
        epi(3 * (int64_t)a + 2, s2v);
      }
    }
  } else {
    const int64_t G = gridDim.x, lb = xcd_block_id();
    const int64_t r0 = (lb * M.n) / G, r1 = ((lb + 1) * M.n) / G;
    const int g = threadIdx.x / kLanesPerRow, lane = threadIdx.x % kLanesPerRow;
    constexpr int NG = kBlock / kLanesPerRow;
    for (int64_t rb = r0; rb < r1; rb += NG) {
      const int64_t r = rb + g;
      const ACC acc = csr_row_sum<NT, V, ACC>(M, r, r < r1, lane, xval);
      if (r < r1 && lane == 0) epi(r, acc);
    }
  }
}

template <int KIND, class V, class ACC, class F, class E>
__device__ inline void matvec_rows(const MatFmt<V> &M, F xval, E epi) {
  if constexpr (KIND == kBsr3W) {  // larger than the caches
    matvec_rows_as<true, KIND, V, ACC>(M, xval, epi);
  } else {
    if (M.nt) matvec_rows_as<true, KIND, V, ACC>(M, xval, epi);
    else matvec_rows_as<false, KIND, V, ACC>(M, xval, epi);
  }
}

// Calls epi(r, sum_k a_rk X(j_k), pre(r), row) for the rows r of this block's
// range, row = false for the padding lanes of the last kSell16 slice (their
// r is past n: epi stores nothing there, and pre was given a clamped row);
// pre(r) (operands of the epilogue) is loaded ahead where the layout allows.
// For kCsrV only the first lane of each 16-lane group calls epi.
template <int KIND, class V, class ACC, class F, class P, class E>
__device__ inline void matvec_rows_pre(const MatFmt<V> &M, F xval, P pre, E epi) {
  if constexpr (KIND == kSell16 && sizeof(V) == 8) {
    if (M.nt) sell16_walk<true, ACC>(M, xval, pre, epi);
    else sell16_walk<false, ACC>(M, xval, pre, epi);
  } else {
    matvec_rows<KIND, V, ACC>(M, xval, [&](int64_t r, ACC acc) { epi(r, acc, pre(r), true); });
  }
}

// ---------------------------------------------------------------- FP64 PCG
// G = A x - b, CG = D^-1 G, H0 = 0, partial (G, CG)
template <int KIND>
__global__ FFHIP_MATVEC_ATTR void k_pcg_init(MatFmt<double> M, const double *__restrict__ x,
                                             const double *__restrict__ b,
                                             const double *__restrict__ dinv, double *__restrict__ G,
                                             double *__restrict__ CG, double *__restrict__ H0,
                                             double *__restrict__ pout, CgState *st) {
  __shared__ double lds[kBlock / kWave];
  double part = 0.;
  matvec_rows<KIND, double, double>(
      M, [&](int32_t j) { return x[j]; },
      [&](int64_t r, double acc) {
        const double g = acc + -1. * b[r];
        const double c = dinv[r] * g;
        G[r] = g; CG[r] = c; H0[r] = 0.;
        part += g * c;
      });
  const double tot = block_sum<kBlock>(part, lds);
  if (threadIdx.x == 0) pout[xcd_block_id()] = tot;
  if (blockIdx.x == 0 && threadIdx.x == 0) { st->done = 0; st->stop = 0; st->iters = 0; st->rho = 0.; }
}

// Start of FP64 PCG iteration it = it0 + c: (g, Cg) from the last update's
// partials, the stop tests of ConjugueGradient (CG.cpp:226-252) and gamma.
// Returns false when the solve stops (the lead thread records why in stop;
// the next launch turns it into done).
__device__ inline bool pcg_begin(int c, const double *__restrict__ pin, CgState *st, double *lds,
                                 double &gamma) {
  const int it = st->it0 + c, itmax = st->itmax;
  const double eps = st->eps;
  const double gcg = reduce_partials(pin, gridDim.x, 1, 0, lds);
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  gamma = 0.;
  int done = 0;
  if (it == 1) {
    const double eps2 = eps > 0 ? eps * eps * gcg : eps * eps;
    if (gcg != gcg) done = 4;
    else if (gcg < 1e-30) done = 2;
    if (lead) {
      st->gcg0 = gcg; st->eps2 = eps2; st->gcg_prev[1] = gcg;
      if (done) { st->stop = done; st->iters = 0; }
    }
  } else {
    const double gcgp = st->gcg_prev[(it - 1) & 1];
    gamma = gcg / gcgp;
    if (gcg != gcg) done = 4;
    else if (gcg < st->eps2) done = 1;
    else if (it - 1 >= itmax) done = 3;
    if (lead) {
      st->gcg_prev[it & 1] = gcg;
      if (done) { st->stop = done; st->iters = it - 1; }
    }
  }
  return done == 0;
}

// this block's row range for the row-wise vector kernels
__device__ inline void block_rows(int64_t n, int64_t &r0, int64_t &r1) {
  const int64_t G = gridDim.x, lb = xcd_block_id();
  r0 = (lb * n) / G;
  r1 = ((lb + 1) * n) / G;
}

// the 4-aligned middle [a4, b4) of [r0, r1), for 16-byte FP32 accesses
// (vectors start 256-byte aligned); head [r0, a4) and tail [b4, r1) go scalar
__device__ inline void block_rows4(int64_t r0, int64_t r1, int64_t &a4, int64_t &b4) {
  a4 = (r0 + 3) & ~int64_t(3);
  if (a4 > r1) a4 = r1;
  b4 = r1 & ~int64_t(3);
  if (b4 < a4) b4 = a4;
}

// K1: the direction H = gamma H_prev - Cg, written by an elementwise pass so
// that the mat-vec gathers one vector (forming H on the fly from two gathered
// vectors per column made the cube(160) mat-vec 17 % slower and the
// [P2,P2,P2] block mat-vec 50 % slower; smaller systems: k_pcg_dir_matvec).
// It also applies the last update's step x += rho H_prev (ConjugueGradient's
// x += ro*h, CG.cpp:241), moved here from the update kernel: this pass reads
// H_prev anyway, so the step costs 16 instead of 24 bytes per row.  x enters
// nothing else of the iteration; the stopping launch still applies it.
__global__ __launch_bounds__(kBlock) void k_pcg_dirvec(int c, int64_t n,
                                                       const double *__restrict__ Hold,
                                                       const double *__restrict__ dinv,
                                                       const double *__restrict__ G,
                                                       double *__restrict__ Hnew,
                                                       double *__restrict__ x,
                                                       const double *__restrict__ pin,
                                                       double *__restrict__ pout, CgState *st) {
  __shared__ double lds[kBlock / kWave];
  if (st->done) return;  // set by an earlier launch only: every block of this one agrees
  double gamma;
  const bool go = pcg_begin(c, pin, st, lds, gamma);
  const bool step = st->it0 + c > 1;  // an update ran before this direction
  const double rho = st->rho;
  int64_t r0, r1;
  block_rows(n, r0, r1);
  if (go) {
    // the new direction and its partial (g, h), the numerator of rho; C g is
    // formed here from D^-1 and g (the update keeps no copy of it), the
    // product rounded on its own as the stored copy was
    double part = 0.;
    for (int64_t r = r0 + threadIdx.x; r < r1; r += kBlock) {
      const double h = Hold[r];
      if (step) x[r] += rho * h;
      const double g = G[r];
      const double hn = gamma * h - __dmul_rn(dinv[r], g);
      Hnew[r] = hn;
      part += g * hn;
    }
    const double gh = block_sum<kBlock>(part, lds);
    if (threadIdx.x == 0) pout[2 * xcd_block_id() + 1] = gh;
  } else if (step) {
    for (int64_t r = r0 + threadIdx.x; r < r1; r += kBlock) x[r] += rho * Hold[r];
  }
}

// K2: AH = A H, partials (H, AH), (g, H)
template <int KIND>
__global__ FFHIP_MATVEC_ATTR void k_pcg_matvec(MatFmt<double> M, const double *__restrict__ H,
                                               double *__restrict__ AH, double *__restrict__ pout,
                                               CgState *st) {
  __shared__ double lds[kBlock / kWave];
  if (st->stop) {  // the direction kernel stopped the solve: publish it
    if (blockIdx.x == 0 && threadIdx.x == 0) st->done = st->stop;
    return;
  }
  if (st->done) return;
  double p_hah = 0.;
  auto epi = [&](int64_t r, double acc, double h, bool row) {
    if (row) AH[r] = acc;
    p_hah += (row ? h : 0.) * acc;
  };
  if constexpr (KIND == kSell16) {
    // gathers through a buffer resource over H (n < 2^28 in this layout)
    const auto hr = slice_rsrc(H, (uint32_t)(M.n * 8));
    matvec_rows_pre<KIND, double, double>(
        M, [&](int32_t j) { return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(hr, j * 8, 0, 0)); },
        [&](int64_t r) { return H[r]; }, epi);
  } else {
    matvec_rows_pre<KIND, double, double>(M, [&](int32_t j) { return H[j]; }, [&](int64_t r) { return H[r]; },
                                          epi);
  }
  const double a = block_sum<kBlock>(p_hah, lds);
  if (threadIdx.x == 0) pout[2 * xcd_block_id()] = a;  // (g, h) comes from the direction kernel
}

// K1 and K2 in one launch: the direction formed for every gathered column from
// two vectors, H_prev and C g (which the update then keeps).  For systems in
// the caches, whose iterations are bound by the latency of their launches
// (cube(24): 3 of about 5 us with the gaps); the rule is at ffhip_cg_s::fuse.
template <int KIND>
__global__ FFHIP_MATVEC_ATTR void k_pcg_dir_matvec(int c, MatFmt<double> M, const double *__restrict__ Hold,
                                                   const double *__restrict__ CG,
                                                   const double *__restrict__ G, double *__restrict__ Hnew,
                                                   double *__restrict__ AH, double *__restrict__ x,
                                                   const double *__restrict__ pin,
                                                   double *__restrict__ pout, CgState *st) {
  __shared__ double lds[kBlock / kWave];
  if (st->done) return;  // set by an earlier launch only: every block of this one agrees
  double gamma;
  const bool go = pcg_begin(c, pin, st, lds, gamma);
  const bool step = st->it0 + c > 1;  // an update ran before this direction
  const double rho = st->rho;
  if (!go) {  // the update publishes the stop
    int64_t r0, r1;
    block_rows(M.n, r0, r1);
    if (step)
      for (int64_t r = r0 + threadIdx.x; r < r1; r += kBlock) x[r] += rho * Hold[r];
    return;
  }
  double p_hah = 0., p_gh = 0.;
  struct Own {
    double h, cg, g, x;
  };
  const auto pre = [&](int64_t r) { return Own{Hold[r], CG[r], G[r], x[r]}; };
  const auto epi = [&](int64_t r, double acc, const Own &o, bool row) {
    if (!row) return;
    const double hn = gamma * o.h - o.cg;
    Hnew[r] = hn;
    AH[r] = acc;
    if (step) x[r] = o.x + rho * o.h;
    p_gh += o.g * hn;
    p_hah += hn * acc;
  };
  if constexpr (KIND == kSell16) {
    const auto hr = slice_rsrc(Hold, (uint32_t)(M.n * 8)), cr = slice_rsrc(CG, (uint32_t)(M.n * 8));
    matvec_rows_pre<KIND, double, double>(
        M,
        [&](int32_t j) {
          const double h = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(hr, j * 8, 0, 0));
          return gamma * h - __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(cr, j * 8, 0, 0));
        },
        pre, epi);
  } else {
    matvec_rows_pre<KIND, double, double>(M, [&](int32_t j) { return gamma * Hold[j] - CG[j]; }, pre, epi);
  }
  const double a = block_sum<kBlock>(p_hah, lds);
  const double b = block_sum<kBlock>(p_gh, lds);
  if (threadIdx.x == 0) {
    pout[2 * xcd_block_id()] = a;
    pout[2 * xcd_block_id() + 1] = b;
  }
}

// ---------------------------------------------------------------- symmetric values
// K2 over half of the values.  The mat-vec is bound by the bytes of the matrix,
// 10 per entry.  Where A is symmetric (bit for bit) and its rows follow few
// patterns (the rows of a box: the same column distances inside, others at its
// faces), a row needs its entries from the diagonal on from memory and no
// index: the entries before it are those of the rows above, read a short while
// ago, and a byte names the row's pattern.  65 bytes a row for 147 (P1 on a
// cube).  The same entries in the same order: the bits of k_pcg_matvec.
//
// us per mat-vec, half against whole: cube(64) 8.9 / 10.9, cube(96) 18.8 / 24.6,
// cube(112) 26.2 / 39.0, cube(128) 38.1 / 70.9, cube(160) 96 / 137 (366 MB from
// HBM; the vector kernels lose 18 us there, their vectors in the Infinity Cache
// no more).  Not faster at cube(160): non-temporal loads of the values (111), of
// some of the planes (98 to 103), the next slice's values loaded ahead (102), 3
// blocks per CU (102), slices in columns that keep a plane's values in the L2
// (98: a fifth fewer misses).
//
// Up to 8 entries before the diagonal and NU from it on, NU 4 or 8:
// [slice][entry from the diagonal on][64 rows].
constexpr int kSymHalf = 8, kSymSlots = 256, kSymMax = 192;  // patterns: slots of the table, most taken
constexpr uint16_t kSymNone = 0xffffu;
struct SymPattern {
  uint16_t off[kSymHalf];   // entry i before the diagonal: its owner's entry, in bytes; kSymNone: none
  int16_t d[2 * kSymHalf];  // column distances before the diagonal, from it on (0: none)
};
struct SymFmt {
  int64_t n, S;
  const double *val;
  const uint8_t *cls;
  const SymPattern *table;
};

template <int NL, int NU>
__global__ FFHIP_MATVEC_ATTR void k_pcg_matvec_sym(SymFmt M, const double *__restrict__ H,
                                                   double *__restrict__ AH, double *__restrict__ pout,
                                                   CgState *st) {
  __shared__ double lds[kBlock / kWave];
  __shared__ __align__(16) SymPattern tab[kSymSlots];
  if (st->stop) {  // the direction kernel stopped the solve: publish it
    if (blockIdx.x == 0 && threadIdx.x == 0) st->done = st->stop;
    return;
  }
  if (st->done) return;
  for (int i = threadIdx.x; i < (int)(sizeof(tab) / 16); i += kBlock)
    reinterpret_cast<u32x4 *>(tab)[i] = reinterpret_cast<const u32x4 *>(M.table)[i];
  __syncthreads();
  const auto hr = slice_rsrc(H, (uint32_t)(M.n * 8));
  const auto vr = slice_rsrc(M.val, (uint32_t)(M.S * (NU * kSlice * 8)));
  // a load past the values' end gives 0
  const auto val = [&](uint32_t o, uint32_t plane) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(vr, o, plane, 0));
  };
  // byte offset of row r's diagonal
  const auto at = [](uint32_t r) { return r * 8u + (r / kSlice) * ((NU - 1) * kSlice * 8u); };
  double p_hah = 0.;
  int64_t s, s1, ds;
  wave_slices(M.S, s, s1, ds);
  const int lane = threadIdx.x % kSlice;
  for (; s < s1; s += ds) {
    const int64_t r = s * kSlice + lane;
    const uint32_t rc = (uint32_t)(r < M.n ? r : M.n - 1);  // past n: the last row's sum, not stored
    const int c = M.cls[rc];
    const uint32_t own = at(rc);
    double u[NU];
#pragma unroll
    for (int k = 0; k < NU; ++k) u[k] = val(own, k * (kSlice * 8));
    const u32x4 *t = reinterpret_cast<const u32x4 *>(&tab[c]);
    const u32x4 w = t[0], e0 = t[1], e1 = t[2];
    const uint32_t oo[4] = {w.x, w.y, w.z, w.w};
    const uint32_t dd[8] = {e0.x, e0.y, e0.z, e0.w, e1.x, e1.y, e1.z, e1.w};
    const auto off = [&](int k) { return k & 1 ? oo[k >> 1] >> 16 : oo[k >> 1] & 0xffffu; };
    const auto col = [&](int k) {
      return rc + (uint32_t)(k & 1 ? (int32_t)dd[k >> 1] >> 16 : (int32_t)(int16_t)dd[k >> 1]);
    };
    const auto xof = [&](int k) {
      return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(hr, col(k) * 8u, 0, 0));
    };
    double a[NL], xl[NL], xu[NU];
#pragma unroll
    for (int k = 0; k < NL; ++k) a[k] = val(off(k) == kSymNone ? 0xffffffffu : off(k) + at(col(k)), 0);
#pragma unroll
    for (int k = 0; k < NL; ++k) xl[k] = xof(k);
#pragma unroll
    for (int k = 0; k < NU; ++k) xu[k] = xof(kSymHalf + k);
    const double h = H[rc];
    double acc = 0.;
#pragma unroll
    for (int k = 0; k < NL; ++k) acc += a[k] * xl[k];
#pragma unroll
    for (int k = 0; k < NU; ++k) acc += u[k] * xu[k];
    if (r < M.n) AH[r] = acc;
    p_hah += (r < M.n ? h : 0.) * acc;
  }
  const double tot = block_sum<kBlock>(p_hah, lds);
  if (threadIdx.x == 0) pout[2 * xcd_block_id()] = tot;
}

// A row of the kSell16 layout as the pattern search sees it: its distances as
// stored (4 packed groups: rows of up to 16 entries), the counts before the
// diagonal and from it on.
struct SymRow {
  u32x2 pk[4];
  int nl, nu, L;
  __device__ int32_t delta(int k) const {
    const uint32_t w = k & 2 ? pk[k >> 2].y : pk[k >> 2].x;
    return k & 1 ? (int32_t)w >> 16 : (int32_t)(int16_t)w;
  }
};
__device__ inline SymRow sym_row(const MatFmt<double> &M, int64_t r) {
  SymRow R;
  const int64_t s = r / kSlice;
  const int lane = (int)(r % kSlice);
  R.L = M.len[s];
  const int64_t cb = M.ptr16[s];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    R.pk[g] = u32x2{0u, 0u};
    if (4 * g < R.L) R.pk[g] = *reinterpret_cast<const u32x2 *>(M.col16 + cb + ((int64_t)g * kSlice + lane) * 4);
  }
  R.nl = R.nu = 0;
  bool past = false;  // the diagonal or a column after it was seen: distance 0 is padding
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int32_t d = R.delta(k);
    R.nl += d < 0;
    R.nu += d > 0 || (d == 0 && !past && k < R.L);
    past |= d >= 0;
  }
  return R;
}
// the positions, from the diagonal on, that row r's entries before the diagonal
// have in the rows of their columns (4 bits each); bad: not all there (kSymForm),
// or not with the same value (kSymValues)
constexpr int kSymForm = 1, kSymValues = 2;
__device__ inline uint32_t sym_owners(const MatFmt<double> &M, int64_t r, const SymRow &R, int &bad) {
  const int64_t vb = M.ptr[r / kSlice];
  uint32_t pw = 0;
#pragma unroll 1
  for (int k = 0; k < R.nl; ++k) {
    const u32x2 g = k < 4 ? R.pk[0] : R.pk[1];  // nl <= 8
    const uint32_t w = k & 2 ? g.y : g.x;
    const int32_t d = k & 1 ? (int32_t)w >> 16 : (int32_t)(int16_t)w;
    const int64_t j = r + d;
    const SymRow J = sym_row(M, j);
    int kj = -1;
#pragma unroll
    for (int q = 0; q < 16; ++q) kj = J.delta(q) == -d ? q : kj;
    if (kj < 0 || J.L > 16 || kj - J.nl >= kSymHalf) { bad = kSymForm; return 0; }
    const double mine = M.val[vb + pair_pos(R.L, k, (int)(r % kSlice))];
    const double theirs = M.val[M.ptr[j / kSlice] + pair_pos(J.L, kj, (int)(j % kSlice))];
    if (__builtin_bit_cast(uint64_t, mine) != __builtin_bit_cast(uint64_t, theirs)) bad = kSymValues;
    pw |= (uint32_t)(kj - J.nl) << (4 * k);
  }
  return pw;
}
struct SymTables {
  unsigned long long key[kSymSlots];  // hash of the pattern, 0: free
  int64_t rep[kSymSlots];             // a row of the pattern
  SymRow row[kSymSlots];
  uint32_t owners[kSymSlots];
  int bad, count, nl, nu;  // some row does not fit (kSymForm, kSymValues); patterns; most entries before a diagonal, from it on
};
// every row's slot in the table of patterns.  Once a row fails (or the table
// fills, as on an unstructured mesh within its first blocks) the rest is left.
__global__ __launch_bounds__(256) void k_sym_rows(MatFmt<double> M, SymTables *T, uint8_t *__restrict__ cls,
                                                  uint32_t *__restrict__ owners) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= M.n || __hip_atomic_load(&T->bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const SymRow R = sym_row(M, r);
  int bad = R.L <= 16 && R.nl <= kSymHalf && R.nu <= kSymHalf ? 0 : kSymForm;
  const uint32_t pw = bad ? 0 : sym_owners(M, r, R, bad);
  if (!bad) {
    unsigned long long h = 0x9e3779b97f4a7c15ull ^ ((unsigned long long)pw << 16 | R.nl << 8 | R.nu);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      h = (h ^ ((unsigned long long)R.pk[g].y << 32 | R.pk[g].x)) * 0xbf58476d1ce4e5b9ull;
      h ^= h >> 29;
    }
    h |= 1;
    bad = kSymForm;  // until a slot is found
    for (int p = 0; p < 16 && bad; ++p) {
      const int t = (int)(((h >> 8) + p) & (kSymSlots - 1));
      unsigned long long k = __hip_atomic_load(&T->key[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (k == 0) {
        k = atomicCAS(&T->key[t], 0ull, h);
        if (k == 0) {
          T->rep[t] = r;
          if (atomicAdd(&T->count, 1) >= kSymMax) break;
          k = h;
        }
      }
      if (k == h) {
        cls[r] = (uint8_t)t;
        owners[r] = pw;
        bad = 0;
      }
    }
  }
  if (bad) atomicOr(&T->bad, bad);
}
// the patterns from their rows
__global__ __launch_bounds__(kSymSlots) void k_sym_table(MatFmt<double> M, SymTables *T,
                                                         const uint32_t *__restrict__ owners,
                                                         SymPattern *__restrict__ table) {
  const int t = threadIdx.x;
  SymPattern P;
  for (int k = 0; k < kSymHalf; ++k) {
    P.off[k] = kSymNone;
    P.d[k] = P.d[kSymHalf + k] = 0;
  }
  if (T->key[t] && !T->bad) {
    const int64_t r = T->rep[t];
    const SymRow R = sym_row(M, r);
    const uint32_t pw = owners[r];
    T->row[t] = R;
    T->owners[t] = pw;
    atomicMax(&T->nl, R.nl);
    atomicMax(&T->nu, R.nu);
    for (int k = 0; k < 16; ++k) {
      const int32_t d = R.delta(k);
      if (k < R.nl) {
        P.d[k] = (int16_t)d;
        P.off[k] = (uint16_t)((pw >> (4 * k) & 15u) * (kSlice * 8u));
      } else if (k - R.nl < R.nu) {
        P.d[kSymHalf + k - R.nl] = (int16_t)d;
      }
    }
  }
  table[t] = P;
}
// the values from the diagonal on; every row compared with its pattern's
__global__ __launch_bounds__(256) void k_sym_fill(MatFmt<double> M, SymTables *T, const uint8_t *__restrict__ cls,
                                                  const uint32_t *__restrict__ owners, int NU,
                                                  double *__restrict__ val) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= M.n || __hip_atomic_load(&T->bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const SymRow R = sym_row(M, r);
  const int t = cls[r];
  const SymRow &Q = T->row[t];
  bool same = owners[r] == T->owners[t] && R.nl == Q.nl && R.nu == Q.nu;
#pragma unroll
  for (int g = 0; g < 4; ++g) same &= R.pk[g].x == Q.pk[g].x && R.pk[g].y == Q.pk[g].y;
  if (!same) {  // a hash met twice
    atomicOr(&T->bad, kSymForm);
    return;
  }
  const int64_t vb = M.ptr[r / kSlice];
  for (int p = 0; p < NU; ++p)
    val[(r / kSlice * NU + p) * kSlice + r % kSlice] =
        p < R.nu ? M.val[vb + pair_pos(R.L, R.nl + p, (int)(r % kSlice))] : 0.;
}

__global__ __launch_bounds__(kBlock) void k_pcg_update(
    int64_t n, const double *__restrict__ AH, const double *__restrict__ dinv,
    double *__restrict__ G, double *__restrict__ CG, const double *__restrict__ pin,
    double *__restrict__ pout, CgState *st) {
  __shared__ double lds[kBlock / kWave];
  if (st->stop) {  // k_pcg_dir_matvec stopped the solve: publish it
    if (blockIdx.x == 0 && threadIdx.x == 0) st->done = st->stop;
    return;
  }
  if (st->done) return;
  const int P = gridDim.x;
  const double hah = reduce_partials(pin, P, 2, 0, lds);
  const double gh = reduce_partials(pin, P, 2, 1, lds);
  const double rho = -gh / hah;
  if (blockIdx.x == 0 && threadIdx.x == 0) st->rho = rho;  // x += rho H: next direction kernel
  int64_t r0, r1;
  block_rows(n, r0, r1);
  double part = 0.;
  for (int64_t r = r0 + threadIdx.x; r < r1; r += kBlock) {
    const double g = G[r] + rho * AH[r];
    G[r] = g;
    const double c = __dmul_rn(dinv[r], g);  // C g, formed again by the next direction kernel
    if (CG) CG[r] = c;                        // but kept for k_pcg_dir_matvec
    part += g * c;
  }
  const double tot = block_sum<kBlock>(part, lds);
  if (threadIdx.x == 0) pout[xcd_block_id()] = tot;
}

// ---------------------------------------------------------------- residual check
// r = b - A x (FP64); partials (r,r), (b,b), (r, D^-1 r)
template <int KIND>
__global__ FFHIP_MATVEC_ATTR void k_residual(MatFmt<double> M, const double *__restrict__ x,
                                             const double *__restrict__ b,
                                             const double *__restrict__ dinv,
                                             double *__restrict__ rout, double *__restrict__ pout) {
  __shared__ double lds[kBlock / kWave];
  double prr = 0., pbb = 0., prc = 0.;
  matvec_rows<KIND, double, double>(
      M, [&](int32_t j) { return x[j]; },
      [&](int64_t r, double acc) {
        const double rr = b[r] - acc;
        if (rout) rout[r] = rr;
        prr += rr * rr;
        pbb += b[r] * b[r];
        prc += rr * (dinv[r] * rr);
      });
  const double a = block_sum<kBlock>(prr, lds);
  const double c = block_sum<kBlock>(pbb, lds);
  const double e = block_sum<kBlock>(prc, lds);
  if (threadIdx.x == 0) {
    const int lb = xcd_block_id();
    pout[3 * lb] = a; pout[3 * lb + 1] = c; pout[3 * lb + 2] = e;
  }
}

// ---------------------------------------------------------------- small systems
// A whole FP64 solve of a small system in one workgroup: the start
// (SetInitWithBC, G = A x - b), the iterations of the three kernels above and
// the residual sums.  Up to some thousand rows an iteration is nothing but the
// latency of three launches (12 us with the gaps between them) and a solve
// waits for the set-up of a captured chunk; here it is three barriers, with h,
// A h and x in LDS and g and D^-1 in registers, bound by the latency of a row
// (slice offsets, entries from L2, gathers from LDS).  us per iteration, this
// against launches (set-up included): 216 rows 2.3 / 17.7, 1000 rows 4.0 / 15.1,
// 1728 rows 6.9 / 13.2, 4096 rows 10.9 / 12.4 (P1 cubes); CSR 216 rows 5.6 / 19.4.
//
// The sums are those of the launches, bit for bit: virtual block vb of the G
// that the launches would use is played by four waves (up to four blocks at a
// time, the others in turn), rows and slices go to the same threads, and
// partials are added in the same order.
constexpr int kSmallBlocks = 16;                         // virtual blocks
constexpr int kSmallRows = kSmallBlocks * kBlock;        // kSell16: 256 rows each
constexpr int kSmallRowsCsr = kSmallBlocks * kBlock / kLanesPerRow;  // kCsrV: 16 rows
struct SmallOut {
  CgState st;
  double res[3 * kSmallBlocks];  // k_residual's partials
};
template <int KIND, int Q>  // Q: rows of a thread in the vector passes
__global__ __launch_bounds__(1024) void k_pcg_small(MatFmt<double> M, int G, const double *b, double *x,
                                                    const double *__restrict__ dinv,
                                                    const uint8_t *__restrict__ wcl, double tgv,
                                                    double eps, int itmax, SmallOut *__restrict__ out) {
  constexpr bool SELL = KIND == kSell16;
  constexpr int T = SELL ? Q : 4;  // virtual blocks that a wave plays in a mat-vec
  __shared__ double H[Q * 1024], A[Q * 1024], X[Q * 1024];
  __shared__ double ws[3][kSmallBlocks * kWavesPerBlock];  // wave sums
  const int n = (int)M.n, S = (int)M.S, t = threadIdx.x % kBlock, lane = threadIdx.x % kWave;
  const int W = wave_id(), w = W % kWavesPerBlock, nv = blockDim.x / kBlock;
  int row[Q];  // this thread's rows in the vector passes; -1: none
  double g[Q], di[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    // block_rows; a kCsrV block's up to 16 rows take 16 lanes here
    const int vb = SELL ? q * nv + W / kWavesPerBlock : threadIdx.x / kLanesPerRow;
    const int r = vb * n / G + (SELL ? t : threadIdx.x % kLanesPerRow);
    row[q] = vb < G && r < (vb + 1) * n / G ? r : -1;
    di[q] = 0.; g[q] = 0.;
    if (row[q] >= 0) {
      di[q] = dinv[row[q]];
      const double x0 = wcl && wcl[row[q]] ? b[row[q]] / tgv : x[row[q]];
      X[row[q]] = x0;
      H[row[q]] = x0;
    }
  }
  // the rows of A H of this wave in turn q: epi(r, acc, row) as in matvec_rows_pre
  auto matvec = [&](int q, auto epi) {
    const auto xval = [&](int32_t j) { return H[j]; };
    const int vb = q * nv + W / kWavesPerBlock;
    if (vb >= G) return;
    if constexpr (SELL) {  // wave_slices: at most one slice
      const int groups = G % 8 ? 1 : 8, nloc = G / groups, grp = vb / nloc, loc = vb - grp * nloc;
      const int s = grp * S / groups + loc * kWavesPerBlock + w;
      if (s >= (grp + 1) * S / groups) return;
      const int r = s * kSlice + lane, rc = r < n ? r : n - 1;
      int pv;
      const double acc =
          sell16_slice_row<false, double>(M, s, lane, rc, xval, [](int32_t) { return 0; }, pv);
      epi(r, acc, r < n);
    } else {
      const int r = vb * n / G + t / kLanesPerRow;
      const bool in = r < (vb + 1) * n / G;
      const double acc = csr_row_sum<false, double, double>(M, r, in, t % kLanesPerRow, xval);
      if (in && t % kLanesPerRow == 0) epi(r, acc, true);
    }
  };
  // wave sums of one value per thread: of a mat-vec's turn q, of a vector pass
  auto put = [&](int k, int q, double v) {
    v = wave_sum(v);
    const int vb = q * nv + W / kWavesPerBlock;
    if (lane == 0 && vb < G) ws[k][vb * kWavesPerBlock + w] = v;
  };
  auto put_rows = [&](int k, int q, double v) {
    if constexpr (SELL) put(k, q, v);
    else {  // the first wave of the block, its other lanes and the other waves without rows
      v = row16_sum(v);
      const int vb = threadIdx.x / kLanesPerRow, l = threadIdx.x % kLanesPerRow;
      if (vb < G && l < kWavesPerBlock) ws[k][vb * kWavesPerBlock + l] = l == 0 ? v : 0.;
    }
  };
  auto partial = [&](int k) {  // block_sum of virtual block `lane`
    double p = 0.;
    if (lane < G) {
#pragma unroll
      for (int i = 0; i < kWavesPerBlock; ++i) p += ws[k][lane * kWavesPerBlock + i];
    }
    return p;
  };
  auto total = [&](int k) { return 0. + wave_sum(partial(k)); };  // reduce_partials
  __syncthreads();
#pragma unroll 1
  for (int q = 0; q < T; ++q) {  // k_pcg_init
    double part = 0.;
    matvec(q, [&](int r, double acc, bool in) {
      if (!in) return;
      const double gv = acc + -1. * b[r];
      const double c = dinv[r] * gv;
      A[r] = gv;
      part += gv * c;
    });
    put(0, q, part);
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (row[q] >= 0) g[q] = A[row[q]];
  double gcg0 = 0., eps2 = 0., gcgp = 0., gcg, rho = 0.;
  int it = 1, done = 0;
  for (;; ++it) {
    // pcg_begin
    gcg = total(0);
    double gamma = 0.;
    if (it == 1) {
      gcg0 = gcg;
      eps2 = eps > 0 ? eps * eps * gcg : eps * eps;
      if (gcg != gcg) done = 4;
      else if (gcg < 1e-30) done = 2;
    } else {
      gamma = gcg / gcgp;
      if (gcg != gcg) done = 4;
      else if (gcg < eps2) done = 1;
      else if (it - 1 >= itmax) done = 3;
    }
    gcgp = gcg;
    if (done) break;  // the same in every thread
    // k_pcg_dirvec
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      double part = 0.;
      if (row[q] >= 0) {
        const double h = it > 1 ? H[row[q]] : 0.;
        if (it > 1) X[row[q]] += rho * h;
        const double hn = gamma * h - __dmul_rn(di[q], g[q]);
        H[row[q]] = hn;
        part += g[q] * hn;
      }
      put_rows(1, q, part);
    }
    __syncthreads();
    // k_pcg_matvec
#pragma unroll 1
    for (int q = 0; q < T; ++q) {
      double part = 0.;
      matvec(q, [&](int r, double acc, bool in) {
        if (in) A[r] = acc;
        part += (in ? H[r] : 0.) * acc;
      });
      put(2, q, part);
    }
    __syncthreads();
    // k_pcg_update
    const double hah = total(2), gh = total(1);
    rho = -gh / hah;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      double part = 0.;
      if (row[q] >= 0) {
        const double gn = g[q] + rho * A[row[q]];
        g[q] = gn;
        const double c = __dmul_rn(di[q], gn);
        part += gn * c;
      }
      put_rows(0, q, part);
    }
    __syncthreads();
  }
  // the stopping launch's step, then the residual of the solution
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (row[q] >= 0) {
      if (it > 1) X[row[q]] += rho * H[row[q]];
      H[row[q]] = X[row[q]];
    }
  __syncthreads();
#pragma unroll 1
  for (int q = 0; q < T; ++q) {  // k_residual
    double rr = 0., bb = 0., rc = 0.;
    matvec(q, [&](int r, double acc, bool in) {
      if (!in) return;
      const double v = b[r] - acc;
      rr += v * v;
      bb += b[r] * b[r];
      rc += v * (dinv[r] * v);
    });
    put(0, q, rr);
    put(1, q, bb);
    put(2, q, rc);
  }
  __syncthreads();  // b has been read: x may be the same array
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (row[q] >= 0) x[row[q]] = X[row[q]];
  if (W == 0) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double p = partial(c);
      if (lane < G) out->res[3 * lane + c] = p;
    }
    if (lane == 0) {
      out->st.gcg0 = gcg0;
      out->st.eps2 = eps2;
      out->st.gcg_prev[it & 1] = gcg;
      out->st.done = done;
      out->st.iters = it - 1;
    }
  }
}

// ---------------------------------------------------------------- affine CG
// LinearCG / AffineCG with the matrix product as the operator:
// ConjuguedGradient2 (src/femlib/MatriceCreuse.hpp:180-240).  Iteration it:
//   k_cg2_step:   (Cg, g) of the last update, stop test, gamma = g2/g2p;
//                 h = gamma h - Cg (it > 0); x += rop h
//   k_cg2_dir:    Ah = A x - b - g; partials (h, Ah), (g, h)
//   k_cg2_update: ro = -(g, h) rop / (h, Ah); x += (ro - rop) h;
//                 g += (ro / rop) Ah; Cg = C g; partial (Cg, g)
// C is the identity (dinv null) or the Jacobi diagonal inverse.  Scalars
// written by a kernel's lead thread are kept by parity of the iteration, so
// no block reads a slot another block of the same kernel writes.
struct Cg2State {
  double g2[2];    // (Cg, g) reduced by the step kernel of iteration it, slot it & 1
  double ro[2];    // ro of iteration it, slot it & 1
  double g20, reps2, g2last;
  int done;        // 0 run, 1 converged, 2 g2_0 < 1e-30, 3 itmax, 5 (h,Ah)^2 < 1e-60, 6 ro NaN
  int iters;
};

// g = A x - b, Cg = C g, h = -Cg; partial (Cg, g)
template <int KIND>
__global__ FFHIP_MATVEC_ATTR void k_cg2_init(MatFmt<double> M, const double *__restrict__ x,
                                             const double *__restrict__ b,
                                             const double *__restrict__ dinv, double *__restrict__ g,
                                             double *__restrict__ Cg, double *__restrict__ h,
                                             double *__restrict__ pout, Cg2State *st) {
  __shared__ double lds[kBlock / kWave];
  double part = 0.;
  matvec_rows<KIND, double, double>(
      M, [&](int32_t j) { return x[j]; },
      [&](int64_t r, double acc) {
        const double gv = b ? acc - b[r] : acc;
        const double c = dinv ? dinv[r] * gv : gv;
        g[r] = gv; Cg[r] = c; h[r] = -c;
        part += c * gv;
      });
  const double tot = block_sum<kBlock>(part, lds);
  if (threadIdx.x == 0) pout[xcd_block_id()] = tot;
  if (blockIdx.x == 0 && threadIdx.x == 0) { st->done = 0; st->iters = 0; }
}

__global__ __launch_bounds__(kBlock) void k_cg2_step(int it, int itmax, double eps, int64_t n,
                                                     double *__restrict__ h,
                                                     const double *__restrict__ Cg,
                                                     double *__restrict__ x,
                                                     const double *__restrict__ pin, Cg2State *st) {
  __shared__ double lds[kBlock / kWave];
  if (st->done) return;
  const double g2 = reduce_partials(pin, gridDim.x, 1, 0, lds);
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  double gamma = 0., rop = 1.;
  if (it == 0) {
    int done = 0;
    if (g2 != g2) done = 6;  // the reference's first ro would be NaN
    else if (g2 < 1e-30) done = 2;
    if (lead) {
      st->g20 = g2; st->g2last = g2; st->g2[0] = g2;
      st->reps2 = eps > 0 ? eps * eps * g2 : -eps;
      if (done) { st->done = done; st->iters = 0; }
    }
    if (done) return;
  } else {
    int done = 0;
    if (g2 < st->reps2) done = 1;
    else if (it - 1 >= itmax) done = 3;
    if (lead) {
      st->g2[it & 1] = g2; st->g2last = g2;
      if (done) { st->done = done; st->iters = it; }
    }
    if (done) return;
    gamma = g2 / st->g2[(it - 1) & 1];
    rop = st->ro[(it - 1) & 1];
  }
  int64_t r0, r1;
  block_rows(n, r0, r1);
  for (int64_t r = r0 + threadIdx.x; r < r1; r += kBlock) {
    double hv = h[r];
    if (it > 0) { hv = hv * gamma - Cg[r]; h[r] = hv; }
    x[r] += rop * hv;
  }
}

template <int KIND>
__global__ FFHIP_MATVEC_ATTR void k_cg2_dir(MatFmt<double> M, const double *__restrict__ x,
                                            const double *__restrict__ b,
                                            const double *__restrict__ g,
                                            const double *__restrict__ h, double *__restrict__ Ah,
                                            double *__restrict__ pout, const Cg2State *st) {
  __shared__ double lds[kBlock / kWave];
  if (st->done) return;
  double p_hah = 0., p_gh = 0.;
  matvec_rows<KIND, double, double>(
      M, [&](int32_t j) { return x[j]; },
      [&](int64_t r, double acc) {
        const double a = (b ? acc - b[r] : acc) - g[r];
        Ah[r] = a;
        p_hah += h[r] * a;
        p_gh += g[r] * h[r];
      });
  const double a = block_sum<kBlock>(p_hah, lds);
  const double c = block_sum<kBlock>(p_gh, lds);
  if (threadIdx.x == 0) {
    const int lb = xcd_block_id();
    pout[2 * lb] = a;
    pout[2 * lb + 1] = c;
  }
}

__global__ __launch_bounds__(kBlock) void k_cg2_update(
    int it, int64_t n, const double *__restrict__ h, const double *__restrict__ Ah,
    const double *__restrict__ dinv, double *__restrict__ x, double *__restrict__ g,
    double *__restrict__ Cg, const double *__restrict__ pin, double *__restrict__ pout,
    Cg2State *st) {
  __shared__ double lds[kBlock / kWave];
  if (st->done) return;
  const int P = gridDim.x;
  const double hah = reduce_partials(pin, P, 2, 0, lds);
  const double gh = reduce_partials(pin, P, 2, 1, lds);
  const double rop = it == 0 ? 1. : st->ro[(it - 1) & 1];
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  if (hah * hah < 1e-60) {
    if (lead) { st->done = 5; st->iters = it; }
    return;
  }
  const double ro = -gh * rop / hah;
  if (ro != ro) {
    if (lead) { st->done = 6; st->iters = it; }
    return;
  }
  if (lead) st->ro[it & 1] = ro;
  const double dx = ro - rop, dg = ro / rop;
  int64_t r0, r1;
  block_rows(n, r0, r1);
  double part = 0.;
  for (int64_t r = r0 + threadIdx.x; r < r1; r += kBlock) {
    x[r] += dx * h[r];
    const double gv = g[r] + dg * Ah[r];
    g[r] = gv;
    const double c = dinv ? dinv[r] * gv : gv;
    Cg[r] = c;
    part += c * gv;
  }
  const double tot = block_sum<kBlock>(part, lds);
  if (threadIdx.x == 0) pout[xcd_block_id()] = tot;
}

// ---------------------------------------------------------------- GMRES
// Restarted right-preconditioned GMRES with modified Gram-Schmidt
// (SolverGMRES::dosolver + fgmres, VirtualSolverCG.hpp:236-255, CG.cpp:347-517).
// Inner iteration it: k_gm_prec (V_it = w / ||w|| and Vp_it = C V_it),
// k_gm_matvec (w = A Vp_it), then the modified Gram-Schmidt coefficients of all
// basis vectors from one pass over the basis: h_i = (w - sum_{j<i} h_j V_j, V_i)
// = (w, V_i) - sum_{j<i} (V_i, V_j) h_j, so k_gm_dots forms the products (w, V_i)
// and (V_it, V_i), k_gm_coefs solves that unit lower triangular system and
// k_gm_project subtracts sum h_i V_i with the partial (w, w).  One kernel per
// basis vector, each waiting for the dot product of the one before, took 5.0 ms
// for the 36 iterations of a cube(20) system (666 dependent launches), this
// takes 1.1 ms (22 us of kernels per iteration, launch latency; the host looks
// every 8 iterations); for large n it reads the basis twice instead of three
// times and writes w once.  The Hessenberg column's Givens rotations and the convergence
// test are the reference's scalar code on the host.

// partial (r, r) of the right-hand side off the tgv rows: ||b|| of fgmres
__global__ __launch_bounds__(kBlock) void k_gm_normb(int64_t n, const double *__restrict__ b,
                                                     const uint8_t *__restrict__ wcl,
                                                     double *__restrict__ pout) {
  __shared__ double lds[kBlock / kWave];
  int64_t r0, r1;
  block_rows(n, r0, r1);
  double part = 0.;
  for (int64_t r = r0 + threadIdx.x; r < r1; r += kBlock) {
    const double v = (wcl && wcl[r]) ? 0. : b[r];
    part += v * v;
  }
  const double tot = block_sum<kBlock>(part, lds);
  if (threadIdx.x == 0) pout[xcd_block_id()] = tot;
}

// z = -(A u - b) (fgmres' ri, pCl the identity); partial (z, z)
template <int KIND>
__global__ FFHIP_MATVEC_ATTR void k_gm_residual(MatFmt<double> M, const double *__restrict__ u,
                                                const double *__restrict__ b,
                                                double *__restrict__ z,
                                                double *__restrict__ pout) {
  __shared__ double lds[kBlock / kWave];
  double part = 0.;
  matvec_rows<KIND, double, double>(
      M, [&](int32_t j) { return u[j]; },
      [&](int64_t r, double acc) {
        const double v = (acc + -1. * b[r]) * -1.;
        z[r] = v;
        part += v * v;
      });
  const double tot = block_sum<kBlock>(part, lds);
  if (threadIdx.x == 0) pout[xcd_block_id()] = tot;
}

// V = w / ||w||, ||w||^2 from the last projection's partials (pin null: the
// factor inv); Vp = C V (dinv null: the identity)
__global__ __launch_bounds__(kBlock) void k_gm_prec(int64_t n, double inv,
                                                    const double *__restrict__ pin,
                                                    const double *__restrict__ w,
                                                    const double *__restrict__ dinv,
                                                    double *__restrict__ V, double *__restrict__ Vp) {
  __shared__ double lds[kBlock / kWave];
  if (pin) inv = 1. / sqrt(reduce_partials(pin, gridDim.x, 1, 0, lds));
  int64_t r0, r1;
  block_rows(n, r0, r1);
  for (int64_t r = r0 + threadIdx.x; r < r1; r += kBlock) {
    const double v = inv * w[r];
    V[r] = v;
    Vp[r] = dinv ? dinv[r] * v : v;
  }
}

// w = A Vp
template <int KIND>
__global__ FFHIP_MATVEC_ATTR void k_gm_matvec(MatFmt<double> M, const double *__restrict__ Vp,
                                              double *__restrict__ w) {
  matvec_rows<KIND, double, double>(
      M, [&](int32_t j) { return Vp[j]; }, [&](int64_t r, double acc) { w[r] = acc; });
}

// partials of (w, V_i) and (V_it, V_i), i <= it, over the rows of block b.x:
// the waves of the blocks b.x, * share the i (a wave per i while the chip has
// room); component c of block b.x at part[c gridDim.x + b.x]
__global__ __launch_bounds__(kBlock) void k_gm_dots(int it, int64_t n, int64_t rows,
                                                    const double *const *__restrict__ V,
                                                    const double *__restrict__ w,
                                                    double *__restrict__ part) {
  const int lane = threadIdx.x % kWave;
  const int64_t r0 = blockIdx.x * rows, r1 = r0 + rows < n ? r0 + rows : n;
  const double *vit = V[it];
  for (int i = blockIdx.y * kWavesPerBlock + wave_id(); i <= it; i += gridDim.y * kWavesPerBlock) {
    const double *vi = V[i];
    double a = 0., b = 0.;
#pragma unroll 4
    for (int64_t r = r0 + lane; r < r1; r += kWave) {
      const double v = vi[r];
      a += v * w[r];
      b += v * vit[r];
    }
    a = wave_sum(a);
    b = wave_sum(b);
    if (lane == 0) {
      part[(int64_t)(2 * i) * gridDim.x + blockIdx.x] = a;
      part[(int64_t)(2 * i + 1) * gridDim.x + blockIdx.x] = b;
    }
  }
}

// The coefficients h_0..h_it (into h) from the P partials per component, one
// block.  L holds the products (V_i, V_j), j < i, packed by rows (row i at
// i (i - 1) / 2); row it is written here.
constexpr int kGmBlock = 1024;
__global__ __launch_bounds__(kGmBlock) void k_gm_coefs(int it, int P, const double *__restrict__ part,
                                                       double *__restrict__ L, double *__restrict__ h) {
  __shared__ double cur;
  const int t = threadIdx.x, lane = t % kWave;
  auto row = [&](int64_t i) { return L + i * (i - 1) / 2; };
  constexpr int NW = kGmBlock / kWave, C = 4;  // components a wave sums at a time
  for (int c0 = t / kWave; c0 < 2 * (it + 1); c0 += C * NW) {
    double s[C] = {0., 0., 0., 0.};
    for (int b = lane; b < P; b += kWave)
#pragma unroll
      for (int u = 0; u < C; ++u)
        if (c0 + u * NW < 2 * (it + 1)) s[u] += part[(int64_t)(c0 + u * NW) * P + b];
#pragma unroll
    for (int u = 0; u < C; ++u) {
      const int c = c0 + u * NW, i = c >> 1;
      s[u] = wave_sum(s[u]);
      if (lane != 0 || c >= 2 * (it + 1)) continue;
      if (!(c & 1)) h[i] = s[u];
      else if (i < it) row(it)[i] = s[u];
    }
  }
  __syncthreads();
  constexpr int U = 8;  // columns whose entries are loaded ahead
  if (it < kWave) {  // one wave, the unknowns in its lanes
    if (t >= kWave) return;
    double s = lane <= it ? h[lane] : 0.;
    const double *l = row(lane);
    for (int j0 = 0; j0 <= it; j0 += U) {
      double e[U];
#pragma unroll
      for (int u = 0; u < U; ++u) e[u] = lane <= it && j0 + u < lane ? l[j0 + u] : 0.;
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (j0 + u < it) s -= e[u] * __shfl(s, j0 + u, kWave);
    }
    if (lane <= it) h[lane] = s;
    return;
  }
  // columns in order; thread t holds the unknowns t, t + kGmBlock, ... of one
  // sweep at a time, so a sweep's unknowns are first freed of the earlier ones
  for (int i0 = 0; i0 <= it; i0 += kGmBlock) {
    const int i = i0 + t;
    double s = i <= it ? h[i] : 0.;
    if (i <= it)
      for (int j = 0; j < i0; ++j) s -= row(i)[j] * h[j];
    const int iend = i0 + kGmBlock - 1 < it ? i0 + kGmBlock - 1 : it;
    for (int j0 = i0; j0 <= iend; j0 += U) {
      double e[U];
#pragma unroll
      for (int u = 0; u < U; ++u) e[u] = i <= it && j0 + u < i ? row(i)[j0 + u] : 0.;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (j0 + u > iend) break;  // uniform
        if (i == j0 + u) cur = s;
        __syncthreads();
        s -= e[u] * cur;
        __syncthreads();
      }
    }
    if (i <= it) h[i] = s;
    __syncthreads();
  }
}

// w -= sum_{i <= it} h_i V_i, in order; partial (w, w)
__global__ __launch_bounds__(kBlock) void k_gm_project(int it, int64_t n,
                                                       const double *const *__restrict__ V,
                                                       const double *__restrict__ h,
                                                       double *__restrict__ w,
                                                       double *__restrict__ pout) {
  __shared__ double lds[kBlock / kWave];
  int64_t r0, r1;
  block_rows(n, r0, r1);
  double part = 0.;
  for (int64_t r = r0 + threadIdx.x; r < r1; r += kBlock) {
    double v = w[r];
#pragma unroll 8
    for (int i = 0; i <= it; ++i) v -= h[i] * V[i][r];
    w[r] = v;
    part += v * v;
  }
  const double tot = block_sum<kBlock>(part, lds);
  if (threadIdx.x == 0) pout[xcd_block_id()] = tot;
}

// x = (sum_i y_i Vp_i) + x0, the sum taken in order i = 0..k-1
__global__ __launch_bounds__(kBlock) void k_gm_update(int64_t n, int k, const double *__restrict__ y,
                                                      const double *const *__restrict__ Vp,
                                                      const double *__restrict__ x0,
                                                      double *__restrict__ x) {
  int64_t r0, r1;
  block_rows(n, r0, r1);
  for (int64_t r = r0 + threadIdx.x; r < r1; r += kBlock) {
    double acc = 0.;
#pragma unroll 8
    for (int i = 0; i < k; ++i) acc += y[i] * Vp[i][r];
    x[r] = acc + x0[r];
  }
}

// plain mat-vec for measurement: y = A x
template <int KIND, class V, class X>
__global__ FFHIP_MATVEC_ATTR void k_matvec(MatFmt<V> M, const X *__restrict__ x, X *__restrict__ y) {
  if constexpr (KIND == kSell16 && sizeof(X) == 8) {
    const auto xr = slice_rsrc(x, (uint32_t)(M.n * 8));  // n < 2^28 in this layout
    matvec_rows<KIND, V, X>(
        M, [&](int32_t j) { return __builtin_bit_cast(X, __builtin_amdgcn_raw_buffer_load_b64(xr, j * 8, 0, 0)); },
        [&](int64_t r, X acc) { y[r] = acc; });
  } else {
    matvec_rows<KIND, V, X>(M, [&](int32_t j) { return x[j]; }, [&](int64_t r, X acc) { y[r] = acc; });
  }
}

// ---------------------------------------------------------------- MIXED (FP32 inner)
// Mixed-precision state lives in CgState: sigma (scale of r32), rho32 (last
// (r32,r32)), and the per-parity (r32,r32) history below.
struct MixState {
  double rho_prev[2];   // (r32, r32) at the start of inner iteration, by parity
  double cbeta;         // coefficient of p_old in the first iteration after an update
  int first_it;         // inner iteration that uses cbeta
  int since_update;     // host-side bookkeeping copy
};

// K_m1: p = r32 + cb*p_old (on the fly for every gathered column); q = Ahat p;
// partial (p, q).  Requests a reliable update when (r32, r32) fell by
// kMixUpdate
// since the last update, or the recurrence says the FP64 criterion is met.
// Start of inner iteration it = it0 + c: rho = (r32, r32) from the last
// update's partials, the requests (reliable update, itmax, NaN) and the
// coefficient of p_old.  Returns false when the chunk stops.
__device__ inline bool mix_begin(int c, const double *__restrict__ pin, CgState *st, MixState *ms,
                                 double *lds, float &cbf) {
  const int it = st->it0 + c, itmax = st->itmax;
  const double rho = reduce_partials(pin, gridDim.x, 1, 0, lds);
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  const double sig = st->sigma;
  int req = 0;
  if (rho != rho) req = 4;
  else if (rho * sig * sig < st->eps2 || rho < kMixUpdate) req = 1;  // check on the FP64 residual
  else if (it - 1 >= itmax) req = 3;
  if (req) {
    if (lead) {
      if (req == 4) st->done = 4;
      else if (req == 3) st->done = 3;
      else st->need_update = 1;
      // (r32, r32) of the last executed iteration: the denominator of beta once
      // the newest recurrence residual is replaced by the FP64 one
      st->rho32 = ms->rho_prev[(it - 1) & 1];
      st->iters = it - 1;
    }
    return false;
  }
  const double cb = (it == ms->first_it) ? ms->cbeta : rho / ms->rho_prev[(it - 1) & 1];
  if (lead) { ms->rho_prev[it & 1] = rho; st->iters = it - 1; }
  cbf = (float)cb;
  return true;
}

// K_m1: p = r32 + cb p_old (elementwise); K_m2: q = Ahat p, partial (p, q).
// Requests a reliable update when (r32, r32) fell by kMixUpdate since the last
// update, or the recurrence says the FP64 criterion is met.
__global__ __launch_bounds__(kBlock) void k_mix_dirvec(int c, int64_t n,
                                                       const float *__restrict__ pold,
                                                       const float *__restrict__ r32,
                                                       float *__restrict__ pnew,
                                                       const double *__restrict__ pin, CgState *st,
                                                       MixState *ms) {
  __shared__ double lds[kBlock / kWave];
  if (st->done || st->need_update) return;
  float cbf;
  if (!mix_begin(c, pin, st, ms, lds, cbf)) return;
  int64_t r0, r1, a4, b4;
  block_rows(n, r0, r1);
  block_rows4(r0, r1, a4, b4);
  for (int64_t r = r0 + threadIdx.x; r < a4; r += kBlock) pnew[r] = r32[r] + cbf * pold[r];
  for (int64_t i = a4 / 4 + threadIdx.x; i < b4 / 4; i += kBlock) {
    const float4 rv = reinterpret_cast<const float4 *>(r32)[i];
    const float4 po = reinterpret_cast<const float4 *>(pold)[i];
    float4 pn;
    pn.x = rv.x + cbf * po.x; pn.y = rv.y + cbf * po.y;
    pn.z = rv.z + cbf * po.z; pn.w = rv.w + cbf * po.w;
    reinterpret_cast<float4 *>(pnew)[i] = pn;
  }
  for (int64_t r = b4 + threadIdx.x; r < r1; r += kBlock) pnew[r] = r32[r] + cbf * pold[r];
}

template <int KIND>
__global__ FFHIP_MATVEC_ATTR void k_mix_matvec(MatFmt<float> M, const float *__restrict__ p,
                                               float *__restrict__ q, double *__restrict__ pout,
                                               const CgState *st) {
  __shared__ double lds[kBlock / kWave];
  if (st->done || st->need_update) return;
  double part = 0.;
  matvec_rows<KIND, float, float>(
      M, [&](int32_t j) { return p[j]; },
      [&](int64_t r, float acc) {
        q[r] = acc;
        part += (double)p[r] * (double)acc;
      });
  const double tot = block_sum<kBlock>(part, lds);
  if (threadIdx.x == 0) pout[xcd_block_id()] = tot;
}

// K_m1 and K_m2 in one launch: p formed for every gathered column
template <int KIND>
__global__ FFHIP_MATVEC_ATTR void k_mix_dir_matvec(int c, MatFmt<float> M, const float *__restrict__ pold,
                                                   const float *__restrict__ r32, float *__restrict__ pnew,
                                                   float *__restrict__ q, const double *__restrict__ pin,
                                                   double *__restrict__ pout, CgState *st, MixState *ms) {
  __shared__ double lds[kBlock / kWave];
  if (st->done || st->need_update) return;
  float cbf;
  if (!mix_begin(c, pin, st, ms, lds, cbf)) return;
  const auto p = [&](int64_t j) { return r32[j] + cbf * pold[j]; };
  double part = 0.;
  matvec_rows<KIND, float, float>(
      M, [&](int32_t j) { return p(j); },
      [&](int64_t r, float acc) {
        const float pr = p(r);
        pnew[r] = pr;
        q[r] = acc;
        part += (double)pr * (double)acc;
      });
  const double tot = block_sum<kBlock>(part, lds);
  if (threadIdx.x == 0) pout[xcd_block_id()] = tot;
}

// K_m3: alpha = rho/(p,q); y32 += alpha p; r32 -= alpha q; partial (r32, r32)
__global__ __launch_bounds__(kBlock) void k_mix_update(
    int c, int64_t n, const float *__restrict__ p, const float *__restrict__ q,
    float *__restrict__ y32, float *__restrict__ r32, const double *__restrict__ pin,
    double *__restrict__ pout, CgState *st, MixState *ms) {
  __shared__ double lds[kBlock / kWave];
  if (st->done || st->need_update) return;
  const int it = st->it0 + c;
  const int P = gridDim.x;
  const double pq = reduce_partials(pin, P, 1, 0, lds);
  const double alpha = ms->rho_prev[it & 1] / pq;
  const float af = (float)alpha;
  if (blockIdx.x == 0 && threadIdx.x == 0) st->iters = it;
  int64_t r0, r1, a4, b4;
  block_rows(n, r0, r1);
  block_rows4(r0, r1, a4, b4);
  double part = 0.;
  auto one = [&](int64_t r) {
    y32[r] += af * p[r];
    const float rr = r32[r] - af * q[r];
    r32[r] = rr;
    part += (double)rr * (double)rr;
  };
  for (int64_t r = r0 + threadIdx.x; r < a4; r += kBlock) one(r);
  for (int64_t i = a4 / 4 + threadIdx.x; i < b4 / 4; i += kBlock) {
    const float4 pv = reinterpret_cast<const float4 *>(p)[i];
    const float4 qv = reinterpret_cast<const float4 *>(q)[i];
    float4 yv = reinterpret_cast<const float4 *>(y32)[i];
    float4 rv = reinterpret_cast<const float4 *>(r32)[i];
    yv.x += af * pv.x; yv.y += af * pv.y; yv.z += af * pv.z; yv.w += af * pv.w;
    rv.x -= af * qv.x; rv.y -= af * qv.y; rv.z -= af * qv.z; rv.w -= af * qv.w;
    reinterpret_cast<float4 *>(y32)[i] = yv;
    reinterpret_cast<float4 *>(r32)[i] = rv;
    part += (double)rv.x * (double)rv.x;
    part += (double)rv.y * (double)rv.y;
    part += (double)rv.z * (double)rv.z;
    part += (double)rv.w * (double)rv.w;
  }
  for (int64_t r = b4 + threadIdx.x; r < r1; r += kBlock) one(r);
  const double tot = block_sum<kBlock>(part, lds);
  if (threadIdx.x == 0) pout[xcd_block_id()] = tot;
}

// end of a chunk of CG launches: the next chunk starts `chunk` iterations on;
// the state goes to the host's copy
__global__ void k_cg_advance(CgState *st, int chunk, CgState *host) {
  if (threadIdx.x != 0) return;
  st->it0 += chunk;
  *host = *st;
}
// a small struct from the launch's arguments to the device
template <class T>
__global__ void k_put(T *dst, T v) {
  *dst = v;
}

// fold the FP32 correction into the FP64 solution: x += D^-1/2 (sigma y32); y32 = 0
__global__ void k_mix_fold(int64_t n, double sigma, const double *__restrict__ dsc,
                           float *__restrict__ y32, double *__restrict__ x) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  x[i] += dsc[i] * (sigma * (double)y32[i]);
  y32[i] = 0.f;
}

// new scaled residual r32 = D^-1/2 r / sigma (r = b - A x in FP64); partial (r32,r32)
__global__ __launch_bounds__(kBlock) void k_mix_rescale(
    int64_t n, double inv_sigma, const double *__restrict__ dsc,
    const double *__restrict__ r, float *__restrict__ r32, double *__restrict__ pout) {
  __shared__ double lds[kBlock / kWave];
  int64_t r0, r1;
  block_rows(n, r0, r1);
  double part = 0.;
  for (int64_t i = r0 + threadIdx.x; i < r1; i += kBlock) {
    const float v = (float)(dsc[i] * r[i] * inv_sigma);
    r32[i] = v;
    part += (double)v * (double)v;
  }
  const double tot = block_sum<kBlock>(part, lds);
  if (threadIdx.x == 0) pout[xcd_block_id()] = tot;
}

static unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

// CG iterations launched per host poll of the device state; one chunk is
// captured once into a hipGraph and replayed (even, so the two-buffer
// parities of a chunk repeat)
constexpr int kChunk = 16;

// stream-captures the launches of f() into an executable graph
template <class F>
hipGraphExec_t capture_graph(hipStream_t s, F f) {
  hipGraph_t g = nullptr;
  hipGraphExec_t e = nullptr;
  FFHIP_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeRelaxed));
  try {
    f();
  } catch (...) {  // the stream must leave capture mode whatever happened
    if (hipStreamEndCapture(s, &g) == hipSuccess && g) (void)hipGraphDestroy(g);
    (void)hipGetLastError();
    throw;
  }
  const hipError_t le = hipGetLastError();
  const hipError_t ce = hipStreamEndCapture(s, &g);
  if (le != hipSuccess || ce != hipSuccess) {
    if (g) (void)hipGraphDestroy(g);
    FFHIP_CHECK(le);
    FFHIP_CHECK(ce);
  }
  const hipError_t ie = hipGraphInstantiate(&e, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  FFHIP_CHECK(ie);
  return e;
}

}  // namespace ffhip

using namespace ffhip;

struct ffhip_cg_s {
  ffhip_ctx ctx = nullptr;
  ffhip_mat A = nullptr;
  int mode = 0;
  int fmt = kSell;
  int far_pending = 0;  // kSell16 chosen before the fill has checked every column delta
  int64_t n = 0, S = 0, ents = 0;
  int grid = 0;
  // kSell layout (kCsrV streams A's own rowptr/colidx)
  int64_t *sptr = nullptr;
  int32_t *slen = nullptr, *scol = nullptr;
  int16_t *scol16 = nullptr;  // kSell16
  int64_t *sptr16 = nullptr;  // kSell16 slice offsets of scol16
  int32_t *bcol = nullptr;    // kBsr3 block columns (slices over sorted node rows)
  int32_t *bperm = nullptr;   // kBsr3 node row of each sorted position
  bool bshare = false;        // kBsr3 a mat-vec block's waves take its slices together
  int32_t *bwave = nullptr;   // kBsr3 first slice of each mat-vec block or wave, and the end
  // values in the solver's layout; for kCsrV, sval is A's value array (borrowed)
  double *sval = nullptr;    // A
  double *svalT = nullptr;   // A^T (built on first transposed solve)
  float *sval32 = nullptr;   // D^-1/2 A D^-1/2 (MIXED)
  float *sval32T = nullptr;
  // Jacobi / tgv
  double *dinv = nullptr, *dsc = nullptr;
  uint8_t *wcl = nullptr;
  double tgvm = 0.;
  int ntgv = 0;
  SetupRb *rb = nullptr;  // set-up figures for the host (one copy per set-up)
  // work
  double *xw = nullptr, *bw = nullptr, *G = nullptr, *CG = nullptr, *H[2] = {nullptr, nullptr},
         *AH = nullptr;
  float *r32 = nullptr, *p32[2] = {nullptr, nullptr}, *q32 = nullptr, *y32 = nullptr;
  double *pA = nullptr, *pB = nullptr;
  CgState *st = nullptr;
  MixState *ms = nullptr;
  Cg2State *st2 = nullptr;  // affine CG (LinearCG)
  // GMRES: Krylov basis V_i and C V_i, allocated vector by vector as a solve
  // first reaches them (as the reference's KN<KN<K>> are) and kept; the device
  // tables of their pointers; w, x0, y, the partials of the dot products, the
  // packed products (V_i, V_j), and per iteration of a batch the coefficients
  // with the partials of ||w||^2 (gmOut, and its page-locked host copy)
  static constexpr int kGmBatch = 8;
  std::vector<double *> gmV, gmVp;
  double **gmVDev = nullptr, **gmVpDev = nullptr;
  int gmCap = 0;  // vectors the tables and the buffers below are sized for
  double *gmW = nullptr, *gmX0 = nullptr, *gmY = nullptr, *gmS = nullptr, *gmL = nullptr, *gmOut = nullptr;
  double *gmOutH = nullptr;
  int gm_blocks() const {  // blocks of the dot products
    const int64_t b = (n + 255) / 256;
    return (int)(b < 256 ? b : 256);
  }
  int64_t gm_out() const { return (int64_t)gmCap + grid; }  // doubles per iteration of gmOut
  // room for `need` vectors, and for up to `want` while device memory lasts
  void gm_basis(int need, int want) {
    if (!gmW) gmW = dalloc<double>(n);
    if (!gmX0) gmX0 = dalloc<double>(n);
    if (want > gmCap) {
      try {
        gm_tables(std::max(std::max(want, 2 * gmCap), 64));
      } catch (const Error &) {
        if (need > gmCap) throw;
      }
    }
    const size_t k0 = gmV.size(), k = (size_t)std::min(want, gmCap);
    if (k <= k0) return;
    gmV.reserve(k);
    gmVp.reserve(k);
    while (gmV.size() < k) {
      double *v = nullptr, *vp = nullptr;
      try {
        v = dalloc<double>(n);
        vp = dalloc<double>(n);
      } catch (const Error &) {
        dfree(v);
        break;
      }
      gmV.push_back(v);
      gmVp.push_back(vp);
    }
    if (const size_t c = gmV.size() - k0) {
      FFHIP_CHECK(hipMemcpy(gmVDev + k0, gmV.data() + k0, sizeof(double *) * c, hipMemcpyHostToDevice));
      FFHIP_CHECK(hipMemcpy(gmVpDev + k0, gmVp.data() + k0, sizeof(double *) * c, hipMemcpyHostToDevice));
    }
    FFHIP_REQUIRE((int)gmV.size() >= need, FFHIP_ERR_HIP,
                  "ffhip_gmres_solve: out of device memory at %d basis vectors", (int)gmV.size());
  }
  // the tables and buffers for cap vectors: all of them, or as they were
  void gm_tables(int cap) {
    double **pv = nullptr, **p = nullptr, *y = nullptr, *S = nullptr, *L = nullptr, *out = nullptr;
    void *outH = nullptr;
    try {
      pv = dalloc<double *>(cap);
      p = dalloc<double *>(cap);
      y = dalloc<double>(cap + 1);
      S = dalloc<double>(2 * (int64_t)cap * gm_blocks());
      L = dalloc<double>((int64_t)cap * (cap - 1) / 2);
      out = dalloc<double>(kGmBatch * ((int64_t)cap + grid));
      FFHIP_CHECK(hipHostMalloc(&outH, 8 * kGmBatch * ((int64_t)cap + grid), hipHostMallocDefault));
      if (gmCap) {
        FFHIP_CHECK(hipMemcpy(L, gmL, 8 * (size_t)gmCap * (gmCap - 1) / 2, hipMemcpyDeviceToDevice));
        FFHIP_CHECK(hipMemcpy(pv, gmV.data(), sizeof(double *) * gmV.size(), hipMemcpyHostToDevice));
        FFHIP_CHECK(hipMemcpy(p, gmVp.data(), sizeof(double *) * gmVp.size(), hipMemcpyHostToDevice));
      }
    } catch (...) {
      dfree(pv); dfree(p); dfree(y); dfree(S); dfree(L); dfree(out);
      if (outH) (void)hipHostFree(outH);
      throw;
    }
    dfree(gmVDev); dfree(gmVpDev); dfree(gmY); dfree(gmS); dfree(gmL); dfree(gmOut);
    if (gmOutH) (void)hipHostFree(gmOutH);
    gmVDev = pv; gmVpDev = p; gmY = y; gmS = S; gmL = L; gmOut = out; gmOutH = (double *)outH; gmCap = cap;
  }
  // captured chunks of CG launches, keyed by (mode, value array, parity of the
  // chunk's first iteration); kernel by kernel when eager or profiling (event
  // records captured in a graph carry no timestamps hipEventElapsedTime reads)
  struct Chunk {
    int kind;
    const void *val;
    int par;
    hipGraphExec_t exec;
  };
  std::vector<Chunk> graphs;
  int use_graph = 1;
  // symmetric values of an FP64 kSell16 solver (k_pcg_matvec_sym)
  enum Sym { kSymUnknown, kSymThere, kSymNot, kSymNever };  // not looked for since the values
  // changed; there; not with these values (or no room); the pattern has not that form
  Sym sym = kSymUnknown;
  int sym_nl = 0, sym_nu = 0;
  double *symval = nullptr;
  uint8_t *symcls = nullptr;
  SymPattern *symtab = nullptr;
  template <class F>
  hipGraphExec_t graph(int kind, const void *val, int par, F launch) {
    if (!use_graph || profile) return nullptr;
    for (const Chunk &c : graphs)
      if (c.kind == kind && c.val == val && c.par == par) return c.exec;
    graphs.push_back({kind, val, par, capture_graph(ctx->stream, launch)});
    return graphs.back().exec;
  }
  // per-kernel timing (measurement only): 4 events per iteration of a chunk,
  // around the direction, mat-vec and update kernels
  int profile = 0;
  std::vector<hipEvent_t> ev;
  double t_dv = 0., t_mv = 0., t_up = 0.;
  int n_timed = 0;
  void ensure_events(int k) {
    while ((int)ev.size() < k) {
      hipEvent_t e;
      FFHIP_CHECK(hipEventCreate(&e));
      ev.push_back(e);
    }
  }
  void mark(int slot) {
    if (profile) FFHIP_CHECK(hipEventRecord(ev[slot], ctx->stream));
  }
  // after a synchronised chunk: accumulate the iterations [it0, it1] that ran
  void collect(int chunk_first_it, int nits, int last_exec_it) {
    if (!profile) return;
    for (int c = 0; c < nits; ++c) {
      const int it = chunk_first_it + c;
      if (it > last_exec_it) break;
      float d = 0.f, a = 0.f, b = 0.f;
      FFHIP_CHECK(hipEventElapsedTime(&d, ev[4 * c], ev[4 * c + 1]));
      FFHIP_CHECK(hipEventElapsedTime(&a, ev[4 * c + 1], ev[4 * c + 2]));
      FFHIP_CHECK(hipEventElapsedTime(&b, ev[4 * c + 2], ev[4 * c + 3]));
      t_dv += d; t_mv += a; t_up += b; ++n_timed;
    }
  }
  // The direction formed in the mat-vec (not for 3x3 blocks, whose mat-vec gains
  // little from one launch less), up to where the second gathered vector costs
  // what the launch did.  That depends on the gathers: a wave's 64 of them take 4
  // lines where consecutive rows hold consecutive columns (box meshes), up to 64
  // in an arbitrary numbering.  us per iteration, apart / together, FP64 on
  // cubes: 15.6 k rows 12.7 / 10.6, 69 k 15.4 / 14.3, 314 k 24.6 / 23.5 (531 k 42 /
  // 48); the vertices shuffled within 30: 97 k 15.6 / 14.6, 227 k 21.7 / 20.9, within
  // 300: 227 k 22.6 / 22.8; numbered at random: 9.3 k 14.0 / 13.8, 15.6 k 14.3 / 14.2,
  // 30 k 16.5 / 17.7, 69 k 20.5 / 24.7, 314 k 41.3 / 66.5; scalar P2 (CSR) 24 k 16.0 /
  // 15.1, 69 k 26.4 / 27.7, 275 k 73.4 / 86.4.  MIXED on cubes: 69 k 19.3 / 16.4, 1.03 M
  // 35.6 / 34.1 (cube(128) 36.9 / 37.9 ms a solve); within 30: 227 k 21.0 / 19.4, 531 k
  // 28.3 / 28.6, 1.03 M 36.7 / 39.9; at random 30 k 20.8 / 20.7, 69 k 23.8 / 25.7, 1.03 M
  // 102 / 230; P2 24 k 21.1 / 18.6, 149 k 41.3 / 41.4.  FP64 systems of one workgroup's
  // size keep the launches' bits of k_pcg_small.
  // order (kSell16, sample_order): most sampled entries are followed by the next column (2), by
  // one near it (1), or not (0)
  int order = 0;
  int64_t fuse_small() const { return mode == FFHIP_CG_MIXED ? 1 << 15 : 1 << 14; }
  int64_t fuse_large() const { return mode == FFHIP_CG_MIXED ? 1 << 20 : 5 << 16; }
  bool fuse() const {
    if (fmt == kBsr3 || (mode == FFHIP_CG_FP64 && n <= kSmallRows)) return false;
    const int64_t most = fmt != kSell16 || order == 0 ? fuse_small() : order == 1 ? 1 << 18 : fuse_large();
    return n <= most;
  }
  // the state as the host reads it after a chunk (k_cg_advance writes it)
  CgState *host_state() const { return static_cast<CgState *>(ctx->pinned_data()); }
  // bytes of the matrix that one mat-vec streams, with values of `size` bytes
  int64_t matrix_bytes(size_t size) const {
    if (fmt == kBsr3) return ents * (int64_t)(9 * size + 4);
    return ents * (int64_t)(size + (fmt == kSell16 ? 2 : 4));
  }
  template <class V>
  MatFmt<V> fmt_of(const V *val) const {
    MatFmt<V> M;
    M.n = n;
    M.S = S;
    M.col16 = scol16;
    M.ptr16 = sptr16;
    M.nb = 0;
    M.perm = bperm;
    if (fmt == kSell || fmt == kSell16) { M.ptr = sptr; M.len = slen; M.col = scol; }
    else if (fmt == kBsr3) { M.ptr = sptr; M.len = slen; M.col = bcol; M.nb = n / 3; }
    else { M.ptr = A->rowptr; M.len = nullptr; M.col = A->colidx; }
    M.wstart = bwave;
    M.val = val;
    M.nt = matrix_bytes(sizeof(V)) > kCachedMatrix;
    return M;
  }
};

// launch a layout-templated mat-vec kernel with the solver's layout (_ROWS: not
// the 3x3 blocks)
#define FFHIP_LAUNCH_ROWS(cg, kern, grid, stream, ...)                       \
  do {                                                                       \
    if ((cg)->fmt == kSell) kern<kSell><<<(grid), kBlock, 0, (stream)>>>(__VA_ARGS__); \
    else if ((cg)->fmt == kSell16) kern<kSell16><<<(grid), kBlock, 0, (stream)>>>(__VA_ARGS__); \
    else kern<kCsrV><<<(grid), kBlock, 0, (stream)>>>(__VA_ARGS__);           \
  } while (0)
#define FFHIP_LAUNCH_FMT(cg, kern, grid, stream, ...)                        \
  do {                                                                       \
    if ((cg)->fmt == kBsr3 && (cg)->bshare) kern<kBsr3><<<(grid), kBlock, 0, (stream)>>>(__VA_ARGS__); \
    else if ((cg)->fmt == kBsr3) kern<kBsr3W><<<(grid), kBlock, 0, (stream)>>>(__VA_ARGS__); \
    else FFHIP_LAUNCH_ROWS(cg, kern, grid, stream, __VA_ARGS__);              \
  } while (0)

#define FFHIP_LAUNCH_MATVEC(cg, T, M, x, y, stream)                                          \
  do {                                                                                      \
    if ((cg)->fmt == kSell)                                                                 \
      k_matvec<kSell, T, T><<<(cg)->grid, kBlock, 0, (stream)>>>(M, (const T *)(x), (T *)(y)); \
    else if ((cg)->fmt == kSell16)                                                          \
      k_matvec<kSell16, T, T><<<(cg)->grid, kBlock, 0, (stream)>>>(M, (const T *)(x), (T *)(y)); \
    else if ((cg)->fmt == kBsr3 && !(cg)->bshare)                                           \
      k_matvec<kBsr3W, T, T><<<(cg)->grid, kBlock, 0, (stream)>>>(M, (const T *)(x), (T *)(y)); \
    else if ((cg)->fmt == kBsr3)                                                            \
      k_matvec<kBsr3, T, T><<<(cg)->grid, kBlock, 0, (stream)>>>(M, (const T *)(x), (T *)(y)); \
    else                                                                                    \
      k_matvec<kCsrV, T, T><<<(cg)->grid, kBlock, 0, (stream)>>>(M, (const T *)(x), (T *)(y)); \
  } while (0)

// the set-up figures to the host (one copy, after the stream's work so far);
// the tgv figures into the solver
static SetupRb setup_readback(ffhip_cg cg) {
  SetupRb h;
  fetch(cg->ctx, {{&h, cg->rb, sizeof(h)}});
  cg->tgvm = h.ttgv;
  cg->ntgv = (int)h.ntgv;
  return h;
}

// Layout choice: sliced ELL unless its slices pad the matrix by more than 25 %
// (rows of very different lengths), then CSR with 16 lanes per row.
static void cg_plan_layout(ffhip_cg cg, int layout, bool index32) {
  ffhip_ctx ctx = cg->ctx;
  ffhip_mat A = cg->A;
  hipStream_t s = ctx->stream;
  cg->S = (A->n + kSlice - 1) / kSlice;
  if (A->nodeptr && A->ncomp == 3 &&
      (layout == FFHIP_CG_LAYOUT_AUTO || layout == FFHIP_CG_LAYOUT_BSR3)) {
    // vector P2: the node rows are 3x3 blocks; slices over node rows sorted by
    // length inside windows of 4096 rows
    cg->fmt = kBsr3;
    const int64_t nb = A->n / 3, S3 = (nb + kSlice - 1) / kSlice;
    uint32_t *keys = dalloc<uint32_t>(nb), *skeys = dalloc<uint32_t>(nb);
    int32_t *vals = dalloc<int32_t>(nb);
    cg->bperm = dalloc<int32_t>(nb);
    k_bsr_keys<<<nblk(nb, 256), 256, 0, s>>>(nb, A->nodeptr, keys, vals);
    size_t tb = 0;
    FFHIP_CHECK(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, keys, skeys, vals, cg->bperm, (int)nb,
                                                   0, 32, s));
    char *tmp = dalloc<char>(tb);
    FFHIP_CHECK(hipcub::DeviceRadixSort::SortPairs(tmp, tb, keys, skeys, vals, cg->bperm, (int)nb, 0,
                                                   32, s));
    cg->sptr = dalloc<int64_t>(S3 + 1);
    cg->slen = dalloc<int32_t>(S3);
    int64_t *cnt = dalloc<int64_t>(S3 + 1);
    k_bsr_len<<<nblk(S3 * kSlice, 256), 256, 0, s>>>(nb, S3, A->nodeptr, cg->bperm, cg->slen, cnt);
    exclusive_scan_i64(ctx, cnt, cg->sptr, S3 + 1);
    k_setup_sizes<<<1, 1, 0, s>>>(cg->rb, cg->sptr + S3, nullptr, 1);
    cg->ents = setup_readback(cg).ents;
    dfree(cnt); dfree(tmp); dfree(keys); dfree(skeys); dfree(vals);
    cg->bcol = dalloc<int32_t>(cg->ents);
  } else if (layout == FFHIP_CG_LAYOUT_BSR3) {
    FFHIP_REQUIRE(false, FFHIP_ERR_UNSUPPORTED, "ffhip_cg_create: 3x3 blocks need a [P2,P2,P2] matrix");
  } else if (layout != FFHIP_CG_LAYOUT_CSR) {
    // slice widths and offsets and the offsets of the packed 16-bit deltas,
    // then one read-back decides among sliced ELL with 16-bit deltas (the fill
    // then checks them), with int32 columns, and CSR
    Arena ar(ctx, 2 * Arena::bytes(cg->S + 1, 8));
    cg->sptr = dalloc<int64_t>(cg->S + 1);
    cg->slen = dalloc<int32_t>(cg->S);
    cg->sptr16 = dalloc<int64_t>(cg->S + 1);
    int64_t *cnt = ar.take<int64_t>(cg->S + 1);
    int64_t *cnt4 = ar.take<int64_t>(cg->S + 1);
    const bool sample = cg->n > cg->fuse_small() && cg->n <= cg->fuse_large();
    k_sell_len<<<nblk(cg->S * kSlice, kOrderBlock) + (sample ? 1 : 0), kOrderBlock, 0, s>>>(
        A->n, cg->S, A->rowptr, sample ? A->colidx : nullptr, cg->rb, cg->slen, cnt);
    exclusive_scan_i64(ctx, cnt, cg->sptr, cg->S + 1);
    // 16-bit column deltas unless index32: the fill checks every delta
    // against 2^15 and falls back to int32 columns (far_pending)
    k_sell_len4<<<nblk(cg->S, 256), 256, 0, s>>>(cg->S, cg->slen, cnt4);
    exclusive_scan_i64(ctx, cnt4, cg->sptr16, cg->S + 1);
    k_setup_sizes<<<1, 1, 0, s>>>(cg->rb, cg->sptr + cg->S, cg->sptr16 + cg->S, index32);
    FFHIP_CHECK(hipGetLastError());
    const SetupRb h = setup_readback(cg);
    cg->ents = h.ents;
    if (sample) cg->order = 2 * h.next >= h.entries ? 2 : 2 * h.near_ >= h.entries ? 1 : 0;
    if (layout == FFHIP_CG_LAYOUT_SELL || 4 * cg->ents <= 5 * A->nnz) {
      // 16-bit deltas, and gathers through buffer resources with 32-bit byte offsets
      if (h.far || A->n >= ((int64_t)1 << 28)) {
        cg->fmt = kSell;
        cg->scol = dalloc<int32_t>(cg->ents);
        dfree(cg->sptr16);
      } else {
        cg->fmt = kSell16;
        cg->scol16 = dalloc<int16_t>(h.ents16);
        cg->far_pending = 1;
      }
    } else {
      dfree(cg->sptr); dfree(cg->slen); dfree(cg->sptr16);
      cg->fmt = kCsrV;
    }
  } else {
    cg->fmt = kCsrV;
    setup_readback(cg);  // the tgv figures
  }
  int64_t g;
  if (cg->fmt == kBsr3) {
    g = (A->n / 3 + kSlice - 1) / kSlice;  // a block per slice, or a wave
    cg->bshare = g <= (int64_t)kWavesPerBlock * FFHIP_GRID_PER_CU * ctx->num_cu ||
                 cg->matrix_bytes(cg->mode == FFHIP_CG_MIXED ? 4 : 8) <= kCachedMatrix;
    if (!cg->bshare) g = (g + kWavesPerBlock - 1) / kWavesPerBlock;
  } else if (cg->fmt != kCsrV) {
    g = (cg->S + kWavesPerBlock - 1) / kWavesPerBlock;
  } else {
    cg->ents = A->nnz;
    g = (A->n + kBlock / kLanesPerRow - 1) / (kBlock / kLanesPerRow);
  }
  // resident blocks per CU: 3 of an FP32 solver and of 3x3-block slices that are not
  // shared, 2 of another FP64 one (FP64 mat-vecs at
  // 2 against 3: cube(160) 136.9 / 139.4 us, cube(96) 24.8 / 25.4, cube(20) 3x3 blocks
  // 29.1 / 29.7, the vector kernels within 3 %; FP32 cube(64) 6.6 / 5.6, cube(128)
  // 32.4 / 30.1)
  const bool three = cg->mode == FFHIP_CG_MIXED || (cg->fmt == kBsr3 && !cg->bshare);
  const int64_t gmax = (three ? FFHIP_GRID_PER_CU : 2) * (int64_t)ctx->num_cu;
  if (g > gmax) g = gmax;
  if (g >= 64) g -= g % 8;  // whole XCD groups
  if (g < 1) g = 1;
  cg->grid = (int)g;
  if (cg->fmt == kBsr3) {
    const int nw = cg->bshare ? cg->grid : cg->grid * kWavesPerBlock;
    cg->bwave = dalloc<int32_t>(nw + 1);
    k_bsr_waves<<<nblk(nw + 1, 256), 256, 0, s>>>((A->n / 3 + kSlice - 1) / kSlice, cg->sptr, nw,
                                                  cg->bwave);
    FFHIP_CHECK(hipGetLastError());
  }
}

// The diagonal values and presence flags the Jacobi set-up starts from, and
// the partials of its tgv passes.
struct DiagBufs {
  static constexpr int GB = 512;  // blocks of a tgv pass
  double *d;
  uint8_t *has;
  double *part;
  static size_t bytes(int64_t n) { return Arena::bytes(n, 8) + Arena::bytes(n, 1) + Arena::bytes(2 * GB, 8); }
  DiagBufs(Arena &ar, int64_t n) : d(ar.take<double>(n)), has(ar.take<uint8_t>(n)), part(ar.take<double>(2 * GB)) {}
};
static void cg_jacobi_tail(ffhip_cg cg, const DiagBufs &b);

// values in the solver's layout (A or A^T; FP32 scaled copy for MIXED).  With
// db the sliced-ELL fill also writes the diagonal and the Jacobi set-up runs
// behind it; with read_rb the tgv figures come back with the fill's wait.
static void cg_fill_values(ffhip_cg cg, bool transposed, const DiagBufs *db = nullptr,
                           bool read_rb = false) {
  ffhip_ctx ctx = cg->ctx;
  ffhip_mat A = cg->A;
  hipStream_t s = ctx->stream;
  int64_t *tmap = nullptr;
  if (transposed) {
    tmap = dalloc<int64_t>(A->nnz);
    // transposed values through the symmetric-pattern slot map
    const bool ok = transpose_map(ctx, A, tmap);
    if (!ok) dfree(tmap);
    FFHIP_REQUIRE(ok, FFHIP_ERR_UNSUPPORTED, "transposed solve needs a symmetric pattern");
  }
  const bool mixed = cg->mode == FFHIP_CG_MIXED;
  const bool check_far = !transposed && cg->far_pending && cg->fmt == kSell16;
  double *&dv = transposed ? cg->svalT : cg->sval;
  float *&fv = transposed ? cg->sval32T : cg->sval32;
  const int64_t nval = cg->fmt == kBsr3 ? 9 * cg->ents : cg->ents;
  if (mixed && !fv) fv = dalloc<float>(nval);
  if (cg->fmt == kBsr3) {
    if (!dv) dv = dalloc<double>(nval);
    const int64_t nb = A->n / 3, S3 = (nb + kSlice - 1) / kSlice;
    auto fill = tmap ? k_bsr_fill<true> : k_bsr_fill<false>;
    fill<<<S3, 256, 0, s>>>(nb, A->nodeptr, cg->bperm, cg->sptr, cg->slen, A->rowptr, A->colidx, A->vals,
                            tmap, cg->dsc, transposed ? nullptr : cg->bcol, dv, mixed ? fv : nullptr);
  } else if (cg->fmt != kCsrV) {
    if (!dv) dv = dalloc<double>(cg->ents);
    k_sell_fill<<<cg->S, 256, 0, s>>>(
        A->n, cg->S, A->rowptr, A->colidx, A->vals, tmap, cg->sptr, cg->slen, cg->dsc,
        transposed ? nullptr : cg->scol, cg->sptr16, transposed ? nullptr : cg->scol16, dv,
        mixed ? fv : nullptr, cg->fmt == kSell16, A->diag, db ? db->d : nullptr,
        db ? db->has : nullptr, check_far ? &cg->rb->far : nullptr);
    if (db) {
      FFHIP_CHECK(hipGetLastError());
      cg_jacobi_tail(cg, *db);
    }
  } else {
    double *dst = nullptr;
    if (transposed) {
      if (!dv) dv = dalloc<double>(cg->ents);
      dst = dv;
    } else {
      dv = A->vals;  // borrowed: A's CSR order is the layout
    }
    if (dst || mixed)
      k_csr_fill<<<nblk(A->n * kLanesPerRow, 256), 256, 0, s>>>(
          A->n, A->rowptr, A->colidx, A->vals, tmap, cg->dsc, dst, mixed ? fv : nullptr);
  }
  FFHIP_CHECK(hipGetLastError());
  SetupRb h{};
  if (read_rb || check_far) fetch(ctx, {{&h, cg->rb, sizeof(h)}});
  else FFHIP_CHECK(hipStreamSynchronize(s));
  if (read_rb) {
    cg->tgvm = h.ttgv;
    cg->ntgv = (int)h.ntgv;
  }
  dfree(tmap);
  if (check_far) {
    cg->far_pending = 0;
    if (h.far) {  // some column more than 2^15 from its row: int32 columns, filled again
      dfree(cg->scol16);
      dfree(cg->sptr16);
      cg->fmt = kSell;
      cg->scol = dalloc<int32_t>(cg->ents);
      cg_fill_values(cg, transposed, db, read_rb);
    }
  }
}

// Jacobi scaling and the tgv rows, on the device (the tgv figures reach the
// host with the next setup_readback)
static void cg_setup_jacobi(ffhip_cg cg) {
  const int64_t n = cg->A->n;
  Arena ar(cg->ctx, DiagBufs::bytes(n));
  const DiagBufs b(ar, n);
  k_diag_vals<<<nblk(n, 256), 256, 0, cg->ctx->stream>>>(n, cg->A->diag, cg->A->vals, b.d, b.has);
  cg_jacobi_tail(cg, b);
}

// the tgv passes and the Jacobi scaling from the diagonal in b
static void cg_jacobi_tail(ffhip_cg cg, const DiagBufs &b) {
  hipStream_t s = cg->ctx->stream;
  const int64_t n = cg->A->n;
  const int GB = DiagBufs::GB;
  const double *d = b.d;
  const uint8_t *has = b.has;
  double *part = b.part;
  k_tgv_pass<<<GB, kBlock, 0, s>>>(n, d, has, nullptr, 1, part);
  k_tgv_reduce<<<1, kBlock, 0, s>>>(GB, part, 1, cg->rb);
  k_tgv_pass<<<GB, kBlock, 0, s>>>(n, d, has, &cg->rb->ttgv, 2, part);
  k_tgv_reduce<<<1, kBlock, 0, s>>>(GB, part, 2, cg->rb);
  k_jacobi<<<nblk(n, 256), 256, 0, s>>>(n, d, has, cg->rb, cg->dinv, cg->dsc, cg->wcl);
  FFHIP_CHECK(hipGetLastError());
}

// r = b - A x (rout may be null); the three partial sums of k_residual added on
// the host in block order
static void residual_sums(ffhip_cg cg, const double *val, const double *x, const double *b,
                          double *rout, double out[3]) {
  hipStream_t s = cg->ctx->stream;
  FFHIP_REQUIRE(24 * (size_t)cg->grid <= ffhip_ctx_s::kPinnedData, FFHIP_ERR_INTERNAL, "residual partials");
  double *h = static_cast<double *>(cg->ctx->pinned_data());
  FFHIP_LAUNCH_FMT(cg, k_residual, cg->grid, s, cg->fmt_of(val), x, b, cg->dinv, rout, h);
  FFHIP_CHECK(hipGetLastError());
  FFHIP_CHECK(hipStreamSynchronize(s));
  out[0] = out[1] = out[2] = 0.;
  for (int i = 0; i < cg->grid; ++i)
    for (int c = 0; c < 3; ++c) out[c] += h[3 * i + c];
}

// residual r = b - A x into cg->G; returns (r, D^-1 r)
static double mix_residual(ffhip_cg cg, const double *sval) {
  double r[3];
  residual_sums(cg, sval, cg->xw, cg->bw, cg->G, r);
  return r[2];
}

// One chunk of FP64 PCG iterations it0 + c, c < kChunk, it0 = 1 (mod kChunk):
// the H buffer parity follows c.
static void launch_pcg_chunk(ffhip_cg cg, const double *sval, bool sym, bool marks) {
  hipStream_t s = cg->ctx->stream;
  const int G = cg->grid;
  const bool fused = cg->fuse();
  const MatFmt<double> M = cg->fmt_of(sval);
  for (int c = 0; c < kChunk; ++c) {
    if (marks) cg->mark(4 * c);
    if (!fused)
      k_pcg_dirvec<<<G, kBlock, 0, s>>>(c, cg->n, cg->H[c & 1], cg->dinv, cg->G, cg->H[(c + 1) & 1],
                                        cg->xw, cg->pA, cg->pB, cg->st);
    if (marks) cg->mark(4 * c + 1);
    if (fused)
      FFHIP_LAUNCH_ROWS(cg, k_pcg_dir_matvec, G, s, c, M, cg->H[c & 1], cg->CG, cg->G, cg->H[(c + 1) & 1],
                       cg->AH, cg->xw, cg->pA, cg->pB, cg->st);
    else if (sym)
      (cg->sym_nu == 4              ? k_pcg_matvec_sym<3, 4>
       : cg->sym_nl == kSymHalf - 1 ? k_pcg_matvec_sym<kSymHalf - 1, kSymHalf>
                                    : k_pcg_matvec_sym<kSymHalf, kSymHalf>)<<<G, kBlock, 0, s>>>(
          SymFmt{cg->n, cg->S, cg->symval, cg->symcls, cg->symtab}, cg->H[(c + 1) & 1], cg->AH, cg->pB, cg->st);
    else
      FFHIP_LAUNCH_FMT(cg, k_pcg_matvec, G, s, M, cg->H[(c + 1) & 1], cg->AH, cg->pB, cg->st);
    if (marks) cg->mark(4 * c + 2);
    k_pcg_update<<<G, kBlock, 0, s>>>(cg->n, cg->AH, cg->dinv, cg->G, fused ? cg->CG : nullptr, cg->pB,
                                      cg->pA, cg->st);
    if (marks) cg->mark(4 * c + 3);
  }
  k_cg_advance<<<1, 64, 0, s>>>(cg->st, kChunk, cg->host_state());
}

// One chunk of MIXED inner iterations it0 + c, par = it0 & 1.
static void launch_mix_chunk(ffhip_cg cg, const float *sval32, int par, bool marks) {
  hipStream_t s = cg->ctx->stream;
  const int G = cg->grid;
  const MatFmt<float> M32 = cg->fmt_of(sval32);
  const bool fused = cg->fuse();
  for (int c = 0; c < kChunk; ++c) {
    const float *pold = cg->p32[(par + c + 1) & 1];
    float *pnew = cg->p32[(par + c) & 1];
    if (marks) cg->mark(4 * c);
    if (!fused) k_mix_dirvec<<<G, kBlock, 0, s>>>(c, cg->n, pold, cg->r32, pnew, cg->pA, cg->st, cg->ms);
    if (marks) cg->mark(4 * c + 1);
    if (fused)
      FFHIP_LAUNCH_ROWS(cg, k_mix_dir_matvec, G, s, c, M32, pold, cg->r32, pnew, cg->q32, cg->pA, cg->pB, cg->st,
                       cg->ms);
    else
      FFHIP_LAUNCH_FMT(cg, k_mix_matvec, G, s, M32, pnew, cg->q32, cg->pB, cg->st);
    if (marks) cg->mark(4 * c + 2);
    k_mix_update<<<G, kBlock, 0, s>>>(c, cg->n, pnew, cg->q32, cg->y32, cg->r32, cg->pB, cg->pA,
                                      cg->st, cg->ms);
    if (marks) cg->mark(4 * c + 3);
  }
  k_cg_advance<<<1, 64, 0, s>>>(cg->st, kChunk, cg->host_state());
}

static hipGraphExec_t pcg_chunk_graph(ffhip_cg cg, const double *sval, bool sym) {
  return cg->graph(sym ? 2 : 0, sval, 1, [&] { launch_pcg_chunk(cg, sval, sym, false); });
}

// The symmetric values of a solver in its kSymAfter-th iteration of a solve; true
// when they are there.  The search and the copy cost 0.2 to 0.6 ms (cube(96),
// cube(160)) and give 6 to 23 us an iteration: worth it in a solve that has run
// a while, for a matrix past kSymMinBytes (cube(64), 39 MB, would gain 2 us an
// iteration for 0.15 ms).  A matrix of another form is seen as one within the
// search's first blocks, once per solver; values that are not symmetric, or no
// room for the copy, count until the values change.
constexpr int kSymAfter = 4 * kChunk;
constexpr int64_t kSymMinBytes = 64000000;
static bool sym_build(ffhip_cg cg) {
  if (cg->sym != cg->kSymUnknown) return cg->sym == cg->kSymThere;
  ffhip_ctx ctx = cg->ctx;
  hipStream_t s = ctx->stream;
  const int64_t n = cg->n;
  cg->sym = cg->kSymNever;
  // 32-bit byte offsets of the values
  if (cg->fmt != kSell16 || cg->mode != FFHIP_CG_FP64 || cg->matrix_bytes(8) <= kSymMinBytes ||
      cg->S * (kSymHalf * kSlice * 8) >= (int64_t)UINT32_MAX)
    return false;
  SymTables *T = nullptr;
  uint32_t *owners = nullptr;
  const MatFmt<double> M = cg->fmt_of(cg->sval);
  int end[4] = {1, 0, 0, 0};  // SymTables' bad, count, nl, nu
  try {
    T = dalloc<SymTables>(1);
    owners = dalloc<uint32_t>(n);
    if (!cg->symcls) cg->symcls = dalloc<uint8_t>(n);
    if (!cg->symtab) cg->symtab = dalloc<SymPattern>(kSymSlots);
    clear(ctx, {{T, sizeof(SymTables)}});
    k_sym_rows<<<nblk(n, 256), 256, 0, s>>>(M, T, cg->symcls, owners);
    k_sym_table<<<1, kSymSlots, 0, s>>>(M, T, owners, cg->symtab);
    FFHIP_CHECK(hipGetLastError());
    fetch(ctx, {{end, &T->bad, sizeof(end)}});
    if (!end[0]) {
      cg->sym_nl = end[2];
      cg->sym_nu = end[2] <= 3 && end[3] <= 4 ? 4 : kSymHalf;
      if (!cg->symval) cg->symval = dalloc<double>(cg->S * cg->sym_nu * kSlice);
      k_sym_fill<<<nblk(n, 256), 256, 0, s>>>(M, T, cg->symcls, owners, cg->sym_nu, cg->symval);
      FFHIP_CHECK(hipGetLastError());
      fetch(ctx, {{end, &T->bad, sizeof(end)}});
    }
  } catch (const Error &) {  // no room for them: the solve goes on without
    (void)hipStreamSynchronize(s);
    end[0] = kSymValues;
  }
  dfree(T);
  dfree(owners);
  if (end[0]) {
    cg->sym = end[0] & kSymForm ? cg->kSymNever : cg->kSymNot;
    // the captured chunks that read the buffers go with them
    auto gone = std::remove_if(cg->graphs.begin(), cg->graphs.end(), [](const ffhip_cg_s::Chunk &c) {
      if (c.kind == 2) (void)hipGraphExecDestroy(c.exec);
      return c.kind == 2;
    });
    cg->graphs.erase(gone, cg->graphs.end());
    dfree(cg->symval);
    dfree(cg->symcls);
    dfree(cg->symtab);
    return false;
  }
  cg->sym = cg->kSymThere;
  return true;
}
static hipGraphExec_t mix_chunk_graph(ffhip_cg cg, const float *sval32, int par) {
  return cg->graph(1, sval32, par, [&] { launch_mix_chunk(cg, sval32, par, false); });
}

// FP32 Jacobi-scaled CG with FP64 reliable updates (see the file comment).
int ffhip_cg_solve_mixed(ffhip_cg cg, const double *sval, const float *sval32, double eps,
                         int itmax, CgState &hs) {
  ffhip_ctx ctx = cg->ctx;
  hipStream_t s = ctx->stream;
  const int64_t n = cg->n;
  const int G = cg->grid;
  const int chunk = kChunk;
  hipGraphExec_t gx[2] = {mix_chunk_graph(cg, sval32, 0), mix_chunk_graph(cg, sval32, 1)};
  clear(ctx, {{cg->p32[0], 4 * (size_t)n}, {cg->p32[1], 4 * (size_t)n}, {cg->y32, 4 * (size_t)n}});
  memset(&hs, 0, sizeof(hs));
  MixState hm;
  memset(&hm, 0, sizeof(hm));
  double gcg = mix_residual(cg, sval);
  hs.refinements = 1;
  hs.gcg0 = gcg;
  hs.eps2 = eps > 0 ? eps * eps * gcg : eps * eps;
  if (gcg != gcg) { hs.done = 4; return 0; }
  if (gcg < 1e-30) { hs.done = 2; return 0; }
  double sigma = std::sqrt(gcg);
  double rho_last = 0.;
  int it = 1;
  hm.cbeta = 0.;
  hm.first_it = 1;
  for (;;) {
    // (re)start the FP32 recurrence from the FP64 residual
    k_mix_rescale<<<G, kBlock, 0, s>>>(n, 1. / sigma, cg->dsc, cg->G, cg->r32, cg->pA);
    hs.sigma = sigma;
    hs.need_update = 0;
    hs.iters = it - 1;
    hs.it0 = it;
    hs.itmax = itmax;
    hs.eps = eps;
    k_put<<<1, 1, 0, s>>>(cg->st, hs);
    k_put<<<1, 1, 0, s>>>(cg->ms, hm);
    cg->ensure_events(4 * chunk);
    const int par = it & 1;
    for (;;) {
      const int it0 = it;
      if (gx[par]) FFHIP_CHECK(hipGraphLaunch(gx[par], s));
      else launch_mix_chunk(cg, sval32, par, cg->profile != 0);
      it += chunk;
      FFHIP_CHECK(hipGetLastError());
      FFHIP_CHECK(hipStreamSynchronize(s));
      hs = *cg->host_state();
      cg->collect(it0, chunk, hs.iters);
      if (hs.done || hs.need_update) break;
    }
    if (hs.done) {  // NaN or itmax: fold what we have
      k_mix_fold<<<nblk(n, 256), 256, 0, s>>>(n, sigma, cg->dsc, cg->y32, cg->xw);
      return 0;
    }
    // reliable update: fold, recompute the FP64 residual, accept or rescale
    if (hs.iters + 1 == hm.first_it && hs.refinements > 1) {  // no inner progress since the last update
      hs.done = 3;
      k_mix_fold<<<nblk(n, 256), 256, 0, s>>>(n, sigma, cg->dsc, cg->y32, cg->xw);
      return 0;
    }
    it = hs.iters + 1;
    rho_last = hs.rho32;
    k_mix_fold<<<nblk(n, 256), 256, 0, s>>>(n, sigma, cg->dsc, cg->y32, cg->xw);
    gcg = mix_residual(cg, sval);
    hs.refinements += 1;
    if (gcg != gcg) { hs.done = 4; return 0; }
    if (gcg < hs.eps2) { hs.done = 1; return 0; }
    if (it - 1 >= itmax) { hs.done = 3; return 0; }
    const double sig_new = std::sqrt(gcg);
    // p_true = r_true + beta p_true_old, beta = gcg / (rho_last sigma^2), in units of sig_new
    hm.cbeta = (gcg / (rho_last * sigma * sigma)) * (sigma / sig_new);
    hm.first_it = it;
    sigma = sig_new;
  }
}

// the figures of a finished solve for the caller, and the errors of one that
// did not converge (res: the sums of k_residual)
static void solve_result(ffhip_cg cg, const CgState &hs, const double res[3], double ms, int itmax,
                         int half_from, bool small, ffhip_cg_stats *stats) {
  if (stats) {
    stats->iters = hs.iters;
    stats->converged = hs.done == 1 ? 1 : (hs.done == 2 ? 2 : 0);
    stats->refinements = hs.refinements;
    stats->half_from = half_from;
    stats->gcg0 = hs.gcg0;
    stats->gcg = cg->mode == FFHIP_CG_FP64 ? hs.gcg_prev[(hs.iters + 1) & 1] : res[2];
    stats->true_gcg = res[2];
    stats->true_relres = res[1] > 0 ? std::sqrt(res[0] / res[1]) : std::sqrt(res[0]);
    stats->ms_solve = ms;
    stats->timed = cg->n_timed;
    stats->ms_matvec_avg = cg->n_timed ? cg->t_mv / cg->n_timed : 0.;
    stats->ms_update_avg = cg->n_timed ? cg->t_up / cg->n_timed : 0.;
    stats->fused = small ? 0 : cg->fuse();
    stats->ms_direction_avg = cg->n_timed ? cg->t_dv / cg->n_timed : 0.;
  }
  FFHIP_REQUIRE(hs.done != 4, FFHIP_ERR_NAN, "ffhip_cg_solve: NaN in CG (bad matrix)");
  FFHIP_REQUIRE(hs.done != 3, FFHIP_ERR_NOCONV,
                "ffhip_cg_solve: ConjugueGradient did not converge in %d iterations", itmax);
}

// Systems that k_pcg_small solves: FP64 in the 16-bit sliced layout up to
// kSmallRows rows, in CSR (taken where slices would pad) up to kSmallRowsCsr,
// unless kernel-by-kernel launches are asked for.  One CU reads the matrix at
// about 64 bytes a cycle: past 2^16 entries (the 4096 rows of a P1 cube) the
// launches win.  The iteration cap bounds the one launch.
static bool pcg_small(ffhip_cg cg, int itmax) {
  const bool fits = (cg->fmt == kSell16 && cg->n <= kSmallRows) || (cg->fmt == kCsrV && cg->n <= kSmallRowsCsr);
  return cg->mode == FFHIP_CG_FP64 && fits && cg->ents <= 1 << 16 && cg->grid <= kSmallBlocks &&
         cg->use_graph && !cg->profile && itmax <= 65536;
}
static void pcg_solve_small(ffhip_cg cg, const double *b, double *x, int on_device, const double *sval,
                            double eps, int itmax, double tgv, ffhip_cg_stats *stats) {
  ffhip_ctx ctx = cg->ctx;
  hipStream_t s = ctx->stream;
  const int64_t n = cg->n;
  const double *bd = b;
  double *xd = x;
  if (!on_device) {
    FFHIP_CHECK(hipMemcpyAsync(cg->bw, b, 8 * n, hipMemcpyHostToDevice, s));
    FFHIP_CHECK(hipMemcpyAsync(cg->xw, x, 8 * n, hipMemcpyHostToDevice, s));
    bd = cg->bw;
    xd = cg->xw;
  }
  static_assert(sizeof(SmallOut) <= ffhip_ctx_s::kPinnedData, "page-locked read-back");
  SmallOut *out = static_cast<SmallOut *>(ctx->pinned_data());
  memset(out, 0, sizeof(*out));
  const int G = cg->grid;
  ctx->tic();
  const auto kernel = cg->fmt == kCsrV ? k_pcg_small<kCsrV, 1>
                      : G <= 4         ? k_pcg_small<kSell16, 1>
                                       : k_pcg_small<kSell16, kSmallBlocks / 4>;
  kernel<<<1, kBlock * std::min(G, 4), 0, s>>>(cg->fmt_of(sval), G, bd, xd, cg->dinv,
                                               cg->ntgv > 0 ? cg->wcl : nullptr, tgv, eps, itmax, out);
  FFHIP_CHECK(hipGetLastError());
  ctx->toc();
  if (!on_device) {
    FFHIP_CHECK(hipMemcpyAsync(x, cg->xw, 8 * n, hipMemcpyDeviceToHost, s));
    FFHIP_CHECK(hipStreamSynchronize(s));
  }
  double res[3] = {0., 0., 0.};
  for (int i = 0; i < G; ++i)
    for (int c = 0; c < 3; ++c) res[c] += out->res[3 * i + c];
  cg->t_dv = cg->t_mv = cg->t_up = 0.;
  cg->n_timed = 0;
  solve_result(cg, out->st, res, ctx->last_ms, itmax, 0, true, stats);
}

static void cg_release(ffhip_cg cg) {
  for (hipEvent_t e : cg->ev) (void)hipEventDestroy(e);
  for (auto &g : cg->graphs) (void)hipGraphExecDestroy(g.exec);
  if (cg->fmt == kCsrV) cg->sval = nullptr;  // A's array
  dfree(cg->sptr); dfree(cg->slen); dfree(cg->scol); dfree(cg->scol16); dfree(cg->sptr16); dfree(cg->bcol); dfree(cg->bperm); dfree(cg->bwave); dfree(cg->sval); dfree(cg->rb);
  dfree(cg->svalT);
  dfree(cg->sval32); dfree(cg->sval32T); dfree(cg->dinv); dfree(cg->dsc); dfree(cg->wcl);
  dfree(cg->xw); dfree(cg->bw); dfree(cg->G); dfree(cg->CG); dfree(cg->H[0]); dfree(cg->H[1]);
  dfree(cg->AH); dfree(cg->r32); dfree(cg->q32); dfree(cg->y32); dfree(cg->p32[0]);
  dfree(cg->p32[1]); dfree(cg->pA); dfree(cg->pB); dfree(cg->st); dfree(cg->ms);
  dfree(cg->st2);
  dfree(cg->symval); dfree(cg->symcls); dfree(cg->symtab);
  for (double *&p : cg->gmV) dfree(p);
  for (double *&p : cg->gmVp) dfree(p);
  dfree(cg->gmVDev); dfree(cg->gmVpDev); dfree(cg->gmW); dfree(cg->gmX0); dfree(cg->gmY);
  dfree(cg->gmS); dfree(cg->gmL); dfree(cg->gmOut);
  if (cg->gmOutH) (void)hipHostFree(cg->gmOutH);
  delete cg;
}

extern "C" {

int ffhip_cg_create(ffhip_ctx ctx, ffhip_mat A, int mode, ffhip_cg *out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && A && out, FFHIP_ERR_ARG, "ffhip_cg_create: null argument");
    FFHIP_REQUIRE(!A->half, FFHIP_ERR_UNSUPPORTED,
                  "ffhip_cg_create: a half (sym=1) matrix; expand it with ffhip_mat_full");
    const int prec = mode & 0xf, layout = mode & 0x130;
    const bool index32 = (mode & FFHIP_CG_INDEX32) != 0;
    FFHIP_REQUIRE((prec == FFHIP_CG_FP64 || prec == FFHIP_CG_MIXED) &&
                      (mode & ~(0x13f | FFHIP_CG_INDEX32 | FFHIP_CG_EAGER)) == 0 &&
                      (layout == 0 || layout == FFHIP_CG_LAYOUT_SELL || layout == FFHIP_CG_LAYOUT_CSR ||
                       layout == FFHIP_CG_LAYOUT_BSR3),
                  FFHIP_ERR_ARG, "ffhip_cg_create: mode %d", mode);
    ffhip_cg cg = new ffhip_cg_s();
    cg->ctx = ctx; cg->A = A; cg->mode = prec; cg->n = A->n;
    cg->use_graph = (mode & FFHIP_CG_EAGER) ? 0 : 1;
    try {
      const int64_t n = A->n;
      cg->dinv = dalloc<double>(n);
      cg->dsc = dalloc<double>(n);
      cg->wcl = dalloc<uint8_t>(n);
      cg->rb = dalloc<SetupRb>(1);
      if (prec == FFHIP_CG_MIXED) {  // the FP32 fill scales by the Jacobi diagonal
        cg_setup_jacobi(cg);
        cg_plan_layout(cg, layout, index32);  // reads the tgv figures back with its sizes
        cg_fill_values(cg, false);
      } else {  // FP64: the Jacobi set-up after the layout, from the fill's diagonal on sliced ELL
        clear(ctx, {{cg->rb, sizeof(SetupRb)}});
        cg_plan_layout(cg, layout, index32);
        Arena ar(ctx, DiagBufs::bytes(n));
        const DiagBufs b(ar, n);
        const bool in_fill = cg->fmt == kSell || cg->fmt == kSell16;
        if (!in_fill) {
          k_diag_vals<<<nblk(n, 256), 256, 0, ctx->stream>>>(n, A->diag, A->vals, b.d, b.has);
          cg_jacobi_tail(cg, b);
        }
        cg_fill_values(cg, false, in_fill ? &b : nullptr, true);
      }
      cg->xw = dalloc<double>(n); cg->bw = dalloc<double>(n);
      cg->G = dalloc<double>(n); cg->CG = dalloc<double>(n);
      cg->H[0] = dalloc<double>(n); cg->H[1] = dalloc<double>(n);
      cg->AH = dalloc<double>(n);
      if (prec == FFHIP_CG_MIXED) {
        cg->r32 = dalloc<float>(n); cg->q32 = dalloc<float>(n); cg->y32 = dalloc<float>(n);
        cg->p32[0] = dalloc<float>(n); cg->p32[1] = dalloc<float>(n);
      }
      cg->pA = dalloc<double>(3 * (int64_t)cg->grid);
      cg->pB = dalloc<double>(3 * (int64_t)cg->grid);
      cg->st = dalloc<CgState>(1);
      cg->ms = dalloc<MixState>(1);
      cg->st2 = dalloc<Cg2State>(1);
    } catch (...) {
      (void)hipStreamSynchronize(ctx->stream);
      cg_release(cg);
      throw;
    }
    *out = cg;
  });
}

int ffhip_cg_layout(ffhip_cg cg, int *layout, int64_t *entries) {
  return guard([&] {
    FFHIP_REQUIRE(cg, FFHIP_ERR_ARG, "ffhip_cg_layout: null solver");
    if (layout)
      *layout = cg->fmt == kCsrV    ? FFHIP_CG_LAYOUT_CSR
                : cg->fmt == kBsr3 ? FFHIP_CG_LAYOUT_BSR3
                                   : (FFHIP_CG_LAYOUT_SELL | (cg->fmt == kSell16 ? FFHIP_CG_INDEX16 : 0));
    if (entries) *entries = cg->fmt == kBsr3 ? 9 * cg->ents : cg->ents;
  });
}

int ffhip_cg_update_values(ffhip_cg cg) {
  return guard([&] {
    FFHIP_REQUIRE(cg, FFHIP_ERR_ARG, "ffhip_cg_update_values: null solver");
    if (cg->sym != cg->kSymNever) cg->sym = cg->kSymUnknown;
    cg_setup_jacobi(cg);
    setup_readback(cg);
    cg_fill_values(cg, false);
    if (cg->svalT) cg_fill_values(cg, true);
  });
}

int ffhip_cg_solve(ffhip_cg cg, const double *b, double *x, int on_device, double eps, int itmax,
                   double tgv, int trans, ffhip_cg_stats *stats) {
  return guard([&] {
    FFHIP_REQUIRE(cg && b && x, FFHIP_ERR_ARG, "ffhip_cg_solve: null argument");
    ffhip_ctx ctx = cg->ctx;
    hipStream_t s = ctx->stream;
    const int64_t n = cg->n;
    if (trans && !cg->svalT) cg_fill_values(cg, true);
    const double *sval = trans ? cg->svalT : cg->sval;
    const float *sval32 = trans ? cg->sval32T : cg->sval32;
    if (itmax <= 0) itmax = (int)n;  // SolverCG(ds): itmax > 0 ? itmax : n
    if (pcg_small(cg, itmax)) {
      pcg_solve_small(cg, b, x, on_device, sval, eps, itmax, tgv, stats);
      return;
    }
    // captured before this solve's first launch (kept for later solves)
    if (cg->mode == FFHIP_CG_FP64) (void)pcg_chunk_graph(cg, sval, !trans && cg->sym == cg->kSymThere);
    else { (void)mix_chunk_graph(cg, sval32, 0); (void)mix_chunk_graph(cg, sval32, 1); }
    FFHIP_CHECK(hipMemcpyAsync(cg->bw, b, 8 * n, on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, s));
    FFHIP_CHECK(hipMemcpyAsync(cg->xw, x, 8 * n, on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, s));
    ctx->tic();
    if (cg->ntgv > 0) k_init_bc<<<nblk(n, 256), 256, 0, s>>>(n, cg->wcl, cg->bw, tgv, cg->xw);
    CgState hs;
    int half_from = 0;
    memset(&hs, 0, sizeof(hs));
    cg->t_dv = cg->t_mv = cg->t_up = 0.;
    cg->n_timed = 0;
    if (cg->mode == FFHIP_CG_FP64) {
      const int G = cg->grid;
      const MatFmt<double> M = cg->fmt_of(sval);
      const int chunk = kChunk;
      bool sym = !trans && cg->sym == cg->kSymThere;
      half_from = sym ? 1 : 0;
      hipGraphExec_t gx = pcg_chunk_graph(cg, sval, sym);
      hs.it0 = 1;
      hs.itmax = itmax;
      hs.eps = eps;
      k_put<<<1, 1, 0, s>>>(cg->st, hs);
      FFHIP_LAUNCH_FMT(cg, k_pcg_init, G, s, M, cg->xw, cg->bw, cg->dinv, cg->G, cg->CG, cg->H[0],
                       cg->pA, cg->st);
      FFHIP_CHECK(hipGetLastError());
      cg->ensure_events(4 * chunk);
      for (int it = 1;; it += chunk) {
        if (gx) FFHIP_CHECK(hipGraphLaunch(gx, s));
        else launch_pcg_chunk(cg, sval, sym, cg->profile != 0);
        FFHIP_CHECK(hipGetLastError());
        FFHIP_CHECK(hipStreamSynchronize(s));
        hs = *cg->host_state();
        cg->collect(it, chunk, hs.done ? hs.iters : it + chunk - 1);
        if (hs.done) break;
        if (!sym && !trans && it + chunk > kSymAfter && sym_build(cg)) {
          sym = true;
          half_from = it + chunk;
          gx = pcg_chunk_graph(cg, sval, sym);
        }
      }
    } else {
      ffhip_cg_solve_mixed(cg, sval, sval32, eps, itmax, hs);
    }
    ctx->toc();
    const double ms = ctx->last_ms;
    double res[3];
    residual_sums(cg, sval, cg->xw, cg->bw, nullptr, res);
    FFHIP_CHECK(hipMemcpyAsync(x, cg->xw, 8 * n, on_device ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, s));
    FFHIP_CHECK(hipStreamSynchronize(s));
    solve_result(cg, hs, res, ms, itmax, half_from, false, stats);
  });
}

int ffhip_cg_solve_affine(ffhip_cg cg, const double *b, double *x, int on_device, double eps,
                          int itmax, int precon, double *eps_out, ffhip_cg_stats *stats) {
  return guard([&] {
    FFHIP_REQUIRE(cg && x, FFHIP_ERR_ARG, "ffhip_cg_solve_affine: null argument");
    FFHIP_REQUIRE(precon == FFHIP_CG2_IDENTITY || precon == FFHIP_CG2_JACOBI, FFHIP_ERR_ARG,
                  "ffhip_cg_solve_affine: precon %d", precon);
    FFHIP_REQUIRE(itmax >= 0, FFHIP_ERR_ARG, "ffhip_cg_solve_affine: nbiter %d", itmax);
    ffhip_ctx ctx = cg->ctx;
    hipStream_t s = ctx->stream;
    const int64_t n = cg->n;
    const hipMemcpyKind kin = on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
    if (b) FFHIP_CHECK(hipMemcpyAsync(cg->bw, b, 8 * n, kin, s));
    FFHIP_CHECK(hipMemcpyAsync(cg->xw, x, 8 * n, kin, s));
    const double *bd = b ? cg->bw : nullptr;
    const double *dinv = precon == FFHIP_CG2_JACOBI ? cg->dinv : nullptr;
    double *h = cg->H[0];
    const int G = cg->grid;
    const MatFmt<double> M = cg->fmt_of(cg->sval);
    ctx->tic();
    FFHIP_LAUNCH_FMT(cg, k_cg2_init, G, s, M, cg->xw, bd, dinv, cg->G, cg->CG, h, cg->pA, cg->st2);
    FFHIP_CHECK(hipGetLastError());
    Cg2State hs;
    const int chunk = 16;
    for (int it = 0;; ++it) {
      k_cg2_step<<<G, kBlock, 0, s>>>(it, itmax, eps, n, h, cg->CG, cg->xw, cg->pA, cg->st2);
      FFHIP_LAUNCH_FMT(cg, k_cg2_dir, G, s, M, cg->xw, bd, cg->G, h, cg->AH, cg->pB, cg->st2);
      k_cg2_update<<<G, kBlock, 0, s>>>(it, n, h, cg->AH, dinv, cg->xw, cg->G, cg->CG, cg->pB,
                                        cg->pA, cg->st2);
      if ((it + 1) % chunk == 0) {
        FFHIP_CHECK(hipGetLastError());
        fetch(ctx, {{&hs, cg->st2, sizeof(hs)}});
        if (hs.done) break;
      }
    }
    ctx->toc();
    const double ms = ctx->last_ms;
    double res[3] = {0., 0., 0.};
    if (!b) FFHIP_CHECK(hipMemsetAsync(cg->bw, 0, 8 * n, s));
    residual_sums(cg, cg->sval, cg->xw, cg->bw, nullptr, res);
    FFHIP_CHECK(hipMemcpyAsync(x, cg->xw, 8 * n, on_device ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, s));
    FFHIP_CHECK(hipStreamSynchronize(s));
    if (eps_out) *eps_out = hs.done == 2 ? eps : hs.reps2;
    if (stats) {
      memset(stats, 0, sizeof(*stats));
      stats->iters = hs.iters;
      stats->converged = hs.done == 1 ? 1 : (hs.done == 2 ? 2 : 0);
      stats->refinements = 0;
      stats->gcg0 = hs.g20;
      stats->gcg = hs.g2last;
      stats->true_gcg = dinv ? res[2] : res[0];
      stats->true_relres = res[1] > 0 ? std::sqrt(res[0] / res[1]) : std::sqrt(res[0]);
      stats->ms_solve = ms;
    }
    FFHIP_REQUIRE(hs.done != 5, FFHIP_ERR_NAN, "CG2: Matrix is not defined (/0), sorry");
    FFHIP_REQUIRE(hs.done != 6, FFHIP_ERR_NAN, "CG2: Bug : ro is NaN");
  });
}

int ffhip_gmres_solve(ffhip_cg cg, const double *b, double *x, int on_device, double eps,
                      int itmax, int restart, double tgv, int trans, ffhip_cg_stats *stats) {
  return guard([&] {
    FFHIP_REQUIRE(cg && b && x, FFHIP_ERR_ARG, "ffhip_gmres_solve: null argument");
    FFHIP_REQUIRE(restart >= 1, FFHIP_ERR_ARG, "ffhip_gmres_solve: restart %d", restart);
    ffhip_ctx ctx = cg->ctx;
    hipStream_t s = ctx->stream;
    const int64_t n = cg->n;
    const int G = cg->grid, m = restart;
    if (trans && !cg->svalT) cg_fill_values(cg, true);
    const double *sval = trans ? cg->svalT : cg->sval;
    const MatFmt<double> M = cg->fmt_of(sval);
    const hipMemcpyKind kin = on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
    cg->gm_basis(1, 1);
    FFHIP_CHECK(hipMemcpyAsync(cg->bw, b, 8 * n, kin, s));
    FFHIP_CHECK(hipMemcpyAsync(cg->xw, x, 8 * n, kin, s));
    std::vector<double> part(G);
    // block partials written by the last kernel, added on the host in block order
    auto host_sum = [&](const double *p) {
      FFHIP_CHECK(hipMemcpyAsync(part.data(), p, 8 * G, hipMemcpyDeviceToHost, s));
      FFHIP_CHECK(hipStreamSynchronize(s));
      double t = 0.;
      for (int i = 0; i < G; ++i) t += part[i];
      return t;
    };
    ctx->tic();
    if (cg->ntgv > 0) k_init_bc<<<nblk(n, 256), 256, 0, s>>>(n, cg->wcl, cg->bw, tgv, cg->xw);
    const int nbitermx = itmax > 0 ? itmax : (int)n;  // SolverGMRES(ds)
    // fgmres (CG.cpp:347-517) with leftC = 0: the scalar part as the reference's
    std::vector<double> rot0(m + 2), rot1(m + 2), g(m + 1), g1(m + 1), y(m + 1);
    // (m + 2) x (m + 1), zero; calloc leaves the pages that are never reached
    // untouched (8 MB for the default restart of 1000)
    const std::unique_ptr<double, decltype(&std::free)> Hn(
        (double *)std::calloc((size_t)(m + 2) * (m + 1), sizeof(double)), &std::free);
    FFHIP_REQUIRE(Hn, FFHIP_ERR_INTERNAL, "ffhip_gmres_solve: out of memory for restart %d", m);
    auto HN = [&](int i, int j) -> double & { return Hn.get()[(size_t)i * (m + 1) + j]; };
    k_gm_normb<<<G, kBlock, 0, s>>>(n, cg->bw, cg->ntgv > 0 ? cg->wcl : nullptr, cg->pA);
    double normb = std::sqrt(host_sum(cg->pA));
    double relres = 1e100, rate = std::log(10.);  // decrease per iteration (log), first a fast solve's
    bool noconv = true;
    int iter = 0, nrestart = 0;
    while (noconv) {
      FFHIP_CHECK(hipMemcpyAsync(cg->gmX0, cg->xw, 8 * n, hipMemcpyDeviceToDevice, s));
      FFHIP_LAUNCH_FMT(cg, k_gm_residual, G, s, M, cg->xw, cg->bw, cg->gmW, cg->pA);
      FFHIP_CHECK(hipGetLastError());
      g[0] = std::sqrt(host_sum(cg->pA));
      if (normb < 1.e-20 || eps < 0) normb = 1.;
      double inv = 1. / g[0];
      const double g0 = g[0];
      int it, ahead = 0;  // iterations launched beyond the ones looked at, of the current batch
      int batch = 0;
      const int P = cg->gm_blocks();
      const int64_t rows = (n + P - 1) / P;
      for (it = 0; it < m; it++, iter++) {
        if (ahead == 0) {
          // a batch of iterations in one go, then one copy of what the host
          // needs of each; those after a convergence are dropped, so a batch is
          // no longer than the rest at the rate so far.  (8 from the start, 1000
          // to 227 k rows: 355 to 465 us for a solve of one iteration that took 285.)
          // Past 2^18 rows an iteration costs more than the wait it saves.
          if (it > 0) rate = std::fmax(std::log(std::fabs(g0) / relres) / it, 0.);
          const double left = std::ceil(std::log((it ? relres : std::fabs(g0)) / (std::fabs(eps) * normb)) / rate);
          const int most = n <= (1 << 18) ? ffhip_cg_s::kGmBatch : 1;
          batch = std::min(!(left > 1.) ? 1 : left < most ? (int)left : most, m - it);  // left may be NaN
          cg->gm_basis(it + 1, it + batch);
          batch = std::min(batch, (int)cg->gmV.size() - it);
          const int64_t ld = cg->gm_out();
          for (int c = 0; c < batch; ++c) {
            const int j = it + c;
            double *out = cg->gmOut + c * ld, *norms = out + cg->gmCap;
            const double *pin = c ? cg->gmOut + (c - 1) * ld + cg->gmCap : nullptr;
            k_gm_prec<<<G, kBlock, 0, s>>>(n, inv, pin, cg->gmW, cg->dinv, cg->gmV[j], cg->gmVp[j]);
            FFHIP_LAUNCH_FMT(cg, k_gm_matvec, G, s, M, cg->gmVp[j], cg->gmW);
            const int share = std::max(1, std::min((j + kWavesPerBlock) / kWavesPerBlock, 2048 / P));
            k_gm_dots<<<dim3(P, share), kBlock, 0, s>>>(j, n, rows, cg->gmVDev, cg->gmW, cg->gmS);
            k_gm_coefs<<<1, kGmBlock, 0, s>>>(j, P, cg->gmS, cg->gmL, out);
            k_gm_project<<<G, kBlock, 0, s>>>(j, n, cg->gmVDev, out, cg->gmW, norms);
          }
          FFHIP_CHECK(hipGetLastError());
          FFHIP_CHECK(hipMemcpyAsync(cg->gmOutH, cg->gmOut, 8 * batch * ld, hipMemcpyDeviceToHost, s));
          FFHIP_CHECK(hipStreamSynchronize(s));
          ahead = batch;
        }
        const double *hc = cg->gmOutH + (batch - ahead) * cg->gm_out(), *wp = hc + cg->gmCap;
        --ahead;
        double ww = 0.;
        for (int i = 0; i < G; ++i) ww += wp[i];
        for (int i = 0; i <= it; ++i) HN(i, it) = hc[i];
        const double aux = HN(it + 1, it) = std::sqrt(ww);
        inv = 1. / aux;
        for (int i = 0; i < it; i++) {
          const double aa = rot0[i] * HN(i, it) + rot1[i] * HN(i + 1, it);
          const double bb = -rot1[i] * HN(i, it) + rot0[i] * HN(i + 1, it);
          HN(i, it) = aa;
          HN(i + 1, it) = bb;
        }
        const double sq = std::sqrt(HN(it, it) * HN(it, it) + HN(it + 1, it) * HN(it + 1, it));
        rot0[it] = HN(it, it) / sq;
        rot1[it] = HN(it + 1, it) / sq;
        HN(it, it) = rot0[it] * HN(it, it) + rot1[it] * HN(it + 1, it);
        HN(it + 1, it) = 0.;
        g[it + 1] = -rot1[it] * g[it];
        g[it] = rot0[it] * g[it];
        relres = std::fabs(g[it + 1]);
        if (relres / normb < std::fabs(eps)) { noconv = false; break; }
        if (it > nbitermx) break;
      }
      it = std::min(it, m - 1);
      for (int i = it; i >= 0; i--) {  // reconstruction
        g1[i] = g[i];
        for (int j = i + 1; j < it + 1; j++) g1[i] = g1[i] - HN(i, j) * y[j];
        y[i] = g1[i] / HN(i, i);
      }
      FFHIP_CHECK(hipMemcpyAsync(cg->gmY, y.data(), 8 * (it + 1), hipMemcpyHostToDevice, s));
      k_gm_update<<<G, kBlock, 0, s>>>(n, it + 1, cg->gmY, cg->gmVpDev, cg->gmX0, cg->xw);
      FFHIP_CHECK(hipGetLastError());
      if (!noconv) break;
      if (iter > nbitermx) break;
      nrestart++;
    }
    ctx->toc();
    const double ms = ctx->last_ms;
    double res[3];
    residual_sums(cg, sval, cg->xw, cg->bw, nullptr, res);
    FFHIP_CHECK(hipMemcpyAsync(x, cg->xw, 8 * n, on_device ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, s));
    FFHIP_CHECK(hipStreamSynchronize(s));
    if (stats) {
      memset(stats, 0, sizeof(*stats));
      stats->iters = iter;
      stats->converged = noconv ? 0 : 1;
      stats->refinements = nrestart;
      stats->gcg0 = normb;
      stats->gcg = relres / normb;
      stats->true_gcg = res[2];
      stats->true_relres = res[1] > 0 ? std::sqrt(res[0] / res[1]) : std::sqrt(res[0]);
      stats->ms_solve = ms;
    }
    FFHIP_REQUIRE(!noconv, FFHIP_ERR_NOCONV, "ffhip_gmres_solve: fgmres did not converge in %d iterations",
                  iter);
  });
}

int ffhip_cg_set_profiling(ffhip_cg cg, int on) {
  return guard([&] {
    FFHIP_REQUIRE(cg, FFHIP_ERR_ARG, "ffhip_cg_set_profiling: null solver");
    cg->profile = on ? 1 : 0;
  });
}

int ffhip_cg_free(ffhip_cg cg) {
  return guard([&] {
    if (!cg) return;
    (void)hipStreamSynchronize(cg->ctx->stream);
    cg_release(cg);
  });
}

int ffhip_bench_spmv(ffhip_cg cg, int mode, int reps, const void *x, void *y, double *avg_ms) {
  return guard([&] {
    FFHIP_REQUIRE(cg && x && y && avg_ms && reps > 0, FFHIP_ERR_ARG, "ffhip_bench_spmv: bad arguments");
    FFHIP_REQUIRE(mode == FFHIP_CG_FP64 || cg->sval32, FFHIP_ERR_ARG,
                  "ffhip_bench_spmv: FP32 matrix only exists for a MIXED solver");
    ffhip_ctx ctx = cg->ctx;
    hipStream_t s = ctx->stream;
    auto launch = [&] {
      if (mode == FFHIP_CG_FP64) {
        const MatFmt<double> M = cg->fmt_of<double>(cg->sval);
        FFHIP_LAUNCH_MATVEC(cg, double, M, x, y, s);
      } else {
        const MatFmt<float> M = cg->fmt_of<float>(cg->sval32);
        FFHIP_LAUNCH_MATVEC(cg, float, M, x, y, s);
      }
    };
    launch();  // warm
    FFHIP_CHECK(hipGetLastError());
    ctx->tic();
    for (int i = 0; i < reps; ++i) launch();
    FFHIP_CHECK(hipGetLastError());
    ctx->toc();
    *avg_ms = ctx->last_ms / reps;
  });
}

}  // extern "C"
