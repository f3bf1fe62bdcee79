// ffhip_assembly.hip — P1 sparsity pattern, atomic-free assembly, Dirichlet
// rows, right-hand side and CSR mat-vec.
//
// Design (MI355X-first, deterministic):
//   1. dof -> (element, local vertex) incidence lists, sorted by element id:
//      each block counts its items per dof in an LDS hash set and reserves
//      their places in the dofs' 32-entry buckets with one global atomic per
//      dof, a scan gives the list offsets, and every entry goes to its rank
//      among its dof's entries (k_v2e_sort_bucket, or the fused pattern pass
//      of the one-call assembly).  Lists longer than 32: an atomic fill, a
//      bitonic sort of the first 32 in a half-wave, insertion sort beyond.
//   2. pattern: one half-wave per row loads the vertices of the row's
//      incident elements (4 per lane), deduplicates them in an LDS hash set
//      (the lanes step together: no atomics) and orders the unique columns by
//      a counting sort.  One pass writes
//      each row's sorted columns to a row buffer, its length and, for every
//      incidence entry, the offsets of that element's vertices inside the row
//      (the element-to-row map); after a scan of the lengths the buffers are
//      compacted into the CSR arrays.  Rows with more than 32 incident
//      elements use a lane-per-row merge in LDS.
//   3. values: one thread per element evaluates the 14-point Tet_5 integral
//      of kappa and the P1 gradients (VALU FP64) and writes the 4 rows of its
//      symmetric 4x4 matrix where its incidence entries sit in the vertices'
//      lists; then one half-wave per row loads them contiguously (one lane
//      per element) into LDS, and the lane owning each slot adds them in
//      element order.  No atomics: every slot is summed by one lane in
//      element order, the order in which HashMatrix::operator+= accumulates
//      (src/femlib/HashMatrix.cpp:1294-1332).  2D triangles and the rows with
//      more than 32 elements use a lane-per-row walk with the row staged in
//      LDS.
//   4. right-hand sides, the adjoint's M (u - u_d) and CSR products: a pass over
//      the elements leaves each its terms, and a wave per 16 or 64 rows stages
//      the rows' entries in LDS with coalesced loads, added by a lane per row in
//      their order.
#include <hipcub/hipcub.hpp>

#include <cstring>
#include <mutex>
#include <type_traits>
#include <vector>

#include "ffhip_fem.hpp"

namespace ffhip {

// T_5 (src/femlib/QuadratureFormular.cpp:172-186), filled from the host
__constant__ double c_qt5_pts[7][2];
__constant__ double c_qt5_w[7];

// ---------------------------------------------------------------- incidence
__global__ void k_u32_to_i64(int64_t n, const uint32_t *__restrict__ a, int64_t *__restrict__ b) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
  if (i == 0) b[n] = 0;  // the scan's last input
}

__global__ void k_v2e_fill(const int32_t *__restrict__ elems, int64_t m,
                           const int64_t *__restrict__ ptr, int32_t *__restrict__ cur,
                           int32_t *__restrict__ v2e) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  const int32_t v = elems[i];
  const int32_t pos = atomicAdd(&cur[v], 1);
  v2e[ptr[v] + pos] = (int32_t)i;
}

// ---------------------------------------------------------------- half-wave sorting networks
// A 32-lane half of a wave holds one row's list; bitonic compare-exchange
// across lanes (lane xor m, m <= 16, never leaves the half) and inside a lane.
constexpr int kHalf = 32;  // rows of up to 32 incident elements use the half-wave kernels

template <class T>
__device__ inline T tmin(T a, T b) { return a < b ? a : b; }
template <class T>
__device__ inline T tmax(T a, T b) { return a < b ? b : a; }

// one value per lane, sequence index = lane within the half
template <class T>
__device__ inline T bitonic32(T x, int hl) {
#pragma unroll
  for (int k = 2; k <= 32; k <<= 1)
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1) {
      const T p = __shfl_xor(x, j, kWave);
      const bool up = (hl & k) == 0, lower = (hl & j) == 0;
      x = (lower == up) ? tmin(x, p) : tmax(x, p);
    }
  return x;
}

// incidence lists of up to 32 entries sorted into element order, two rows
// per wave; longer lists are left to k_v2e_sort (flagged in *big)
__global__ __launch_bounds__(256) void k_v2e_sort_half(int64_t n, const int64_t *__restrict__ ptr,
                                                       int32_t *__restrict__ v2e, int *__restrict__ big) {
  const int hl = threadIdx.x % kHalf;
  const int64_t v = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kHalf;
  int64_t k0 = 0;
  int deg = 0;
  if (v < n) { k0 = ptr[v]; deg = (int)(ptr[v + 1] - k0); }
  if (deg > kHalf) {
    if (hl == 0) atomicOr(big, 1);
    deg = 0;
  }
  int32_t x = hl < deg ? v2e[k0 + hl] : INT_MAX;
  x = bitonic32(x, hl);
  if (hl < deg) v2e[k0 + hl] = x;
}

// Incidence buckets (up to 32 entries per dof, in no particular order; the
// sort below puts them in element order) with the atomics aggregated per
// block: the block's 256 x kBucketIpt items are counted per dof in an LDS hash set (an
// item's rank among the block's items of its dof from the LDS atomicAdd),
// then each distinct dof of the block reserves its positions with one
// atomicAdd on its global count.
#ifndef FFHIP_BUCKET_IPT
#define FFHIP_BUCKET_IPT 2
#endif
// items per thread (cube(160): 1 -> 2 saves about 0.15 ms of the one-call
// assembly, 4 loses it again)
constexpr int kBucketIpt = FFHIP_BUCKET_IPT;
constexpr int kBucketLog = 9 + (kBucketIpt >= 4 ? 2 : kBucketIpt >= 2 ? 1 : 0);
constexpr int kBucketHash = 1 << kBucketLog;              // >= 2x the items of a block: probing always ends
static_assert(kBucketHash >= 2 * 256 * kBucketIpt, "hash set of twice the block's items");
__global__ __launch_bounds__(256) void k_v2e_bucket_block(const int32_t *__restrict__ elems, int64_t m,
                                                          uint32_t *__restrict__ deg,
                                                          int32_t *__restrict__ bucket,
                                                          int *__restrict__ ovf) {
  __shared__ int32_t hkey[kBucketHash];
  __shared__ uint32_t hcnt[kBucketHash];
  __shared__ uint32_t hbase[kBucketHash];
  const int t = threadIdx.x;
  for (int i = t; i < kBucketHash; i += blockDim.x) { hkey[i] = -1; hcnt[i] = 0; }
  __syncthreads();
  int32_t v[kBucketIpt];
  uint32_t h[kBucketIpt], rank[kBucketIpt];
#pragma unroll
  for (int j = 0; j < kBucketIpt; ++j) {
    const int64_t i = (int64_t)blockIdx.x * (256 * kBucketIpt) + j * 256 + t;
    v[j] = i < m ? elems[i] : -1;
  }
#pragma unroll
  for (int j = 0; j < kBucketIpt; ++j) {
    h[j] = 0;
    rank[j] = 0;
    if (v[j] >= 0) {
      h[j] = ((uint32_t)v[j] * 2654435761u) >> (32 - kBucketLog);
      for (;;) {  // ends: at most half the slots hold keys
        const int32_t old = atomicCAS(&hkey[h[j]], -1, v[j]);
        if (old == -1 || old == v[j]) break;
        h[j] = (h[j] + 1) & (kBucketHash - 1);
      }
      rank[j] = atomicAdd(&hcnt[h[j]], 1u);
    }
  }
  __syncthreads();
  for (int q = t; q < kBucketHash; q += blockDim.x) {
    const int32_t key = hkey[q];
    if (key >= 0) hbase[q] = atomicAdd(&deg[key], hcnt[q]);
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kBucketIpt; ++j) {
    if (v[j] < 0) continue;
    const int64_t i = (int64_t)blockIdx.x * (256 * kBucketIpt) + j * 256 + t;
    const uint32_t pos = hbase[h[j]] + rank[j];
    if (pos < 32) bucket[32 * (int64_t)v[j] + pos] = (int32_t)i;
    else atomicOr(ovf, 1);
  }
}

// bucketed lists (up to 32 entries) put into element order and packed at
// their CSR offsets, two dofs per wave: each entry goes to its rank among
// the dof's entries (distinct items), counted over the bucket staged in LDS
__global__ __launch_bounds__(256) void k_v2e_sort_bucket(int64_t n, const int64_t *__restrict__ ptr,
                                                         const int32_t *__restrict__ bucket,
                                                         int32_t *__restrict__ v2e,
                                                         int32_t *__restrict__ inv) {
  __shared__ __align__(16) int32_t ids[256];
  const int hl = threadIdx.x % kHalf;
  const int64_t v = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kHalf;
  int64_t k0 = 0;
  int deg = 0;
  if (v < n) { k0 = ptr[v]; deg = (int)(ptr[v + 1] - k0); }
  const int32_t x = hl < deg ? bucket[32 * v + hl] : INT_MAX;
  ids[threadIdx.x] = x;
  wave_lds_sync();
  const int4 *row = reinterpret_cast<const int4 *>(ids + (threadIdx.x & ~(kHalf - 1)));
  int rho = 0;
#pragma unroll
  for (int g = 0; g < kHalf / 4; ++g) {
    const int4 w = row[g];
    rho += (w.x < x) + (w.y < x) + (w.z < x) + (w.w < x);
  }
  if (hl < deg) {
    v2e[k0 + rho] = x;
    if (inv) inv[x] = (int32_t)(k0 + rho);
  }
}

// position of every (element, local dof) item in the incidence lists
__global__ void k_v2e_inverse(int64_t m, const int32_t *__restrict__ v2e, int32_t *__restrict__ inv) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < m) inv[v2e[k]] = (int32_t)k;
}

// per-dof insertion sort of the lists longer than 32 entries
__global__ void k_v2e_sort(int64_t n, const int64_t *__restrict__ ptr, int32_t *__restrict__ v2e) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  const int64_t a = ptr[v], b = ptr[v + 1];
  if (b - a <= kHalf) return;
  for (int64_t i = a + 1; i < b; ++i) {
    const int32_t key = v2e[i];
    int64_t j = i - 1;
    while (j >= a && v2e[j] > key) { v2e[j + 1] = v2e[j]; --j; }
    v2e[j + 1] = key;
  }
}

// ---------------------------------------------------------------- pattern (half-wave rows)
// One row per 32-lane half-wave: lane q loads incidence q's element vertices,
// places those other than the row's own in an open-addressing set in LDS (all
// of them step together: read, write where free, read back), the set is
// compacted by ballots and the columns are ordered by a counting sort (rank =
// number of smaller columns).  One pass writes the row length, the sorted
// columns to a 64-entry row buffer, the relative diagonal slot and the
// element-to-row map (each lane kept its columns' slots in the set, which get
// their ranks); after the scan, k_pattern_compact moves the buffered columns to
// their CSR place.  Rows with more than 32 incident elements or 64 columns are
// flagged in big[] for the lane-per-row merge (k_pattern_rows).
constexpr int kRowBuf = 64;

constexpr int kHash = 128;  // LDS hash slots per row (a row has at most 3 * 32 columns besides its own)

// Where the pass writes a row it builds.  Buffered: the 64-entry row
// buffers (rowbuf, rowval), the length and the diagonal offset, moved to CSR
// by k_pattern_compact after the scan of the lengths.  DIRECT: the row
// pointers are known beforehand (the vertex-link counts, k_link_len) and the
// row goes straight to colidx / vals / diag; a row whose length differs from
// its pointers sets *mismatch and is not written (the caller then takes the
// buffered pass).
struct PatternOut {
  int64_t *rowlen = nullptr;
  int32_t *rowbuf = nullptr;
  int8_t *dposr = nullptr;
  double *rowval = nullptr;
  const int64_t *rowptr = nullptr;
  int32_t *colidx = nullptr;
  int64_t *diag = nullptr;
  double *vals = nullptr;
  int *mismatch = nullptr;
};

// VALS (3D P1 stiffness): the same pass also forms the row's values from the
// element scales Ce (the rows of k_p1_values_rows).
//
// With bucket (the incidence lists unsorted, 32 entries per row, every list
// within its bucket; VALS only): each lane ranks its incidence among the
// row's and writes it to v2e at that rank, in place of k_v2e_sort_bucket.
// Bound by its vector instructions (cube(160): 600 per wave, nine tenths of the
// issue slots).  cube(160), 2.84 -> 2.27 ms: an atomic compare-and-swap per
// candidate, an atomic count and a second search per column took 770; a third of
// the rest is the values' geometry and sums.
template <int NLOC, bool VALS, bool DIRECT>
__global__ __launch_bounds__(256) void k_pattern_half(
    int64_t n, const int32_t *__restrict__ elems, const int64_t *__restrict__ v2e_ptr,
    int32_t *__restrict__ v2e, uint32_t *__restrict__ slotmap, uint8_t *__restrict__ big,
    int *__restrict__ any_big, PatternOut out, const double *__restrict__ xyz = nullptr,
    const double *__restrict__ Ce = nullptr, const int32_t *__restrict__ bucket = nullptr) {
  constexpr int NH = 256 / kHalf, R = NLOC - 1, kFree = INT_MAX;
  // every LDS array below is per row (half-wave), so a wave orders its own
  // accesses (wave_lds_sync) and the waves of a block run independently
  __shared__ __align__(16) int32_t hk[NH][kHash];     // open-addressing set of the row's columns but its own
  __shared__ uint8_t hrank[NH][kHash];                // the offset in the row of the column in each set slot
  __shared__ __align__(16) int32_t ucol[NH][kRowBuf];  // the set's columns
  __shared__ uint8_t uslot[NH][kRowBuf];              // and their slots
  // VALS: incidence q's entries at [(column - own - 1) mod 4][q] ([3]: the diagonal),
  // its slot bytes in that order (own first), and for every slot of the row and each
  // of the three the incidences that hold it there
  __shared__ __align__(16) double sv[VALS ? NH : 1][VALS ? 4 * kHalf : 1];
  __shared__ __align__(16) uint32_t so[VALS ? NH : 1][VALS ? kHalf : 1];
  __shared__ uint32_t smask[VALS ? NH : 1][VALS ? 3 : 1][VALS ? kHalf + 1 : 1];
  const int hl = threadIdx.x % kHalf, hid = threadIdx.x / kHalf;
  const bool upper = threadIdx.x % kWave >= kHalf;
  const int64_t v = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kHalf;
  int64_t k0 = 0, p0 = 0, p1 = 0;
  int deg = 0;
  if (v < n) {
    k0 = v2e_ptr[v];
    deg = (int)(v2e_ptr[v + 1] - k0);
    if (DIRECT) { p0 = out.rowptr[v]; p1 = out.rowptr[v + 1]; }
  }
  bool mine = v < n && deg <= kHalf;
  if (!mine) deg = 0;
  // this half's bits of a wave's ballot
  const auto half = [&](bool x) {
    const uint64_t w = __builtin_amdgcn_ballot_w64(x);
    return upper ? (uint32_t)(w >> 32) : (uint32_t)w;
  };
  *reinterpret_cast<int4 *>(&hk[hid][4 * hl]) = make_int4(kFree, kFree, kFree, kFree);
  *reinterpret_cast<int2 *>(&ucol[hid][2 * hl]) = make_int2(kFree, kFree);
  if constexpr (VALS) {
#pragma unroll
    for (int r = 0; r < 3; ++r) smask[hid][r][hl] = 0;
  }
  int32_t c[4] = {kFree, kFree, kFree, kFree};
  int64_t e = 0;
  int lv = 0;
  int32_t idx = kFree;
  int qp = hl;  // the incidence's position in the row's list (element order)
  bool ranked = false;
  if constexpr (VALS) {
    if (bucket) {
      // unsorted bucket: each lane's rank among the row's entries (element
      // ids are distinct) places its incidence, and everything it stores
      // per incidence below, in element order
      idx = hl < deg ? bucket[32 * v + hl] : kFree;
      so[hid][hl] = (uint32_t)idx;
      wave_lds_sync();
      int rho = 0;
#pragma unroll
      for (int g = 0; g < kHalf / 4; ++g) {
        if (__builtin_amdgcn_ballot_w64(deg > 4 * g) == 0) break;
        const uint4 w = *reinterpret_cast<const uint4 *>(&so[hid][4 * g]);
        rho += ((int32_t)w.x < idx) + ((int32_t)w.y < idx) + ((int32_t)w.z < idx) + ((int32_t)w.w < idx);
      }
      if (hl < deg) {
        qp = rho;
        v2e[k0 + qp] = idx;
      }
      ranked = true;
    }
  }
  if (!ranked && hl < deg) idx = v2e[k0 + hl];
  if (hl < deg) {
    e = idx / NLOC;
    lv = idx - (int)e * NLOC;
    if (NLOC == 4) {
      const int4 t = reinterpret_cast<const int4 *>(elems)[e];
      c[0] = t.x; c[1] = t.y; c[2] = t.z; c[3] = t.w;
    } else {
#pragma unroll
      for (int m = 0; m < NLOC; ++m) c[m] = elems[e * NLOC + m];
    }
  }
  // the other vertices, from the one after the row's own on (cyclic)
  int32_t key[R];
  if (NLOC == 4) {
    const int32_t b0 = lv & 1 ? c[1] : c[0], b1 = lv & 1 ? c[2] : c[1], b2 = lv & 1 ? c[3] : c[2],
                  b3 = lv & 1 ? c[0] : c[3];
    key[0] = lv & 2 ? b3 : b1;
    key[1] = lv & 2 ? b0 : b2;
    key[R - 1] = lv & 2 ? b1 : b3;
  } else {
    key[0] = lv == 0 ? c[1] : lv == 1 ? c[2] : c[0];
    key[1] = lv == 0 ? c[2] : lv == 1 ? c[0] : c[1];
  }
  // Equal keys are at the same slot in every step: a slot that was free is
  // written by all of them, and they all see it taken by theirs or by another.
  // Ends: the set holds at most 96 columns of its 128 slots.
  uint32_t slot[R];
  bool open[R];  // still looking (a repeated own vertex is no other column)
#pragma unroll
  for (int r = 0; r < R; ++r) {
    slot[r] = ((uint32_t)__umul24((uint32_t)key[r], 0x9e3779u) >> 17) % kHash;
    open[r] = key[r] != kFree && key[r] != (int32_t)v;
  }
  const auto at = [&](int r) -> int32_t & { return hk[hid][slot[r]]; };
  for (;;) {
    int32_t was[R], is[R];
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < R; ++r) was[r] = __hip_atomic_load(&at(r), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (open[r] && was[r] == kFree)
        __hip_atomic_store(&at(r), key[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    wave_lds_sync();
    bool more = false;
#pragma unroll
    for (int r = 0; r < R; ++r) is[r] = __hip_atomic_load(&at(r), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      open[r] = open[r] && is[r] != key[r];
      if (open[r]) slot[r] = (slot[r] + 1) % kHash;
      more |= open[r];
    }
    if (__builtin_amdgcn_ballot_w64(more) == 0) break;
  }
  // compaction: lane hl's four slots
  int nset = 0;  // columns in the set
  {
    const int4 w = *reinterpret_cast<const int4 *>(&hk[hid][4 * hl]);
    const int32_t k4[4] = {w.x, w.y, w.z, w.w};
    const uint32_t below = (1u << hl) - 1;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool full = k4[j] != kFree;
      const uint32_t mk = half(full);
      const int at_ = nset + __builtin_popcount(mk & below);
      if (full && at_ < kRowBuf) {
        ucol[hid][at_] = k4[j];
        uslot[hid][at_] = (uint8_t)(4 * hl + j);
      }
      nset += __builtin_popcount(mk);
    }
  }
  wave_lds_sync();
  const int len = nset + (deg > 0);  // and the row's own column
  if (len > kRowBuf) mine = false;
  const bool wrong = DIRECT && mine && p1 - p0 != len;  // the row's length is not its pointers'
  const bool write = mine && !wrong;
  // counting sort: the rank of a column is the number of smaller columns
  int dpos = 0;
#pragma unroll
  for (int h2 = 0; h2 < 2; ++h2) {
    const int j = hl + h2 * kHalf;
    if (h2 == 1 && __builtin_amdgcn_ballot_w64(mine && nset > kHalf) == 0) break;
    const bool on = mine && j < nset;
    const int32_t u = on ? ucol[hid][j] : kFree;
    const bool less = u < (int32_t)v;  // before the row's own column
    int rk = less ? 0 : 1;
    for (int g = 0; __builtin_amdgcn_ballot_w64(on && 4 * g < nset); ++g) {  // past nset: kFree
      const int4 w = *reinterpret_cast<const int4 *>(&ucol[hid][(4 * g) % kRowBuf]);
      rk += (w.x < u) + (w.y < u) + (w.z < u) + (w.w < u);
    }
    dpos += __builtin_popcount(half(on && less));
    if (on) {
      hrank[hid][uslot[hid][j]] = (uint8_t)rk;
      if (!DIRECT) out.rowbuf[kRowBuf * v + rk] = u;
      else if (write) out.colidx[p0 + rk] = u;
    }
  }
  wave_lds_sync();
  if (v < n && hl == 0) {
    big[v] = mine ? 0 : 1;
    if (!mine) atomicOr(any_big, 1);
    if (DIRECT && wrong) atomicOr(out.mismatch, 1);
    if (mine && len) {
      if (!DIRECT) out.rowbuf[kRowBuf * v + dpos] = (int32_t)v;
      else if (write) out.colidx[p0 + dpos] = (int32_t)v;
    }
    if (mine && !DIRECT) { out.rowlen[v] = len; out.dposr[v] = (int8_t)(len ? dpos : -1); }
    if (write && DIRECT) out.diag[v] = len ? p0 + dpos : -1;
  }
  if (mine && hl < deg) {
    uint32_t pk = (uint32_t)dpos, rank[R];  // own first
#pragma unroll
    for (int r = 0; r < R; ++r) {
      rank[r] = key[r] == (int32_t)v ? dpos : hrank[hid][slot[r]];
      pk |= rank[r] << (8 * r + 8);
    }
    if (NLOC == 4) slotmap[k0 + qp] = __builtin_rotateleft32(pk, 8 * lv);
    else
      slotmap[k0 + qp] = lv == 0 ? pk : lv == 1 ? (pk << 8 & 0xffff00u) | pk >> 16
                                                : (pk << 16 & 0xff0000u) | pk >> 8;
    if constexpr (VALS) {
      // the vertices are read here, not with the element: the registers that they
      // held through the passes above left 6 waves per SIMD instead of 8
      double vv[4][3], r4[4];
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int k = 0; k < 3; ++k) vv[m][k] = xyz[3 * (int64_t)c[m] + k];
      p1_row_entries(vv, lv, Ce[e], r4);
#pragma unroll
      for (int m = 0; m < 4; ++m) sv[hid][((m - lv - 1) & 3) * kHalf + qp] = r4[m];
#pragma unroll
      for (int r = 0; r < 3; ++r)  // slots past 32 to the word that nobody reads
        atomicOr(&smask[hid][r][min(rank[r < R ? r : 0], (uint32_t)kHalf)], 1u << qp);
      so[hid][qp] = pk;
    }
  }
  if constexpr (VALS) {  // the row's values, each slot summed by its lane in element order
    const int nq = mine ? deg : 0;
    if (hl >= nq) sv[hid][3 * kHalf + hl] = 0.;
    wave_lds_sync();
    double acc0 = 0., acc1 = 0.;
    // Every incidence holds the diagonal slot: its lane adds the incidences'
    // diagonal entries in order, 8 per round (past the row's count +0.0, which
    // leaves the sum unchanged: it starts at +0.0 and is never -0.0).  Another
    // slot's lane adds the entries of the incidences in its masks (bit q:
    // incidence q holds the slot), lowest first, 3 per round.  Both orders are
    // the element order.
    if (hl == dpos) {
      for (int q0 = 0; q0 < nq; q0 += 8) {
        double a[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) a[i] = sv[hid][3 * kHalf + q0 + i];
#pragma unroll
        for (int i = 0; i < 8; ++i) acc0 += a[i];
      }
    } else if (mine && hl < len) {
      const uint32_t m1 = smask[hid][1][hl], m2 = smask[hid][2][hl];
      uint32_t mask = smask[hid][0][hl] | m1 | m2;
      while (mask) {
        constexpr int U = 3;
        double a[U];
        bool ok[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
          ok[i] = mask != 0;
          const int q = (__ffs(mask) - 1) & (kHalf - 1);
          const int r = (int)(m1 >> q & 1) + 2 * (int)(m2 >> q & 1);
          a[i] = sv[hid][r * kHalf + q];
          mask &= mask - 1;
        }
#pragma unroll
        for (int i = 0; i < U; ++i) acc0 += ok[i] ? a[i] : 0.;
      }
    }
    if (__builtin_amdgcn_ballot_w64(mine && len > kHalf)) {  // rows of more than 32 columns: the second slot of each lane
      const uint32_t me1 = (uint32_t)(hl + kHalf) * 0x01010101u;
      if (len > kHalf)
        for (int q = 0; q < nq; ++q) {
          const uint32_t t1 = so[hid][q] ^ me1, z1 = (t1 - 0x01010101u) & ~t1 & 0x80808080u;
          if (z1) acc1 += sv[hid][(((__builtin_ctz(z1) >> 3) - 1) & 3) * kHalf + q];
        }
    }
    if (mine && !DIRECT) {
      if (hl < len) out.rowval[kRowBuf * v + hl] = acc0;
      if (hl + kHalf < len) out.rowval[kRowBuf * v + hl + kHalf] = acc1;
    }
    if (write && DIRECT) {
      if (hl < len) out.vals[p0 + hl] = acc0;
      if (hl + kHalf < len) out.vals[p0 + hl + kHalf] = acc1;
    }
  }
}

// The P1 row lengths a manifold simplicial mesh implies, from the counts of
// incident elements (deg) and boundary elements (b) of each vertex: the link
// of a vertex is a sphere (3D) / circle (2D) inside and a disk / path on the
// boundary, so Euler's formula gives its vertex count — 3D: 2 + deg/2 inside,
// 1 + (deg + b)/2 on the boundary; 2D: deg inside, deg + 1 on the boundary —
// and the row holds those vertices and its own.  Meshes where this does not
// hold (boundary elements inside the domain, non-manifold vertices) are found
// by the pattern pass, which compares every row with these lengths.
__global__ void k_bcount(int64_t m, const int32_t *__restrict__ belems, uint32_t *__restrict__ cnt) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < m) atomicAdd(&cnt[belems[i]], 1u);
}

__global__ void k_link_len(int64_t n, int dim, const int64_t *__restrict__ v2e_ptr,
                           const uint32_t *__restrict__ bcnt, int64_t *__restrict__ len) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  const int64_t deg = v2e_ptr[v + 1] - v2e_ptr[v], b = bcnt[v];
  int64_t l;
  if (dim == 3) l = b == 0 ? 3 + deg / 2 : 2 + (deg + b) / 2;
  else l = b == 0 ? 1 + deg : 2 + deg;
  len[v] = deg == 0 ? 0 : l;
  if (v == 0) len[n] = 0;  // the scan's last input
}

// buffered columns to their CSR place; diagonal slots.  One lane per row:
// the row's buffer is read as 16-byte groups, all issued before the stores,
// so a wave keeps 64 rows' loads in flight.
// With rowval, the row values too (2 doubles per 16-byte load).
__global__ __launch_bounds__(256) void k_pattern_compact(
    int64_t n, const int64_t *__restrict__ rowptr, const int32_t *__restrict__ rowbuf,
    const int8_t *__restrict__ dposr, const uint8_t *__restrict__ big,
    int32_t *__restrict__ colidx, int64_t *__restrict__ diag,
    const double *__restrict__ rowval = nullptr, double *__restrict__ vals = nullptr) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n || big[v]) return;
  const int64_t r0 = rowptr[v];
  const int len = (int)(rowptr[v + 1] - r0);
  if (rowval) {
    const double2 *vs = reinterpret_cast<const double2 *>(rowval + kRowBuf * v);
    double *vd = vals + r0;
    for (int g0 = 0; g0 < len; g0 += 8) {  // 8 values (4 loads) per round
      double2 q[4];
#pragma unroll
      for (int g = 0; g < 4; ++g)
        if (g0 + 2 * g < len) q[g] = vs[(g0 >> 1) + g];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (g0 + 2 * g < len) vd[g0 + 2 * g] = q[g].x;
        if (g0 + 2 * g + 1 < len) vd[g0 + 2 * g + 1] = q[g].y;
      }
    }
  }
  const int4 *src = reinterpret_cast<const int4 *>(rowbuf + kRowBuf * v);
  int32_t *dst = colidx + r0;
  for (int g0 = 0; g0 < len; g0 += 16) {  // 16 columns (4 groups) per round
    int4 q[4];
#pragma unroll
    for (int g = 0; g < 4; ++g)
      if (g0 + 4 * g < len) q[g] = src[(g0 >> 2) + g];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int32_t e[4] = {q[g].x, q[g].y, q[g].z, q[g].w};
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (g0 + 4 * g + t < len) dst[g0 + 4 * g + t] = e[t];
    }
  }
  diag[v] = dposr[v] < 0 ? -1 : r0 + dposr[v];
}

// ---------------------------------------------------------------- element matrices
// 3D P1: Ke_ij = S grad l_i . grad l_j with S = sum_q |K| w_q kappa(x_q)
// (problem.cpp:6387-6392); the 10 unique entries per element.
__device__ inline double p1_kappa_integral(int64_t e, const int32_t id[4], const double v[4][3],
                                           double mes, int kind, double c0,
                                           const double *__restrict__ kappa_e) {
  double S = 0.;
  if (kind == FFHIP_COEF_P1) {
    const double u[4] = {kappa_e[id[0]], kappa_e[id[1]], kappa_e[id[2]], kappa_e[id[3]]};
    S = mes * (0.25 * ((u[0] + u[1]) + (u[2] + u[3])));  // the rule is exact here
  } else if (kind == FFHIP_COEF_SIN3) {
#pragma unroll 1
    for (int q = 0; q < 14; ++q) {
      const double px = c_qf5_pts[q][0], py = c_qf5_pts[q][1], pz = c_qf5_pts[q][2];
      const double l0 = 1. - (px + py + pz);
      double P[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) P[k] = l0 * v[0][k] + px * v[1][k] + py * v[2][k] + pz * v[3][k];
      S += (mes * qf5_weight(q)) * kappa_sin3(P[0], P[1], P[2]);
    }
  } else if (kind == FFHIP_COEF_QP) {
#pragma unroll
    for (int q = 0; q < 14; ++q) S += (mes * qf5_weight(q)) * kappa_e[14 * e + q];
  } else {
    S = mes * ((kind == FFHIP_COEF_P0) ? kappa_e[e] : c0);
  }
  return S;
}

__device__ inline void load_tet(const double *__restrict__ xyz, const int32_t *__restrict__ tets,
                                int64_t e, int32_t id[4], double v[4][3]) {
  const int4 tv = reinterpret_cast<const int4 *>(tets)[e];
  id[0] = tv.x; id[1] = tv.y; id[2] = tv.z; id[3] = tv.w;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int k = 0; k < 3; ++k) v[i][k] = xyz[3 * (int64_t)id[i] + k];
}

// the reaction term of int3d(m*u*v): K(i,j) += sum_q |K| w_q m(x_q) l_i(q) l_j(q)
// for the 10 entries i <= j (P1 values l = barycentrics of the Tet_5 point)
__device__ inline void p1_mass_3d(int64_t e, const int32_t id[4], const double v[4][3], double mes,
                                  int mkind, double m0, const double *__restrict__ mass_e,
                                  double K[10]) {
  // m constant or linear: the rule is exact (degree 5 for an integrand of 3), so
  // the integrals of l_i l_j l_k, |K| / 120 (all different; 2 and 6 times that with
  // two and three equal).  Its 14 points took 41 us on a 61 x 50 x 43 box, now 34.
  if (mkind == FFHIP_COEF_CONST || mkind == FFHIP_COEF_P0 || mkind == FFHIP_COEF_P1) {
    double mu[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      mu[i] = mkind == FFHIP_COEF_P1 ? mass_e[id[i]] : mkind == FFHIP_COEF_P0 ? mass_e[e] : m0;
    const double w = mes * (1. / 120.), S = (mu[0] + mu[1]) + (mu[2] + mu[3]);
    int o = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = i; j < 4; ++j) {
        const double t = S + mu[i] + mu[j];
        K[o++] += w * (i == j ? t + t : t);
      }
    return;
  }
#pragma unroll 2
  for (int q = 0; q < 14; ++q) {
    const double px = c_qf5_pts[q][0], py = c_qf5_pts[q][1], pz = c_qf5_pts[q][2];
    const double l[4] = {1. - (px + py + pz), px, py, pz};
    double mq;
    if (mkind == FFHIP_COEF_SIN3) {
      double P[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) P[k] = l[0] * v[0][k] + px * v[1][k] + py * v[2][k] + pz * v[3][k];
      mq = kappa_sin3(P[0], P[1], P[2]);
    } else {
      mq = mass_e[14 * e + q];
    }
    const double W = (mes * qf5_weight(q)) * mq;
    int o = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = i; j < 4; ++j) K[o++] += (W * l[i]) * l[j];
  }
}

// entry (i, j), i <= j, of the P1 element matrix: sum_k (S G_ik) G_jk
__device__ inline double p1_entry(double S, const double G[4][3], int i, int j) {
  double a = 0.;
#pragma unroll
  for (int k = 0; k < 3; ++k) a += (S * G[i][k]) * G[j][k];
  return a;
}

// the element's 4 rows, each written where its incidence entry sits in the
// vertex's list (inv): Kinc[4k + m] = Ke(l, m) for the incidence k of (e, l),
// so the row gather reads them contiguously; with Ke != null also the 10
// unique entries per element (i <= j, row-major upper triangle) for the
// lane-per-row gather
// MASS: with the reaction term m*u*v (coefficient kind mkind, m0, mass_e)
template <bool MASS>
__global__ __launch_bounds__(256) void k_p1_element_3d(
    int64_t nt, const double *__restrict__ xyz, const int32_t *__restrict__ tets,
    int kind, double c0, const double *__restrict__ kappa_e, int mkind, double m0,
    const double *__restrict__ mass_e, const int32_t *__restrict__ inv,
    double *__restrict__ Kinc, double *__restrict__ Ke) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nt) return;
  double v[4][3], G[4][3];
  int32_t id[4];
  load_tet(xyz, tets, e, id, v);
  const double mes = tet_geom(v, G);
  const double S = p1_kappa_integral(e, id, v, mes, kind, c0, kappa_e);
  double K[10];
  int o = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = i; j < 4; ++j) K[o++] = p1_entry(S, G, i, j);
  if (MASS) p1_mass_3d(e, id, v, mes, mkind, m0, mass_e, K);
  const int4 pos = reinterpret_cast<const int4 *>(inv)[e];
  const int32_t kk[4] = {pos.x, pos.y, pos.z, pos.w};
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    double4 row;
    row.x = K[sym4(l, 0)]; row.y = K[sym4(l, 1)]; row.z = K[sym4(l, 2)]; row.w = K[sym4(l, 3)];
    reinterpret_cast<double4 *>(Kinc)[kk[l]] = row;
  }
  if (Ke) {
    double *dst = Ke + 10 * e;
#pragma unroll
    for (int i = 0; i < 10; ++i) dst[i] = K[i];
  }
}


// 2D P1: 6 unique entries; TTriangle area and H(i) (fem.hpp:290-325)
__global__ __launch_bounds__(256) void k_p1_element_2d(
    int64_t nt, const double *__restrict__ xy, const int32_t *__restrict__ tris,
    int kind, double c0, const double *__restrict__ kappa_e, int mkind, double m0,
    const double *__restrict__ mass_e, double *__restrict__ Ke) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nt) return;
  double v[3][2];
  int32_t id[3];
  for (int i = 0; i < 3; ++i) {
    id[i] = tris[3 * e + i];
    for (int k = 0; k < 2; ++k) v[i][k] = xy[2 * (int64_t)id[i] + k];
  }
  const double area = ((v[1][0] - v[0][0]) * (v[2][1] - v[0][1]) -
                       (v[1][1] - v[0][1]) * (v[2][0] - v[0][0])) * 0.5;
  double G[3][2];
  for (int i = 0; i < 3; ++i) {
    const int a = (i + 2) % 3, b = (i + 1) % 3;
    const double Ex = v[a][0] - v[b][0], Ey = v[a][1] - v[b][1];
    G[i][0] = -Ey / (2 * area);
    G[i][1] = Ex / (2 * area);
  }
  double S = 0.;
  for (int q = 0; q < 7; ++q) {
    double kc;
    if (kind == FFHIP_COEF_SIN3) {
      const double px = c_qt5_pts[q][0], py = c_qt5_pts[q][1];
      const double l0 = 1. - px - py;
      const double X = l0 * v[0][0] + px * v[1][0] + py * v[2][0];
      const double Y = l0 * v[0][1] + px * v[1][1] + py * v[2][1];
      const double tp = 2 * M_PI;
      kc = 1 + (0.5 * sin(tp * X)) * sin(tp * Y);
    } else if (kind == FFHIP_COEF_QP) {
      kc = kappa_e[7 * e + q];
    } else if (kind == FFHIP_COEF_P1) {
      const double u[3] = {kappa_e[id[0]], kappa_e[id[1]], kappa_e[id[2]]};
      kc = p1_value2(u, c_qt5_pts[q][0], c_qt5_pts[q][1]);
    } else {
      kc = (kind == FFHIP_COEF_P0) ? kappa_e[e] : c0;
    }
    S += (area * c_qt5_w[q]) * kc;
  }
  double K[6];
  int o = 0;
  for (int i = 0; i < 3; ++i)
    for (int j = i; j < 3; ++j) {
      double a = 0.;
      for (int k = 0; k < 2; ++k) a += (S * G[i][k]) * G[j][k];
      K[o++] = a;
    }
  if (mkind >= 0) {  // the reaction term m*u*v with T_5
    for (int q = 0; q < 7; ++q) {
      const double px = c_qt5_pts[q][0], py = c_qt5_pts[q][1];
      const double l[3] = {1. - px - py, px, py};
      double mq = (mkind == FFHIP_COEF_P0) ? mass_e[e] : m0;
      if (mkind == FFHIP_COEF_SIN3) {
        const double X = l[0] * v[0][0] + px * v[1][0] + py * v[2][0];
        const double Y = l[0] * v[0][1] + px * v[1][1] + py * v[2][1];
        const double tp = 2 * M_PI;
        mq = 1 + (0.5 * sin(tp * X)) * sin(tp * Y);
      } else if (mkind == FFHIP_COEF_QP) {
        mq = mass_e[7 * e + q];
      } else if (mkind == FFHIP_COEF_P1) {
        const double u[3] = {mass_e[id[0]], mass_e[id[1]], mass_e[id[2]]};
        mq = p1_value2(u, px, py);
      }
      const double W = (area * c_qt5_w[q]) * mq;
      o = 0;
      for (int i = 0; i < 3; ++i)
        for (int j = i; j < 3; ++j) K[o++] += (W * l[i]) * l[j];
    }
  }
  for (int i = 0; i < 6; ++i) Ke[6 * e + i] = K[i];
}

// ---------------------------------------------------------------- row gather
// Block of BLOCK rows; the block's CSR segment is staged in LDS when it fits
// (STAGE doubles), else each lane accumulates its own row in global memory.
template <int BLOCK, int STAGE, int NLOC>
__global__ __launch_bounds__(BLOCK) void k_p1_gather(
    int64_t n, const int64_t *__restrict__ rowptr, const int64_t *__restrict__ v2e_ptr,
    const int32_t *__restrict__ v2e, const uint32_t *__restrict__ slotmap,
    const double *__restrict__ Ke, double *__restrict__ vals,
    const uint8_t *__restrict__ only = nullptr) {
  constexpr int NU = NLOC * (NLOC + 1) / 2;
  __shared__ double S[STAGE];
  const int t = threadIdx.x;
  const int64_t v0 = (int64_t)blockIdx.x * BLOCK;
  const int64_t v = v0 + t;
  const int64_t vend = (v0 + BLOCK < n) ? v0 + BLOCK : n;
  const int64_t seg0 = rowptr[v0], seg1 = rowptr[vend];
  const bool staged = (seg1 - seg0) <= STAGE;
  if (staged) {
    for (int64_t i = t; i < seg1 - seg0; i += BLOCK) S[i] = 0.;
    __syncthreads();
  }
  if (v < n && (!only || only[v])) {  // only[]: the rows this kernel owns
    const int64_t r0 = rowptr[v];
    double *acc = staged ? S + (r0 - seg0) : vals + r0;
    if (!staged)
      for (int64_t i = r0; i < rowptr[v + 1]; ++i) vals[i] = 0.;
    const int64_t k0 = v2e_ptr[v], k1 = v2e_ptr[v + 1];
    for (int64_t k = k0; k < k1; ++k) {
      const int32_t idx = v2e[k];
      const int64_t e = idx / NLOC;
      const int l = idx - (int)e * NLOC;
      const uint32_t pk = slotmap[k];
      const double *ke = Ke + NU * e;
#pragma unroll
      for (int m = 0; m < NLOC; ++m) {
        const int off = (pk >> (8 * m)) & 0xff;
        const double a = ke[NLOC == 4 ? sym4(l, m) : sym3(l, m)];
        acc[off] += a;
      }
    }
  }
  if (staged) {
    __syncthreads();
    if (!only) {
      for (int64_t i = t; i < seg1 - seg0; i += BLOCK) vals[seg0 + i] = S[i];
    } else {
      for (int64_t i = t; i < seg1 - seg0; i += BLOCK) {
        const int64_t g = seg0 + i;
        int64_t lo = v0, hi = vend - 1;  // the row of slot g
        while (lo < hi) {
          const int64_t mid = (lo + hi + 1) >> 1;
          if (rowptr[mid] <= g) lo = mid; else hi = mid - 1;
        }
        if (only[lo]) vals[g] = S[i];
      }
    }
  }
}

// 3D values, one row per 32-lane half-wave: lane q takes incidence q (element
// order), whose 4 row entries the element kernel stored at Kinc[4k..4k+3],
// and stages them and their 4 slot bytes in LDS; lane j then walks the
// incidences in order and adds the entry (if any) whose slot is j (lanes own
// slots j and j + 32) — the same sums, in the same order, as a sequential walk
// over the row's elements.  Rows flagged big[] (more than 32 elements or 64
// columns) are left to k_p1_gather.
__global__ __launch_bounds__(256) void k_p1_values_half(
    int64_t n, const int64_t *__restrict__ rowptr, const int64_t *__restrict__ v2e_ptr,
    const uint32_t *__restrict__ slotmap, const double *__restrict__ Kinc,
    const uint8_t *__restrict__ big, double *__restrict__ vals) {
  __shared__ double sv[256 / kHalf][4 * kHalf];
  __shared__ uint32_t so[256 / kHalf][kHalf];  // 4 slot bytes per incidence
  const int hl = threadIdx.x % kHalf, hid = threadIdx.x / kHalf;
  const int64_t v = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kHalf;
  int64_t k0 = 0, r0 = 0;
  int deg = 0, len = 0;
  if (v < n && !big[v]) {
    k0 = v2e_ptr[v];
    deg = (int)(v2e_ptr[v + 1] - k0);
    r0 = rowptr[v];
    len = (int)(rowptr[v + 1] - r0);
  }
  if (hl < deg) {
    const double4 row = reinterpret_cast<const double4 *>(Kinc)[k0 + hl];
    sv[hid][4 * hl + 0] = row.x;
    sv[hid][4 * hl + 1] = row.y;
    sv[hid][4 * hl + 2] = row.z;
    sv[hid][4 * hl + 3] = row.w;
    so[hid][hl] = slotmap[k0 + hl];
  }
  __syncthreads();
  const uint32_t me0 = (uint32_t)hl * 0x01010101u, me1 = (uint32_t)(hl + kHalf) * 0x01010101u;
  double acc0 = 0., acc1 = 0.;
  for (int q = 0; q < deg; ++q) {
    // lowest byte of so[q] equal to the lane's slot (at most one is)
    const uint32_t pk = so[hid][q];
    const uint32_t t0 = pk ^ me0, z0 = (t0 - 0x01010101u) & ~t0 & 0x80808080u;
    if (z0) acc0 += sv[hid][4 * q + (__builtin_ctz(z0) >> 3)];
    if (len > kHalf) {
      const uint32_t t1 = pk ^ me1, z1 = (t1 - 0x01010101u) & ~t1 & 0x80808080u;
      if (z1) acc1 += sv[hid][4 * q + (__builtin_ctz(z1) >> 3)];
    }
  }
  if (hl < len) vals[r0 + hl] = acc0;
  if (hl + kHalf < len) vals[r0 + hl + kHalf] = acc1;
}

// ---------------------------------------------------------------- 3D stiffness in two passes
// K_e(l, m) = S_e grad l_l . grad l_m (problem.cpp:6387-6392) with
// grad l_l = N_l / (6 |K|), N_l the cross products of the edge vectors from
// vertex 0 (Tet::Gradlambda, Mesh3dn.hpp:126-137, before its division) and
// N_0 = -(N_1 + N_2 + N_3): the element pass stores the one scale
// C_e = S_e / (6 |K|)^2 per element, and the row pass forms the row's entries
// C_e N_l . N_m from the vertices — no element rows through HBM.
__global__ __launch_bounds__(256) void k_p1_scale_3d(int64_t nt, const double *__restrict__ xyz,
                                                     const int32_t *__restrict__ tets, int kind,
                                                     double c0, const double *__restrict__ kappa_e,
                                                     double *__restrict__ Ce) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nt) return;
  double v[4][3];
  int32_t id[4];
  load_tet(xyz, tets, e, id, v);
  const double mes = tet_mesure(v);
  const double S = p1_kappa_integral(e, id, v, mes, kind, c0, kappa_e);
  const double d1 = 1. / (6. * mes);
  Ce[e] = (S * d1) * d1;
}

// The incidence buckets of k_v2e_bucket_block fused with the element scales
// of k_p1_scale_3d (tets): a block takes 256 tets (1024 items, 4 per thread,
// a 2048-slot LDS hash set); the thread's tet is loaded with its items, the
// block's global count atomics are issued before the tet's scale is
// computed (their round trip hidden by the arithmetic), and the items are
// placed after it.  The scale is the same computation as k_p1_scale_3d's.
// (5 waves per SIMD, no spills; uncapped it takes 108 registers and runs 4.  One
// point of the rule at a time: cube(160) 1150 us for 1210 with two, now 1107)
constexpr int kFuseLog = 11;
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5, 5))) void k_v2e_bucket_scale(const int32_t *__restrict__ tets, int64_t nt,
                                                          ScaleArgs sc, uint32_t *__restrict__ deg,
                                                          int32_t *__restrict__ bucket,
                                                          int *__restrict__ ovf) {
  constexpr int IPT = 4, HS = 1 << kFuseLog;
  __shared__ int32_t hkey[HS];
  __shared__ uint32_t hcnt[HS];
  __shared__ uint32_t hbase[HS];
  const int t = threadIdx.x;
  const int64_t m = 4 * nt, b0 = (int64_t)blockIdx.x * (256 * IPT);
  for (int i = t; i < HS; i += blockDim.x) { hkey[i] = -1; hcnt[i] = 0; }
  int32_t v[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const int64_t i = b0 + j * 256 + t;
    v[j] = i < m ? tets[i] : -1;
  }
  const int64_t e = (int64_t)blockIdx.x * 256 + t;
  double tv[4][3];
  int32_t id[4];
  if (e < nt) load_tet(sc.xyz, tets, e, id, tv);
  __syncthreads();
  uint32_t h[IPT], rank[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    h[j] = 0;
    rank[j] = 0;
    if (v[j] >= 0) {
      h[j] = ((uint32_t)v[j] * 2654435761u) >> (32 - kFuseLog);
      for (;;) {  // ends: at most half the slots hold keys
        const int32_t old = atomicCAS(&hkey[h[j]], -1, v[j]);
        if (old == -1 || old == v[j]) break;
        h[j] = (h[j] + 1) & (HS - 1);
      }
      rank[j] = atomicAdd(&hcnt[h[j]], 1u);
    }
  }
  __syncthreads();
  uint32_t hb[HS / 256];
#pragma unroll
  for (int q = 0; q < HS / 256; ++q) {
    const int32_t key = hkey[t + q * 256];
    hb[q] = key >= 0 ? atomicAdd(&deg[key], hcnt[t + q * 256]) : 0u;
  }
  if (e < nt) {
    const double mes = tet_mesure(tv);
    const double S = p1_kappa_integral(e, id, tv, mes, sc.kind, sc.c0, sc.kappa_e);
    const double d1 = 1. / (6. * mes);
    sc.Ce[e] = (S * d1) * d1;
  }
#pragma unroll
  for (int q = 0; q < HS / 256; ++q) hbase[t + q * 256] = hb[q];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    if (v[j] < 0) continue;
    const int64_t i = b0 + j * 256 + t;
    const uint32_t pos = hbase[h[j]] + rank[j];
    if (pos < 32) bucket[32 * (int64_t)v[j] + pos] = (int32_t)i;
    else atomicOr(ovf, 1);
  }
}

// values, one row per 32-lane half-wave (rows of up to 32 elements and 64
// columns; big[] rows are left to the lane-per-row gather): lane q takes
// incidence q (element order), forms its element's row l from the vertices
// and C_e, and stages the 4 entries with their slot bytes (the element-to-row
// map of the pattern) in LDS; lane j then adds, in element order, the entries
// whose slot is j (lanes own slots j and j + 32) — the summation order of
// HashMatrix::operator+= over the element loop.  Blocks take contiguous row
// ranges per XCD (the gathered vertices and element scales of neighbouring
// rows stay in that XCD's L2).
__global__ __launch_bounds__(256) void k_p1_values_rows(
    int64_t n, const int64_t *__restrict__ rowptr, const int64_t *__restrict__ v2e_ptr,
    const int32_t *__restrict__ v2e, const uint32_t *__restrict__ slotmap,
    const double *__restrict__ xyz, const int32_t *__restrict__ tets, const double *__restrict__ Ce,
    const uint8_t *__restrict__ big, double *__restrict__ vals) {
  __shared__ double sv[256 / kHalf][4 * kHalf];
  __shared__ uint32_t so[256 / kHalf][kHalf];
  const int hl = threadIdx.x % kHalf, hid = threadIdx.x / kHalf;
  const int64_t v = ((int64_t)xcd_block_id() * blockDim.x + threadIdx.x) / kHalf;
  int64_t k0 = 0, r0 = 0;
  int deg = 0, len = 0;
  if (v < n && !big[v]) {
    k0 = v2e_ptr[v];
    deg = (int)(v2e_ptr[v + 1] - k0);
    r0 = rowptr[v];
    len = (int)(rowptr[v + 1] - r0);
  }
  if (hl < deg) {
    const int32_t idx = v2e[k0 + hl];
    const int64_t e = idx >> 2;
    const int l = idx & 3;
    const uint32_t pk = slotmap[k0 + hl];
    const int4 tv = reinterpret_cast<const int4 *>(tets)[e];
    const int32_t id[4] = {tv.x, tv.y, tv.z, tv.w};
    const double C = Ce[e];
    double vv[4][3], r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int k = 0; k < 3; ++k) vv[i][k] = xyz[3 * (int64_t)id[i] + k];
    p1_row_entries(vv, l, C, r);
#pragma unroll
    for (int m = 0; m < 4; ++m) sv[hid][4 * hl + m] = r[m];
    so[hid][hl] = pk;
  }
  wave_lds_sync();  // sv / so are this row's (half-wave's) own
  const uint32_t me0 = (uint32_t)hl * 0x01010101u, me1 = (uint32_t)(hl + kHalf) * 0x01010101u;
  double acc0 = 0., acc1 = 0.;
  for (int q = 0; q < deg; ++q) {
    const uint32_t pk = so[hid][q];
    const uint32_t t0 = pk ^ me0, z0 = (t0 - 0x01010101u) & ~t0 & 0x80808080u;
    if (z0) acc0 += sv[hid][4 * q + (__builtin_ctz(z0) >> 3)];
    if (len > kHalf) {
      const uint32_t t1 = pk ^ me1, z1 = (t1 - 0x01010101u) & ~t1 & 0x80808080u;
      if (z1) acc1 += sv[hid][4 * q + (__builtin_ctz(z1) >> 3)];
    }
  }
  if (hl < len) vals[r0 + hl] = acc0;
  if (hl + kHalf < len) vals[r0 + hl + kHalf] = acc1;
}

// ---------------------------------------------------------------- Dirichlet
__global__ void k_mark_bc(int64_t nbe, int nbloc, const int32_t *__restrict__ belems,
                          const int32_t *__restrict__ blab, Labels labels, uint8_t *__restrict__ onbc) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= nbe || !labels.has(blab[f])) return;
  for (int q = 0; q < nbloc; ++q) onbc[belems[nbloc * f + q]] = 1;  // same value from every writer
}

__global__ void k_set_diag(int64_t n, const uint8_t *__restrict__ onbc,
                           const int64_t *__restrict__ diag, double tgv,
                           double *__restrict__ vals, int *__restrict__ missing) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !onbc[i]) return;
  const int64_t s = diag[i];
  if (s < 0) { *missing = 1; return; }
  vals[s] = tgv;
}

// ---------------------------------------------------------------- right-hand side
// b[v] = sum over the incident elements (element order) of int_K f l_v with
// the element's rule (Element_rhs, problem.cpp:7940-7978); f: CONST f0, SIN3,
// P0 fcoef[e], QP fcoef[e * nq + q], P1 fcoef[vertex] interpolated at the
// point.  Dirichlet rows: tgv * (gvals[v] or g0).
__device__ inline double rhs_coef(int kind, double f0, const double *__restrict__ fcoef, int64_t e,
                                  int q, int nq, double x, double y, double z, int dim) {
  if (kind == FFHIP_COEF_SIN3) {
    if (dim == 3) return kappa_sin3(x, y, z);
    const double tp = 2 * M_PI;
    return 1 + (0.5 * sin(tp * x)) * sin(tp * y);
  }
  if (kind == FFHIP_COEF_QP) return fcoef[e * nq + q];
  if (kind == FFHIP_COEF_P0) return fcoef[e];
  return f0;
}

// LDS position of staged item i of a wave's 64 rows: one item of padding per
// 32, so that rows of 8, 16 or 24 items do not start in the same banks
__device__ inline int stage_pos(int i) { return i + (i >> 5); }

// What the row pass below needs of each tet for the terms of its 4 vertices
// (rule of Tet_5, exact for these products):
//   kRowScale  f constant on the tet:  E = |K| f, term E / 4
//   kRowPair   f P1:                   E = (|K| / 20, sum of the 4 f's), term E.x (f_v + E.y)
//   kRowQuad   f at the 14 points:     E = the 4 integrals, term E[l]
constexpr int kRowScale = 0, kRowPair = 1, kRowQuad = 2;
template <int RM>
__global__ __launch_bounds__(256) void k_p1_load_elem(int64_t nt, const double *__restrict__ xyz,
                                                      const int32_t *__restrict__ tets, int kind,
                                                      double f0, const double *__restrict__ fcoef,
                                                      double *__restrict__ E) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nt) return;
  double v[4][3];
  int32_t id[4];
  load_tet(xyz, tets, e, id, v);
  const double mes = tet_mesure(v);
  if constexpr (RM == kRowScale) {
    E[e] = mes * (kind == FFHIP_COEF_P0 ? fcoef[e] : f0);
  } else if constexpr (RM == kRowPair) {
    const double se = fcoef[id[0]] + fcoef[id[1]] + fcoef[id[2]] + fcoef[id[3]];
    reinterpret_cast<double2 *>(E)[e] = double2{mes / 20., se};
  } else {
    double r[4] = {0., 0., 0., 0.};
    for (int q = 0; q < 14; ++q) {
      const double px = c_qf5_pts[q][0], py = c_qf5_pts[q][1], pz = c_qf5_pts[q][2];
      const double l[4] = {1. - (px + py + pz), px, py, pz};
      double P[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) P[k] = l[0] * v[0][k] + px * v[1][k] + py * v[2][k] + pz * v[3][k];
      const double W = (mes * qf5_weight(q)) * rhs_coef(kind, f0, fcoef, e, q, 14, P[0], P[1], P[2], 3);
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] += W * l[i];
    }
    double4 o;
    o.x = r[0]; o.y = r[1]; o.z = r[2]; o.w = r[3];
    reinterpret_cast<double4 *>(E)[e] = o;
  }
}

// b_v = the sum of v's incidence terms in element order.  A wave takes 64 rows:
// it reads their incidence lists consecutively (lane on incidence), stages what
// it gathers in LDS chunk by chunk, and each lane adds its own row from there
// in order.  Bound by the bytes of the lists and of E (4 + 8..16 per
// incidence), so the stage is small (4.2 KB: the waves of a CU are limited by
// registers, not LDS): 187 us for a constant f at cube(160), 98 M incidences,
// 3.3 TB/s; with 2048 staged items per wave (9 waves per CU) 422 us, with
// 1024 and 16 in flight 260 us.  A half-wave per row whose 32 lanes each added
// all 32 slots issued 32 LDS reads for two rows and took 1660 us.  PAIR at
// cube(96), 21 M incidences: 70 us (half-wave: 378 us with |K| recomputed).
// PAIR terms need the row's own value (own, minus own2 when given); the
// product and the sum are rounded on their own, as the term and its addition
// were.  tgv rows: tgv * (gvals[v] or g0).
// PART (a device without room for every tet's E): E holds the tets [e0, e1), the
// row's sum goes on from b, and the last part (e1 = nt) writes the tgv rows.  A
// row's list is in element order, so the additions are the same.
struct RowPart {
  int64_t e0, e1, nt;
};
template <int RM, int ROWS, bool PART = false>
__global__ __launch_bounds__(64) void k_row_sum(
    int64_t n, const int64_t *__restrict__ v2e_ptr, const int32_t *__restrict__ v2e,
    const double *__restrict__ E, const double *__restrict__ own, const double *__restrict__ own2,
    const uint8_t *__restrict__ onbc, double tgv, double g0, const double *__restrict__ gvals,
    double *__restrict__ b, RowPart part = {}) {
  constexpr int U = RM == kRowPair ? 4 : 8, CAP = kWave * U;  // one round of gathers per chunk
  using T = typename std::conditional<RM == kRowPair, double2, double>::type;
  __shared__ T st[CAP + CAP / 32];
  const int lane = threadIdx.x;
  const int64_t r0 = (int64_t)xcd_block_id() * ROWS, rend = r0 + ROWS < n ? r0 + ROWS : n;
  if (r0 >= n) return;  // one wave per block
  const int64_t r = r0 + lane;  // lanes past the rows hold an empty range at the end
  int64_t p0 = v2e_ptr[r < rend ? r : rend], p1 = v2e_ptr[r + 1 < rend ? r + 1 : rend];
  const int64_t seg0 = v2e_ptr[r0], seg1 = v2e_ptr[rend];
  double me = 0.;
  if (RM == kRowPair && r < rend) me = own2 ? own[r] - own2[r] : own[r];
  double s = 0.;
  if constexpr (PART) {
    auto first = [&](int64_t e) {  // the row's first incidence of a tet >= e
      int64_t lo = p0, hi = p1;
      while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (v2e[mid] >> 2 < e) lo = mid + 1; else hi = mid;
      }
      return lo;
    };
    const int64_t a = first(part.e0), z = first(part.e1);
    p0 = a;
    p1 = z;
    if (part.e0 > 0 && r < rend) s = b[r];
  }
  for (int64_t c0 = seg0; c0 < seg1; c0 += CAP) {
    const int cnt = (int)(seg1 - c0 < CAP ? seg1 - c0 : CAP);
    for (int i0 = lane; i0 < cnt; i0 += kWave * U) {
      int32_t idx[U];
      T t[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + u * kWave;
        idx[u] = i < cnt ? v2e[c0 + i] : 0;
        if (PART) {  // another part's tets are staged too, but not added
          const int64_t e = idx[u] >> 2;
          idx[u] = e >= part.e0 && e < part.e1 ? idx[u] - 4 * (int32_t)part.e0 : 0;
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        t[u] = reinterpret_cast<const T *>(E)[RM == kRowQuad ? idx[u] : idx[u] >> 2];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + u * kWave;
        if (i < cnt) st[stage_pos(i)] = t[u];
      }
    }
    wave_lds_sync();
    const int b0 = (int)((p0 > c0 ? p0 : c0) - c0);
    const int b1 = (int)((p1 < c0 + cnt ? p1 : c0 + cnt) - c0);
    if constexpr (RM == kRowPair) {
      for (int k = b0; k < b1; ++k) {
        const double2 q = st[stage_pos(k)];
        double t = q.x * (me + q.y);
        asm("" : "+v"(t));  // rounded before it is added (no fused multiply-add)
        s += t;
      }
    } else {
#pragma unroll 4
      for (int k = b0; k < b1; ++k) s += RM == kRowScale ? 0.25 * st[stage_pos(k)] : st[stage_pos(k)];
    }
    wave_lds_sync();
  }
  if (r >= rend) return;
  if (onbc && onbc[r]) {
    if (PART && part.e1 < part.nt) return;
    s = tgv * (gvals ? gvals[r] : g0);
  }
  b[r] = s;
}

__global__ void k_rhs_p1_2d(int64_t n, const double *__restrict__ xy,
                            const int32_t *__restrict__ tris, const int64_t *__restrict__ v2e_ptr,
                            const int32_t *__restrict__ v2e, int kind, double f0,
                            const double *__restrict__ fcoef, const uint8_t *__restrict__ onbc,
                            double tgv, double g0, const double *__restrict__ gvals,
                            double *__restrict__ b) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  if (onbc && onbc[v]) { b[v] = tgv * (gvals ? gvals[v] : g0); return; }
  double s = 0.;
  for (int64_t k = v2e_ptr[v]; k < v2e_ptr[v + 1]; ++k) {
    const int32_t idx = v2e[k];
    const int64_t e = idx / 3;
    const int l = idx - 3 * (int)e;
    double p[3][2], fu[3] = {0., 0., 0.};
    for (int i = 0; i < 3; ++i)
      for (int kk = 0; kk < 2; ++kk) p[i][kk] = xy[2 * (int64_t)tris[3 * e + i] + kk];
    if (kind == FFHIP_COEF_P1)
      for (int i = 0; i < 3; ++i) fu[i] = fcoef[tris[3 * e + i]];
    const double area = ((p[1][0] - p[0][0]) * (p[2][1] - p[0][1]) -
                         (p[1][1] - p[0][1]) * (p[2][0] - p[0][0])) * 0.5;
    double r = 0.;
    for (int q = 0; q < 7; ++q) {
      const double px = c_qt5_pts[q][0], py = c_qt5_pts[q][1];
      const double l0 = 1 - px - py;
      const double lam = l == 0 ? l0 : (l == 1 ? px : py);
      double f = f0;
      if (kind == FFHIP_COEF_P1) {
        f = p1_value2(fu, px, py);
      } else if (kind != FFHIP_COEF_CONST) {
        const double X = l0 * p[0][0] + px * p[1][0] + py * p[2][0];
        const double Y = l0 * p[0][1] + px * p[1][1] + py * p[2][1];
        f = rhs_coef(kind, f0, fcoef, e, q, 7, X, Y, 0., 2);
      }
      r += (area * c_qt5_w[q]) * f * lam;
    }
    s += r;
  }
  b[v] = s;
}

// ---------------------------------------------------------------- adjoint blocks
// per element: misfit 1/2 int_K e^2 = |K|/40 (sum e_i^2 + (sum e_i)^2), e = u - ud;
// with pair also (|K|/20, sum e_i), the element's part of M e (kRowPair)
__global__ __launch_bounds__(256) void k_p1_misfit_elem(
    int64_t nt, const double *__restrict__ xyz, const int32_t *__restrict__ tets,
    const double *__restrict__ u, const double *__restrict__ ud, double *__restrict__ part,
    double2 *__restrict__ pair) {
  __shared__ double lds[256 / kWave];
  double acc = 0.;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < nt; e += (int64_t)gridDim.x * 256) {
    const int4 tv = reinterpret_cast<const int4 *>(tets)[e];
    const int32_t id[4] = {tv.x, tv.y, tv.z, tv.w};
    double v[4][3], ev[4];
    for (int i = 0; i < 4; ++i) {
      for (int k = 0; k < 3; ++k) v[i][k] = xyz[3 * (int64_t)id[i] + k];
      ev[i] = u[id[i]] - ud[id[i]];
    }
    const double mes = tet_mesure(v);
    const double s1 = ev[0] + ev[1] + ev[2] + ev[3];
    const double s2 = ev[0] * ev[0] + ev[1] * ev[1] + ev[2] * ev[2] + ev[3] * ev[3];
    acc += mes / 40. * (s2 + s1 * s1);
    if (pair) pair[e] = double2{mes / 20., s1};
  }
  const double tot = block_sum<256>(acc, lds);
  if (part && threadIdx.x == 0) part[blockIdx.x] = tot;
}

// Sum of a row's incidence terms in element order, one row per 32-lane
// half-wave: lane q computes the term of incidence c0 + q of each chunk of 32
// into its LDS slot, and every lane then adds the 32 slots in order (the order
// of the element loop, so the sum rounds as FreeFEM's accumulation into the
// row).  Slots past the row's end hold +0.0, and adding +0.0 leaves the sum
// unchanged: a sum that starts at +0.0 is never -0.0 under round-to-nearest.
template <class F>
__device__ inline double row_sum_in_order(double *__restrict__ slot, int hl, int64_t deg, F term) {
  double s = 0.;
  for (int64_t c0 = 0; c0 < deg; c0 += kHalf) {
    slot[hl] = c0 + hl < deg ? term(c0 + hl) : 0.;
    wave_lds_sync();
#pragma unroll
    for (int q = 0; q < kHalf; ++q) s += slot[q];
    wave_lds_sync();
  }
  return s;
}

// (M e)_v = sum over incident elements of |K|/20 (e_v + sum_K e_j); 0 on
// Dirichlet rows: the pass where there is no per-element temporary (the entry
// point that allocates nothing, a device without room for one; else the pairs
// are stored with the misfit and added in k_row_sum, the same terms in the same
// order)
__global__ __launch_bounds__(256) void k_p1_mass_apply(
    int64_t n, const double *__restrict__ xyz, const int32_t *__restrict__ tets,
    const int64_t *__restrict__ v2e_ptr, const int32_t *__restrict__ v2e,
    const double *__restrict__ u, const double *__restrict__ ud, const uint8_t *__restrict__ onbc,
    double *__restrict__ r) {
  const int hl = threadIdx.x % kHalf;
  const int64_t v = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kHalf;
  if (v >= n) return;  // uniform in the half-wave
  if (onbc && onbc[v]) {
    if (hl == 0) r[v] = 0.;
    return;
  }
  const double ev = u[v] - ud[v];
  __shared__ double slots[256];
  const int64_t k0 = v2e_ptr[v];
  const double s = row_sum_in_order(slots + (threadIdx.x & ~(kHalf - 1)), hl, v2e_ptr[v + 1] - k0,
                                    [&](int64_t k) {
    const int64_t e = v2e[k0 + k] >> 2;
    const int4 tv = reinterpret_cast<const int4 *>(tets)[e];
    const int32_t id[4] = {tv.x, tv.y, tv.z, tv.w};
    double vv[4][3], se = 0.;
    for (int i = 0; i < 4; ++i) {
      for (int kk = 0; kk < 3; ++kk) vv[i][kk] = xyz[3 * (int64_t)id[i] + kk];
      se += u[id[i]] - ud[id[i]];
    }
    return tet_mesure(vv) / 20. * (ev + se);
  });
  if (hl == 0) r[v] = s;
}

// g_e = -|K| grad u_K . grad lambda_K
__global__ __launch_bounds__(256) void k_p1_grad_kappa(
    int64_t nt, const double *__restrict__ xyz, const int32_t *__restrict__ tets,
    const double *__restrict__ u, const double *__restrict__ lam, double *__restrict__ g) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nt) return;
  const int4 tv = reinterpret_cast<const int4 *>(tets)[e];
  const int32_t id[4] = {tv.x, tv.y, tv.z, tv.w};
  double v[4][3], G[4][3];
  for (int i = 0; i < 4; ++i)
    for (int k = 0; k < 3; ++k) v[i][k] = xyz[3 * (int64_t)id[i] + k];
  const double mes = tet_geom(v, G);
  double gu[3] = {0., 0., 0.}, gl[3] = {0., 0., 0.};
  for (int i = 0; i < 4; ++i) {
    const double ui = u[id[i]], li = lam[id[i]];
    for (int k = 0; k < 3; ++k) { gu[k] += ui * G[i][k]; gl[k] += li * G[i][k]; }
  }
  g[e] = -mes * (gu[0] * gl[0] + gu[1] * gl[1] + gu[2] * gl[2]);
}

// ---------------------------------------------------------------- CSR mat-vec
// y = A x over a CSR pattern, the value of entry k read as vals[k] (kPlain),
// vals[slot[k]] (kSlots: the full view of a half matrix) or the entry (j, i)
// of a symmetric pattern (kTrans: y = A^T x, *missing raised where the pattern
// holds no such entry; y's old values go to keep, for a call that is refused).
//
// Bound by HBM (12 nnz + 20 n bytes), so every matrix load is coalesced: a wave
// takes 64 rows, reads their entries consecutively (lane on entry, up to 8
// independent load pairs per lane in flight), stages the pairs (a, x_j) in LDS
// and each lane then adds its own row in entry order with fused multiply-adds,
// bit for bit the sum of a lane that walks its row in memory.  The stage is one
// round of loads (4 or 8 KB, so that LDS does not limit the waves per CU).
// cube(72) (n = 389,017, nnz = 5.7 M): A x 19 us, half 25 us, A^T x 63 us (29,
// 41 and 74 us with a 16 KB stage); with a lane per row in memory, the lanes
// 120 bytes apart, 130 us, 180 us, and 215 us after a 161 us pass that wrote
// the transposed slots.
constexpr int kPlain = 0, kSlots = 1, kTrans = 2;

// slot of column i among the sorted columns [lo, end) of a row, or -1
__device__ inline int64_t find_entry(int64_t lo, int64_t end, const int32_t *__restrict__ colidx,
                                     int32_t i) {
  int64_t hi = end - 1;
  while (lo <= hi) {
    const int64_t mid = (lo + hi) >> 1;
    const int32_t c = colidx[mid];
    if (c == i) return mid;
    if (c < i) lo = mid + 1; else hi = mid - 1;
  }
  return -1;
}

template <int MODE, int ROWS>
__global__ __launch_bounds__(64) void k_spmv_stage(int64_t n, const int64_t *__restrict__ rowptr,
                                                   const int32_t *__restrict__ colidx,
                                                   const double *__restrict__ vals,
                                                   const int64_t *__restrict__ slot,
                                                   const double *__restrict__ x, double *__restrict__ y,
                                                   int *__restrict__ missing, double *__restrict__ keep) {
  constexpr int U = MODE == kTrans ? 8 : 4, CAP = kWave * U;  // one round of loads per chunk
  __shared__ double2 st[CAP + CAP / 32];
  __shared__ int64_t rs[kWave];  // kTrans: the rows' starts
  const int lane = threadIdx.x;
  const int64_t r0 = (int64_t)xcd_block_id() * ROWS, rend = r0 + ROWS < n ? r0 + ROWS : n;
  if (r0 >= n) return;  // one wave per block
  const int64_t r = r0 + lane;  // lanes past the rows hold an empty range at the end
  const int64_t p0 = rowptr[r < rend ? r : rend], p1 = rowptr[r + 1 < rend ? r + 1 : rend];
  const int64_t seg0 = rowptr[r0], seg1 = rowptr[rend];
  if constexpr (MODE == kTrans) {
    rs[lane] = p0;
    wave_lds_sync();
  }
  double acc = 0.;
  for (int64_t c0 = seg0; c0 < seg1; c0 += CAP) {
    const int cnt = (int)(seg1 - c0 < CAP ? seg1 - c0 : CAP);
    for (int i0 = lane; i0 < cnt; i0 += kWave * U) {
      int32_t j[U];
      double a[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + u * kWave;
        j[u] = i < cnt ? colidx[c0 + i] : 0;
        if (MODE == kPlain) a[u] = i < cnt ? vals[c0 + i] : 0.;
        if (MODE == kSlots) a[u] = i < cnt ? vals[slot[c0 + i]] : 0.;
      }
      if constexpr (MODE == kTrans) {
        // Entry k of row i at (i, j): (j, i) is first looked for where it lies
        // when row j's offsets mirror row i's (structured meshes), so the
        // chain is row j's ends, one column, one value with U of them in
        // flight; a binary search finds the others.
        int64_t q0[U], q1[U], g[U];
        int32_t ri[U], cg[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int i = i0 + u * kWave;
          int lo = 0, hi = ROWS - 1;  // the row of this entry: the last that starts at or before it
          while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (rs[mid] <= c0 + i) lo = mid; else hi = mid - 1;
          }
          ri[u] = lo;
          q0[u] = rowptr[j[u]];
          q1[u] = rowptr[j[u] + 1];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t m = q1[u] - 1 - (c0 + i0 + u * kWave - rs[ri[u]]);
          g[u] = m > q0[u] ? m : q0[u];
          ri[u] += (int32_t)r0;
          cg[u] = g[u] < q1[u] ? colidx[g[u]] : -1;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          a[u] = 0.;
          if (i0 + u * kWave < cnt) {
            const int64_t s = cg[u] == ri[u] ? g[u] : find_entry(q0[u], q1[u], colidx, ri[u]);
            if (s >= 0) a[u] = vals[s];
            else *missing = 1;
          }
        }
      }
      double xv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) xv[u] = x[j[u]];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + u * kWave;
        if (i < cnt) st[stage_pos(i)] = double2{a[u], xv[u]};
      }
    }
    wave_lds_sync();
    const int b0 = (int)((p0 > c0 ? p0 : c0) - c0);
    const int b1 = (int)((p1 < c0 + cnt ? p1 : c0 + cnt) - c0);
#pragma unroll 4
    for (int k = b0; k < b1; ++k) {
      const double2 q = st[stage_pos(k)];
      acc = fma(q.x, q.y, acc);
    }
    wave_lds_sync();
  }
  if (r >= rend) return;
  if (MODE == kTrans) keep[r] = y[r];
  y[r] = acc;
}

// slot of the transposed entry: (i,j) at k  ->  (j,i); -1 if absent
__global__ void k_transpose_map(int64_t n, const int64_t *__restrict__ rowptr,
                                const int32_t *__restrict__ colidx, int64_t *__restrict__ tmap,
                                int *__restrict__ missing) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int64_t k = rowptr[i]; k < rowptr[i + 1]; ++k) {
    const int32_t j = colidx[k];
    int64_t lo = rowptr[j], hi = rowptr[j + 1] - 1, f = -1;
    while (lo <= hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (colidx[mid] == i) { f = mid; break; }
      if (colidx[mid] < i) lo = mid + 1; else hi = mid - 1;
    }
    tmap[k] = f;
    if (f < 0) atomicMax(missing, 1);
  }
}

static unsigned nblocks(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }
// Rows per wave of the staged row kernels: 64, or 16 where 64 would leave under
// 16 waves per CU, each with several chunks one after the other.  PAIR sums and
// A x, 64 against 16 rows: cube(12) 20.0 / 7.4 and 8.0 / 4.0 us, cube(40) 22.0 /
// 10.3 and 10.8 / 6.4, cube(60) (227 k rows) 25.8 / 20.8 and 13.9 / 12.6,
// cube(72) A x 18.9 / 20.1, cube(96) PAIR 70 / 76, cube(160) SCALE 188 / 226.
static bool few_rows(int64_t n) { return n < 64 * 16 * 256; }
// one wave per `rows` rows, whole XCD groups
static unsigned row_grid(int64_t n, int rows) { return (nblocks(n, rows) + 7) / 8 * 8; }
void half_view(ffhip_mat L);

// once per device (__constant__ memory is per device): the context's device,
// the caller's current device restored afterwards
static void upload_t5_once(int dev) {
  static bool done[64] = {};
  FFHIP_REQUIRE(dev >= 0 && dev < 64, FFHIP_ERR_UNSUPPORTED, "device id %d", dev);
  if (done[dev]) return;
  int cur = 0;
  FFHIP_CHECK(hipGetDevice(&cur));
  if (cur != dev) FFHIP_CHECK(hipSetDevice(dev));
  const double sqrt15 = 3.87298334620741688517926539978;
  const double t = 1.E0 / 3.E0, A = 0.225E0;
  const double r = (6 - sqrt15) / 21, s = (9 + 2 * sqrt15) / 21, B = (155 - sqrt15) / 1200;
  const double u = (6 + sqrt15) / 21, v = (9 - 2 * sqrt15) / 21, C = (155 + sqrt15) / 1200;
  const double P[7][2] = {{t, t}, {r, r}, {r, s}, {s, r}, {u, u}, {u, v}, {v, u}};
  const double W[7] = {A, B, B, B, C, C, C};
  FFHIP_CHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_qt5_pts), P, sizeof(P)));
  FFHIP_CHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_qt5_w), W, sizeof(W)));
  if (cur != dev) FFHIP_CHECK(hipSetDevice(cur));
  done[dev] = true;
}

// dof -> (element * nloc + local) incidence lists in element order, for any
// element-to-dof table (P1 vertices, P2 nodes)
// The lists when some exceeds its 32-entry bucket: an atomic fill at the
// list offsets, then the lists of up to 32 entries sorted in a half-wave and
// the longer ones per dof (temporaries from the block cache: callable while
// an arena is held).
void v2e_fill_sort(ffhip_ctx ctx, const int32_t *elems, int64_t M, int64_t n, const int64_t *ptr,
                   int32_t *list, int32_t *inv) {
  hipStream_t s = ctx->stream;
  int32_t *cur = dalloc<int32_t>(n);
  int *flag = dalloc<int>(1);
  clear(ctx, {{cur, 4 * (size_t)n}, {flag, sizeof(int)}});
  k_v2e_fill<<<nblocks(M, 256), 256, 0, s>>>(elems, M, ptr, cur, list);
  k_v2e_sort_half<<<nblocks(n * kHalf, 256), 256, 0, s>>>(n, ptr, list, flag);
  k_v2e_sort<<<nblocks(n, 256), 256, 0, s>>>(n, ptr, list);
  if (inv) k_v2e_inverse<<<nblocks(M, 256), 256, 0, s>>>(M, list, inv);
  FFHIP_CHECK(hipGetLastError());
  dfree(cur);
  dfree(flag);
}

void build_incidence(ffhip_ctx ctx, const int32_t *elems, int64_t nt, int nloc, int64_t n,
                     int64_t **ptr_out, int32_t **list_out, int *big_out, int32_t **inv_out,
                     int32_t **bucket_out, const ScaleArgs *sc, int *ovf_dev) {
  hipStream_t s = ctx->stream;
  const int64_t M = nt * nloc;
  Arena ar(ctx, Arena::bytes(n, 4) + Arena::bytes(n + 1, 8) + (bucket_out ? 0 : Arena::bytes(32 * n, 4)) +
                    Arena::bytes(1, 4) + Arena::bytes(n, 4));
  uint32_t *deg = ar.take<uint32_t>(n);
  int64_t *deg64 = ar.take<int64_t>(n + 1);
  int32_t *bucket = bucket_out ? dalloc<int32_t>(32 * n) : ar.take<int32_t>(32 * n);
  if (bucket_out) *bucket_out = nullptr;
  // with ovf_dev (and bucket_out) the overflow flag is the caller's, read by
  // the caller later: nothing here waits for the device
  int *flag = ovf_dev && bucket_out ? ovf_dev : ar.take<int>(1);
  int64_t *ptr = dalloc<int64_t>(n + 1);
  int32_t *list = dalloc<int32_t>(M);
  int32_t *inv = inv_out ? dalloc<int32_t>(M) : nullptr;
  clear(ctx, {{deg, 4 * (size_t)n}, {flag, sizeof(int)}});
  if (sc && nloc == 4)  // the element scales computed in the same pass
    k_v2e_bucket_scale<<<nblocks(nt, 256), 256, 0, s>>>(elems, nt, *sc, deg, bucket, flag);
  else
    k_v2e_bucket_block<<<nblocks(M, 256 * kBucketIpt), 256, 0, s>>>(elems, M, deg, bucket, flag);
  k_u32_to_i64<<<nblocks(n, 256), 256, 0, s>>>(n, deg, deg64);
  exclusive_scan_i64(ctx, deg64, ptr, n + 1);
  FFHIP_CHECK(hipGetLastError());
  if (ovf_dev && bucket_out) {  // the caller checks the flag and sorts the buckets
    *bucket_out = bucket;
    if (big_out) *big_out = 0;
    if (inv_out) *inv_out = inv;
    *ptr_out = ptr;
    *list_out = list;
    return;
  }
  const int has_big = read_flag(ctx, flag);
  if (!has_big && bucket_out) {
    *bucket_out = bucket;  // the caller sorts the buckets into the lists
  } else if (!has_big) {
    k_v2e_sort_bucket<<<nblocks(n * kHalf, 256), 256, 0, s>>>(n, ptr, bucket, list, inv);
  } else {  // some list exceeds its bucket: fill by atomics, then sort
    if (bucket_out) dfree(bucket);
    v2e_fill_sort(ctx, elems, M, n, ptr, list, inv);
  }
  FFHIP_CHECK(hipGetLastError());
  FFHIP_CHECK(hipStreamSynchronize(s));
  if (big_out) *big_out = has_big;
  if (inv_out) *inv_out = inv;
  *ptr_out = ptr;
  *list_out = list;
}

// vertex -> incidence lists of a mesh (built once per mesh), and the position
// of every (element, local vertex) item in them
void build_v2e(ffhip_mesh m) {
  if (m->v2e_ptr) return;
  build_incidence(m->ctx, m->elems, m->nt, m->nloc, m->nv, &m->v2e_ptr, &m->v2e, &m->v2e_big,
                  nullptr, nullptr, nullptr);
}

// As build_v2e, but where every list fits its 32-entry bucket the buckets are
// returned unsorted and m->v2e is left unfilled: the caller must sort them
// into m->v2e (k_pattern_half with the buckets does, k_v2e_sort_bucket
// otherwise) and free the buckets before anything else reads m->v2e.
// With sc (a tetrahedral mesh), the incidence build also computes the
// element scales (*scaled = true); when the lists exist already it does not.
// ovf (device int): raised when some list exceeds its bucket; the caller
// reads it and then builds the lists with v2e_fill_sort instead.
int32_t *build_v2e_unsorted(ffhip_mesh m, const ScaleArgs *sc, bool *scaled, int *ovf) {
  *scaled = false;
  if (m->v2e_ptr) return nullptr;
  int32_t *bucket = nullptr;
  build_incidence(m->ctx, m->elems, m->nt, m->nloc, m->nv, &m->v2e_ptr, &m->v2e, &m->v2e_big,
                  nullptr, &bucket, sc, ovf);
  *scaled = sc && m->nloc == 4;
  return bucket;
}

// the position of every (element, local vertex) item in the incidence lists
// (built on first use: only the element-row assembly path scatters by it)
void build_v2e_inv(ffhip_mesh m) {
  build_v2e(m);
  if (m->v2e_inv) return;
  const int64_t M = m->nt * m->nloc;
  m->v2e_inv = dalloc<int32_t>(M);
  k_v2e_inverse<<<nblocks(M, 256), 256, 0, m->ctx->stream>>>(M, m->v2e, m->v2e_inv);
  FFHIP_CHECK(hipGetLastError());
}

// a_ii = tgv on the marked rows (HashMatrix::SetBC); *missing set when a
// marked row has no diagonal slot
void set_diag_rows(ffhip_ctx ctx, int64_t n, const uint8_t *onbc, const int64_t *diag, double tgv,
                   double *vals, int *missing) {
  k_set_diag<<<nblocks(n, 256), 256, 0, ctx->stream>>>(n, onbc, diag, tgv, vals, missing);
  FFHIP_CHECK(hipGetLastError());
}

// tmap[k] = slot of the transposed entry; false if the pattern is not symmetric
bool transpose_map(ffhip_ctx ctx, ffhip_mat A, int64_t *tmap) {
  int *missing = dalloc<int>(1);
  clear(ctx, {{missing, sizeof(int)}});
  k_transpose_map<<<nblocks(A->n, 256), 256, 0, ctx->stream>>>(A->n, A->rowptr, A->colidx, tmap,
                                                                missing);
  FFHIP_CHECK(hipGetLastError());
  const int miss = read_flag(ctx, missing);
  dfree(missing);
  return miss == 0;
}

// ---------------------------------------------------------------- misfit
// J = 1/2 int (u - ud)^2 (partials of kMisfitBlocks blocks, summed on the host
// in block order; they go to page-locked memory) and r = M (u - ud) with the
// Dirichlet rows zeroed, on the given buffers: onbc (nv bytes, when r and
// nlab > 0), labs (nlab int32, where there are more labels than kernels take
// by value), pair (nt, when r; without it r's terms are formed per incidence)
constexpr int kMisfitBlocks = 1024;
static_assert(8 * kMisfitBlocks <= ffhip_ctx_s::kPinnedData, "page-locked partials");
struct MisfitBuffers {
  uint8_t *onbc = nullptr;
  int32_t *labs = nullptr;
  double2 *pair = nullptr;
};

// the vertices of the boundary elements with these labels
void mark_bc(ffhip_ctx ctx, ffhip_mesh m, const Labels &labels, uint8_t *onbc) {
  clear(ctx, {{onbc, (size_t)m->nv}});
  if (m->nbe)
    k_mark_bc<<<nblocks(m->nbe, 256), 256, 0, ctx->stream>>>(m->nbe, m->nbloc, m->belems, m->blab, labels, onbc);
  FFHIP_CHECK(hipGetLastError());
}

void misfit_run(ffhip_ctx ctx, ffhip_mesh m, const double *u, const double *ud,
                const int32_t *labels, int nlab, double *J, double *r, const MisfitBuffers &b) {
  hipStream_t s = ctx->stream;
  ctx->tic();
  double *part = J ? static_cast<double *>(ctx->pinned_data()) : nullptr;
  if (J || b.pair) {
    k_p1_misfit_elem<<<kMisfitBlocks, 256, 0, s>>>(m->nt, m->xyz, m->elems, u, ud, part, b.pair);
    FFHIP_CHECK(hipGetLastError());
  }
  if (r) {
    const uint8_t *onbc = nullptr;
    if (nlab > 0) {
      mark_bc(ctx, m, LabelArg(ctx, labels, nlab, b.labs).L, b.onbc);
      onbc = b.onbc;
    }
    if (b.pair) {
      auto sum = few_rows(m->nv) ? k_row_sum<kRowPair, 16> : k_row_sum<kRowPair, 64>;
      sum<<<row_grid(m->nv, few_rows(m->nv) ? 16 : 64), kWave, 0, s>>>(
          m->nv, m->v2e_ptr, m->v2e, reinterpret_cast<const double *>(b.pair), u, ud, onbc, 0., 0.,
          nullptr, r, RowPart{});
    } else
      k_p1_mass_apply<<<nblocks(m->nv * kHalf, 256), 256, 0, s>>>(m->nv, m->xyz, m->elems, m->v2e_ptr,
                                                                  m->v2e, u, ud, onbc, r);
    FFHIP_CHECK(hipGetLastError());
  }
  ctx->toc();
  if (J) {
    double tot = 0.;
    for (int i = 0; i < kMisfitBlocks; ++i) tot += part[i];
    *J = tot;
  }
}

// ---------------------------------------------------------------- no-allocation scratch
// The scratch of ffhip_p1_misfit_noalloc: a file-scope device array, one copy
// per device, reached through the address hipGetSymbolAddress gives on that
// device (the array's name is a host-side stand-in in host code).  Layout:
// labels | Dirichlet marks.  Every call on a device shares
// it: overlapping calls on one device race.
constexpr int64_t kNoallocMaxVertices = (int64_t)1 << 24;
constexpr int kNoallocMaxLabels = 64;
constexpr size_t kScratchLabelsOff = 0;
constexpr size_t kScratchOnbcOff = kScratchLabelsOff + 4 * kNoallocMaxLabels;
constexpr size_t kScratchBytes = kScratchOnbcOff + (size_t)kNoallocMaxVertices;
constexpr int kMaxDevices = 64;

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

std::mutex &scratch_mutex() {
  static std::mutex mu;
  return mu;
}
unsigned char *&scratch_ptr(int device) {
  static unsigned char *ptr[kMaxDevices] = {};
  return ptr[device];
}

// resolves the device address of the scratch array on `device`, which must be
// the current device (called by ffhip_init, once per device)
void noalloc_scratch_setup(int device) {
  FFHIP_REQUIRE(device >= 0 && device < kMaxDevices, FFHIP_ERR_UNSUPPORTED, "device %d", device);
  std::lock_guard<std::mutex> g(scratch_mutex());
  if (scratch_ptr(device)) return;
  void *p = nullptr;
  FFHIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  scratch_ptr(device) = static_cast<unsigned char *>(p);
}

unsigned char *noalloc_scratch(int device) {
  std::lock_guard<std::mutex> g(scratch_mutex());
  unsigned char *p = (device >= 0 && device < kMaxDevices) ? scratch_ptr(device) : nullptr;
  FFHIP_REQUIRE(p, FFHIP_ERR_INTERNAL, "no-allocation scratch not set up on device %d", device);
  return p;
}

// The P1 pattern (ffhip_pattern_p1).  With Ce (3D: the element scales,
// computed from sc by the incidence build, or by k_p1_scale_3d when the
// mesh's lists exist) the half-wave pattern pass also forms the values of
// the rows it builds; *values_done tells whether that covered every row (no
// lane-per-row rows).
//
// First try: the row pointers from the vertex-link counts (k_link_len), the
// pattern pass writing straight to CSR.  If some row is not what they
// predict, or needs the lane-per-row kernels, the buffered passes run.
ffhip_mat pattern_p1(ffhip_ctx ctx, ffhip_mesh m, const double *Ce, bool *values_done,
                     const ScaleArgs *sc) {
  hipStream_t s = ctx->stream;
  const bool vals_pass = Ce && m->nloc == 4;
  // the fused pass sorts the incidence buckets into the lists itself; with
  // sc the incidence build computes the element scales Ce as well (or, on a
  // mesh whose lists exist, k_p1_scale_3d does)
  int32_t *bucket = nullptr;
  int *ovf = nullptr;  // bucket overflow, read back with the row pointers
  if (vals_pass) {
    bool scaled = false;
    ovf = dalloc<int>(1);
    clear(ctx, {{ovf, sizeof(int)}});
    bucket = build_v2e_unsorted(m, sc, &scaled, ovf);
    if (sc && !scaled) {
      k_p1_scale_3d<<<nblocks(m->nt, 256), 256, 0, s>>>(m->nt, sc->xyz, m->elems, sc->kind, sc->c0,
                                                        sc->kappa_e, sc->Ce);
      FFHIP_CHECK(hipGetLastError());
    }
  } else {
    build_v2e(m);
  }
  const int64_t n = m->nv;
  ffhip_mat A = new ffhip_mat_s();
  A->ctx = ctx; A->n = n; A->mesh = m;
  // the lists sorted from the buckets by k_v2e_sort_bucket (when the fused
  // pass did not run, or not for every row)
  auto sort_buckets = [&] {
    if (!bucket) return;
    k_v2e_sort_bucket<<<nblocks(n * kHalf, 256), 256, 0, s>>>(n, m->v2e_ptr, bucket, m->v2e, nullptr);
    FFHIP_CHECK(hipGetLastError());
    dfree(bucket);
  };
  try {
    A->rowptr = dalloc<int64_t>(n + 1);
    A->diag = dalloc<int64_t>(n);
    A->slotmap = dalloc<uint32_t>(m->nt * m->nloc);
    A->big = dalloc<uint8_t>(n);
    bool direct_ok = false;
    {  // direct pass
      Arena ar(ctx, Arena::bytes(n, 4) + Arena::bytes(n + 1, 8) + Arena::bytes(2, 4));
      uint32_t *bcnt = ar.take<uint32_t>(n);
      int64_t *len = ar.take<int64_t>(n + 1);
      int *flags = ar.take<int>(2);  // any big row, any row unlike its link count
      clear(ctx, {{bcnt, 4 * (size_t)n}, {flags, 2 * sizeof(int)}});
      if (m->nbe)
        k_bcount<<<nblocks(m->nbe * m->nbloc, 256), 256, 0, s>>>(m->nbe * m->nbloc, m->belems, bcnt);
      k_link_len<<<nblocks(n, 256), 256, 0, s>>>(n, m->dim, m->v2e_ptr, bcnt, len);
      FFHIP_CHECK(hipGetLastError());
      exclusive_scan_i64(ctx, len, A->rowptr, n + 1);
      if (bucket) {  // the entry count and the bucket overflow flag in one wait
        int64_t nnz = 0;
        int of = 0;
        fetch(ctx, {{&nnz, A->rowptr + n, sizeof(nnz)}, {&of, ovf, sizeof(of)}});
        A->nnz = nnz;
        if (of) {  // some list exceeds its bucket: the lists by the atomic fill
          dfree(bucket);
          v2e_fill_sort(ctx, m->elems, m->nt * m->nloc, n, m->v2e_ptr, m->v2e, nullptr);
          m->v2e_big = 1;
        }
      } else {
        A->nnz = read_i64(ctx, A->rowptr + n);
      }
      A->colidx = dalloc<int32_t>(A->nnz);
      A->vals = dalloc<double>(A->nnz);
      PatternOut out;
      out.rowptr = A->rowptr; out.colidx = A->colidx; out.diag = A->diag; out.vals = A->vals;
      out.mismatch = flags + 1;
      if (vals_pass)
        k_pattern_half<4, true, true><<<nblocks(n * kHalf, 256), 256, 0, s>>>(
            n, m->elems, m->v2e_ptr, m->v2e, A->slotmap, A->big, flags, out, m->xyz, Ce, bucket);
      else if (m->nloc == 4)
        k_pattern_half<4, false, true><<<nblocks(n * kHalf, 256), 256, 0, s>>>(
            n, m->elems, m->v2e_ptr, m->v2e, A->slotmap, A->big, flags, out);
      else
        k_pattern_half<3, false, true><<<nblocks(n * kHalf, 256), 256, 0, s>>>(
            n, m->elems, m->v2e_ptr, m->v2e, A->slotmap, A->big, flags, out);
      FFHIP_CHECK(hipGetLastError());
      int h[2] = {0, 0};
      fetch(ctx, {{h, flags, sizeof(h)}});
      direct_ok = !h[0] && !h[1];
      if (!direct_ok) { dfree(A->colidx); dfree(A->vals); }
      if (direct_ok) dfree(bucket);  // every list sorted by the pass
      else sort_buckets();
      dfree(ovf);
    }
    if (direct_ok) {
      if (!vals_pass) FFHIP_CHECK(hipMemsetAsync(A->vals, 0, 8 * A->nnz, s));
      A->any_big = 0;
      A->max_row = kRowBuf;
      if (values_done) *values_done = vals_pass;
      return A;
    }
    // buffered passes
    Arena ar(ctx, Arena::bytes(n + 1, 8) + Arena::bytes(1, 4) + Arena::bytes(kRowBuf * n, 4) +
                      Arena::bytes(n, 1) + Arena::bytes(1, 4) +
                      (vals_pass ? Arena::bytes(kRowBuf * n, 8) : 0));
    int64_t *len = ar.take<int64_t>(n + 1);
    int *ovf = ar.take<int>(1);
    FFHIP_CHECK(hipMemsetAsync(len, 0, 8 * (n + 1), s));
    FFHIP_CHECK(hipMemsetAsync(ovf, 0, sizeof(int), s));
    // rows with up to 32 incident elements and 64 columns: one half-wave
    // pass into row buffers (big = 0); the rest: the lane-per-row merge with
    // 64 LDS columns per lane (big = 1), then with 256 (big = 2: the slot
    // offsets of the element-to-row map are bytes)
    constexpr int B = 128, CAP = 64, BW = 32, CAPW = 256;
    PatternOut out;
    out.rowlen = len;
    out.rowbuf = ar.take<int32_t>(kRowBuf * n);
    out.dposr = ar.take<int8_t>(n);
    int *anyb = ar.take<int>(1);
    out.rowval = vals_pass ? ar.take<double>(kRowBuf * n) : nullptr;
    FFHIP_CHECK(hipMemsetAsync(anyb, 0, sizeof(int), s));
    if (vals_pass)
      k_pattern_half<4, true, false><<<nblocks(n * kHalf, 256), 256, 0, s>>>(
          n, m->elems, m->v2e_ptr, m->v2e, A->slotmap, A->big, anyb, out, m->xyz, Ce);
    else if (m->nloc == 4)
      k_pattern_half<4, false, false><<<nblocks(n * kHalf, 256), 256, 0, s>>>(
          n, m->elems, m->v2e_ptr, m->v2e, A->slotmap, A->big, anyb, out);
    else
      k_pattern_half<3, false, false><<<nblocks(n * kHalf, 256), 256, 0, s>>>(
          n, m->elems, m->v2e_ptr, m->v2e, A->slotmap, A->big, anyb, out);
    FFHIP_CHECK(hipGetLastError());
    A->any_big = read_flag(ctx, anyb);
    bool wide = false;
    if (A->any_big) {
      k_pattern_rows<B, CAP, false><<<nblocks(n, B), B, 0, s>>>(
          n, m->nloc, m->elems, m->v2e_ptr, m->v2e, len, nullptr, nullptr, nullptr, nullptr,
          nullptr, ovf, A->big, 1);
      FFHIP_CHECK(hipGetLastError());
      wide = read_flag(ctx, ovf) != 0;
    }
    if (wide) {
      FFHIP_CHECK(hipMemsetAsync(ovf, 0, sizeof(int), s));
      k_pattern_rows<BW, CAPW, false><<<nblocks(n, BW), BW, 0, s>>>(
          n, m->nloc, m->elems, m->v2e_ptr, m->v2e, len, nullptr, nullptr, nullptr, nullptr,
          nullptr, ovf, A->big, 2);
      FFHIP_CHECK(hipGetLastError());
      FFHIP_REQUIRE(read_flag(ctx, ovf) == 0, FFHIP_ERR_UNSUPPORTED,
                    "ffhip_pattern_p1: a row has more than %d columns", CAPW);
    }
    exclusive_scan_i64(ctx, len, A->rowptr, n + 1);
    A->nnz = read_i64(ctx, A->rowptr + n);
    A->colidx = dalloc<int32_t>(A->nnz);
    A->vals = dalloc<double>(A->nnz);
    k_pattern_compact<<<nblocks(n, 256), 256, 0, s>>>(n, A->rowptr, out.rowbuf, out.dposr, A->big,
                                                      A->colidx, A->diag, out.rowval,
                                                      vals_pass ? A->vals : nullptr);
    if (A->any_big)
      k_pattern_rows<B, CAP, true><<<nblocks(n, B), B, 0, s>>>(
          n, m->nloc, m->elems, m->v2e_ptr, m->v2e, nullptr, A->rowptr, A->colidx, A->diag,
          A->slotmap, nullptr, ovf, A->big, 1);
    if (wide)
      k_pattern_rows<BW, CAPW, true><<<nblocks(n, BW), BW, 0, s>>>(
          n, m->nloc, m->elems, m->v2e_ptr, m->v2e, nullptr, A->rowptr, A->colidx, A->diag,
          A->slotmap, nullptr, ovf, A->big, 2);
    FFHIP_CHECK(hipGetLastError());
    if (!vals_pass) FFHIP_CHECK(hipMemsetAsync(A->vals, 0, 8 * A->nnz, s));
    if (values_done) *values_done = vals_pass && !A->any_big;
    A->max_row = wide ? CAPW : CAP;
  } catch (...) {
    (void)hipStreamSynchronize(s);
    dfree(ovf);
    if (bucket) {  // the lists were never sorted: the mesh builds them again when next needed
      dfree(bucket);
      dfree(m->v2e_ptr);
      dfree(m->v2e);
    }
    dfree(A->rowptr); dfree(A->colidx); dfree(A->vals); dfree(A->diag);
    dfree(A->slotmap); dfree(A->big);
    delete A;
    throw;
  }
  return A;
}

}  // namespace ffhip

using namespace ffhip;

extern "C" {

int ffhip_pattern_p1(ffhip_ctx ctx, ffhip_mesh m, ffhip_mat *out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && m && out, FFHIP_ERR_ARG, "ffhip_pattern_p1: null argument");
    FFHIP_REQUIRE(m->nloc <= 4, FFHIP_ERR_UNSUPPORTED, "ffhip_pattern_p1: P1 on simplices only");
    ctx->tic();
    ffhip_mat A = pattern_p1(ctx, m, nullptr, nullptr, nullptr);
    ctx->toc();
    *out = A;
  });
}

int ffhip_pattern_assemble_p1(ffhip_ctx ctx, ffhip_mesh m, int kind, double c0, const double *kappa_e,
                              int kappa_on_device, ffhip_mat *out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && m && out, FFHIP_ERR_ARG, "ffhip_pattern_assemble_p1: null argument");
    FFHIP_REQUIRE(m->dim == 3 && m->nloc == 4, FFHIP_ERR_UNSUPPORTED,
                  "ffhip_pattern_assemble_p1: 3D P1 meshes (2D: ffhip_pattern_p1 + ffhip_assemble_p1)");
    FFHIP_REQUIRE(kind == FFHIP_COEF_CONST || kind == FFHIP_COEF_SIN3 || kind == FFHIP_COEF_P0 ||
                      kind == FFHIP_COEF_QP || kind == FFHIP_COEF_P1,
                  FFHIP_ERR_ARG, "ffhip_pattern_assemble_p1: coefficient kind %d", kind);
    const bool arr = kind == FFHIP_COEF_P0 || kind == FFHIP_COEF_QP || kind == FFHIP_COEF_P1;
    FFHIP_REQUIRE(!arr || kappa_e, FFHIP_ERR_ARG, "ffhip_pattern_assemble_p1: kappa_e");
    hipStream_t s = ctx->stream;
    const double *kd = kappa_e;
    double *kbuf = nullptr, *Ce = nullptr;
    ffhip_mat A = nullptr;
    try {
      if (arr && !kappa_on_device) {
        const int64_t cnt = kind == FFHIP_COEF_P1 ? m->nv : kind == FFHIP_COEF_P0 ? m->nt : 14 * m->nt;
        kbuf = dalloc<double>(cnt);
        FFHIP_CHECK(hipMemcpyAsync(kbuf, kappa_e, 8 * cnt, hipMemcpyHostToDevice, s));
        kd = kbuf;
      }
      Ce = dalloc<double>(m->nt);
      ctx->tic();
      // the element scales are computed by the incidence build (one pass:
      // the coefficient at 14 points per tet hides the atomics' round trips),
      // then the pattern pass forms the row values from them
      const ScaleArgs sc{m->xyz, kind, c0, kd, Ce};
      bool done = false;
      A = pattern_p1(ctx, m, Ce, &done, &sc);
      ctx->toc();
      if (!done) {  // rows for the lane-per-row kernels: all values by the element-row path
        const int rc = ffhip_assemble_p1(ctx, m, A, kind, c0, kd, 1);
        FFHIP_REQUIRE(rc == FFHIP_OK, rc, "ffhip_pattern_assemble_p1: %s", ffhip_last_error());
      }
    } catch (...) {
      (void)hipStreamSynchronize(s);
      dfree(Ce); dfree(kbuf);
      if (A) ffhip_mat_free(A);
      throw;
    }
    dfree(Ce); dfree(kbuf);
    *out = A;
  });
}

int ffhip_mat_info(ffhip_mat A, int64_t *n, int64_t *nnz) {
  return guard([&] {
    FFHIP_REQUIRE(A, FFHIP_ERR_ARG, "ffhip_mat_info: null matrix");
    if (n) *n = A->n;
    if (nnz) *nnz = A->nnz;
  });
}

int ffhip_assemble_p1(ffhip_ctx ctx, ffhip_mesh m, ffhip_mat A, int kind, double c0,
                      const double *kappa_e, int kappa_on_device) {
  return ffhip_assemble_p1_form(ctx, m, A, kind, c0, kappa_e, FFHIP_COEF_NONE, 0., nullptr,
                                kappa_on_device);
}

int ffhip_assemble_p1_form(ffhip_ctx ctx, ffhip_mesh m, ffhip_mat A, int kind, double c0,
                           const double *kappa_e, int mkind, double m0, const double *mass_e,
                           int on_device) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && m && A && A->mesh == m && A->slotmap, FFHIP_ERR_ARG,
                  "ffhip_assemble_p1: matrix pattern was not built from this mesh");
    auto valid = [](int k) {
      return k == FFHIP_COEF_CONST || k == FFHIP_COEF_SIN3 || k == FFHIP_COEF_P0 ||
             k == FFHIP_COEF_QP || k == FFHIP_COEF_P1;
    };
    FFHIP_REQUIRE(valid(kind), FFHIP_ERR_ARG, "ffhip_assemble_p1: coefficient kind %d", kind);
    FFHIP_REQUIRE(mkind == FFHIP_COEF_NONE || valid(mkind), FFHIP_ERR_ARG,
                  "ffhip_assemble_p1_form: mass coefficient kind %d", mkind);
    auto is_array = [](int k) {
      return k == FFHIP_COEF_P0 || k == FFHIP_COEF_QP || k == FFHIP_COEF_P1;
    };
    const bool arr = is_array(kind), marr = is_array(mkind);
    FFHIP_REQUIRE(!arr || kappa_e, FFHIP_ERR_ARG, "ffhip_assemble_p1: kappa_e");
    FFHIP_REQUIRE(!marr || mass_e, FFHIP_ERR_ARG, "ffhip_assemble_p1_form: mass_e");
    const int kappa_on_device = on_device;
    hipStream_t s = ctx->stream;
    const int nu = m->nloc == 4 ? 10 : 6;
    // 3D stiffness without a reaction term and with every row in the
    // half-wave kernels: element scales, then rows formed from the vertices.
    // Otherwise the element rows in incidence order (3D), and Ke for the
    // lane-per-row gather of long rows and 2D.
    const bool rows_path = m->dim == 3 && mkind == FFHIP_COEF_NONE && !A->any_big;
    const bool needKe = m->nloc != 4 || A->any_big;
    Arena ar(ctx, (rows_path ? Arena::bytes(m->nt, 8) : 0) +
                      (!rows_path && m->dim == 3 ? Arena::bytes(16 * m->nt, 8) : 0) +
                      (needKe ? Arena::bytes(nu * m->nt, 8) : 0));
    double *Ke = needKe ? ar.take<double>(nu * m->nt) : nullptr;
    const double *kd = kappa_e, *md = mass_e;
    double *kbuf = nullptr, *mbuf = nullptr;
    auto count = [&](int k) {
      return k == FFHIP_COEF_P1 ? m->nv : k == FFHIP_COEF_P0 ? m->nt : m->nt * (m->dim == 3 ? 14 : 7);
    };
    if (arr && !kappa_on_device) {
      const int64_t cnt = count(kind);
      kbuf = dalloc<double>(cnt);
      FFHIP_CHECK(hipMemcpyAsync(kbuf, kappa_e, 8 * cnt, hipMemcpyHostToDevice, s));
      kd = kbuf;
    }
    if (marr && !on_device) {
      const int64_t cnt = count(mkind);
      mbuf = dalloc<double>(cnt);
      FFHIP_CHECK(hipMemcpyAsync(mbuf, mass_e, 8 * cnt, hipMemcpyHostToDevice, s));
      md = mbuf;
    }
    if (m->dim == 2) upload_t5_once(ctx->device);
    if (!rows_path && m->dim == 3) build_v2e_inv(m);
    ctx->tic();
    double *Kinc = nullptr;
    if (rows_path) {
      double *Ce = ar.take<double>(m->nt);
      k_p1_scale_3d<<<nblocks(m->nt, 256), 256, 0, s>>>(m->nt, m->xyz, m->elems, kind, c0, kd, Ce);
      const int64_t g = (nblocks(A->n * kHalf, 256) + 7) / 8 * 8;  // a multiple of the 8 XCDs
      k_p1_values_rows<<<(unsigned)g, 256, 0, s>>>(A->n, A->rowptr, m->v2e_ptr, m->v2e, A->slotmap,
                                                   m->xyz, m->elems, Ce, A->big, A->vals);
    } else if (m->dim == 3) {
      Kinc = ar.take<double>(16 * m->nt);
      if (mkind == FFHIP_COEF_NONE)
        k_p1_element_3d<false><<<nblocks(m->nt, 256), 256, 0, s>>>(
            m->nt, m->xyz, m->elems, kind, c0, kd, mkind, m0, md, m->v2e_inv, Kinc,
            A->any_big ? Ke : nullptr);
      else
        k_p1_element_3d<true><<<nblocks(m->nt, 256), 256, 0, s>>>(
            m->nt, m->xyz, m->elems, kind, c0, kd, mkind, m0, md, m->v2e_inv, Kinc,
            A->any_big ? Ke : nullptr);
    } else
      k_p1_element_2d<<<nblocks(m->nt, 256), 256, 0, s>>>(m->nt, m->xyz, m->elems, kind, c0, kd,
                                                           mkind, m0, md, Ke);
    constexpr int B = 256, STAGE = 6144;
    if (!rows_path && m->nloc == 4) {
      k_p1_values_half<<<nblocks(A->n * kHalf, 256), 256, 0, s>>>(
          A->n, A->rowptr, m->v2e_ptr, A->slotmap, Kinc, A->big, A->vals);
      if (A->any_big)
        k_p1_gather<B, STAGE, 4><<<nblocks(A->n, B), B, 0, s>>>(
            A->n, A->rowptr, m->v2e_ptr, m->v2e, A->slotmap, Ke, A->vals, A->big);
    } else if (m->nloc == 3) {
      k_p1_gather<B, STAGE, 3><<<nblocks(A->n, B), B, 0, s>>>(A->n, A->rowptr, m->v2e_ptr, m->v2e,
                                                               A->slotmap, Ke, A->vals);
    }
    FFHIP_CHECK(hipGetLastError());
    ctx->toc();
    dfree(kbuf);
    dfree(mbuf);
  });
}

int ffhip_set_bc(ffhip_ctx ctx, ffhip_mesh m, ffhip_mat A, const int32_t *labels, int nlab,
                 double tgv, uint8_t *onbc_out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && m && A && A->n == m->nv, FFHIP_ERR_ARG, "ffhip_set_bc: bad arguments");
    FFHIP_REQUIRE(nlab >= 0 && (nlab == 0 || labels), FFHIP_ERR_ARG, "ffhip_set_bc: labels");
    FFHIP_REQUIRE(tgv > 0, FFHIP_ERR_UNSUPPORTED, "ffhip_set_bc: only tgv > 0 is supported");
    hipStream_t s = ctx->stream;
    uint8_t *onbc = dalloc<uint8_t>(A->n);
    const LabelArg labs(ctx, labels, nlab);
    int *missing = ctx->flag(0);
    ctx->tic();
    mark_bc(ctx, m, labs.L, onbc);
    k_set_diag<<<nblocks(A->n, 256), 256, 0, s>>>(A->n, onbc, A->diag, tgv, A->vals, missing);
    FFHIP_CHECK(hipGetLastError());
    ctx->toc();
    if (onbc_out) FFHIP_CHECK(hipMemcpy(onbc_out, onbc, A->n, hipMemcpyDeviceToHost));
    const int miss = *missing;
    dfree(onbc);
    FFHIP_REQUIRE(miss == 0, FFHIP_ERR_INTERNAL, "ffhip_set_bc: a Dirichlet row has no diagonal");
  });
}

int ffhip_rhs_p1_form(ffhip_ctx ctx, ffhip_mesh m, int kind, double f0, const double *fcoef,
                      const int32_t *labels, int nlab, double tgv, double g0, const double *gvals,
                      double *b, int on_device) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && m && b, FFHIP_ERR_ARG, "ffhip_rhs_p1: bad arguments");
    FFHIP_REQUIRE(kind == FFHIP_COEF_CONST || kind == FFHIP_COEF_SIN3 || kind == FFHIP_COEF_P0 ||
                      kind == FFHIP_COEF_QP || kind == FFHIP_COEF_P1,
                  FFHIP_ERR_ARG, "ffhip_rhs_p1_form: coefficient kind");
    const bool arr = kind == FFHIP_COEF_P0 || kind == FFHIP_COEF_QP || kind == FFHIP_COEF_P1;
    FFHIP_REQUIRE(!arr || fcoef, FFHIP_ERR_ARG, "ffhip_rhs_p1_form: coefficient array missing");
    hipStream_t s = ctx->stream;
    build_v2e(m);
    const int64_t n = m->nv;
    uint8_t *onbc = nullptr;
    const LabelArg labs(ctx, labels, nlab > 0 ? nlab : 0);
    if (nlab > 0) {
      onbc = dalloc<uint8_t>(n);
      mark_bc(ctx, m, labs.L, onbc);
    }
    double *bd = on_device ? b : dalloc<double>(n);
    const double *fd = fcoef, *gd = gvals;
    double *fown = nullptr, *gown = nullptr;
    if (arr && !on_device) {
      const int64_t cnt = kind == FFHIP_COEF_P1   ? m->nv
                          : kind == FFHIP_COEF_P0 ? m->nt
                                                  : m->nt * (m->dim == 3 ? 14 : 7);
      fown = dalloc<double>(cnt);
      FFHIP_CHECK(hipMemcpyAsync(fown, fcoef, 8 * cnt, hipMemcpyHostToDevice, s));
      fd = fown;
    }
    if (gvals && !on_device) {
      gown = dalloc<double>(n);
      FFHIP_CHECK(hipMemcpyAsync(gown, gvals, 8 * n, hipMemcpyHostToDevice, s));
      gd = gown;
    }
    if (m->dim == 2) upload_t5_once(ctx->device);
    // 3D: one pass over the tets, then one over the rows; part by part where a
    // device has no room for every tet's terms (8 to 32 bytes each)
    const int rm = kind == FFHIP_COEF_P1 ? kRowPair
                   : kind == FFHIP_COEF_SIN3 || kind == FFHIP_COEF_QP ? kRowQuad : kRowScale;
    const int ed = rm == kRowPair ? 2 : rm == kRowQuad ? 4 : 1;
    double *E = nullptr;
    int64_t part = m->nt;
    while (m->dim == 3 && !E) {
      try {
        E = dalloc<double>(part * ed);
      } catch (const Error &) {
        if (part <= 256) throw;
        part = (part + 1) / 2;
      }
    }
    ctx->tic();
    if (m->dim == 3) {
#define FFHIP_RHS(RM)                                                                              \
  do {                                                                                             \
    int64_t e0 = 0;                                                                                \
    do {                                                                                           \
      const int64_t cnt = m->nt - e0 < part ? m->nt - e0 : part;                                   \
      const double *fe = !fd || kind == FFHIP_COEF_P1 ? fd                                         \
                                                      : fd + e0 * (kind == FFHIP_COEF_QP ? 14 : 1); \
      k_p1_load_elem<RM><<<nblocks(cnt, 256), 256, 0, s>>>(cnt, m->xyz, m->elems + 4 * e0, kind, f0, fe, E); \
      auto sum = part < m->nt ? k_row_sum<RM, 64, true>                                            \
                 : few_rows(n) ? k_row_sum<RM, 16> : k_row_sum<RM, 64>;                            \
      sum<<<row_grid(n, part == m->nt && few_rows(n) ? 16 : 64), kWave, 0, s>>>(                   \
          n, m->v2e_ptr, m->v2e, E, fd, nullptr, onbc, tgv, g0, gd, bd, RowPart{e0, e0 + cnt, m->nt}); \
    } while ((e0 += part) < m->nt);                                                                \
  } while (0)
      if (rm == kRowScale) FFHIP_RHS(kRowScale);
      else if (rm == kRowPair) FFHIP_RHS(kRowPair);
      else FFHIP_RHS(kRowQuad);
#undef FFHIP_RHS
    } else
      k_rhs_p1_2d<<<nblocks(n, 256), 256, 0, s>>>(n, m->xyz, m->elems, m->v2e_ptr, m->v2e, kind, f0,
                                                   fd, onbc, tgv, g0, gd, bd);
    FFHIP_CHECK(hipGetLastError());
    ctx->toc();
    if (!on_device) {
      FFHIP_CHECK(hipMemcpy(b, bd, 8 * n, hipMemcpyDeviceToHost));
      dfree(bd);
    }
    FFHIP_CHECK(hipStreamSynchronize(s));
    dfree(onbc);
    dfree(fown);
    dfree(gown);
    dfree(E);
  });
}

int ffhip_rhs_p1(ffhip_ctx ctx, ffhip_mesh m, double f, const int32_t *labels, int nlab,
                 double tgv, double g, double *b, int on_device) {
  return ffhip_rhs_p1_form(ctx, m, FFHIP_COEF_CONST, f, nullptr, labels, nlab, tgv, g, nullptr, b,
                           on_device);
}

int ffhip_p1_misfit(ffhip_ctx ctx, ffhip_mesh m, const double *u, const double *ud,
                    const int32_t *labels, int nlab, double *J, double *r) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && m && u && ud && m->dim == 3, FFHIP_ERR_ARG, "ffhip_p1_misfit: bad arguments");
    FFHIP_REQUIRE(nlab >= 0 && (nlab == 0 || labels), FFHIP_ERR_ARG, "ffhip_p1_misfit: labels");
    build_v2e(m);
    MisfitBuffers b;
    try {
      if (r && nlab > 0) {
        b.onbc = dalloc<uint8_t>(m->nv);
        b.labs = dalloc<int32_t>(nlab);
      }
      if (r) {
        try {
          b.pair = dalloc<double2>(m->nt);
        } catch (const Error &) {  // no room for the pairs: r without them, the same bits
        }
      }
      misfit_run(ctx, m, u, ud, labels, nlab, J, r, b);
    } catch (...) {
      (void)hipStreamSynchronize(ctx->stream);
      dfree(b.onbc); dfree(b.labs); dfree(b.pair);
      throw;
    }
    dfree(b.onbc); dfree(b.labs); dfree(b.pair);
  });
}

int ffhip_p1_misfit_noalloc(ffhip_ctx ctx, ffhip_mesh m, const double *u, const double *ud,
                            const int32_t *labels, int nlab, double *J, double *r) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && m && u && ud && m->dim == 3, FFHIP_ERR_ARG,
                  "ffhip_p1_misfit_noalloc: bad arguments");
    FFHIP_REQUIRE(nlab >= 0 && (nlab == 0 || labels), FFHIP_ERR_ARG, "ffhip_p1_misfit_noalloc: labels");
    FFHIP_REQUIRE(m->nv <= kNoallocMaxVertices, FFHIP_ERR_ARG,
                  "ffhip_p1_misfit_noalloc: %lld vertices, more than its maximum %lld",
                  (long long)m->nv, (long long)kNoallocMaxVertices);
    FFHIP_REQUIRE(nlab <= kNoallocMaxLabels, FFHIP_ERR_ARG,
                  "ffhip_p1_misfit_noalloc: %d labels, more than its maximum %d", nlab, kNoallocMaxLabels);
    FFHIP_REQUIRE(!r || m->v2e_ptr, FFHIP_ERR_ARG,
                  "ffhip_p1_misfit_noalloc: the mesh's vertex incidence is not built yet (an assembly "
                  "or ffhip_p1_misfit on this mesh builds it; this entry point allocates nothing)");
    unsigned char *base = noalloc_scratch(ctx->device);
    MisfitBuffers b;
    b.labs = reinterpret_cast<int32_t *>(base + kScratchLabelsOff);
    b.onbc = base + kScratchOnbcOff;
    misfit_run(ctx, m, u, ud, labels, nlab, J, r, b);
  });
}

int ffhip_p1_grad_kappa(ffhip_ctx ctx, ffhip_mesh m, const double *u, const double *lambda,
                        double *g) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && m && u && lambda && g && m->dim == 3, FFHIP_ERR_ARG,
                  "ffhip_p1_grad_kappa: bad arguments");
    ctx->tic();
    k_p1_grad_kappa<<<nblocks(m->nt, 256), 256, 0, ctx->stream>>>(m->nt, m->xyz, m->elems, u, lambda, g);
    FFHIP_CHECK(hipGetLastError());
    ctx->toc();
  });
}

int ffhip_mat_download(ffhip_mat A, int64_t *rowptr, int32_t *colidx, double *vals) {
  return guard([&] {
    FFHIP_REQUIRE(A, FFHIP_ERR_ARG, "ffhip_mat_download: null matrix");
    hipStream_t s = A->ctx->stream;
    if (rowptr) FFHIP_CHECK(hipMemcpyAsync(rowptr, A->rowptr, 8 * (A->n + 1), hipMemcpyDeviceToHost, s));
    if (colidx) FFHIP_CHECK(hipMemcpyAsync(colidx, A->colidx, 4 * A->nnz, hipMemcpyDeviceToHost, s));
    if (vals) FFHIP_CHECK(hipMemcpyAsync(vals, A->vals, 8 * A->nnz, hipMemcpyDeviceToHost, s));
    FFHIP_CHECK(hipStreamSynchronize(s));
  });
}

int ffhip_mat_upload(ffhip_ctx ctx, int64_t n, int64_t nnz, const int64_t *rowptr,
                     const int32_t *colidx, const double *vals, ffhip_mat *out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && out && rowptr && colidx && vals && n > 0 && nnz > 0, FFHIP_ERR_ARG,
                  "ffhip_mat_upload: bad arguments");
    FFHIP_REQUIRE(rowptr[0] == 0 && rowptr[n] == nnz, FFHIP_ERR_ARG, "ffhip_mat_upload: rowptr");
    FFHIP_REQUIRE(n < (1ll << 31), FFHIP_ERR_UNSUPPORTED, "ffhip_mat_upload: n too large");
    for (int64_t i = 0; i < n; ++i) {
      FFHIP_REQUIRE(rowptr[i + 1] >= rowptr[i], FFHIP_ERR_ARG, "ffhip_mat_upload: rowptr not monotone");
      for (int64_t k = rowptr[i]; k < rowptr[i + 1]; ++k) {
        FFHIP_REQUIRE(colidx[k] >= 0 && colidx[k] < n, FFHIP_ERR_ARG, "ffhip_mat_upload: column out of range");
        FFHIP_REQUIRE(k == rowptr[i] || colidx[k] > colidx[k - 1], FFHIP_ERR_ARG,
                      "ffhip_mat_upload: columns must be sorted and unique (HashMatrix::CSR order)");
      }
    }
    hipStream_t s = ctx->stream;
    ffhip_mat A = new ffhip_mat_s();
    A->ctx = ctx; A->n = n; A->nnz = nnz;
    A->rowptr = dalloc<int64_t>(n + 1);
    A->colidx = dalloc<int32_t>(nnz);
    A->vals = dalloc<double>(nnz);
    A->diag = dalloc<int64_t>(n);
    std::vector<int64_t> d(n, -1);
    for (int64_t i = 0; i < n; ++i)
      for (int64_t k = rowptr[i]; k < rowptr[i + 1]; ++k)
        if (colidx[k] == i) d[i] = k;
    FFHIP_CHECK(hipMemcpyAsync(A->rowptr, rowptr, 8 * (n + 1), hipMemcpyHostToDevice, s));
    FFHIP_CHECK(hipMemcpyAsync(A->colidx, colidx, 4 * nnz, hipMemcpyHostToDevice, s));
    FFHIP_CHECK(hipMemcpyAsync(A->vals, vals, 8 * nnz, hipMemcpyHostToDevice, s));
    FFHIP_CHECK(hipMemcpyAsync(A->diag, d.data(), 8 * n, hipMemcpyHostToDevice, s));
    FFHIP_CHECK(hipStreamSynchronize(s));
    *out = A;
  });
}

int ffhip_mat_set_values(ffhip_mat A, const double *vals) {
  return guard([&] {
    FFHIP_REQUIRE(A && vals, FFHIP_ERR_ARG, "ffhip_mat_set_values: null argument");
    FFHIP_CHECK(hipMemcpyAsync(A->vals, vals, 8 * A->nnz, hipMemcpyHostToDevice, A->ctx->stream));
    FFHIP_CHECK(hipStreamSynchronize(A->ctx->stream));
  });
}

int ffhip_mat_device_ptrs(ffhip_mat A, int64_t **rowptr, int32_t **colidx, double **vals) {
  return guard([&] {
    FFHIP_REQUIRE(A, FFHIP_ERR_ARG, "ffhip_mat_device_ptrs: null matrix");
    if (rowptr) *rowptr = A->rowptr;
    if (colidx) *colidx = A->colidx;
    if (vals) *vals = A->vals;
  });
}

int ffhip_mat_free(ffhip_mat A) {
  return guard([&] {
    if (!A) return;
    (void)hipStreamSynchronize(A->ctx->stream);
    dfree(A->rowptr); dfree(A->colidx); dfree(A->vals); dfree(A->diag); dfree(A->slotmap);
    dfree(A->nodeptr); dfree(A->slot8); dfree(A->big);
    dfree(A->fptr); dfree(A->fcol); dfree(A->fslot);
    delete A;
  });
}

int ffhip_spmv(ffhip_ctx ctx, ffhip_mat A, const double *x, double *y, int trans) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && A && x && y, FFHIP_ERR_ARG, "ffhip_spmv: null argument");
    hipStream_t s = ctx->stream;
    const unsigned grid = row_grid(A->n, few_rows(A->n) ? 16 : 64);
    auto product = [&](auto small, auto large, const int64_t *ptr, const int32_t *col, int *missing, double *keep) {
      ctx->tic();
      (few_rows(A->n) ? small : large)<<<grid, kWave, 0, s>>>(A->n, ptr, col, A->vals, A->fslot, x, y, missing, keep);
      FFHIP_CHECK(hipGetLastError());
      ctx->toc();
    };
    if (A->half) {  // y = (L + L^T - diag L) x over the full view; symmetric: trans alike
      half_view(A);
      product(k_spmv_stage<kSlots, 16>, k_spmv_stage<kSlots, 64>, A->fptr, A->fcol, nullptr, nullptr);
      return;
    }
    if (!trans) {
      product(k_spmv_stage<kPlain, 16>, k_spmv_stage<kPlain, 64>, A->rowptr, A->colidx, nullptr, nullptr);
      return;
    }
    int *missing = ctx->flag(0);
    double *keep = dalloc<double>(A->n);
    try {
      product(k_spmv_stage<kTrans, 16>, k_spmv_stage<kTrans, 64>, A->rowptr, A->colidx, missing, keep);
      if (*missing) {
        FFHIP_CHECK(hipMemcpyAsync(y, keep, 8 * A->n, hipMemcpyDeviceToDevice, s));
        FFHIP_CHECK(hipStreamSynchronize(s));
      }
    } catch (...) {
      (void)hipStreamSynchronize(s);
      dfree(keep);
      throw;
    }
    dfree(keep);
    FFHIP_REQUIRE(*missing == 0, FFHIP_ERR_UNSUPPORTED, "ffhip_spmv: transpose needs a symmetric pattern");
  });
}

}  // extern "C"
