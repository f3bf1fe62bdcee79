// ffhip_internal.hpp — shared internals of libffhip (not part of the C-ABI).
//
// Device-memory objects behind the opaque handles of include/ffhip.h, error
// plumbing, and small device helpers.  Everything here targets gfx950
// (CDNA4, wave64).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <string>

#include "../../include/ffhip.h"

namespace ffhip {

// ---------------------------------------------------------------- errors
void set_error(const char *fmt, ...);

struct Error {
  int code;
};

// (A failed call's error stays the thread's last error until it is read, also
// over calls that succeed: read here, so that no later launch check reports it.)
#define FFHIP_CHECK(expr)                                                      \
  do {                                                                         \
    hipError_t e_ = (expr);                                                    \
    if (e_ != hipSuccess) {                                                    \
      (void)hipGetLastError();                                                 \
      ::ffhip::set_error("%s:%d: %s -> %s", __FILE__, __LINE__, #expr,         \
                         hipGetErrorString(e_));                               \
      throw ::ffhip::Error{FFHIP_ERR_HIP};                                     \
    }                                                                          \
  } while (0)

#define FFHIP_REQUIRE(cond, code, ...)                                         \
  do {                                                                         \
    if (!(cond)) {                                                             \
      ::ffhip::set_error(__VA_ARGS__);                                         \
      throw ::ffhip::Error{code};                                              \
    }                                                                          \
  } while (0)

// Runs f() and maps exceptions to C-ABI return codes.
template <class F>
int guard(F &&f) {
  try {
    f();
    return FFHIP_OK;
  } catch (const Error &e) {
    return e.code;
  } catch (...) {
    set_error("unexpected C++ exception");
    return FFHIP_ERR_INTERNAL;
  }
}

// ---------------------------------------------------------------- memory
// Device blocks: released blocks are kept per device and handed out again for
// requests of about the same size (a solve or an assembly repeated on the same
// mesh re-allocates the same sizes), so steady-state calls do not pay
// hipMalloc / hipFree (tens to hundreds of microseconds per large block).
// All work of a context is ordered on its one stream; with several contexts
// on a device, a release first waits for the device.
void *block_alloc(size_t bytes);
void block_free(void *p);
void blocks_context(int device, int delta);  // context count per device; trims at 0
template <class T>
T *dalloc(size_t n) {
  if (n == 0) n = 1;
  return (T *)block_alloc(n * sizeof(T));
}
template <class T>
void dfree(T *&p) {
  if (p) block_free(p);
  p = nullptr;
}

}  // namespace ffhip

// ---------------------------------------------------------------- handles
struct ffhip_ctx_s {
  int device = 0;
  hipStream_t stream = nullptr;  // default priority (never a priority stream)
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  int num_cu = 256;
  // reusable scratch for library-internal temporaries (scans, partials)
  void *scratch = nullptr;
  size_t scratch_bytes = 0;
  void *ensure_scratch(size_t bytes);
  // work buffer the assembly and solver-setup temporaries are carved from
  // (grows to the largest request and is kept: no allocation on repeat calls)
  void *work = nullptr;
  size_t work_bytes = 0;
  void *ensure_work(size_t bytes);
  // page-locked host memory that kernels write small results to, read after the
  // call's wait (a context serves one call at a time): 16 flags, then data.  A
  // read-back this way is a launch and a wait; a copy to pageable memory cost
  // about 15 us more.
  static constexpr size_t kPinnedFlags = 64, kPinnedData = 65536;
  void *pinned = nullptr;
  int *flag(int i) {  // cleared flag i: kernels store 1 (plain stores: no atomics on host memory)
    int *p = static_cast<int *>(pinned) + i;
    *p = 0;
    return p;
  }
  void *pinned_data() { return static_cast<char *>(pinned) + kPinnedFlags; }
  double last_ms = 0.;  // device time of the last timed call
  void tic();           // record ev0 on the stream
  void toc();           // record ev1, synchronise, set last_ms
};

struct ffhip_mesh_s {
  ffhip_ctx ctx = nullptr;
  int dim = 3;      // 3: tetrahedra, 2: triangles
  int nloc = 4;     // vertices per element
  int nbloc = 3;    // vertices per boundary element
  int64_t nv = 0, nt = 0, nbe = 0;
  double *xyz = nullptr;    // nv * dim, vertex-major (x,y,z per vertex)
  int32_t *elems = nullptr; // nt * nloc
  int32_t *belems = nullptr;// nbe * nbloc
  int32_t *blab = nullptr;  // nbe
  // dof -> incident (element, local vertex) list, element order (built lazily)
  int64_t *v2e_ptr = nullptr;  // nv + 1
  int32_t *v2e = nullptr;      // nt * nloc entries: e * nloc + l
  int v2e_big = 0;             // some vertex has more than 32 incident elements
  int32_t *v2e_inv = nullptr;  // nt * nloc: position of item e * nloc + l in v2e
  // dof -> incident (boundary element, local vertex) list, boundary-element
  // order (built lazily by the boundary-integral calls)
  int64_t *b2e_ptr = nullptr;  // nv + 1
  int32_t *b2e = nullptr;      // nbe * nbloc entries: f * nbloc + l
};

struct ffhip_mat_s {
  ffhip_ctx ctx = nullptr;
  int64_t n = 0, nnz = 0;
  int64_t *rowptr = nullptr;   // n + 1
  int32_t *colidx = nullptr;   // nnz (sorted within each row)
  double *vals = nullptr;      // nnz
  int64_t *diag = nullptr;     // n: slot of (i,i), -1 if absent
  // element-to-row map: for incidence entry k of row i (mesh v2e order), the
  // offsets within row i of the columns of that element's vertices
  uint32_t *slotmap = nullptr; // (nt*nloc) packed 4 x uint8 (P1, nloc <= 4)
  int max_row = 0;
  ffhip_mesh mesh = nullptr;   // mesh the pattern was built from (if any)
  // P1 rows built by the lane-per-row kernels (more than 32 incident elements
  // or 64 columns); the others by the half-wave kernels
  uint8_t *big = nullptr;      // n
  int any_big = 0;
  // vector-P2 matrices: node-level rows (the scalar rows 3a..3a+2 of node a
  // hold 3 x 3 blocks of its node columns) and the byte slot map, 10 offsets
  // per node incidence
  ffhip_p2v p2v = nullptr;
  int ncomp = 0;               // P2 matrices: 3 for [P2,P2,P2], 1 for scalar P2
  int64_t *nodeptr = nullptr;  // nnodes + 1
  uint8_t *slot8 = nullptr;    // (nt * 10) * 10
  // half storage (FreeFEM's sym=1): only row >= column is stored; the full
  // view lists every full row as slots of vals (built once, by half_view)
  int half = 0;
  int64_t fnnz = 0;
  int64_t *fptr = nullptr;     // n + 1
  int32_t *fcol = nullptr;     // fnnz
  int64_t *fslot = nullptr;    // fnnz: slot in vals
};

// [P2,P2,P2] space on a tetrahedral mesh (FESpace3 with GTypeOfFESum of three
// P2): nodes numbered by first appearance over the elements, then dof
// 3 * node + component.
struct ffhip_p2v_s {
  ffhip_ctx ctx = nullptr;
  ffhip_mesh mesh = nullptr;
  int64_t nnodes = 0, ne = 0;
  int32_t *elem_nodes = nullptr;  // nt * 10: 4 vertex nodes, 6 edge nodes
  int32_t *vnode = nullptr;       // nv: node of each vertex
  uint64_t *ekeys = nullptr;      // ne: sorted edge keys (min << 32 | max)
  int32_t *enode = nullptr;       // ne: node of each edge
  int64_t *n2e_ptr = nullptr;     // nnodes + 1
  int32_t *n2e = nullptr;         // nt * 10: element * 10 + local node, element order
};

namespace ffhip {

// ---------------------------------------------------------------- device helpers
constexpr int kWave = 64;

// wave64 sum of a double, the same in every lane: lane i adds lane i ^ 32's
// value, then i ^ 16's, ... i ^ 1's.  The first two exchanges swap halves and
// rows between two registers, the others rotate within the rows of 16 lanes: a
// rotation by m is the exchange with i ^ m once the values repeat every 2 m
// lanes, as they do after the steps before.  Vector instructions only: about
// 100 cycles, where six shuffles through LDS took about 800 (the solver's
// kernels sum twice each: its update at 252 rows 2.49 -> 2.03 us, its direction
// 2.68 -> 2.36).
template <int CTRL>
__device__ inline double dpp_row(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, false);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ inline double join_halves(unsigned lo, unsigned hi) {
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ inline double row16_sum(double v) {  // over each 16 lanes
  v += dpp_row<0x128>(v);                       // row_ror:8
  v += dpp_row<0x124>(v);
  v += dpp_row<0x122>(v);
  v += dpp_row<0x121>(v);
  return v;
}
__device__ inline double wave_sum(double v) {
  {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const auto l = __builtin_amdgcn_permlane32_swap((unsigned)b, (unsigned)b, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
    v = join_halves(l[0], h[0]) + join_halves(l[1], h[1]);
  }
  {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const auto l = __builtin_amdgcn_permlane16_swap((unsigned)b, (unsigned)b, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
    v = join_halves(l[0], h[0]) + join_halves(l[1], h[1]);
  }
  return row16_sum(v);
}

// Deterministic block reduction of one double; result valid in every thread.
template <int BLOCK>
__device__ inline double block_sum(double v, double *lds /* BLOCK/64 */) {
  v = wave_sum(v);
  const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  __syncthreads();
  if (lane == 0) lds[w] = v;
  __syncthreads();
  double s = 0.;
#pragma unroll
  for (int i = 0; i < BLOCK / kWave; ++i) s += lds[i];
  return s;
}

// orders the LDS accesses of one wave (cross-lane reuse of the row staging)
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// XCD-aware logical block id: the hardware dispatches block b to XCD b % 8;
// logical ids are renumbered so each XCD owns a contiguous block range (and
// so a contiguous row range whose x-gathers stay in that XCD's L2).
__device__ inline int xcd_block_id() {
  const int G = gridDim.x, b = blockIdx.x;
  if (G % 8) return b;
  return (b % 8) * (G / 8) + (b / 8);
}

// What the one-call P1 assembly needs for the element scales (C_e of the
// stiffness); the incidence build of a tetrahedral mesh computes them when
// given these.
struct ScaleArgs {
  const double *xyz;
  int kind;
  double c0;
  const double *kappa_e;
  double *Ce;
};

// dof -> (element, local dof) incidence lists in element order (ffhip_assembly.hip)
void build_incidence(ffhip_ctx ctx, const int32_t *elems, int64_t nt, int nloc, int64_t n,
                     int64_t **ptr_out, int32_t **list_out, int *big_out, int32_t **inv_out,
                     int32_t **bucket_out, const ScaleArgs *sc = nullptr, int *ovf_dev = nullptr);

void exclusive_scan_i64(ffhip_ctx ctx, const int64_t *in, int64_t *out,
                        int64_t n);

// 256-byte aligned temporaries carved from the context's work buffer; one
// arena at a time per context (the calls that use one are sequential)
struct Arena {
  static size_t bytes(size_t count, size_t size) { return (count * size + 255) & ~size_t(255); }
  char *base;
  size_t cap, off = 0;
  Arena(ffhip_ctx ctx, size_t total) : base((char *)ctx->ensure_work(total)), cap(total) {}
  template <class T>
  T *take(size_t count) {
    const size_t b = bytes(count ? count : 1, sizeof(T));
    FFHIP_REQUIRE(off + b <= cap, FFHIP_ERR_INTERNAL, "work arena overflow");
    T *p = (T *)(base + off);
    off += b;
    return p;
  }
};
int64_t read_i64(ffhip_ctx ctx, const int64_t *p);
int read_flag(ffhip_ctx ctx, const int *p);
// Small device values to the host: one launch that writes them to page-locked
// memory, then a wait for the stream (bytes: multiples of 4, 256 at most in all).
struct Fetch {
  void *dst;
  const void *src;
  unsigned bytes;
};
void fetch(ffhip_ctx ctx, std::initializer_list<Fetch> list);
// Clears up to 4 buffers in one launch (16-byte aligned; a memset each was a
// launch each).
struct Clear {
  void *p;
  size_t bytes;
};
void clear(ffhip_ctx ctx, std::initializer_list<Clear> list);

// Boundary labels as a kernel takes them: up to kNear by value (no copy to the
// device), more in an array that lives as long as the LabelArg.
struct Labels {
  static constexpr int kNear = 16;
  int n;
  int32_t near_[kNear];
  const int32_t *far;
  __device__ bool has(int32_t lab) const {
    bool on = false;
    for (int k = 0; k < n; ++k) on |= lab == (far ? far[k] : near_[k]);
    return on;
  }
};
struct LabelArg {
  Labels L{};
  int32_t *own = nullptr;
  // buf: device room for the labels (else allocated where needed)
  LabelArg(ffhip_ctx ctx, const int32_t *labels, int nlab, int32_t *buf = nullptr) {
    L.n = nlab;
    if (nlab <= Labels::kNear) {
      for (int k = 0; k < nlab; ++k) L.near_[k] = labels[k];
      return;
    }
    if (!buf) buf = own = dalloc<int32_t>(nlab);
    L.far = buf;
    if (hipError_t e = hipMemcpyAsync(buf, labels, 4 * (size_t)nlab, hipMemcpyHostToDevice, ctx->stream)) {
      dfree(own);
      FFHIP_CHECK(e);
    }
  }
  LabelArg(const LabelArg &) = delete;
  LabelArg &operator=(const LabelArg &) = delete;
  ~LabelArg() { dfree(own); }
};
// the vertices of the boundary elements with these labels
void mark_bc(ffhip_ctx ctx, ffhip_mesh m, const Labels &labels, uint8_t *onbc);

// the per-device address of the no-allocation entry points' scratch array
// (ffhip_assembly.hip); set up by ffhip_init with the device current
void noalloc_scratch_setup(int device);

}  // namespace ffhip
