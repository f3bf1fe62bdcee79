// ffhip_core.hip — context, errors, scans and device-built meshes.
//
// cube(nx,ny,nz) and square(nx,ny) are generated on the GPU with the exact
// vertex numbering, coordinates, element vertex order, boundary elements and
// labels of FreeFEM's BuildCube (src/fflib/msh3.cpp:7879-8132) and Carre_
// (src/fflib/lgmesh.cpp:1229-1384), each in one pass.
#include <hipcub/hipcub.hpp>

#include <cstdarg>
#include <map>
#include <mutex>
#include <unordered_map>
#include <cstring>
#include <vector>

#include "ffhip_internal.hpp"

namespace ffhip {

static thread_local char g_err[1024] = "";

void set_error(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

void exclusive_scan_i64(ffhip_ctx ctx, const int64_t *in, int64_t *out,
                        int64_t n) {
  size_t bytes = 0;
  FFHIP_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, in, out, n,
                                               ctx->stream));
  void *tmp = ctx->ensure_scratch(bytes);
  FFHIP_CHECK(hipcub::DeviceScan::ExclusiveSum(tmp, bytes, in, out, n,
                                               ctx->stream));
}

struct FetchArgs {
  const uint32_t *src[4];
  int end[4];  // words up to and with this source
};
__global__ __launch_bounds__(64) void k_fetch(FetchArgs a, uint32_t *__restrict__ dst) {
  const int i = threadIdx.x;
  int k = 0, base = 0;
  while (k < 4 && i >= a.end[k]) base = a.end[k++];
  if (k < 4) dst[i] = a.src[k][i - base];
}
void fetch(ffhip_ctx ctx, std::initializer_list<Fetch> list) {
  FetchArgs a{};
  int k = 0, words = 0;
  FFHIP_REQUIRE(list.size() <= 4, FFHIP_ERR_INTERNAL, "fetch: %d values", (int)list.size());
  for (const Fetch &f : list) {
    a.src[k] = static_cast<const uint32_t *>(f.src);
    a.end[k++] = words += f.bytes / 4;
  }
  FFHIP_REQUIRE(words <= 64, FFHIP_ERR_INTERNAL, "fetch: %d words", words);
  for (; k < 4; ++k) a.end[k] = words;
  k_fetch<<<1, 64, 0, ctx->stream>>>(a, static_cast<uint32_t *>(ctx->pinned_data()));
  FFHIP_CHECK(hipGetLastError());
  FFHIP_CHECK(hipStreamSynchronize(ctx->stream));
  const char *p = static_cast<const char *>(ctx->pinned_data());
  for (const Fetch &f : list) {
    memcpy(f.dst, p, f.bytes);
    p += f.bytes;
  }
}
int64_t read_i64(ffhip_ctx ctx, const int64_t *p) {
  int64_t v = 0;
  fetch(ctx, {{&v, p, sizeof(v)}});
  return v;
}
int read_flag(ffhip_ctx ctx, const int *p) {
  int v = 0;
  fetch(ctx, {{&v, p, sizeof(v)}});
  return v;
}

struct ClearArgs {
  char *p[4];
  size_t bytes[4];
  int64_t end[4];  // 16-byte units up to and with this buffer
};
__global__ __launch_bounds__(256) void k_clear(ClearArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  int k = 0;
  int64_t base = 0;
  while (k < 4 && i >= a.end[k]) base = a.end[k++];
  if (k == 4) return;
  const size_t o = 16 * (size_t)(i - base);
  if (o + 16 <= a.bytes[k]) {
    *reinterpret_cast<uint4 *>(a.p[k] + o) = make_uint4(0, 0, 0, 0);
  } else {
    for (size_t b = o; b < a.bytes[k]; ++b) a.p[k][b] = 0;
  }
}
void clear(ffhip_ctx ctx, std::initializer_list<Clear> list) {
  ClearArgs a{};
  int k = 0;
  int64_t units = 0;
  for (const Clear &c : list) {
    FFHIP_REQUIRE(k < 4 && (uintptr_t)c.p % 16 == 0, FFHIP_ERR_INTERNAL, "clear: buffers");
    a.p[k] = static_cast<char *>(c.p);
    a.bytes[k] = c.bytes;
    a.end[k++] = units += (int64_t)((c.bytes + 15) / 16);
  }
  for (; k < 4; ++k) a.end[k] = units;
  if (!units) return;
  k_clear<<<(unsigned)((units + 255) / 256), 256, 0, ctx->stream>>>(a);
  FFHIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------- cube
// hex split selected by BuildCube for kind = 6 (hex_decoupe[70] of the table
// at msh3.cpp:7682-7742, simplexes {7,15,19,27,26,11}), hex-local numbering
// a + 2b + 4c (msh3.cpp:8039-8045)
__constant__ int c_split6[6][4] = {{4, 0, 6, 7}, {0, 4, 5, 7}, {1, 0, 5, 7},
                                   {0, 1, 3, 7}, {2, 0, 3, 7}, {0, 2, 6, 7}};
// Tet faces (Mesh3dn.cpp:72)
__constant__ int c_tetface[4][3] = {{3, 2, 1}, {0, 2, 3}, {3, 1, 0}, {0, 1, 2}};

struct CubeLabels {
  int32_t lab[6];
};

// boundary triangles of the hexes before hex (i, j, k) in hex order: two per
// hex face on the boundary, counted plane by plane
__device__ inline int cube_bfaces_before(int i, int j, int k, int nx, int ny, int nz) {
  const int row = k * ny + j, in_plane = i + nx * j;
  return 2 * (row + (i > 0) + row +                                        // x = 0, x = 1
              k * nx + (j > 0 ? nx : i) + k * nx + (j == ny - 1 ? i : 0) +  // y = 0, y = 1
              (k > 0 ? nx * ny : in_plane) + (k == nz - 1 ? in_plane : 0)); // z = 0, z = 1
}

// The whole mesh in one pass: thread p writes vertex p, the block its 256
// hexes' 1536 tets (consecutive threads on consecutive tets, from the hexes'
// first vertices in LDS) and each boundary hex its triangles in BuildCube's
// order, hex, tet, face (msh3.cpp:8090-8110), at the offset counted above.
// Bound by the tets' store (16 B each): 114 us for 24.6 M tets at cube(160).  A
// thread per hex that found its triangles by comparing the vertices' labels
// (64-bit divisions) took 450 us there and about 60 us on the smallest box,
// after a scan of the hexes' counts.
__global__ __launch_bounds__(256) void k_cube_mesh(int nx, int ny, int nz, double xd, double yd,
                                                   double zd, CubeLabels L, double *__restrict__ xyz,
                                                   int32_t *__restrict__ tets,
                                                   int32_t *__restrict__ btri,
                                                   int32_t *__restrict__ blab) {
  __shared__ int32_t first[256];
  __shared__ int4 off[6];  // the tets' vertex offsets from the hex's first vertex
  const int nv = (nx + 1) * (ny + 1) * (nz + 1), nc = nx * ny * nz;
  const int nj = nx + 1, nk = nj * (ny + 1);
  const int t = threadIdx.x, p = blockIdx.x * 256 + t;
  if (p < nv) {
    const int i = p % nj, r = p / nj, j = r % (ny + 1), k = r / (ny + 1);
    xyz[3 * (int64_t)p + 0] = 0. + xd * i;
    xyz[3 * (int64_t)p + 1] = 0. + yd * j;
    xyz[3 * (int64_t)p + 2] = 0. + zd * k;
  }
  auto corner = [&](int c) { return (c & 1) + ((c >> 1) & 1) * nj + (c >> 2) * nk; };
  const int i = p % nx, r = p / nx, j = r % ny, k = r / ny;  // hex p
  const int f0 = i + nj * j + nk * k;
  first[t] = f0;
  if (t < 6)
    off[t] = int4{corner(c_split6[t][0]), corner(c_split6[t][1]), corner(c_split6[t][2]),
                  corner(c_split6[t][3])};
  __syncthreads();
  const int h0 = blockIdx.x * 256, ntb = 6 * (nc - h0 < 256 ? nc - h0 : 256);
  for (int q = t; q < ntb; q += 256) {
    const int h = q / 6, b = first[h];
    const int4 o = off[q - 6 * h];
    reinterpret_cast<int4 *>(tets)[6 * (int64_t)h0 + q] = int4{b + o.x, b + o.y, b + o.z, b + o.w};
  }
  if (p >= nc) return;
  // the hex's faces on the boundary, bits as the vertex labels of BuildCube
  const int on = 1 * (i == 0) + 2 * (i == nx - 1) + 4 * (j == 0) + 8 * (j == ny - 1) + 16 * (k == 0) +
                 32 * (k == nz - 1);
  if (!on) return;
  const int nff[6] = {3, 1, 0, 2, 4, 5};  // msh3.cpp:8050
  int64_t o = cube_bfaces_before(i, j, k, nx, ny, nz);
  for (int d = 0; d < 6; ++d)
    for (int f = 0; f < 4; ++f) {
      int c[3], side = on;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        c[q] = c_split6[d][c_tetface[f][q]];
        // the hex faces that corner c lies on
        side &= (c[q] & 1 ? 2 : 1) | (c[q] & 2 ? 8 : 4) | (c[q] & 4 ? 32 : 16);
      }
      if (!side) continue;  // three corners share at most one face
      btri[3 * o + 0] = f0 + corner(c[0]);
      btri[3 * o + 1] = f0 + corner(c[1]);
      btri[3 * o + 2] = f0 + corner(c[2]);
      blab[o] = L.lab[nff[__builtin_ctz(side)]];
      ++o;
    }
}

// ---------------------------------------------------------------- square
struct SquareLabels {
  int32_t lab[4];
};

__global__ void k_square(int nx, int ny, SquareLabels L, double *__restrict__ xy,
                         int32_t *__restrict__ tris, int32_t *__restrict__ bed,
                         int32_t *__restrict__ blab) {
  const int64_t nv = (int64_t)(nx + 1) * (ny + 1), nc = (int64_t)nx * ny;
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < nv) {
    const int i = (int)(p % (nx + 1)), j = (int)(p / (nx + 1));
    xy[2 * p] = (double)i / nx;  // R2 P((R) i/nx,(R) j/ny)  (lgmesh.cpp:1258)
    xy[2 * p + 1] = (double)j / ny;
  }
  if (p < nc) {
    const int i = (int)(p % nx), j = (int)(p / nx);
    const int32_t i0 = i + j * (nx + 1), i1 = i0 + 1, i2 = i1 + nx + 1, i3 = i2 - 1;
    int32_t *t = tris + 6 * p;  // diag 1 (lgmesh.cpp:1300-1306)
    t[0] = i0; t[1] = i1; t[2] = i2; t[3] = i0; t[4] = i2; t[5] = i3;
  }
  // boundary edges (2 (nx + ny) may exceed the vertices of a thin square: the grid covers both)
  const int64_t b = p, nbe = 2 * ((int64_t)nx + ny);
  if (b >= nbe) return;
  const int nx1 = nx + 1;
  int32_t i1, i2, l;
  if (b < nx) { i1 = (int32_t)b; i2 = i1 + 1; l = L.lab[0]; }                       // bottom
  else if (b < nx + ny) { int j = (int)(b - nx); i1 = nx + j * nx1; i2 = i1 + nx1; l = L.lab[1]; }  // right
  else if (b < 2 * nx + ny) { int i = (int)(b - nx - ny); i1 = i + ny * nx1; i2 = i1 + 1; l = L.lab[2]; }  // up
  else { int j = (int)(b - 2 * nx - ny); i1 = j * nx1; i2 = i1 + nx1; l = L.lab[3]; }  // left
  bed[2 * b] = i1; bed[2 * b + 1] = i2; blab[b] = l;
}

// plain streaming copy, 16 B per lane per step (measurement reference)
typedef int v4i __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void k_copy(int64_t n16, const v4i *__restrict__ src,
                                              v4i *__restrict__ dst) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16;
       i += (int64_t)gridDim.x * blockDim.x)
    dst[i] = __builtin_nontemporal_load(src + i);
}

}  // namespace ffhip

using namespace ffhip;

void *ffhip_ctx_s::ensure_scratch(size_t bytes) {
  if (bytes > scratch_bytes) {
    if (scratch) (void)hipFree(scratch);
    scratch = nullptr;
    scratch_bytes = 0;
    FFHIP_CHECK(hipMalloc(&scratch, bytes));
    scratch_bytes = bytes;
  }
  return scratch;
}

void *ffhip_ctx_s::ensure_work(size_t bytes) {
  if (bytes > work_bytes) {
    if (work) (void)hipFree(work);
    work = nullptr;
    work_bytes = 0;
    FFHIP_CHECK(hipMalloc(&work, bytes));
    work_bytes = bytes;
  }
  return work;
}

void ffhip_ctx_s::tic() { FFHIP_CHECK(hipEventRecord(ev0, stream)); }
void ffhip_ctx_s::toc() {
  FFHIP_CHECK(hipEventRecord(ev1, stream));
  FFHIP_CHECK(hipEventSynchronize(ev1));
  float ms = 0.f;
  FFHIP_CHECK(hipEventElapsedTime(&ms, ev0, ev1));
  last_ms = ms;
}

extern "C" {

const char *ffhip_last_error(void) { return g_err; }
const char *ffhip_version(void) { return "ffhip 0.1 (gfx950)"; }

}  // extern "C"

namespace ffhip {
namespace {
struct BlockCache {
  std::mutex mu;
  std::map<int, std::multimap<size_t, void *>> free_;       // per device, by size
  std::unordered_map<void *, std::pair<int, size_t>> info;  // every block: device, size
  std::map<int, int> contexts;
  size_t cached = 0;  // bytes in the free lists
};
BlockCache &blocks() {
  static BlockCache *c = new BlockCache();  // never destroyed: used until process exit
  return *c;
}
constexpr size_t kCacheCap = size_t(32) << 30;  // cached bytes kept at most

size_t round_block(size_t b) {
  const size_t g = b >= (size_t(1) << 20) ? (size_t(2) << 20) : 256;
  return (b + g - 1) / g * g;
}

void trim_device(BlockCache &c, int dev) {  // caller holds c.mu
  auto it = c.free_.find(dev);
  if (it == c.free_.end()) return;
  for (auto &kv : it->second) {
    (void)hipFree(kv.second);
    c.info.erase(kv.second);
    c.cached -= kv.first;
  }
  it->second.clear();
}
}  // namespace

void *block_alloc(size_t bytes) {
  BlockCache &c = blocks();
  int dev = 0;
  FFHIP_CHECK(hipGetDevice(&dev));
  const size_t want = round_block(bytes);
  {
    std::lock_guard<std::mutex> g(c.mu);
    auto &fl = c.free_[dev];
    auto it = fl.lower_bound(want);
    // a cached block at most 1/8 larger (small blocks: at most twice as large)
    if (it != fl.end() && it->first <= (want >= (size_t(1) << 20) ? want + want / 8 : 2 * want)) {
      void *p = it->second;
      c.cached -= it->first;
      fl.erase(it);
      return p;
    }
  }
  void *p = nullptr;
  hipError_t e = hipMalloc(&p, want);
  if (e != hipSuccess) {  // give the cached blocks back and try once more
    (void)hipGetLastError();
    {
      std::lock_guard<std::mutex> g(c.mu);
      trim_device(c, dev);
    }
    e = hipMalloc(&p, want);
  }
  if (e != hipSuccess) {
    (void)hipGetLastError();
    set_error("hipMalloc(%zu bytes) -> %s", want, hipGetErrorString(e));
    throw Error{FFHIP_ERR_HIP};
  }
  std::lock_guard<std::mutex> g(c.mu);
  c.info[p] = {dev, want};
  return p;
}

void block_free(void *p) {
  BlockCache &c = blocks();
  int dev = 0;
  size_t size = 0;
  bool shared = false;
  {
    std::lock_guard<std::mutex> g(c.mu);
    auto it = c.info.find(p);
    if (it == c.info.end()) {  // not a cached block
      (void)hipFree(p);
      return;
    }
    dev = it->second.first;
    size = it->second.second;
    shared = c.contexts[dev] > 1;
    if (c.cached + size > kCacheCap) {
      c.info.erase(it);
      (void)hipFree(p);
      return;
    }
  }
  if (shared) {  // another context's stream could reuse it: let this one's work finish
    int cur = 0;
    (void)hipGetDevice(&cur);
    (void)hipSetDevice(dev);
    (void)hipDeviceSynchronize();
    (void)hipSetDevice(cur);
  }
  std::lock_guard<std::mutex> g(c.mu);
  c.free_[dev].emplace(size, p);
  c.cached += size;
}

void blocks_context(int device, int delta) {
  BlockCache &c = blocks();
  std::lock_guard<std::mutex> g(c.mu);
  c.contexts[device] += delta;
  if (c.contexts[device] <= 0) trim_device(c, device);
}
}  // namespace ffhip

extern "C" {

int ffhip_init(int device, ffhip_ctx *out) {
  return guard([&] {
    FFHIP_REQUIRE(out, FFHIP_ERR_ARG, "ffhip_init: null output");
    int ndev = 0;
    FFHIP_CHECK(hipGetDeviceCount(&ndev));
    FFHIP_REQUIRE(device >= 0 && device < ndev, FFHIP_ERR_ARG,
                  "ffhip_init: device %d of %d", device, ndev);
    FFHIP_CHECK(hipSetDevice(device));
    noalloc_scratch_setup(device);
    ffhip_ctx c = new ffhip_ctx_s();
    c->device = device;
    // a blocking stream: ordered with the legacy default stream, which is
    // where a host framework sharing the process (torch) enqueues its work
    FFHIP_CHECK(hipStreamCreate(&c->stream));
    FFHIP_CHECK(hipEventCreate(&c->ev0));
    FFHIP_CHECK(hipEventCreate(&c->ev1));
    FFHIP_CHECK(hipHostMalloc(&c->pinned, ffhip_ctx_s::kPinnedFlags + ffhip_ctx_s::kPinnedData, hipHostMallocDefault));
    hipDeviceProp_t prop;
    FFHIP_CHECK(hipGetDeviceProperties(&prop, device));
    c->num_cu = prop.multiProcessorCount;
    blocks_context(device, +1);
    *out = c;
  });
}

int ffhip_ctx_free(ffhip_ctx c) {
  return guard([&] {
    if (!c) return;
    (void)hipStreamSynchronize(c->stream);
    if (c->scratch) (void)hipFree(c->scratch);
    if (c->work) (void)hipFree(c->work);
    if (c->pinned) (void)hipHostFree(c->pinned);
    (void)hipEventDestroy(c->ev0);
    (void)hipEventDestroy(c->ev1);
    (void)hipStreamDestroy(c->stream);
    blocks_context(c->device, -1);
    delete c;
  });
}

int ffhip_sync(ffhip_ctx c) {
  return guard([&] { FFHIP_CHECK(hipStreamSynchronize(c->stream)); });
}

double ffhip_last_ms(ffhip_ctx c) { return c ? c->last_ms : 0.; }

int ffhip_bench_copy(ffhip_ctx ctx, int64_t nbytes, int reps, double *avg_ms) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && avg_ms && reps > 0 && nbytes >= 16, FFHIP_ERR_ARG, "ffhip_bench_copy: bad arguments");
    const int64_t n16 = nbytes / 16;
    v4i *a = dalloc<v4i>(n16), *b = dalloc<v4i>(n16);
    FFHIP_CHECK(hipMemsetAsync(a, 0, 16 * n16, ctx->stream));
    // 4 blocks of 256 per CU: the fastest plain copy in a sweep of grid sizes
    // (4..32 blocks per CU) and unroll depths on MI355X
    const unsigned grid = 4 * (unsigned)ctx->num_cu;
    k_copy<<<grid, 256, 0, ctx->stream>>>(n16, a, b);
    FFHIP_CHECK(hipGetLastError());
    ctx->tic();
    for (int r = 0; r < reps; ++r) k_copy<<<grid, 256, 0, ctx->stream>>>(n16, a, b);
    FFHIP_CHECK(hipGetLastError());
    ctx->toc();
    *avg_ms = ctx->last_ms / reps;
    dfree(a);
    dfree(b);
  });
}

int ffhip_mesh3_cube(ffhip_ctx ctx, int nx, int ny, int nz, const int32_t labels[6],
                     ffhip_mesh *out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && out, FFHIP_ERR_ARG, "ffhip_mesh3_cube: null argument");
    FFHIP_REQUIRE(nx >= 1 && ny >= 1 && nz >= 1, FFHIP_ERR_ARG,
                  "ffhip_mesh3_cube: bad sizes %d %d %d", nx, ny, nz);
    const int64_t nv = (int64_t)(nx + 1) * (ny + 1) * (nz + 1);
    const int64_t nc = (int64_t)nx * ny * nz, nt = 6 * nc;
    const int64_t nbe = 4 * ((int64_t)nx * ny + (int64_t)nx * nz + (int64_t)ny * nz);
    FFHIP_REQUIRE(nv < (1ll << 31) && 4 * nt < (1ll << 31), FFHIP_ERR_UNSUPPORTED,
                  "ffhip_mesh3_cube: mesh too large for int32 element ids");
    CubeLabels lab = {{1, 2, 3, 4, 5, 6}};
    if (labels) memcpy(lab.lab, labels, sizeof(lab.lab));
    ffhip_mesh m = new ffhip_mesh_s();
    m->ctx = ctx; m->dim = 3; m->nloc = 4; m->nbloc = 3;
    m->nv = nv; m->nt = nt; m->nbe = nbe;
    m->xyz = dalloc<double>(3 * nv);
    m->elems = dalloc<int32_t>(4 * nt);
    m->belems = dalloc<int32_t>(3 * nbe);
    m->blab = dalloc<int32_t>(nbe);
    ctx->tic();
    k_cube_mesh<<<(unsigned)((nv + 255) / 256), 256, 0, ctx->stream>>>(  // nv > nc
        nx, ny, nz, 1. / nx, 1. / ny, 1. / nz, lab, m->xyz, m->elems, m->belems, m->blab);
    FFHIP_CHECK(hipGetLastError());
    ctx->toc();
    *out = m;
  });
}

int ffhip_mesh2_square(ffhip_ctx ctx, int nx, int ny, const int32_t labels[4],
                       ffhip_mesh *out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && out && nx >= 1 && ny >= 1, FFHIP_ERR_ARG, "ffhip_mesh2_square: bad args");
    const int64_t nv = (int64_t)(nx + 1) * (ny + 1), nt = 2 * (int64_t)nx * ny;
    const int64_t nbe = 2 * ((int64_t)nx + ny);
    FFHIP_REQUIRE(nv < (1ll << 31) && 3 * nt < (1ll << 31), FFHIP_ERR_UNSUPPORTED,
                  "ffhip_mesh2_square: mesh too large");
    SquareLabels lab = {{1, 2, 3, 4}};
    if (labels) memcpy(lab.lab, labels, sizeof(lab.lab));
    ffhip_mesh m = new ffhip_mesh_s();
    m->ctx = ctx; m->dim = 2; m->nloc = 3; m->nbloc = 2;
    m->nv = nv; m->nt = nt; m->nbe = nbe;
    m->xyz = dalloc<double>(2 * nv);
    m->elems = dalloc<int32_t>(3 * nt);
    m->belems = dalloc<int32_t>(2 * nbe);
    m->blab = dalloc<int32_t>(nbe);
    const int64_t nn = nv > nbe ? nv : nbe;
    ctx->tic();
    k_square<<<(unsigned)((nn + 255) / 256), 256, 0, ctx->stream>>>(nx, ny, lab, m->xyz, m->elems,
                                                                    m->belems, m->blab);
    FFHIP_CHECK(hipGetLastError());
    ctx->toc();
    *out = m;
  });
}

int ffhip_mesh3_upload(ffhip_ctx ctx, int64_t nv, int64_t nt, int64_t nbe,
                       const double *xyz, const int32_t *tets, const int32_t *btri,
                       const int32_t *blab, ffhip_mesh *out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && out && xyz && tets && nv > 0 && nt > 0 && nbe >= 0, FFHIP_ERR_ARG,
                  "ffhip_mesh3_upload: bad arguments");
    FFHIP_REQUIRE(nbe == 0 || (btri && blab), FFHIP_ERR_ARG, "ffhip_mesh3_upload: boundary arrays");
    FFHIP_REQUIRE(nv < (1ll << 31) && 4 * nt < (1ll << 31), FFHIP_ERR_UNSUPPORTED,
                  "ffhip_mesh3_upload: mesh too large for int32 ids");
    for (int64_t k = 0; k < 4 * nt; ++k)
      FFHIP_REQUIRE(tets[k] >= 0 && tets[k] < nv, FFHIP_ERR_ARG,
                    "ffhip_mesh3_upload: tet vertex id %d out of range", tets[k]);
    for (int64_t k = 0; k < 3 * nbe; ++k)
      FFHIP_REQUIRE(btri[k] >= 0 && btri[k] < nv, FFHIP_ERR_ARG,
                    "ffhip_mesh3_upload: boundary vertex id out of range");
    ffhip_mesh m = new ffhip_mesh_s();
    m->ctx = ctx; m->dim = 3; m->nloc = 4; m->nbloc = 3;
    m->nv = nv; m->nt = nt; m->nbe = nbe;
    m->xyz = dalloc<double>(3 * nv);
    m->elems = dalloc<int32_t>(4 * nt);
    m->belems = dalloc<int32_t>(3 * nbe);
    m->blab = dalloc<int32_t>(nbe);
    FFHIP_CHECK(hipMemcpyAsync(m->xyz, xyz, 24 * nv, hipMemcpyHostToDevice, ctx->stream));
    FFHIP_CHECK(hipMemcpyAsync(m->elems, tets, 16 * nt, hipMemcpyHostToDevice, ctx->stream));
    if (nbe) {
      FFHIP_CHECK(hipMemcpyAsync(m->belems, btri, 12 * nbe, hipMemcpyHostToDevice, ctx->stream));
      FFHIP_CHECK(hipMemcpyAsync(m->blab, blab, 4 * nbe, hipMemcpyHostToDevice, ctx->stream));
    }
    FFHIP_CHECK(hipStreamSynchronize(ctx->stream));
    *out = m;
  });
}

int ffhip_mesh2_upload(ffhip_ctx ctx, int64_t nv, int64_t nt, int64_t nbe, const double *xy,
                       const int32_t *tris, const int32_t *bedges, const int32_t *blab,
                       ffhip_mesh *out) {
  return guard([&] {
    FFHIP_REQUIRE(ctx && out && xy && tris && nv > 0 && nt > 0 && nbe >= 0, FFHIP_ERR_ARG,
                  "ffhip_mesh2_upload: bad arguments");
    FFHIP_REQUIRE(nbe == 0 || (bedges && blab), FFHIP_ERR_ARG, "ffhip_mesh2_upload: boundary arrays");
    FFHIP_REQUIRE(nv < (1ll << 31) && 3 * nt < (1ll << 31), FFHIP_ERR_UNSUPPORTED,
                  "ffhip_mesh2_upload: mesh too large for int32 ids");
    for (int64_t k = 0; k < 3 * nt; ++k)
      FFHIP_REQUIRE(tris[k] >= 0 && tris[k] < nv, FFHIP_ERR_ARG,
                    "ffhip_mesh2_upload: triangle vertex id %d out of range", tris[k]);
    for (int64_t k = 0; k < 2 * nbe; ++k)
      FFHIP_REQUIRE(bedges[k] >= 0 && bedges[k] < nv, FFHIP_ERR_ARG,
                    "ffhip_mesh2_upload: boundary vertex id out of range");
    ffhip_mesh m = new ffhip_mesh_s();
    m->ctx = ctx; m->dim = 2; m->nloc = 3; m->nbloc = 2;
    m->nv = nv; m->nt = nt; m->nbe = nbe;
    m->xyz = dalloc<double>(2 * nv);
    m->elems = dalloc<int32_t>(3 * nt);
    m->belems = dalloc<int32_t>(2 * nbe);
    m->blab = dalloc<int32_t>(nbe);
    FFHIP_CHECK(hipMemcpyAsync(m->xyz, xy, 16 * nv, hipMemcpyHostToDevice, ctx->stream));
    FFHIP_CHECK(hipMemcpyAsync(m->elems, tris, 12 * nt, hipMemcpyHostToDevice, ctx->stream));
    if (nbe) {
      FFHIP_CHECK(hipMemcpyAsync(m->belems, bedges, 8 * nbe, hipMemcpyHostToDevice, ctx->stream));
      FFHIP_CHECK(hipMemcpyAsync(m->blab, blab, 4 * nbe, hipMemcpyHostToDevice, ctx->stream));
    }
    FFHIP_CHECK(hipStreamSynchronize(ctx->stream));
    *out = m;
  });
}

int ffhip_mesh_info(ffhip_mesh m, int64_t *nv, int64_t *nt, int64_t *nbe) {
  return guard([&] {
    FFHIP_REQUIRE(m, FFHIP_ERR_ARG, "ffhip_mesh_info: null mesh");
    if (nv) *nv = m->nv;
    if (nt) *nt = m->nt;
    if (nbe) *nbe = m->nbe;
  });
}

int ffhip_mesh_download(ffhip_mesh m, double *xyz, int32_t *elems, int32_t *belems,
                        int32_t *blab) {
  return guard([&] {
    FFHIP_REQUIRE(m, FFHIP_ERR_ARG, "ffhip_mesh_download: null mesh");
    hipStream_t s = m->ctx->stream;
    if (xyz) FFHIP_CHECK(hipMemcpyAsync(xyz, m->xyz, 8 * m->dim * m->nv, hipMemcpyDeviceToHost, s));
    if (elems) FFHIP_CHECK(hipMemcpyAsync(elems, m->elems, 4 * m->nloc * m->nt, hipMemcpyDeviceToHost, s));
    if (belems && m->nbe)
      FFHIP_CHECK(hipMemcpyAsync(belems, m->belems, 4 * m->nbloc * m->nbe, hipMemcpyDeviceToHost, s));
    if (blab && m->nbe) FFHIP_CHECK(hipMemcpyAsync(blab, m->blab, 4 * m->nbe, hipMemcpyDeviceToHost, s));
    FFHIP_CHECK(hipStreamSynchronize(s));
  });
}

int ffhip_mesh_free(ffhip_mesh m) {
  return guard([&] {
    if (!m) return;
    (void)hipStreamSynchronize(m->ctx->stream);
    dfree(m->xyz); dfree(m->elems); dfree(m->belems); dfree(m->blab);
    dfree(m->v2e_ptr); dfree(m->v2e); dfree(m->v2e_inv);
    dfree(m->b2e_ptr); dfree(m->b2e);
    delete m;
  });
}

}  // extern "C"
