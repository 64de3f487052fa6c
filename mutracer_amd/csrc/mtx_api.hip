// C ABI of libmtx: handle registry, BLAS / scene acceleration objects and the
// ray-query kernels.
#include <atomic>
#include <map>
#include <mutex>

#include "mtx_fetch.h"
#include "mtx_registry.h"
#include "mtx_walk.h"

namespace mtx {

// ------------------------------------------------------------------ registry
Registry &registry() {
  static Registry r;
  return r;
}

uint64_t Registry::next() { return nextHandle.fetch_add(1); }

// ------------------------------------------------------------- trace kernels
constexpr int kTraceBlock = 128;

__global__ void k_zero_counters(uint32_t *__restrict__ c) {
  if (threadIdx.x < (uint32_t)kXcds) c[threadIdx.x * kCtrStride] = 0u;
}

// Ray queries: the traversal of the wavefront trace (closest hit) and shadow
// (any hit) kernels over a caller's rays; `ctr` holds the queue's chunk
// counters, zeroed before the launch.
// Mode 4 uses no counters, for queries recorded into a graph (graphs recorded
// on one stream may be replayed on several at once, where they would share
// that stream's counters) and on hipStreamPerThread, which is another stream
// in each thread. Elsewhere mode 1 stays: it is 6 to 9% faster
// where waves take many chunks (6M occlusion rays in 24 x 60k triangles 2.65 ms
// against 2.82) and on short queries (40k 0.277 against 0.285), slower in
// between (1.5M 0.99 against 0.92).
template <int kMode>  // 0 closest, 1 any, 2 counters, 3 closest with visit counts, 4 any, chunks shared out beforehand
__global__ void __launch_bounds__(kTraceBlock, kMode == 1 || kMode == 4 ? kOcclusionWaves : kTraceWaves)
k_trace(const AccelView *__restrict__ viewp, const mtx_ray *__restrict__ rays, uint32_t n,
        mtx_hit *__restrict__ hits, uint32_t *__restrict__ out, uint32_t flags, int32_t *__restrict__ spill,
        uint32_t *__restrict__ ctr) {
  constexpr bool kAny = kMode == 1 || kMode == 4;
  __shared__ int32_t lds[kMinLdsStack * kTraceBlock];
  const AccelView acc = *viewp;
  // Only the lanes that take rays have a spill slice.
  const uint32_t wave = blockIdx.x * (kTraceBlock / 64) + (threadIdx.x >> 6);
  const uint32_t lanes = queue_lanes(n, gridDim.x * (kTraceBlock / 64));
  LaneStackT<kMinLdsStack> st{
      lds + threadIdx.x, kTraceBlock,
      spill + ((size_t)wave * lanes + min(lane_id(), lanes - 1u)) * (kMaxStack - kMinLdsStack)};
  const bool doubleSided = kAny || (flags & MTX_TRACE_DOUBLE_SIDED) != 0;
  auto load = [&](uint32_t i, RayIn &r) {
    const float4 *r4 = reinterpret_cast<const float4 *>(rays + i);
    const float4 a = r4[0], b = r4[1];
    r.o = f3of(a);
    r.d = f3of(b);
    r.tMax = kAny ? fminf(fmaxf(a.w, 0.0f), kRayMaxDistance) : kRayMaxDistance;
    r.curTri = r.curSlot = -1;
    r.id = i;
  };
  auto covers = [](uint32_t, int32_t, int32_t, f3) { return true; };
  auto hit = [&](uint32_t i, float t, f3 b, int32_t slot, int32_t, int32_t source) {
    if (kMode == 2) return;
    hits[i] = mtx_hit{1u, fint(acc.slots[slot].c2.w), source, t, {b.x, b.y, b.z}, 0u};
  };
  auto done = [&](uint32_t i, bool any, const TraceCounters &c) {
    if (kAny) {
      out[i] = any ? 1u : 0u;
      return;
    }
    if (kMode == 2) {
      out[(size_t)i * 3] = c.boxes;
      out[(size_t)i * 3 + 1] = c.tris;
      out[(size_t)i * 3 + 2] = c.instances;
      return;
    }
    if (!any) hits[i] = mtx_hit{0u, -1, -1, kRayMaxDistance, {0.0f, 0.0f, 0.0f}, 0u};
    if (kMode == 3) hits[i].visits = c.boxes + c.tris;
  };
  trace_queue<kAny, kMode == 2 || kMode == 3, false, false, false, kMode == 4>(
      n, ctr, acc, doubleSided, st, load, hit, covers, done);
}

// Spill slices of the traversal stacks and chunk counters of the ray queries,
// one set per stream: launches of one stream follow one another. `m` is held
// over a query's launches (its counters are zeroed by one and used by the
// next, and another thread's pair on the stream must not come in between).
struct StreamScratch {
  std::mutex m;
  DevBuf<int32_t> spill;
  DevBuf<uint32_t> counters;
  std::weak_ptr<OwnStream> last;  // whose launches used `spill` last, in place of this stream's
  hipEvent_t used = nullptr;      // their end, once another's have to wait for it
  ~StreamScratch() {
    if (used) (void)hipEventDestroy(used);
  }
};
static std::mutex gScratchesMutex;
static std::map<std::pair<int, hipStream_t>, std::shared_ptr<StreamScratch>> gScratches;

static std::shared_ptr<StreamScratch> scratch_of(hipStream_t s) {
  int dev = 0;
  MTX_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> g(gScratchesMutex);
  auto &b = gScratches[{dev, s}];
  if (!b) b = std::make_shared<StreamScratch>();
  return b;
}

uint32_t trace_grid() {
  static uint32_t grid = 0;
  if (!grid) {
    int dev = 0, cus = 0;
    MTX_HIP(hipGetDevice(&dev));
    MTX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    grid = (uint32_t)std::max(8, cus) * 8u;
    grid = (grid + 7u) & ~7u;
  }
  return grid;
}

// Each lane owns kMaxStack - kLds entries at lane * (kMaxStack - kLds): sized
// for the smallest LDS depth any kernel uses. The caller holds S.m.
static int32_t *spill_of(StreamScratch &S, size_t lanes) {
  const size_t need = lanes * (kMaxStack - kMinLdsStack);
  if (S.spill.count < need) S.spill = DevBuf<int32_t>(need);
  return S.spill.ptr;
}
SpillLease::SpillLease(hipStream_t s, uint32_t blocks, uint32_t blockThreads)
    : scratch(scratch_of(s)), lock(scratch->m) {
  ptr = spill_of(*scratch, (size_t)blocks * blockThreads);
}
void SpillLease::enter(const std::shared_ptr<OwnStream> &own) {
  const auto last = scratch->last.lock();  // gone: its stream has been waited for
  if (last && last != own && hipStreamQuery(last->s) != hipSuccess) {  // not yet done
    (void)hipGetLastError();
    if (!scratch->used) MTX_HIP(hipEventCreateWithFlags(&scratch->used, hipEventDisableTiming));
    MTX_HIP(hipEventRecord(scratch->used, last->s));
    MTX_HIP(hipStreamWaitEvent(own->s, scratch->used, 0));
  }
  scratch->last = own;
}
// Whether launches on s are being recorded into a graph.
static bool recording(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (!s) return false;  // the null stream cannot be
  if (hipStreamIsCapturing(s, &st) != hipSuccess) (void)hipGetLastError();
  return st == hipStreamCaptureStatusActive;
}

static const void *trace_kernel(int mode) {
  return mode == 0   ? (const void *)k_trace<0>
         : mode == 1 ? (const void *)k_trace<1>
         : mode == 2 ? (const void *)k_trace<2> : (const void *)k_trace<3>;
}
// Blocks of a query of n rays: at most `most` (a multiple of 8, one share per
// XCD), and at most one wave per ray (short queries run with one ray or a few
// per wave, see WorkQueue).
static uint32_t query_grid(uint32_t n, uint32_t most) {
  constexpr uint32_t wpb = kTraceBlock / 64;
  return std::max<uint32_t>(8u, std::min<uint64_t>(most, ((uint64_t)n + wpb - 1) / wpb + 7) & ~7u);
}
static uint32_t resident_grid(int mode) {
  static uint32_t bpc[4] = {0, 0, 0, 0};
  if (!bpc[mode]) {
    int b = 0;
    MTX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, trace_kernel(mode), kTraceBlock, 0));
    bpc[mode] = (uint32_t)std::max(1, b);
  }
  return trace_grid() / 8u * bpc[mode];
}
static void launch_query(int mode, uint32_t grid, const Accel &A, const mtx_ray *rays, uint32_t n, mtx_hit *hits,
                         uint32_t *out, uint32_t flags, int32_t *spill, uint32_t *ctr, hipStream_t s) {
  if (mode != 4) hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, s, ctr);
  const dim3 g(grid), b(kTraceBlock);
  switch (mode) {
    case 0: hipLaunchKernelGGL(k_trace<0>, g, b, 0, s, A.view.ptr, rays, n, hits, out, flags, spill, ctr); break;
    case 1: hipLaunchKernelGGL(k_trace<1>, g, b, 0, s, A.view.ptr, rays, n, hits, out, flags, spill, ctr); break;
    case 2: hipLaunchKernelGGL(k_trace<2>, g, b, 0, s, A.view.ptr, rays, n, hits, out, flags, spill, ctr); break;
    case 3: hipLaunchKernelGGL(k_trace<3>, g, b, 0, s, A.view.ptr, rays, n, hits, out, flags, spill, ctr); break;
    default: hipLaunchKernelGGL(k_trace<4>, g, b, 0, s, A.view.ptr, rays, n, hits, out, flags, spill, ctr); break;
  }
  MTX_HIP(hipGetLastError());
}

static void launch_trace(int mode, const Accel &A, const mtx_ray *rays, uint32_t n, mtx_hit *hits, uint32_t *out,
                         uint32_t flags, hipStream_t s) {
  MTX_REQUIRE(A.max_stack() <= (uint32_t)kMaxStack, MTX_INVALID_STATE, "scene deeper than the traversal stack");
  if (!n) return;
  if (mode == 0 && (flags & MTX_TRACE_COUNT)) mode = 3;
  // The same grid recorded or not: the scratch of a query made before suffices.
  const uint32_t grid = query_grid(n, resident_grid(mode));
  if (mode == 1 && (s == hipStreamPerThread || recording(s))) mode = 4;
  auto S = scratch_of(s);
  std::lock_guard<std::mutex> g(S->m);
  const uint32_t waves = grid * (kTraceBlock / 64);
  int32_t *spill = spill_of(*S, (size_t)waves * queue_lanes(n, waves));
  if (mode != 4 && !S->counters.ptr) S->counters.alloc(kXcds * kCtrStride);
  launch_query(mode, grid, A, rays, n, hits, out, flags, spill, S->counters.ptr, s);
}

// ----------------------------------------------- allocation-free ray query
// mtx_trace_closest_noalloc runs k_trace<0> on a fixed persistent grid of
// kNoAllocBlocks blocks whose traversal-stack spill slices and chunk counters
// live in `scratch`, a file-scope device array: each device holds its own copy
// from module load until the process ends, and nothing is allocated per call.
constexpr uint32_t kNoAllocBlocks = 1024;
constexpr size_t kNoAllocSpillInts = (size_t)kNoAllocBlocks * kTraceBlock * (kMaxStack - kMinLdsStack);
constexpr size_t kNoAllocScratchBytes = kNoAllocSpillInts * sizeof(int32_t) + kXcds * kCtrStride * sizeof(uint32_t);
constexpr uint32_t kNoAllocMaxRays = 1u << 30;
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

// Device address of `scratch` per device, looked up once with that device
// current (the host-side symbol is only a stand-in, not a device address).
static std::mutex gScratchMutex;
static std::map<int, uint8_t *> gScratchPtr;

static uint8_t *scratch_for_current_device() {
  int dev = 0;
  MTX_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> g(gScratchMutex);
  auto it = gScratchPtr.find(dev);
  if (it != gScratchPtr.end()) return it->second;
  void *p = nullptr;
  MTX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  MTX_REQUIRE(p != nullptr, MTX_CONTEXT_FAILED, "scratch symbol has no device address");
  gScratchPtr[dev] = (uint8_t *)p;
  return (uint8_t *)p;
}

static void launch_trace_noalloc(const Accel &A, const mtx_ray *rays, uint32_t n, mtx_hit *hits, uint32_t flags,
                                 hipStream_t s) {
  MTX_REQUIRE(A.max_stack() <= (uint32_t)kMaxStack, MTX_INVALID_ARGUMENT, "scene deeper than the traversal stack");
  MTX_REQUIRE(n <= kNoAllocMaxRays, MTX_INVALID_ARGUMENT, "more than 2^30 rays in one allocation-free query");
  uint8_t *base = scratch_for_current_device();
  if (!n) return;
  int32_t *spill = reinterpret_cast<int32_t *>(base);
  uint32_t *ctr = reinterpret_cast<uint32_t *>(base + kNoAllocSpillInts * sizeof(int32_t));
  const int mode = (flags & MTX_TRACE_COUNT) ? 3 : 0;
  const uint32_t grid = query_grid(n, std::min<uint32_t>(resident_grid(mode), kNoAllocBlocks));
  launch_query(mode, grid, A, rays, n, hits, nullptr, flags, spill, ctr, s);
}

}  // namespace mtx

using namespace mtx;

#define MTX_API_BEGIN try {
#define MTX_API_END(err, cap)                                     \
  }                                                               \
  catch (const mtx::Error &e) {                                   \
    set_error(err, cap, e.what());                                \
    return e.code;                                                \
  }                                                               \
  catch (const std::bad_alloc &) {                                \
    set_error(err, cap, "out of host memory");                    \
    return MTX_ERROR;                                             \
  }                                                               \
  catch (const std::exception &e) {                               \
    set_error(err, cap, e.what());                                \
    return MTX_ERROR;                                             \
  }

extern "C" {

uint32_t mtx_abi_version(void) { return MTX_ABI_VERSION; }

int32_t mtx_device_info(char *name, size_t cap, int32_t *cus) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return MTX_UNAVAILABLE;
  int dev = 0;
  hipDeviceProp_t p;
  if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&p, dev) != hipSuccess) return MTX_UNAVAILABLE;
  set_error(name, cap, std::string(p.name) + " " + p.gcnArchName);
  if (cus) *cus = p.multiProcessorCount;
  return MTX_OK;
}

int32_t mtx_blas_build(const float *positions, uint32_t vertex_count, const uint32_t *indices,
                       uint32_t triangle_count, uint32_t bins, uint32_t flags, mtx_handle *out, char *err,
                       size_t cap) {
  MTX_API_BEGIN
  MTX_REQUIRE(out, MTX_INVALID_ARGUMENT, "out_blas is NULL");
  MTX_REQUIRE(triangle_count == 0 || (positions && indices), MTX_INVALID_ARGUMENT, "positions/indices are NULL");
  MTX_REQUIRE(bins >= 2 && bins <= 64, MTX_INVALID_ARGUMENT, "bins must be in [2, 64]");
  auto B = build_blas(positions, vertex_count, indices, triangle_count, bins, (flags & MTX_INPUT_DEVICE) != 0, 0);
  auto &R = registry();
  std::lock_guard<std::mutex> g(R.m);
  uint64_t h = R.next();
  R.blas[h] = B;
  *out = h;
  return MTX_OK;
  MTX_API_END(err, cap)
}

int32_t mtx_blas_info(mtx_handle blas, uint32_t info[8]) {
  MTX_API_BEGIN
  auto B = registry().get_blas(blas);
  MTX_REQUIRE(info, MTX_INVALID_ARGUMENT, "info is NULL");
  info[0] = B->topo.nodeCount;
  info[1] = B->topo.nodeCount * 2 + B->topo.primCount;
  info[2] = B->topo.maxDepth;
  info[3] = B->maxLeaf;
  info[4] = B->topo.primCount;
  uint64_t bytes = B->resident_bytes();
  info[5] = (uint32_t)bytes;
  info[6] = (uint32_t)(bytes >> 32);
  info[7] = B->layout.interiorCount;
  return MTX_OK;
  MTX_API_END(nullptr, 0)
}

int32_t mtx_blas_refit(mtx_handle blas, const float *positions, uint32_t vertex_count, const uint32_t *indices,
                       uint32_t triangle_count, uint32_t flags, uint32_t *rebuild_advised, char *err, size_t cap) {
  MTX_API_BEGIN
  auto B = registry().get_blas(blas);
  MTX_REQUIRE(positions && indices, MTX_INVALID_ARGUMENT, "positions/indices are NULL");
  MTX_REQUIRE(vertex_count == B->vertexInput && triangle_count == B->triangleInput, MTX_INVALID_ARGUMENT,
              "refit needs the build's vertex and triangle counts");
  const bool dev = (flags & MTX_INPUT_DEVICE) != 0;
  DevBuf<float> hpos;
  DevBuf<uint32_t> hidx;
  const float *dpos = positions;
  const uint32_t *didx = indices;
  if (!dev) {
    hpos.upload(positions, (size_t)vertex_count * 3, 0);
    hidx.upload(indices, (size_t)triangle_count * 3, 0);
    dpos = hpos.ptr;
    didx = hidx.ptr;
  }
  const bool advise = refit_blas(*B, dpos, didx, 0);
  if (rebuild_advised) *rebuild_advised = advise ? 1u : 0u;
  return MTX_OK;
  MTX_API_END(err, cap)
}

int32_t mtx_blas_export(mtx_handle blas, const uint32_t *indices, uint32_t *words, size_t capacity,
                        size_t *written, uint32_t *source_of_record) {
  MTX_API_BEGIN
  auto B = registry().get_blas(blas);
  size_t need = export_blas(*B, indices, nullptr, 0, nullptr, 0);
  if (written) *written = need;
  if (!words) return MTX_OK;
  if (capacity < need) return MTX_BUFFER_TOO_SMALL;
  export_blas(*B, indices, words, capacity, source_of_record, 0);
  return MTX_OK;
  MTX_API_END(nullptr, 0)
}

int32_t mtx_blas_destroy(mtx_handle blas) {
  auto &R = registry();
  std::lock_guard<std::mutex> g(R.m);
  return R.blas.erase(blas) ? MTX_OK : MTX_INVALID_HANDLE;
}

int32_t mtx_accel_create(const mtx_handle *blases, uint32_t blas_count, const mtx_instance_desc *instances,
                         uint32_t instance_count, uint32_t tlas_bins, uint32_t flags, mtx_handle *out, char *err,
                         size_t cap) {
  MTX_API_BEGIN
  MTX_REQUIRE(out, MTX_INVALID_ARGUMENT, "out_accel is NULL");
  MTX_REQUIRE(instance_count == 0 || instances, MTX_INVALID_ARGUMENT, "instances is NULL");
  MTX_REQUIRE(tlas_bins >= 2 && tlas_bins <= 64, MTX_INVALID_ARGUMENT, "tlas_bins must be in [2, 64]");
  for (uint32_t i = 0; i < instance_count; i++)
    MTX_REQUIRE(instances[i].struct_size >= sizeof(mtx_instance_desc), MTX_INVALID_ARGUMENT,
                "mtx_instance_desc.struct_size too small");
  std::vector<std::shared_ptr<Blas>> bl;
  for (uint32_t i = 0; i < blas_count; i++) bl.push_back(registry().get_blas(blases[i]));
  auto A = build_accel(bl, instances, instance_count, tlas_bins, flags, 0);
  auto &R = registry();
  std::lock_guard<std::mutex> g(R.m);
  uint64_t h = R.next();
  R.accel[h] = A;
  *out = h;
  return MTX_OK;
  MTX_API_END(err, cap)
}

int32_t mtx_accel_refit(mtx_handle accel, const mtx_instance_desc *instances, uint32_t count, const uint32_t *dirty,
                        uint32_t dirty_count, char *err, size_t cap) {
  MTX_API_BEGIN
  auto A = registry().get_accel(accel);
  MTX_REQUIRE(count == 0 || instances, MTX_INVALID_ARGUMENT, "instances is NULL");
  refit_accel(*A, instances, count, dirty, dirty_count, 0);
  return MTX_OK;
  MTX_API_END(err, cap)
}

int32_t mtx_accel_export_tlas(mtx_handle accel, uint32_t *tlas_words, size_t tlas_capacity, size_t *tlas_written,
                              uint32_t *instance_words, size_t instance_capacity, size_t *instance_written) {
  MTX_API_BEGIN
  auto A = registry().get_accel(accel);
  std::vector<uint32_t> tw, iw;
  export_tlas(*A, tw, iw, 0);
  if (tlas_written) *tlas_written = tw.size();
  if (instance_written) *instance_written = iw.size();
  if (tlas_words) {
    if (tlas_capacity < tw.size()) return MTX_BUFFER_TOO_SMALL;
    std::memcpy(tlas_words, tw.data(), tw.size() * 4);
  }
  if (instance_words) {
    if (instance_capacity < iw.size()) return MTX_BUFFER_TOO_SMALL;
    std::memcpy(instance_words, iw.data(), iw.size() * 4);
  }
  return MTX_OK;
  MTX_API_END(nullptr, 0)
}

int32_t mtx_accel_destroy(mtx_handle accel) {
  auto &R = registry();
  std::lock_guard<std::mutex> g(R.m);
  return R.accel.erase(accel) ? MTX_OK : MTX_INVALID_HANDLE;
}

int32_t mtx_trace_closest(mtx_handle accel, const mtx_ray *rays, uint32_t count, mtx_hit *hits, uint32_t flags,
                          void *stream) {
  MTX_API_BEGIN
  auto A = registry().get_accel(accel);
  MTX_REQUIRE(count == 0 || (rays && hits), MTX_INVALID_ARGUMENT, "rays/hits are NULL");
  launch_trace(0, *A, rays, count, hits, nullptr, flags, (hipStream_t)stream);
  return MTX_OK;
  MTX_API_END(nullptr, 0)
}

int32_t mtx_trace_closest_noalloc(mtx_handle accel, const mtx_ray *rays, uint32_t count, mtx_hit *hits,
                                  uint32_t flags, void *stream) {
  MTX_API_BEGIN
  auto A = registry().get_accel(accel);
  MTX_REQUIRE(count == 0 || (rays && hits), MTX_INVALID_ARGUMENT, "rays/hits are NULL");
  launch_trace_noalloc(*A, rays, count, hits, flags, (hipStream_t)stream);
  return MTX_OK;
  MTX_API_END(nullptr, 0)
}

int32_t mtx_trace_any(mtx_handle accel, const mtx_ray *rays, uint32_t count, uint32_t *occluded, void *stream) {
  MTX_API_BEGIN
  auto A = registry().get_accel(accel);
  MTX_REQUIRE(count == 0 || (rays && occluded), MTX_INVALID_ARGUMENT, "rays/occluded are NULL");
  launch_trace(1, *A, rays, count, nullptr, occluded, 0, (hipStream_t)stream);
  return MTX_OK;
  MTX_API_END(nullptr, 0)
}

int32_t mtx_trace_count(mtx_handle accel, const mtx_ray *rays, uint32_t count, uint32_t *counters, uint32_t flags,
                        void *stream) {
  MTX_API_BEGIN
  auto A = registry().get_accel(accel);
  MTX_REQUIRE(count == 0 || (rays && counters), MTX_INVALID_ARGUMENT, "rays/counters are NULL");
  launch_trace(2, *A, rays, count, nullptr, counters, flags, (hipStream_t)stream);
  return MTX_OK;
  MTX_API_END(nullptr, 0)
}

}  // extern "C"
