// lg_order.hip — a traced segment buffer as trace_all's return value (tracer.rs:276-330): the
// vertex pairs in emission order, on the host.
//
// A trace appends its segments in no fixed order; ascending keys (ray << kPathBits | path) are the
// reference's order. A ray's segments are few, so the buffer is grouped by ray first (count,
// scan, place) and each segment then finds its rank among its ray's paths by comparing: three
// passes over 8 bytes per segment instead of the passes of a 64-bit sort, and every segment writes
// its record straight to its place. One copy per chunk brings the ordered records to pinned
// memory, from which the host writes the caller's arrays (doubles, and the colour once per
// vertex), a chunk ahead of it being on its way.
//
// The host did all of this on the downloaded arrays before (trace_all, us: 20k rays, 50,518 segments
// 1120 -> 328; 40k rays in FP64, 136k segments 2298 -> 400).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <new>
#include <numeric>
#include <thread>
#include <vector>

#include "lg_host.h"

namespace lg {

// Segments of one ray that are ranked by comparing (the work is the sum of their squares); a
// buffer with a longer ray is ordered on the host. (Ordered vertices, ms, by the device and by the host:
// 655k segments, the longest ray 16381: 7.3 and 14.2; 2.6M, 65491: 40 and 73; 1.0M, 261625: 46 and 29.)
constexpr uint32_t kMaxRankedPerRay = 65536;
constexpr int kOrderBlock = 256;
// Records per copy to the host, how many a thread of the host writes at least, and its threads. What
// takes the time is the caller's fresh pages, so the copies are few and the threads several. (Ordered
// vertices, us, medians of 40. 1.26M segments, chunks of 2^14 records 6900, 2^15 5900, 2^16 4400,
// 2^17 3900, 2^18 3700; one thread 5800, two 5600, four 3900, eight 3600. 5042 segments, a thread from
// 2^12 records on 76, from 2^13 to 2^16 60; 1.26M from 2^16 on 4140.)
constexpr uint64_t kChunkRecords = 1u << 17;
constexpr uint64_t kShareRecords = 1u << 14;
constexpr unsigned kHostThreads = 4;

struct OrderScratch {
  DevBuf count, start, scan, place, path, records;
  PinnedBuf stage[2];
  PinnedBuf flag;
  hipEvent_t landed[2] = {nullptr, nullptr};
  ~OrderScratch() {
    for (hipEvent_t e : landed)
      if (e) (void)hipEventDestroy(e);
  }
};

void OrderScratchDeleter::operator()(OrderScratch* s) const { delete s; }

static size_t scratch_bytes(const OrderScratch& s) {
  size_t b = 0;
  for (const DevBuf* d : {&s.count, &s.start, &s.scan, &s.place, &s.path, &s.records}) b += d->bytes;
  return b;
}

// One segment as the host reads it: 32 bytes, 48 with FP64 end points.
struct Record32 {
  float4 pos, col;
};
struct alignas(16) Record64 {
  double pos[4];
  float4 col;
};

// count[ray] = segments of the ray; place[i] = how many of them were counted before segment i. A
// buffer whose keys name a ray that it does not have goes to the host too: *by_host ends the
// kernels that follow before they index by a ray.
__global__ __launch_bounds__(kOrderBlock) void order_count_kernel(const uint64_t* __restrict__ key, uint32_t n,
                                                                  uint32_t n_rays, uint32_t* count,
                                                                  uint32_t* __restrict__ place, uint32_t* by_host) {
  const uint32_t i = blockIdx.x * kOrderBlock + threadIdx.x;
  if (i >= n) return;
  const uint64_t ray = key[i] >> kPathBits;
  if (ray >= n_rays) {
    *by_host = 1u;
    return;
  }
  const uint32_t a = atomicAdd(&count[ray], 1u);
  place[i] = a;
  if (a == kMaxRankedPerRay) *by_host = 1u;
}

// The paths grouped by ray, in arrival order.
__global__ __launch_bounds__(kOrderBlock) void order_group_kernel(const uint64_t* __restrict__ key, uint32_t n,
                                                                  const uint32_t* __restrict__ start,
                                                                  const uint32_t* __restrict__ place,
                                                                  uint32_t* __restrict__ path,
                                                                  const uint32_t* __restrict__ by_host) {
  const uint32_t i = blockIdx.x * kOrderBlock + threadIdx.x;
  if (i >= n || *by_host) return;
  const uint64_t k = key[i];
  path[start[k >> kPathBits] + place[i]] = (uint32_t)(k & ((1ull << kPathBits) - 1ull));
}

// Segment i's record to its ray's start plus its rank among the ray's paths (all different).
template <typename R>
__global__ __launch_bounds__(kOrderBlock) void order_write_kernel(const uint64_t* __restrict__ key, uint32_t n,
                                                                  const uint32_t* __restrict__ start,
                                                                  const uint32_t* __restrict__ path,
                                                                  const float4* __restrict__ pos,
                                                                  const double* __restrict__ pos64,
                                                                  const float4* __restrict__ col, R* __restrict__ out,
                                                                  const uint32_t* __restrict__ by_host) {
  const uint32_t i = blockIdx.x * kOrderBlock + threadIdx.x;
  if (i >= n || *by_host) return;
  const uint64_t k = key[i];
  const uint32_t mine = (uint32_t)(k & ((1ull << kPathBits) - 1ull));
  const uint32_t b = start[k >> kPathBits], e = start[(k >> kPathBits) + 1];
  uint32_t rank = 0;
#pragma unroll 8
  for (uint32_t j = b; j < e; j++) rank += path[j] < mine ? 1u : 0u;
  R r;
  if constexpr (sizeof(R) == sizeof(Record64)) {
    for (int c = 0; c < 4; c++) r.pos[c] = pos64[4 * (size_t)i + c];
  } else {
    r.pos = pos[i];
  }
  r.col = col[i];
  out[b + rank] = r;
}

// The caller's vertices of n records: two points and the colour twice.
template <typename R>
static void expand(const R* rec, uint64_t n, double* xy, float* rgba) {
  for (uint64_t i = 0; i < n; i++) {
    if constexpr (sizeof(R) == sizeof(Record64)) {
      std::memcpy(xy + 4 * i, rec[i].pos, 32);
    } else {
      xy[4 * i] = (double)rec[i].pos.x;
      xy[4 * i + 1] = (double)rec[i].pos.y;
      xy[4 * i + 2] = (double)rec[i].pos.z;
      xy[4 * i + 3] = (double)rec[i].pos.w;
    }
    std::memcpy(rgba + 8 * i, &rec[i].col, 16);
    std::memcpy(rgba + 8 * i + 4, &rec[i].col, 16);
  }
}

// part(begin, end) over n records, shared by a few threads from kShareRecords on (the host writes
// 64 bytes per record into fresh pages: one thread keeps up with neither the link nor the memory).
template <typename F>
static void share(uint64_t n, F&& part) {
  const uint64_t parts = std::min<uint64_t>(kHostThreads, n / kShareRecords + 1);
  const uint64_t per = (n + parts - 1) / parts;
  std::thread th[kHostThreads];
  uint64_t begun = 1;  // part 0 is this thread's
  for (; begun < parts; begun++) {
    const uint64_t b = std::min(n, begun * per), e = std::min(n, b + per);
    try {
      th[begun] = std::thread([&part, b, e] { part(b, e); });
    } catch (...) {
      break;  // no more threads: the rest is this thread's
    }
  }
  part(0, std::min(n, per));
  if (begun < parts) part(std::min(n, begun * per), n);
  for (uint64_t p = 1; p < begun; p++) th[p].join();
}

// The indices of the keys in ascending order: a radix sort, 11 bits to a pass, over the bits that any
// key has. Keys in order already (uploads, StringMods) take the first pass over them only.
static std::vector<uint32_t> key_order(std::vector<uint64_t> key) {
  const uint64_t n = key.size();
  std::vector<uint32_t> order(n);
  std::iota(order.begin(), order.end(), 0u);
  if (std::is_sorted(key.begin(), key.end())) return order;
  uint64_t bits = 0;
  for (uint64_t k : key) bits |= k;
  std::vector<uint64_t> key2(n);
  std::vector<uint32_t> order2(n);
  constexpr int kDigit = 11;
  for (int shift = 0; shift < 64 && bits >> shift; shift += kDigit) {
    auto digit = [&](uint64_t k) { return (uint32_t)(k >> shift) & ((1u << kDigit) - 1u); };
    std::vector<uint32_t> at((1u << kDigit) + 1, 0u);
    for (uint64_t k : key) at[digit(k) + 1]++;
    for (uint32_t d = 0; d < 1u << kDigit; d++) at[d + 1] += at[d];
    for (uint64_t i = 0; i < n; i++) {
      const uint32_t to = at[digit(key[i])]++;
      key2[to] = key[i];
      order2[to] = order[i];
    }
    key.swap(key2);
    order.swap(order2);
  }
  return order;
}

// The buffer ordered by the host: any buffer, whatever its keys, and without device memory.
static int order_on_host(lg_segments* s, double* xy, float* rgba) {
  const uint64_t n = s->count;
  auto room = [](bool wanted, uint64_t m) { return std::unique_ptr<float[]>(wanted ? new float[m] : nullptr); };
  const auto pos = room(!s->has_pos64, 4 * n), c0 = room(true, 4 * n), c1 = room(!s->one_color, 4 * n);
  const std::unique_ptr<double[]> pos64(s->has_pos64 ? new double[4 * n] : nullptr);
  std::vector<uint64_t> key(n);
  int rc;
  if ((rc = lg_segments_download(s, pos.get(), c0.get(), c1.get(), key.data(), n, nullptr))) return rc;
  if (pos64 && (rc = lg_segments_download_pos64(s, pos64.get(), n, nullptr))) return rc;
  const std::vector<uint32_t> order = key_order(std::move(key));
  const float *const p = pos.get(), *const a = c0.get(), *const b = c1 ? c1.get() : c0.get();
  const double* const p64 = pos64.get();
  share(n, [&](uint64_t i, uint64_t e) {
    for (; i < e; i++) {
      const uint64_t k = order[i];
      for (int c = 0; c < 4; c++) xy[4 * i + c] = p64 ? p64[4 * k + c] : (double)p[4 * k + c];
      std::memcpy(rgba + 8 * i, a + 4 * k, 16);
      std::memcpy(rgba + 8 * i + 4, b + 4 * k, 16);
    }
  });
  return LG_OK;
}

template <typename R>
static int order_on_device(lg_segments* s, OrderScratch& S, double* xy, float* rgba, bool* done) {
  lg_ctx* ctx = s->ctx;
  hipStream_t st = ctx->stream;
  const uint64_t n = s->count, n_rays = s->n_rays;
  const uint64_t stage_records = std::min(n, kChunkRecords);
  int rc;
  *done = false;
  // count: a word per ray, the end, and the flag of a buffer for the host
  if ((rc = S.count.ensure((n_rays + 2) * 4)) || (rc = S.start.ensure((n_rays + 1) * 4)) ||
      (rc = S.scan.ensure(scan_scratch_elems(n_rays + 1) * 4)) || (rc = S.place.ensure(n * 4)) ||
      (rc = S.path.ensure(n * 4)) || (rc = S.records.ensure(n * sizeof(R))) ||
      (rc = S.stage[0].ensure(stage_records * sizeof(R))) || (rc = S.flag.ensure(16)))
    return rc;
  if (n > kChunkRecords && (rc = S.stage[1].ensure(stage_records * sizeof(R)))) return rc;
  for (hipEvent_t& e : S.landed)
    if (!e) LG_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  uint32_t* const by_host = S.count.as<uint32_t>() + n_rays + 1;
  const uint64_t* key = s->key.as<const uint64_t>();
  R* const records = S.records.as<R>();
  const dim3 grid((unsigned)((n + kOrderBlock - 1) / kOrderBlock)), block(kOrderBlock);
  LG_HIP(launch_fill_u32(S.count.as<uint32_t>(), n_rays + 2, 0u, st));
  hipLaunchKernelGGL(order_count_kernel, grid, block, 0, st, key, (uint32_t)n, (uint32_t)n_rays,
                     S.count.as<uint32_t>(), S.place.as<uint32_t>(), by_host);
  LG_HIP(hipGetLastError());
  LG_HIP(launch_scan_exclusive(S.count.as<const uint32_t>(), S.start.as<uint32_t>(), n_rays + 1,
                               S.scan.as<uint32_t>(), st, nullptr));
  hipLaunchKernelGGL(order_group_kernel, grid, block, 0, st, key, (uint32_t)n, S.start.as<const uint32_t>(),
                     S.place.as<const uint32_t>(), S.path.as<uint32_t>(), by_host);
  LG_HIP(hipGetLastError());
  hipLaunchKernelGGL(order_write_kernel<R>, grid, block, 0, st, key, (uint32_t)n, S.start.as<const uint32_t>(),
                     S.path.as<const uint32_t>(), s->pos.as<const float4>(), s->pos64.as<const double>(),
                     s->col0.as<const float4>(), records, by_host);
  LG_HIP(hipGetLastError());
  auto copy = [&](uint64_t chunk) -> int {
    const uint64_t b = chunk * kChunkRecords, m = std::min(kChunkRecords, n - b);
    LG_HIP(hipMemcpyAsync(S.stage[chunk & 1].p, records + b, m * sizeof(R), hipMemcpyDeviceToHost, st));
    LG_HIP(hipEventRecord(S.landed[chunk & 1], st));
    return LG_OK;
  };
  LG_HIP(hipMemcpyAsync(S.flag.p, by_host, 4, hipMemcpyDeviceToHost, st));
  if ((rc = copy(0))) return rc;
  for (uint64_t c = 0; c * kChunkRecords < n; c++) {
    if ((c + 1) * kChunkRecords < n && (rc = copy(c + 1))) return rc;
    LG_HIP(hipEventSynchronize(S.landed[c & 1]));
    if (*S.flag.as<const uint32_t>()) {  // nothing was written
      LG_HIP(hipStreamSynchronize(st));
      return LG_OK;
    }
    const uint64_t b = c * kChunkRecords, m = std::min(kChunkRecords, n - b);
    const R* const rec = S.stage[c & 1].as<const R>();
    share(m, [=](uint64_t i, uint64_t e) { expand(rec + i, e - i, xy + 4 * (b + i), rgba + 8 * (b + i)); });
  }
  *done = true;
  return LG_OK;
}

}  // namespace lg

using namespace lg;

extern "C" {

int lg_segments_download_vertices(lg_segments* s, double* xy, float* rgba, uint64_t cap_vertices,
                                  uint64_t* n_vertices) {
  if (!s || !n_vertices) return fail(LG_E_INVALID, "segments or n_vertices is NULL");
  const uint64_t n = s->count;
  *n_vertices = 2 * n;
  if (cap_vertices < 2 * n || (n && (!xy || !rgba))) return fail(LG_E_CAPACITY, "vertices: output too small");
  if (n == 0) return LG_OK;
  lg_ctx* ctx = s->ctx;
  LG_HIP(hipSetDevice(ctx->device));
  // rays are counted in 32 bits; segments that were not traced (no rays) are in order already,
  // and may carry a colour per vertex
  if (s->n_rays && s->n_rays < 0x7fffffffull) {
    if (!ctx->order) ctx->order.reset(new OrderScratch());
    bool done = false;
    const int rc = s->has_pos64 ? order_on_device<Record64>(s, *ctx->order, xy, rgba, &done)
                                : order_on_device<Record32>(s, *ctx->order, xy, rgba, &done);
    if (rc || scratch_bytes(*ctx->order) > kKeptScratch) {
      (void)hipStreamSynchronize(ctx->stream);
      ctx->order.reset();
    }
    if (rc == LG_E_OOM)
      (void)hipGetLastError();  // (no room for the scratch: nothing was launched)
    else if (rc || done)
      return rc;
  }
  try {
    return order_on_host(s, xy, rgba);
  } catch (const std::bad_alloc&) {
    return fail(LG_E_OOM, "vertices: host memory");
  }
}

}  // extern "C"
