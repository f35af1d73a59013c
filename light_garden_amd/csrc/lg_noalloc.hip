// lg_noalloc.hip — lg_accumulate_noalloc: lg_accumulate without any device allocation.
//
// lg_accumulate sizes its frame scratch (the bin chunks' places, row totals, pair list, tile work items,
// merge slots, control block) on demand and grows it with hipMalloc when a frame overflows. Callers
// that may not allocate (a serving loop with a fixed footprint, a harness that forbids
// allocation) call this variant instead: the same kernels in the same order, with every
// scratch buffer carved out of one file-scope device array, `scratch`, of fixed size. Its
// limits are the array's partition below; a call beyond them fails with LG_E_CAPACITY before
// anything is deposited, and the image is left unchanged.
//
// Each device holds its own copy of `scratch`, from the moment the library is loaded until
// the process ends. Its device address is looked up once per device (hipGetSymbolAddress,
// lg_ctx_create calls noalloc_init with the device current) and only that address is ever
// handed to kernels. All calls on one device share the array: the library serialises them
// with a per-device lock (each call runs to completion before it returns), so calls that
// would overlap on one GPU from several threads wait for each other instead of racing.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>

#include "lg_host.h"

namespace lg {

// ---- limits of the static scratch --------------------------------------------------------------
constexpr int kNaMaxTiles = 4096;           // tiles of the image: 4096 x 4096 at 64 px, 2048 x 2048 at 32
constexpr uint64_t kNaPairs = 8ull << 20;   // segment-tile pairs of one call
constexpr uint32_t kNaSplit = 128;          // tiles split over several work items
constexpr uint32_t kNaBinTarget = 128;      // bin chunks of one call
constexpr uint32_t kNaChunkMin = 256;       // segments per bin chunk, at least
constexpr uint32_t kNaMinPiece = 4096;      // smallest tile work item (bounds the item count)
constexpr uint64_t kNaCounts = 2 * (uint64_t)kNaMaxTiles * (kNaBinTarget + kMaxLayers);  // [chunk][tile][axis]
constexpr uint64_t kNaRows = 2 * (uint64_t)kNaMaxTiles * kMaxLayers + 1;
constexpr uint64_t kNaScan = 64;  // >= work_items_scratch_elems(kNaMaxTiles)
constexpr uint64_t kNaItems = kNaMaxTiles + kNaPairs / kNaMinPiece + 1024;

constexpr uint64_t na_align(uint64_t x) { return (x + 255) & ~uint64_t(255); }
// byte offsets of the partition
constexpr uint64_t kOffDesc = 0;
constexpr uint64_t kOffCtl = na_align(kOffDesc + kMaxLayers * sizeof(SceneDesc));
constexpr uint64_t kOffChunkPre = na_align(kOffCtl + sizeof(BatchCtl));
constexpr uint64_t kOffCbase = na_align(kOffChunkPre + (kMaxLayers + 1) * 4);
constexpr uint64_t kOffCounts = na_align(kOffCbase + (kMaxLayers + 1) * 4);
constexpr uint64_t kOffRowCount = na_align(kOffCounts + kNaCounts * 4);
constexpr uint64_t kOffRowStart = na_align(kOffRowCount + kNaRows * 4);
constexpr uint64_t kOffScan = na_align(kOffRowStart + kNaRows * 4);
constexpr uint64_t kOffTileScene = na_align(kOffScan + kNaScan * 4);
constexpr uint64_t kOffSplitTiles = na_align(kOffTileScene + (uint64_t)kNaMaxTiles * 4);
constexpr uint64_t kOffItems = na_align(kOffSplitTiles + (uint64_t)kNaSplit * 4);
constexpr uint64_t kOffPairs = na_align(kOffItems + kNaItems * sizeof(WorkItem));
constexpr uint64_t kOffSplitFx = na_align(kOffPairs + kNaPairs * 4);
constexpr uint64_t kScratchBytes = na_align(kOffSplitFx + (uint64_t)kNaSplit * kMergeSlotU64 * 8);
static_assert(kScratchBytes < (64ull << 20), "the static scratch stays below 64 MiB");

// The scratch of every call on a device. In host code this name is only a handle for
// hipGetSymbolAddress; kernels get the looked-up device address.
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kNaMaxDevices = 64;
static std::mutex g_init_mu;
static void* g_scratch_dev[kNaMaxDevices];  // device address of `scratch`, per device
static std::mutex g_call_mu[kNaMaxDevices];

__global__ void na_put_desc_kernel(SceneDesc d, SceneDesc* dst) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *dst = d;
}

// Looks up the device address of `scratch` on `device` (which must be current) and zeroes
// its merge slots, which every later call leaves zeroed again. Once per device; any thread.
int noalloc_init(int device, hipStream_t st) {
  if (device < 0 || device >= kNaMaxDevices) return fail(LG_E_UNSUPPORTED, "noalloc: device ordinal above 63");
  std::lock_guard<std::mutex> lk(g_init_mu);
  if (g_scratch_dev[device]) return LG_OK;
  void* p = nullptr;
  hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) return hip_fail(e != hipSuccess ? e : hipErrorInvalidSymbol, "hipGetSymbolAddress(scratch)");
  unsigned char* base = static_cast<unsigned char*>(p);
  LG_HIP(launch_fill_u32(reinterpret_cast<uint32_t*>(base + kOffSplitFx), (uint64_t)kNaSplit * kMergeSlotU64 * 2, 0u,
                         st));
  LG_HIP(hipStreamSynchronize(st));
  g_scratch_dev[device] = p;
  return LG_OK;
}

uint64_t noalloc_scratch_bytes() { return kScratchBytes; }

}  // namespace lg

using namespace lg;

extern "C" {

int lg_accumulate_noalloc(lg_ctx* ctx, const lg_segments* segs, lg_image* img) {
  if (!ctx || !segs || !img) return fail(LG_E_INVALID, "ctx, segments or image is NULL");
  if (segs->ctx != ctx || img->ctx != ctx) return fail(LG_E_INVALID, "accumulate: objects of another context");
  if (ctx->device < 0 || ctx->device >= kNaMaxDevices) return fail(LG_E_UNSUPPORTED, "noalloc: device ordinal above 63");
  LG_HIP(hipSetDevice(ctx->device));
  if (segs->count == 0) return LG_OK;
  if (segs->count > 0xffffffffull) return fail(LG_E_UNSUPPORTED, "accumulate: more than 2^32 segments");
  void* dev = g_scratch_dev[ctx->device];
  if (!dev) {
    int rc = noalloc_init(ctx->device, ctx->stream);
    if (rc) return rc;
    dev = g_scratch_dev[ctx->device];
  }
  const int tile = (int)ctx->tune.tile;
  const AccumView view = make_view(img->view, tile);
  const int n_tiles = view.tiles_x * view.tiles_y;
  if (n_tiles > kNaMaxTiles)
    return fail(LG_E_CAPACITY, tile == 64 ? "lg_accumulate_noalloc: image above 4096x4096 pixels (4096 tiles)"
                                          : "lg_accumulate_noalloc: image above 2048x2048 pixels at 32-pixel tiles");

  // the descriptor lg_accumulate builds for its one entry (segments, image; no trace)
  SceneDesc D;
  std::memset(&D, 0, sizeof(D));
  D.seg_pos = gbl(segs->pos.as<float4>());
  D.seg_col = gbl(segs->col0.as<float4>());
  D.seg_col1 = gbl(segs->one_color ? nullptr : segs->col1.as<const float4>());
  D.seg_key = gbl(segs->key.as<uint64_t>());
  D.seg_cap = segs->cap;
  D.flags = SCENE_FIXED_COUNT;
  D.seg_fixed = segs->count;
  D.view = view;
  D.accum = gbl(img->accum.as<float4>());
  D.out16 = gbl(img->out16.as<ushort4>());
  D.color_max = segs->max_abs;
  D.blend_code = img->blend_code;
  for (int c = 0; c < 4; c++) D.blend_k[c] = img->blend.constant[c];
  blend_factor_bounds(D.blend_code, D.color_max, D.blend_k, D.factor_max);
  const bool packed = ctx->packed_accum && segs->nonneg && std::isfinite(segs->max_abs) &&
                      blend_nonneg(D.blend_code, segs->max_abs, D.blend_k);
  if (packed) D.flags |= SCENE_PACKED;
  const bool hues = packed && segs->hues.n && D.blend_code == kBlendDefault && tile == 64;
  if (hues) set_hues(D, segs->hues);
  D.row_stride = 1u;
  const bool runs = packed && tile == 64 && use_runs(*segs, img->view, ctx->n_cu);
  const int layers = runs ? run_layers(segs->runs) : 1;
  const uint32_t min_piece = std::max(kNaMinPiece, std::min(ctx->tune.min_piece, kPackedPiece));
  const uint32_t max_piece = std::max(min_piece, std::min(ctx->tune.max_piece, kPackedPiece));

  unsigned char* b = static_cast<unsigned char*>(dev);
  SceneDesc* d_desc = reinterpret_cast<SceneDesc*>(b + kOffDesc);
  BatchCtl* d_ctl = reinterpret_cast<BatchCtl*>(b + kOffCtl);
  uint32_t* chunk_pre = reinterpret_cast<uint32_t*>(b + kOffChunkPre);
  uint32_t* cbase = reinterpret_cast<uint32_t*>(b + kOffCbase);
  uint32_t* counts = reinterpret_cast<uint32_t*>(b + kOffCounts);
  uint32_t* row_count = reinterpret_cast<uint32_t*>(b + kOffRowCount);
  uint32_t* row_start = reinterpret_cast<uint32_t*>(b + kOffRowStart);
  uint32_t* scan = reinterpret_cast<uint32_t*>(b + kOffScan);
  uint32_t* tile_scene = reinterpret_cast<uint32_t*>(b + kOffTileScene);
  uint32_t* split_tiles = reinterpret_cast<uint32_t*>(b + kOffSplitTiles);
  WorkItem* items = reinterpret_cast<WorkItem*>(b + kOffItems);
  uint32_t* pairs = reinterpret_cast<uint32_t*>(b + kOffPairs);
  unsigned long long* split_fx = reinterpret_cast<unsigned long long*>(b + kOffSplitFx);

  const hipStream_t st = ctx->stream;
  BatchCtl hc;
  {
    std::lock_guard<std::mutex> lk(g_call_mu[ctx->device]);
    for (int l = 0; l < layers; l++) {
      hipLaunchKernelGGL(na_put_desc_kernel, dim3(1), dim3(64), 0, st, runs ? run_layer(D, segs->runs, l, layers) : D,
                         d_desc + l);
      LG_HIP(hipGetLastError());
    }
    LG_HIP(launch_fill_u32(reinterpret_cast<uint32_t*>(d_ctl), sizeof(BatchCtl) / 4, 0u, st));
    LG_HIP(launch_fill_u32(tile_scene, (uint64_t)n_tiles, 0u, st));
    LG_HIP(launch_fill_u32(row_count, 2 * (uint64_t)n_tiles * layers + 1, 0u, st));
    const int bin_grid = ctx->n_cu * (int)kBinWaves;
    LG_HIP(launch_bin_count(d_desc, layers, kNaChunkMin, kNaBinTarget, chunk_pre, cbase, d_ctl, counts, row_count,
                            n_tiles, bin_grid, st));
    LG_HIP(launch_work_items(d_desc, tile_scene, n_tiles, layers, row_count, row_start, scan, d_ctl, items, (uint32_t)kNaItems,
                             split_tiles, kNaSplit, kNaPairs, min_piece, max_piece, (uint32_t)ctx->n_cu, false, st));
    LG_HIP(launch_bin_fill(d_desc, layers, chunk_pre, cbase, d_ctl, counts, row_start, pairs, kNaPairs, n_tiles,
                           bin_grid, st));
    LG_HIP(launch_tile_accum(d_desc, pairs, items, row_start, split_fx, d_ctl, tile, packed,
                             hues ? 1024 : (int)ctx->tune.tile_block, runs, false, ctx->n_cu, st));
    LG_HIP(launch_tile_merge(d_desc, tile_scene, row_start, split_tiles, d_ctl, split_fx, kNaSplit, tile, ctx->n_cu,
                             st));
    LG_HIP(hipMemcpyAsync(&hc, d_ctl, sizeof(BatchCtl), hipMemcpyDeviceToHost, st));
    LG_HIP(hipStreamSynchronize(st));
  }
  // an overflow turned the tile stage into a no-op: nothing was deposited
  if (hc.flags & CTL_PAIRS_OVERFLOW)
    return fail(LG_E_CAPACITY, "lg_accumulate_noalloc: " + std::to_string(hc.total_pairs) +
                                   " segment-tile pairs, above the static scratch's 8388608");
  if (hc.flags & CTL_ITEMS_OVERFLOW) return fail(LG_E_CAPACITY, "lg_accumulate_noalloc: too many tile work items");
  if (hc.flags & CTL_SPLIT_OVERFLOW)
    return fail(LG_E_CAPACITY, "lg_accumulate_noalloc: " + std::to_string(hc.n_split) +
                                   " tiles split over several work items, above the static scratch's 128");
  return LG_OK;
}

}  // extern "C"
