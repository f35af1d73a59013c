// lg_host.h — host-side objects behind the C ABI handles, shared by lg_api.hip (the ABI and
// scene compilation) and lg_pipeline.hip (the batched frame pipeline).
#pragma once

#include <atomic>
#include <memory>
#include <string>
#include <vector>

#include "lg_internal.h"

namespace lg {

// ---- device buffer ---------------------------------------------------------------------------
struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { reset(); }
  void reset() {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  }
  // Grows to at least `need` bytes (contents are not kept).
  int ensure(size_t need);
  template <typename U>
  U* as() const {
    return reinterpret_cast<U*>(p);
  }
};

// Pinned host staging buffer.
struct PinnedBuf {
  void* p = nullptr;
  size_t bytes = 0;
  PinnedBuf() = default;
  PinnedBuf(const PinnedBuf&) = delete;
  PinnedBuf& operator=(const PinnedBuf&) = delete;
  ~PinnedBuf() { reset(); }
  void reset() {
    if (p) (void)hipHostFree(p);
    p = nullptr;
    bytes = 0;
  }
  int ensure(size_t need);
  template <typename U>
  U* as() const {
    return reinterpret_cast<U*>(p);
  }
};

struct StageRec {
  std::string name;
  hipEvent_t start, stop;
  uint64_t work;
  uint64_t work2 = 0;
};

struct Pipeline;
struct PipelineDeleter {
  void operator()(Pipeline* p) const;
};
struct SmScratch;  // string-mod generator buffers (lg_stringmod.hip)
struct SmScratchDeleter {
  void operator()(SmScratch* p) const;
};

// Device scratch of an ordered download that its context keeps for the next one, at most: more is
// given back when the call ends.
constexpr size_t kKeptScratch = 64u << 20;
struct OrderScratch;  // ordered downloads (lg_order.hip)
struct OrderScratchDeleter {
  void operator()(OrderScratch* s) const;
};

int fail(int code, const std::string& msg);

// ---- kernel launchers (lg_trace.hip, lg_accum.hip) ---------------------------------------------
// LDS bytes of a trace workgroup; `chunk` bounce generations per launch (1 .. trace_max_chunk()).
template <typename T>
size_t trace_lds_bytes(int n_recs, int n_objs, int n_verts, uint32_t chunk);
uint32_t trace_max_chunk();
// One trace launch: generations gen .. gen + chunk - 1 of every scene; launch_ix = its index in
// the frame (it picks the ping-pong ray queues).
template <typename T>
hipError_t launch_trace(const SceneDesc* descs, int n_scenes, uint32_t gen, uint32_t chunk, uint32_t launch_ix,
                        const uint32_t* item_pre, BatchCtl* ctl, uint32_t rpi, int cap_recs, int cap_objs,
                        int cap_verts, uint32_t* item_pre_next, int grid, hipStream_t stream);
int trace_block();
bool tile_size_supported(int tile);
// Exclusive scan of n u32 (out may not alias in). scratch holds scan_scratch_elems(n) u32. With
// total (zeroed by an earlier kernel): *total += the 64-bit sum of the elements, or bit 63 set when
// 2048 consecutive elements sum to 2^32 or more (the 32-bit offsets wrapped).
uint64_t scan_scratch_elems(uint64_t n);
hipError_t launch_scan_exclusive(const uint32_t* in, uint32_t* out, uint64_t n, uint32_t* scratch, hipStream_t st,
                                 unsigned long long* total);
hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t st);
hipError_t launch_iota_u64(uint64_t* p, uint64_t n, hipStream_t st);  // p[i] = i
// bin workgroups per compute unit (as many as the LDS allows run at once)
constexpr uint32_t kBinWaves = 6;
// The bin layout (chunk_pre, cbase: see the kernels) and the count pass: row_count are the row totals
// (2 per tile, zeroed by the caller), places the [scene][chunk][tile][axis] matrix.
hipError_t launch_bin_count(const SceneDesc* descs, int n_scenes, uint32_t chunk_min, uint32_t target,
                            uint32_t* chunk_pre, uint32_t* cbase, BatchCtl* ctl, uint32_t* places, uint32_t* row_count,
                            int max_tiles, int grid, hipStream_t st);
// The fill pass, of the same grid: row_start are the rows' starts.
hipError_t launch_bin_fill(const SceneDesc* descs, int n_scenes, uint32_t* chunk_pre, uint32_t* cbase, BatchCtl* ctl,
                           uint32_t* places, uint32_t* row_start, uint32_t* pairs, uint64_t pairs_cap, int max_tiles,
                           int grid, hipStream_t st);
// row_count and row_start hold 2 * n_tiles_total + 1 entries (row_count's last is zero): per tile
// its y-major and x-major pairs, and where they start; scan_scratch holds
// work_items_scratch_elems(n_tiles_total) u32.
uint64_t work_items_scratch_elems(int n_tiles_total);
// layers: pairs of rows per tile (1, or a SCENE_RUNS frame's layers)
hipError_t launch_work_items(const SceneDesc* descs, const uint32_t* tile_scene, int n_tiles_total, int layers,
                             const uint32_t* row_count, uint32_t* row_start, uint32_t* scan_scratch, BatchCtl* ctl,
                             WorkItem* items, uint32_t items_cap, uint32_t* split_tiles, uint32_t split_cap,
                             uint64_t pairs_cap, uint32_t min_piece, uint32_t max_piece, uint32_t grid,
                             bool whole_images, hipStream_t st);
// Workgroups of the tile kernel per compute unit (launch_tile_accum).
int tile_groups_per_cu(int tile, bool packed_only, int block, bool runs);
hipError_t launch_tile_accum(const SceneDesc* descs, const uint32_t* pairs, const WorkItem* items,
                             const uint32_t* row_start, unsigned long long* split_fx, BatchCtl* ctl, int tile,
                             bool packed_only, int block, bool runs, bool count_work, int n_cu, hipStream_t st);
hipError_t launch_tile_merge(const SceneDesc* descs, const uint32_t* tile_scene, const uint32_t* row_start,
                             const uint32_t* split_tiles, const BatchCtl* ctl, unsigned long long* split_fx,
                             uint32_t split_cap, int tile, int n_cu, hipStream_t st);
uint64_t merge_slot_u64();
// The 64-bit LDS atomic issue-rate probe (lg_calibrate_lds_atomics): `sink` holds 2 * n_cu
// words; *wave_instructions = the atomic wave instructions the launch issues.
hipError_t launch_lds_atomic_rate(int n_cu, uint32_t iters, unsigned long long* sink, hipStream_t st,
                                  uint64_t* wave_instructions);
// lg_noalloc.hip: the device address of the static scratch of lg_accumulate_noalloc, looked up
// once per device (the device must be current); its size in bytes.
int noalloc_init(int device, hipStream_t st);
uint64_t noalloc_scratch_bytes();
// Clears (mode 0) or resolves (1) the n pixels of an image.
hipError_t launch_pixels(int mode, float4* accum, ushort4* out16, uint64_t n, hipStream_t st);

}  // namespace lg

struct lg_ctx {
  int device = 0;
  int n_cu = 256;
  hipStream_t stream = nullptr;
  std::atomic<int> children{0};  // live scenes, segment buffers, images and servers (any thread)
  bool closing = false;  // lg_ctx_destroy was called while children were alive
  bool profiling = false;
  bool use_graphs = true;
  bool packed_accum = true;   // two channels per LDS word for scenes whose deposits are all >= 0
  // Pieces: half a tile workgroup's even share, within [2048, 32768]. Below 2048 pairs the merge
  // costs what the balance gains, above, the piece at a light's centre is the frame's tail (tile
  // walk + merge, us, at 1024 / 2048 / 4096: 20k-ray frame 64 / 61 / 70, 75k-ray frame 93 / 91 /
  // 101, 60k lines with vertex colours 319 / 316 / 362); a cap of 8192 splits tiles for nothing
  // where the share is larger (8192 / 32768: 1M-ray frame 720 / 622, 1.6M segments at 4096x4096
  // 4350 / 3730, 20 uneven scenes 736 / 678).
  lg_tuning tune{1024u, 2048u, 32768u, 4u, 8u, 64u, 2u, 1024u};
  std::vector<lg::StageRec> pending;  // events of the current call
  std::vector<hipEvent_t> event_pool;
  std::vector<lg_stage_time> last_times;
  std::unique_ptr<lg::Pipeline, lg::PipelineDeleter> pipe;
  std::unique_ptr<lg::SmScratch, lg::SmScratchDeleter> sm;
  std::unique_ptr<lg::OrderScratch, lg::OrderScratchDeleter> order;
  lg::DevBuf encode_table;  // 65536 u8: the 8-bit encode of every half (built on first use)
  bool encode_table_ready = false;

  hipEvent_t get_event() {
    if (!event_pool.empty()) {
      hipEvent_t e = event_pool.back();
      event_pool.pop_back();
      return e;
    }
    hipEvent_t e;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
  }
};

struct lg_scene {
  lg_ctx* ctx = nullptr;
  std::vector<lg_object> objects;
  std::vector<lg_light> lights;
  bool dirty = true;
  std::vector<lg::Rec<double>> h_recs64;
  std::vector<int32_t> h_obj_rec;
  std::vector<double> h_verts64;
  int n_recs = 0, n_objs = 0, n_verts = 0;
  // The compiled scene on the device: one allocation, written with one copy; byte offsets of its
  // tables.
  lg::DevBuf tables;
  struct {
    size_t recs32, recs64, obj_n64, obj_flags, obj_rec, obj_box, medium, verts32, verts64, lights;
    size_t blocks, block_box, block_rec;  // culling blocks (CullBlock)
    size_t tree_rec;                      // first records of the Logic trees of more than two primitives
  } at{};
  template <typename U>
  const U* table(size_t off) const {
    return reinterpret_cast<const U*>(tables.as<char>() + off);
  }
  int n_blocks = 0;
  double reach = 0.0;         // largest |coordinate| that a ray starts from
  float medium_map[4] = {};
  int n_trees = 0;
  lg::DevBuf q0, q1;          // ray queues (QRay<double>)
  uint64_t q_cap = 0;         // rays per queue
  uint64_t seg_hint = 0;      // high-water segment count
  uint64_t n_primary = 0;
  float light_max = 0.0f;     // largest |light colour channel|
  bool light_nonneg = true;   // every light colour channel is >= 0 (so is every traced segment's)
};

struct lg_segments {
  lg_ctx* ctx = nullptr;
  uint32_t flags = 0;
  uint64_t count = 0, cap = 0;
  float max_abs = 0.0f;       // largest |colour channel| of the stored segments (host-side bound)
  bool nonneg = true;         // every colour channel of the stored segments is >= 0
  // both vertices of every stored segment have colour col0 (traced segments, uploads without
  // or with an identical color1, StringMods without modulo colours): col1 is not read
  bool one_color = true;
  lg::SceneHues hues;         // traced segments: the colours of their lights
  lg::SegRuns runs;           // segments of one colour each: their runs of equal colours, if few
  double extent[2] = {0.0, 0.0};  // with runs: mean |dx| and |dy| of a sample of the segments
  uint64_t n_rays = 0;        // traced segments: the scene's rays (keys hold their index); else 0
  lg::DevBuf pos, col0, col1, key, pos64;
  bool has_pos64 = false;
};

struct lg_image {
  lg_ctx* ctx = nullptr;
  lg_view view{};
  lg::DevBuf accum, out16;
  lg_blend blend{{LG_BF_ONE, LG_BF_ONE, LG_BO_ADD}, {LG_BF_SRC_ALPHA, LG_BF_ONE, LG_BO_ADD}, {0.f, 0.f, 0.f, 0.f}};
  uint32_t blend_code = lg::kBlendDefault;
  lg::DevBuf enc8;  // 8-bit encode output
};

namespace lg {

// ST_FRESH with ST_ACCUM: the frame clears, accumulates into and resolves every image (lg_render,
// lg_batch_render, the server), clear and resolve as part of the tile flushes.
enum Stage : uint32_t { ST_TRACE = 1u, ST_ACCUM = 2u, ST_FRESH = 4u };

struct Entry {
  lg_scene* scene = nullptr;
  lg_params params{};
  lg_segments* segs = nullptr;
  lg_image* img = nullptr;
};

int compile_scene(lg_scene* sc, hipStream_t st);
// Whatever is going to overwrite a buffer's segments (or move them: seg_ensure) forgets them first and
// publishes the new ones when they are complete, so that a call that fails in between leaves an empty
// buffer and not the old counts over other contents.
void seg_forget(lg_segments* s);
int seg_ensure(lg_segments* s, uint64_t cap, bool need64);
AccumView make_view(const lg_view& v, int tile);
int check_params(const lg_params* p);
// A scene, segment buffer, image or server of ctx was destroyed (frees ctx when it was
// closed and this was its last child).
void ctx_child_gone(lg_ctx* ctx);
void begin_call(lg_ctx* ctx);
void end_call(lg_ctx* ctx);
// per channel, max |blend factor| of a BlendCode word over colours with |channel| <= m
void blend_factor_bounds(uint32_t code, float m, const float k[4], float out[4]);
// The hues of a scene's traced segments (n = 0 when its lights are more than kMaxHues), and their
// form in a frame's descriptor.
SceneHues scene_hues(const lg_scene* sc);
void set_hues(SceneDesc& D, const SceneHues& h);
// The mean extent of a buffer's segments comes from kExtentSamples of them, the same wherever they
// came from: sample k of n segments, and the mean from the samples' end points.
constexpr int kExtentSamples = 64;
__host__ __device__ inline uint64_t extent_sample(int k, uint64_t n) {
  const uint64_t spread = (uint64_t)(k + 1) * 0x9E3779B97F4A7C15ull;  // (evenly, and in step with no pattern)
  return ((spread >> 32) * n) >> 32;  // (n < 2^32)
}
void set_extent(lg_segments& s, const float4* samples);
// Whether an accumulation into the view goes by runs; the layers of such a frame, and the descriptor of one of them
// from the whole scene's. All layers of a frame have the same tiles.
bool use_runs(const lg_segments& s, const lg_view& view, int n_cu);
int run_layers(const SegRuns& r);
SceneDesc run_layer(const SceneDesc& D, const SegRuns& r, int layer, int n_layers);
// Whether every value colour * factor is >= 0 for colour channels in [0, m].
bool blend_nonneg(uint32_t code, float m, const float k[4]);

// Runs `stages` for every entry as one batched frame on ctx's stream and waits for it.
int pipeline_run(lg_ctx* ctx, const std::vector<Entry>& entries, uint32_t stages);
void pipeline_destroy(lg_ctx* ctx);

// A batched frame in flight on a stream of its own, with its own scratch and graph cache
// (the serving loop keeps several). start() validates and launches; poll() returns with
// *finished once the frame is complete (relaunching it when a buffer overflowed).
struct FrameJob;
FrameJob* frame_job_new(lg_ctx* ctx);
void frame_job_free(FrameJob* job);
int frame_job_start(FrameJob* job, std::vector<Entry>&& entries, uint32_t stages);
int frame_job_poll(FrameJob* job, bool wait, bool* finished);
const std::vector<Entry>& frame_job_entries(const FrameJob* job);
size_t frame_job_scratch_bytes(const FrameJob* job);

struct StageScope {
  lg_ctx* ctx;
  size_t idx = (size_t)-1;
  StageScope(lg_ctx* c, const char* name, uint64_t work);
  ~StageScope();
};

}  // namespace lg
