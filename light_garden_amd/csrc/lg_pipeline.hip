// lg_pipeline.hip — one batched frame: clear, trace, accumulate and resolve any number of
// scenes in the same launches.
//
// Every stage's work list is built on the device from device-side counts (trace items per
// bounce generation, bin chunks, tile work items), and every kernel is persistent over its
// list, so a frame needs no host synchronisation until its end. Buffers are sized from
// capacities; the end-of-frame readback reports any overflow, the capacities grow and the
// frame runs again (this happens on the first frames of a scene only). Because the launch
// sequence is fixed for a given batch shape (buffers and sizes), it is captured once in a
// hipGraph and replayed.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "lg_host.h"

namespace lg {

// per scene: the u64 segment count, and one cache line further the u32 children per
// generation (the trace's appends add to both; apart, they do not contend for one L2 line)
constexpr size_t kCounterStride = 256;
constexpr size_t kGenCountOffset = 128;
constexpr uint32_t kChunkMin = 256;     // segments per bin chunk, at least
// Bin chunks per workgroup: 8, so that the persistent workgroups end close together although
// chunks of one segment count differ in pairs (image size, segment length), fewer (down to 2)
// when the [tile][axis][chunk] matrix would pass kBinMatrixMax entries (the largest images).
constexpr uint32_t kChunksPerBinGroup = 8;
constexpr uint64_t kBinMatrixMax = 1ull << 26;
static_assert(kGenCountOffset + 4 * kMaxGen <= kCounterStride, "counter stride");
// Pairs per tile work item: total / (2 * n_cu) + 1, clamped to [min_piece, max_piece]. A tile
// is split when it holds more than one piece. The merge buffer holds a slot per split tile:
// it starts at 2 * n_cu + 64 slots and grows to what frames report (overflow -> rerun).

// A part of a larger device allocation.
struct DevView {
  void* p = nullptr;
  template <typename U>
  U* as() const {
    return reinterpret_cast<U*>(p);
  }
};

// Byte offsets of a frame's parts in frame_in and stage_in, each a multiple of 128.
struct FrameLayout {
  size_t tile_scene, item_pre0, counters, ctl, row_count, total;
  FrameLayout(int n, int n_tiles, int layers) {
    auto up = [](size_t b) { return (b + 127) & ~size_t(127); };  // (the control block's lines)
    tile_scene = up((size_t)n * sizeof(SceneDesc));
    item_pre0 = tile_scene + up((size_t)n_tiles * 4);
    counters = item_pre0 + up((size_t)(n + 1) * 4);
    ctl = counters + (size_t)n * kCounterStride;
    row_count = ctl + up(sizeof(BatchCtl));
    total = row_count + up((size_t)(2 * n_tiles * layers + 1) * 4);
  }
  size_t out_bytes() const { return row_count - counters; }
};

struct Pipeline {
  // One allocation that a frame uploads with one copy: descs | tile_scene | item_pre0 |
  // counters | ctl | row_count (FrameLayout; the layout of stage_in, whose counters, control block
  // and row totals are the frame's zeros). One copy reads counters | ctl back.
  DevBuf frame_in;
  DevView descs, tile_scene, item_pre0, counters, ctl, row_count;
  DevBuf item_pre, chunk_pre, cbase, places, row_start, scan_scratch;
  DevBuf pairs, items;
  DevBuf split_tiles, split_fx;  // merge slots of tiles split over several items
  uint64_t pairs_cap = 1u << 20;
  uint32_t items_cap = 0;
  uint32_t split_cap = 0, split_min = 0;
  PinnedBuf stage_in;   // as frame_in
  PinnedBuf stage_out;  // counters | ctl
  // Captured frames keyed on their shape (sizes, knobs and every buffer address they bake
  // in), least recently used evicted first.
  struct Graph {
    std::vector<uint64_t> shape;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    uint64_t used = 0;
  };
  static constexpr size_t kMaxGraphs = 8;
  std::vector<Graph> graphs;
  uint64_t tick = 0;

  static void release(Graph& g) {
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
    if (g.graph) (void)hipGraphDestroy(g.graph);
    g.exec = nullptr;
    g.graph = nullptr;
  }
  Graph* find(const std::vector<uint64_t>& shape) {
    for (Graph& g : graphs)
      if (g.shape == shape) return &g;
    return nullptr;
  }
  // Room for one more graph.
  void make_room() {
    while (graphs.size() >= kMaxGraphs) {
      size_t lru = 0;
      for (size_t i = 1; i < graphs.size(); i++)
        if (graphs[i].used < graphs[lru].used) lru = i;
      release(graphs[lru]);
      graphs.erase(graphs.begin() + lru);
    }
  }
  ~Pipeline() {
    for (Graph& g : graphs) release(g);
  }
};

void PipelineDeleter::operator()(Pipeline* p) const { delete p; }

void pipeline_destroy(lg_ctx* ctx) { ctx->pipe.reset(); }

// Whether a scene's culling pass goes by its objects' boxes, which may not change a result. An FP32
// ray from far outside reports hits that it does not have, beyond any padding where it grazes a
// surface, and with them goes the FP64 rescan that they bring about: of 2M rays at 9 or 70 objects
// none came out otherwise from up to 100 units, 3 from 300, up to 2500 from 1000. Such scenes test
// every object. (FP64 rays carry a slack of their own, good below 1e20: walk_boxes.)
constexpr double kBoxReach = 64.0;
static bool scene_uses_boxes(const lg_ctx* ctx, const lg_scene* sc, bool fp64) {
  return sc->n_blocks > 0 && (uint32_t)sc->n_objs >= ctx->tune.bvh_min_objects &&
         sc->reach <= (fp64 ? 1e18 : kBoxReach);
}

// Workgroups of a trace launch over n scenes: as many as the chip holds at once, twice as many over
// several scenes, whose items take unequal times. The second half starts, without a trip to the cursor, as
// workgroups of the first end, and the items past them, off the cursor, are begun before the
// second half is through. (Trace launches of 1.4M rays in 20 scenes: 646 us with one time, 527 with
// two; 24 requests of a server in frames of several: no difference.)
static uint32_t trace_groups(const lg_ctx* ctx, int n) {
  return (uint32_t)ctx->n_cu * ctx->tune.trace_waves * (n > 1 ? 2u : 1u);
}

struct Layout {
  int n = 0;                         // descriptors: one per entry, or one per layer
  int layers = 1;                    // of a frame over segments in runs (SCENE_RUNS)
  bool fp64 = false;
  uint32_t max_bounce = 0;
  int cap_recs = 0, cap_objs = 0, cap_verts = 0;
  uint32_t chunk = 1;                // bounce generations per trace launch
  int n_tiles = 0, max_tiles = 0;
  int tile = 64;                     // screen tile edge of the frame
  bool packed_only = false;          // every accumulated scene keeps two channels per LDS word
  bool hues = false;                 // some scene's deposits are one LDS word (SCENE_HUES)
  bool runs = false;                 // the frame's tiles sum weights of runs (SCENE_RUNS)
  bool streams = false;              // every accumulated scene is walked as streams of samples
  uint64_t n_counts = 0;             // capacity of the per-frame [chunk][tile][axis] matrix
  uint32_t bin_target = 0;           // bin chunks per frame
  std::vector<int> tile_base;
};

SceneHues scene_hues(const lg_scene* sc) {
  SceneHues h;
  if (sc->lights.empty() || sc->lights.size() > (size_t)kMaxHues) return h;
  uint64_t ray = 0;
  for (const lg_light& l : sc->lights) {
    h.first_ray[h.n] = ray;
    for (int c = 0; c < 4; c++) h.color[h.n][c] = l.color[c];
    h.n++;
    ray += l.num_rays;
  }
  return h;
}

void set_hues(SceneDesc& D, const SceneHues& h) {
  D.flags |= SCENE_HUES;
  D.n_hues = h.n;
  for (int f = 0; f < h.n; f++) {
    const float* c = h.color[f];
    const int p = c[1] > c[0] ? (c[2] > c[1] ? 2 : 1) : (c[2] > c[0] ? 2 : 0);
    D.hue_ch[f] = p;
    D.hue_ray[f] = h.first_ray[f];
    D.hue_bound[f][0] = c[p];
    D.hue_bound[f][1] = c[3];
    for (int k = 0; k < 3; k++) D.hue_ratio[f][k] = c[p] > 0.0f ? (double)c[k] / (double)c[p] : 0.0;
  }
}

void set_extent(lg_segments& s, const float4* samples) {
  s.extent[0] = s.extent[1] = 0.0;
  int n = 0;
  for (int k = 0; k < kExtentSamples; k++) {
    const double dx = std::fabs((double)samples[k].z - samples[k].x), dy = std::fabs((double)samples[k].w - samples[k].y);
    if (!std::isfinite(dx) || !std::isfinite(dy)) continue;
    s.extent[0] += dx;
    s.extent[1] += dy;
    n++;
  }
  for (double& e : s.extent) e = n ? e / n : 0.0;
}

// Summing weights saves 0.4 ps per sample of the frame where the whole chip walks them (more where
// tiles and pieces are fewer than its workgroups). It costs each of a workgroup's tiles some 6 us for
// every layer after the first (its planes, phases and barriers) and 0.25 us for every plane, of which
// the channels' walk has about three. The samples are estimated from the segments' mean extent, a
// tile's piece as 88000 of them. (Accumulation, us, by weights and by channels. 4096x4096, 24 runs:
// 409600 StringMod lines 1143 and 1282, 102400 759 and 451; 1.6M lines of 400 px 1423 and 1131, in
// 12 runs 1033 and 1136; 25000 lines of 4 px in 7 runs 304 and 230, in one 208 and 229. 2048x2048,
// 24 runs: 409600 StringMod lines 510 and 668, 102400 278 and 249. 1920x1080, 100000 lines of 4 px
// in 24 runs 128 and 79, in 6 84 and 80; 400000 of 400 px in 12 runs 292 and 298. 256x256, 7 runs:
// 25600 StringMod lines 74 and 82, 1600 65 and 59.)
bool use_runs(const lg_segments& s, const lg_view& view, int n_cu) {
  if (s.runs.n == 0) return false;
  const uint64_t tiles = (uint64_t)((view.width + 63) / 64) * ((view.height + 63) / 64);
  const double rounds = (double)((tiles + n_cu - 1) / n_cu);
  const double cost = rounds * (6.0 * (run_layers(s.runs) - 1) + 0.25 * (s.runs.n - 3));
  const double px = std::max(std::min(s.extent[0] / (view.right - view.left), 1.0) * view.width,
                             std::min(s.extent[1] / (view.top - view.bottom), 1.0) * view.height);
  const double samples = (double)s.count * px;
  const double groups = std::min(std::max((double)tiles, samples / 88000.0), (double)n_cu);
  return 4e-7 * samples * n_cu / groups >= cost;
}

int run_layers(const SegRuns& r) { return (r.n + kRunPlanes - 1) / kRunPlanes; }

SceneDesc run_layer(const SceneDesc& D, const SegRuns& r, int layer, int n_layers) {
  SceneDesc d = D;
  const int per = (r.n + n_layers - 1) / n_layers;
  const int a = std::min(layer * per, r.n), b = std::min(a + per, r.n);
  const uint64_t first = a < r.n ? r.first[a] : D.seg_fixed;
  const uint64_t end = b < r.n ? r.first[b] : D.seg_fixed;
  d.flags |= SCENE_RUNS;
  d.seg_pos = D.seg_pos + first;
  d.seg_fixed = end - first;
  d.row_base = (uint32_t)layer;
  d.row_stride = (uint32_t)n_layers;
  d.n_runs = b - a;
  for (int f = 0; f < kRunPlanes; f++) {
    d.run_first[f] = f < d.n_runs ? (uint32_t)(r.first[a + f] - first) : 0xffffffffu;
    for (int c = 0; c < 4; c++) d.run_color[f][c] = f < d.n_runs ? r.color[a + f][c] : 0.0f;
  }
  return d;
}

// Whether every deposit of the segments into the image is non-negative (SCENE_PACKED).
static bool scene_packed(const lg_ctx* ctx, const lg_segments& segs, const lg_image& img) {
  return ctx->packed_accum && segs.nonneg && std::isfinite(segs.max_abs) &&
         blend_nonneg(img.blend_code, segs.max_abs, img.blend.constant);
}

// The pieces that the tiles' lists are cut into, and the share that they are measured by. Where the
// walk goes by streams a piece is half a workgroup's even share of the pairs, within the tuning's
// limits. Pair by pair each one takes longer, so the piece that ends last costs more than a merge:
// a quarter of the share, and at most 8192 pairs. (Accumulation, us, with pieces of half a compute
// unit's share up to 32768 pairs / with these: 32-pixel tiles, colours per vertex, 770k string-mod
// lines at 36x2111 5102 / 3513, 1.6M at 1024x1024 6843 / 5620; one channel per word, 770k lines at
// 36x2111 2136 / 1962, 800k at 640x480 1274 / 1168.)
struct TilePieces {
  uint32_t groups, min_piece, max_piece;
};
constexpr uint32_t kPairWalkPiece = 8192;
static int frame_block(const lg_ctx* ctx, const Layout& L) { return L.hues ? 1024 : (int)ctx->tune.tile_block; }
static TilePieces tile_pieces(const lg_ctx* ctx, const Layout& L) {
  TilePieces p;
  p.groups = (uint32_t)(ctx->n_cu * tile_groups_per_cu(L.tile, L.packed_only, frame_block(ctx, L), L.runs));
  p.min_piece = std::min(ctx->tune.min_piece, kPackedPiece);
  p.max_piece = std::min(ctx->tune.max_piece, kPackedPiece);
  if (!L.streams) {
    p.groups *= 2;
    p.max_piece = std::max(p.min_piece, std::min(p.max_piece, kPairWalkPiece));
  }
  return p;
}

// Stage events only where the caller asked for them (the synchronous entry points on the
// context's own stream).
struct Scope {
  StageScope* s = nullptr;
  Scope(lg_ctx* ctx, bool on, const char* name, uint64_t work) {
    if (on) s = new StageScope(ctx, name, work);
  }
  ~Scope() { delete s; }
};

static int enqueue(lg_ctx* ctx, Pipeline& P, hipStream_t st, bool profile, const Layout& L, uint32_t stages) {
  const int n = L.n;
  const bool whole = stages & ST_FRESH;
  SceneDesc* d_descs = P.descs.as<SceneDesc>();
  BatchCtl* d_ctl = P.ctl.as<BatchCtl>();
  const FrameLayout F(n, L.n_tiles, L.layers);
  LG_HIP(hipMemcpyAsync(P.frame_in.p, P.stage_in.p, F.total, hipMemcpyHostToDevice, st));
  if (stages & ST_TRACE) {
    Scope s(ctx, profile, L.fp64 ? "trace_fp64" : "trace", L.max_bounce);
    const int grid = (int)trace_groups(ctx, n);
    // generation 0's work list comes with the frame's upload; each later one is built by the last
    // workgroup of the previous launch
    uint32_t li = 0;  // launch index: `chunk` generations per launch
    for (uint32_t g = 0; g < L.max_bounce; g += L.chunk, li++) {
      uint32_t* const next_pre = P.item_pre.as<uint32_t>() + (size_t)li * (n + 1);
      const uint32_t* pre = li ? next_pre - (n + 1) : P.item_pre0.as<uint32_t>();
      uint32_t* next = g + L.chunk < L.max_bounce ? next_pre : nullptr;
      if (L.fp64)
        LG_HIP(launch_trace<double>(d_descs, n, g, L.chunk, li, pre, d_ctl, ctx->tune.rays_per_item, L.cap_recs,
                                    L.cap_objs, L.cap_verts, next, grid, st));
      else
        LG_HIP(launch_trace<float>(d_descs, n, g, L.chunk, li, pre, d_ctl, ctx->tune.rays_per_item, L.cap_recs,
                                   L.cap_objs, L.cap_verts, next, grid, st));
    }
  }
  if (stages & ST_ACCUM) {
    const int grid = ctx->n_cu * (int)kBinWaves;
    {
      Scope s(ctx, profile, "bin_count", 0);
      LG_HIP(launch_bin_count(d_descs, n, kChunkMin, L.bin_target, P.chunk_pre.as<uint32_t>(), P.cbase.as<uint32_t>(),
                              d_ctl, P.places.as<uint32_t>(), P.row_count.as<uint32_t>(), L.max_tiles, grid, st));
    }
    {
      Scope s(ctx, profile, "bin_scan", 2 * (uint64_t)L.n_tiles);
      const TilePieces tp = tile_pieces(ctx, L);
      LG_HIP(launch_work_items(d_descs, P.tile_scene.as<uint32_t>(), L.n_tiles, L.layers, P.row_count.as<uint32_t>(),
                               P.row_start.as<uint32_t>(), P.scan_scratch.as<uint32_t>(), d_ctl,
                               P.items.as<WorkItem>(), P.items_cap, P.split_tiles.as<uint32_t>(), P.split_cap,
                               P.pairs_cap, tp.min_piece, tp.max_piece, tp.groups, whole, st));
    }
    {
      Scope s(ctx, profile, "bin_fill", 0);
      LG_HIP(launch_bin_fill(d_descs, n, P.chunk_pre.as<uint32_t>(), P.cbase.as<uint32_t>(), d_ctl,
                             P.places.as<uint32_t>(), P.row_start.as<uint32_t>(), P.pairs.as<uint32_t>(), P.pairs_cap,
                             L.max_tiles, grid, st));
    }
    {
      Scope s(ctx, profile, "tile_accum", 0);
      LG_HIP(launch_tile_accum(d_descs, P.pairs.as<uint32_t>(), P.items.as<WorkItem>(), P.row_start.as<uint32_t>(),
                               P.split_fx.as<unsigned long long>(), d_ctl, L.tile, L.packed_only,
                               frame_block(ctx, L), L.runs, profile, ctx->n_cu, st));
    }
    {
      Scope s(ctx, profile, "tile_merge", 0);
      LG_HIP(launch_tile_merge(d_descs, P.tile_scene.as<uint32_t>(), P.row_start.as<uint32_t>(),
                               P.split_tiles.as<uint32_t>(), d_ctl, P.split_fx.as<unsigned long long>(), P.split_cap,
                               L.tile, ctx->n_cu, st));
    }
  }
  LG_HIP(hipMemcpyAsync(P.stage_out.p, P.counters.p, F.out_bytes(), hipMemcpyDeviceToHost, st));
  return LG_OK;
}

// One batched frame: its entries, its stages and the layout of its current attempt.
struct Batch {
  std::vector<Entry> E;
  uint32_t stages = 0;
  Layout L;
  size_t first_stage = 0;  // first stage event of the current attempt
};

static int batch_validate(lg_ctx* ctx, hipStream_t st, Batch& B) {
  const std::vector<Entry>& E = B.E;
  const uint32_t stages = B.stages;
  const int n = (int)E.size();
  const bool trace = stages & ST_TRACE, accum = stages & ST_ACCUM;
  int rc;
  Layout& L = B.L;
  L.n = n;
  // ---- validate ----
  for (int i = 0; i < n; i++) {
    const Entry& e = E[i];
    if (trace) {
      if (!e.scene || !e.segs) return fail(LG_E_INVALID, "batch: trace needs a scene and a segment buffer");
      if ((rc = check_params(&e.params))) return rc;
      if (e.scene->ctx != ctx || e.segs->ctx != ctx) return fail(LG_E_INVALID, "batch: objects of another context");
      bool f = (e.params.flags & LG_TRACE_FP64) != 0;
      if (i == 0) L.fp64 = f;
      if (f != L.fp64) return fail(LG_E_INVALID, "batch: mixed FP32/FP64 traces");
      if ((rc = compile_scene(e.scene, st))) return rc;
    }
    if (accum && !e.segs) return fail(LG_E_INVALID, "batch: accumulation needs a segment buffer");
    if (accum && !e.img) return fail(LG_E_INVALID, "batch: an image is needed");
    if (e.img && e.img->ctx != ctx) return fail(LG_E_INVALID, "batch: image of another context");
    for (int j = 0; j < i; j++) {
      if ((e.scene && e.scene == E[j].scene) || (e.segs && e.segs == E[j].segs) || (e.img && e.img == E[j].img))
        return fail(LG_E_INVALID, "batch: scenes, segment buffers and images must be distinct");
    }
  }

  return LG_OK;
}

// Sizes every buffer for the attempt, writes the descriptors and launches the frame on `st`
// (graph replay when its shape is known). Does not wait.
static int batch_launch(lg_ctx* ctx, Pipeline& P, hipStream_t st, bool profile, bool allow_graph, Batch& B) {
  const std::vector<Entry>& E = B.E;
  const uint32_t stages = B.stages;
  const bool trace = stages & ST_TRACE, accum = stages & ST_ACCUM;
  int rc;
  Layout& L = B.L;
  // Segments in runs of one colour, every deposit non-negative: the tiles sum weights (not with
  // 32-pixel tiles, whose kernels do not have that walk, nor where the flush is to clear and
  // resolve the image, which that of the weights does not)
  L.runs = accum && !trace && !(stages & ST_FRESH) && E.size() == 1 && ctx->tune.tile == 64 &&
           use_runs(*E[0].segs, E[0].img->view, ctx->n_cu) && scene_packed(ctx, *E[0].segs, *E[0].img);
  L.layers = L.runs ? run_layers(E[0].segs->runs) : 1;
  const int entries = (int)E.size();
  const int n = L.n = L.runs ? L.layers : entries;
  // ---- limits (what they refuse has changed no buffer) ----
  L.max_bounce = 0;
  L.cap_recs = L.cap_objs = L.cap_verts = 1;
  for (const Entry& e : E) {
    if (trace) {
      const lg_scene* sc = e.scene;
      L.max_bounce = std::max(L.max_bounce, e.params.max_bounce);
      L.cap_recs = std::max(L.cap_recs, sc->n_recs);
      L.cap_objs = std::max(L.cap_objs, sc->n_objs);
      L.cap_verts = std::max(L.cap_verts, sc->n_verts);
    }
  }
  if (trace) {
    // bounce generations per launch, fewer when the on-chip level buffers do not fit beside the
    // scene (results do not depend on it)
    L.chunk = std::max(1u, std::min(ctx->tune.trace_chunk, trace_max_chunk()));
    auto lds = [&](uint32_t chunk) {
      return L.fp64 ? trace_lds_bytes<double>(L.cap_recs, L.cap_objs, L.cap_verts, chunk)
                    : trace_lds_bytes<float>(L.cap_recs, L.cap_objs, L.cap_verts, chunk);
    };
    if (lds(1) > 64 * 1024) return fail(LG_E_UNSUPPORTED, "scene too large for the LDS-resident trace");
    while (L.chunk > 1 && lds(L.chunk) > 64 * 1024) L.chunk--;
  }
  // ---- layout ----
  L.tile_base.assign(n, 0);
  L.n_tiles = 0;
  L.max_tiles = 1;
  L.n_counts = 0;
  L.tile = (int)ctx->tune.tile;
  for (int i = 0; i < entries; i++) {
    const Entry& e = E[i];
    if (accum) {
      AccumView v = make_view(e.img->view, L.tile);
      int t = v.tiles_x * v.tiles_y;
      // the binning keeps one LDS counter per tile of an image
      if (t > 16384)
        return fail(LG_E_UNSUPPORTED, L.tile == 64 ? "accumulate: image above 8192x8192"
                                                   : "accumulate: image above 4096x4096 with 32-pixel tiles");
      L.tile_base[i] = L.n_tiles;
      L.n_tiles += t;
      L.max_tiles = std::max(L.max_tiles, t);
    }
  }
  {
    const uint64_t groups = (uint64_t)ctx->n_cu * kBinWaves;
    uint64_t t = kBinMatrixMax / (2 * (uint64_t)L.max_tiles);
    t = std::min<uint64_t>(t, kChunksPerBinGroup * groups);
    L.bin_target = (uint32_t)std::max<uint64_t>(t, 2 * groups);
  }
  // chunks hold at least total / bin_target segments, so a scene has at most
  // n_s * bin_target / total + 1 of them and the batch fewer than bin_target + n
  if (accum) L.n_counts = 2 * (uint64_t)L.max_tiles * (L.bin_target + (uint64_t)n);
  if (L.n_counts > 0xffffffffull) return fail(LG_E_UNSUPPORTED, "batch too large for one frame");
  // ---- queues and segments ----
  for (const Entry& e : E) {
    if (trace) {
      lg_scene* sc = e.scene;
      uint64_t qn = std::max<uint64_t>(sc->q_cap, std::min<uint64_t>(2 * sc->n_primary, 0xffffffffull));
      qn = std::max<uint64_t>(qn, 1);
      if ((rc = sc->q0.ensure(qn * sizeof(QRay<double>)))) return rc;
      if ((rc = sc->q1.ensure(qn * sizeof(QRay<double>)))) return rc;
      sc->q_cap = qn;
      uint64_t need = std::max<uint64_t>(sc->seg_hint + sc->seg_hint / 8,
                                         sc->n_primary * std::min<uint32_t>(e.params.max_bounce, 4u) + 1024);
      need = std::max<uint64_t>(need, e.segs->cap);
      if ((rc = seg_ensure(e.segs, need, L.fp64))) return rc;
      seg_forget(e.segs);
    }
  }
  // ---- scratch ----
  // pieces hold at least min_piece pairs, so a frame without pair overflow has fewer than
  // n_tiles + pairs_cap / min_piece items
  const uint32_t items_need =
      (uint32_t)std::min<uint64_t>(0xffffffffull, (uint64_t)L.n_tiles + P.pairs_cap / ctx->tune.min_piece + 1024);
  P.items_cap = std::max(P.items_cap, items_need);
  const FrameLayout F(n, L.n_tiles, L.layers);
  {
    if ((rc = P.frame_in.ensure(F.total))) return rc;
    char* fi = P.frame_in.as<char>();
    P.descs.p = fi;
    P.tile_scene.p = fi + F.tile_scene;
    P.item_pre0.p = fi + F.item_pre0;
    P.counters.p = fi + F.counters;
    P.ctl.p = fi + F.ctl;
    P.row_count.p = fi + F.row_count;
  }
  if ((rc = P.item_pre.ensure((size_t)kMaxGen * (n + 1) * 4))) return rc;
  if ((rc = P.chunk_pre.ensure((size_t)(n + 1) * 4))) return rc;
  if ((rc = P.cbase.ensure((size_t)(n + 1) * 4))) return rc;
  if ((rc = P.places.ensure(std::max<uint64_t>(L.n_counts, 1) * 4))) return rc;
  if ((rc = P.scan_scratch.ensure(work_items_scratch_elems(L.n_tiles * L.layers) * 4))) return rc;
  if ((rc = P.row_start.ensure((size_t)(2 * L.n_tiles * L.layers + 1) * 4))) return rc;
  if ((rc = P.pairs.ensure(P.pairs_cap * 4))) return rc;
  if ((rc = P.items.ensure((size_t)P.items_cap * sizeof(WorkItem)))) return rc;
  {
    uint64_t sc = std::max<uint64_t>(2ull * ctx->n_cu + 64, P.split_min);
    sc = std::min<uint64_t>(sc, (uint64_t)std::max(L.n_tiles, 1));
    P.split_cap = (uint32_t)sc;
    if ((rc = P.split_tiles.ensure((size_t)P.split_cap * 4))) return rc;
    const size_t fx_bytes = (size_t)P.split_cap * merge_slot_u64() * 8;
    if (P.split_fx.bytes < fx_bytes) {
      // slots start zeroed; tile_merge leaves every slot it reads zeroed again
      if ((rc = P.split_fx.ensure(fx_bytes))) return rc;
      LG_HIP(launch_fill_u32(P.split_fx.as<uint32_t>(), P.split_fx.bytes / 4, 0u, st));
      LG_HIP(hipStreamSynchronize(st));
    }
  }
  if ((rc = P.stage_in.ensure(F.total))) return rc;
  if ((rc = P.stage_out.ensure(F.out_bytes()))) return rc;
  // ---- descriptors ----
  L.packed_only = accum;
  L.hues = false;
  char* in = P.stage_in.as<char>();
  SceneDesc* hd = reinterpret_cast<SceneDesc*>(in);
  uint32_t* h_tile_scene = reinterpret_cast<uint32_t*>(in + F.tile_scene);
  uint32_t* h_pre = reinterpret_cast<uint32_t*>(in + F.item_pre0);
  std::memset(in + F.counters, 0, F.total - F.counters);
  h_pre[0] = 0;
  uint64_t rays = 0;
  for (const Entry& e : E)
    if (trace && e.params.max_bounce) rays += e.scene->n_primary;
  const uint32_t rpi = trace_item_rays(rays, ctx->tune.rays_per_item, trace_groups(ctx, L.n), L.n);
  for (int i = 0; i < entries; i++) {
    const Entry& e = E[i];
    SceneDesc& D = hd[i];
    std::memset(&D, 0, sizeof(D));
    D.seg_count = gbl(reinterpret_cast<unsigned long long*>(P.counters.as<char>() + i * kCounterStride));
    D.gen_count = gbl(reinterpret_cast<uint32_t*>(P.counters.as<char>() + i * kCounterStride + kGenCountOffset));
    float max_abs = 0.0f;
    bool nonneg = true;
    SceneHues hues;
    if (trace) {
      lg_scene* sc = e.scene;
      D.recs = gbl(sc->table<void>(L.fp64 ? sc->at.recs64 : sc->at.recs32));
      D.recs64 = gbl(sc->table<Rec<double>>(sc->at.recs64));
      D.obj_n64 = gbl(sc->table<double>(sc->at.obj_n64));
      D.obj_flags = gbl(sc->table<uint32_t>(sc->at.obj_flags));
      D.obj_rec = gbl(sc->table<int32_t>(sc->at.obj_rec));
      D.obj_box = gbl(sc->table<float4>(sc->at.obj_box));
      D.medium = gbl(sc->table<MediumMasks>(sc->at.medium));
      std::memcpy(D.medium_map, sc->medium_map, sizeof(D.medium_map));
      D.verts = gbl(sc->table<void>(L.fp64 ? sc->at.verts64 : sc->at.verts32));
      D.verts64 = gbl(sc->table<double>(sc->at.verts64));
      D.lights = gbl(sc->table<DevLight>(sc->at.lights));
      D.blocks = gbl(sc->table<CullBlock>(sc->at.blocks));
      D.block_box = gbl(sc->table<float4>(sc->at.block_box));
      D.block_rec = gbl(sc->table<int32_t>(sc->at.block_rec));
      D.n_blocks = sc->n_blocks;
      D.by_boxes = scene_uses_boxes(ctx, sc, L.fp64) ? 1 : 0;
      D.tree_rec = gbl(sc->table<int32_t>(sc->at.tree_rec));
      D.n_trees = sc->n_trees;
      D.n_recs = sc->n_recs;
      D.n_objs = sc->n_objs;
      D.n_verts = sc->n_verts;
      D.n_lights = (int32_t)sc->lights.size();
      D.n_primary = sc->n_primary;
      // trace items of the first launch
      h_pre[i + 1] = h_pre[i] + (e.params.max_bounce ? (uint32_t)((sc->n_primary + rpi - 1) / rpi) : 0u);
      D.max_bounce = e.params.max_bounce;
      for (int c = 0; c < 4; c++) D.cutoff[c] = e.params.cutoff_color[c];
      for (int c = 0; c < 4; c++) D.canvas[c] = e.params.canvas[c];
      D.q0 = gbl(sc->q0.as<QRay<double>>());
      D.q1 = gbl(sc->q1.as<QRay<double>>());
      D.q_cap = sc->q_cap;
      max_abs = sc->light_max;
      nonneg = sc->light_nonneg;
      hues = scene_hues(sc);
    }
    if (e.segs) {
      D.seg_pos = gbl(e.segs->pos.as<float4>());
      D.seg_col = gbl(e.segs->col0.as<float4>());
      // a frame that traces writes one colour per segment (col0), whatever the buffer holds
      D.seg_col1 = gbl((!trace && !e.segs->one_color) ? e.segs->col1.as<const float4>() : nullptr);
      D.seg_key = gbl(e.segs->key.as<uint64_t>());
      D.seg_pos64 = gbl((trace && L.fp64) ? e.segs->pos64.as<double>() : nullptr);
      D.seg_cap = e.segs->cap;
      if (!trace) {
        D.flags |= SCENE_FIXED_COUNT;
        D.seg_fixed = e.segs->count;
        max_abs = e.segs->max_abs;
        nonneg = e.segs->nonneg;
        hues = e.segs->hues;
      }
    }
    if (e.img) {
      if (stages & ST_FRESH) D.flags |= SCENE_FRESH_IMAGE;
      D.view = make_view(e.img->view, L.tile);
      D.accum = gbl(e.img->accum.as<float4>());
      D.out16 = gbl(e.img->out16.as<ushort4>());
    }
    D.color_max = max_abs;
    D.blend_code = e.img ? e.img->blend_code : kBlendDefault;
    for (int c = 0; c < 4; c++) D.blend_k[c] = e.img ? e.img->blend.constant[c] : 0.0f;
    blend_factor_bounds(D.blend_code, max_abs, D.blend_k, D.factor_max);
    // two channels per LDS word when every deposit of the scene is non-negative
    if (ctx->packed_accum && nonneg && std::isfinite(max_abs) && blend_nonneg(D.blend_code, max_abs, D.blend_k)) {
      D.flags |= SCENE_PACKED;
      // one LDS word per deposit where the blend keeps the hue: RGB One, alpha SrcAlpha (the
      // default); not with 32-pixel tiles, whose kernels do not have that walk
      if (hues.n && D.blend_code == kBlendDefault && L.tile == 64) {
        set_hues(D, hues);
        L.hues = true;
      }
    } else if (accum) {
      L.packed_only = false;
    }
    D.tile_base = L.tile_base[i];
    D.row_base = (uint32_t)L.tile_base[i];
    D.row_stride = 1u;
    if (accum) {
      int t = D.view.tiles_x * D.view.tiles_y;
      for (int k = 0; k < t; k++) h_tile_scene[L.tile_base[i] + k] = (uint32_t)i;
    }
  }
  // colours per vertex go pair by pair under every blend but the default
  L.streams = accum && L.tile == 64 && L.packed_only && (L.runs || frame_block(ctx, L) == 1024);
  for (const Entry& e : E)
    if (accum && !trace && !e.segs->one_color && e.img->blend_code != kBlendDefault) L.streams = false;
  if (L.runs) {
    const SceneDesc whole = hd[0];
    for (int l = 0; l < n; l++) hd[l] = run_layer(whole, E[0].segs->runs, l, n);
  }
  if (trace) {
    BatchCtl* c = reinterpret_cast<BatchCtl*>(in + F.ctl);
    c->n_items_gen[0] = h_pre[n];
    c->item_rays[0] = rpi;
  }
  // ---- launch (graph replay when the shape is unchanged) ----
  std::vector<uint64_t> shape = {(uint64_t)n, stages, L.fp64, L.max_bounce, (uint64_t)L.cap_recs,
                                 (uint64_t)L.cap_objs, (uint64_t)L.cap_verts, (uint64_t)L.n_tiles,
                                 (uint64_t)L.max_tiles, L.n_counts, L.bin_target, P.pairs_cap, P.items_cap,
                                 P.split_cap, ctx->tune.rays_per_item, ctx->tune.min_piece, ctx->tune.max_piece,
                                 ctx->tune.trace_waves, ctx->tune.bvh_min_objects,
                                 (uint64_t)L.tile, (uint64_t)L.packed_only, (uint64_t)L.hues, (uint64_t)L.runs,
                                 (uint64_t)L.streams, L.chunk,
                                 ctx->tune.tile_block};
  for (DevBuf* b : {&P.frame_in, &P.item_pre, &P.chunk_pre, &P.cbase, &P.places, &P.scan_scratch, &P.row_start,
                    &P.pairs, &P.items, &P.split_tiles, &P.split_fx})
    shape.push_back((uint64_t)b->p);
  shape.push_back((uint64_t)P.stage_in.p);
  shape.push_back((uint64_t)P.stage_out.p);
  const bool use_graph = allow_graph && ctx->use_graphs && !profile;
  if (use_graph) {
    Pipeline::Graph* G = P.find(shape);
    if (!G) {
      P.make_room();
      LG_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
      rc = enqueue(ctx, P, st, profile, L, stages);
      hipGraph_t g = nullptr;
      hipError_t ce = hipStreamEndCapture(st, &g);
      if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
      }
      if (ce != hipSuccess) return hip_fail(ce, "hipStreamEndCapture");
      Pipeline::Graph ng;
      ng.shape = shape;
      ng.graph = g;
      hipError_t ie = hipGraphInstantiate(&ng.exec, g, nullptr, nullptr, 0);
      if (ie != hipSuccess) {
        (void)hipGraphDestroy(g);
        return hip_fail(ie, "hipGraphInstantiate");
      }
      P.graphs.push_back(ng);
      G = &P.graphs.back();
    }
    G->used = ++P.tick;
    LG_HIP(hipGraphLaunch(G->exec, st));
  } else {
    if ((rc = enqueue(ctx, P, st, profile, L, stages))) return rc;
  }
  return LG_OK;
}

// After the frame's stream has completed: grows whatever overflowed (*rerun = true: launch
// again) or publishes the segment counts.
static int batch_finish(lg_ctx* ctx, Pipeline& P, bool profile, Batch& B, bool* rerun) {
  const std::vector<Entry>& E = B.E;
  const uint32_t stages = B.stages;
  const Layout& L = B.L;
  const int n = L.n;
  const bool trace = stages & ST_TRACE, accum = stages & ST_ACCUM;
  // ---- overflow check ----
  const char* out = P.stage_out.as<const char>();
  const BatchCtl* hc = reinterpret_cast<const BatchCtl*>(out + n * kCounterStride);
  if (profile) {  // device-side work counts of this attempt's stages
    uint64_t segs_total = 0;
    for (int i = 0; trace && i < n; i++) segs_total += *reinterpret_cast<const uint64_t*>(out + i * kCounterStride);
    for (size_t k = B.first_stage; k < ctx->pending.size(); k++) {
      StageRec& r = ctx->pending[k];
      if (r.name.compare(0, 5, "trace") == 0) r.work = segs_total;
      if (r.name == "bin_count" || r.name == "bin_fill") r.work = hc->total_pairs;
      if (r.name == "tile_accum") {
        r.work = hc->samples;
        r.work2 = hc->lds_atomics;
      }
    }
  }
  bool over = false;
  for (int i = 0; trace && i < n; i++) {
    const Entry& e = E[i];
    const uint64_t segs = *reinterpret_cast<const uint64_t*>(out + i * kCounterStride);
    const uint32_t* gc = reinterpret_cast<const uint32_t*>(out + i * kCounterStride + kGenCountOffset);
    uint64_t qmax = 0;
    for (uint32_t g = 0; g < e.params.max_bounce; g++) qmax = std::max<uint64_t>(qmax, gc[g]);
    if (segs > e.segs->cap) {
      e.scene->seg_hint = std::max<uint64_t>(e.scene->seg_hint, segs + segs / 4 + 1024);
      over = true;
    }
    if (qmax > e.scene->q_cap) {
      e.scene->q_cap = std::min<uint64_t>(qmax + qmax / 4 + 1024, 0xffffffffull);
      if (qmax >= 0xffffffffull) return fail(LG_E_UNSUPPORTED, "ray queue exceeds 2^32 entries");
      over = true;
    }
  }
  if (accum) {
    if (hc->total_pairs > 0xffffffffull) return fail(LG_E_UNSUPPORTED, "more than 2^32 segment-tile pairs");
    if (hc->flags & CTL_PAIRS_OVERFLOW) {
      P.pairs_cap = hc->total_pairs + hc->total_pairs / 4 + 1024;
      over = true;
    }
    if (hc->flags & CTL_ITEMS_OVERFLOW) {
      P.items_cap *= 2;
      over = true;
    }
    if (hc->flags & CTL_SPLIT_OVERFLOW) {
      P.split_min = std::max<uint32_t>(hc->n_split + hc->n_split / 4 + 64, P.split_cap);
      over = true;
    }
  }
  *rerun = over;
  if (!over) {
    for (int i = 0; trace && i < n; i++) {
      const Entry& e = E[i];
      const uint64_t segs = *reinterpret_cast<const uint64_t*>(out + i * kCounterStride);
      e.segs->count = segs;
      e.segs->has_pos64 = L.fp64;
      e.segs->max_abs = e.scene->light_max;
      e.segs->nonneg = e.scene->light_nonneg;
      e.segs->hues = scene_hues(e.scene);
      e.segs->n_rays = e.scene->n_primary;
      e.scene->seg_hint = std::max(e.scene->seg_hint, segs);
    }
  }
  return LG_OK;
}

constexpr int kMaxAttempts = 8;

int pipeline_run(lg_ctx* ctx, const std::vector<Entry>& E, uint32_t stages) {
  if (!ctx->pipe) ctx->pipe.reset(new Pipeline());
  Pipeline& P = *ctx->pipe;
  if (E.empty()) return LG_OK;
  Batch B;
  B.E = E;
  B.stages = stages;
  int rc;
  if ((rc = batch_validate(ctx, ctx->stream, B))) return rc;
  for (int attempt = 0; attempt < kMaxAttempts; attempt++) {
    B.first_stage = ctx->pending.size();
    if ((rc = batch_launch(ctx, P, ctx->stream, ctx->profiling, true, B))) return rc;
    LG_HIP(hipStreamSynchronize(ctx->stream));
    bool rerun = false;
    if ((rc = batch_finish(ctx, P, ctx->profiling, B, &rerun))) return rc;
    if (!rerun) return LG_OK;
  }
  return fail(LG_E_CAPACITY, "batch: buffers kept overflowing");
}

// ---- asynchronous frames (the serving loop) ----------------------------------------------------
struct FrameJob {
  lg_ctx* ctx = nullptr;
  hipStream_t st = nullptr;
  hipEvent_t done = nullptr;
  Pipeline P;
  Batch B;
  int attempts = 0;
  bool busy = false;
};

FrameJob* frame_job_new(lg_ctx* ctx) {
  FrameJob* j = new FrameJob();
  j->ctx = ctx;
  if (hipStreamCreateWithFlags(&j->st, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreateWithFlags(&j->done, hipEventDisableTiming) != hipSuccess) {
    frame_job_free(j);
    return nullptr;
  }
  return j;
}

void frame_job_free(FrameJob* j) {
  if (!j) return;
  if (j->st) (void)hipStreamSynchronize(j->st);
  if (j->done) (void)hipEventDestroy(j->done);
  if (j->st) (void)hipStreamDestroy(j->st);
  delete j;
}

static int job_launch(FrameJob* j) {
  int rc;
  // eager: the batches of a serving mix rarely repeat a shape, so a capture would not pay
  if ((rc = batch_launch(j->ctx, j->P, j->st, false, false, j->B))) return rc;
  LG_HIP(hipEventRecord(j->done, j->st));
  j->attempts++;
  return LG_OK;
}

int frame_job_start(FrameJob* j, std::vector<Entry>&& E, uint32_t stages) {
  if (j->busy) return fail(LG_E_INVALID, "frame job already running");
  j->B = Batch();
  j->B.E = std::move(E);
  j->B.stages = stages;
  j->attempts = 0;
  int rc;
  if ((rc = batch_validate(j->ctx, j->st, j->B))) return rc;
  if ((rc = job_launch(j))) return rc;
  j->busy = true;
  return LG_OK;
}

int frame_job_poll(FrameJob* j, bool wait, bool* finished) {
  *finished = false;
  if (!j->busy) {
    *finished = true;
    return LG_OK;
  }
  hipError_t q = wait ? hipEventSynchronize(j->done) : hipEventQuery(j->done);
  if (q == hipErrorNotReady) return LG_OK;
  j->busy = false;
  if (q != hipSuccess) return hip_fail(q, "frame job");
  bool rerun = false;
  int rc;
  if ((rc = batch_finish(j->ctx, j->P, false, j->B, &rerun))) return rc;
  if (!rerun) {
    *finished = true;
    return LG_OK;
  }
  if (j->attempts >= kMaxAttempts) return fail(LG_E_CAPACITY, "batch: buffers kept overflowing");
  if ((rc = job_launch(j))) return rc;
  j->busy = true;
  return LG_OK;
}

const std::vector<Entry>& frame_job_entries(const FrameJob* j) { return j->B.E; }

size_t frame_job_scratch_bytes(const FrameJob* j) {
  const Pipeline& P = j->P;
  size_t b = 0;
  for (const DevBuf* d : {&P.frame_in, &P.item_pre, &P.chunk_pre, &P.cbase, &P.places, &P.scan_scratch, &P.row_start,
                          &P.pairs, &P.items, &P.split_tiles, &P.split_fx})
    b += d->bytes;
  return b;
}

}  // namespace lg
