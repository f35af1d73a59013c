// lg_internal.h — layouts shared by the host side (lg_api.hip) and the kernels
// (lg_trace.hip, lg_accum.hip). gfx950 only.
#pragma once
#include <cstring>

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <vector>

#include "../../include/lg.h"

namespace lg {

// ---- trace constants ------------------------------------------------------------------
// Hits with t <= kTMin along a ray are ignored: a child ray starts on the surface it left.
constexpr double kTMin = 1e-5;
// Spot lights with |spot_direction.x| below this point straight up or down (light.rs:230).
constexpr double kEpsilon = 1e-9;
// Path bits kept in a segment key (ray_index << kPathBits | path).
constexpr int kPathBits = 24;
constexpr uint32_t kMaxBounce = kPathBits - 1;

// ---- device scene records ------------------------------------------------------------
// One record per shape in object order; a Logic record is followed by its two operand
// records. Everything is in world coordinates.
enum RecKind : int32_t {
  REC_SEG = LG_SHAPE_LINE_SEGMENT,      // p: ax ay ex ey nx ny   (e = b - a, n = left unit normal)
  REC_BEZ = LG_SHAPE_CUBIC_BEZIER,      // p: a3 a2 a1 a0 (power basis, x/y pairs)
  REC_CIRCLE = LG_SHAPE_CIRCLE,         // p: cx cy r r^2
  REC_RECT = LG_SHAPE_RECT,             // p: cx cy ux uy vx vy hw hh
  REC_LOGIC = LG_SHAPE_LOGIC,           // op = lg_logic_op; aux = records of the subtree
  REC_POLY = LG_SHAPE_CONVEX_POLYGON,   // p: cx cy ux uy vx vy; aux = first vertex, op = count
  REC_ELLIPSE = LG_SHAPE_ELLIPSE,       // p: cx cy ux uy vx vy a b
  REC_TREE = 7                          // the root Logic record of a tree of more than two
                                        // primitives: as REC_LOGIC, p[0..4] list its leaves
};

template <typename T>
struct alignas(16) Rec {
  int32_t kind;
  int32_t obj;
  int32_t op;
  int32_t aux;
  T p[12];
};
static_assert(sizeof(Rec<float>) == 64, "Rec<float> is four float4");

// ---- containment (strict; open curves contain nothing), host and device -------------
template <typename T>
__host__ __device__ inline T abs_hd(T x) {
  return x < (T)0 ? -x : x;
}

template <typename T>
__host__ __device__ inline bool contains_prim(const Rec<T>& R, const T* verts, T px, T py) {
  switch (R.kind) {
    case REC_CIRCLE: {
      T x = px - R.p[0], y = py - R.p[1];
      return x * x + y * y < R.p[3];
    }
    case REC_RECT: {
      T lx = px - R.p[0], ly = py - R.p[1];
      T x = lx * R.p[2] + ly * R.p[3], y = lx * R.p[4] + ly * R.p[5];
      return abs_hd(x) < R.p[6] && abs_hd(y) < R.p[7];
    }
    case REC_ELLIPSE: {
      T lx = px - R.p[0], ly = py - R.p[1];
      T x = (lx * R.p[2] + ly * R.p[3]) / R.p[6], y = (lx * R.p[4] + ly * R.p[5]) / R.p[7];
      return x * x + y * y < (T)1;
    }
    case REC_POLY: {
      T lx = px - R.p[0], ly = py - R.p[1];
      T x = lx * R.p[2] + ly * R.p[3], y = lx * R.p[4] + ly * R.p[5];
      int first = R.aux, nv = R.op;
      if (nv < 3) return false;
      for (int i = 0; i < nv; i++) {
        int j = (i + 1 == nv) ? 0 : i + 1;
        T ax = verts[2 * (first + i)], ay = verts[2 * (first + i) + 1];
        T bx = verts[2 * (first + j)], by = verts[2 * (first + j) + 1];
        T cr = (bx - ax) * (y - ay) - (by - ay) * (x - ax);
        if (!(cr > (T)0)) return false;
      }
      return true;
    }
    default: return false;
  }
}

// A Logic tree is stored in prefix order: a Logic record (op; aux = records of its subtree,
// itself included), its operand a's subtree, then b's. A two-primitive object is REC_LOGIC
// with aux = 3; the root of a larger tree is REC_TREE and also lists its leaves: p[0..3] their
// record offsets from the root, p[4] their count (at most kLogicLeaves: an object's tree has
// at most LG_MAX_SHAPES = 7 nodes).
constexpr int kLogicLeaves = 4;

__host__ __device__ inline bool logic_combine(int op, bool a, bool b) {
  return op == LG_LOGIC_AND ? (a && b) : op == LG_LOGIC_OR ? (a || b) : (a && !b);
}

// Containment in a Logic tree of more than two primitives (records [first, first + aux)):
// the records in reverse prefix order, a primitive pushes its value, a Logic record pops its
// operands (a on top of b) and pushes their combination.
template <typename T>
__host__ __device__ inline bool contains_tree(const Rec<T>* recs, const T* verts, int first, T px, T py) {
  const Rec<T>& R = recs[first];
  uint32_t st = 0;
  int sp = 0;
  for (int k = first + R.aux - 1; k >= first; k--) {
    const Rec<T>& Q = recs[k];
    bool v;
    if (Q.kind == REC_LOGIC || Q.kind == REC_TREE) {
      const bool a = (st >> (sp - 1)) & 1u, b = (st >> (sp - 2)) & 1u;
      sp -= 2;
      v = logic_combine(Q.op, a, b);
    } else {
      v = contains_prim(Q, verts, px, py);
    }
    st = (st & ~(1u << sp)) | ((uint32_t)v << sp);
    sp++;
  }
  return st & 1u;
}

// Object::contains (object.rs:240-259) over the object's records starting at `first`.
template <typename T>
__host__ __device__ inline bool contains_object(const Rec<T>* recs, const T* verts, int first,
                                                T px, T py) {
  const Rec<T>& R = recs[first];
  if (R.kind == REC_LOGIC)
    return logic_combine(R.op, contains_prim(recs[first + 1], verts, px, py),
                         contains_prim(recs[first + 2], verts, px, py));
  if (R.kind == REC_TREE) return contains_tree(recs, verts, first, px, py);
  return contains_prim(R, verts, px, py);
}

// Per-object flags.
enum ObjFlags : uint32_t { OBJ_MATERIAL = 1u, OBJ_CLOSED = 2u };

// Bounding volumes over a scene's objects (Logic trees of more than two primitives aside): the
// objects in Morton order of their box centres, cut into blocks of up to kCullBlock. A block has
// the union of its objects' boxes and, per shape kind, the objects of that kind as bits. The
// boxes, kBoxGroup to a read (a block's are padded to that), are FP32 and padded so that every hit
// the FP32 culling pass can report lies inside its object's box.
constexpr int kCullBlock = 64;
constexpr int kBoxGroup = 4;
struct alignas(16) CullBlock {
  float box[4];         // centre x, y, half sizes x, y
  uint64_t kind[8];     // n_kinds masks, disjoint, together the block's objects
  int32_t first;        // of its boxes and first records
  int32_t n;
  int32_t n_kinds;
  uint32_t kinds;       // their RecKinds, 4 bits each
};
static_assert(sizeof(CullBlock) == 96, "six float4");

constexpr int kMaxRecords = 1024;      // records resident in LDS per trace workgroup
constexpr int kMaxObjects = 1024;
constexpr int kMaxPolyVertices = 1024; // vertices of all polygons in a scene
constexpr int kMaxLights = 64;
// Segments in one buffer: the accumulation's pair entries hold a segment index in 31 bits.
constexpr uint64_t kMaxSegments = (1ull << 31) - 1;

// ---- lights --------------------------------------------------------------------------
struct DevLight {
  int32_t kind;
  int32_t _pad;
  uint64_t num_rays;
  uint64_t ray_base;    // global index of the light's first ray
  float color[4];
  double a[2];          // point/spot position; directional band start
  double e[2];          // directional: b - a
  double nrm[2];        // directional: unit normal
  double min_angle;     // spot
  double spot_angle;    // spot
  double sign;          // spot: f64::signum(spot_direction.x)
  double ior;           // starting refractive index (tracer.rs:280-287)
};

// ---- rays in flight -------------------------------------------------------------------
template <typename T>
struct alignas(16) QRay {
  T o[2];
  T d[2];
  float c[4];
  T ior;
  uint64_t key;
};

// ---- batched pipeline: one descriptor per scene ------------------------------------------
struct AccumView {
  double left, top;
  double sx, sy;              // pixels per world unit
  int32_t width, height;
  int32_t tiles_x, tiles_y;
  int32_t tile;               // screen tile edge in pixels (32 or 64), the same for a whole frame
  int32_t tile_shift;         // log2(tile)
};

enum SceneFlags : uint32_t {
  SCENE_FIXED_COUNT = 1u,     // accumulate `seg_fixed` uploaded segments (no trace)
  SCENE_FRESH_IMAGE = 2u,     // the frame clears, accumulates and resolves the image: the tile
                              // flushes write the accumulator and the RGBA16F target directly
  SCENE_PACKED = 4u,          // every deposit is non-negative: two channels per LDS word
  SCENE_HUES = 8u,            // with SCENE_PACKED: the segments' colours are fractions of at most
                              // kMaxHues light colours (SceneHues): one LDS word per deposit
  SCENE_RUNS = 16u            // with SCENE_PACKED: runs of segments of one colour (SegRuns): the
                              // tiles sum one weight per run. The frame's only scene, cut into
                              // layers of up to kRunPlanes runs with a descriptor each
};

// Segments in runs of one colour (StringMods without modulo colours, or uploads): run r holds the segments from
// first[r] (first[0] = 0) up to the next run's, all of colour color[r].
constexpr int kRunPlanes = 6;   // runs whose weight planes fit a tile kernel's LDS
constexpr int kMaxLayers = 4;
constexpr int kMaxRuns = kRunPlanes * kMaxLayers;
struct SegRuns {
  int32_t n = 0;                // 0: the segments are not known to be of this form
  uint32_t first[kMaxRuns] = {};
  float color[kMaxRuns][4] = {};
  // A segment of the given colour at index i follows; false: too many runs (n = 0 from then on).
  bool add(uint64_t i, const float* c) {
    if (n && std::memcmp(color[n - 1], c, sizeof(color[0])) == 0) return true;
    if (n == kMaxRuns || i > 0xffffffffull) {
      n = 0;
      return false;
    }
    first[n] = (uint32_t)i;
    std::memcpy(color[n++], c, sizeof(color[0]));
    return true;
  }
};

// The colours of traced segments. A ray's RGB is its light's, scaled by one factor per surface it
// met, and its alpha is its light's (tracer.rs:454-457): a segment's colour is one number times
// its light's hue, and its light follows from the ray index in its key. Hue h covers the rays
// from first_ray[h] (first_ray[0] = 0) up to the next hue's.
constexpr int kMaxHues = 3;
struct SceneHues {
  int32_t n = 0;               // 0: the colours are not known to be of this form
  uint64_t first_ray[kMaxHues] = {0, 0, 0};
  float color[kMaxHues][4] = {};
};

// Device pointers kept in descriptors carry the global address space in their type: kernels
// read them from memory rather than from their arguments, and a plain (generic) pointer
// loaded from memory makes the compiler emit flat accesses, which tie up more registers and
// wait on the LDS counter too. gen() turns one back into a plain pointer whose global origin
// the compiler still sees.
#define LG_G __attribute__((address_space(1)))
template <typename T>
__host__ __device__ __forceinline__ LG_G T* gbl(T* p) {
  return (LG_G T*)p;
}
template <typename T>
__host__ __device__ __forceinline__ T* gen(LG_G T* p) {
  return (T*)p;
}

// Which of 64 objects (with a material and an inside; others have no bit) have a padded box over a
// bucket of x, and of y: a point lies in none but those of both its buckets.
constexpr int kMediumBuckets = 64;
struct MediumMasks {
  uint64_t x[kMediumBuckets], y[kMediumBuckets];
};
// Monotone in v, so a point between a box's ends has a bucket between theirs.
__host__ __device__ inline int medium_bucket(float v, float scale, float offset) {
  const float b = __builtin_fmaf(v, scale, offset);
  const float c = __builtin_fminf(__builtin_fmaxf(b, 0.0f), (float)(kMediumBuckets - 1));
  return (int)c;
}

struct SceneDesc {
  // geometry (device buffers of the lg_scene)
  const LG_G void* recs;           // culling records, Rec<float> or Rec<double>
  const LG_G Rec<double>* recs64;  // FP64 records: re-evaluation of winners and shading
  const LG_G double* obj_n64;
  const LG_G uint32_t* obj_flags;
  const LG_G int32_t* obj_rec;
  const LG_G float4* obj_box;      // per object: padded world box {lo.x, lo.y, hi.x, hi.y}
  const LG_G MediumMasks* medium;  // per 64 objects
  float medium_map[4];             // bucket of x: x * [0] + [1]; of y: y * [2] + [3] (medium_bucket)
  const LG_G void* verts;          // polygon vertices in the culling precision
  const LG_G double* verts64;
  const LG_G DevLight* lights;
  const LG_G CullBlock* blocks;    // culling by boxes (every object's; see by_boxes)
  const LG_G float4* block_box;    // the blocks' objects: padded boxes (centre and half sizes),
  const LG_G int32_t* block_rec;   // and first records
  const LG_G int32_t* tree_rec;    // first record of each object that is a Logic tree of more
                                   // than two primitives (the object walk skips these)
  int32_t n_blocks;
  int32_t by_boxes;                // 0: the culling pass walks every record
  int32_t n_trees;
  int32_t n_recs, n_objs, n_verts, n_lights;
  uint64_t n_primary;
  uint32_t max_bounce;
  uint32_t flags;             // SceneFlags
  float cutoff[4];
  double canvas[4];           // left right bottom top
  // ray queues (lg_scene)
  LG_G QRay<double>* q0;
  LG_G QRay<double>* q1;
  uint64_t q_cap;
  // segments (lg_segments)
  LG_G float4* seg_pos;
  LG_G float4* seg_col;
  const LG_G float4* seg_col1;
  LG_G uint64_t* seg_key;
  LG_G double* seg_pos64;
  uint64_t seg_cap;
  uint64_t seg_fixed;         // SCENE_FIXED_COUNT: number of segments present
  // per-scene counters (pipeline scratch): segments, then children per generation
  LG_G unsigned long long* seg_count;
  LG_G uint32_t* gen_count;
  // accumulation (lg_image)
  AccumView view;
  LG_G float4* accum;
  LG_G ushort4* out16;
  int32_t tile_base;          // first global tile of this scene
  float color_max;            // bound on |colour channel| of the scene's segments
  // blend of the image (lg_image_set_blend): per channel (r, g, b, a) 4 bits at 4 * channel,
  // a BlendCode factor in the low 3 bits and bit 3 set for ReverseSubtract; the constant;
  // per channel, the largest |factor| over |colour| <= color_max
  uint32_t blend_code;
  float blend_k[4];
  float factor_max[4];
  // SCENE_HUES: per hue the light's brightest RGB channel, the bound of what a segment of it
  // deposits there and its alpha (whose square a segment deposits), and the RGB channels over the
  // brightest
  int32_t n_hues;
  int32_t hue_ch[kMaxHues];
  uint64_t hue_ray[kMaxHues];
  float hue_bound[kMaxHues][2];
  double hue_ratio[kMaxHues][3];
  // Tile t's pair rows (y-major, x-major) are rows 2 (row_base + row_stride t) and the next.
  // row_stride is 1 but for the layers of a SCENE_RUNS frame, whose rows of a tile follow each other.
  uint32_t row_base, row_stride;
  // SCENE_RUNS: this layer's runs, by first segment in the layer, and their colours
  int32_t n_runs;
  uint32_t run_first[kRunPlanes];
  float run_color[kRunPlanes][4];
};

// Source factors of the supported blends, per channel c of the interpolated colour (a = its
// alpha, k = the blend constant): each sample adds +-w * c * factor.
enum BlendCode : uint32_t {
  BC_ZERO = 0, BC_ONE = 1, BC_SRC = 2, BC_ONE_MINUS_SRC = 3, BC_SRC_ALPHA = 4, BC_ONE_MINUS_SRC_ALPHA = 5,
  BC_CONST = 6, BC_ONE_MINUS_CONST = 7, BC_NEGATE = 8
};
// rgb: One; alpha: SrcAlpha (mod.rs:57-73)
constexpr uint32_t kBlendDefault = BC_ONE | (BC_ONE << 4) | (BC_ONE << 8) | (BC_SRC_ALPHA << 12);

constexpr int kMaxGen = kPathBits;

// Rays of a trace item when a launch of n_scenes has `total`: a workgroup's share of them, at
// least 64 and at most the tuning's (`rpi`). A workgroup waits for its slowest wave at every
// append, and a launch for its slowest workgroup, so few rays are done sooner by workgroups of one
// wave. (us of trace launches, items of 256 rays and so: 20000 rays, 4 objects 94 and 86; 12000
// rays, 3 objects 97 and 79; 75011 rays, 23 objects 213 and 214. Sharing the rays of an item out
// over its four waves gave no more: every further wave fetches the kernel's code through its own
// compute unit's cache.) Between two items lies a chain of trips to memory (the cursor, the item's
// scene, its tables), so many rays are done sooner in one item to a workgroup than in several (1M
// rays, 64 objects: items of 256 576 us, 512 484, 1024 469), unless they are of several scenes:
// their shares are halves, as the launch has twice the workgroups (trace_groups), and halved
// again down to 512 rays where they are larger, since the items' costs differ (1.4M rays in 20
// scenes, items of 256 714 us, 512 621, whole shares 748, so 527).
__host__ __device__ inline uint32_t trace_item_rays(uint64_t total, uint32_t rpi, uint32_t groups, int n_scenes) {
  const uint64_t waves = (total + 64ull * groups - 1) / (64ull * groups);  // per share
  uint64_t m = waves > 1 ? 64 * waves : 64;
  if (n_scenes > 1 && m > 512) m = m > 1024 ? (waves + 1) / 2 * 64 : 512;
  return m < rpi ? (uint32_t)m : rpi;
}

// Device-side control block of one batched frame. Atomic adds to one line of memory are served one
// after another, 12 ns each over the whole chip, so the words that persistent workgroups count on
// have lines of their own: a workgroup waits for its claim, and behind other words' adds it waits
// for those too.
struct BatchCtl {
  uint32_t n_items_gen[kMaxGen];   // trace items per generation
  uint32_t item_rays[kMaxGen];     // rays of an item, per generation
  uint32_t n_chunks;
  uint32_t chunk;                  // segments per bin chunk (at least; see scene_chunk)
  uint32_t bin_groups;             // bin workgroups of the frame
  uint32_t spread;                 // segments per bin workgroup of the frame (see scene_chunk)
  unsigned long long total_pairs;
  uint32_t n_work;
  uint32_t flags;                  // CTL_* overflow bits
  uint32_t n_split;                // tiles split over several work items
  uint32_t pad0;
  // profiled frames only: anti-aliased samples walked by tile_accum (2 pixels x 4 channels each),
  // and the 64-bit LDS atomic wave instructions its walk issued
  unsigned long long samples;
  unsigned long long lds_atomics;
  // tile work items ordered by size class (floor(log2(pairs))), largest class first: items per
  // class, and the slots each class has handed out (frames above kPlanTiles tiles)
  uint32_t class_count[32];
  uint32_t class_cursor[32];
  alignas(128) uint32_t item_cursor[kMaxGen];
  alignas(128) uint32_t gen_done[kMaxGen];  // trace workgroups finished per generation
  alignas(128) uint32_t chunk_cursor0;  // bin_count
  alignas(128) uint32_t chunk_cursor1;  // bin_fill
  alignas(128) uint32_t work_cursor;    // tile_accum
  uint32_t pad[31];
};
static_assert(sizeof(BatchCtl) % 128 == 0, "the cursors' lines end with the block");

enum CtlFlags : uint32_t { CTL_PAIRS_OVERFLOW = 1u, CTL_ITEMS_OVERFLOW = 2u, CTL_SPLIT_OVERFLOW = 4u };
// Any of these makes the frame's tile stage a no-op; the host grows the buffer and reruns.
constexpr uint32_t kCtlStop = CTL_PAIRS_OVERFLOW | CTL_ITEMS_OVERFLOW | CTL_SPLIT_OVERFLOW;

// Everything the tile kernel needs of its tile besides the scene, so that an item costs one
// 32-byte load (prefetched while the previous item runs).
struct alignas(16) WorkItem {
  uint32_t scene;             // bit 31: the tile is split over several items (merge buffer)
  uint32_t tile;              // tile index inside the scene
  uint32_t begin, end;        // range in the pair list
  uint32_t mid;               // the tile's first x-major pair (its y-major pairs come first)
  uint32_t tile_pairs;        // the tile's pair count, at most kPackedPiece (packed fixed point)
  uint32_t slot;              // merge slot of a split tile
  uint32_t pad;
};
constexpr uint32_t kSplitBit = 0x80000000u;
// One merge slot of a tile split over several work items: 4 channel planes of the largest
// tile (64 x 64), or two per hue, 64-bit fixed point.
constexpr int kMergeSlotU64 = 2 * kMaxHues * 64 * 64;
// Pairs per tile work item at most: the fixed point of a tile that accumulates two channels
// per LDS word follows min(pairs of the tile, kPackedPiece), whatever the launch tuning, so
// results do not depend on it.
constexpr uint32_t kPackedPiece = 32768u;

// Work distribution of the persistent kernels: workgroup b first takes item b; workgroups
// that finish it take further items from `cursor`, which counts up from gridDim.x. A plain
// (coherent) read of the cursor lets workgroups leave without touching the atomic once the
// items are gone, so a launch that has fewer items than workgroups costs no atomics at all
// beyond one per worked item.
__device__ __forceinline__ uint32_t next_work_item(uint32_t* cursor, uint32_t n_items, bool first) {
  if (first) return blockIdx.x;
  if (__hip_atomic_load(cursor, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + gridDim.x >= n_items)
    return n_items;
  return atomicAdd(cursor, 1u) + gridDim.x;
}

// ---- error helpers (host) -------------------------------------------------------------
void set_error(const std::string& msg);
int hip_fail(hipError_t e, const char* what);

}  // namespace lg

#define LG_HIP(call)                                   \
  do {                                                 \
    hipError_t _e = (call);                            \
    if (_e != hipSuccess) return lg::hip_fail(_e, #call); \
  } while (0)
