/*
 * lg.h — C ABI of the MI355X light_garden path: per-ray 2-D trace and additive line
 * accumulation into an RGBA16F image.
 *
 * The reference is in-process Rust (sphereflow/light_garden) with no FFI. Its seam is
 * the `Tracer` scene API (src/light_garden/tracer.rs:4-17, 48-116) and
 * `Tracer::trace_all() -> Vec<(P2, Color)>` (tracer.rs:276), whose output is drawn by
 * `SubRenderPass::update_vertex_buffer` + a LineList draw with additive blend into an
 * Rgba16Float texture (src/sub_render_pass.rs:188-212, src/light_garden/mod.rs:57-73,
 * src/texture_renderer.rs:5). Every entry point below names the reference item it
 * replaces. The structs are plain data with fixed-width fields and explicit padding,
 * so a Rust `#[repr(C)]` mirror binds them one to one.
 *
 * Conventions
 *   - Every call returns an int status (LG_OK == 0). lg_last_error() gives a message for
 *     the last failing call on the calling thread.
 *   - Host arrays passed in are copied during the call; the caller keeps ownership.
 *   - Device buffers behind lg_segments / lg_image belong to the library until the
 *     matching *_destroy.
 *   - One host thread per lg_ctx at a time. Each context owns one HIP stream; separate
 *     contexts are independent. A scene must not be edited while a trace of it runs
 *     (the reference's `&self` trace / `&mut self` edit split, tracer.rs:360).
 */
#ifndef LG_H
#define LG_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define LG_ABI_VERSION 1

/* ---- status codes -------------------------------------------------------------- */
enum lg_status {
  LG_OK = 0,
  LG_E_INVALID = 1,     /* malformed argument or scene                              */
  LG_E_OOM = 2,         /* device allocation failed or memory budget exceeded        */
  LG_E_CAPACITY = 3,    /* caller's output array too small; *needed says how large   */
  LG_E_HIP = 4,         /* HIP runtime error                                         */
  LG_E_UNSUPPORTED = 5, /* valid in the reference but not handled by this build      */
  LG_E_NODEVICE = 6,    /* no usable gfx950 device                                   */
  LG_E_TIMEOUT = 7,     /* serving: request deadline passed                          */
  LG_E_NOTFOUND = 8     /* serving: unknown request or scene id                       */
};

/* ---- geometry (collision2d::Geo variants reachable from ObjectE, object.rs:6-16) -- */
enum lg_shape_kind {
  LG_SHAPE_LINE_SEGMENT = 0,   /* Geo::GeoLineSegment — StraightMirror (object.rs:315)  */
  LG_SHAPE_CUBIC_BEZIER = 1,   /* Geo::GeoCubicBezier — CurvedMirror (object.rs:345)    */
  LG_SHAPE_CIRCLE = 2,         /* Geo::GeoCircle (object.rs:287)                        */
  LG_SHAPE_RECT = 3,           /* Geo::GeoRect, rotated (object.rs:288)                 */
  LG_SHAPE_LOGIC = 4,          /* Geo::GeoLogic — Lens and boolean ops (object.rs:387)  */
  LG_SHAPE_CONVEX_POLYGON = 5, /* Geo::GeoConvexPolygon (object.rs:290)                 */
  LG_SHAPE_ELLIPSE = 6         /* Geo::GeoEllipse (object.rs:291)                       */
};

enum lg_logic_op { LG_LOGIC_AND = 0, LG_LOGIC_OR = 1, LG_LOGIC_AND_NOT = 2 };

#define LG_MAX_SHAPES 7          /* nodes of one object's Logic tree (<= 4 leaves)    */
#define LG_MAX_POLY_VERTICES 16  /* vertices of all polygons of one object            */

/*
 * One node of an object's shape tree. Node 0 is the root. A node's frame is
 * world = parent_frame(origin + R * local), R column-major [m00, m10, m01, m11]
 * (the RON `rotation: [..4]` layout, default.ron:24-29).
 *   LINE_SEGMENT   p = {ax, ay, bx, by}                         (origin/rotation unused)
 *   CUBIC_BEZIER   p = {p0x, p0y, p1x, p1y, p2x, p2y, p3x, p3y} (origin/rotation unused)
 *   CIRCLE         origin = centre, p[0] = radius
 *   RECT           origin = centre, rotation, p[0] = width, p[1] = height
 *   ELLIPSE        origin = centre, rotation, p[0] = a (local x semi-axis), p[1] = b
 *   CONVEX_POLYGON origin, rotation; vertices (local, counter-clockwise) at
 *                  lg_object.vertices[2*vertex_offset ..], n_vertices of them
 *   LOGIC          origin, rotation = local frame of the two operands; op,
 *                  child_a / child_b = node indices (> this node's index); an operand
 *                  is a closed primitive (circle, rect, ellipse, polygon) or LOGIC
 */
typedef struct lg_shape {
  int32_t kind;
  int32_t op;
  int32_t child_a;
  int32_t child_b;
  int32_t n_vertices;
  int32_t vertex_offset;
  double origin[2];
  double rotation[4];
  double p[8];
} lg_shape;

/* Object {object_enum, material_opt: Option<Material>, moved} (object.rs:50-55). */
typedef struct lg_object {
  int32_t has_material;      /* material_opt.is_some(); without it the object mirrors */
  int32_t n_shapes;          /* nodes used in shapes[]                                 */
  double refractive_index;   /* Material::refractive_index (default 1.2, object.rs:444) */
  lg_shape shapes[LG_MAX_SHAPES];
  double vertices[2 * LG_MAX_POLY_VERTICES];
} lg_object;

/* ---- lights (light.rs:9-14) -------------------------------------------------------- */
enum lg_light_kind {
  LG_LIGHT_POINT = 0,        /* PointLight{position, color, num_rays}  light.rs:139       */
  LG_LIGHT_DIRECTIONAL = 1,  /* DirectionalLight{color, num_rays, start} light.rs:79      */
  LG_LIGHT_SPOT = 2          /* SpotLight{position, color, num_rays, spot_angle, dir} 190 */
};

typedef struct lg_light {
  int32_t kind;
  int32_t _pad0;
  uint64_t num_rays;
  float color[4];            /* Color = [f32; 4] (light.rs:7), RGB plus alpha            */
  double position[2];        /* point/spot: position; directional: band start a          */
  double direction[2];       /* spot: spot_direction; directional: band end b            */
  double spot_angle;         /* spot: full cone angle in radians                          */
} lg_light;

/* ---- trace parameters (Tracer fields, tracer.rs:9-13, 37-39) ------------------------ */
enum lg_trace_flags {
  LG_TRACE_FP64 = 1u << 0    /* trace in FP64 end to end instead of FP32 + FP64 islands */
};

typedef struct lg_params {
  uint32_t max_bounce;       /* generations traced (default 5)                          */
  uint32_t flags;            /* lg_trace_flags                                           */
  float cutoff_color[4];     /* default {0.001, 0.001, 0.001, 0.001}                     */
  double canvas[4];          /* canvas_bounds as {left, right, bottom, top}               */
} lg_params;

/* Image view: world rect projected onto width x height pixels, row 0 at the top
 * (ortho(-a, a, -1, 1) of renderer.rs:120-124 generalised to any rect). */
typedef struct lg_view {
  double left, right, bottom, top;
  uint32_t width, height;
} lg_view;

/* ---- opaque handles ------------------------------------------------------------------ */
typedef struct lg_ctx lg_ctx;
typedef struct lg_scene lg_scene;
typedef struct lg_segments lg_segments;
typedef struct lg_image lg_image;

/* ---- context ------------------------------------------------------------------------- */
const char* lg_last_error(void);
int lg_version(void);
/* Opens `device` (HIP ordinal), creates the context's stream and scratch arenas. */
int lg_ctx_create(int device, lg_ctx** out);
/* Releases the context; while scenes, segment buffers or images made from it are alive the
 * release waits for the last of them to be destroyed. */
int lg_ctx_destroy(lg_ctx* ctx);
int lg_ctx_synchronize(lg_ctx* ctx);
/* Per-stage HIP-event timing of the context's next calls (off by default). */
int lg_ctx_set_profiling(lg_ctx* ctx, int enable);
typedef struct lg_stage_time {
  char name[24];
  float ms;                  /* sum over the stage's launches in the last profiled call */
  uint32_t launches;
  uint64_t work;             /* stage-specific unit count (segments, pairs, pixels)     */
  uint64_t work2;            /* a second count where a stage has one: tile_accum's 64-bit
                                LDS atomic wave instructions (work: its samples)       */
} lg_stage_time;
int lg_ctx_stage_times(lg_ctx* ctx, lg_stage_time* out, int cap, int* n_out);
/* Measures the device's issue rate of 64-bit LDS atomic adds in wave instructions per second
 * (workgroups shaped like the tile accumulation's, conflict-free addresses; best of 3 runs of
 * about a millisecond each). No counterpart in the reference: it is the roof that the tile
 * walk's atomic count (lg_stage_time.work2 of "tile_accum") is measured against. */
int lg_calibrate_lds_atomics(lg_ctx* ctx, double* wave_instructions_per_s);

/* ---- scene: the Tracer's object/light container (tracer.rs:4-17, 48-116) ------------- */
int lg_scene_create(lg_ctx* ctx, lg_scene** out);
int lg_scene_destroy(lg_scene* scene);
/* Tracer::clear (tracer.rs:54) / clear_objects (tracer.rs:48). */
int lg_scene_clear(lg_scene* scene);
int lg_scene_clear_objects(lg_scene* scene);
/* Tracer::push_object (tracer.rs:87) / push_light (tracer.rs:92). */
int lg_scene_push_object(lg_scene* scene, const lg_object* obj);
int lg_scene_push_light(lg_scene* scene, const lg_light* light);
/* Bulk forms of push_*: replace all objects / all lights (Tracer::load, tracer.rs:190). */
int lg_scene_set_objects(lg_scene* scene, const lg_object* objs, uint32_t n);
int lg_scene_set_lights(lg_scene* scene, const lg_light* lights, uint32_t n);
/* Tracer::replace_object (tracer.rs:104), remove_object (109), remove_light (114). */
int lg_scene_replace_object(lg_scene* scene, uint32_t ix, const lg_object* obj);
int lg_scene_remove_object(lg_scene* scene, uint32_t ix);
int lg_scene_remove_light(lg_scene* scene, uint32_t ix);
int lg_scene_counts(const lg_scene* scene, uint32_t* n_objects, uint32_t* n_lights,
                    uint64_t* n_rays);

/* ---- RON scene files: `(Vec<Object>, Vec<Light>)` as ron reads and writes it ----------
 * Host only; no device work. The text is the reference's save format (default.ron; objects
 * by object_enum variant, material_opt, moved; lights by variant). LineSegment is written
 * `(a: [x, y], b: [x, y])` and ConvexPolygon `(points: [[x, y], ...])`, which the reference's
 * files do not show. Errors: LG_E_INVALID for malformed text (the reference panics,
 * tracer.rs:191-192), LG_E_CAPACITY with the needed count/length returned. */
/* Tracer::load (tracer.rs:190-204): replaces all objects and lights; the scene is unchanged
 * when the text does not parse. Light rays are regenerated from num_rays at trace time. */
int lg_scene_load_ron(lg_scene* scene, const char* text, uint64_t len);
/* Tracer::serialize (tracer.rs:183-188): ron::ser::to_string_pretty with PrettyConfig::default
 * (4-space indent, trailing commas, floats in Rust's shortest Display form). `buf` gets the
 * text and a NUL; *len is the text length without it. */
int lg_scene_save_ron(const lg_scene* scene, char* buf, uint64_t cap, uint64_t* len);
/* Context-free forms of the two above (LightGarden::load_from_file / save_to_file read and
 * write the same text, mod.rs:698-725). Shape trees are decoded as lg_object nodes: Lens,
 * Geo(GeoLogic) -> LOGIC root with children; a LOGIC root of two equal circles at (+-d, 0)
 * under And is written back as Lens, other LOGIC roots as Geo(GeoLogic(...)). */
int lg_ron_parse_scene(const char* text, uint64_t len, lg_object* objects, uint32_t cap_objects,
                       uint32_t* n_objects, lg_light* lights, uint32_t cap_lights,
                       uint32_t* n_lights);
int lg_ron_write_scene(const lg_object* objects, uint32_t n_objects, const lg_light* lights,
                       uint32_t n_lights, char* buf, uint64_t cap, uint64_t* len);

/* ---- segments: the `Vec<(P2, Color)>` vertex pairs of trace_all (tracer.rs:451-486) --- */
/* Device SoA: pos float4 {x0,y0,x1,y1}; color0 float4; optional color1 float4 (per-vertex
 * colours, string_mod.rs:118-119); key uint64 (ray index << 24 | path bits). */
enum lg_segment_flags { LG_SEG_VERTEX_COLORS = 1u << 0 };
/* A buffer holds at most 2^31 - 1 segments: LG_E_OOM for a larger capacity, and for a trace,
 * upload or string mod that would need more. */
int lg_segments_create(lg_ctx* ctx, uint64_t capacity, uint32_t flags, lg_segments** out);
int lg_segments_destroy(lg_segments* segs);
int lg_segments_count(const lg_segments* segs, uint64_t* count);
/* Host -> device (replaces update_vertex_buffer's upload, sub_render_pass.rs:188-203).
 * color1 may be NULL unless the buffer was created with LG_SEG_VERTEX_COLORS. A buffer whose
 * segments have one colour for both ends (color1 NULL or equal to color0 bit for bit, traced
 * segments, StringMods without modulo colours) keeps color0 only: its download returns color0
 * as color1, and its accumulation takes the one-colour walk (the same image bits). */
int lg_segments_upload(lg_segments* segs, const float* pos, const float* color0,
                       const float* color1, uint64_t n);
/* Device -> host; any output pointer may be NULL. Fails with LG_E_CAPACITY if cap < count. */
int lg_segments_download(lg_segments* segs, float* pos, float* color0, float* color1,
                         uint64_t* key, uint64_t cap, uint64_t* count);

/* FP64 end points {x0,y0,x1,y1} of the last LG_TRACE_FP64 trace into `out` (the
 * reference's P2 = Point2<f64> vertices, tracer.rs:451-452). */
int lg_segments_download_pos64(lg_segments* segs, double* pos64, uint64_t cap, uint64_t* count);

/* The buffer's vertex pairs in ascending key order, which for traced segments is trace_all's
 * order: xy gets 2 doubles and rgba 4 floats per vertex, 2 vertices per segment (FP64 end points
 * of an LG_TRACE_FP64 trace, else the stored FP32 ones). LG_E_CAPACITY with *n_vertices set to the
 * needed count when cap_vertices is too small. The call's device scratch, 40 to 56 bytes per segment
 * and 8 per ray, stays with the context up to 64 MiB, and some 12 MB of pinned host memory; without
 * room for it the host orders the buffer. */
int lg_segments_download_vertices(lg_segments* segs, double* xy, float* rgba, uint64_t cap_vertices,
                                  uint64_t* n_vertices);

/* ---- trace: Tracer::trace_all / Tracer::trace (tracer.rs:276-358, 360-493) ------------ */
/* Traces every light of the scene into `out` (device). Segment order in the buffer is
 * unspecified; the key gives each segment's identity and the reference's emission order. */
int lg_trace(lg_scene* scene, const lg_params* params, lg_segments* out);
/* Drop-in for trace_all's return value: vertex pairs in the reference's order
 * (light, ray, depth, parent, reflected before refracted). xy gets 2 doubles and rgba 4
 * floats per vertex, 2 vertices per segment. Fails with LG_E_CAPACITY and *n_vertices set
 * to the needed count when cap_vertices is too small. */
int lg_trace_all(lg_scene* scene, const lg_params* params, double* xy, float* rgba,
                 uint64_t cap_vertices, uint64_t* n_vertices);

/* ---- image: the Rgba16Float render target (texture_renderer.rs:5, 69-80) --------------- */
int lg_image_create(lg_ctx* ctx, const lg_view* view, lg_image** out);
int lg_image_destroy(lg_image* img);
/* Clears the FP32 accumulator to zero (the resolve adds the target's clear alpha of 1,
 * renderer.rs:175). */
int lg_image_clear(lg_image* img);
/* Device pointers for zero-copy interop: accum is float4 per pixel (row-major), rgba16f is
 * 4 half per pixel. */
int lg_image_device_ptrs(lg_image* img, void** accum, void** rgba16f);
int lg_image_download_rgba16f(lg_image* img, uint16_t* host, uint64_t cap_halves);
int lg_image_download_accum(lg_image* img, float* host, uint64_t cap_floats);

/* ---- blend state of an image: the lines pipeline's BlendState (mod.rs:57-73), selectable
 * in the reference's settings window (gui/settings.rs:57-133). Values follow wgpu's enums in
 * the order that window lists them. */
enum lg_blend_factor {
  LG_BF_ZERO = 0, LG_BF_ONE = 1, LG_BF_SRC = 2, LG_BF_ONE_MINUS_SRC = 3, LG_BF_SRC_ALPHA = 4,
  LG_BF_ONE_MINUS_SRC_ALPHA = 5, LG_BF_DST = 6, LG_BF_ONE_MINUS_DST = 7, LG_BF_DST_ALPHA = 8,
  LG_BF_ONE_MINUS_DST_ALPHA = 9, LG_BF_SRC_ALPHA_SATURATED = 10, LG_BF_CONSTANT = 11,
  LG_BF_ONE_MINUS_CONSTANT = 12
};
enum lg_blend_op { LG_BO_MIN = 0, LG_BO_MAX = 1, LG_BO_ADD = 2, LG_BO_SUBTRACT = 3, LG_BO_REVERSE_SUBTRACT = 4 };
typedef struct lg_blend_component {   /* wgpu::BlendComponent */
  uint32_t src_factor;                /* lg_blend_factor */
  uint32_t dst_factor;
  uint32_t operation;                 /* lg_blend_op */
} lg_blend_component;
typedef struct lg_blend {             /* wgpu::BlendState + the blend constant */
  lg_blend_component color;           /* default: One, One, Add        (mod.rs:66-70) */
  lg_blend_component alpha;           /* default: SrcAlpha, One, Add   (mod.rs:61-65) */
  float constant[4];                  /* default 0 (never set by the reference) */
} lg_blend;
/* Sets the blend of every later accumulation into img. Supported: the states whose result
 * does not depend on the order of the fragments nor on the target's value, i.e. dst factor
 * One with Add or ReverseSubtract and a source factor among Zero, One, Src, OneMinusSrc,
 * SrcAlpha, OneMinusSrcAlpha, Constant, OneMinusConstant: each sample then adds
 * +-w * src * factor, which the exact integer tile sums take in any order. The others (Dst*
 * factors, SrcAlphaSaturated, a dst factor other than One, Subtract, Min, Max) return
 * LG_E_UNSUPPORTED; out-of-range values LG_E_INVALID. */
int lg_image_set_blend(lg_image* img, const lg_blend* blend);
int lg_image_get_blend(const lg_image* img, lg_blend* out);

/* ---- 8-bit encode: Renderer::make_screenshot's pixel conversion (renderer.rs:313-328) ---- */
enum lg_encode_order {
  LG_ENCODE_BGRA = 0,  /* the reference's bytes: B, G, R, A (it then saves them as RGBA) */
  LG_ENCODE_RGBA = 1
};
/* Each RGBA16F channel of img's resolved target -> f32 -> powf(f, 1/2.2) * 255 -> u8 with
 * Rust's saturating `as` (NaN and values <= 0 give 0, >= 255 give 255, else truncation), on the
 * GPU; host gets width * height * 4 bytes, row 0 at the top (the copy of renderer.rs:271-291
 * with its row padding removed). The JPEG file write is not part of it. */
int lg_image_encode_8bit(lg_image* img, uint32_t order, uint8_t* host, uint64_t cap_bytes);
/* The conversion as a table: table[h] = the u8 of the half with bits h (65536 entries). It is
 * computed on the device (FP64 pow rounded to FP32) and is what lg_image_encode_8bit applies. */
int lg_encode_table(lg_ctx* ctx, uint8_t* table);

/* ---- accumulation: LineList draw + One/One blend (shader.wgsl:14-28, mod.rs:57-73) ---- */
/* Adds every segment into img's FP32 accumulator: rgb += w*rgb, a += w*a*a, with the
 * anti-aliased column/row sampling rule of this build. */
int lg_accumulate(lg_ctx* ctx, const lg_segments* segs, lg_image* img);
/* lg_accumulate without device allocation. No counterpart in the reference: it is for callers
 * that cannot allocate device memory (serving loops with a fixed footprint, harnesses that
 * forbid hipMalloc). The same kernels and the same result bits as lg_accumulate, with their
 * scratch in one static device array of about 64 MB (60.6 MiB) per device (kept until the
 * process ends): an image of at most 4096 x 4096 pixels (2048 x 2048 with 32-pixel tiles), at
 * most 8,388,608 segment-tile pairs and at most 128 tiles split over several work items per
 * call. Beyond a limit it returns LG_E_CAPACITY and deposits nothing. Calls on one device share
 * the array and are serialised by the library (each finishes before it returns). */
int lg_accumulate_noalloc(lg_ctx* ctx, const lg_segments* segs, lg_image* img);
/* FP32 accumulator -> RGBA16F target (round to nearest even), alpha += 1 (clear value). */
int lg_resolve(lg_ctx* ctx, lg_image* img);
/* One frame: clear, trace, accumulate, resolve (LightGarden::draw + Renderer::render,
 * mod.rs:680-696, renderer.rs:420). `segs` receives the trace output. */
int lg_render(lg_scene* scene, const lg_params* params, lg_segments* segs, lg_image* img);

/* ---- string mod: StringMod::draw on the GPU (string_mod.rs:3-158) ---------------------- */
enum lg_sm_mode { LG_SM_ADD = 0, LG_SM_MUL = 1, LG_SM_POW = 2, LG_SM_BASE = 3 };  /* StringModMode */
enum lg_sm_curve {                                                    /* Curve (string_mod.rs:182-188) */
  LG_CURVE_CIRCLE = 0,        /* unit circle                                                  */
  LG_CURVE_COMPLEX_EXP = 1,   /* c^(turns n): curve_f = {c.re, c.im}                          */
  LG_CURVE_HYPOTROCHOID = 2,  /* curve_u = {r, s, d}                                          */
  LG_CURVE_LISSAJOUS = 3      /* curve_u = {a, b}, curve_f[0] = delta                         */
};
#define LG_MAX_MOD_COLORS 256           /* modulo colours per StringMod                         */
#define LG_MAX_CROSSING_LINES (1u << 18) /* lines of a nested StringMod's outer (O(L^2) pairs)   */
typedef struct lg_mod_rem_color {       /* ModRemColor (string_mod.rs:166-171)                  */
  uint64_t modulo;                      /* > 0                                                   */
  uint64_t rem;
  float color[4];
} lg_mod_rem_color;
typedef struct lg_string_mod {          /* StringMod (string_mod.rs:3-15)                        */
  uint64_t modulo;
  uint64_t num;
  uint64_t turns;
  uint32_t mode;                        /* lg_sm_mode                                            */
  uint32_t curve;                       /* lg_sm_curve                                           */
  uint64_t curve_u[3];
  double curve_f[2];
  double scale;                         /* curve radius; 1 = the reference's curves              */
  float color[4];
  const lg_mod_rem_color* modulo_colors;
  uint32_t n_modulo_colors;
  uint32_t _pad0;
  const struct lg_string_mod* nested;   /* Option<Box<StringMod>>; NULL = None. Its own nested
                                           is not read (draw() nests one level)             */
} lg_string_mod;
/* LightGarden::draw in Mode::StringMod (mod.rs:681-689): the segments of every StringMod's
 * draw() (string_mod.rs:152-158), concatenated in order, into `out` (device; created with
 * LG_SEG_VERTEX_COLORS; replaces its contents). A nested StringMod draws over the crossing
 * points of its outer lines. Points in FP64, stored as FP32 vertices; key = emission index.
 * LG_E_INVALID for an unknown mode/curve, a modulo colour with modulo 0 (the reference divides
 * by it), more than LG_MAX_MOD_COLORS colours or a nested outer above LG_MAX_CROSSING_LINES. */
int lg_string_mod_draw(lg_ctx* ctx, uint32_t n, const lg_string_mod* mods, lg_segments* out);
/* StringMod::line_crossings_as_points (string_mod.rs:87-102): the crossing points of sm's
 * lines, every ordered pair in the reference's order, 2 doubles each into xy. LG_E_CAPACITY
 * with *n_points set when cap_points is too small. */
int lg_string_mod_crossings(lg_ctx* ctx, const lg_string_mod* sm, double* xy, uint64_t cap_points,
                            uint64_t* n_points);

/* ---- batched form (no reference counterpart: the reference renders one scene per frame) --
 * lg_render for n scenes in one frame: every stage runs once over all scenes (persistent
 * work-queue kernels over device-built work lists) and the launch sequence is replayed from a
 * hipGraph while the batch keeps its shape. Scenes, segment buffers and images must be
 * distinct; all params must agree on LG_TRACE_FP64. Results equal n separate lg_render
 * calls bit for bit (accumulation sums are exact integers until one final conversion). */
int lg_batch_render(lg_ctx* ctx, uint32_t n, lg_scene* const* scenes, const lg_params* params,
                    lg_segments* const* segs, lg_image* const* images);
/* Launch tuning of a context. No counterpart in the reference (its trace is one CPU pass):
 * these are the knobs of the persistent GPU work lists, read by the autotuner. Apart from
 * `tile` none of them changes results: images are the same bits for every setting. */
typedef struct lg_tuning {
  uint32_t rays_per_item;  /* rays per trace work item, at most, [64, 2^20]; default 1024 */
  uint32_t min_piece;      /* smallest tile work item in segment-tile pairs, >= 64; default 2048 */
  uint32_t max_piece;      /* largest tile work item, >= min_piece; default 32768; work items
                              hold at most 32768 pairs whatever the setting (the fixed point
                              of two channels per LDS word is sized for that), and at most
                              max(min_piece, 8192) where the tile walk goes pair by pair
                              (32-pixel tiles, one channel per LDS word, tile_block 512) */
  uint32_t trace_waves;    /* trace workgroups per compute unit, [1, 16]; default 4 */
  uint32_t bvh_min_objects; /* scenes with at least this many objects cull by their objects'
                               bounding boxes, others test every object (as FP32 traces
                               do of scenes with an object or a light beyond 64 units from
                               the origin); 0xffffffff: never; default 8 */
  uint32_t tile;           /* screen tile edge of the accumulation, 32 or 64 pixels; default 64.
                              Unlike the other knobs it moves sample positions by FP32
                              rounding and the two-channel fixed point's scale with the tile's
                              pair count, so images differ within the accumulation's error
                              bound (not bit for bit) between the two sizes; at 32 an image
                              has at most 4096 x 4096 pixels */
  uint32_t trace_chunk;    /* bounce generations per trace launch, [1, 3]; default 2. Above 1 a
                              trace workgroup keeps its rays' children on chip (LDS) for the
                              launch's further generations and writes only the last one's to
                              the ray queue in HBM (bounce-chunking); lowered for a frame whose
                              scene leaves no LDS room for it */
  uint32_t tile_block;     /* threads per tile workgroup, 1024 (one per compute unit) or 512
                              (two per compute unit), for frames at 64-pixel tiles whose every
                              scene keeps two colour channels per LDS word; default 1024.
                              Frames with traced scenes of one to three lights under the
                              default blend always take 1024 */
} lg_tuning;
int lg_ctx_get_tuning(const lg_ctx* ctx, lg_tuning* out);
int lg_ctx_set_tuning(lg_ctx* ctx, const lg_tuning* tuning);
/* Replay frames from a hipGraph while the batch keeps its shape (default on). */
int lg_ctx_set_graphs(lg_ctx* ctx, int enable);
/* Tile accumulation with two colour channels per 64-bit LDS add (default on). It applies to
 * each scene of a frame whose every deposit is non-negative (colours >= 0, no ReverseSubtract,
 * no blend factor below 0 on them); other scenes take one channel per add, so a scene's image
 * does not depend on the scenes batched with it. No reference counterpart (the reference
 * blends in wgpu). Off: every scene takes one channel per add. */
int lg_ctx_set_packed_accumulation(lg_ctx* ctx, int enable);

/* ---- serving (no reference counterpart: the reference renders one scene per event-loop
 * frame, LightGarden::draw mod.rs:680-696; this is the batch/serve seam lg_server_*) ----
 * A server owns a worker thread that keeps up to `slots` batched frames in flight, each on a
 * stream of its own, and forms the next frame from waiting requests whenever a slot frees up
 * (continuous batching). Requests are admitted in arrival order while the resident working
 * set fits the HBM budget: every resident scene's ray queues and segment buffer (owned by the
 * server, kept across requests and edits) plus the images of admitted requests and the
 * frames' scratch; idle scenes are evicted least-recently-used first. Requests for one scene
 * run in submission order; an edit replaces one object right before its render. A scene's
 * image is the same bits whatever else shares its frame.
 * Scenes and images given to a server are the server's until their requests complete (do
 * not change or render them meanwhile); destroy the server before them. */
typedef struct lg_server lg_server;
typedef struct lg_server_config {
  uint64_t hbm_budget;  /* bytes; 0 = 64 GiB */
  uint32_t max_batch;   /* scenes per frame; 0 = 256 */
  uint32_t slots;       /* frames in flight, 1..4; 0 = 2 */
} lg_server_config;
typedef struct lg_request {
  lg_scene* scene;      /* resident scene, rendered with `params` into `image` (lg_render) */
  lg_image* image;
  lg_params params;     /* FP32 trace */
  int32_t edit_index;   /* >= 0: lg_scene_replace_object(scene, edit_index, &edit) first */
  int32_t _pad0;
  lg_object edit;
  lg_segments* segments; /* optional: before the request is reported done, its traced segments
                            are copied here (the buffer grows as needed; the caller's until
                            then, like the image) */
} lg_request;
typedef struct lg_result {
  int32_t status;       /* LG_OK or the error of the frame that rendered the request */
  uint32_t batch_size;  /* requests in that frame */
  uint64_t segments;    /* segments traced for the request */
  double submit_us;     /* server clock, microseconds: submitted, */
  double start_us;      /* its frame launched, */
  double end_us;        /* its frame completed */
} lg_result;
typedef struct lg_server_stats {
  uint64_t submitted, completed, frames, evictions;
  uint64_t resident_bytes, peak_resident_bytes;
  double busy_us;       /* time with at least one frame in flight */
} lg_server_stats;
int lg_server_create(lg_ctx* ctx, const lg_server_config* cfg, lg_server** out);
/* Finishes every submitted request, then stops. */
int lg_server_destroy(lg_server* server);
int lg_server_submit(lg_server* server, const lg_request* request, uint64_t* ticket);
/* Waits up to timeout_s (< 0: forever) for a request; LG_E_TIMEOUT if it has not finished.
 * Each ticket's result is returned once. */
int lg_server_wait(lg_server* server, uint64_t ticket, double timeout_s, lg_result* out);
int lg_server_get_stats(lg_server* server, lg_server_stats* out);

#ifdef __cplusplus
}
#endif

#endif /* LG_H */
