// lg_api.hip — the C ABI of include/lg.h: contexts, scenes, buffers, images, and the entry
// points trace / accumulate / resolve / render / batch render, all of which run through the
// batched frame pipeline (lg_pipeline.hip).
//
// The scene API mirrors Tracer (src/light_garden/tracer.rs:4-17, 48-116). A scene keeps
// the caller's lg_object / lg_light values on the host (FP64, as the reference does) and
// compiles them into world-space device records on the first trace after an edit.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "lg_host.h"

namespace lg {

// ---- errors --------------------------------------------------------------------------------
static thread_local std::string g_error;

void set_error(const std::string& msg) { g_error = msg; }

int hip_fail(hipError_t e, const char* what) {
  g_error = std::string(what) + ": " + hipGetErrorString(e);
  return e == hipErrorOutOfMemory ? LG_E_OOM : LG_E_HIP;
}

int fail(int code, const std::string& msg) {
  g_error = msg;
  return code;
}

// ---- buffers -------------------------------------------------------------------------------
int DevBuf::ensure(size_t need) {
  if (need <= bytes && p) return LG_OK;
  reset();
  size_t b = need ? need : 16;
  LG_HIP(hipMalloc(&p, b));
  bytes = b;
  return LG_OK;
}

int PinnedBuf::ensure(size_t need) {
  if (need <= bytes && p) return LG_OK;
  reset();
  size_t b = need ? need : 16;
  LG_HIP(hipHostMalloc(&p, b));
  bytes = b;
  return LG_OK;
}

// ---- profiling -----------------------------------------------------------------------------
StageScope::StageScope(lg_ctx* c, const char* name, uint64_t work) : ctx(c) {
  if (!ctx->profiling) return;
  StageRec r;
  r.name = name;
  r.work = work;
  r.start = ctx->get_event();
  r.stop = ctx->get_event();
  if (!r.start || !r.stop) return;
  (void)hipEventRecord(r.start, ctx->stream);
  ctx->pending.push_back(r);
  idx = ctx->pending.size() - 1;
}

StageScope::~StageScope() {
  if (idx != (size_t)-1) (void)hipEventRecord(ctx->pending[idx].stop, ctx->stream);
}

void begin_call(lg_ctx* ctx) {
  for (auto& r : ctx->pending) {
    ctx->event_pool.push_back(r.start);
    ctx->event_pool.push_back(r.stop);
  }
  ctx->pending.clear();
}

// Resolves event times after the stream has been synchronised.
void end_call(lg_ctx* ctx) {
  if (!ctx->profiling) return;
  std::vector<lg_stage_time> out;
  for (auto& r : ctx->pending) {
    float ms = 0.0f;
    (void)hipEventElapsedTime(&ms, r.start, r.stop);
    auto it = std::find_if(out.begin(), out.end(), [&](const lg_stage_time& t) {
      return std::strncmp(t.name, r.name.c_str(), sizeof(t.name)) == 0;
    });
    if (it == out.end()) {
      lg_stage_time t{};
      std::snprintf(t.name, sizeof(t.name), "%s", r.name.c_str());
      out.push_back(t);
      it = out.end() - 1;
    }
    it->ms += ms;
    it->launches += 1;
    it->work += r.work;
    it->work2 += r.work2;
  }
  ctx->last_times = out;
}

// ---- scene compilation -------------------------------------------------------------------
struct Frame {
  double o[2];
  double r[4];  // column-major
};

static Frame frame_identity() { return Frame{{0, 0}, {1, 0, 0, 1}}; }

static Frame frame_compose(const Frame& parent, const double origin[2], const double rot[4]) {
  Frame f;
  f.o[0] = parent.o[0] + parent.r[0] * origin[0] + parent.r[2] * origin[1];
  f.o[1] = parent.o[1] + parent.r[1] * origin[0] + parent.r[3] * origin[1];
  // parent.R * rot (column-major)
  f.r[0] = parent.r[0] * rot[0] + parent.r[2] * rot[1];
  f.r[1] = parent.r[1] * rot[0] + parent.r[3] * rot[1];
  f.r[2] = parent.r[0] * rot[2] + parent.r[2] * rot[3];
  f.r[3] = parent.r[1] * rot[2] + parent.r[3] * rot[3];
  return f;
}

static void frame_point(const Frame& f, double x, double y, double& ox, double& oy) {
  ox = f.o[0] + f.r[0] * x + f.r[2] * y;
  oy = f.o[1] + f.r[1] * x + f.r[3] * y;
}

static bool finite_all(const double* v, int n) {
  for (int i = 0; i < n; i++)
    if (!std::isfinite(v[i])) return false;
  return true;
}

static bool rotation_ok(const double r[4]) {
  if (!finite_all(r, 4)) return false;
  // columns unit length and orthogonal
  double c0 = r[0] * r[0] + r[1] * r[1], c1 = r[2] * r[2] + r[3] * r[3];
  double d = r[0] * r[2] + r[1] * r[3];
  return std::fabs(c0 - 1.0) < 1e-6 && std::fabs(c1 - 1.0) < 1e-6 && std::fabs(d) < 1e-6;
}

static bool is_closed_prim(int kind) {
  return kind == LG_SHAPE_CIRCLE || kind == LG_SHAPE_RECT || kind == LG_SHAPE_ELLIPSE ||
         kind == LG_SHAPE_CONVEX_POLYGON;
}

static bool shape_is_framed(int kind) { return is_closed_prim(kind) || kind == LG_SHAPE_LOGIC; }

// One primitive shape node -> world-space record. Polygon vertices are appended to verts.
static int compile_prim(const lg_object& obj, int oi, const lg_shape& s, const Frame& parent,
                        std::vector<Rec<double>>& out, std::vector<double>& verts) {
  Rec<double> R;
  std::memset(&R, 0, sizeof(R));
  R.kind = s.kind;
  R.obj = oi;
  switch (s.kind) {
    case LG_SHAPE_LINE_SEGMENT: {
      if (!finite_all(s.p, 4)) return fail(LG_E_INVALID, "line segment: non-finite point");
      double ax, ay, bx, by;
      frame_point(parent, s.p[0], s.p[1], ax, ay);
      frame_point(parent, s.p[2], s.p[3], bx, by);
      double ex = bx - ax, ey = by - ay;
      double l = std::sqrt(ex * ex + ey * ey);
      if (!(l > 0)) return fail(LG_E_INVALID, "line segment: zero length");
      R.p[0] = ax; R.p[1] = ay; R.p[2] = ex; R.p[3] = ey;
      R.p[4] = -ey / l; R.p[5] = ex / l;
      break;
    }
    case LG_SHAPE_CUBIC_BEZIER: {
      if (!finite_all(s.p, 8)) return fail(LG_E_INVALID, "bezier: non-finite point");
      double P[8];
      for (int i = 0; i < 4; i++) frame_point(parent, s.p[2 * i], s.p[2 * i + 1], P[2 * i], P[2 * i + 1]);
      for (int c = 0; c < 2; c++) {
        double p0 = P[c], p1 = P[2 + c], p2 = P[4 + c], p3 = P[6 + c];
        R.p[0 + c] = -p0 + 3.0 * p1 - 3.0 * p2 + p3;
        R.p[2 + c] = 3.0 * p0 - 6.0 * p1 + 3.0 * p2;
        R.p[4 + c] = 3.0 * (p1 - p0);
        R.p[6 + c] = p0;
      }
      // bounding box of the control points (the curve lies in their convex hull), padded so
      // that the FP32 culling test never rejects a hit
      double x0 = P[0], x1 = P[0], y0 = P[1], y1 = P[1], mag = 0.0;
      for (int i = 0; i < 4; i++) {
        x0 = std::min(x0, P[2 * i]);
        x1 = std::max(x1, P[2 * i]);
        y0 = std::min(y0, P[2 * i + 1]);
        y1 = std::max(y1, P[2 * i + 1]);
        mag = std::max(mag, std::max(std::fabs(P[2 * i]), std::fabs(P[2 * i + 1])));
      }
      const double pad = 1e-5 * (1.0 + mag);
      R.p[8] = x0 - pad;
      R.p[9] = y0 - pad;
      R.p[10] = x1 + pad;
      R.p[11] = y1 + pad;
      break;
    }
    case LG_SHAPE_CIRCLE: {
      if (!finite_all(s.origin, 2) || !std::isfinite(s.p[0]) || !(s.p[0] > 0))
        return fail(LG_E_INVALID, "circle: bad centre or radius");
      double cx, cy;
      frame_point(parent, s.origin[0], s.origin[1], cx, cy);
      R.p[0] = cx; R.p[1] = cy; R.p[2] = s.p[0]; R.p[3] = s.p[0] * s.p[0];
      break;
    }
    case LG_SHAPE_RECT:
    case LG_SHAPE_ELLIPSE:
    case LG_SHAPE_CONVEX_POLYGON: {
      if (!finite_all(s.origin, 2) || !rotation_ok(s.rotation))
        return fail(LG_E_INVALID, "shape: bad origin or rotation (must be a 2x2 rotation)");
      Frame f = frame_compose(parent, s.origin, s.rotation);
      R.p[0] = f.o[0]; R.p[1] = f.o[1];
      R.p[2] = f.r[0]; R.p[3] = f.r[1];  // local x axis
      R.p[4] = f.r[2]; R.p[5] = f.r[3];  // local y axis
      if (s.kind == LG_SHAPE_RECT || s.kind == LG_SHAPE_ELLIPSE) {
        if (!std::isfinite(s.p[0]) || !std::isfinite(s.p[1]) || !(s.p[0] > 0) || !(s.p[1] > 0))
          return fail(LG_E_INVALID, "rect/ellipse: sizes must be positive");
        if (s.kind == LG_SHAPE_RECT) {
          R.p[6] = 0.5 * s.p[0];
          R.p[7] = 0.5 * s.p[1];
        } else {
          R.p[6] = s.p[0];
          R.p[7] = s.p[1];
        }
      } else {
        int nv = s.n_vertices, first = s.vertex_offset;
        if (nv < 3 || first < 0 || first + nv > LG_MAX_POLY_VERTICES)
          return fail(LG_E_INVALID, "polygon: bad vertex range");
        const double* v = obj.vertices + 2 * first;
        if (!finite_all(v, 2 * nv)) return fail(LG_E_INVALID, "polygon: non-finite vertex");
        for (int i = 0; i < nv; i++) {
          const double* a = v + 2 * i;
          const double* b = v + 2 * ((i + 1) % nv);
          const double* c = v + 2 * ((i + 2) % nv);
          double cr = (b[0] - a[0]) * (c[1] - b[1]) - (b[1] - a[1]) * (c[0] - b[0]);
          if (!(cr > 0)) return fail(LG_E_INVALID, "polygon: vertices must be convex and counter-clockwise");
        }
        R.aux = (int32_t)(verts.size() / 2);
        R.op = nv;
        if ((int)(verts.size() / 2) + nv > kMaxPolyVertices)
          return fail(LG_E_UNSUPPORTED, "scene: too many polygon vertices");
        for (int i = 0; i < 2 * nv; i++) verts.push_back(v[i]);
      }
      break;
    }
    default: return fail(LG_E_INVALID, "unknown shape kind");
  }
  out.push_back(R);
  return LG_OK;
}

// Node ni of obj's shape tree and its subtree, in prefix order, in frame f (a Logic node's
// origin and rotation compose with its parent's). Children come after their parent in
// shapes[], so the tree has no cycles; leaves are closed primitives.
static int compile_node(const lg_object& obj, int oi, int ni, const Frame& f, std::vector<Rec<double>>& recs,
                        std::vector<double>& verts, std::vector<int>& leaves) {
  const lg_shape& s = obj.shapes[ni];
  if (s.kind != LG_SHAPE_LOGIC) {
    if (!is_closed_prim(s.kind))
      return fail(LG_E_UNSUPPORTED, "logic: operands must be circles, rects, ellipses, convex polygons or logic");
    leaves.push_back((int)recs.size());
    return compile_prim(obj, oi, s, f, recs, verts);
  }
  if (s.op < LG_LOGIC_AND || s.op > LG_LOGIC_AND_NOT) return fail(LG_E_INVALID, "logic: bad op");
  if (s.child_a <= ni || s.child_b <= ni || s.child_a >= obj.n_shapes || s.child_b >= obj.n_shapes ||
      s.child_a == s.child_b)
    return fail(LG_E_INVALID, "logic: bad operand index (operands follow their node in shapes[])");
  if (!finite_all(s.origin, 2) || !rotation_ok(s.rotation)) return fail(LG_E_INVALID, "logic: bad origin or rotation");
  const Frame g = frame_compose(f, s.origin, s.rotation);
  const size_t at = recs.size();
  Rec<double> L;
  std::memset(&L, 0, sizeof(L));
  L.kind = REC_LOGIC;
  L.obj = oi;
  L.op = s.op;
  recs.push_back(L);
  int rc = compile_node(obj, oi, s.child_a, g, recs, verts, leaves);
  if (rc) return rc;
  if ((rc = compile_node(obj, oi, s.child_b, g, recs, verts, leaves))) return rc;
  recs[at].aux = (int32_t)(recs.size() - at);
  return LG_OK;
}

static int compile_object(const lg_object& obj, int oi, std::vector<Rec<double>>& recs,
                          std::vector<double>& verts) {
  if (obj.n_shapes < 1 || obj.n_shapes > LG_MAX_SHAPES)
    return fail(LG_E_INVALID, "object " + std::to_string(oi) + ": n_shapes out of range");
  if (obj.has_material && (!std::isfinite(obj.refractive_index) || !(obj.refractive_index > 0)))
    return fail(LG_E_INVALID, "object " + std::to_string(oi) + ": bad refractive index");
  const lg_shape& root = obj.shapes[0];
  Frame id = frame_identity();
  if (root.kind == LG_SHAPE_LOGIC) {
    const size_t top = recs.size();
    std::vector<int> leaves;
    const int rc = compile_node(obj, oi, 0, id, recs, verts, leaves);
    if (rc) return rc;
    if ((int)leaves.size() > kLogicLeaves) return fail(LG_E_UNSUPPORTED, "logic: more than 4 primitives");
    Rec<double>& R = recs[top];
    if (R.aux != 3) R.kind = REC_TREE;
    for (size_t k = 0; k < leaves.size(); k++) R.p[k] = (double)(leaves[k] - (int)top);
    R.p[4] = (double)leaves.size();
    return LG_OK;
  }
  return compile_prim(obj, oi, root, id, recs, verts);
}

// A scene's tables packed for one copy to the device, each from a 256-byte boundary. (A copy of
// its own for each of fourteen tables cost an edited scene about 3 us each on the device, and the
// calls.)
struct TablePack {
  std::vector<char> bytes;
  template <typename U>
  size_t add(const std::vector<U>& v) {
    const size_t off = (bytes.size() + 255) & ~size_t(255);
    bytes.resize(off + v.size() * sizeof(U));
    if (!v.empty()) std::memcpy(bytes.data() + off, v.data(), v.size() * sizeof(U));
    return off;
  }
};

// ---- object bounding volumes -------------------------------------------------------------
struct Box2 {
  double lo[2], hi[2];
  void add(double x, double y) {
    lo[0] = std::min(lo[0], x);
    lo[1] = std::min(lo[1], y);
    hi[0] = std::max(hi[0], x);
    hi[1] = std::max(hi[1], y);
  }
  void add(const Box2& b) {
    add(b.lo[0], b.lo[1]);
    add(b.hi[0], b.hi[1]);
  }
};

static Box2 empty_box() { return Box2{{INFINITY, INFINITY}, {-INFINITY, -INFINITY}}; }

// World box of one primitive record (REC_* parameterisation).
static Box2 rec_box(const Rec<double>& R, const std::vector<double>& verts) {
  Box2 b = empty_box();
  const double* p = R.p;
  switch (R.kind) {
    case REC_SEG: b.add(p[0], p[1]); b.add(p[0] + p[2], p[1] + p[3]); break;
    case REC_BEZ: b.add(p[8], p[9]); b.add(p[10], p[11]); break;
    case REC_CIRCLE: b.add(p[0] - p[2], p[1] - p[2]); b.add(p[0] + p[2], p[1] + p[2]); break;
    case REC_RECT: {
      // world = c + x u + y v, u = (p2, p3), v = (p4, p5), |x| <= hw, |y| <= hh
      const double hx = std::fabs(p[2]) * p[6] + std::fabs(p[4]) * p[7];
      const double hy = std::fabs(p[3]) * p[6] + std::fabs(p[5]) * p[7];
      b.add(p[0] - hx, p[1] - hy);
      b.add(p[0] + hx, p[1] + hy);
      break;
    }
    case REC_ELLIPSE: {
      const double hx = std::hypot(p[6] * p[2], p[7] * p[4]);
      const double hy = std::hypot(p[6] * p[3], p[7] * p[5]);
      b.add(p[0] - hx, p[1] - hy);
      b.add(p[0] + hx, p[1] + hy);
      break;
    }
    case REC_POLY:
      for (int i = 0; i < R.op; i++) {
        const double x = verts[2 * (R.aux + i)], y = verts[2 * (R.aux + i) + 1];
        b.add(p[0] + p[2] * x + p[4] * y, p[1] + p[3] * x + p[5] * y);
      }
      break;
    default: break;
  }
  return b;
}

static float round_down(double v) {
  float f = (float)v;
  return (double)f > v ? std::nextafter(f, -INFINITY) : f;
}
static float round_up(double v) {
  float f = (float)v;
  return (double)f < v ? std::nextafter(f, INFINITY) : f;
}

static uint32_t spread_bits(uint32_t v) {  // 16 bits -> even bit positions
  v &= 0xffffu;
  v = (v | (v << 8)) & 0x00ff00ffu;
  v = (v | (v << 4)) & 0x0f0f0f0fu;
  v = (v | (v << 2)) & 0x33333333u;
  v = (v | (v << 1)) & 0x55555555u;
  return v;
}

// Object boxes padded by 1e-5 (1 + |coordinates|) + 2e-6 reach, far more than the FP32 culling
// pass's error and than the rounding of an FP64 inside test: a point outside an object's padded box
// is neither hit by a culled ray nor contained. *reach: the largest |coordinate| that a ray
// starts from, at a light or on an object; both the box test and the FP32 hits are off by some
// 2^-21 of the ray's origin (5e-7), whatever the object's own coordinates.
static std::vector<Box2> object_boxes(const std::vector<Rec<double>>& recs, const std::vector<double>& verts,
                                      const std::vector<int32_t>& obj_rec, const std::vector<lg_light>& lights,
                                      double* reach) {
  const int n = (int)obj_rec.size();
  std::vector<Box2> boxes(n);
  for (int o = 0; o < n; o++) {
    const int top = obj_rec[o];
    Box2 b = empty_box();
    if (recs[top].kind == REC_LOGIC || recs[top].kind == REC_TREE) {
      for (int k = top + 1; k < top + recs[top].aux; k++)
        if (recs[k].kind != REC_LOGIC) b.add(rec_box(recs[k], verts));
    } else {
      b = rec_box(recs[top], verts);
    }
    boxes[o] = b;
  }
  auto magnitude = [](const Box2& b) {
    return std::max(std::max(std::fabs(b.lo[0]), std::fabs(b.lo[1])), std::max(std::fabs(b.hi[0]), std::fabs(b.hi[1])));
  };
  double r = 0.0;
  for (const Box2& b : boxes) r = std::max(r, magnitude(b));
  for (const lg_light& l : lights) {
    Box2 b = empty_box();
    b.add(l.position[0], l.position[1]);
    if (l.kind == LG_LIGHT_DIRECTIONAL) b.add(l.direction[0], l.direction[1]);
    if (std::isfinite(magnitude(b))) r = std::max(r, magnitude(b));  // (others are refused later)
  }
  for (Box2& b : boxes) {
    const double pad = 1e-5 * (1.0 + magnitude(b)) + 2e-6 * r;
    b.lo[0] -= pad;
    b.lo[1] -= pad;
    b.hi[0] += pad;
    b.hi[1] += pad;
  }
  *reach = r;
  return boxes;
}

// Objects in Morton order of their box centres.
static std::vector<int> morton_order(const std::vector<Box2>& boxes) {
  const int n = (int)boxes.size();
  Box2 all = empty_box();
  for (int o = 0; o < n; o++) all.add(boxes[o]);
  std::vector<uint32_t> code(n);
  const double sx = all.hi[0] > all.lo[0] ? 65535.0 / (all.hi[0] - all.lo[0]) : 0.0;
  const double sy = all.hi[1] > all.lo[1] ? 65535.0 / (all.hi[1] - all.lo[1]) : 0.0;
  for (int o = 0; o < n; o++) {
    const double cx = 0.5 * (boxes[o].lo[0] + boxes[o].hi[0]), cy = 0.5 * (boxes[o].lo[1] + boxes[o].hi[1]);
    const uint32_t qx = (uint32_t)std::min(65535.0, std::max(0.0, (cx - all.lo[0]) * sx));
    const uint32_t qy = (uint32_t)std::min(65535.0, std::max(0.0, (cy - all.lo[1]) * sy));
    code[o] = spread_bits(qx) | (spread_bits(qy) << 1);
  }
  std::vector<int> order(n);
  for (int o = 0; o < n; o++) order[o] = o;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return code[a] < code[b]; });
  return order;
}

static float4 box_f32(const Box2& b) {
  return make_float4(round_down(b.lo[0]), round_down(b.lo[1]), round_up(b.hi[0]), round_up(b.hi[1]));
}

// MediumMasks of objects with the given boxes, and the map of their buckets.
static std::vector<MediumMasks> medium_masks(const std::vector<float4>& box, const std::vector<uint32_t>& flags,
                                             float map[4]) {
  std::vector<MediumMasks> M((box.size() + 63) / 64);
  if (!M.empty()) std::memset(M.data(), 0, M.size() * sizeof(M[0]));
  auto has = [&](size_t o) {
    return (flags[o] & (OBJ_MATERIAL | OBJ_CLOSED)) == (OBJ_MATERIAL | OBJ_CLOSED);
  };
  float4 all = make_float4(INFINITY, INFINITY, -INFINITY, -INFINITY);
  for (size_t o = 0; o < box.size(); o++)
    if (has(o))
      all = make_float4(std::min(all.x, box[o].x), std::min(all.y, box[o].y), std::max(all.z, box[o].z),
                        std::max(all.w, box[o].w));
  auto axis = [](float lo, float hi, float* m) {
    m[0] = kMediumBuckets / (hi - lo);
    m[1] = -lo * m[0];
    if (!std::isfinite(m[0]) || !std::isfinite(m[1])) m[0] = m[1] = 0.0f;  // one bucket for all
  };
  axis(all.x, all.z, map);
  axis(all.y, all.w, map + 2);
  for (size_t o = 0; o < box.size(); o++) {
    if (!has(o)) continue;
    MediumMasks& m = M[o / 64];
    const uint64_t bit = 1ull << (o % 64);
    for (int k = medium_bucket(box[o].x, map[0], map[1]); k <= medium_bucket(box[o].z, map[0], map[1]); k++) m.x[k] |= bit;
    for (int k = medium_bucket(box[o].y, map[2], map[3]); k <= medium_bucket(box[o].w, map[2], map[3]); k++) m.y[k] |= bit;
  }
  return M;
}

// Centre and half sizes of a box, in FP32 and not smaller.
static float4 centre_f32(const Box2& b) {
  const float cx = (float)(0.5 * (b.lo[0] + b.hi[0])), cy = (float)(0.5 * (b.lo[1] + b.hi[1]));
  return make_float4(cx, cy, round_up(std::max(b.hi[0] - cx, cx - b.lo[0])),
                     round_up(std::max(b.hi[1] - cy, cy - b.lo[1])));
}

// The culling blocks of objects with the given boxes and first records (CullBlock).
struct CullLists {
  std::vector<CullBlock> blocks;
  std::vector<float4> box;
  std::vector<int32_t> rec;
};
static CullLists build_blocks(const std::vector<Box2>& boxes, const std::vector<int32_t>& top,
                              const std::vector<Rec<double>>& recs) {
  CullLists C;
  const std::vector<int> order = morton_order(boxes);
  for (size_t b = 0; b < order.size(); b += kCullBlock) {
    const size_t n = std::min<size_t>(kCullBlock, order.size() - b);
    CullBlock B;
    std::memset(&B, 0, sizeof(B));
    B.first = (int32_t)C.box.size();
    B.n = (int32_t)n;
    Box2 all = empty_box();
    uint64_t mask[8] = {};
    for (size_t k = 0; k < n; k++) {
      const int o = order[b + k];
      all.add(boxes[o]);
      mask[recs[top[o]].kind & 7] |= 1ull << k;
      C.box.push_back(centre_f32(boxes[o]));
      C.rec.push_back(top[o]);
    }
    const float4 u = centre_f32(all);
    B.box[0] = u.x;
    B.box[1] = u.y;
    B.box[2] = u.z;
    B.box[3] = u.w;
    for (int k = 0; k < 8; k++)
      if (mask[k]) {
        B.kinds |= (uint32_t)k << (4 * B.n_kinds);
        B.kind[B.n_kinds++] = mask[k];
      }
    while (C.box.size() % kBoxGroup) {  // (no kind has a bit for these)
      C.box.push_back(u);
      C.rec.push_back(-1);
    }
    C.blocks.push_back(B);
  }
  return C;
}

// Copies the tables on `st`, the stream of the frame that will read the scene.
int compile_scene(lg_scene* sc, hipStream_t st) {
  if (!sc->dirty) return LG_OK;
  std::vector<Rec<double>> recs;
  std::vector<double> verts;
  std::vector<int32_t> obj_rec;
  std::vector<uint32_t> flags;
  std::vector<double> n64;
  if (sc->objects.size() > (size_t)kMaxObjects) return fail(LG_E_UNSUPPORTED, "scene: too many objects");
  for (size_t i = 0; i < sc->objects.size(); i++) {
    const lg_object& o = sc->objects[i];
    obj_rec.push_back((int32_t)recs.size());
    int rc = compile_object(o, (int)i, recs, verts);
    if (rc) return rc;
    uint32_t f = 0;
    if (o.has_material) f |= OBJ_MATERIAL;
    if (shape_is_framed(o.shapes[0].kind)) f |= OBJ_CLOSED;
    flags.push_back(f);
    n64.push_back(o.has_material ? o.refractive_index : 1.0);
  }
  if ((int)recs.size() > kMaxRecords) return fail(LG_E_UNSUPPORTED, "scene: too many shape records");
  // The records of Logic trees of more than two primitives move after every other object's:
  // the object walk covers the records before the first tree, and the trees are tested in a
  // loop of their own (records are relocatable: a Logic record refers to its operands by
  // offset). Objects keep their order within each group.
  std::vector<int32_t> tree_rec;
  {
    std::vector<Rec<double>> ordered;
    ordered.reserve(recs.size());
    std::vector<int32_t> at(obj_rec.size());
    for (int trees = 0; trees < 2; trees++)
      for (size_t o = 0; o < obj_rec.size(); o++) {
        if ((recs[obj_rec[o]].kind == REC_TREE) != (trees == 1)) continue;
        const size_t end = o + 1 < obj_rec.size() ? (size_t)obj_rec[o + 1] : recs.size();
        at[o] = (int32_t)ordered.size();
        if (trees) tree_rec.push_back(at[o]);
        ordered.insert(ordered.end(), recs.begin() + obj_rec[o], recs.begin() + end);
      }
    recs.swap(ordered);
    obj_rec.swap(at);
  }
  std::vector<Rec<float>> recs32(recs.size());
  for (size_t i = 0; i < recs.size(); i++) {
    recs32[i].kind = recs[i].kind;
    recs32[i].obj = recs[i].obj;
    recs32[i].op = recs[i].op;
    recs32[i].aux = recs[i].aux;
    for (int k = 0; k < 12; k++) recs32[i].p[k] = (float)recs[i].p[k];
  }
  std::vector<float> verts32(verts.begin(), verts.end());
  TablePack pack;
  decltype(sc->at) at{};
  at.recs32 = pack.add(recs32);
  at.recs64 = pack.add(recs);
  at.obj_n64 = pack.add(n64);
  at.obj_flags = pack.add(flags);
  at.obj_rec = pack.add(obj_rec);
  at.tree_rec = pack.add(tree_rec);
  at.verts32 = pack.add(verts32);
  at.verts64 = pack.add(verts);
  double reach = 0.0;
  const std::vector<Box2> boxes = object_boxes(recs, verts, obj_rec, sc->lights, &reach);
  std::vector<float4> box32(boxes.size());
  for (size_t o = 0; o < boxes.size(); o++) box32[o] = box_f32(boxes[o]);
  at.obj_box = pack.add(box32);
  float medium_map[4];
  at.medium = pack.add(medium_masks(box32, flags, medium_map));
  std::vector<Box2> walk_boxes;  // the blocks hold the objects of the walk
  std::vector<int32_t> walk_rec;
  for (size_t o = 0; o < obj_rec.size(); o++)
    if (recs[obj_rec[o]].kind != REC_TREE) {
      walk_boxes.push_back(boxes[o]);
      walk_rec.push_back(obj_rec[o]);
    }
  const CullLists cull = build_blocks(walk_boxes, walk_rec, recs);
  at.blocks = pack.add(cull.blocks);
  at.block_box = pack.add(cull.box);
  at.block_rec = pack.add(cull.rec);
  // lights
  if (sc->lights.size() > (size_t)kMaxLights) return fail(LG_E_UNSUPPORTED, "scene: too many lights");
  std::vector<DevLight> dl;
  uint64_t base = 0;
  for (size_t l = 0; l < sc->lights.size(); l++) {
    const lg_light& L = sc->lights[l];
    DevLight d;
    std::memset(&d, 0, sizeof(d));
    d.kind = L.kind;
    d.num_rays = L.num_rays;
    d.ray_base = base;
    base += L.num_rays;
    std::memcpy(d.color, L.color, sizeof(d.color));
    if (!finite_all(L.position, 2)) return fail(LG_E_INVALID, "light: non-finite position");
    d.a[0] = L.position[0];
    d.a[1] = L.position[1];
    if (L.kind == LG_LIGHT_SPOT) {
      double dx = L.direction[0], dy = L.direction[1];
      double ang = std::fabs(dx) < kEpsilon ? (dy >= 0.0 ? M_PI * 0.5 : -M_PI * 0.5) : std::atan(dy / dx);
      d.min_angle = ang - 0.5 * L.spot_angle;
      d.spot_angle = L.spot_angle;
      d.sign = std::signbit(dx) ? -1.0 : 1.0;
    } else if (L.kind == LG_LIGHT_DIRECTIONAL) {
      double ex = L.direction[0] - L.position[0], ey = L.direction[1] - L.position[1];
      double l = std::sqrt(ex * ex + ey * ey);
      if (!(l > 0)) return fail(LG_E_INVALID, "directional light: zero-length band");
      d.e[0] = ex;
      d.e[1] = ey;
      d.nrm[0] = -ey / l;
      d.nrm[1] = ex / l;
    } else if (L.kind != LG_LIGHT_POINT) {
      return fail(LG_E_INVALID, "light: unknown kind");
    }
    // starting refractive index: last object with a material containing the origin
    double ior = 1.0;
    for (size_t o = 0; o < sc->objects.size(); o++)
      if ((flags[o] & OBJ_MATERIAL) && contains_object<double>(recs.data(), verts.data(), obj_rec[o],
                                                               L.position[0], L.position[1]))
        ior = n64[o];
    d.ior = ior;
    dl.push_back(d);
  }
  if (base >= (1ull << (64 - kPathBits))) return fail(LG_E_UNSUPPORTED, "scene: too many rays");
  at.lights = pack.add(dl);
  int rc;
  if ((rc = sc->tables.ensure((pack.bytes.size() + 4095) & ~size_t(4095)))) return rc;
  if (!pack.bytes.empty())
    LG_HIP(hipMemcpyAsync(sc->tables.p, pack.bytes.data(), pack.bytes.size(), hipMemcpyHostToDevice, st));
  sc->at = at;
  sc->n_trees = (int)tree_rec.size();
  sc->n_blocks = (int)cull.blocks.size();
  sc->reach = reach;
  std::memcpy(sc->medium_map, medium_map, sizeof(medium_map));
  sc->n_primary = base;
  float lmax = 0.0f;
  bool nonneg = true;
  for (const lg_light& L : sc->lights)
    for (int c = 0; c < 4; c++) {
      lmax = std::max(lmax, std::fabs(L.color[c]));
      nonneg = nonneg && L.color[c] >= 0.0f;
    }
  sc->light_max = lmax;
  sc->light_nonneg = nonneg;
  sc->h_recs64 = recs;
  sc->h_obj_rec = obj_rec;
  sc->h_verts64 = verts;
  sc->n_recs = (int)recs.size();
  sc->n_objs = (int)sc->objects.size();
  sc->n_verts = (int)(verts.size() / 2);
  sc->dirty = false;
  return LG_OK;
}

void seg_forget(lg_segments* s) {
  s->count = 0;
  s->n_rays = 0;
  s->has_pos64 = false;
  s->one_color = true;
  s->max_abs = 0.0f;
  s->nonneg = true;
  s->hues = SceneHues{};
  s->runs = SegRuns{};
  s->extent[0] = s->extent[1] = 0.0;
}

int seg_ensure(lg_segments* s, uint64_t cap, bool need64) {
  int rc;
  if (cap > kMaxSegments) return fail(LG_E_OOM, "segments: at most 2^31 - 1 in one buffer");
  if (cap > s->cap || !s->pos.p) {
    seg_forget(s);
    s->cap = 0;  // (of the smallest of the buffers, should one of them fail)
    if ((rc = s->pos.ensure(cap * sizeof(float4)))) return rc;
    if ((rc = s->col0.ensure(cap * sizeof(float4)))) return rc;
    if ((rc = s->key.ensure(cap * sizeof(uint64_t)))) return rc;
    if (s->flags & LG_SEG_VERTEX_COLORS)
      if ((rc = s->col1.ensure(cap * sizeof(float4)))) return rc;
    s->cap = cap;
    s->pos64.reset();
  }
  if (need64 && s->pos64.bytes < cap * 4 * sizeof(double))
    if ((rc = s->pos64.ensure(s->cap * 4 * sizeof(double)))) return rc;
  return LG_OK;
}


AccumView make_view(const lg_view& v, int tile) {
  AccumView a;
  a.left = v.left;
  a.top = v.top;
  a.sx = (double)v.width / (v.right - v.left);
  a.sy = (double)v.height / (v.top - v.bottom);
  a.width = (int32_t)v.width;
  a.height = (int32_t)v.height;
  a.tile = tile;
  a.tile_shift = tile == 32 ? 5 : 6;
  a.tiles_x = (int32_t)((v.width + tile - 1) / tile);
  a.tiles_y = (int32_t)((v.height + tile - 1) / tile);
  return a;
}

int check_params(const lg_params* p) {
  if (!p) return fail(LG_E_INVALID, "params is NULL");
  if (p->max_bounce > kMaxBounce) return fail(LG_E_UNSUPPORTED, "max_bounce above 23");
  if (!finite_all(p->canvas, 4) || !(p->canvas[1] > p->canvas[0]) || !(p->canvas[3] > p->canvas[2]))
    return fail(LG_E_INVALID, "canvas must be {left < right, bottom < top}");
  return LG_OK;
}

}  // namespace lg

using namespace lg;

// =============================================================================================
// C ABI
// =============================================================================================
extern "C" {

const char* lg_last_error(void) { return g_error.c_str(); }

int lg_version(void) { return LG_ABI_VERSION; }

int lg_ctx_create(int device, lg_ctx** out) {
  if (!out) return fail(LG_E_INVALID, "lg_ctx_create: out is NULL");
  *out = nullptr;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return fail(LG_E_NODEVICE, "no HIP device");
  if (device < 0 || device >= n) return fail(LG_E_NODEVICE, "device ordinal out of range");
  LG_HIP(hipSetDevice(device));
  hipDeviceProp_t prop;
  LG_HIP(hipGetDeviceProperties(&prop, device));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return fail(LG_E_NODEVICE, std::string("device is ") + prop.gcnArchName + ", this build targets gfx950");
  lg_ctx* c = new lg_ctx();
  c->device = device;
  c->n_cu = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
  hipError_t e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
  if (e != hipSuccess) {
    delete c;
    return hip_fail(e, "hipStreamCreate");
  }
  // the static scratch of lg_accumulate_noalloc on this device (looked up once per device)
  int rc = noalloc_init(device, c->stream);
  if (rc) {
    (void)hipStreamDestroy(c->stream);
    delete c;
    return rc;
  }
  *out = c;
  return LG_OK;
}

static void ctx_free(lg_ctx* ctx) {
  (void)hipSetDevice(ctx->device);
  pipeline_destroy(ctx);
  (void)hipStreamSynchronize(ctx->stream);
  begin_call(ctx);
  for (hipEvent_t e : ctx->event_pool) (void)hipEventDestroy(e);
  (void)hipStreamDestroy(ctx->stream);
  delete ctx;
}

// A context outlives its children: destroying it while scenes, segment buffers or images
// are alive defers the release to the last child's destroy.
int lg_ctx_destroy(lg_ctx* ctx) {
  if (!ctx) return LG_OK;
  if (ctx->children > 0) {
    ctx->closing = true;
    return LG_OK;
  }
  ctx_free(ctx);
  return LG_OK;
}

}  // extern "C"

void lg::ctx_child_gone(lg_ctx* ctx) {
  if (--ctx->children == 0 && ctx->closing) ctx_free(ctx);
}

extern "C" {

int lg_ctx_synchronize(lg_ctx* ctx) {
  if (!ctx) return fail(LG_E_INVALID, "ctx is NULL");
  LG_HIP(hipStreamSynchronize(ctx->stream));
  return LG_OK;
}

int lg_ctx_set_profiling(lg_ctx* ctx, int enable) {
  if (!ctx) return fail(LG_E_INVALID, "ctx is NULL");
  ctx->profiling = enable != 0;
  return LG_OK;
}

int lg_ctx_stage_times(lg_ctx* ctx, lg_stage_time* out, int cap, int* n_out) {
  if (!ctx || !n_out) return fail(LG_E_INVALID, "ctx or n_out is NULL");
  *n_out = (int)ctx->last_times.size();
  if (cap < *n_out) return fail(LG_E_CAPACITY, "stage array too small");
  for (int i = 0; i < *n_out; i++) out[i] = ctx->last_times[i];
  return LG_OK;
}

// ---- scene ---------------------------------------------------------------------------------
int lg_scene_create(lg_ctx* ctx, lg_scene** out) {
  if (!ctx || !out) return fail(LG_E_INVALID, "ctx or out is NULL");
  lg_scene* s = new lg_scene();
  s->ctx = ctx;
  ctx->children++;
  *out = s;
  return LG_OK;
}

int lg_scene_destroy(lg_scene* scene) {
  if (!scene) return LG_OK;
  lg_ctx* ctx = scene->ctx;
  (void)hipSetDevice(ctx->device);
  (void)hipStreamSynchronize(ctx->stream);
  delete scene;
  ctx_child_gone(ctx);
  return LG_OK;
}

int lg_scene_clear(lg_scene* s) {
  if (!s) return fail(LG_E_INVALID, "scene is NULL");
  s->objects.clear();
  s->lights.clear();
  s->dirty = true;
  return LG_OK;
}

int lg_scene_clear_objects(lg_scene* s) {
  if (!s) return fail(LG_E_INVALID, "scene is NULL");
  s->objects.clear();
  s->dirty = true;
  return LG_OK;
}

int lg_scene_push_object(lg_scene* s, const lg_object* obj) {
  if (!s || !obj) return fail(LG_E_INVALID, "scene or object is NULL");
  s->objects.push_back(*obj);
  s->dirty = true;
  return LG_OK;
}

int lg_scene_push_light(lg_scene* s, const lg_light* light) {
  if (!s || !light) return fail(LG_E_INVALID, "scene or light is NULL");
  s->lights.push_back(*light);
  s->dirty = true;
  return LG_OK;
}

int lg_scene_set_objects(lg_scene* s, const lg_object* objs, uint32_t n) {
  if (!s || (n && !objs)) return fail(LG_E_INVALID, "scene or objects is NULL");
  s->objects.assign(objs, objs + n);
  s->dirty = true;
  return LG_OK;
}

int lg_scene_set_lights(lg_scene* s, const lg_light* lights, uint32_t n) {
  if (!s || (n && !lights)) return fail(LG_E_INVALID, "scene or lights is NULL");
  s->lights.assign(lights, lights + n);
  s->dirty = true;
  return LG_OK;
}

int lg_scene_replace_object(lg_scene* s, uint32_t ix, const lg_object* obj) {
  if (!s || !obj) return fail(LG_E_INVALID, "scene or object is NULL");
  if (ix >= s->objects.size()) return fail(LG_E_INVALID, "object index out of range");
  s->objects[ix] = *obj;
  s->dirty = true;
  return LG_OK;
}

int lg_scene_remove_object(lg_scene* s, uint32_t ix) {
  if (!s) return fail(LG_E_INVALID, "scene is NULL");
  if (ix >= s->objects.size()) return fail(LG_E_INVALID, "object index out of range");
  s->objects.erase(s->objects.begin() + ix);
  s->dirty = true;
  return LG_OK;
}

int lg_scene_remove_light(lg_scene* s, uint32_t ix) {
  if (!s) return fail(LG_E_INVALID, "scene is NULL");
  if (ix >= s->lights.size()) return fail(LG_E_INVALID, "light index out of range");
  s->lights.erase(s->lights.begin() + ix);
  s->dirty = true;
  return LG_OK;
}

int lg_scene_counts(const lg_scene* s, uint32_t* n_objects, uint32_t* n_lights, uint64_t* n_rays) {
  if (!s) return fail(LG_E_INVALID, "scene is NULL");
  if (n_objects) *n_objects = (uint32_t)s->objects.size();
  if (n_lights) *n_lights = (uint32_t)s->lights.size();
  if (n_rays) {
    uint64_t r = 0;
    for (auto& l : s->lights) r += l.num_rays;
    *n_rays = r;
  }
  return LG_OK;
}

// ---- segments ------------------------------------------------------------------------------
int lg_segments_create(lg_ctx* ctx, uint64_t capacity, uint32_t flags, lg_segments** out) {
  if (!ctx || !out) return fail(LG_E_INVALID, "ctx or out is NULL");
  lg_segments* s = new lg_segments();
  s->ctx = ctx;
  s->flags = flags;
  int rc = seg_ensure(s, std::max<uint64_t>(capacity, 1), false);
  if (rc) {
    delete s;
    return rc;
  }
  ctx->children++;
  *out = s;
  return LG_OK;
}

int lg_segments_destroy(lg_segments* s) {
  if (!s) return LG_OK;
  lg_ctx* ctx = s->ctx;
  (void)hipSetDevice(ctx->device);
  (void)hipStreamSynchronize(ctx->stream);
  delete s;
  ctx_child_gone(ctx);
  return LG_OK;
}

int lg_segments_count(const lg_segments* s, uint64_t* count) {
  if (!s || !count) return fail(LG_E_INVALID, "segments or count is NULL");
  *count = s->count;
  return LG_OK;
}

// The largest |value| and whether every value is >= 0, over the bits, in 32-bit integer
// operations that the compiler vectorises (with float comparisons, whose order NaN fixes, one value
// after another: 100003 segments took 150 us of an upload's 266). NaN, rare, goes value by value.
struct ColorBounds {
  uint32_t top = 0, sign = 0;  // the largest magnitude's bits; some value is below zero, or NaN
  float rest = 0.0f;
  void add(const float* v, uint64_t n) {
    uint32_t t = 0, neg = 0;
    for (uint64_t i = 0; i < n; i++) {
      uint32_t b;
      std::memcpy(&b, v + i, sizeof(b));
      const uint32_t m = b & 0x7fffffffu;
      t = t > m ? t : m;
      neg |= b > 0x80000000u ? 1u : 0u;  // (-0 is not below zero)
    }
    sign |= neg;
    if (t <= 0x7f800000u) {
      top = std::max(top, t);
      return;
    }
    sign = 1u;
    for (uint64_t i = 0; i < n; i++) rest = std::max(rest, std::fabs(v[i]));
  }
  float max_abs() const {
    float m;
    std::memcpy(&m, &top, sizeof(m));
    return std::max(m, rest);
  }
  bool nonneg() const { return sign == 0u; }
};

// The runs of n colours. A stretch that equals itself moved by one colour goes on with the run: one long
// comparison where a comparison per colour took 120 us of an upload of 100000 segments of a colour.
static void add_runs(SegRuns& runs, const float* c, uint64_t n) {
  constexpr uint64_t kStretch = 256;
  for (uint64_t i = 0; i < n;) {
    const uint64_t e = std::min(n, i + kStretch);
    if (i && std::memcmp(c + 4 * (i - 1), c + 4 * i, (e - i) * 16) == 0) {
      i = e;
      continue;
    }
    for (; i < e; i++)
      if (!runs.add(i, c + 4 * i)) return;
  }
}

int lg_segments_upload(lg_segments* s, const float* pos, const float* color0, const float* color1,
                       uint64_t n) {
  if (!s || (n && (!pos || !color0))) return fail(LG_E_INVALID, "segments, pos or color0 is NULL");
  if (color1 && !(s->flags & LG_SEG_VERTEX_COLORS))
    return fail(LG_E_INVALID, "color1 given but the buffer has no per-vertex colours");
  hipStream_t st = s->ctx->stream;
  int rc = seg_ensure(s, std::max<uint64_t>(n, 1), false);
  if (rc) return rc;
  seg_forget(s);
  // a color1 equal to color0 bit for bit is no per-vertex colour: the accumulation then takes
  // the one-colour walk, which deposits the same bits
  const bool one_color = !color1 || !n || std::memcmp(color0, color1, n * 16) == 0;
  ColorBounds b;
  SegRuns runs;
  if (n) {
    LG_HIP(hipMemcpyAsync(s->pos.p, pos, n * 16, hipMemcpyHostToDevice, st));
    LG_HIP(hipMemcpyAsync(s->col0.p, color0, n * 16, hipMemcpyHostToDevice, st));
    if (!one_color) LG_HIP(hipMemcpyAsync(s->col1.p, color1, n * 16, hipMemcpyHostToDevice, st));
    LG_HIP(launch_iota_u64(s->key.as<uint64_t>(), n, st));
    b.add(color0, 4 * n);
    if (color1) b.add(color1, 4 * n);
    if (one_color) add_runs(runs, color0, n);
    LG_HIP(hipStreamSynchronize(st));
  }
  s->count = n;
  s->one_color = one_color;
  s->max_abs = b.max_abs();
  s->nonneg = b.nonneg();
  s->runs = runs;
  if (runs.n) {
    float4 samples[kExtentSamples];
    for (int k = 0; k < kExtentSamples; k++) std::memcpy(&samples[k], pos + 4 * extent_sample(k, n), sizeof(float4));
    set_extent(*s, samples);
  }
  return LG_OK;
}

int lg_segments_download(lg_segments* s, float* pos, float* color0, float* color1, uint64_t* key,
                         uint64_t cap, uint64_t* count) {
  if (!s) return fail(LG_E_INVALID, "segments is NULL");
  if (count) *count = s->count;
  if (cap < s->count) return fail(LG_E_CAPACITY, "download: capacity below segment count");
  hipStream_t st = s->ctx->stream;
  uint64_t n = s->count;
  if (n) {
    if (pos) LG_HIP(hipMemcpyAsync(pos, s->pos.p, n * 16, hipMemcpyDeviceToHost, st));
    if (color0) LG_HIP(hipMemcpyAsync(color0, s->col0.p, n * 16, hipMemcpyDeviceToHost, st));
    if (color1)
      LG_HIP(hipMemcpyAsync(color1, s->one_color ? s->col0.p : s->col1.p, n * 16,
                            hipMemcpyDeviceToHost, st));
    if (key) LG_HIP(hipMemcpyAsync(key, s->key.p, n * 8, hipMemcpyDeviceToHost, st));
  }
  LG_HIP(hipStreamSynchronize(st));
  return LG_OK;
}

int lg_segments_download_pos64(lg_segments* s, double* pos64, uint64_t cap, uint64_t* count) {
  if (!s || !pos64) return fail(LG_E_INVALID, "segments or pos64 is NULL");
  if (count) *count = s->count;
  if (!s->has_pos64) return fail(LG_E_INVALID, "no FP64 end points: trace with LG_TRACE_FP64");
  if (cap < s->count) return fail(LG_E_CAPACITY, "download: capacity below segment count");
  if (s->count)
    LG_HIP(hipMemcpyAsync(pos64, s->pos64.p, s->count * 32, hipMemcpyDeviceToHost, s->ctx->stream));
  LG_HIP(hipStreamSynchronize(s->ctx->stream));
  return LG_OK;
}

// ---- trace ---------------------------------------------------------------------------------
int lg_trace(lg_scene* scene, const lg_params* params, lg_segments* out) {
  if (!scene || !out) return fail(LG_E_INVALID, "scene or out is NULL");
  int rc = check_params(params);
  if (rc) return rc;
  lg_ctx* ctx = scene->ctx;
  LG_HIP(hipSetDevice(ctx->device));
  begin_call(ctx);
  Entry e;
  e.scene = scene;
  e.params = *params;
  e.segs = out;
  if ((rc = pipeline_run(ctx, {e}, ST_TRACE))) return rc;
  end_call(ctx);
  return LG_OK;
}

int lg_trace_all(lg_scene* scene, const lg_params* params, double* xy, float* rgba,
                 uint64_t cap_vertices, uint64_t* n_vertices) {
  if (!scene || !n_vertices) return fail(LG_E_INVALID, "scene or n_vertices is NULL");
  lg_segments* segs = nullptr;
  int rc = lg_segments_create(scene->ctx, 1024, 0, &segs);
  if (rc) return rc;
  rc = lg_trace(scene, params, segs);
  if (rc) {
    lg_segments_destroy(segs);
    return rc;
  }
  rc = lg_segments_download_vertices(segs, xy, rgba, cap_vertices, n_vertices);
  lg_segments_destroy(segs);
  return rc;
}

// ---- image ---------------------------------------------------------------------------------
int lg_image_create(lg_ctx* ctx, const lg_view* view, lg_image** out) {
  if (!ctx || !view || !out) return fail(LG_E_INVALID, "ctx, view or out is NULL");
  if (view->width == 0 || view->height == 0 || view->width > 8192 || view->height > 8192)
    return fail(LG_E_INVALID, "image size must be 1..8192");
  double b[4] = {view->left, view->right, view->bottom, view->top};
  if (!finite_all(b, 4) || !(view->right > view->left) || !(view->top > view->bottom))
    return fail(LG_E_INVALID, "view must be {left < right, bottom < top}");
  lg_image* im = new lg_image();
  im->ctx = ctx;
  im->view = *view;
  size_t px = (size_t)view->width * view->height;
  int rc = im->accum.ensure(px * 16);
  if (!rc) rc = im->out16.ensure(px * 8);
  if (rc) {
    delete im;
    return rc;
  }
  ctx->children++;
  *out = im;
  return lg_image_clear(im);
}

int lg_image_destroy(lg_image* img) {
  if (!img) return LG_OK;
  lg_ctx* ctx = img->ctx;
  (void)hipSetDevice(ctx->device);
  (void)hipStreamSynchronize(ctx->stream);
  delete img;
  ctx_child_gone(ctx);
  return LG_OK;
}

// Clears (mode 0) or resolves (1) an image.
static int image_pass(lg_ctx* ctx, lg_image* img, int mode) {
  begin_call(ctx);
  const uint64_t n = (uint64_t)img->view.width * img->view.height;
  {
    StageScope s(ctx, mode ? "resolve" : "clear", n);
    LG_HIP(launch_pixels(mode, img->accum.as<float4>(), img->out16.as<ushort4>(), n, ctx->stream));
  }
  LG_HIP(hipStreamSynchronize(ctx->stream));
  end_call(ctx);
  return LG_OK;
}

int lg_image_clear(lg_image* img) {
  if (!img) return fail(LG_E_INVALID, "image is NULL");
  lg_ctx* ctx = img->ctx;
  LG_HIP(hipSetDevice(ctx->device));
  return image_pass(ctx, img, 0);
}

int lg_image_device_ptrs(lg_image* img, void** accum, void** rgba16f) {
  if (!img) return fail(LG_E_INVALID, "image is NULL");
  if (accum) *accum = img->accum.p;
  if (rgba16f) *rgba16f = img->out16.p;
  return LG_OK;
}

int lg_image_download_rgba16f(lg_image* img, uint16_t* host, uint64_t cap_halves) {
  if (!img || !host) return fail(LG_E_INVALID, "image or host is NULL");
  size_t n = (size_t)img->view.width * img->view.height * 4;
  if (cap_halves < n) return fail(LG_E_CAPACITY, "download: capacity below 4*W*H");
  LG_HIP(hipMemcpyAsync(host, img->out16.p, n * 2, hipMemcpyDeviceToHost, img->ctx->stream));
  LG_HIP(hipStreamSynchronize(img->ctx->stream));
  return LG_OK;
}

int lg_image_download_accum(lg_image* img, float* host, uint64_t cap_floats) {
  if (!img || !host) return fail(LG_E_INVALID, "image or host is NULL");
  size_t n = (size_t)img->view.width * img->view.height * 4;
  if (cap_floats < n) return fail(LG_E_CAPACITY, "download: capacity below 4*W*H");
  LG_HIP(hipMemcpyAsync(host, img->accum.p, n * 4, hipMemcpyDeviceToHost, img->ctx->stream));
  LG_HIP(hipStreamSynchronize(img->ctx->stream));
  return LG_OK;
}

// ---- accumulate / resolve / render --------------------------------------------------------------
int lg_accumulate(lg_ctx* ctx, const lg_segments* segs, lg_image* img) {
  if (!ctx || !segs || !img) return fail(LG_E_INVALID, "ctx, segments or image is NULL");
  LG_HIP(hipSetDevice(ctx->device));
  begin_call(ctx);
  if (segs->count == 0) return LG_OK;
  if (segs->count > 0xffffffffull) return fail(LG_E_UNSUPPORTED, "accumulate: more than 2^32 segments");
  Entry e;
  e.segs = const_cast<lg_segments*>(segs);
  e.img = img;
  int rc = pipeline_run(ctx, {e}, ST_ACCUM);
  if (rc) return rc;
  end_call(ctx);
  return LG_OK;
}

int lg_resolve(lg_ctx* ctx, lg_image* img) {
  if (!ctx || !img) return fail(LG_E_INVALID, "ctx or image is NULL");
  LG_HIP(hipSetDevice(ctx->device));
  if (img->ctx != ctx) return fail(LG_E_INVALID, "resolve: image of another context");
  return image_pass(ctx, img, 1);
}

int lg_render(lg_scene* scene, const lg_params* params, lg_segments* segs, lg_image* img) {
  if (!scene || !segs || !img) return fail(LG_E_INVALID, "scene, segments or image is NULL");
  return lg_batch_render(scene->ctx, 1, &scene, params, &segs, &img);
}

int lg_batch_render(lg_ctx* ctx, uint32_t n, lg_scene* const* scenes, const lg_params* params,
                    lg_segments* const* segs, lg_image* const* images) {
  if (!ctx) return fail(LG_E_INVALID, "ctx is NULL");
  if (n && (!scenes || !params || !segs || !images)) return fail(LG_E_INVALID, "batch arrays are NULL");
  LG_HIP(hipSetDevice(ctx->device));
  begin_call(ctx);
  std::vector<Entry> E(n);
  for (uint32_t i = 0; i < n; i++) {
    if (!scenes[i] || !segs[i] || !images[i]) return fail(LG_E_INVALID, "batch entry is NULL");
    int rc = check_params(&params[i]);
    if (rc) return rc;
    E[i].scene = scenes[i];
    E[i].params = params[i];
    E[i].segs = segs[i];
    E[i].img = images[i];
  }
  int rc = pipeline_run(ctx, E, ST_TRACE | ST_ACCUM | ST_FRESH);
  if (rc) return rc;
  end_call(ctx);
  return LG_OK;
}

int lg_ctx_set_graphs(lg_ctx* ctx, int enable) {
  if (!ctx) return fail(LG_E_INVALID, "ctx is NULL");
  ctx->use_graphs = enable != 0;
  return LG_OK;
}

int lg_ctx_set_packed_accumulation(lg_ctx* ctx, int enable) {
  if (!ctx) return fail(LG_E_INVALID, "ctx is NULL");
  ctx->packed_accum = enable != 0;
  return LG_OK;
}

int lg_calibrate_lds_atomics(lg_ctx* ctx, double* rate) {
  if (!ctx || !rate) return fail(LG_E_INVALID, "ctx or rate is NULL");
  LG_HIP(hipSetDevice(ctx->device));
  DevBuf sink;
  int rc;
  if ((rc = sink.ensure((size_t)2 * ctx->n_cu * sizeof(unsigned long long)))) return rc;
  hipEvent_t a = nullptr, b = nullptr;
  LG_HIP(hipEventCreate(&a));
  if (hipEventCreate(&b) != hipSuccess) {
    (void)hipEventDestroy(a);
    return fail(LG_E_HIP, "hipEventCreate");
  }
  double best = 0.0;
  hipError_t e = hipSuccess;
  for (int run = 0; run < 4 && e == hipSuccess; run++) {  // the first run warms up
    uint64_t n = 0;
    e = hipEventRecord(a, ctx->stream);
    if (e == hipSuccess) e = launch_lds_atomic_rate(ctx->n_cu, 1u << 14, sink.as<unsigned long long>(), ctx->stream, &n);
    if (e == hipSuccess) e = hipEventRecord(b, ctx->stream);
    if (e == hipSuccess) e = hipEventSynchronize(b);
    float ms = 0.0f;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, a, b);
    if (e == hipSuccess && run > 0 && ms > 0.0f) best = std::max(best, (double)n / (ms * 1e-3));
  }
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  if (e != hipSuccess) return hip_fail(e, "lds atomic rate probe");
  *rate = best;
  return LG_OK;
}

int lg_ctx_get_tuning(const lg_ctx* ctx, lg_tuning* out) {
  if (!ctx || !out) return fail(LG_E_INVALID, "ctx or out is NULL");
  *out = ctx->tune;
  return LG_OK;
}

int lg_ctx_set_tuning(lg_ctx* ctx, const lg_tuning* t) {
  if (!ctx || !t) return fail(LG_E_INVALID, "ctx or tuning is NULL");
  if (t->rays_per_item < 64 || t->rays_per_item > (1u << 20))
    return fail(LG_E_INVALID, "rays_per_item must be in [64, 2^20]");
  if (t->min_piece < 64 || t->max_piece < t->min_piece)
    return fail(LG_E_INVALID, "tile pieces need 64 <= min_piece <= max_piece");
  if (t->trace_waves < 1 || t->trace_waves > 16) return fail(LG_E_INVALID, "trace_waves must be in [1, 16]");
  if (!tile_size_supported((int)t->tile)) return fail(LG_E_INVALID, "tile must be 32 or 64");
  if (t->trace_chunk < 1 || t->trace_chunk > trace_max_chunk()) return fail(LG_E_INVALID, "trace_chunk must be in [1, 3]");
  if (t->tile_block != 512 && t->tile_block != 1024) return fail(LG_E_INVALID, "tile_block must be 512 or 1024");
  ctx->tune = *t;
  return LG_OK;
}

}  // extern "C"
