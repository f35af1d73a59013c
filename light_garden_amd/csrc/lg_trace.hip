// lg_trace.hip — the per-ray trace on gfx950.
//
// Replaces Tracer::trace_all / Tracer::trace (src/light_garden/tracer.rs:276-330,
// 360-493) and the collision2d ray/shape arithmetic it calls. The reference walks each
// primary ray's bounce tree breadth-first on a rayon worker; here one kernel launch is one
// to three generations of ALL rays: each lane owns one live ray and culls the scene's objects
// by their boxes, read as wave-uniform scalars, to a bit mask; the candidates are then tested
// lane by lane (scenes of few objects test every record, wave-uniformly). A lane shades its
// nearest hit, and appends its segment and surviving children with one global
// atomic per workgroup (wave64 ballot + mbcnt prefix, then a cross-wave LDS prefix).
// Children that the cutoff (tracer.rs:378-384) would skip are never queued, which is the
// same as queueing and skipping them.
//
// Precision: T = float is the bulk path. The steps whose branch decides the ray tree are
// redone in FP64 when FP32 cannot decide them: the circle/ellipse discriminant near
// tangency, the Bezier sign tests near a double root or an end point, and the Snell
// critical-angle (total internal reflection) test. T = double runs the whole trace in
// FP64.
#include <float.h>

#include "lg_internal.h"

namespace lg {

template <typename T>
struct RayT {
  T ox, oy, dx, dy;
};

template <typename T>
__device__ __forceinline__ T tmin_v() {
  return (T)kTMin;
}
template <typename T>
__device__ __forceinline__ T inf_v() {
  return (T)INFINITY;
}
template <typename T>
__device__ __forceinline__ T sqrt_v(T x) {
  if constexpr (sizeof(T) == 4)
    return __builtin_sqrtf(x);
  else
    return __builtin_sqrt(x);
}
template <typename T>
__device__ __forceinline__ T abs_v(T x) {
  if constexpr (sizeof(T) == 4)
    return __builtin_fabsf(x);
  else
    return __builtin_fabs(x);
}
template <typename T>
__device__ __forceinline__ T rcp_v(T x) {
  if constexpr (sizeof(T) == 4)
    return __builtin_amdgcn_rcpf(x);
  else
    return (T)1 / x;
}
template <typename T>
__device__ __forceinline__ void normalize_v(T& x, T& y) {
  T l2 = x * x + y * y;
  if (l2 > (T)0) {
    if constexpr (sizeof(T) == 4) {
      T r = __builtin_amdgcn_rsqf(l2);
      x *= r;
      y *= r;
    } else {
      T l = sqrt_v(l2);
      x /= l;
      y /= l;
    }
  }
}

// The FP32 culling pass over every object reads its records with wave-uniform indices (the object
// loop is the same for every lane). Read through the constant address space from the scene's
// device buffers, those loads become scalar loads: a record's fields arrive in SGPRs and feed
// the vector ALU directly, instead of taking VGPRs after an LDS read, and the scalar data
// cache holds a scene's records (64 B each) for every wave of the compute unit. The pass by boxes
// reads the boxes so, and the records of its candidates, each lane its own, as four 16-byte vector
// loads (they hit the L1).
#define LG_K __attribute__((address_space(4)))
typedef int lg_v4i __attribute__((ext_vector_type(4)));
template <typename P>
struct RecAt {
  P p;  // four lg_v4i per record
  __device__ __forceinline__ Rec<float> operator[](int i) const {
    struct V {
      lg_v4i a, b, c, d;
    };
    const V v{p[4 * i], p[4 * i + 1], p[4 * i + 2], p[4 * i + 3]};
    return __builtin_bit_cast(Rec<float>, v);
  }
};
using RecK = RecAt<const LG_K lg_v4i*>;  // the same record for every lane
using RecV = RecAt<const lg_v4i*>;       // a record per lane

// One field of a record at an index known only at run time: read from the source itself, since
// indexing into a copy of the whole record would put the copy on the stack.
template <typename T>
__device__ __forceinline__ T rec_param(const Rec<T>* recs, int i, int m) {
  return recs[i].p[m];
}
__device__ __forceinline__ float rec_param(const RecK& recs, int i, int m) {
  return reinterpret_cast<const LG_K float*>(recs.p + 4 * i)[offsetof(Rec<float>, p) / 4 + m];
}

// FP32 -> FP64 step threshold: a branch quantity q is recomputed in FP64 when
// |q| < kIsland * (magnitude of the terms it was computed from).
constexpr float kIsland = 1.0e-5f;

// ---------------------------------------------------------------------------------------
// chords of closed convex primitives: the parameter interval [tin, tout] the full line
// o + t d spends inside (tin may be negative). Returns false when the line misses.
// ---------------------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ bool chord_circle(const RayT<T>& r, const T* p, const Rec<double>* r64, T& tin,
                             T& tout) {
  T lx = r.ox - p[0], ly = r.oy - p[1];
  T b = lx * r.dx + ly * r.dy;
  T ll = lx * lx + ly * ly;
  T cc = ll - p[3];
  T disc = b * b - cc;
  if constexpr (sizeof(T) == 4) {
    if (__builtin_fabsf(disc) < kIsland * (b * b + ll + p[3])) {
      RayT<double> rd{(double)r.ox, (double)r.oy, (double)r.dx, (double)r.dy};
      double ti, to;
      bool ok = chord_circle<double>(rd, r64->p, nullptr, ti, to);
      tin = (float)ti;
      tout = (float)to;
      return ok;
    }
  }
  if (disc < (T)0) return false;
  T sq = sqrt_v(disc);
  T q = b > (T)0 ? -b - sq : -b + sq;
  if (q == (T)0) {
    tin = tout = (T)0;
    return true;
  }
  T ra = q, rb = cc / q;
  tin = ra < rb ? ra : rb;
  tout = ra < rb ? rb : ra;
  return true;
}

// Local coordinates of the ray in a frame {c, u, v} (p[0..5]).
template <typename T>
__device__ __forceinline__ void to_local(const RayT<T>& r, const T* p, T& ox, T& oy, T& dx,
                                         T& dy) {
  T lx = r.ox - p[0], ly = r.oy - p[1];
  ox = lx * p[2] + ly * p[3];
  oy = lx * p[4] + ly * p[5];
  dx = r.dx * p[2] + r.dy * p[3];
  dy = r.dx * p[4] + r.dy * p[5];
}

// Rect faces: 0 bottom (0,-1), 1 right (1,0), 2 top (0,1), 3 left (-1,0).
template <typename T>
__device__ __forceinline__ bool chord_rect(const RayT<T>& r, const T* p, T& tin, T& tout, int& fin, int& fout) {
  T ox, oy, dx, dy;
  to_local(r, p, ox, oy, dx, dy);
  T hw = p[6], hh = p[7];
  T t0 = -inf_v<T>(), t1 = inf_v<T>();
  int f0 = -1, f1 = -1;
  if (dx != (T)0) {
    T inv = rcp_v(dx);
    T ta = (-hw - ox) * inv, tb = (hw - ox) * inv;
    if (ta < tb) {
      t0 = ta; f0 = 3; t1 = tb; f1 = 1;
    } else {
      t0 = tb; f0 = 1; t1 = ta; f1 = 3;
    }
  } else if (ox < -hw || ox > hw) {
    return false;
  }
  if (dy != (T)0) {
    T inv = rcp_v(dy);
    T ta = (-hh - oy) * inv, tb = (hh - oy) * inv;
    T lo = ta < tb ? ta : tb, hi = ta < tb ? tb : ta;
    int flo = ta < tb ? 0 : 2, fhi = ta < tb ? 2 : 0;
    if (lo > t0) { t0 = lo; f0 = flo; }
    if (hi < t1) { t1 = hi; f1 = fhi; }
  } else if (oy < -hh || oy > hh) {
    return false;
  }
  if (!(t0 <= t1)) return false;
  tin = t0; tout = t1; fin = f0; fout = f1;
  return true;
}

template <typename T>
__device__ __forceinline__ bool chord_ellipse(const RayT<T>& r, const T* p, const Rec<double>* r64, T& tin,
                              T& tout) {
  T ox, oy, dx, dy;
  to_local(r, p, ox, oy, dx, dy);
  T ia = (T)1 / p[6], ib = (T)1 / p[7];
  T osx = ox * ia, osy = oy * ib, dsx = dx * ia, dsy = dy * ib;
  T A = dsx * dsx + dsy * dsy, B = osx * dsx + osy * dsy, C = osx * osx + osy * osy - (T)1;
  T disc = B * B - A * C;
  if constexpr (sizeof(T) == 4) {
    if (__builtin_fabsf(disc) < kIsland * (B * B + __builtin_fabsf(A * C) + A)) {
      RayT<double> rd{(double)r.ox, (double)r.oy, (double)r.dx, (double)r.dy};
      double ti, to;
      bool ok = chord_ellipse<double>(rd, r64->p, nullptr, ti, to);
      tin = (float)ti;
      tout = (float)to;
      return ok;
    }
  }
  if (disc < (T)0 || A == (T)0) return false;
  T sq = sqrt_v(disc);
  T q = B > (T)0 ? -B - sq : -B + sq;
  if (q == (T)0) {
    tin = tout = (T)0;
    return true;
  }
  T ra = q / A, rb = C / q;
  tin = ra < rb ? ra : rb;
  tout = ra < rb ? rb : ra;
  return true;
}

// Convex polygon (counter-clockwise local vertices), Cyrus-Beck clipping of the line.
template <typename T>
__device__ __forceinline__ bool chord_poly(const RayT<T>& r, const T* p, const T* verts, int first, int nv,
                           T& tin, T& tout, int& ein, int& eout) {
  T ox, oy, dx, dy;
  to_local(r, p, ox, oy, dx, dy);
  T t0 = -inf_v<T>(), t1 = inf_v<T>();
  int e0 = -1, e1 = -1;
  for (int i = 0; i < nv; i++) {
    int j = (i + 1 == nv) ? 0 : i + 1;
    T ax = verts[2 * (first + i)], ay = verts[2 * (first + i) + 1];
    T bx = verts[2 * (first + j)], by = verts[2 * (first + j) + 1];
    T nx = by - ay, ny = -(bx - ax);  // outward for CCW
    T num = nx * (ax - ox) + ny * (ay - oy);
    T den = nx * dx + ny * dy;
    if (den == (T)0) {
      if (num < (T)0) return false;
      continue;
    }
    T t = num / den;
    if (den < (T)0) {
      if (t > t0) { t0 = t; e0 = i; }
    } else {
      if (t < t1) { t1 = t; e1 = i; }
    }
  }
  if (!(t0 <= t1)) return false;
  tin = t0; tout = t1; ein = e0; eout = e1;
  return true;
}

// ---------------------------------------------------------------------------------------
// open primitives
// ---------------------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ bool hit_segment(const RayT<T>& r, const T* p, T& t_out) {
  T ex = p[2], ey = p[3];
  T den = r.dx * ey - r.dy * ex;
  if (den == (T)0) return false;
  T wx = p[0] - r.ox, wy = p[1] - r.oy;
  T inv = rcp_v(den);
  T t = (wx * ey - wy * ex) * inv;
  T s = (wx * r.dy - wy * r.dx) * inv;
  if (!(t > tmin_v<T>()) || s < (T)0 || s > (T)1) return false;
  t_out = t;
  return true;
}

template <typename T>
__device__ __forceinline__ T horner3(T A, T B, T C, T D, T s) {
  return ((A * s + B) * s + C) * s + D;
}

// Nearest hit (smallest t > kTMin) of the ray with the cubic Bezier given in power basis
// a = {a3x a3y a2x a2y a1x a1y a0x a0y}. [0,1] is split at the roots of the derivative of
// f(s) = n . (B(s) - o) into monotone pieces and each piece with a sign change is
// bisected (the oracle's rule). Returns false on a miss; sets `ambiguous` (FP32 only)
// when a sign test at a piece end is too close to zero to trust.
// Whether the ray (t > T_MIN) can meet the padded box b = {x0, y0, x1, y1} (slab test).
template <typename T>
__device__ __forceinline__ bool ray_meets_box(const RayT<T>& r, const T* b) {
  T lo = tmin_v<T>(), hi = inf_v<T>();
  if (r.dx == (T)0) {
    if (r.ox < b[0] || r.ox > b[2]) return false;
  } else {
    const T inv = (T)1 / r.dx;
    T t0 = (b[0] - r.ox) * inv, t1 = (b[2] - r.ox) * inv;
    if (t0 > t1) {
      const T u = t0;
      t0 = t1;
      t1 = u;
    }
    lo = t0 > lo ? t0 : lo;
    hi = t1 < hi ? t1 : hi;
  }
  if (r.dy == (T)0) {
    if (r.oy < b[1] || r.oy > b[3]) return false;
  } else {
    const T inv = (T)1 / r.dy;
    T t0 = (b[1] - r.oy) * inv, t1 = (b[3] - r.oy) * inv;
    if (t0 > t1) {
      const T u = t0;
      t0 = t1;
      t1 = u;
    }
    lo = t0 > lo ? t0 : lo;
    hi = t1 < hi ? t1 : hi;
  }
  return lo <= hi;
}

template <typename T>
__device__ __forceinline__ bool bezier_nearest(const RayT<T>& r, const T* a, T& t_best, T& s_best,
                               bool& ambiguous) {
  T nx = -r.dy, ny = r.dx;
  T A = nx * a[0] + ny * a[1];
  T B = nx * a[2] + ny * a[3];
  T C = nx * a[4] + ny * a[5];
  T D = nx * (a[6] - r.ox) + ny * (a[7] - r.oy);
  T knots[4];
  int nk = 0;
  knots[nk++] = (T)0;
  T qa = (T)3 * A, qb = (T)2 * B, qc = C;
  T crit[2];
  int nc = 0;
  if (qa == (T)0) {
    if (qb != (T)0) crit[nc++] = -qc / qb;
  } else {
    T disc = qb * qb - (T)4 * qa * qc;
    if (disc >= (T)0) {
      T sq = sqrt_v(disc);
      T q = (T)(-0.5) * (qb + (qb >= (T)0 ? sq : -sq));
      if (q != (T)0) {
        crit[nc++] = q / qa;
        crit[nc++] = qc / q;
      } else {
        crit[nc++] = (T)0;
      }
    }
  }
  if (nc == 2 && crit[0] > crit[1]) {
    T tmp = crit[0];
    crit[0] = crit[1];
    crit[1] = tmp;
  }
  knots[1] = knots[2] = knots[3] = (T)1;
  if (nc >= 1 && crit[0] > (T)0 && crit[0] < (T)1) {
    knots[1] = crit[0];
    nk = 2;
  }
  if (nc == 2 && crit[1] > (T)0 && crit[1] < (T)1 && crit[1] != (nk == 2 ? knots[1] : knots[0])) {
    if (nk == 2) knots[2] = crit[1]; else knots[1] = crit[1];
    nk++;
  }
  nk++;  // the end knot s = 1 (already stored)
  T fk[4];
  T scale = abs_v(A) + abs_v(B) + abs_v(C) + abs_v(D);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if (i >= nk) break;
    fk[i] = horner3(A, B, C, D, knots[i]);
    if constexpr (sizeof(T) == 4) {
      if (__builtin_fabsf(fk[i]) < kIsland * scale) ambiguous = true;
    }
  }
  if constexpr (sizeof(T) == 4) {
    if (ambiguous) return false;
  }
  bool found = false;
  t_best = inf_v<T>();
  constexpr int kMaxIt = sizeof(T) == 4 ? 48 : 200;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    if (i + 1 >= nk) break;
    T l = knots[i], rr = knots[i + 1];
    T fl = fk[i], fr = fk[i + 1];
    T root;
    if (fl == (T)0) {
      root = l;
    } else {
      if (fr == (T)0) continue;
      if ((fl < (T)0) == (fr < (T)0)) continue;
      // safeguarded Newton on the bracket [lo, hi] (f(lo), f(hi) of opposite signs): a Newton
      // step that leaves the bracket is replaced by its midpoint, so it converges like
      // bisection in the worst case and quadratically near a simple root
      T lo = l, hi = rr, flo = fl;
      T x = (T)0.5 * (lo + hi);
      for (int it = 0; it < kMaxIt; it++) {
        const T fm = horner3(A, B, C, D, x);
        if (fm == (T)0) {
          lo = hi = x;
          break;
        }
        if ((fm < (T)0) == (flo < (T)0)) {
          lo = x;
          flo = fm;
        } else {
          hi = x;
        }
        const T dfm = ((T)3 * A * x + (T)2 * B) * x + C;
        T xn = x - fm / dfm;
        // converged: the step no longer moves x (tested before the safeguard, which would
        // otherwise replace the converged x, now an end of the bracket, by the midpoint)
        if (xn == x) break;
        if (!(xn > lo && xn < hi)) xn = (T)0.5 * (lo + hi);
        if (xn <= lo || xn >= hi) break;  // the bracket cannot shrink further
        x = xn;
      }
      root = lo == hi ? lo : x;
    }
    T px = ((a[0] * root + a[2]) * root + a[4]) * root + a[6];
    T py = ((a[1] * root + a[3]) * root + a[5]) * root + a[7];
    T t = (px - r.ox) * r.dx + (py - r.oy) * r.dy;
    if (t > tmin_v<T>() && t < t_best) {
      t_best = t;
      s_best = root;
      found = true;
    }
  }
  T f_last = nk == 2 ? fk[1] : (nk == 3 ? fk[2] : fk[3]);
  if (f_last == (T)0) {
    T px = a[0] + a[2] + a[4] + a[6], py = a[1] + a[3] + a[5] + a[7];
    T t = (px - r.ox) * r.dx + (py - r.oy) * r.dy;
    if (t > tmin_v<T>() && t < t_best) {
      t_best = t;
      s_best = (T)1;
      found = true;
    }
  }
  return found;
}

// ---------------------------------------------------------------------------------------
// Chord of any closed primitive record (used for top-level shapes and Logic operands).
// aux_in / aux_out: face or edge index of the chord ends (rect/polygon).
// ---------------------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ bool chord_any(const RayT<T>& r, int kind, const Rec<T>& R,
                                          const Rec<double>* R64, const T* verts, T& tin,
                                          T& tout, int& ain, int& aout) {
  ain = aout = 0;
  switch (kind) {
    case REC_CIRCLE: return chord_circle(r, R.p, R64, tin, tout);
    case REC_RECT: return chord_rect(r, R.p, tin, tout, ain, aout);
    case REC_ELLIPSE: return chord_ellipse(r, R.p, R64, tin, tout);
    case REC_POLY: return chord_poly(r, R.p, verts, R.aux, R.op, tin, tout, ain, aout);
    default: return false;
  }
}

// Nearest-hit state. code: bit0 = chord exit (else entry), bit1 = flip the normal,
// bits 8.. = face/edge index. `rec` is the record whose surface was hit (a Logic operand
// for boolean objects), `top` the object's first record. The runner-up from another
// object (t2, top2) lets the FP32 pass hand near-ties to FP64.
template <typename T>
struct Nearest {
  T t;
  T s;        // Bezier parameter
  int rec;
  int top;
  int code;
  T t2;
  int top2;
};

template <typename T>
__device__ __forceinline__ void nearest_init(Nearest<T>& nb) {
  nb.t = inf_v<T>();
  nb.s = (T)0;
  nb.rec = -1;
  nb.top = -1;
  nb.code = 0;
  nb.t2 = inf_v<T>();
  nb.top2 = -1;
}

// The first minimum in object order (tracer.rs:404,417): a smaller t wins, and an equal t
// from an object earlier in the scene. With objects offered in scene order this is the strict
// <; with the hierarchy's order it gives the same winner, and t2 is the smallest t of the
// other objects either way.
template <typename T>
__device__ __forceinline__ void consider(Nearest<T>& nb, T t, int rec, int code, T s, int top) {
  if (!(t > tmin_v<T>())) return;
  if (t < nb.t || (t == nb.t && top < nb.top)) {
    if (top != nb.top) {
      nb.t2 = nb.t;
      nb.top2 = nb.top;
    }
    nb.t = t;
    nb.rec = rec;
    nb.top = top;
    nb.code = code;
    nb.s = s;
  } else if (t < nb.t2 && top != nb.top) {
    nb.t2 = t;
    nb.top2 = top;
  }
}

// `consider` for a Logic tree of more than two primitives. Such trees' records follow every
// other object's, so on an exact tie in t the scene order of the objects decides: `first` says
// that the tree's object comes before the current winner's.
template <typename T>
__device__ __forceinline__ void consider_tree(Nearest<T>& nb, T t, int rec, int code, int top, bool first) {
  if (!(t > tmin_v<T>())) return;
  if (t < nb.t || (t == nb.t && first)) {
    if (top != nb.top) {
      nb.t2 = nb.t;
      nb.top2 = nb.top;
    }
    nb.t = t;
    nb.rec = rec;
    nb.top = top;
    nb.code = code;
    nb.s = (T)0;
  } else if (t < nb.t2 && top != nb.top) {
    nb.t2 = t;
    nb.top2 = top;
  }
}

// Boolean combination of two chords (closed convex operands). Candidate boundary points
// are offered to `consider` in a-then-b order.
template <typename T>
__device__ __forceinline__ void logic_candidates(Nearest<T>& nb, int op, bool hitA, T inA, T outA, int ainA,
                                 int aoutA, int recA, bool hitB, T inB, T outB, int ainB,
                                 int aoutB, int recB, int top) {
  const int cA_in = (ainA << 8), cA_out = 1 | (aoutA << 8);
  const int cB_in = (ainB << 8), cB_out = 1 | (aoutB << 8);
  if (op == LG_LOGIC_AND) {
    if (!hitA || !hitB) return;
    // a-boundary points inside b, then b-boundary points inside a
    if (inA > inB && inA < outB) consider(nb, inA, recA, cA_in, (T)0, top);
    if (outA > inB && outA < outB) consider(nb, outA, recA, cA_out, (T)0, top);
    if (inB > inA && inB < outA) consider(nb, inB, recB, cB_in, (T)0, top);
    if (outB > inA && outB < outA) consider(nb, outB, recB, cB_out, (T)0, top);
  } else if (op == LG_LOGIC_OR) {
    // a-boundary points outside b, b-boundary points outside a
    if (hitA) {
      bool in_b_in = hitB && inA > inB && inA < outB;
      bool in_b_out = hitB && outA > inB && outA < outB;
      if (!in_b_in) consider(nb, inA, recA, cA_in, (T)0, top);
      if (!in_b_out) consider(nb, outA, recA, cA_out, (T)0, top);
    }
    if (hitB) {
      bool in_a_in = hitA && inB > inA && inB < outA;
      bool in_a_out = hitA && outB > inA && outB < outA;
      if (!in_a_in) consider(nb, inB, recB, cB_in, (T)0, top);
      if (!in_a_out) consider(nb, outB, recB, cB_out, (T)0, top);
    }
  } else {
    // a minus b: a-boundary outside b; b-boundary inside a with the normal flipped
    if (hitA) {
      bool in_b_in = hitB && inA > inB && inA < outB;
      bool in_b_out = hitB && outA > inB && outA < outB;
      if (!in_b_in) consider(nb, inA, recA, cA_in, (T)0, top);
      if (!in_b_out) consider(nb, outA, recA, cA_out, (T)0, top);
    }
    if (hitB && hitA) {
      if (inB > inA && inB < outA) consider(nb, inB, recB, cB_in | 2, (T)0, top);
      if (outB > inA && outB < outA) consider(nb, outB, recB, cB_out | 2, (T)0, top);
    }
  }
}

template <typename T>
struct TreeHit {
  T t;
  int rec;  // -1: nothing kept
  int code;
};

// A Logic tree of three or four primitives (records [i, i + n), prefix order). A leaf's
// entry or exit point is kept by the two-operand rule applied at every Logic node above it:
// And keeps it inside the other operand, Or outside it, AndNot outside b on the a side and
// inside a on the b side (normal flipped). Insideness at a point's t comes from the other
// leaves' chords (convex leaves: inside iff t lies strictly within the chord), combined
// bottom-up. Returns the object's nearest kept point (the first in leaf order, entry before
// exit, among equal ones): `consider` never makes an object its own runner-up, so that is
// what offering every kept point would leave. Trees this size are rare, so the chords are
// recomputed rather than held in registers.
template <typename T, typename RS>
__device__ __forceinline__ TreeHit<T> logic_tree(const RayT<T>& r, RS recs, const Rec<double>* recs64,
                                                 const T* verts, int i, int n) {
  const int nl = (int)recs[i].p[4];
  T best = (T)0;
  int best_k = -1, best_code = 0;
  for (int m = 0; m < nl; m++) {
    const int leaf = i + (int)rec_param(recs, i, m);
    T tin, tout;
    int ain, aout;
    if (!chord_any(r, recs[leaf].kind, recs[leaf], recs64 + leaf, verts, tin, tout, ain, aout)) continue;
    for (int side = 0; side < 2; side++) {
      const T t = side ? tout : tin;
      if (!(t > tmin_v<T>()) || (best_k >= 0 && !(t < best))) continue;
      uint32_t leaf_in = 0;  // the point lies on leaf m's boundary: not inside it
      for (int q = 0; q < nl; q++) {
        if (q == m) continue;
        const int kq = i + (int)rec_param(recs, i, q);
        T qin, qout;
        int qa, qb;
        if (chord_any(r, recs[kq].kind, recs[kq], recs64 + kq, verts, qin, qout, qa, qb) && t > qin && t < qout)
          leaf_in |= 1u << q;
      }
      // insideness of every subtree at t (bit k - i for the subtree whose root record is k)
      uint32_t node_in = 0, st = 0;
      int sp = 0, lq = nl - 1;
      for (int k = i + n - 1; k >= i; k--) {
        bool v;
        if (recs[k].kind == REC_LOGIC || recs[k].kind == REC_TREE) {
          const bool a = (st >> (sp - 1)) & 1u, b = (st >> (sp - 2)) & 1u;
          sp -= 2;
          v = logic_combine(recs[k].op, a, b);
        } else {
          v = (leaf_in >> lq) & 1u;
          lq--;
        }
        st = (st & ~(1u << sp)) | ((uint32_t)v << sp);
        sp++;
        node_in |= (uint32_t)v << (k - i);
      }
      // the rules of the Logic nodes from the root down to the leaf
      bool keep = true, flip = false;
      int node = i;
      while (node != leaf) {
        const int a = node + 1;
        const int b = a + (recs[a].kind == REC_LOGIC ? recs[a].aux : 1);
        const bool a_side = leaf < b;
        const bool other_in = (node_in >> ((a_side ? b : a) - i)) & 1u;
        const int op = recs[node].op;
        if (op == LG_LOGIC_AND) {
          keep = keep && other_in;
        } else if (op == LG_LOGIC_OR) {
          keep = keep && !other_in;
        } else if (a_side) {
          keep = keep && !other_in;
        } else {
          keep = keep && other_in;
          flip = !flip;
        }
        node = a_side ? a : b;
      }
      if (keep) {
        best = t;
        best_k = leaf;
        best_code = side | ((side ? aout : ain) << 8) | (flip ? 2 : 0);
      }
    }
  }
  return TreeHit<T>{best, best_k, best_code};
}

// Tests one object (records starting at i) and returns the index of the next object. The
// object walk (kTrees false) never meets a Logic tree of more than two primitives: their
// records follow the walk's.
template <typename T, bool kTrees = true, typename RS>
__device__ __forceinline__ int eval_object(const RayT<T>& r, RS recs, const Rec<double>* recs64, const T* verts,
                                           int i, int kind, Nearest<T>& nb) {
  const Rec<T>& R = recs[i];
  if (kind == REC_SEG) {
    T t;
    if (hit_segment(r, R.p, t)) consider(nb, t, i, 0, (T)0, i);
    return i + 1;
  }
  if (kind == REC_BEZ) {
    if (!ray_meets_box(r, R.p + 8)) return i + 1;
    T t, s = (T)0;
    bool amb = false;
    bool hit = bezier_nearest(r, R.p, t, s, amb);
    if constexpr (sizeof(T) == 4) {
      if (amb) {
        RayT<double> rd{(double)r.ox, (double)r.oy, (double)r.dx, (double)r.dy};
        double td, sd;
        bool a2 = false;
        hit = bezier_nearest<double>(rd, recs64[i].p, td, sd, a2);
        t = (float)td;
        s = (float)sd;
      }
    }
    if (hit) consider(nb, t, i, 0, s, i);
    return i + 1;
  }
  if constexpr (kTrees) {
    if (kind == REC_TREE) {
      const TreeHit<T> h = logic_tree<T>(r, recs, recs64, verts, i, R.aux);
      if (h.rec >= 0) consider_tree(nb, h.t, h.rec, h.code, i, nb.top < 0 || R.obj < recs[nb.top].obj);
      return i + R.aux;
    }
  }
  if (kind == REC_LOGIC) {
    T inA = 0, outA = 0, inB = 0, outB = 0;
    int ainA, aoutA, ainB, aoutB;
    bool hA = chord_any(r, recs[i + 1].kind, recs[i + 1], recs64 + i + 1, verts, inA, outA, ainA, aoutA);
    bool hB = chord_any(r, recs[i + 2].kind, recs[i + 2], recs64 + i + 2, verts, inB, outB, ainB, aoutB);
    logic_candidates(nb, R.op, hA, inA, outA, ainA, aoutA, i + 1, hB, inB, outB, ainB, aoutB,
                     i + 2, i);
    return i + 3;
  }
  T tin, tout;
  int ain, aout;
  if (chord_any(r, kind, R, recs64 + i, verts, tin, tout, ain, aout)) {
    if (tin > tmin_v<T>())
      consider(nb, tin, i, ain << 8, (T)0, i);
    else
      consider(nb, tout, i, 1 | (aout << 8), (T)0, i);
  }
  return i + 1;
}

// The culling pass for one ray over every object in scene order. Logic trees of more than two
// primitives are not among them. Inlined, so that the compiler sees which records are in LDS and
// which in global memory.
template <typename T, typename RS>
__device__ __forceinline__ void walk_objects(const RayT<T>& r, RS recs, const Rec<double>* recs64, const T* verts,
                                             int n_recs, Nearest<T>& nb) {
  for (int rec = 0; rec < n_recs;) rec = eval_object<T, false>(r, recs, recs64, verts, rec, recs[rec].kind, nb);
}

// a + b + the lane's bit of `carry`.
__device__ __forceinline__ uint32_t add_carry(uint32_t a, uint32_t b, uint64_t carry) {
  uint32_t r;
  uint64_t out;
  asm("v_addc_co_u32 %0, %1, %2, %3, %4" : "=v"(r), "=s"(out) : "v"(a), "v"(b), "s"(carry));
  return r;
}

// The scene's culling blocks; tops: the blocks' first records in LDS.
struct CullView {
  const LG_K CullBlock* blocks;
  const LG_K float* box;
  const int32_t* tops;
  int n;
};

// The culling pass by boxes: every lane tests its ray against the boxes of a block's objects
// (uniform, branch-free, four boxes to a scalar load, ten vector instructions each) for a t in
// [tmin, t_best + 4e-5 (1 + t_best)], which leaves a bit per candidate; then, kind by kind, each
// lane evaluates its own candidates, as many rounds as the lane with the most has of that kind. A
// walk that evaluates an object for the whole wave when one lane needs it (a hierarchy does that
// too) runs nearly all of them once rays have split up, since a wave's rays are in no order then.
// Bound: instruction issue and the serial loads of the rounds. A million rays, 64 objects, 10
// bounces: trace launches 894 us over every object, 716 us through a hierarchy of boxes, 553 us
// so (573 with the kind read from each lane's record: branches over execution masks); 75011 rays,
// 23 objects, 8 bounces: 263, 256 and 200 us; FP64, 40009 rays, 12 objects, 6
// bounces: 110 and 97 us (records in LDS). Few objects are tested as soon as their boxes (trace calls of
// 20000 rays, 6 bounces, us, over every object and by boxes: 4 objects 77 and 78, 6 93 and 92, 8 101
// and 95, 12 111 and 100): by boxes from lg_tuning.bvh_min_objects (8) objects.
//
// Every object that can hit within the window is a candidate (boxes are padded beyond the FP32
// error of the test and of the hits, for the scene's farthest ray origins: object_boxes), so the
// winner, and any runner-up that the FP64 refinement looks at (within 1e-5 (1 + t)), are those of
// the full walk: `consider` does not depend on the order.
template <typename T, typename RS>
__device__ __forceinline__ void walk_boxes(const RayT<T>& r, RS recs, const Rec<double>* recs64, const T* verts,
                                           const CullView& C, Nearest<T>& nb) {
  // (1e-18: the products stay finite for coordinates below 1e20)
  const float ox = (float)r.ox, oy = (float)r.oy, dx = (float)r.dx, dy = (float)r.dy;
  const float ix = 1.0f / (fabsf(dx) > 1e-18f ? dx : __builtin_copysignf(1e-18f, dx));
  const float iy = 1.0f / (fabsf(dy) > 1e-18f ? dy : __builtin_copysignf(1e-18f, dy));
  const float ax = -ox * ix, ay = -oy * iy;
  // an FP64 ray's rounding to FP32 moves it by up to 2^-24 of its origin's coordinates; the boxes'
  // padding covers the same of theirs
  const float slack = sizeof(T) == 8 ? 6e-7f * (fabsf(ax) + fabsf(ay)) : 0.0f;
  const float wx = fabsf(ix), wy = fabsf(iy);
  // whether the ray meets the box (centre and half sizes) within [1e-5, lim]
  auto meets = [&](const LG_K float* b, float lim) {
    const float cx = __builtin_fmaf(b[0], ix, ax), cy = __builtin_fmaf(b[1], iy, ay);
    const float tn = fmaxf(fmaxf(__builtin_fmaf(-b[2], wx, cx), __builtin_fmaf(-b[3], wy, cy)), 1e-5f);
    const float tf = fminf(fminf(__builtin_fmaf(b[2], wx, cx), __builtin_fmaf(b[3], wy, cy)), lim);
    if constexpr (sizeof(T) == 8) return !(tn > tf + slack);  // (NaN: a candidate)
    return tn <= tf;
  };
  for (int b = 0; b < C.n; b++) {
    const LG_K CullBlock* const B = C.blocks + b;
    const float bt = (float)nb.t;
    const float lim = bt + 4e-5f * (1.0f + bt);
    if (C.n > 1 && !__ballot(meets(B->box, lim))) continue;
    const int n = B->n, first = B->first;
    // from the last box down: each moves the bits up by one and adds its own, one instruction (an
    // add with the comparison as carry)
    uint32_t half[2] = {0u, 0u};
#pragma unroll
    for (int h = 1; h >= 0; h--)
      for (int o = (n < 32 * (h + 1) ? n + kBoxGroup - 1 : 32 * (h + 1)) / kBoxGroup * kBoxGroup - kBoxGroup; o >= 32 * h;
           o -= kBoxGroup) {
        const LG_K float* const x = C.box + 4 * (first + o);
#pragma unroll
        for (int k = kBoxGroup - 1; k >= 0; k--) half[h] = add_carry(half[h], half[h], __ballot(meets(x + 4 * k, lim)));
      }
    const uint64_t cand = (uint64_t)half[1] << 32 | half[0];
    for (int k = 0; k < B->n_kinds; k++) {
      uint64_t m = cand & B->kind[k];
      const int kind = (int)(B->kinds >> (4 * k) & 15u);  // the same for every lane: scalar branches
      while (__ballot(m != 0ull)) {
        if (m) {
          const int top = C.tops[first + __builtin_ctzll(m)];
          m &= m - 1ull;
          eval_object<T, false>(r, recs, recs64, verts, top, kind, nb);
        }
      }
    }
  }
}

// The objects that are Logic trees of more than two primitives: first records and the
// per-object boxes (padded world boxes, indexed by the records' object).
struct TreeList {
  const int32_t* top;
  const float4* box;
  int n;
};

// Records of the object walk: those before the first such tree.
__device__ __forceinline__ int walk_records(const TreeList& trees, int n_recs) {
  return trees.n ? __builtin_amdgcn_readfirstlane(trees.top[0]) : n_recs;
}

// Nearest hit over every object: walk(nb) offers those before the first Logic tree of more than
// two primitives, then come those trees in a wave-uniform loop of their own, where the
// walk's state is no longer live (such trees are rare; a test for them inside the walk raises
// its register pressure). `consider` keeps the lexicographic minimum of (t, scene order) and
// the nearest t of another object, so the order in which objects are offered does not change
// the result. A tree whose box the ray does not enter within the window of the walk by boxes is
// skipped, for the same reason.
template <typename T, typename RS, typename Walk>
__device__ __forceinline__ Nearest<T> nearest_hit(const RayT<T>& r, RS recs, const Rec<double>* recs64,
                                                  const T* verts, const TreeList& trees, Walk&& walk) {
  Nearest<T> nb;
  nearest_init(nb);
  walk(nb);
  if (trees.n == 0) return nb;
  const T ix = (T)1 / (fabs(r.dx) > (T)1e-30 ? r.dx : (T)__builtin_copysign(1e-30, (double)r.dx));
  const T iy = (T)1 / (fabs(r.dy) > (T)1e-30 ? r.dy : (T)__builtin_copysign(1e-30, (double)r.dy));
  for (int k = 0; k < trees.n; k++) {
    const int top = __builtin_amdgcn_readfirstlane(trees.top[k]);
    const float4 bx = trees.box[recs[top].obj];
    const T tx0 = ((T)bx.x - r.ox) * ix, tx1 = ((T)bx.z - r.ox) * ix;
    const T ty0 = ((T)bx.y - r.oy) * iy, ty1 = ((T)bx.w - r.oy) * iy;
    const T tn = fmax(fmin(tx0, tx1), fmin(ty0, ty1));
    const T tf = fmin(fmax(tx0, tx1), fmax(ty0, ty1));
    const T lim = nb.t + (T)4e-5 * ((T)1 + nb.t);
    if (!(tn <= tf && tf >= (T)1e-5 && tn <= lim)) continue;
    const TreeHit<T> h = logic_tree<T>(r, recs, recs64, verts, top, recs[top].aux);
    if (h.rec >= 0) consider_tree(nb, h.t, h.rec, h.code, top, nb.top < 0 || recs[top].obj < recs[nb.top].obj);
  }
  return nb;
}

// Outward (closed) or left (open) unit normal of the winning surface at p.
template <typename T>
__device__ __forceinline__ void hit_normal(const Rec<T>& R, const T* verts, int code, T s, T px, T py, T& nx,
                           T& ny) {
  int face = code >> 8;
  switch (R.kind) {
    case REC_SEG: nx = R.p[4]; ny = R.p[5]; break;
    case REC_BEZ: {
      T tx = ((T)3 * R.p[0] * s + (T)2 * R.p[2]) * s + R.p[4];
      T ty = ((T)3 * R.p[1] * s + (T)2 * R.p[3]) * s + R.p[5];
      if (tx == (T)0 && ty == (T)0) {
        // cusp: chord direction P3 - P0 = a3 + a2 + a1
        tx = R.p[0] + R.p[2] + R.p[4];
        ty = R.p[1] + R.p[3] + R.p[5];
      }
      nx = -ty;
      ny = tx;
      break;
    }
    case REC_CIRCLE: nx = px - R.p[0]; ny = py - R.p[1]; break;
    case REC_RECT: {
      T lx = (face == 1) ? (T)1 : (face == 3) ? (T)-1 : (T)0;
      T ly = (face == 2) ? (T)1 : (face == 0) ? (T)-1 : (T)0;
      nx = lx * R.p[2] + ly * R.p[4];
      ny = lx * R.p[3] + ly * R.p[5];
      break;
    }
    case REC_ELLIPSE: {
      T lx = px - R.p[0], ly = py - R.p[1];
      T x = lx * R.p[2] + ly * R.p[3], y = lx * R.p[4] + ly * R.p[5];
      T gx = x / (R.p[6] * R.p[6]), gy = y / (R.p[7] * R.p[7]);
      nx = gx * R.p[2] + gy * R.p[4];
      ny = gx * R.p[3] + gy * R.p[5];
      break;
    }
    case REC_POLY: {
      int first = R.aux, nv = R.op;
      int j = (face + 1 == nv) ? 0 : face + 1;
      T ex = verts[2 * (first + j)] - verts[2 * (first + face)];
      T ey = verts[2 * (first + j) + 1] - verts[2 * (first + face) + 1];
      T lx = ey, ly = -ex;
      nx = lx * R.p[2] + ly * R.p[4];
      ny = lx * R.p[3] + ly * R.p[5];
      break;
    }
    default: nx = (T)0; ny = (T)1; break;
  }
  normalize_v(nx, ny);
  if (code & 2) {
    nx = -nx;
    ny = -ny;
  }
}

// Ray::refract (tracer.rs:444-450): reflected and refracted directions and the
// unpolarised Fresnel reflectance; false on total internal reflection.
template <typename T>
__device__ __forceinline__ bool refract_dir(T dx, T dy, T nx, T ny, T n1, T n2, T& rx, T& ry, T& tx, T& ty,
                            T& R) {
  T ci = -(dx * nx + dy * ny);
  if (ci < (T)0) {
    nx = -nx;
    ny = -ny;
    ci = -ci;
  }
  rx = dx + (T)2 * ci * nx;
  ry = dy + (T)2 * ci * ny;
  normalize_v(rx, ry);
  T eta = n1 / n2;
  T k = (T)1 - eta * eta * ((T)1 - ci * ci);
  if constexpr (sizeof(T) == 4) {
    if (__builtin_fabsf(k) < kIsland) {
      double rxd, ryd, txd, tyd, Rd;
      bool ok = refract_dir<double>(dx, dy, nx, ny, n1, n2, rxd, ryd, txd, tyd, Rd);
      rx = (float)rxd;
      ry = (float)ryd;
      tx = (float)txd;
      ty = (float)tyd;
      R = (float)Rd;
      return ok;
    }
  }
  if (k < (T)0) {
    R = (T)1;
    return false;
  }
  T ct = sqrt_v(k);
  tx = eta * dx + (eta * ci - ct) * nx;
  ty = eta * dy + (eta * ci - ct) * ny;
  normalize_v(tx, ty);
  T ds = n1 * ci + n2 * ct, dp = n2 * ci + n1 * ct;
  T rs = ds != (T)0 ? (n1 * ci - n2 * ct) / ds : (T)1;
  T rp = dp != (T)0 ? (n2 * ci - n1 * ct) / dp : (T)1;
  R = (T)0.5 * (rs * rs + rp * rp);
  return true;
}

// key = ray_index << kPathBits | path; a child appends one bit to the path
// (0 reflected, 1 refracted).
__device__ __forceinline__ uint64_t child_key(uint64_t key, uint64_t bit) {
  const uint64_t mask = (1ull << kPathBits) - 1ull;
  return (key & ~mask) | (((key & mask) << 1) & mask) | bit;
}

__device__ __forceinline__ bool below_cutoff(const float c[4], const float cut[4]) {
  return (c[0] < cut[0] && c[1] < cut[1] && c[2] < cut[2]) || c[3] < cut[3];
}

// Light ray i of the scene (light.rs:103-115, 163-174, 225-249), generated in FP64.
__device__ __forceinline__ void gen_ray(const DevLight* lights, int n_lights, uint64_t gi, double& ox, double& oy,
                        double& dx, double& dy, float c[4], double& ior) {
  int l = 0;
  while (l + 1 < n_lights && gi >= lights[l + 1].ray_base) l++;
  const DevLight& L = lights[l];
  uint64_t i = gi - L.ray_base;
  double n = (double)L.num_rays;
  if (L.kind == LG_LIGHT_POINT) {
    double f = (double)i * M_PI * 2.0 / n;
    ox = L.a[0];
    oy = L.a[1];
    dx = cos(f);
    dy = sin(f);
  } else if (L.kind == LG_LIGHT_SPOT) {
    double angle = L.min_angle + ((double)(i + 1) / n) * L.spot_angle;
    ox = L.a[0];
    oy = L.a[1];
    dx = L.sign * cos(angle);
    dy = L.sign * sin(angle);
  } else {
    double r = (double)i / n;
    ox = L.a[0] + r * L.e[0];
    oy = L.a[1] + r * L.e[1];
    dx = L.nrm[0];
    dy = L.nrm[1];
  }
  c[0] = L.color[0];
  c[1] = L.color[1];
  c[2] = L.color[2];
  c[3] = L.color[3];
  ior = L.ior;
}

// Canvas exit (tracer.rs:484-486): nearest intersection with the canvas rect.
template <typename T>
__device__ __forceinline__ bool canvas_exit(const RayT<T>& r, const double* cv, T& px, T& py) {
  T t0 = -inf_v<T>(), t1 = inf_v<T>();
  if (r.dx != (T)0) {
    T ta = (cv[0] - r.ox) / r.dx, tb = (cv[1] - r.ox) / r.dx;
    t0 = ta < tb ? ta : tb;
    t1 = ta < tb ? tb : ta;
  } else if (r.ox < cv[0] || r.ox > cv[1]) {
    return false;
  }
  if (r.dy != (T)0) {
    T ta = (cv[2] - r.oy) / r.dy, tb = (cv[3] - r.oy) / r.dy;
    T lo = ta < tb ? ta : tb, hi = ta < tb ? tb : ta;
    t0 = lo > t0 ? lo : t0;
    t1 = hi < t1 ? hi : t1;
  } else if (r.oy < cv[2] || r.oy > cv[3]) {
    return false;
  }
  if (!(t0 <= t1)) return false;
  T t;
  if (t0 > tmin_v<T>())
    t = t0;
  else if (t1 > tmin_v<T>())
    t = t1;
  else
    return false;
  px = r.ox + t * r.dx;
  py = r.oy + t * r.dy;
  return true;
}

// ---------------------------------------------------------------------------------------
// One bounce generation of every scene of a batch.
//
// Work items are ranges of `rpi` rays of one scene; item i belongs to the scene s with
// item_pre[s] <= i < item_pre[s + 1]. A persistent workgroup takes items with an atomic
// cursor and reloads the scene into LDS only when the scene changes.
//
// Ray state (origin, direction, refractive index) is FP64. The O(objects) culling loop runs
// in T over the LDS records; for T = float the winning object (and a runner-up within the
// tie tolerance) is re-evaluated in FP64, and the whole FP64 scan is redone when that
// re-evaluation no longer clearly wins. Shading (normal, inside test, Snell/Fresnel, total
// internal reflection, children) is FP64.
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ double tie_tol(double t) { return 1e-5 * (1.0 + t); }

// Full FP64 scan for the rare ray whose FP32 winner was not confirmed, by boxes whatever the scene's
// size: a wave waits for its slowest lane. (Over every object, with a record's loads waited for one
// after another, one such ray of a scene of 64 objects took 225 us, most of a launch of a million.)
__device__ __forceinline__ Nearest<double> rescan_fp64(const RayT<double>& rd, const Rec<double>* recs64,
                                                    const double* verts64, const CullView& blocks,
                                                    const TreeList& trees) {
  return nearest_hit<double>(rd, recs64, recs64, verts64, trees, [&](Nearest<double>& nb) {
    walk_boxes<double>(rd, recs64, recs64, verts64, blocks, nb);
  });
}

// FP64 answer for a ray whose FP32 culling pass found `nb`.
__device__ __forceinline__ void refine_fp64(const RayT<double>& rd, const Nearest<float>& nb,
                                            const Rec<double>* recs64, const double* verts64,
                                            const CullView& blocks, const TreeList& trees, Nearest<double>& h) {
  const bool tie = nb.top2 >= 0 && (double)nb.t2 <= (double)nb.t + tie_tol(nb.t);
  if (tie) {
    int a = nb.top < nb.top2 ? nb.top : nb.top2;
    int b = nb.top < nb.top2 ? nb.top2 : nb.top;
    eval_object<double>(rd, recs64, recs64, verts64, a, recs64[a].kind, h);
    eval_object<double>(rd, recs64, recs64, verts64, b, recs64[b].kind, h);
  } else {
    eval_object<double>(rd, recs64, recs64, verts64, nb.top, recs64[nb.top].kind, h);
  }
  const bool unsure = h.top < 0 || (!tie && nb.top2 >= 0 && h.t > (double)nb.t2 - tie_tol(nb.t2));
  if (unsure) h = rescan_fp64(rd, recs64, verts64, blocks, trees);
}

__device__ __forceinline__ uint64_t gen_input_count(const SceneDesc& D, uint32_t gen_ix) {
  if (gen_ix == 0) return D.n_primary;
  uint64_t c = D.gen_count[gen_ix - 1];
  return c < D.q_cap ? c : D.q_cap;
}

// Largest s in [0, n) with pre[s] <= x (pre is non-decreasing, pre[0] = 0).
__device__ __forceinline__ int find_scene(const uint32_t* pre, int n, uint32_t x) {
  int lo = 0, hi = n;
  while (hi - lo > 1) {
    int mid = (lo + hi) >> 1;
    if (pre[mid] <= x)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// item_pre[s] = first item of scene s for generation `gen_ix` > 0; item_pre[n] = total, run by
// one workgroup of BLOCK threads (generation 0's comes from the host, which knows the primary
// rays). The previous generation's child counts were written by other workgroups of the running
// kernel, so they are read with device-scope atomic loads (not through this CU's cache).
template <int BLOCK>
__device__ __forceinline__ void build_items_block(const SceneDesc* __restrict__ descs, int n_scenes,
                                                  uint32_t gen_ix, uint32_t max_rpi, uint32_t* item_pre,
                                                  BatchCtl* ctl) {
  constexpr int kW = BLOCK / 64;
  __shared__ uint32_t s_w[kW];
  __shared__ uint32_t s_carry;
  __shared__ unsigned long long s_rays;
  auto scene_rays = [&](int sid) -> uint64_t {
    if (sid >= n_scenes) return 0;
    const SceneDesc& D = descs[sid];
    if (gen_ix >= D.max_bounce) return 0;
    const uint32_t g = __hip_atomic_load(gen(D.gen_count) + gen_ix - 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return g < D.q_cap ? g : D.q_cap;
  };
  if (threadIdx.x == 0) {
    s_carry = 0;
    s_rays = 0;
  }
  __syncthreads();
  for (int sid = threadIdx.x; sid < n_scenes; sid += BLOCK) {
    const uint64_t c = scene_rays(sid);
    if (c) atomicAdd(&s_rays, (unsigned long long)c);
  }
  __syncthreads();
  const uint32_t rpi = trace_item_rays(s_rays, max_rpi, gridDim.x, n_scenes);
  for (int base = 0; base < n_scenes; base += BLOCK) {
    const int sid = base + threadIdx.x;
    const uint32_t n_it = (uint32_t)((scene_rays(sid) + rpi - 1) / rpi);
    // block exclusive scan
    uint32_t x = n_it;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      uint32_t y = __shfl_up(x, d, 64);
      if (lane >= d) x += y;
    }
    if (lane == 63) s_w[wave] = x;
    __syncthreads();
    uint32_t wofs = 0;
    for (int w = 0; w < wave; w++) wofs += s_w[w];
    const uint32_t carry = s_carry;
    if (sid < n_scenes) item_pre[sid] = carry + wofs + x - n_it;
    __syncthreads();
    if (threadIdx.x == BLOCK - 1) s_carry = carry + wofs + x;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    item_pre[n_scenes] = s_carry;
    ctl->n_items_gen[gen_ix] = s_carry;
    ctl->item_rays[gen_ix] = rpi;
    ctl->item_cursor[gen_ix] = 0;
  }
}

// One launch traces `chunk` bounce generations, gen_ix .. gen_ix + chunk - 1 (bounce-chunking).
// A work item is `rpi` rays of generation gen_ix of one scene, traced BLOCK at a time; the
// children of a sub-batch at level j < chunk - 1 (generation gen_ix + j) stay on chip, in the
// LDS buffer of level j + 1 (2 * BLOCK rays: the children of one sub-batch), and are traced
// depth-first before the next sub-batch of level j, so a level's buffer is empty whenever its
// parents' level appends to it. Only the last level's children go to the scene's ray queue in
// HBM (counted at gen_count[gen_ix + chunk - 1]) for the next launch; launch_ix (the launch's
// index in the frame) picks the ping-pong queues.
constexpr uint32_t kMaxChunk = 3;

// LDS of one trace workgroup: the objects' first records and flags in scene order, first records
// in the culling blocks' order (without padding, which only the last block has), polygon
// vertices, the FP64 trace's records (the FP32 culling pass reads its records from global
// memory), then the level buffers of a chunked launch.
struct TraceLds {
  size_t obj, tops, verts, recs, levels, total;
};
template <typename T>
__host__ __device__ inline TraceLds trace_lds(int n_recs, int n_objs, int n_verts, uint32_t chunk, int block) {
  TraceLds L;
  L.obj = 0;
  L.tops = (size_t)n_objs * 4;
  L.verts = (L.tops + (size_t)n_objs * 4 + 15) & ~size_t(15);
  L.recs = (L.verts + (size_t)n_verts * 2 * sizeof(T) + 15) & ~size_t(15);
  const bool fp64 = sizeof(T) == 8;
  L.levels = (L.recs + (fp64 ? (size_t)n_recs * sizeof(Rec<T>) : 0) + 15) & ~size_t(15);
  L.total = L.levels + (size_t)(chunk > 1 ? chunk - 1 : 0) * 2 * block * sizeof(QRay<double>);
  return L;
}

template <typename T, int BLOCK>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void trace_kernel(const SceneDesc* __restrict__ descs, int n_scenes,
                                                      uint32_t gen_ix, uint32_t chunk, uint32_t launch_ix,
                                                      const uint32_t* __restrict__ item_pre,
                                                      BatchCtl* ctl, uint32_t max_rpi, int cap_recs,
                                                      int cap_objs, int cap_verts,
                                                      uint32_t* __restrict__ item_pre_next) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int kWaves = BLOCK / 64;
  __shared__ uint32_t s_wseg[kWaves];
  __shared__ uint32_t s_wch[kWaves];
  __shared__ unsigned long long s_seg_base;
  __shared__ uint32_t s_ch_base;
  __shared__ uint32_t s_item;
  __shared__ uint32_t s_lcnt[kMaxChunk];  // rays in the LDS buffer of each level (1 .. chunk - 1)

  const TraceLds lay = trace_lds<T>(cap_recs, cap_objs, cap_verts, chunk, BLOCK);
  uint32_t* s_obj = reinterpret_cast<uint32_t*>(smem + lay.obj);  // first record << 2 | ObjFlags
  int32_t* s_tops = reinterpret_cast<int32_t*>(smem + lay.tops);
  T* s_verts = reinterpret_cast<T*>(smem + lay.verts);
  Rec<T>* s_rec = reinterpret_cast<Rec<T>*>(smem + lay.recs);
  QRay<double>* s_lvl = reinterpret_cast<QRay<double>*>(smem + lay.levels);  // level j at (j - 1) * 2 * BLOCK

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const uint32_t n_items = ctl->n_items_gen[gen_ix];
  const uint32_t rpi = ctl->item_rays[gen_ix];
  // Workgroup b's first item is b: the others have none. They leave before any atomic or fence
  // (with both, the 900 idle workgroups of a late generation held up the working ones by 13 us).
  if (blockIdx.x >= n_items) return;
  int loaded = -1;
  if (threadIdx.x < kMaxChunk) s_lcnt[threadIdx.x] = 0;

  bool first = true;
  for (;;) {
    if (threadIdx.x == 0) s_item = next_work_item(&ctl->item_cursor[gen_ix], n_items, first);
    first = false;
    __syncthreads();
    // the item (and so the scene) is the same for the whole workgroup: keep it scalar
    const uint32_t it = __builtin_amdgcn_readfirstlane(s_item);
    if (it >= n_items) break;
    const int sid = __builtin_amdgcn_readfirstlane(find_scene(item_pre, n_scenes, it));
    const SceneDesc& D = descs[sid];
    const Rec<double>* recs64 = gen(D.recs64);
    const double* verts64 = gen(D.verts64);
    const int n_recs = D.n_recs, n_objs = D.n_objs;
    const TreeList trees{gen(D.tree_rec), gen(D.obj_box), D.n_trees};
    const CullView blocks{(const LG_K CullBlock*)D.blocks, (const LG_K float*)D.block_box, s_tops, D.n_blocks};
    CullView cull = blocks;
    if (!D.by_boxes) cull.n = 0;
    if (sid != loaded) {
      if (sizeof(T) == 8) {  // the FP32 pass reads its records with scalar loads instead
        const int4* src = reinterpret_cast<const int4*>(gen(D.recs));
        int4* dst = reinterpret_cast<int4*>(s_rec);
        const int n16 = n_recs * (int)(sizeof(Rec<T>) / 16);
        for (int k = threadIdx.x; k < n16; k += BLOCK) dst[k] = src[k];
      }
      const int n_walk = n_objs - D.n_trees;  // the objects that the blocks hold
      for (int k = threadIdx.x; k < n_objs; k += BLOCK) {
        s_obj[k] = (uint32_t)gen(D.obj_rec)[k] << 2 | gen(D.obj_flags)[k];
        if (k < n_walk) s_tops[k] = gen(D.block_rec)[k];
      }
      const T* vsrc = reinterpret_cast<const T*>(gen(D.verts));
      for (int k = threadIdx.x; k < 2 * D.n_verts; k += BLOCK) s_verts[k] = vsrc[k];

      loaded = sid;
    }
    __syncthreads();

    const uint64_t count = gen_input_count(D, gen_ix);
    const uint64_t begin = (uint64_t)(it - item_pre[sid]) * rpi;
    const uint64_t end = begin + rpi < count ? begin + rpi : count;
    const QRay<double>* in_q = gen(launch_ix & 1 ? D.q0 : D.q1);
    QRay<double>* out_q = gen(launch_ix & 1 ? D.q1 : D.q0);
    // levels of this launch the scene has (gen_ix < max_bounce: the item exists)
    const uint32_t levels = D.max_bounce - gen_ix < chunk ? D.max_bounce - gen_ix : chunk;

    for (uint64_t base = begin; base < end; base += BLOCK) {
      // Depth-first over the levels: the sub-batch at `level` is rays [head, head + BLOCK) of
      // its input (the item's rays at level 0, the level's LDS buffer above). h1 and h2 are the
      // heads of levels 1 and 2 (kMaxChunk = 3).
      uint32_t level = 0, h1 = 0, h2 = 0;
      for (;;) {
      const uint32_t g = gen_ix + level;  // the sub-batch's bounce generation
      const bool last_gen = g + 1 >= D.max_bounce;
      const bool to_lds = level + 1 < chunk;  // children stay on chip (else the HBM queue)
      const uint64_t idx = level == 0 ? base + threadIdx.x : (uint64_t)(level == 1 ? h1 : h2) + threadIdx.x;
      bool active = level == 0 ? idx < end : idx < (uint64_t)s_lcnt[level];
      double ox = 0, oy = 0, dx = 1, dy = 0, ior = 1;
      float c[4] = {0, 0, 0, 0};
      uint64_t key = 0;
      if (active) {
        if (g == 0) {
          gen_ray(gen(D.lights), D.n_lights, idx, ox, oy, dx, dy, c, ior);
          key = (idx << kPathBits) | 1ull;
          if (below_cutoff(c, D.cutoff)) active = false;
        } else {
          auto take = [&](const QRay<double>& q) {
            ox = q.o[0]; oy = q.o[1]; dx = q.d[0]; dy = q.d[1];
            c[0] = q.c[0]; c[1] = q.c[1]; c[2] = q.c[2]; c[3] = q.c[3];
            ior = q.ior;
            key = q.key;
          };
          if (level == 0)
            take(in_q[idx]);
          else
            take(s_lvl[(size_t)(level - 1) * 2 * BLOCK + idx]);
        }
      }

      bool emit = false, keep0 = false, keep1 = false;
      double px = 0, py = 0, nx = 0, ny = 0;
      double d0x = 0, d0y = 0, d1x = 0, d1y = 0;
      float c0[4] = {0, 0, 0, 0}, c1[4] = {0, 0, 0, 0};
      double n_refr = ior;
      bool hit = false, seek = false;  // seek: exiting a closed object, medium not yet found
      int obj = -1;
      uint32_t fl = 0;
      double n2 = 1.0;
      if (active) {
        const RayT<double> rd{ox, oy, dx, dy};
        Nearest<double> h;
        if constexpr (sizeof(T) == 8) {
          h = nearest_hit<double>(rd, s_rec, recs64, s_verts, trees, [&](Nearest<double>& nb) {
            if (cull.n)
              walk_boxes<double>(rd, s_rec, recs64, s_verts, cull, nb);
            else
              walk_objects<double>(rd, s_rec, recs64, s_verts, walk_records(trees, n_recs), nb);
          });
        } else {
          const RayT<float> rf{(float)ox, (float)oy, (float)dx, (float)dy};
          const RecK krec{(const LG_K lg_v4i*)D.recs};
          const RecV vrec{(const lg_v4i*)gen(D.recs)};
          Nearest<float> nb = nearest_hit<float>(rf, krec, recs64, s_verts, trees, [&](Nearest<float>& nf) {
            if (cull.n)
              walk_boxes<float>(rf, vrec, recs64, s_verts, cull, nf);
            else
              walk_objects<float>(rf, krec, recs64, s_verts, walk_records(trees, n_recs), nf);
          });
          nearest_init(h);
          if (nb.top >= 0) refine_fp64(rd, nb, recs64, verts64, blocks, trees, h);
        }
        if (h.rec >= 0) {
          const Rec<double>& R = recs64[h.rec];
          if (R.kind == REC_BEZ) {
            double sp = h.s;
            px = ((R.p[0] * sp + R.p[2]) * sp + R.p[4]) * sp + R.p[6];
            py = ((R.p[1] * sp + R.p[3]) * sp + R.p[5]) * sp + R.p[7];
          } else {
            px = ox + h.t * dx;
            py = oy + h.t * dy;
          }
          hit_normal<double>(R, verts64, h.code, h.s, px, py, nx, ny);
          obj = R.obj;
          fl = s_obj[obj] & 3u;
          hit = true;
          emit = true;
          if (fl & OBJ_MATERIAL) {
            seek = (fl & OBJ_CLOSED) && (dx * nx + dy * ny > 0.0);
            if (!seek) n2 = gen(D.obj_n64)[obj];
          }
        } else {
          emit = canvas_exit<double>(rd, D.canvas, px, py);
        }
      }
      // The medium a ray exits into: the first other material object, in scene order, that
      // contains the exit point (tracer.rs:431-440), else air. The masks of the point's bucket in x
      // and in y give the few of 64 objects at a time that can; a lane looks at its own, in
      // order, up to the first whose padded box holds the point (in FP32: the padding of 1e-5 (1 +
      // |coordinates|) covers that) and that contains it by the exact FP64 test. (A test of every
      // box by every lane, without branches, was a quarter of the vector instructions of a step with
      // 64 objects. With ten instead of thirteen instructions per box in the culling pass,
      // trace launches: a million rays, 64 objects 618 -> 582 us; 75011 rays, 23 objects 215 -> 204.)
      if (__ballot(seek)) {
        const int kx = medium_bucket((float)px, D.medium_map[0], D.medium_map[1]);
        const int ky = medium_bucket((float)py, D.medium_map[2], D.medium_map[3]);
        for (int base = 0; base < n_objs; base += 64) {
          const MediumMasks* const m = gen(D.medium) + base / 64;
          uint64_t cand = seek ? m->x[kx] & m->y[ky] : 0ull;
          if ((unsigned)(obj - base) < 64u) cand &= ~(1ull << (obj - base));
          while (__ballot(cand != 0ull)) {
            if (cand) {
              const int o = base + __builtin_ctzll(cand);
              cand &= cand - 1ull;
              const float4 b = gen(D.obj_box)[o];
              const float fx = (float)px, fy = (float)py;
              if ((fx >= b.x) & (fy >= b.y) & (fx <= b.z) & (fy <= b.w) &&
                  contains_object<double>(recs64, verts64, (int)(s_obj[o] >> 2), px, py)) {
                n2 = gen(D.obj_n64)[o];
                seek = false;
                cand = 0ull;
              }
            }
          }
          if (!__ballot(seek)) break;
        }
      }
      if (hit) {
        if (fl & OBJ_MATERIAL) {
          double Rf;
          const bool has_refr = refract_dir<double>(dx, dy, nx, ny, ior, n2, d0x, d0y, d1x, d1y, Rf);
          const float rf = (float)Rf;       // tracer.rs:454
          const float omr = 1.0f - rf;      // tracer.rs:455
          c0[0] = c[0] * rf; c0[1] = c[1] * rf; c0[2] = c[2] * rf; c0[3] = c[3];
          keep0 = !below_cutoff(c0, D.cutoff);
          if (has_refr) {
            c1[0] = c[0] * omr; c1[1] = c[1] * omr; c1[2] = c[2] * omr; c1[3] = c[3];
            keep1 = !below_cutoff(c1, D.cutoff);
            n_refr = n2;
          }
        } else {
          // Ray::reflect (tracer.rs:476-480)
          const double dn = dx * nx + dy * ny;
          d0x = dx - 2.0 * dn * nx;
          d0y = dy - 2.0 * dn * ny;
          normalize_v(d0x, d0y);
          c0[0] = c[0]; c0[1] = c[1]; c0[2] = c[2]; c0[3] = c[3];
          keep0 = true;  // same colour as the parent, which passed the cutoff
        }
      }
      if (last_gen) {
        keep0 = false;
        keep1 = false;
      }

      // ---- workgroup-aggregated append ----
      const uint64_t m_seg = __ballot(emit);
      const uint64_t m_c0 = __ballot(keep0);
      const uint64_t m_c1 = __ballot(keep1);
      const uint32_t pre_seg = __builtin_amdgcn_mbcnt_hi((uint32_t)(m_seg >> 32),
                                                         __builtin_amdgcn_mbcnt_lo((uint32_t)m_seg, 0));
      const uint32_t pre_c0 = __builtin_amdgcn_mbcnt_hi((uint32_t)(m_c0 >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((uint32_t)m_c0, 0));
      const uint32_t pre_c1 = __builtin_amdgcn_mbcnt_hi((uint32_t)(m_c1 >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((uint32_t)m_c1, 0));
      if (lane == 0) {
        s_wseg[wave] = (uint32_t)__popcll(m_seg);
        s_wch[wave] = (uint32_t)(__popcll(m_c0) + __popcll(m_c1));
      }
      __syncthreads();
      if (threadIdx.x == 0) {
        uint32_t ts = 0, tc = 0;
        for (int w = 0; w < kWaves; w++) {
          uint32_t a = s_wseg[w], b = s_wch[w];
          s_wseg[w] = ts;
          s_wch[w] = tc;
          ts += a;
          tc += b;
        }
        s_seg_base = ts ? atomicAdd(gen(D.seg_count), (unsigned long long)ts) : 0ull;
        if (to_lds) {
          s_ch_base = s_lcnt[level + 1];
          s_lcnt[level + 1] += tc;
        } else {
          s_ch_base = tc ? atomicAdd(gen(D.gen_count) + gen_ix + chunk - 1, tc) : 0u;
        }
      }
      __syncthreads();
      if (emit) {
        const uint64_t slot = s_seg_base + s_wseg[wave] + pre_seg;
        if (slot < D.seg_cap) {
          gen(D.seg_pos)[slot] = make_float4((float)ox, (float)oy, (float)px, (float)py);
          gen(D.seg_col)[slot] = make_float4(c[0], c[1], c[2], c[3]);
          gen(D.seg_key)[slot] = key;
          if (D.seg_pos64) {
            double* p64 = gen(D.seg_pos64) + 4 * slot;
            p64[0] = ox;
            p64[1] = oy;
            p64[2] = px;
            p64[3] = py;
          }
        }
      }
      uint64_t ch_slot = (uint64_t)s_ch_base + s_wch[wave] + pre_c0 + pre_c1;
      // children: the next level's LDS buffer (at most 2 * BLOCK: it was empty) or the HBM queue
      auto put = [&](uint64_t slot, double ddx, double ddy, const float* cc, double n, uint64_t k) {
        auto fill = [&](QRay<double>& q) {
          q.o[0] = px; q.o[1] = py; q.d[0] = ddx; q.d[1] = ddy;
          q.c[0] = cc[0]; q.c[1] = cc[1]; q.c[2] = cc[2]; q.c[3] = cc[3];
          q.ior = n;
          q.key = k;
        };
        if (to_lds) {
          if (slot < 2u * BLOCK) fill(s_lvl[(size_t)level * 2 * BLOCK + slot]);
        } else if (slot < D.q_cap) {
          fill(out_q[slot]);
        }
      };
      if (keep0) {
        put(ch_slot, d0x, d0y, c0, ior, child_key(key, 0));
        ch_slot++;
      }
      if (keep1) put(ch_slot, d1x, d1y, c1, n_refr, child_key(key, 1));
      __syncthreads();
      // the next sub-batch: the children just written to the next level, else the rest of this
      // level, else up to the levels above (a finished level's buffer is emptied)
      if (level + 1 < levels && s_lcnt[level + 1] > 0) {
        level++;
        if (level == 1) h1 = 0; else h2 = 0;
        continue;
      }
      bool done = false;
      for (;;) {
        if (level == 0) {
          done = true;
          break;
        }
        const uint32_t hn = (level == 1 ? h1 : h2) + BLOCK;
        if (level == 1) h1 = hn; else h2 = hn;
        if (hn < s_lcnt[level]) break;
        __syncthreads();  // every lane has read the count
        if (threadIdx.x == 0) s_lcnt[level] = 0;
        __syncthreads();
        level--;
      }
      if (done) break;
      }
    }
  }
  // The last of the workgroups that had items builds the next launch's work list. Its child counts
  // are final then: every add to them has returned its value before its workgroup counts itself
  // done, and both are performed where all XCDs see them, so no fence is needed (a device-scope
  // release writes back an XCD's whole L2). The rays themselves are read by the next launch only.
  if (item_pre_next) {
    __shared__ bool s_last;
    __syncthreads();
    if (threadIdx.x == 0) {
      const uint32_t working = n_items < gridDim.x ? n_items : gridDim.x;
      s_last = __hip_atomic_fetch_add(&ctl->gen_done[gen_ix], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == working - 1;
    }
    __syncthreads();
    if (s_last) build_items_block<BLOCK>(descs, n_scenes, gen_ix + chunk, max_rpi, item_pre_next, ctl);
  }
}

// ---------------------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------------------
constexpr int kTraceBlock = 256;

template <typename T>
size_t trace_lds_bytes(int n_recs, int n_objs, int n_verts, uint32_t chunk) {
  return trace_lds<T>(n_recs, n_objs, n_verts, chunk, kTraceBlock).total;
}

uint32_t trace_max_chunk() { return kMaxChunk; }

int trace_block() { return kTraceBlock; }

template <typename T>
hipError_t launch_trace(const SceneDesc* descs, int n_scenes, uint32_t gen, uint32_t chunk, uint32_t launch_ix,
                        const uint32_t* item_pre, BatchCtl* ctl, uint32_t rpi, int cap_recs, int cap_objs,
                        int cap_verts, uint32_t* item_pre_next, int grid, hipStream_t stream) {
  size_t lds = trace_lds_bytes<T>(cap_recs, cap_objs, cap_verts, chunk);
  hipLaunchKernelGGL((trace_kernel<T, kTraceBlock>), dim3(grid), dim3(kTraceBlock), lds, stream, descs,
                     n_scenes, gen, chunk, launch_ix, item_pre, ctl, rpi, cap_recs, cap_objs, cap_verts,
                     item_pre_next);
  return hipGetLastError();
}

template hipError_t launch_trace<float>(const SceneDesc*, int, uint32_t, uint32_t, uint32_t, const uint32_t*,
                                        BatchCtl*, uint32_t, int, int, int, uint32_t*, int, hipStream_t);
template hipError_t launch_trace<double>(const SceneDesc*, int, uint32_t, uint32_t, uint32_t, const uint32_t*,
                                         BatchCtl*, uint32_t, int, int, int, uint32_t*, int, hipStream_t);
template size_t trace_lds_bytes<float>(int, int, int, uint32_t);
template size_t trace_lds_bytes<double>(int, int, int, uint32_t);

}  // namespace lg
