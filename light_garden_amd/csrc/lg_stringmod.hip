// lg_stringmod.hip — StringMod::draw on the GPU (src/light_garden/string_mod.rs:3-158): the
// string-art producer that feeds the same accumulation as the trace.
//
//   curve points   init_points (string_mod.rs:33-85): Circle, ComplexExp, Hypotrochoid,
//                  Lissajous, each point computed on the fly from its index in FP64
//   segments       draw_init_points (104-122): segment iix -> ix(iix) for iix in 0..modulo,
//                  per-vertex colours from get_color (124-150), FP64 end points stored as
//                  FP32 like the reference's vertex upload (sub_render_pass.rs:188-196)
//   nested         draw (152-158) with `nested`: the nested StringMod draws over the crossing
//                  points of the outer one's lines, line_crossings_as_points (87-102): every
//                  ordered pair (ixa, (ixa + diff) % L), diff = 1..L-1 outer, ixa inner, in
//                  that order
//
// All FP64 arithmetic here is written without fused multiply-adds (contract off), so every
// value is the IEEE result of the same operations in the same order as the reference's Rust
// (which never fuses): crossings and Mul/Add/Pow/Base indices are bit-exact, ComplexExp points
// too; the trigonometric curves differ from the host's libm by at most an ulp or two.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "lg_host.h"

#pragma clang fp contract(off)

using lg::fail;

namespace lg {

struct SmDev {          // one StringMod as the generator reads it
  uint64_t modulo, num, turns;
  uint32_t mode, curve;
  uint64_t cu[3];
  double cf[2];
  double scale;
  float color[4];
  uint32_t mrc_off, n_mrc;
  uint64_t seg_base;    // first output segment of this StringMod
  uint64_t n_points;    // points indexed: modulo (own curve) or the crossing count (nested)
  const double2* pts;   // NULL: the curve's own points; else the crossing points
};

struct SmScratch {
  DevBuf descs, lines, chunk_counts, masks, row_counts, row_off, total, maxbits;
  std::vector<DevBuf*> crossings;  // crossing points of the i-th nested StringMod of a call (kept, grown)
  PinnedBuf stage;
  ~SmScratch() {
    for (DevBuf* b : crossings) delete b;
  }
};

void SmScratchDeleter::operator()(SmScratch* s) const { delete s; }

}  // namespace lg

namespace {

using lg::SmDev;

constexpr int kBlock = 256;
constexpr double kTau = 6.283185307179586;  // std::f64::consts::TAU

__host__ __device__ inline uint64_t wrapping_pow(uint64_t base, uint32_t exp) {
  // u64::pow; a release build wraps modulo 2^64, where every multiplication order agrees
  uint64_t acc = 1;
  while (exp) {
    if (exp & 1u) acc *= base;
    base *= base;
    exp >>= 1;
  }
  return acc;
}

// x mod m; with 32-bit operands in a third of the instructions.
__device__ inline uint64_t umod(uint64_t x, uint64_t m) {
  return ((x | m) >> 32) == 0 ? (uint64_t)((uint32_t)x % (uint32_t)m) : x % m;
}

// ix for iix (string_mod.rs:111-117)
__device__ inline uint64_t target_index(const SmDev& s, uint64_t iix) {
  const uint64_t m = s.modulo;
  switch (s.mode) {
    case LG_SM_ADD: return umod(iix + s.num, m);
    case LG_SM_MUL: return umod(iix * s.num, m);
    case LG_SM_POW: return umod(wrapping_pow(iix, (uint32_t)s.num), m);
    default: return umod(wrapping_pow(s.num, (uint32_t)iix), m);
  }
}

// Complex::powu (num-complex 0.4.6): square-and-multiply over Complex * Complex =
// (re1 re2 - im1 im2) + (re1 im2 + im1 re2) i.
__device__ inline double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ inline double2 cpowu(double2 base, uint32_t exp) {
  if (exp == 0) return make_double2(1.0, 0.0);
  while ((exp & 1u) == 0) {
    base = cmul(base, base);
    exp >>= 1;
  }
  if (exp == 1) return base;
  double2 acc = base;
  while (exp > 1) {
    exp >>= 1;
    base = cmul(base, base);
    if (exp & 1u) acc = cmul(acc, base);
  }
  return acc;
}

// init_points()[n] (string_mod.rs:35-83), times this build's radius `scale` (exact for 1).
__device__ inline double2 curve_point(const SmDev& s, uint64_t n) {
  const double angle = (double)(s.turns * n) * kTau / (double)s.modulo;
  double x, y;
  switch (s.curve) {
    case LG_CURVE_COMPLEX_EXP: {
      const double2 c = cpowu(make_double2(s.cf[0], s.cf[1]), (uint32_t)(s.turns * n));
      x = c.x;
      y = c.y;
      break;
    }
    case LG_CURVE_HYPOTROCHOID: {
      const double small_r = (double)s.cu[0], big_r = (double)s.cu[1], off = (double)s.cu[2];
      const double smr = big_r - small_r;
      const double ratio = smr + off;
      const double inner = angle * smr / small_r;
      x = (smr * cos(angle) + off * cos(inner)) / ratio;
      y = (smr * sin(angle) - off * sin(inner)) / ratio;
      break;
    }
    case LG_CURVE_LISSAJOUS:
      x = sin((double)s.cu[0] * angle + s.cf[0]);
      y = sin((double)s.cu[1] * angle);
      break;
    default:  // Circle: (y, x) = angle.sin_cos()
      sincos(angle, &y, &x);
      break;
  }
  return make_double2(x * s.scale, y * s.scale);
}

// get_color (string_mod.rs:124-150): the mean of the matching modulo colours, else the colour.
__device__ inline float4 mod_color(const SmDev& s, const lg_mod_rem_color* mrc, uint64_t ix) {
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  uint32_t k = 0;
  for (uint32_t i = 0; i < s.n_mrc; i++) {
    const lg_mod_rem_color& c = mrc[s.mrc_off + i];
    if (umod(ix, c.modulo) == c.rem) {
      acc[0] += c.color[0];
      acc[1] += c.color[1];
      acc[2] += c.color[2];
      acc[3] += c.color[3];
      k++;
    }
  }
  if (k == 0) return make_float4(s.color[0], s.color[1], s.color[2], s.color[3]);
  const float d = (float)k;
  return make_float4(acc[0] / d, acc[1] / d, acc[2] / d, acc[3] / d);
}

__device__ inline float absmax4(float4 c) {
  return fmaxf(fmaxf(fabsf(c.x), fabsf(c.y)), fmaxf(fabsf(c.z), fabsf(c.w)));
}

// One thread per output segment of every StringMod of the call; col1 may be NULL (no modulo
// colours: both ends have the StringMod's colour). Each thread computes its two points: a table of
// them, shared by the StringMods of a curve, costs a launch and 16-byte gathers (draws, us, with a
// table and without: 1 StringMod over 4096 points 21 and 17; 16 over 100000 of a circle 39 and 37, of as
// many circles 66 and 37, of one hypotrochoid 40 and 54; 16 over 20000 with modulo colours 44 and 40).
__global__ void __launch_bounds__(kBlock) sm_segments_kernel(const SmDev* __restrict__ descs, int n_descs,
                                                             const lg_mod_rem_color* __restrict__ mrc,
                                                             uint64_t n_segs, float4* __restrict__ pos,
                                                             float4* __restrict__ col0, float4* __restrict__ col1,
                                                             uint64_t* __restrict__ key,
                                                             unsigned int* __restrict__ maxbits) {
  const uint64_t g = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  float mx = 0.0f;
  if (g < n_segs) {
    int lo = 0, hi = n_descs - 1;  // last descriptor with seg_base <= g
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (descs[mid].seg_base <= g) lo = mid;
      else hi = mid - 1;
    }
    const SmDev& s = descs[lo];
    const uint64_t iix = g - s.seg_base;
    const uint64_t ix = target_index(s, iix);
    double2 p, q;
    if (s.pts) {
      p = s.pts[iix < s.n_points ? iix : umod(iix, s.n_points)];
      q = s.pts[ix < s.n_points ? ix : umod(ix, s.n_points)];
    } else {
      p = curve_point(s, iix);  // points[iix % m] with iix < m
      q = curve_point(s, ix);
    }
    const float4 c0 = mod_color(s, mrc, iix);
    const float4 c1 = mod_color(s, mrc, ix);
    pos[g] = make_float4((float)p.x, (float)p.y, (float)q.x, (float)q.y);
    col0[g] = c0;
    if (col1) col1[g] = c1;
    key[g] = g;
    mx = fmaxf(absmax4(c0), absmax4(c1));
  }
  if (!maxbits) return;
  // |colour| bits order like the floats; one atomic per workgroup (one per wave to this word took half
  // of the kernel)
  __shared__ unsigned int s_max[kBlock / 64];
  unsigned int b = __float_as_uint(mx);
  for (int off = 32; off > 0; off >>= 1) b = max(b, (unsigned int)__shfl_xor((int)b, off, 64));
  if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = b;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kBlock / 64; w++) b = max(b, s_max[w]);
    if (b) atomicMax(maxbits, b);
  }
}

// The outer StringMod's lines: a = points[ixa], r = points[ix(ixa)] - a.
__global__ void __launch_bounds__(kBlock) sm_lines_kernel(SmDev s, double4* __restrict__ lines) {
  const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= s.modulo) return;
  const double2 a = curve_point(s, i);
  const double2 b = curve_point(s, target_index(s, i));
  lines[i] = make_double4(a.x, a.y, b.x - a.x, b.y - a.y);
}

// LineSegment::intersect, restated (collision2d is absent): a + t r = c + u s with
// t = ((c - a) x s) / (r x s), u = ((c - a) x r) / (r x s); a point iff r x s != 0 and
// t, u in [0, 1] (as the divided values); the point is a + t r. Parallel and zero-length
// lines never meet.
//
// The test runs without a division and without branches: with d = |r x s| and n the
// numerator signed as if d > 0, fl(n / d) lies in [0, 1] iff n == 0 or (n > 0, n <= 2d and
// n - d <= d 2^-53): fl(q) <= 1 iff q <= 1 + 2^-53 (round to nearest even), n - d is exact
// for d < n <= 2d (Sterbenz) and d 2^-53 is exact. That holds while the quotient cannot
// underflow or the products overflow (d, |n| in [2^-500, 2^500] or n == 0); a lane outside
// that range (or with NaN/inf) takes the divided test instead.
__device__ inline bool unit_fast(double n, double d, double two_d, double eps) {
  return (n == 0.0) | ((n > 0.0) & (n <= two_d) & (n - d <= eps));
}
__device__ inline bool in_range(double a) { return (a == 0.0) | ((a >= 0x1p-500) & (a <= 0x1p500)); }

__device__ inline bool crosses(const double4 A, const double4 B) {
  const double denom = A.z * B.w - A.w * B.z;
  const double qx = B.x - A.x, qy = B.y - A.y;
  const double tn = qx * B.w - qy * B.z;
  const double un = qx * A.w - qy * A.z;
  const bool neg = denom < 0.0;
  const double d = fabs(denom);
  const double t = neg ? -tn : tn, u = neg ? -un : un;
  const double two_d = d + d, eps = d * 0x1p-53;
  // `&` on the conditions rather than `&&`: every term is evaluated, without branches
  const bool ok = (d >= 0x1p-500) & (d <= 0x1p500) & in_range(fabs(t)) & in_range(fabs(u));
  bool hit = ok & unit_fast(t, d, two_d, eps) & unit_fast(u, d, two_d, eps);
  if (__builtin_expect(!ok & (denom != 0.0), 0)) {
    const double tq = tn / denom, uq = un / denom;
    hit = (tq >= 0.0) & (tq <= 1.0) & (uq >= 0.0) & (uq <= 1.0);
  }
  return hit;
}

// The crossing point of two lines already known to cross (t = tn / denom as above).
__device__ inline double2 crossing_point(const double4 A, const double4 B) {
  const double denom = A.z * B.w - A.w * B.z;
  const double qx = B.x - A.x, qy = B.y - A.y;
  const double t = (qx * B.w - qy * B.z) / denom;
  return make_double2(A.x + t * A.z, A.y + t * A.w);
}

// The pair sweep in blocks of kBlock lines (chunk c = blockIdx.x, ixa = c kBlock + lane) by
// kRows pair offsets (rows diff = d0 .. d0 + kRows - 1, d0 = 1 + blockIdx.y kRows): each
// block keeps its lines in registers and the kBlock + kRows - 1 partner lines
// lines[(ixa + diff) % L] in LDS, so a line is read from memory about twice per kRows pairs.
// PASS 0 classifies every pair, keeps each lane's kRows hit bits in masks and writes the
// crossings of every (row, chunk) to counts[(diff - 1) n_chunks + c]. PASS 1 reads the masks
// back and writes each crossing point at row_off[diff - 1] + chunk_off[(diff - 1) n_chunks + c]
// + its rank in the chunk: the reference's order (diff outer, ixa inner).
constexpr int kRows = 64;  // one bit of a per-lane u64 hit mask per row
constexpr int kWin = kBlock + kRows - 1;

template <int PASS>
__global__ void __launch_bounds__(kBlock) sm_crossings_kernel(const double4* __restrict__ lines, uint32_t L,
                                                              uint32_t n_chunks, uint32_t* __restrict__ counts,
                                                              unsigned long long* __restrict__ masks,
                                                              const uint64_t* __restrict__ row_off,
                                                              double2* __restrict__ out) {
  __shared__ double4 win[kWin];
  __shared__ uint32_t wcnt[kRows][kBlock / 64];
  const uint32_t c = blockIdx.x;
  const uint32_t d0 = 1 + blockIdx.y * kRows;
  const uint32_t w0 = c * kBlock + d0;
  for (uint32_t k = threadIdx.x; k < (uint32_t)kWin; k += kBlock) win[k] = lines[(w0 + k) % L];
  const uint32_t ixa = c * kBlock + threadIdx.x;
  const bool valid = ixa < L;
  const double4 A = lines[valid ? ixa : 0];
  unsigned long long* my_mask = masks + ((uint64_t)blockIdx.y * n_chunks + c) * kBlock + threadIdx.x;
  const uint32_t nr = L - d0 < (uint32_t)kRows ? L - d0 : (uint32_t)kRows;  // rows d0 .. L-1
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  unsigned long long mask = 0;
  if (PASS == 0) {
    for (uint32_t r = 0; r < nr; r++) {
      const bool hit = valid & crosses(A, win[threadIdx.x + r]);
      mask |= (unsigned long long)hit << r;
      const unsigned long long bal = __ballot(hit);
      if (lane == 0) wcnt[r][wave] = (uint32_t)__popcll(bal);
    }
    *my_mask = mask;
    __syncthreads();
    if (threadIdx.x < nr) {
      uint32_t t = 0;
      for (int w = 0; w < kBlock / 64; w++) t += wcnt[threadIdx.x][w];
      counts[(uint64_t)(d0 - 1 + threadIdx.x) * n_chunks + c] = t;
    }
    return;
  }
  mask = *my_mask;
  for (uint32_t r = 0; r < nr; r++) {
    const unsigned long long bal = __ballot((mask >> r) & 1ull);
    if (lane == 0) wcnt[r][wave] = (uint32_t)__popcll(bal);
  }
  __syncthreads();
  const unsigned long long below = (1ull << lane) - 1ull;
  for (uint32_t r = 0; r < nr; r++) {
    const bool hit = (mask >> r) & 1ull;
    const unsigned long long bal = __ballot(hit);
    if (hit) {
      uint32_t before = 0;
      for (int w = 0; w < wave; w++) before += wcnt[r][w];
      const uint64_t row = d0 - 1 + r;
      const uint64_t base = row_off[row] + counts[row * n_chunks + c];
      out[base + before + (uint32_t)__popcll(bal & below)] = crossing_point(A, win[threadIdx.x + r]);
    }
  }
}

// In-place exclusive scan of each row's n_chunks counts (one wave per row); row totals to
// row_tot.
__global__ void __launch_bounds__(kBlock) sm_scan_chunks_kernel(uint32_t* __restrict__ counts, uint32_t n_rows,
                                                                uint32_t n_chunks, uint32_t* __restrict__ row_tot) {
  const uint32_t row = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= n_rows) return;
  uint32_t* v = counts + (uint64_t)row * n_chunks;
  const uint32_t per = (n_chunks + 63) / 64;
  const uint32_t b = lane * per, e = b + per < n_chunks ? b + per : n_chunks;
  uint32_t sum = 0;
  for (uint32_t i = b; i < e; i++) sum += v[i];
  uint32_t inc = sum;
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t o = (uint32_t)__shfl_up((int)inc, off, 64);
    if (lane >= off) inc += o;
  }
  uint32_t run = inc - sum;
  for (uint32_t i = b; i < e; i++) {
    const uint32_t x = v[i];
    v[i] = run;
    run += x;
  }
  if (lane == 63) row_tot[row] = inc;
}

// Exclusive prefix of n row counts into u64 offsets and their total (one block).
__global__ void __launch_bounds__(1024) sm_scan_rows_kernel(const uint32_t* __restrict__ in, uint64_t n,
                                                            uint64_t* __restrict__ out,
                                                            uint64_t* __restrict__ total) {
  __shared__ uint64_t part[1024];
  const uint64_t per = (n + 1023) / 1024;
  const uint64_t b = threadIdx.x * per, e = b + per < n ? b + per : n;
  uint64_t s = 0;
  for (uint64_t i = b; i < e; i++) s += in[i];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const uint64_t v = threadIdx.x >= (unsigned)off ? part[threadIdx.x - off] : 0;
    __syncthreads();
    part[threadIdx.x] += v;
    __syncthreads();
  }
  uint64_t run = part[threadIdx.x] - s;
  for (uint64_t i = b; i < e; i++) {
    out[i] = run;
    run += in[i];
  }
  if (threadIdx.x == 1023) *total = part[1023];
}

// The end points of a sample of the segments (set_extent), into host memory.
__global__ void sm_extent_kernel(const float4* __restrict__ pos, uint64_t n, float4* samples) {
  samples[threadIdx.x] = pos[lg::extent_sample((int)threadIdx.x, n)];
}

__global__ void sm_zero_u32_kernel(unsigned int* p) { *p = 0u; }

int check_mod(const lg_string_mod& m, bool nested) {
  const char* who = nested ? "nested string mod" : "string mod";
  if (m.mode > LG_SM_BASE) return fail(LG_E_INVALID, std::string(who) + ": unknown mode");
  if (m.curve > LG_CURVE_LISSAJOUS) return fail(LG_E_INVALID, std::string(who) + ": unknown curve");
  if (m.n_modulo_colors > LG_MAX_MOD_COLORS)
    return fail(LG_E_INVALID, std::string(who) + ": more than LG_MAX_MOD_COLORS modulo colours");
  if (m.n_modulo_colors && !m.modulo_colors) return fail(LG_E_INVALID, std::string(who) + ": modulo_colors is NULL");
  for (uint32_t i = 0; i < m.n_modulo_colors; i++)
    if (m.modulo_colors[i].modulo == 0)
      return fail(LG_E_INVALID, std::string(who) + ": a modulo colour has modulo 0 (the reference divides by it)");
  return LG_OK;
}

SmDev make_dev(const lg_string_mod& m, uint32_t mrc_off) {
  SmDev d{};
  d.modulo = m.modulo;
  d.num = m.num;
  d.turns = m.turns;
  d.mode = m.mode;
  d.curve = m.curve;
  for (int i = 0; i < 3; i++) d.cu[i] = m.curve_u[i];
  d.cf[0] = m.curve_f[0];
  d.cf[1] = m.curve_f[1];
  d.scale = m.scale;
  for (int c = 0; c < 4; c++) d.color[c] = m.color[c];
  d.mrc_off = mrc_off;
  d.n_mrc = m.n_modulo_colors;
  d.n_points = m.modulo;
  return d;
}

lg::SmScratch& scratch(lg_ctx* ctx) {
  if (!ctx->sm) ctx->sm.reset(new lg::SmScratch());
  return *ctx->sm;
}

// Crossing points of `outer`'s lines into `dst` (device); *count gets their number.
int crossings_device(lg_ctx* ctx, const lg_string_mod& outer, lg::DevBuf& dst, uint64_t* count) {
  lg::SmScratch& S = scratch(ctx);
  hipStream_t st = ctx->stream;
  *count = 0;
  const uint64_t L = outer.modulo;
  if (L > LG_MAX_CROSSING_LINES)
    return fail(LG_E_INVALID, "string mod: line_crossings_as_points over more than LG_MAX_CROSSING_LINES lines");
  if (L < 2) return LG_OK;
  const uint32_t n_rows = (uint32_t)(L - 1);
  const uint32_t n_chunks = (uint32_t)((L + kBlock - 1) / kBlock);
  int rc;
  if ((rc = S.lines.ensure(L * sizeof(double4))) ||
      (rc = S.chunk_counts.ensure((uint64_t)n_rows * n_chunks * sizeof(uint32_t))) ||
      (rc = S.masks.ensure((uint64_t)((n_rows + kRows - 1) / kRows) * n_chunks * kBlock * 8)) ||
      (rc = S.row_counts.ensure(n_rows * sizeof(uint32_t))) || (rc = S.row_off.ensure(n_rows * sizeof(uint64_t))) ||
      (rc = S.total.ensure(sizeof(uint64_t))))
    return rc;
  const SmDev d = make_dev(outer, 0);
  const dim3 grid(n_chunks, (n_rows + kRows - 1) / kRows);
  {
    lg::StageScope sc(ctx, "sm_lines", L);
    hipLaunchKernelGGL(sm_lines_kernel, dim3((unsigned)((L + kBlock - 1) / kBlock)), dim3(kBlock), 0, st, d,
                       S.lines.as<double4>());
  }
  {
    lg::StageScope sc(ctx, "sm_cross_count", L * (L - 1));
    hipLaunchKernelGGL(sm_crossings_kernel<0>, grid, dim3(kBlock), 0, st, S.lines.as<const double4>(), (uint32_t)L,
                       n_chunks, S.chunk_counts.as<uint32_t>(), S.masks.as<unsigned long long>(),
                       (const uint64_t*)nullptr, (double2*)nullptr);
  }
  {
    lg::StageScope sc(ctx, "sm_cross_scan", (uint64_t)n_rows * n_chunks);
    hipLaunchKernelGGL(sm_scan_chunks_kernel, dim3((n_rows + kBlock / 64 - 1) / (kBlock / 64)), dim3(kBlock), 0, st,
                       S.chunk_counts.as<uint32_t>(), n_rows, n_chunks, S.row_counts.as<uint32_t>());
    hipLaunchKernelGGL(sm_scan_rows_kernel, dim3(1), dim3(1024), 0, st, S.row_counts.as<const uint32_t>(),
                       (uint64_t)n_rows, S.row_off.as<uint64_t>(), S.total.as<uint64_t>());
  }
  LG_HIP(hipGetLastError());
  if ((rc = S.stage.ensure(64))) return rc;
  LG_HIP(hipMemcpyAsync(S.stage.p, S.total.p, sizeof(uint64_t), hipMemcpyDeviceToHost, st));
  LG_HIP(hipStreamSynchronize(st));
  const uint64_t n = *S.stage.as<uint64_t>();
  if (n) {
    if ((rc = dst.ensure(n * sizeof(double2)))) return rc;
    lg::StageScope sc(ctx, "sm_cross_write", L * (L - 1));
    hipLaunchKernelGGL(sm_crossings_kernel<1>, grid, dim3(kBlock), 0, st, S.lines.as<const double4>(), (uint32_t)L,
                       n_chunks, S.chunk_counts.as<uint32_t>(), S.masks.as<unsigned long long>(),
                       S.row_off.as<const uint64_t>(), dst.as<double2>());
    LG_HIP(hipGetLastError());
  }
  *count = n;
  return LG_OK;
}

}  // namespace

extern "C" {

int lg_string_mod_draw(lg_ctx* ctx, uint32_t n, const lg_string_mod* mods, lg_segments* out) {
  if (!ctx || !out || (n && !mods)) return fail(LG_E_INVALID, "string mod: ctx, mods or out is NULL");
  if (out->ctx != ctx) return fail(LG_E_INVALID, "string mod: segments belong to another context");
  if (!(out->flags & LG_SEG_VERTEX_COLORS))
    return fail(LG_E_INVALID, "string mod: the segment buffer needs LG_SEG_VERTEX_COLORS");
  int rc;
  for (uint32_t i = 0; i < n; i++) {
    if ((rc = check_mod(mods[i], false))) return rc;
    if (mods[i].nested) {
      if ((rc = check_mod(*mods[i].nested, true))) return rc;
      if (mods[i].modulo > LG_MAX_CROSSING_LINES)
        return fail(LG_E_INVALID, "string mod: nested over more than LG_MAX_CROSSING_LINES lines");
    }
  }
  LG_HIP(hipSetDevice(ctx->device));
  lg::begin_call(ctx);
  hipStream_t st = ctx->stream;
  lg::SmScratch& S = scratch(ctx);
  size_t n_nested = 0;

  // nested StringMods draw over the crossing points of their outer lines (string_mod.rs:153-154)
  std::vector<SmDev> descs;
  std::vector<lg_mod_rem_color> mrc;
  uint64_t total = 0;
  bool nonneg = true;  // a segment's colour is the StringMod's or a mean of its modulo colours
  lg::SegRuns runs;    // consecutive StringMods of one colour
  bool in_runs = true;
  for (uint32_t i = 0; i < n; i++) {
    const lg_string_mod& outer = mods[i];
    const lg_string_mod& m = outer.nested ? *outer.nested : outer;
    SmDev d = make_dev(m, (uint32_t)mrc.size());
    mrc.insert(mrc.end(), m.modulo_colors, m.modulo_colors + m.n_modulo_colors);
    for (int c = 0; c < 4; c++) {
      nonneg = nonneg && m.color[c] >= 0.0f;
      for (uint32_t k = 0; k < m.n_modulo_colors; k++) nonneg = nonneg && m.modulo_colors[k].color[c] >= 0.0f;
    }
    if (outer.nested) {
      if (S.crossings.size() <= n_nested) S.crossings.push_back(new lg::DevBuf());
      lg::DevBuf& buf = *S.crossings[n_nested++];
      uint64_t np = 0;
      if ((rc = crossings_device(ctx, outer, buf, &np))) return rc;
      d.pts = buf.as<const double2>();
      d.n_points = np;
    }
    // draw_init_points returns nothing when there are no points (string_mod.rs:106-108)
    const uint64_t segs = d.n_points ? m.modulo : 0;
    if (!segs) continue;
    d.seg_base = total;
    in_runs = in_runs && !m.n_modulo_colors && runs.add(total, m.color);
    total += segs;
    descs.push_back(d);
  }
  if (total >= (1ull << 32)) return fail(LG_E_INVALID, "string mod: 2^32 or more segments in one call");
  if ((rc = lg::seg_ensure(out, std::max<uint64_t>(total, 1), false))) return rc;
  lg::seg_forget(out);
  uint32_t max_bits = 0;
  if (total) {
    // one upload: descs | modulo colours
    const size_t db = descs.size() * sizeof(SmDev);
    const size_t mb = mrc.size() * sizeof(lg_mod_rem_color);
    if ((rc = S.descs.ensure(db + mb)) || (rc = S.maxbits.ensure(16)) ||
        (rc = S.stage.ensure(std::max<size_t>(db + mb, 64 + lg::kExtentSamples * sizeof(float4)))))
      return rc;
    char* stage = S.stage.as<char>();
    std::memcpy(stage, descs.data(), db);
    if (mb) std::memcpy(stage + db, mrc.data(), mb);
    LG_HIP(hipMemcpyAsync(S.descs.p, stage, db + mb, hipMemcpyHostToDevice, st));
    const char* dev = S.descs.as<const char>();
    // without modulo colours the largest |colour channel| is known here
    unsigned int* const dev_max = mrc.empty() ? nullptr : S.maxbits.as<unsigned int>();
    for (const SmDev& d : descs) {
      const float m = std::fmax(std::fmax(std::fabs(d.color[0]), std::fabs(d.color[1])),
                                std::fmax(std::fabs(d.color[2]), std::fabs(d.color[3])));
      uint32_t b;
      std::memcpy(&b, &m, sizeof(b));
      max_bits = std::max(max_bits, b);
    }
    if (dev_max) hipLaunchKernelGGL(sm_zero_u32_kernel, dim3(1), dim3(1), 0, st, dev_max);
    {
      lg::StageScope sc(ctx, "sm_generate", total);
      hipLaunchKernelGGL(sm_segments_kernel, dim3((unsigned)((total + kBlock - 1) / kBlock)), dim3(kBlock), 0, st,
                         reinterpret_cast<const SmDev*>(dev), (int)descs.size(),
                         reinterpret_cast<const lg_mod_rem_color*>(dev + db), total,
                         out->pos.as<float4>(), out->col0.as<float4>(),
                         mrc.empty() ? nullptr : out->col1.as<float4>(), out->key.as<uint64_t>(), dev_max);
    }
    LG_HIP(hipGetLastError());
    // the staging buffer is free again once the stream has come this far
    if (dev_max) LG_HIP(hipMemcpyAsync(stage, dev_max, sizeof(unsigned int), hipMemcpyDeviceToHost, st));
    // (up to three runs are summed as weights whatever the extent: use_runs)
    float4* const samples = reinterpret_cast<float4*>(stage + 64);
    const bool sampled = in_runs && runs.n > 3;
    if (sampled) {
      hipLaunchKernelGGL(sm_extent_kernel, dim3(1), dim3(lg::kExtentSamples), 0, st, out->pos.as<const float4>(), total,
                         samples);
      LG_HIP(hipGetLastError());
    }
    LG_HIP(hipStreamSynchronize(st));
    if (dev_max) std::memcpy(&max_bits, stage, sizeof(max_bits));
    if (sampled) lg::set_extent(*out, samples);
  } else {
    LG_HIP(hipStreamSynchronize(st));
  }
  float max_abs;
  std::memcpy(&max_abs, &max_bits, sizeof(max_abs));
  out->count = total;
  out->max_abs = max_abs;
  out->nonneg = nonneg;
  if (in_runs) out->runs = runs;
  // without modulo colours both ends of every segment take their StringMod's colour
  // (get_color, string_mod.rs:124-150): col1 is then neither written nor read
  out->one_color = mrc.empty();
  out->has_pos64 = false;
  lg::end_call(ctx);
  return LG_OK;
}

int lg_string_mod_crossings(lg_ctx* ctx, const lg_string_mod* sm, double* xy, uint64_t cap_points,
                            uint64_t* n_points) {
  if (!ctx || !sm || !n_points) return fail(LG_E_INVALID, "string mod: ctx, sm or n_points is NULL");
  int rc;
  if ((rc = check_mod(*sm, false))) return rc;
  LG_HIP(hipSetDevice(ctx->device));
  lg::begin_call(ctx);
  lg::SmScratch& S = scratch(ctx);
  lg::DevBuf pts;
  uint64_t np = 0;
  if ((rc = crossings_device(ctx, *sm, pts, &np))) return rc;
  LG_HIP(hipStreamSynchronize(ctx->stream));
  *n_points = np;
  (void)S;
  if (np > cap_points || (np && !xy)) return fail(LG_E_CAPACITY, "string mod: crossing points exceed cap_points");
  if (np) LG_HIP(hipMemcpy(xy, pts.p, np * sizeof(double2), hipMemcpyDeviceToHost));
  lg::end_call(ctx);
  return LG_OK;
}

}  // extern "C"
