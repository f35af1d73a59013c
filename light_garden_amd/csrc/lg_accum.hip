// lg_accum.hip — additive line accumulation on gfx950.
//
// Replaces the reference's LineList draw with additive blend into an Rgba16Float target
// (src/sub_render_pass.rs:86-95, 188-212; src/shader.wgsl:14-28; blend
// src/light_garden/mod.rs:57-73; target src/texture_renderer.rs:5). HIP has no ROP path,
// so the raster + blend becomes three stages:
//   1. binning: every segment is enumerated against the square screen tiles (64 or 32
//      pixels a side, one size per frame) its deposits can touch. A workgroup owns a chunk
//      of segments, counts its pairs per row (tile, major axis) in an LDS histogram and adds
//      them to the rows' totals; what the adds return is the chunk's place in each row. The
//      row totals are scanned, and a second pass writes segment indices into per-tile lists,
//      y-major pairs first.
//   2. tiles: a persistent workgroup takes a (tile, pair range) work item, walks each of
//      its segments' column (x-major) or row (y-major) samples that fall in the tile (in
//      two-channel frames the samples of 64 pairs laid end to end, two to a lane, 128 per
//      step; else one per lane), and adds the two anti-aliased deposits per sample into a
//      64-bit fixed-point LDS tile: 4 colour planes, or 2 when two channels share a word, or
//      up to 3 hues' or 6 one-colour runs' weight planes, whose colours come in afterwards.
//      Integer sums make the image independent of the order of the deposits. When one item
//      owns the tile it converts the sums to FP32 and adds them to the accumulator with
//      coalesced read-add-write; the items of a heavy tile split over several items add
//      their exact sums into a 64-bit merge slot, converted afterwards by the same
//      expression.
//   3. resolve: FP32 accumulator -> RGBA16F, round to nearest even, alpha + 1 (the
//      target's clear alpha, renderer.rs:175).
//
// The sampling rule (shared with the FP64 oracle): world -> pixel
// X = (x - left) * sx, Y = (top - y) * sy; major axis x if |dX| >= |dY|; one sample per
// major-axis pixel whose centre k + 0.5 lies in the half-open span [M0, M1); with
// s = (k + 0.5 - M0) / dM, minor m = m0 + s dm, v = m - 0.5, j = floor(v), f = v - j,
// pixels j and j + 1 on the minor axis get weights 1 - f and f; a weight w adds w*rgb to
// RGB and w*a*a to alpha. Each (segment, tile) pair is set up in FP64 from the FP32 end
// points; its samples are then stepped in FP32 from the tile's first column.
#include <type_traits>

#include "lg_internal.h"

namespace lg {

// Largest tile edge; merge slots are sized for it. One colour plane of an LDS tile of edge T
// is unpadded: element (minor m, major q) of a walk sits at m * T + q, so the lanes of a
// deposit (consecutive q) fall in distinct banks whatever the segment's slope.
constexpr int kTileMax = 64;

struct SegGeom {
  double M0, m0, slope;  // slope = dm / dM
  int klo, khi;          // sample range on the major axis (clipped to the image)
  int xmajor;
};

// First and last sample (0.5-centred major pixels) of the half-open span from M0 (included) to M1
// (excluded), which differ.
__device__ __forceinline__ void sample_span(double M0, double M1, double& lo, double& hi) {
  if (M1 > M0) {
    lo = ceil(M0 - 0.5);
    hi = ceil(M1 - 0.5) - 1.0;
  } else {
    lo = floor(M1 - 0.5) + 1.0;
    hi = floor(M0 - 0.5);
  }
}

// Returns false when the segment deposits nothing.
__device__ __forceinline__ bool seg_geom(const float4 p, const AccumView& v, SegGeom& g) {
  double X0 = ((double)p.x - v.left) * v.sx;
  double Y0 = (v.top - (double)p.y) * v.sy;
  double X1 = ((double)p.z - v.left) * v.sx;
  double Y1 = (v.top - (double)p.w) * v.sy;
  if (!isfinite(X0) || !isfinite(Y0) || !isfinite(X1) || !isfinite(Y1)) return false;
  double dX = X1 - X0, dY = Y1 - Y0;
  int xm = fabs(dX) >= fabs(dY);
  double M0 = xm ? X0 : Y0, M1 = xm ? X1 : Y1;
  double m0 = xm ? Y0 : X0, dM = xm ? dX : dY, dm = xm ? dY : dX;
  if (M0 == M1) return false;
  double lo, hi;
  sample_span(M0, M1, lo, hi);
  double limit = (double)(xm ? v.width : v.height);
  if (lo < 0.0) lo = 0.0;
  if (hi > limit - 1.0) hi = limit - 1.0;
  if (!(lo <= hi)) return false;
  g.M0 = M0;
  g.m0 = m0;
  g.slope = dm * (1.0 / dM);
  // 0 <= lo <= hi <= limit - 1: one 32-bit conversion each (a 64-bit one takes six instructions)
  g.klo = (int)lo;
  g.khi = (int)hi;
  g.xmajor = xm;
  return true;
}

// 1 / x of a finite x away from the ends of the range, to about an ulp: the hardware's estimate
// and two Newton steps (a division's scaling and fix-up are most of its instructions).
__device__ __forceinline__ double rcp_newton(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
}

// LDS by byte address: a uniform part of an address that comes from a lane read stays an integer.
#define LG_L __attribute__((address_space(3)))
typedef uint32_t lg_v4u __attribute__((ext_vector_type(4)));
typedef uint32_t lg_v2u __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(uintptr_t)(const LG_L char*)p;
}
__device__ __forceinline__ uint4 lds_read16(uint32_t a) {
  return __builtin_bit_cast(uint4, *(const LG_L lg_v4u*)(uintptr_t)a);
}
__device__ __forceinline__ uint2 lds_read8(uint32_t a) {
  return __builtin_bit_cast(uint2, *(const LG_L lg_v2u*)(uintptr_t)a);
}

// Inclusive sum over the lanes of a wave with DPP lane moves (no LDS round trips): shifts by
// 1, 2, 4, 8 within each row of 16 lanes, then the totals of rows 0 and 2 broadcast into rows
// 1 and 3, and the total of rows 0-1 into rows 2-3. Lanes a move has no source for add 0.
__device__ __forceinline__ int wave_sum_incl(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1, 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2, 3
  return x;
}

// One segment of a wave's bin stream (48 bytes: three 16-byte LDS reads). tc is the segment's
// first major-axis tile column minus its first stream position, so stream position k is
// column tc + k.
struct alignas(16) ColumnRec {
  double M0, m0, slope;
  int klo, khi, tc;
  uint32_t seg;  // segment index | major axis << 31 (the pair entry)
  uint32_t pad[2];
};

// Segments per bin stream: one per lane of a wave. A segment spans at most 8192 / 32 = 256
// major-axis tile columns (image sides <= 8192, tiles >= 32), so a wave's stream holds at most
// 64 * 256 positions, 256 words of start bits.
constexpr int kBinMaskWords = 256;

// ---- batch helpers ------------------------------------------------------------------------
__device__ __forceinline__ int find_u32(const uint32_t* pre, int n, uint32_t x) {
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

__device__ __forceinline__ uint64_t scene_segments(const SceneDesc& D) {
  if (D.flags & SCENE_FIXED_COUNT) return D.seg_fixed;
  uint64_t c = *D.seg_count;
  return c < D.seg_cap ? c : D.seg_cap;
}

// Segments per bin chunk of a scene: the frame's chunk size, or a bin workgroup's share of the frame's
// segments, up to kSpreadMax (`spread`), where that is more. Every chunk initialises the scene's [tile][axis]
// histogram and writes it back, which short chunks of a large image would spend their time on, and
// adds it to the row totals, which many chunks of a small image queue up for (its totals are a few
// lines, and a line takes some 15 ns per chunk: a scene of a million segments on 64 tiles, cut
// into 4600 chunks beside 19 others, held the frame's count pass up: 152 us, 60 so; the fill pass
// 210 and 88). A scene with more chunks than workgroups gets a whole multiple of their number (a
// count just above it leaves most workgroups idle while the rest take one more chunk). Never more
// chunks than the frame's chunk size gives, so the count matrix keeps its capacity.
__device__ __forceinline__ uint32_t scene_chunk(uint32_t chunk, uint32_t groups, uint32_t spread, const SceneDesc& D) {
  const uint64_t n = scene_segments(D);
  const uint64_t g = groups ? groups : 1u;
  uint64_t sc = spread > chunk ? spread : chunk;
  const uint64_t nch = (n + sc - 1) / sc;
  if (nch > g) {
    const uint64_t whole = nch / g * g;
    sc = (n + whole - 1) / whole;
  }
  return (uint32_t)(sc < 0x80000000ull ? sc : 0x80000000ull);
}

// Bin layout of one frame, from the segment counts the trace just produced: the chunk size
// gives about `target` chunks over the whole batch (at least `chunk_min` segments each);
// chunk_pre[s] = first chunk of scene s, cbase[s] = first entry of scene s's [chunk][tile][axis]
// matrix (2 x tiles x its chunk count). Frames of up to kBinScenes scenes have a wave of every
// workgroup of the count pass make it (bin_kernel): a launch less, which at 5 us was a twentieth
// of the smallest frames (20000 rays 185 -> 182 us a frame). For more scenes build_chunks_kernel
// does, one block of 1024.
constexpr int kBinScenes = 64;
struct BinPlan {
  uint32_t chunk_min, target, groups;
  uint32_t lds_counters;  // LDS words of the histogram; the layout's follow
};
constexpr uint32_t bin_layout_words(int n_scenes) { return 2u * (uint32_t)n_scenes + 3u; }
// A chunk of kSpreadMax segments keeps its workgroup for longer than the adds of all workgroups to
// one line take (some 20 ns a segment against 15 ns for each of 1536), so no line holds them
// up; longer ones only leave the pass uneven. (256 scenes, 192M segments: count and fill pass
// 5.3 and 7.1 ms with chunks of a whole share, 125k segments, 2.0 and 3.3 so; at 16384 the same.)
constexpr unsigned long long kSpreadMax = 4096;
// Segments per chunk and per workgroup of a frame of `total` segments.
__device__ __forceinline__ uint2 frame_chunk(unsigned long long total, const BinPlan& P) {
  const unsigned long long ch = (total + P.target - 1) / P.target;
  unsigned long long sp = P.groups ? (total + P.groups - 1) / P.groups : total;
  if (sp > kSpreadMax) sp = kSpreadMax;
  return make_uint2((uint32_t)(ch > P.chunk_min ? (ch < 0x80000000ull ? ch : 0x80000000ull) : P.chunk_min),
                    (uint32_t)sp);
}

__global__ __launch_bounds__(1024) void build_chunks_kernel(const SceneDesc* __restrict__ descs, int n_scenes, BinPlan P,
                                                           uint32_t* chunk_pre, uint32_t* cbase, BatchCtl* ctl) {
  __shared__ unsigned long long s_tot[16];
  __shared__ uint32_t s_wa[16], s_wb[16];
  __shared__ uint32_t s_ca, s_cb;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // total segments of the batch
  unsigned long long tot = 0;
  for (int sid = threadIdx.x; sid < n_scenes; sid += 1024) tot += scene_segments(descs[sid]);
  for (int d = 32; d > 0; d >>= 1) tot += __shfl_down(tot, d, 64);
  if (lane == 0) s_tot[wave] = tot;
  if (threadIdx.x == 0) s_ca = s_cb = 0;
  __syncthreads();
  unsigned long long total = 0;
  for (int w = 0; w < 16; w++) total += s_tot[w];
  const uint2 fc = frame_chunk(total, P);
  const uint32_t chunk = fc.x, spread = fc.y, groups = P.groups;
  for (int base = 0; base < n_scenes; base += 1024) {
    const int sid = base + threadIdx.x;
    uint32_t nch = 0, ncnt = 0;
    if (sid < n_scenes) {
      const SceneDesc& D = descs[sid];
      const uint32_t sc = scene_chunk(chunk, groups, spread, D);
      nch = (uint32_t)((scene_segments(D) + sc - 1) / sc);
      ncnt = 2u * nch * (uint32_t)(D.view.tiles_x * D.view.tiles_y);
    }
    uint32_t xa = nch, xb = ncnt;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t ya = __shfl_up(xa, d, 64), yb = __shfl_up(xb, d, 64);
      if (lane >= d) {
        xa += ya;
        xb += yb;
      }
    }
    if (lane == 63) {
      s_wa[wave] = xa;
      s_wb[wave] = xb;
    }
    __syncthreads();
    uint32_t oa = s_ca, ob = s_cb;
    for (int w = 0; w < wave; w++) {
      oa += s_wa[w];
      ob += s_wb[w];
    }
    if (sid < n_scenes) {
      chunk_pre[sid] = oa + xa - nch;
      cbase[sid] = ob + xb - ncnt;
    }
    __syncthreads();
    if (threadIdx.x == 1023) {
      s_ca = oa + xa;
      s_cb = ob + xb;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    chunk_pre[n_scenes] = s_ca;
    cbase[n_scenes] = s_cb;
    ctl->chunk = chunk;
    ctl->spread = spread;
    ctl->bin_groups = groups;
    ctl->n_chunks = s_ca;
  }
}

// Persistent over bin chunks. PASS 0 counts a chunk's pairs per row (2 tile + major axis; axis
// 0: y-major, 1: x-major) in LDS, adds them to the row totals and keeps, in the chunk's row of
// the [chunk][tile][axis] matrix, the totals from before its own adds: the chunk's first place
// in each row's list. PASS 1 writes segment indices from row_start + that place on, so every
// tile's list holds its y-major pairs first, then its x-major ones, and each phase of the tile
// walk reads one contiguous run. (Which chunk comes first within a row changes from run to run;
// the tile sums do not depend on it.) The two rows of a tile share one 64-bit add: a row holds
// fewer than 2^31 pairs.
//
// What the chunks' places cost: one atomic per touched tile and chunk here, against a scan of
// the whole [tile][axis][chunk] matrix, written and read with strides of the chunk count, which
// this replaced (both passes and the scan, us: 1M-ray frame at 2048x2048 262 -> 204; 20 uneven
// scenes in one frame 1210 -> 394, part of it from `spread` being the frame's and not the
// scene's; 1.6M segments at 4096x4096 754 -> 630; 20k-ray frame at 1024x1024 45 -> 25).
template <int PASS>
__global__ __launch_bounds__(256) void bin_kernel(const SceneDesc* __restrict__ descs, int n_scenes,
                                                  BinPlan P, uint32_t* chunk_pre, uint32_t* cbase, BatchCtl* ctl,
                                                  uint32_t* places, uint32_t* rows, uint32_t* pairs,
                                                  uint64_t pairs_cap) {
  // rows: PASS 0 the row totals (zeroed before the frame), PASS 1 the rows' starts; both
  // 2 per tile of the frame
  extern __shared__ __align__(16) uint32_t s_hist[];
  __shared__ uint32_t s_chunk;
  __shared__ ColumnRec s_rec[4][64];
  __shared__ unsigned long long s_mask[4][kBinMaskWords];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  ColumnRec* const rec = s_rec[wave];
  unsigned long long* const mask = s_mask[wave];
  // PASS 0 of a frame of few scenes makes the layout; its first workgroup writes it for PASS 1
  const bool own_layout = PASS == 0 && n_scenes <= kBinScenes;
  // (after the histogram, sized for the frame's scenes: with room for kBinScenes apart, a 4096x4096
  // image's workgroups were two to a compute unit instead of three, count pass 225 -> 282 us)
  uint32_t* const s_pre = s_hist + P.lds_counters;
  uint32_t* const s_cbase = s_pre + n_scenes + 1;
  uint32_t* const s_chunk_spread = s_cbase + n_scenes;
  if (own_layout) {
    if (wave == 0) {
      const SceneDesc& D = descs[lane < n_scenes ? lane : 0];
      const unsigned long long n_own = lane < n_scenes ? scene_segments(D) : 0ull;
      unsigned long long total = n_own;
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) total += __shfl_xor(total, d, 64);
      const uint2 fc = frame_chunk(total, P);
      const uint32_t sc = scene_chunk(fc.x, P.groups, fc.y, D);
      const uint32_t nch = (uint32_t)((n_own + sc - 1) / sc);
      const uint32_t ncnt = 2u * nch * (uint32_t)(D.view.tiles_x * D.view.tiles_y);
      const uint32_t pre = (uint32_t)wave_sum_incl((int)nch) - nch, cb = (uint32_t)wave_sum_incl((int)ncnt) - ncnt;
      if (lane < n_scenes) {
        s_pre[lane] = pre;
        s_cbase[lane] = cb;
        if (lane == n_scenes - 1) s_pre[n_scenes] = pre + nch;
        if (blockIdx.x == 0) {
          chunk_pre[lane] = pre;
          cbase[lane] = cb;
          if (lane == n_scenes - 1) {
            chunk_pre[n_scenes] = pre + nch;
            ctl->n_chunks = pre + nch;
          }
        }
      }
      if (lane == 0) {
        s_chunk_spread[0] = fc.x;
        s_chunk_spread[1] = fc.y;
        if (blockIdx.x == 0) {
          ctl->chunk = fc.x;
          ctl->spread = fc.y;
          ctl->bin_groups = P.groups;
        }
      }
    }
    __syncthreads();
  }
  const uint32_t n_chunks = own_layout ? s_pre[n_scenes] : ctl->n_chunks;
  const uint32_t chunk = own_layout ? s_chunk_spread[0] : ctl->chunk;
  const uint32_t spread = own_layout ? s_chunk_spread[1] : ctl->spread;
  const uint32_t groups = own_layout ? P.groups : ctl->bin_groups;
  bool first = true;
  for (;;) {
    if (threadIdx.x == 0) s_chunk = next_work_item(PASS == 0 ? &ctl->chunk_cursor0 : &ctl->chunk_cursor1, n_chunks, first);
    first = false;
    __syncthreads();
    const uint32_t ci = __builtin_amdgcn_readfirstlane(s_chunk);
    if (ci >= n_chunks) break;
    const int sid = __builtin_amdgcn_readfirstlane(own_layout ? find_u32(s_pre, n_scenes, ci) : find_u32(chunk_pre, n_scenes, ci));
    const SceneDesc& D = descs[sid];
    const AccumView v = D.view;
    const int n_tiles = v.tiles_x * v.tiles_y;
    const uint32_t local = ci - (own_layout ? s_pre[sid] : chunk_pre[sid]);
    uint2* const mat =
        reinterpret_cast<uint2*>(places + (own_layout ? s_cbase[sid] : cbase[sid])) + (uint64_t)local * n_tiles;
    uint2* const tile_rows = reinterpret_cast<uint2*>(rows) + D.row_base;
    const uint32_t row_stride = D.row_stride;
    uint2* const hist2 = reinterpret_cast<uint2*>(s_hist);
    for (int t = threadIdx.x; t < n_tiles; t += blockDim.x) {
      if (PASS == 0) {
        hist2[t] = make_uint2(0u, 0u);
      } else {
        const uint2 a = tile_rows[t * row_stride], b = mat[t];
        hist2[t] = make_uint2(a.x + b.x, a.y + b.y);
      }
    }
    __syncthreads();
    const uint64_t n = scene_segments(D);
    const uint32_t sc = scene_chunk(chunk, groups, spread, D);
    const uint64_t s0 = (uint64_t)local * sc;
    const uint64_t s1 = s0 + sc < n ? s0 + sc : n;
    const int sh = v.tile_shift;
    const int T = v.tile;
    // Each wave takes 64 segments at a time and lays their (segment, major tile column) items
    // end to end; every step gives each lane one item, whatever the segments' lengths. Lane
    // l of step s finds its segment's record from the start bits of the stream, as the tile
    // walk does.
    for (uint64_t wb = s0 + (uint64_t)wave * 64; wb < s1; wb += 256) {
      const uint64_t s = wb + lane;
      SegGeom g{};
      int nc = 0;
      if (s < s1 && seg_geom(gen(D.seg_pos)[s], v, g)) nc = (g.khi >> sh) - (g.klo >> sh) + 1;
      const int incl = wave_sum_incl(nc);
      const int total = __builtin_amdgcn_readlane(incl, 63);
      if (total == 0) continue;
      // the tiles of column tm the segment's deposits can touch (conservative), counted or filled
      auto column = [&](int tm, double M0, double m0, double slope, int klo, int khi, uint32_t seg) {
        const int xmajor = (int)(seg >> 31);
        const int ka = klo > tm * T ? klo : tm * T;
        const int kb = khi < tm * T + T - 1 ? khi : tm * T + T - 1;
        const double ma = m0 + ((double)ka + 0.5 - M0) * slope;
        const double mb = m0 + ((double)kb + 0.5 - M0) * slope;
        const double mn = ma < mb ? ma : mb, mx = ma < mb ? mb : ma;
        const int minor_limit = xmajor ? v.height : v.width;
        // clamped to the image's rows before the (32-bit) conversions
        double f_lo = floor(mn - 0.5) - 1.0, f_hi = floor(mx - 0.5) + 2.0;
        f_lo = f_lo > 0.0 ? f_lo : 0.0;
        f_hi = f_hi < (double)(minor_limit - 1) ? f_hi : (double)(minor_limit - 1);
        if (!(f_lo <= f_hi)) return;
        const int r_lo = (int)f_lo, r_hi = (int)f_hi;
        for (int tn = r_lo >> sh; tn <= r_hi >> sh; tn++) {
          const int tile = xmajor ? tn * v.tiles_x + tm : tm * v.tiles_x + tn;
          const int row = 2 * tile + xmajor;
          if (PASS == 0) {
            // lanes that share the first active lane's counter add to it with one atomic
            const int lt = __builtin_amdgcn_readfirstlane(row);
            const uint64_t same = __ballot(row == lt);
            if (row != lt)
              atomicAdd(&s_hist[row], 1u);
            else if (__lane_id() == (unsigned)__builtin_ctzll(same))
              atomicAdd(&s_hist[lt], (uint32_t)__builtin_popcountll(same));
          } else {
            const uint32_t slot = atomicAdd(&s_hist[row], 1u);
            if (slot < pairs_cap) pairs[slot] = seg;
          }
        }
      };
      const int steps = (total + 63) >> 6;
      const uint32_t seg = (uint32_t)s | ((uint32_t)g.xmajor << 31);
      // A wave whose segments span about as many columns each walks them lane by lane (the
      // stream would cost more per column than the divergence it saves).
      if (__ballot(nc > steps + (steps >> 1) + 1) == 0) {
        const int t0 = nc ? g.klo >> sh : 0;
        for (int j = 0; j < nc; j++) column(t0 + j, g.M0, g.m0, g.slope, g.klo, g.khi, seg);
        continue;
      }
      const int pre = incl - nc;
      const uint64_t live = __ballot(nc != 0);
      const int c = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(live >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)live, 0u));
      // (one wave's LDS operations execute in order: words cleared, then starts set)
      for (int w = lane; w < steps; w += 64) mask[w] = 0ull;
      if (nc) {
        ColumnRec r;
        r.M0 = g.M0;
        r.m0 = g.m0;
        r.slope = g.slope;
        r.klo = g.klo;
        r.khi = g.khi;
        r.tc = (g.klo >> sh) - pre;
        r.seg = seg;
        r.pad[0] = r.pad[1] = 0u;
        rec[c] = r;
        atomicOr(&mask[pre >> 6], 1ull << (pre & 63));
      }
      uint32_t seen = 0;  // starts in the words before the step (wave-uniform)
      for (int st = 0; st < steps; st++) {
        const unsigned long long sw = mask[st];
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)sw);
        const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(sw >> 32));
        const uint64_t X = ((uint64_t)hi << 32 | lo) >> 1;
        const int owner = (int)seen + (int)(lo & 1u) - 1 +
                          (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(X >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)X, 0u));
        seen += (uint32_t)__builtin_popcountll((uint64_t)hi << 32 | lo);
        const int k = st * 64 + lane;
        if (k >= total) continue;
        const ColumnRec r = rec[owner];
        column(r.tc + k, r.M0, r.m0, r.slope, r.klo, r.khi, r.seg);
      }
    }
    __syncthreads();
    if (PASS == 0) {
      for (int t = threadIdx.x; t < n_tiles; t += blockDim.x) {
        const uint2 h = hist2[t];
        if (h.x | h.y) {  // (a tile the chunk does not touch has no pairs to place)
          const unsigned long long before = atomicAdd(reinterpret_cast<unsigned long long*>(tile_rows + t * row_stride),
                                                      (unsigned long long)h.y << 32 | h.x);
          mat[t] = make_uint2((uint32_t)before, (uint32_t)(before >> 32));
        }
      }
    }
    __syncthreads();
  }
}

// ---- tile work items ------------------------------------------------------------------------
// Tile g's list is pairs [rows[2 g], rows[2 g + 2]) of the scanned row totals, its x-major part
// from rows[2 g + 1] on (with layers 2 * layers rows per tile, y-major and x-major of each). A tile
// is cut into full pieces and at most one remainder; the items are ordered by size class
// (floor(log2(pairs))), largest class first. With `whole` (the frame clears, accumulates and
// resolves every image) a tile without pairs gets one empty item (size class 0), which writes its
// cleared pixels.
struct PlanLimits {
  uint64_t pairs_cap;
  uint32_t items_cap, split_cap;
  uint32_t min_piece, max_piece;
  uint32_t grid;   // tile workgroups
  uint32_t whole;
  uint32_t layers; // pairs of rows per tile
};

__device__ __forceinline__ uint32_t piece_size(unsigned long long total, const PlanLimits& L) {
  unsigned long long pc = total / (2ull * L.grid) + 1;
  pc = pc < L.min_piece ? L.min_piece : pc;
  pc = pc > L.max_piece ? L.max_piece : pc;
  return (uint32_t)pc;
}

// A tile of cnt pairs: its full pieces, whether one more item follows (the remainder, or the empty
// item), and that item's class.
struct TileCut {
  uint32_t full, items;
  int cls_rem;
};
__device__ __forceinline__ TileCut cut_tile(uint32_t cnt, uint32_t piece, uint32_t whole) {
  TileCut c;
  c.full = cnt / piece;
  const uint32_t rem = cnt - c.full * piece;
  c.items = cnt ? c.full + (rem ? 1u : 0u) : (whole ? 1u : 0u);
  c.cls_rem = rem ? 31 - __clz(rem) : 0;
  return c;
}

// Writes the items of tile g (list [b, e), x-major from mid); full_slot / rem_slot: the slots of
// its full pieces and of its last item.
__device__ __forceinline__ void put_items(WorkItem* items, uint32_t items_cap, uint32_t sid, uint32_t tile, uint32_t b,
                                          uint32_t e, uint32_t mid, uint32_t piece, const TileCut& c,
                                          uint32_t split_slot, uint32_t full_slot, uint32_t rem_slot) {
  const uint32_t cnt = e - b;
  for (uint32_t p = 0; p < c.items; p++) {
    WorkItem w;
    w.scene = sid | (c.items > 1 ? kSplitBit : 0u);
    w.tile = tile;
    w.begin = b + p * piece;
    w.end = e - w.begin > piece ? w.begin + piece : e;
    w.mid = mid;
    w.tile_pairs = cnt < kPackedPiece ? cnt : kPackedPiece;
    w.slot = split_slot;
    w.pad = 0u;
    const uint32_t slot = p < c.full ? full_slot + p : rem_slot;
    if (slot < items_cap) items[slot] = w;
  }
}

// Scan of the row totals and the work items in one workgroup, for frames of at most kPlanTiles
// tiles: thread t owns consecutive tiles. What it takes is the latency of its few dependent steps,
// so one launch in place of the five to seven of a multi-block scan, a piece count and an item
// writer is what counts here (us, with the launches it replaces: 256 tiles 34 -> 6, 1024 tiles
// 61 -> 18, 4096 tiles 122 -> 33, 6k tiles of 20 images 61 -> 30). One workgroup's time grows with
// its tiles, so frames of more take the multi-block scan.
constexpr int kPlanTiles = 8192;
__global__ __launch_bounds__(1024) void plan_items_kernel(const SceneDesc* __restrict__ descs,
                                                          const uint32_t* __restrict__ tile_scene, int n_tiles,
                                                          const uint32_t* __restrict__ row_count, BatchCtl* ctl,
                                                          uint32_t* row_start, WorkItem* items, uint32_t* split_tiles,
                                                          PlanLimits L) {
  __shared__ unsigned long long s_w[16];
  __shared__ uint32_t s_cls[32], s_cur[32];
  __shared__ uint32_t s_nsplit;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int per = (n_tiles + 1023) / 1024;
  const int t0 = (int)threadIdx.x * per < n_tiles ? (int)threadIdx.x * per : n_tiles;
  const int t1 = t0 + per < n_tiles ? t0 + per : n_tiles;
  const uint2* counts = reinterpret_cast<const uint2*>(row_count);
  uint2* starts = reinterpret_cast<uint2*>(row_start);
  const uint32_t nl = L.layers;
  auto tile_count = [&](int t) {
    uint32_t n = 0;
    for (uint32_t l = 0; l < nl; l++) {
      const uint2 c = counts[t * nl + l];
      n += c.x + c.y;
    }
    return n;
  };
  if (threadIdx.x < 32) s_cls[threadIdx.x] = 0u;
  if (threadIdx.x == 0) s_nsplit = 0u;
  unsigned long long own = 0;
  for (uint32_t t = t0 * nl; t < t1 * nl; t++) {
    const uint2 c = counts[t];
    own += (unsigned long long)c.x + c.y;
  }
  unsigned long long incl = own;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned long long y = __shfl_up(incl, d, 64);
    if (lane >= d) incl += y;
  }
  if (lane == 63) s_w[wave] = incl;
  __syncthreads();
  unsigned long long before = 0, total = 0;
  for (int w = 0; w < 16; w++) {
    before += w < wave ? s_w[w] : 0ull;
    total += s_w[w];
  }
  const uint32_t first = (uint32_t)(before + incl - own);  // (wraps only past pairs_cap: flagged below)
  const uint32_t piece = piece_size(total, L);
  const int cls_full = 31 - __clz(piece);
  uint32_t b = first;
  for (int t = t0; t < t1; t++) {
    const uint32_t b0 = b;
    for (uint32_t l = 0; l < nl; l++) {
      const uint2 c = counts[t * nl + l];
      starts[t * nl + l] = make_uint2(b, b + c.x);
      b += c.x + c.y;
    }
    const TileCut k = cut_tile(b - b0, piece, L.whole);
    if (k.full) atomicAdd(&s_cls[cls_full], k.full);
    if (k.items > k.full) atomicAdd(&s_cls[k.cls_rem], 1u);
  }
  __syncthreads();
  // First slot of each size class, largest class first. (A lane that added up the larger classes by
  // itself read the LDS 31 times in a row: 1.3 us of every frame's 11 to 8 us of this kernel.)
  if (threadIdx.x < 32) {
    const uint32_t n_own = s_cls[threadIdx.x];
    uint32_t upto = n_own;  // of this class and the larger ones
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) {
      const uint32_t y = __shfl_down(upto, d, 32);
      if ((int)threadIdx.x + d < 32) upto += y;
    }
    s_cur[threadIdx.x] = upto - n_own;
    if (threadIdx.x == 0) {
      const uint32_t n_items = upto;
      row_start[2 * n_tiles * nl] = (uint32_t)total;
      ctl->total_pairs = total;
      ctl->n_work = n_items < L.items_cap ? n_items : L.items_cap;
      uint32_t f = 0;
      if (total > L.pairs_cap) f |= CTL_PAIRS_OVERFLOW;
      if (n_items > L.items_cap) f |= CTL_ITEMS_OVERFLOW;
      if (f) atomicOr(&ctl->flags, f);
    }
  }
  __syncthreads();
  b = first;
  for (int t = t0; t < t1; t++) {
    const uint32_t cnt = tile_count(t);
    const TileCut k = cut_tile(cnt, piece, L.whole);
    if (k.items) {
      uint32_t split_slot = 0, full_slot = 0, rem_slot = 0;
      if (k.items > 1) {  // the tile's items merge their sums in a slot of the fixed-point merge buffer
        split_slot = atomicAdd(&s_nsplit, 1u);
        if (split_slot < L.split_cap) split_tiles[split_slot] = (uint32_t)t;
      }
      if (k.full) full_slot = atomicAdd(&s_cur[cls_full], k.full);
      if (k.items > k.full) rem_slot = atomicAdd(&s_cur[k.cls_rem], 1u);
      const uint32_t sid = tile_scene[t];
      put_items(items, L.items_cap, sid, (uint32_t)(t - descs[sid].tile_base), b, b + cnt, b + counts[t * nl].x, piece, k,
                split_slot, full_slot, rem_slot);
    }
    b += cnt;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    ctl->n_split = s_nsplit;
    if (s_nsplit > L.split_cap) atomicOr(&ctl->flags, (uint32_t)CTL_SPLIT_OVERFLOW);
  }
}

// Frames of more tiles: the row totals were scanned into row_start by a multi-block scan. Counts
// the items per size class. A workgroup sums its tiles' classes in LDS and adds each non-zero
// class to the global count once (one global atomic per tile on a handful of class counters
// serialises in the L2 when a frame has 1e5 tiles).
__global__ __launch_bounds__(256) void tile_classes_kernel(int n_tiles, const uint32_t* __restrict__ row_start,
                                                           BatchCtl* ctl, PlanLimits L) {
  __shared__ uint32_t s_cls[32];
  if (threadIdx.x < 32) s_cls[threadIdx.x] = 0u;
  __syncthreads();
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  const unsigned long long total = ctl->total_pairs;
  const uint32_t piece = piece_size(total, L);
  if (g < n_tiles) {
    const TileCut k = cut_tile(row_start[2 * (g + 1) * L.layers] - row_start[2 * g * L.layers], piece, L.whole);
    if (k.full) atomicAdd(&s_cls[31 - __clz(piece)], k.full);
    if (k.items > k.full) atomicAdd(&s_cls[k.cls_rem], 1u);
  }
  if (g == 0 && total > L.pairs_cap) atomicOr(&ctl->flags, (uint32_t)CTL_PAIRS_OVERFLOW);
  __syncthreads();
  if (threadIdx.x < 32 && s_cls[threadIdx.x]) atomicAdd(&ctl->class_count[threadIdx.x], s_cls[threadIdx.x]);
}

// Writes the work items of every tile into the slots of their size classes. The workgroup
// reserves its slots of each class, and its split-tile slots, with one global atomic each; a
// tile's items then take consecutive slots from the offsets its LDS atomics returned.
__global__ __launch_bounds__(256) void write_items_kernel(const SceneDesc* __restrict__ descs,
                                                          const uint32_t* __restrict__ tile_scene,
                                                          const uint32_t* __restrict__ row_start, int n_tiles,
                                                          BatchCtl* ctl, WorkItem* items, uint32_t* split_tiles,
                                                          PlanLimits L) {
  __shared__ uint32_t s_cnt[32], s_base[32], s_cls_base[32];
  __shared__ uint32_t s_nsplit, s_split_base;
  if (threadIdx.x < 32) {
    // first slot of each size class, largest class first
    uint32_t base = 0;
    for (int c = 31; c > (int)threadIdx.x; c--) base += ctl->class_count[c];
    s_cls_base[threadIdx.x] = base;
    s_cnt[threadIdx.x] = 0u;
  }
  if (threadIdx.x == 0) s_nsplit = 0u;
  if (blockIdx.x == 0 && threadIdx.x == 0) {  // the number of work items
    uint32_t n_items = 0;
    for (int c = 0; c < 32; c++) n_items += ctl->class_count[c];
    if (n_items > L.items_cap) atomicOr(&ctl->flags, (uint32_t)CTL_ITEMS_OVERFLOW);
    ctl->n_work = n_items < L.items_cap ? n_items : L.items_cap;
  }
  __syncthreads();
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t piece = piece_size(ctl->total_pairs, L);
  uint32_t b = 0, e = 0, mid = 0;
  TileCut k{0u, 0u, 0};
  if (g < n_tiles) {
    b = row_start[2 * g * L.layers];
    mid = row_start[2 * g * L.layers + 1];
    e = row_start[2 * (g + 1) * L.layers];
    k = cut_tile(e - b, piece, L.whole);
  }
  const int cls_full = 31 - __clz(piece);
  uint32_t off_full = 0, off_rem = 0, off_split = 0;
  if (k.full) off_full = atomicAdd(&s_cnt[cls_full], k.full);
  if (k.items > k.full) off_rem = atomicAdd(&s_cnt[k.cls_rem], 1u);
  if (k.items > 1) off_split = atomicAdd(&s_nsplit, 1u);
  __syncthreads();
  if (threadIdx.x < 32 && s_cnt[threadIdx.x])
    s_base[threadIdx.x] = s_cls_base[threadIdx.x] + atomicAdd(&ctl->class_cursor[threadIdx.x], s_cnt[threadIdx.x]);
  if (threadIdx.x == 32 && s_nsplit) s_split_base = atomicAdd(&ctl->n_split, s_nsplit);
  __syncthreads();
  if (k.items == 0) return;
  const uint32_t sid = tile_scene[g];
  uint32_t split_slot = 0;
  if (k.items > 1) {  // the tile's items merge their sums in a slot of the fixed-point merge buffer
    split_slot = s_split_base + off_split;
    if (split_slot < L.split_cap)
      split_tiles[split_slot] = (uint32_t)g;
    else
      atomicOr(&ctl->flags, (uint32_t)CTL_SPLIT_OVERFLOW);
  }
  put_items(items, L.items_cap, sid, (uint32_t)(g - descs[sid].tile_base), b, e, mid, piece, k, split_slot,
            k.full ? s_base[cls_full] + off_full : 0u, k.items > k.full ? s_base[k.cls_rem] + off_rem : 0u);
}

// ---- exclusive scan of u32 (block sums kept in u32; totals are checked on the host) ------
constexpr int kScanThreads = 256;
constexpr int kScanPer = 8;
constexpr int kScanBlock = kScanThreads * kScanPer;

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    uint32_t y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  return x;
}

// Block-level exclusive scan of kScanBlock elements; writes block total to sums[b]. With
// `total`: a block whose elements sum to 2^32 or more (its u32 total wrapped) sets bit 63 of
// *total, and the launch of a single block (the scan's top level, whose elements are the exact
// block totals of the level below) adds their 64-bit sum to *total.
__global__ __launch_bounds__(kScanThreads) void scan_block_kernel(const uint32_t* in, uint32_t* out,
                                                                  uint64_t n, uint32_t* sums,
                                                                  unsigned long long* total) {
  __shared__ uint32_t s_w[kScanThreads / 64];
  __shared__ unsigned long long s_w64[kScanThreads / 64];
  uint64_t base = (uint64_t)blockIdx.x * kScanBlock + (uint64_t)threadIdx.x * kScanPer;
  uint32_t v[kScanPer];
  uint32_t tot = 0;
  unsigned long long tot64 = 0;
#pragma unroll
  for (int i = 0; i < kScanPer; i++) {
    v[i] = (base + i < n) ? in[base + i] : 0u;
    uint32_t x = v[i];
    v[i] = tot;
    tot += x;
    tot64 += x;
  }
  if (total) {
    for (int d = 32; d > 0; d >>= 1) tot64 += __shfl_down(tot64, d, 64);
    if ((threadIdx.x & 63) == 0) s_w64[threadIdx.x >> 6] = tot64;
  }
  uint32_t incl = wave_incl_scan(tot);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 63) s_w[wave] = incl;
  __syncthreads();
  uint32_t wofs = 0;
  for (int w = 0; w < wave; w++) wofs += s_w[w];
  uint32_t excl = wofs + incl - tot;
#pragma unroll
  for (int i = 0; i < kScanPer; i++)
    if (base + i < n) out[base + i] = v[i] + excl;
  if (threadIdx.x == kScanThreads - 1 && sums) sums[blockIdx.x] = excl + tot;
  if (total && threadIdx.x == 0) {
    unsigned long long b = 0;
    for (int w = 0; w < kScanThreads / 64; w++) b += s_w64[w];
    if (b > 0xffffffffull) atomicOr(total, 1ull << 63);
    if (gridDim.x == 1 && b) atomicAdd(total, b);
  }
}

__global__ __launch_bounds__(kScanThreads) void scan_add_kernel(uint32_t* out, uint64_t n,
                                                                const uint32_t* block_ofs) {
  uint64_t base = (uint64_t)blockIdx.x * kScanBlock;
  uint32_t add = block_ofs[blockIdx.x];
  for (int i = threadIdx.x; i < kScanBlock; i += kScanThreads)
    if (base + i < n) out[base + i] += add;
}

// ---- tile accumulation -----------------------------------------------------------------
// The LDS tile accumulates in 64-bit fixed point: FP32 LDS atomics (ds_add_f32) run ~30x
// slower than 64-bit integer ones (ds_add_u64) on gfx950. A sample's anti-aliasing weight f
// is quantised to wq = round(f * 2^20) and the pixel pair gets (2^20 - wq) * cq and wq * cq,
// where cq = round(c * 2^G) is the channel value in fixed point: the two deposits sum to
// exactly 2^20 * cq. Integer sums do not depend on the order of the deposits, so a frame's
// image is the same bits whatever the batch, the work split or the replay: a tile whose
// pairs are split over several work items adds its exact sums into a 64-bit merge slot, and
// every pixel's sum is converted to FP32 once, by the same expression, whether the tile was
// split or not. (That is the one-channel-per-word form; two-channel scenes split each cq
// between the pixel pair with deposit2.)
constexpr int kWBits = 20;
constexpr int kWOne = 1 << kWBits;
constexpr int kSlotU64 = kMergeSlotU64;
static_assert(kSlotU64 >= 4 * kTileMax * kTileMax && kSlotU64 >= 2 * kMaxHues * kTileMax * kTileMax,
              "a merge slot holds 4 channel planes, or 2 planes per hue, of the largest tile");
// A pair entry is the segment's index in its scene with the segment's major axis in bit 31
// (1 = x); kNoPair marks lanes past the end of an item.
constexpr uint32_t kPairIndex = 0x7FFFFFFFu;
constexpr uint32_t kNoPair = 0xFFFFFFFFu;

// 2^G must stay a finite, normal float: G <= 126 (a colour as faint as 1e-15 has an alpha
// deposit a * a = 1e-30 under the default blend, which wants G of about 122 (two channels per
// word) to 128 (one) for its full precision; at G = 126 one deposit still has about 2^26 levels).
// Below 2^-149 the scale is 0 and such colours deposit nothing.
__device__ __forceinline__ int clamp_fixed_bits(int G) { return G < -250 ? -250 : (G > 126 ? 126 : G); }

// floor(log2(a / b)) of positive finite a and b, exactly (no rounded quotient or logarithm):
// with a = ma * 2^ea and b = mb * 2^eb (mantissas in [1/2, 1)) the quotient is
// (ma / mb) * 2^(ea - eb), and ma / mb lies in [1, 2) when ma >= mb, in (1/2, 1) otherwise.
__device__ __forceinline__ int floor_log2_ratio(double a, double b) {
  int ea, eb;
  const double ma = frexp(a, &ea), mb = frexp(b, &eb);
  return ea - eb - (ma < mb ? 1 : 0);
}

// G of channel c of a scene's fixed point, from the scene's colour bound for that channel and
// its segment count only (never from a buffer capacity, so it is the same alone or in any
// batch). Each channel has its own scale: with the default blend alpha deposits a * a while
// RGB deposit the colour, so for bright colours the two differ by many orders of magnitude.
// A segment deposits at most once into a given pixel, so every partial sum of a pixel is
// bounded by n * 2^20 * max|cq|; with n <= 2^lb and G + log2(bound) <= 41 - lb that stays
// below 2^62, and |cq| <= 2^29. bound = max|colour| * max|blend factor of the channel|.
__device__ __forceinline__ int scene_fixed_bits(const SceneDesc& D, int c) {
  const double m = (double)D.color_max;
  const double bound = m * (double)D.factor_max[c];
  if (!(bound > 0.0) || !(bound < 1e300)) return 30;
  const uint64_t n = scene_segments(D);
  const int lb = n > 1 ? 64 - __clzll((long long)(n - 1)) : 0;  // n <= 2^lb
  const int room = (42 - lb) < 30 ? 42 - lb : 30;
  // floor(room - log2(bound)) - 1, exactly: room is an integer
  const int G = room + floor_log2_ratio(1.0, bound) - 1;
  return clamp_fixed_bits(G);
}

// Packed deposits: two channels per 64-bit LDS word, (R, G) and (B, A) as 32-bit fields, for
// scenes whose every deposit is non-negative (SCENE_PACKED). A sample's value of channel c is
// cq = round(v * 2^G) <= lim <= 2^22 and its two deposits add up to cq; a pair deposits at
// most once into a pixel, so the n pairs of one item keep a field below n * lim <= 2^32 - 1
// and no carry crosses into the other field. Every item of a tile takes G from n = min(pairs
// of the tile, kPackedPiece) (no item holds more), so the items' sums add up in the merge slot
// and the launch tuning changes no bit.
constexpr uint32_t kPackLevels = 1u << 22;
__device__ __forceinline__ uint32_t packed_levels(uint32_t n) {
  const uint32_t q = 0xFFFFFFFFu / (n > 1u ? n : 1u);  // floor((2^32 - 1) / n)
  return q < kPackLevels ? q : kPackLevels;
}
__device__ __forceinline__ int packed_fixed_bits(double bound, uint32_t n) {
  if (!(bound > 0.0) || !(bound < 1e300)) return 0;
  const double lim = (double)packed_levels(n);
  // the largest G with bound * 2^G <= lim - 1/2: v <= bound, rounded once in FP32, keeps
  // v * 2^G + 1/2 below lim + 1
  return clamp_fixed_bits(floor_log2_ratio(lim - 0.5, bound));
}

__device__ __forceinline__ int packed_fixed_bits(const SceneDesc& D, int c, uint32_t n) {
  return packed_fixed_bits((double)D.color_max * (double)D.factor_max[c], n);
}

// Hue deposits (SCENE_HUES): a segment's colour is s times its light's hue, so its samples deposit
// two numbers, s (the brightest channel's value) and the alpha deposit a * a, as the fields of ONE
// word in the plane of its hue, where (R, G, B, A) take two words; the hue's RGB ratios come in
// when a pixel's sums are converted. Half the LDS adds per sample, of which the walk is bound
// (tile walk of the 1M-ray frame, us: 915 -> 776). The
// fields' scales follow the packed rule with the hue's own bounds, so the brightest channel keeps
// the levels it had and the others gain some.
// What a tile's pairs and pixels need of each hue. It sits in LDS: the pairs of a batch mix hues
// (a lane reads its own), and as registers of every wave it spilled the walk.
struct HueScale {
  double us, ua;     // 2^-G of the two fields
  double ratio[3];   // the hue's RGB over its brightest channel
  float ss, sa;      // 2^G
  int32_t ch;        // the brightest channel
  int32_t pad;
};
__device__ __forceinline__ HueScale hue_scale(const SceneDesc& D, int f, uint32_t n) {
  HueScale h{};
  if (f < D.n_hues) {
    const double a = (double)D.hue_bound[f][1];
    const int gs = packed_fixed_bits((double)D.hue_bound[f][0], n), ga = packed_fixed_bits(a * a, n);
    h.us = __builtin_ldexp(1.0, -gs);
    h.ua = __builtin_ldexp(1.0, -ga);
    h.ss = __builtin_ldexpf(1.0f, gs);
    h.sa = __builtin_ldexpf(1.0f, ga);
    for (int k = 0; k < 3; k++) h.ratio[k] = D.hue_ratio[f][k];
    h.ch = D.hue_ch[f];
  }
  return h;
}

// Adds hue h's exact sums s and a of a pixel to p: ratio s 2^-Gs and a 2^-Ga, in FP64 (rounded to
// FP32 once, after the last hue). The one expression of the tile flush and of the merge of split
// tiles.
__device__ __forceinline__ void hue_add(double (&p)[4], const HueScale& h, unsigned long long s, unsigned long long a) {
  const double v = (double)s * h.us;
  p[0] = __builtin_fma(v, h.ratio[0], p[0]);
  p[1] = __builtin_fma(v, h.ratio[1], p[1]);
  p[2] = __builtin_fma(v, h.ratio[2], p[2]);
  p[3] = __builtin_fma((double)a, h.ua, p[3]);
}

// Whether the items of a split tile of two fields to a word add the words as they are to the merge
// slot: with the whole tile's pairs in the fields' bound no sum carries. (n: its pairs, at most
// kPackedPiece.) Half the adds and loads: every item of a tile of nearly full pixels took 17 us for
// them where 256 do so at a time (60033 string-mod lines of two colours, us of walk and merge:
// 135 + 25 and 117 + 23).
__device__ __forceinline__ bool slot_words(uint32_t n) { return n < kPackedPiece; }

// Run weights (SCENE_RUNS). A run's segments have one colour, so a tile sums one number per pixel
// and run: the weights of the deposits, each sample's Q cut into round(fr Q) at pixel jl + 1 and the
// rest at jl, as 32-bit words (a pair deposits at most once into a pixel, so n pairs keep a word
// below n Q <= 2^32 - 1). The colours come in when a layer's sums are converted: channel c of run f
// adds weight times C = round(value 2^K_c), exact 64-bit products, so neither the split of a
// tile's list into items nor the order of anything changes a bit. C <= 2^30, less where the
// tile's pairs would pass 2^62 in total. A deposit costs two 32-bit adds where two-channel words
// take four of 64 bits, no colour is loaded, and instruction issue instead of the LDS is what bounds the
// walk (1.6M segments in 16 runs at 4096x4096, 78M pairs: 3727 us by colours, 2168 us so). Q has all
// the levels that the word has room for, no fewer than the brightest channel by colours, and no
// colour is rounded to them. (Q a power of two, a field of the place's bits cut out: 2122 us, but
// up to half the levels of a channel. Error of 16 x 20000 lines against FP64, rel L1: 7.6e-7 by
// colours, 2.1e-7 with powers of two, 1.6e-7 so.)
constexpr int kFxBits = 22;  // of a sample's place below the pixel; |slope| 2^22 is a 24-bit number
__device__ __forceinline__ uint32_t run_weight(uint32_t n) {
  const uint32_t Q = 0xFFFFFFFFu / (n > 1u ? n : 1u);
  return Q < (1u << kFxBits) ? Q : 1u << kFxBits;
}
// round(fr Q), to nearest even, of the place M: with the fraction as the mantissa of 1 + fr / 2 and
// the integer 2 Q as the bits of a denormal float (2 Q <= 2^23, which the bits hold as well), the
// FMA's one rounding is to a multiple of 2^-149 (see mul_frac).
__device__ __forceinline__ uint32_t cut_weight(int M, uint32_t Q) {
  const uint32_t one_half_fr = ((uint32_t)M & ((1u << kFxBits) - 1u)) | 0x3f800000u;
  const float q2 = __builtin_bit_cast(float, 2u * Q);
  return __builtin_bit_cast(uint32_t, __builtin_fmaf(__builtin_bit_cast(float, one_half_fr), q2, -q2));
}
// K of channel c in a tile of n pairs.
__device__ __forceinline__ int run_color_bits(const SceneDesc& D, int c, uint32_t n) {
  const double bound = (double)D.color_max * (double)D.factor_max[c];
  if (!(bound > 0.0) || !(bound < 1e300)) return 0;
  const uint32_t over = n / kPackedPiece;  // n Q <= 2^32 (over + 1)
  return 30 - (over ? 32 - __clz((int)over) : 0) - 1 - floor_log2_ratio(bound, 1.0);
}
__device__ __forceinline__ uint32_t run_color(float v, int K) {
  const double x = __builtin_ldexp((double)v, K);
  return x > 0.0 ? (uint32_t)__builtin_rint(x < 1073741824.0 ? x : 1073741824.0) : 0u;  // (2^30: an overflown product)
}

// One packed channel value of a sample: cq = round(max(v, 0) * 2^G), the low bits of one FMA against
// 2^23 (round to nearest even; cq <= 2^22 leaves the exponent alone; a NaN deposits nothing).
constexpr float kMagic = 8388608.0f;  // 2^23
__device__ __forceinline__ uint32_t pack_q(float v, float scale) {
  return __builtin_bit_cast(uint32_t, __builtin_fmaf(__builtin_fmaxf(v, 0.0f), scale, kMagic)) & 0x7FFFFFu;
}
// Of a product of two numbers, which may be infinite in FP32 where the bound, in FP64, is finite: then
// all the levels (top: 2^23 + packed_levels), so that the pixel's sum overflows and not vanishes.
__device__ __forceinline__ uint32_t pack_q(float v, float scale, float top) {
  const float x = __builtin_fminf(__builtin_fmaf(__builtin_fmaxf(v, 0.0f), scale, kMagic), top);
  return __builtin_bit_cast(uint32_t, x) & 0x7FFFFFu;
}

// round(f * q) for 0 <= f < 1 and an integer q < 2^23, as one multiplication: the integer's bits
// are the denormal float q * 2^-149, whose product with f rounds (to nearest even) to a multiple
// of 2^-149, so its bits are the rounded integer. Never more than q.
__device__ __forceinline__ uint32_t mul_frac(float f, uint32_t q) {
  return __builtin_bit_cast(uint32_t, f * __builtin_bit_cast(float, q));
}

// The two-channel deposits of one sample at minor position m (fraction fr = m - floor(m))
// into t (pixel jl of planes 0 and 1) and t + T (pixel jl + 1), channel values q0..q3 from
// pack_q. Pixel jl + 1 takes r = round(fr q) and pixel jl the rest, q - r: the two deposits
// always add up to exactly q, at one multiplication and one subtraction per channel (the form
// before, an FMA against 2^23 and the subtractions of its exponent bits, took 14 instructions
// for four channels and the weights where this takes 8; tile walk, us: 1M-ray frame 950 -> 915,
// 1.6M segments at 4096x4096 4440 -> 4330; what binds it is the LDS, see the stream walk).
template <int T, int STRIDE>
__device__ __forceinline__ void deposit2(unsigned long long* t, float m, uint32_t q0, uint32_t q1, uint32_t q2,
                                         uint32_t q3) {
  const float fr = __builtin_amdgcn_fractf(m);
  const uint32_t r0 = mul_frac(fr, q0), r1 = mul_frac(fr, q1), r2 = mul_frac(fr, q2), r3 = mul_frac(fr, q3);
  atomicAdd(t, (unsigned long long)(q1 - r1) << 32 | (q0 - r0));
  atomicAdd(t + STRIDE, (unsigned long long)(q3 - r3) << 32 | (q2 - r2));
  atomicAdd(t + T, (unsigned long long)r1 << 32 | r0);
  atomicAdd(t + T + STRIDE, (unsigned long long)r3 << 32 | r2);
}

// The hue deposits of one sample: (s, a * a) as one word into t (pixel jl of the hue's plane) and
// t + T.
template <int T>
__device__ __forceinline__ void deposit1(unsigned long long* t, float m, uint32_t qs, uint32_t qa) {
  const float fr = __builtin_amdgcn_fractf(m);
  const uint32_t r0 = mul_frac(fr, qs), r1 = mul_frac(fr, qa);
  atomicAdd(t, (unsigned long long)(qa - r1) << 32 | (qs - r0));
  atomicAdd(t + T, (unsigned long long)r1 << 32 | r0);
}

// The value one sample of colour channel c adds per unit weight: +-c * factor (BlendCode).
__device__ __forceinline__ float blend_value(uint32_t code, float c, float a, float k) {
  float f;
  switch (code & 7u) {
    case BC_ZERO: f = 0.0f; break;
    case BC_ONE: f = 1.0f; break;
    case BC_SRC: f = c; break;
    case BC_ONE_MINUS_SRC: f = 1.0f - c; break;
    case BC_SRC_ALPHA: f = a; break;
    case BC_ONE_MINUS_SRC_ALPHA: f = 1.0f - a; break;
    case BC_CONST: f = k; break;
    default: f = 1.0f - k; break;
  }
  const float v = c * f;
  return (code & BC_NEGATE) ? -v : v;
}

__device__ __forceinline__ int bcast_i(int v, int lane) {
  return __builtin_amdgcn_readlane(v, lane);
}
__device__ __forceinline__ float bcast_f(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ __forceinline__ double bcast_d(double v, int lane) {
  long long b = __builtin_bit_cast(long long, v);
  int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), lane);
  int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (long long)(unsigned)lo);
}

__device__ __forceinline__ int fx(float v, float scale) { return (int)__builtin_rintf(v * scale); }

// FP32 accumulator -> RGBA16F, round to nearest even, alpha + 1 (the target's clear alpha,
// renderer.rs:175). The one expression of the resolve pass and the fused flushes.
__device__ __forceinline__ ushort4 resolve_px(const float4 a) {
  ushort4 o;
  o.x = __builtin_bit_cast(unsigned short, (_Float16)a.x);
  o.y = __builtin_bit_cast(unsigned short, (_Float16)a.y);
  o.z = __builtin_bit_cast(unsigned short, (_Float16)a.z);
  o.w = __builtin_bit_cast(unsigned short, (_Float16)(a.w + 1.0f));
  return o;
}

// In-place transpose of the first `planes` TxT planes (STRIDE elements apart), (r, c) <-> (c, r). Job j of planes * T/2
// is plane j / (T/2) and diagonal pair d = j % (T/2) + 1: lanes 0 .. T-1-d swap the elements of
// diagonal c - r = d, lanes T-d .. T-1 those of diagonal T - d (d < T/2; diagonal T/2 takes lanes
// 0 .. T/2-1 alone; lanes from T on idle). Every element off the main diagonal is swapped
// exactly once, and the lanes' addresses step by T + 1 elements, which keeps the swaps free of
// bank conflicts.
template <int T, int STRIDE, int WAVES, typename W>
__device__ __forceinline__ void transpose_tile(W* t, int planes, int wave, int lane) {
  constexpr int H = T / 2;
  for (int j = wave; j < planes * H; j += WAVES) {
    const int d = (j % H) + 1;
    W* pl = t + (j / H) * STRIDE;
    const bool first_diag = lane < T - d;
    const int r = first_diag ? lane : lane - (T - d);
    const int c = first_diag ? lane + d : r + (T - d);
    if (lane < T && (d < H || lane < H)) {
      const int a = r * T + c, b = c * T + r;
      const W va = pl[a], vb = pl[b];
      pl[a] = vb;
      pl[b] = va;
    }
  }
}

// Items of at most this many pairs claim their successor when they start (see the item loop).
constexpr uint32_t kEarlyClaimPairs = 8192;

// One persistent workgroup per (tile, pair range) item. Each wave takes 64 pairs at a time:
// lane l loads pair l's segment and computes its sample range inside the tile plus the
// tile-relative FP32 parameters of its samples. Two-channel frames at T = 64 with 1024-thread
// workgroups then walk the batch as one stream of samples, 128 per step (see the stream
// comment in the walk; not under blends with factors when colours vary along a segment); other
// shapes walk the pairs one after another with one sample per lane, reading the pair's setup
// from scalar registers.
//
// An item is walked twice: first its y-major pairs with the tile held transposed (pixel
// (row y, column x) at x * T + y), then, after an in-place transpose, its x-major pairs with
// the tile row-major (y * T + x). Either way a deposit of the sample at major offset q and
// minor pixel m lands at m * T + q: the lanes of one deposit instruction cover consecutive
// addresses for every slope (a single padded layout serves one orientation's walks without
// conflicts but stacks the lanes of the other's diagonal walks in a few banks).
//
// A pair's sample positions are anchored on the tile's column 0: the sample of column c is at
// m(c) = m_first + c * slope in FP32 relative to the tile's minor origin, m_first rounded once
// from FP64; both walks evaluate exactly this. Two tiles sharing a sample (its two deposits on
// either side of a tile edge) differ only by FP32 rounding (< 1e-5 px).
//
// T is the tile edge of the frame (64 or 32; with 32 a pair has at most 32 samples in the
// tile and lanes 32..63 only set up pairs). A scene with SCENE_PACKED (all its deposits
// non-negative) keeps two channels per 64-bit word in the first two planes
// (packed_fixed_bits); one with SCENE_HUES a word per hue; other scenes one channel per word in
// four. RUNS: the kernel of a SCENE_RUNS frame, whose tiles go through the layers' lists one after
// another with a 32-bit weight plane per run, and keep the pixels' channel sums in registers from
// layer to layer. PACKED_ONLY: every scene of the frame has SCENE_PACKED, so the LDS tile holds two
// planes only (half the LDS: two 512-thread workgroups share a compute unit at T = 64), or three in the
// 1024-thread kernel, which serves up to three hues.
enum WalkMode { WALK_COLOR, WALK_VERTEX_COLORS, WALK_VERTEX_STREAM, WALK_HUES, WALK_RUNS };
template <int T, bool PACKED_ONLY, int BLOCK, bool RUNS>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4)))
void tile_accum_kernel(const SceneDesc* __restrict__ descs,
                                                          const uint32_t* __restrict__ pairs,
                                                          const WorkItem* __restrict__ items,
                                                          const uint32_t* __restrict__ row_start,
                                                          unsigned long long* split_fx, BatchCtl* ctl,
                                                          uint32_t count_work) {
  constexpr int kPlane = T * T;                         // pixels of a plane
  constexpr int kGuard = 2;                             // guard rows on each side of a plane
  constexpr int kStride = (T + 2 * kGuard) * T;         // elements from one plane to the next
  constexpr bool kStreamKernel = PACKED_ONLY && T == 64 && BLOCK == 1024;
  static_assert(!RUNS || kStreamKernel, "runs are walked as streams");
  constexpr bool kHueKernel = T == 64 && BLOCK == 1024 && !RUNS;  // the kernels frames with hues run
  constexpr int kPlanes = kStreamKernel ? 3 : PACKED_ONLY ? 2 : 4;
  static_assert(!kHueKernel || kPlanes >= kMaxHues, "a plane per hue");
  __shared__ unsigned long long s_tile[kPlanes * kStride];
  // the workgroup's next item and its index, double-buffered: thread 0 claims and loads item
  // i + 1 while item i runs and writes it into the other buffer
  __shared__ WorkItem s_w[2];
  __shared__ uint32_t s_item[2];
  __shared__ uint32_t s_batch[2];  // next batch of 64 pairs, per phase
  unsigned long long* const tile = s_tile + kGuard * T;  // row 0 of plane 0
  // RUNS: planes of 32-bit words in the same memory, a weight plane per run of the layer
  static_assert(2 * kPlanes >= kRunPlanes || !RUNS, "a plane per run");
  uint32_t* const tile32 = reinterpret_cast<uint32_t*>(s_tile) + kGuard * T;
  __shared__ uint32_t s_run[RUNS ? kRunPlanes : 1][4];  // the runs' colours (run_color)
  constexpr int kWaves = BLOCK / 64;
  // Sample-stream walk (two-channel frames, T = 64, one workgroup per compute unit; with a colour
  // per vertex under the default blend, whose channel values need no factors): each wave lays the
  // samples of its 64 pairs end to end and walks that stream two samples to a lane, 128 per step,
  // every lane busy, instead of one pair per step. Per wave: a record per
  // pair with samples plus an empty one (two uint4 each) and a start bit per stream position.
  __shared__ HueScale s_hue[kHueKernel ? kMaxHues : 1];
  constexpr int kRecs = 66, kMaskWords = 64;
  __shared__ uint4 s_rec[kStreamKernel ? kWaves * kRecs * 2 : 1];
  __shared__ unsigned long long s_mask[kStreamKernel ? kWaves * kMaskWords : 1];
  const int lane = threadIdx.x & 63;
  const float lane_f = (float)lane;
  const int wave = threadIdx.x >> 6;
  if (ctl->flags & kCtlStop) return;  // a buffer overflowed: the host reruns the frame
  const uint32_t n_items = ctl->n_work;
  unsigned long long wave_samples = 0;  // wave-uniform
  unsigned long long wave_atomics = 0;  // wave-uniform: LDS atomic instructions of the walk steps
  if (threadIdx.x == 0) {
    s_item[0] = blockIdx.x;
    if (blockIdx.x < n_items) s_w[0] = items[blockIdx.x];
  }
  __syncthreads();
  for (int buf = 0;; buf ^= 1) {
    const uint32_t it = __builtin_amdgcn_readfirstlane(s_item[buf]);
    if (it >= n_items) break;
    WorkItem W;
    W.scene = __builtin_amdgcn_readfirstlane(s_w[buf].scene);
    W.tile = __builtin_amdgcn_readfirstlane(s_w[buf].tile);
    W.begin = __builtin_amdgcn_readfirstlane(s_w[buf].begin);
    W.end = __builtin_amdgcn_readfirstlane(s_w[buf].end);
    W.mid = __builtin_amdgcn_readfirstlane(s_w[buf].mid);
    W.tile_pairs = __builtin_amdgcn_readfirstlane(s_w[buf].tile_pairs);
    W.slot = __builtin_amdgcn_readfirstlane(s_w[buf].slot);
    // Thread 0 claims the next item and loads it before the flush, so that the loop's next trip
    // starts from LDS. A small item claims at its start (the claim returns while it runs); a
    // large one at its flush, since a workgroup holding a claimed item while its current one
    // runs for long leaves others idle at the end of the launch. After the last item every
    // workgroup claims one more, past the end; a frame with an item per workgroup or fewer claims
    // none.
    const bool claim_early = W.end - W.begin <= kEarlyClaimPairs;
    uint32_t it_next = 0;
    auto claim = [&]() {
      if (threadIdx.x == 0) it_next = n_items > gridDim.x ? atomicAdd(&ctl->work_cursor, 1u) + gridDim.x : n_items;
    };
    if (claim_early) claim();
    // publishes the next item for the loop's next trip (before the workgroup's last barrier)
    auto publish_next = [&](const WorkItem& wn) {
      if (threadIdx.x == 0) {
        s_item[buf ^ 1] = it_next;
        s_w[buf ^ 1] = wn;
      }
    };
    auto load_next = [&]() {
      WorkItem wn{};
      if (threadIdx.x == 0 && it_next < n_items) wn = items[it_next];
      return wn;
    };
    const bool split = (W.scene & kSplitBit) != 0;
    const SceneDesc& D = descs[W.scene & ~kSplitBit];
    const AccumView v = D.view;
    const float4* __restrict__ pos = gen(D.seg_pos);
    const float4* __restrict__ col0 = gen(D.seg_col);
    const float4* __restrict__ col1 = gen(D.seg_col1);
    const uint64_t* __restrict__ keys = gen(D.seg_key);
    float4* accum = gen(D.accum);
    // two channels per word; uniform
    const bool two_ch = PACKED_ONLY || (D.flags & SCENE_PACKED) != 0;
    const bool hues = kHueKernel && (D.flags & SCENE_HUES) != 0;
    const int n_hues = hues ? D.n_hues : 0;
    if (kHueKernel && hues && threadIdx.x < kMaxHues) s_hue[threadIdx.x] = hue_scale(D, threadIdx.x, W.tile_pairs);
    int G[4] = {0, 0, 0, 0};
    const uint32_t n_layers = RUNS ? D.row_stride : 1u;
    const uint32_t* const tile_rows = row_start + 2u * n_layers * W.tile;
    int K[4] = {0, 0, 0, 0};
    const uint32_t wq = RUNS ? run_weight(W.tile_pairs) : 0u;  // a sample's weight
    unsigned long long acc[RUNS ? T * T / BLOCK : 1][4] = {};
    if constexpr (RUNS) {
      const uint32_t nt = tile_rows[2u * n_layers] - tile_rows[0];
#pragma unroll
      for (int c = 0; c < 4; c++) K[c] = run_color_bits(D, c, nt);
    }
    if (RUNS || hues) {
      // (the channels' scales are not used)
    } else if (two_ch) {
#pragma unroll
      for (int c = 0; c < 4; c++) G[c] = packed_fixed_bits(D, c, W.tile_pairs);
    } else {
#pragma unroll
      for (int c = 0; c < 4; c++) G[c] = scene_fixed_bits(D, c);
    }
    const float cs0 = __builtin_ldexpf(1.0f, G[0]), cs1 = __builtin_ldexpf(1.0f, G[1]);
    const float cs2 = __builtin_ldexpf(1.0f, G[2]), cs3 = __builtin_ldexpf(1.0f, G[3]);
    const float q_top = kMagic + (float)packed_levels(W.tile_pairs);
    const uint32_t bc = __builtin_amdgcn_readfirstlane(D.blend_code);
    const uint32_t bc0 = bc & 15u, bc1 = (bc >> 4) & 15u, bc2 = (bc >> 8) & 15u, bc3 = (bc >> 12) & 15u;
    const float bk0 = D.blend_k[0], bk1 = D.blend_k[1], bk2 = D.blend_k[2], bk3 = D.blend_k[3];
    const int tx = (int)(W.tile % (uint32_t)v.tiles_x);
    const int ty = (int)(W.tile / (uint32_t)v.tiles_x);
    const int x0 = tx * T, y0 = ty * T;
    // the frame clears and resolves the image here: the flush writes the accumulator and the
    // RGBA16F target instead of adding to a cleared accumulator
    const bool whole = (D.flags & SCENE_FRESH_IMAGE) != 0;
    if (W.begin == W.end) {  // a tile without pairs in such a frame: its cleared pixels
      const WorkItem wn = load_next();
      ushort4* out16 = gen(D.out16);
      for (int k = threadIdx.x; k < T * T; k += BLOCK) {
        const int gx = x0 + (k % T), gy = y0 + (k / T);
        if (gx >= v.width || gy >= v.height) continue;
        const size_t px = (size_t)gy * v.width + gx;
        const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
        accum[px] = z;
        out16[px] = resolve_px(z);
      }
      publish_next(wn);
      __syncthreads();
      continue;
    }
    for (uint32_t layer = 0; layer < n_layers; layer++) {
    uint32_t r_beg = W.begin, r_end = W.end;  // the item's part of the layer's list
    // the list holds its y-major pairs before `mid`, its x-major pairs from there
    uint32_t mid = W.mid;
    int planes = hues ? n_hues : two_ch ? 2 : 4;
    uint32_t run1 = 0, run2 = 0, run3 = 0, run4 = 0, run5 = 0;  // RUNS: the layer's first segments
    if constexpr (RUNS) {
      const uint32_t lb = tile_rows[2u * layer], le = tile_rows[2u * layer + 2u];
      mid = tile_rows[2u * layer + 1u];
      r_beg = r_beg > lb ? r_beg : lb;
      r_end = r_end < le ? r_end : le;
      if (r_beg >= r_end) continue;
      const SceneDesc& DL = descs[layer];
      pos = gen(DL.seg_pos);
      planes = DL.n_runs;
      static_assert(kRunPlanes == 6, "run1 .. run5");
      run1 = DL.run_first[1];
      run2 = DL.run_first[2];
      run3 = DL.run_first[3];
      run4 = DL.run_first[4];
      run5 = DL.run_first[5];
      if (threadIdx.x < kRunPlanes * 4) {
        const int f = threadIdx.x >> 2, c = threadIdx.x & 3;
        const uint32_t code = (bc >> (4 * c)) & 15u;
        const float v = blend_value(code, DL.run_color[f][c], DL.run_color[f][3], DL.blend_k[c]);
        s_run[f][c] = run_color(v, c == 0 ? K[0] : c == 1 ? K[1] : c == 2 ? K[2] : K[3]);
      }
      // (a thread zeroes and converts the same pixels, so the layer before needs no barrier here;
      // s_run's readers have all passed the barriers of this layer's walk only after this write)
      for (int k = threadIdx.x; k < planes * kPlane; k += BLOCK) tile32[(k / kPlane) * kStride + k % kPlane] = 0u;
    } else {
      for (int k = threadIdx.x; k < planes * kPlane; k += BLOCK) tile[(k / kPlane) * kStride + k % kPlane] = 0ull;
    }
    if (threadIdx.x == 0) s_batch[0] = s_batch[1] = 2u * kWaves;
    __syncthreads();
    for (int phase = 0; phase < 2; phase++) {  // 0: y-major pairs, 1: x-major pairs
      const uint32_t pb = phase ? (r_beg > mid ? r_beg : mid) : r_beg;
      const uint32_t pe = phase ? r_end : (r_end < mid ? r_end : mid);
      const uint32_t n_batches = pe > pb ? (pe - pb + 63u) >> 6 : 0u;
      // an empty phase deposits nothing: without y-major pairs the tile stays zero, so it
      // needs no transpose either
      if (n_batches == 0u) continue;
      // the tile's place on this phase's axes, and its last column inside the image
      const double maj0 = (double)(phase ? x0 : y0), min0 = (double)(phase ? y0 : x0);
      const int cols = (phase ? v.width : v.height) - (phase ? x0 : y0);
      const double last_col = (double)((cols < T ? cols : T) - 1);
      // pair entry of this lane in batch b, kNoPair past the phase's end
      auto entry = [&](uint32_t b) -> uint32_t {
        const uint32_t pi = pb + b * 64u + (uint32_t)lane;
        return b < n_batches && pi < pe ? pairs[pi] : kNoPair;
      };
      // Batches of 64 pairs come from the phase's counter in LDS, so the waves of an item end
      // a phase together whatever the lengths of their pairs' runs. Each wave works two
      // batches ahead: while it walks batch b0, the end points and colours of b1 and the
      // pair entries of b2 are in flight.
      auto fetch = [&](uint32_t e, float4& p, float4& ca, float4& cb) {
        if (e != kNoPair) {
          const uint32_t s = e & kPairIndex;
          p = pos[s];
          if constexpr (RUNS) return;  // (a run's colour comes in with its sums)
          ca = col0[s];
          if (col1) cb = col1[s];
          if (n_hues > 1) {  // (such a scene has no col1: the key travels in its place)
            const uint64_t k = keys[s];
            cb.x = __uint_as_float((uint32_t)k);
            cb.y = __uint_as_float((uint32_t)(k >> 32));
          }
        }
      };
      uint32_t taken = 0;  // lane 0: the counter's previous value
      // One batch: set up the current batch's pairs from their loaded end points and colours,
      // issue the loads of the next batch and the pair entries of the one after, then walk.
      // mode_tag: a colour per segment, a colour per vertex, or hues (compiled apart, so that
      // with one colour per segment a pair's channel values stay in scalar registers).
      auto step = [&](auto mode_tag, const uint32_t e_cur, const float4& p_cur, const float4& a_cur,
                      const float4& c_cur, const uint32_t e_nxt, float4& p_nxt, float4& a_nxt, float4& c_nxt,
                      uint32_t& b_aft, uint32_t& e_aft) {
        constexpr bool kVS = decltype(mode_tag)::value == WALK_VERTEX_STREAM;
        constexpr bool kVC = kVS || decltype(mode_tag)::value == WALK_VERTEX_COLORS;
        constexpr bool kHues = decltype(mode_tag)::value == WALK_HUES;
        constexpr bool kRuns = decltype(mode_tag)::value == WALK_RUNS;
        int fx_m = 0, fx_s = 0;  // kRuns: m at the tile's middle column and the slope, times 2^kFxBits
        // ---- per-lane setup of one pair of the current batch ----
        int packed = 0;  // n | q0 << 8 | vertex colours << 17 | negative colour << 18
        float m_first = 0.f, slope = 0.f, s_first = 0.f, ds = 0.f;
        float4 ca = make_float4(0.f, 0.f, 0.f, 0.f), dc = ca;
        int cq0 = 0, cq1 = 0, cq2 = 0, cq3 = 0;
        // A pair's segment deposits (the binning listed it), its major axis is the phase's: no test
        // of either here. The sample range and the line are FP64; the samples whose deposits can
        // reach the tile's rows, m in [-1, T), are cut out in FP32, with a margin of 0.02 px
        // (m_first and the reciprocal are off by some 1e-5 px at most; a sample kept for the margin
        // deposits into guard rows). About 100 instructions; in FP64 and 64-bit integers throughout,
        // with divisions, it was 300, as much as a dozen walk steps (tile walk, us: 1M-ray frame
        // 776 -> 704, 1.6M segments at 4096x4096 4330 -> 4170).
        if (e_cur != kNoPair) {
          const float4 pc = p_cur;
          double M0, M1, m0, m1;
          if (phase) {
            M0 = ((double)pc.x - v.left) * v.sx;
            m0 = (v.top - (double)pc.y) * v.sy;
            M1 = ((double)pc.z - v.left) * v.sx;
            m1 = (v.top - (double)pc.w) * v.sy;
          } else {
            m0 = ((double)pc.x - v.left) * v.sx;
            M0 = (v.top - (double)pc.y) * v.sy;
            m1 = ((double)pc.z - v.left) * v.sx;
            M1 = (v.top - (double)pc.w) * v.sy;
          }
          double lo, hi;
          sample_span(M0, M1, lo, hi);
          // columns of the tile (and the image); both in [-1, T] before the conversions
          int a = (int)__builtin_fmin(__builtin_fmax(lo - maj0, 0.0), (double)T);
          int b = (int)__builtin_fmax(__builtin_fmin(hi - maj0, last_col), -1.0);
          const double inv_dM = rcp_newton(M1 - M0);
          const double sl = (m1 - m0) * inv_dM;
          // minor coordinate on the line through the tile's column 0, tile-relative, minus
          // the pixel-centre 0.5: the sample of column c is at m_first + c * slope (both
          // walks evaluate exactly this expression, so they deposit the same bits)
          m_first = (float)(m0 + ((maj0 + 0.5) - M0) * sl - min0 - 0.5);
          slope = (float)sl;
          if (__builtin_fabsf(slope) >= 1e-6f) {  // (else m moves by less than the margin)
            const float rs = __builtin_amdgcn_rcpf(slope);
            const float c1 = (-1.02f - m_first) * rs, c2 = ((float)T + 0.02f - m_first) * rs;
            const float cl = __builtin_amdgcn_fmed3f(__builtin_fminf(c1, c2), -1.0f, (float)T);
            const float ch = __builtin_amdgcn_fmed3f(__builtin_fmaxf(c1, c2), -1.0f, (float)T);
            const int wa = (int)__builtin_ceilf(cl), wb = (int)__builtin_floorf(ch);
            a = a > wa ? a : wa;
            b = b < wb ? b : wb;
          } else if (!(m_first >= -1.02f && m_first <= (float)T + 0.02f)) {
            b = -1;  // (the binning lists a row or two more than the deposits touch)
          }
          if (a <= b) {
            if constexpr (!kRuns) ca = a_cur;
            if constexpr (kRuns) {
              const double ml = (double)m_first + (double)(T / 2) * (double)slope;
              double mc = m0 + ((maj0 + (T / 2 + 0.5)) - M0) * sl - min0 - 0.5;
              // (far outside end points leave FP64 pixels too coarse for two evaluations to agree; the
              // sample range, and so the rows that the walk may touch, follows m_first)
              mc = __builtin_fabs(mc - ml) < 0.25 ? mc : ml;
              fx_m = (int)__builtin_rint(mc * (double)(1 << kFxBits));
              fx_s = (int)__builtin_rint(sl * (double)(1 << kFxBits));
              const uint32_t s = e_cur & kPairIndex;
              cq2 = ((s >= run1) + (s >= run2) + (s >= run3) + (s >= run4) + (s >= run5)) * kStride;  // its plane
            } else if constexpr (kHues) {
              int f = 0;
              if (n_hues > 1) {
                const uint64_t ray = ((uint64_t)__float_as_uint(c_cur.y) << 32 | __float_as_uint(c_cur.x)) >> kPathBits;
                f = (ray >= D.hue_ray[1] ? 1 : 0) + (n_hues > 2 && ray >= D.hue_ray[2] ? 1 : 0);
              }
              const HueScale& h = s_hue[f];
              const int hch = h.ch;
              const float val = hch == 0 ? ca.x : hch == 1 ? ca.y : ca.z;
              cq0 = (int)pack_q(val, h.ss);
              cq1 = (int)pack_q(ca.w * ca.w, h.sa, q_top);
              cq2 = f * kStride;  // its plane
            } else if (two_ch) {
              if (bc == kBlendDefault) {  // (the same values, without the factors' branches)
                cq0 = (int)pack_q(ca.x, cs0);
                cq1 = (int)pack_q(ca.y, cs1);
                cq2 = (int)pack_q(ca.z, cs2);
                cq3 = (int)pack_q(ca.w * ca.w, cs3, q_top);
              } else {
                cq0 = (int)pack_q(blend_value(bc0, ca.x, ca.w, bk0), cs0, q_top);
                cq1 = (int)pack_q(blend_value(bc1, ca.y, ca.w, bk1), cs1, q_top);
                cq2 = (int)pack_q(blend_value(bc2, ca.z, ca.w, bk2), cs2, q_top);
                cq3 = (int)pack_q(blend_value(bc3, ca.w, ca.w, bk3), cs3, q_top);
              }
            } else {
              cq0 = fx(blend_value(bc0, ca.x, ca.w, bk0), cs0);
              cq1 = fx(blend_value(bc1, ca.y, ca.w, bk1), cs1);
              cq2 = fx(blend_value(bc2, ca.z, ca.w, bk2), cs2);
              cq3 = fx(blend_value(bc3, ca.w, ca.w, bk3), cs3);
            }
            int vc = 0;
            if constexpr (kVC) {
              dc = make_float4(c_cur.x - ca.x, c_cur.y - ca.y, c_cur.z - ca.z, c_cur.w - ca.w);
              vc = (dc.x != 0.f || dc.y != 0.f || dc.z != 0.f || dc.w != 0.f) ? 1 : 0;
              s_first = (float)((((double)a + maj0 + 0.5) - M0) * inv_dM);
              ds = (float)inv_dM;
            }
            const int neg = (cq0 | cq1 | cq2 | cq3) < 0 ? 1 : 0;
            packed = (b - a + 1) | (a << 8) | (vc << 17) | (neg << 18);
          }
        }
        // ---- loads for the batches ahead ----
        fetch(e_nxt, p_nxt, a_nxt, c_nxt);
        b_aft = __builtin_amdgcn_readfirstlane(taken);
        e_aft = entry(b_aft);
        if (lane == 0) taken = atomicAdd(&s_batch[phase], 1u);
        // ---- walk the pairs that have samples ----
        if constexpr (kStreamKernel && (kVS || !kVC)) {
          // Sample stream: the c-th lane with samples owns positions pre_c .. pre_c + n_c - 1 of
          // the wave's stream (pre: exclusive prefix sum of n), n_c half its samples, rounded up: at
          // position k a lane takes two, columns k + off_c and k + off_c + delta_c of the tile, so
          // that the search for the record and its reads serve both (at the last position of an odd
          // number the second goes to the guard rows). Record c = {off_c, delta_c and the first
          // position without a second sample, m_first, slope, 8 off_c}, {q0..q3}; with a colour
          // per vertex {q0_c, s_first, ds} in the second part and the first colour and the difference in
          // two more; with hues {off_c, m_first, slope, 8 off_c and the plane}, {s, a a, last position
          // with a second sample, delta_c}. With runs the line is in fixed point, 22 bits below the
          // pixel: m = M + S position, both modulo 2^32 and exact, its pixel M >> 22 and the fraction
          // of its weight the bits below; {M at position 0, S, 4 off_c and the plane, last position with a
          // second sample}, {S delta_c, 4 delta_c}. Record P (after the last pair) is empty, so the
          // positions past the end of the stream need no mask. Stream word i holds a bit per position
          // 64 i .. 64 i + 63 that starts a record; lane l of step s finds its record as the
          // number of starts at positions <= 64 s + l, minus one.
          //
          // A sample's pixel needs no clamp here: the setup keeps samples at m in [-1.02, T + 0.02] only,
          // off by some 1e-5, so jl and jl + 1 lie in the tile's rows and the two guard rows on either side.
          //
          // Hues and runs are bound by instruction issue, channels by the LDS. Tile walk, us, a
          // sample to a lane and two: 1M-ray frame 541 and 506, 20 uneven scenes 604 and 563, 60033
          // string-mod lines of two colours at 2048x1536 142 and 134 (pair by pair 292), 100003 lines of a colour
          // each at 1920x1080 52 and 50.
          const int n_all = packed & 0xff;
          const int n = (n_all + 1) >> 1;  // positions
          const uint64_t live = __ballot(n != 0);
          if (live) {
            const int incl = wave_sum_incl(n);
            const int pre = incl - n;
            const int total = __builtin_amdgcn_readlane(incl, 63);
            const int n_live = __builtin_popcountll(live);
            const int steps = (total + 63) >> 6;
            const int c = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(live >> 32),
                                                         __builtin_amdgcn_mbcnt_lo((uint32_t)live, 0u));
            const int wv = __builtin_amdgcn_readfirstlane(wave);
            uint4* const rec = s_rec + wv * (kRecs * 2);
            // the vertex colours' part of the records: in the third plane, which such frames do not use
            uint4* const vrec = reinterpret_cast<uint4*>(s_tile + 2 * kStride) + wv * (kRecs * 2);
            static_assert(!kVS || (kPlanes > 2 && kWaves * kRecs * 32 <= kStride * 8), "the third plane holds them");
            unsigned long long* const mask = s_mask + wv * kMaskWords;
            // (one wave's LDS operations execute in order: the words are cleared before the
            // starts are set, and the previous batch's reads are done before these writes)
            if (lane < steps) mask[lane] = 0ull;
            if (n) {
              // the two samples of an even record are columns c and c + n, of an odd one c + m and c (m =
              // n_all - n): neighbouring pairs, often of the same columns, then mostly meet other banks
              // (without that the 1M-ray frame's walk took 550 us, 506 so)
              const int m2 = n_all - n;
              const int off = ((packed >> 8) & 0xff) - pre + ((c & 1) ? m2 : 0);
              const int delta = (c & 1) ? -m2 : n;  // from the first sample's column to the second's
              if constexpr (kRuns) {
                rec[2 * c] = make_uint4((uint32_t)(fx_m + __mul24(off - T / 2, fx_s)), (uint32_t)fx_s,
                                        (uint32_t)((off + cq2) * 4), (uint32_t)(pre + m2 - 1));
                *reinterpret_cast<uint2*>(&rec[2 * c + 1]) = make_uint2((uint32_t)__mul24(delta, fx_s), (uint32_t)(4 * delta));
              } else {
                const uint32_t place = kHues ? (uint32_t)off
                                             : (uint32_t)off << 19 | ((uint32_t)delta & 127u) << 12 | (uint32_t)(pre + m2);
                rec[2 * c] = make_uint4(place, __float_as_uint(m_first), __float_as_uint(slope),
                                        (uint32_t)((kHues ? off + cq2 : off) * 8));
              }
              if constexpr (kRuns) {
              } else if constexpr (kHues) {
                rec[2 * c + 1] = make_uint4((uint32_t)cq0, (uint32_t)cq1, (uint32_t)(pre + m2 - 1), (uint32_t)delta);
              } else if constexpr (kVS) {
                rec[2 * c + 1] = make_uint4(__float_as_uint((float)((packed >> 8) & 0xff)), __float_as_uint(s_first),
                                            __float_as_uint(ds), 0u);
                vrec[2 * c] = __builtin_bit_cast(uint4, ca);
                vrec[2 * c + 1] = __builtin_bit_cast(uint4, dc);
              } else {
                rec[2 * c + 1] = make_uint4((uint32_t)cq0, (uint32_t)cq1, (uint32_t)cq2, (uint32_t)cq3);
              }
              atomicOr(&mask[pre >> 6], 1ull << (pre & 63));
            }
            if (lane == 0) {
              if constexpr (kRuns) {
                // (no colour to be zero: the empty record's line lies above the tile, in guard row -2)
                rec[2 * n_live] = make_uint4((uint32_t)(-(kGuard << kFxBits)), 0u, (uint32_t)(-total * 4), 0xffffffffu);
                rec[2 * n_live + 1] = make_uint4(0u, 0u, 0u, 0u);
              } else {
                rec[2 * n_live] = make_uint4(kHues ? (uint32_t)(-total) : (uint32_t)(-total) << 19, 0u, 0u,
                                             (uint32_t)(-total * 8));
                rec[2 * n_live + 1] = make_uint4(0u, 0u, kHues ? 0xffffffffu : 0u, 0u);
              }
              if constexpr (kVS) vrec[2 * n_live] = vrec[2 * n_live + 1] = make_uint4(0u, 0u, 0u, 0u);
              if (total & 63) atomicOr(&mask[total >> 6], 1ull << (total & 63));
            }
            // Lane i keeps, for step i, the stream word's starts at positions 64 i + 1 .. 64 i + 63 and
            // the address of the record before the first of those: a step takes them with three lane
            // reads, and its lane l reads the record that many starts further on. (With the record
            // count kept by scalar instructions, 17 of them a step, the scalar unit took as long as
            // the vector ALU: 1M-ray frame 590 -> 549 us, 1.6M segments in runs 2920 -> 2700.) Past the
            // last step (the read one step ahead, never used) the words are empty and every lane names
            // the last record.
            const unsigned long long my_word = lane < steps ? mask[lane] : 0ull;
            const uint32_t my_lo = (uint32_t)(my_word >> 1), my_hi = (uint32_t)(my_word >> 33);
            const int my_n = __builtin_popcountll(my_word);
            const int my_first = wave_sum_incl(my_n) - my_n + (int)(my_word & 1ull) - 1;
            const uint32_t my_rec = lds_address(rec) + (uint32_t)(my_first * 32);
            struct StepRec {
              uint4 r0, r1, a, d;
            };
            auto read_recs = [&](int s, StepRec& R) {
              const int sl = s < 63 ? s : 63;
              const uint32_t lo = __builtin_amdgcn_readlane(my_lo, sl), hi = __builtin_amdgcn_readlane(my_hi, sl);
              const uint32_t k = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
              const uint32_t ra = __builtin_amdgcn_readlane(my_rec, sl) + k * 32u;
              R.r0 = lds_read16(ra);
              if constexpr (kRuns) {
                const uint2 q = lds_read8(ra + 16u);
                R.r1.x = q.x;
                R.r1.y = q.y;
              } else {
                R.r1 = lds_read16(ra + 16u);
              }
              if constexpr (kVS) {
                const uint32_t rv = ra + (lds_address(vrec) - lds_address(rec));
                R.a = lds_read16(rv);
                R.d = lds_read16(rv + 16u);
              }
            };
            // Step st at stream positions p = 64 st + lane: the sample's column is off + p, its
            // entry in plane 0 jl * T + column.
            auto deposit_step = [&](int st, const StepRec& R) {
              if constexpr (kRuns) {
                const int p = lane + (st << 6);
                auto put = [&](int M, uint32_t b) {
                  const int jl = M >> kFxBits;
                  uint32_t* const t = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(tile32) + (((uint32_t)jl << 8) + b));
                  const uint32_t r = cut_weight(M, wq);
                  atomicAdd(t, wq - r);
                  atomicAdd(t + T, r);
                };
                int M;
                asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(M) : "v"(p), "v"((int)R.r0.y), "v"((int)R.r0.x));
                const uint32_t base = ((uint32_t)p << 2) + R.r0.z;
                put(M, base);
                // (no second sample: above the tile, into the guard rows)
                put(p <= (int)R.r0.w ? M + (int)R.r1.x : -(kGuard << kFxBits), base + R.r1.y);
                return;
              }
              const uint4 r0 = R.r0, r1 = R.r1;
              if constexpr (kHues) {
                const int p = lane + (st << 6), col = (int)r0.x + p;
                auto put = [&](float m, uint32_t b) {
                  int jl;
                  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(jl) : "v"(m));
                  char* const t = reinterpret_cast<char*>(tile) + (((uint32_t)jl << 9) + b);
                  deposit1<T>(reinterpret_cast<unsigned long long*>(t), m, r1.x, r1.y);
                };
                const float m = __builtin_fmaf((float)col, __uint_as_float(r0.z), __uint_as_float(r0.y));
                const float m2 = __builtin_fmaf((float)(col + (int)r1.w), __uint_as_float(r0.z), __uint_as_float(r0.y));
                const uint32_t base = ((uint32_t)p << 3) + r0.w;
                put(m, base);
                put(p <= (int)r1.z ? m2 : (float)-kGuard, base + (r1.w << 3));
                return;
              }
              const int p = lane + (st << 6), col = ((int)r0.x >> 19) + p;
              const int delta = __builtin_amdgcn_sbfe((int)r0.x, 12, 7);
              auto put = [&](int column, float m, uint32_t b) {
                int jl;
                asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(jl) : "v"(m));
                unsigned long long* const t =
                    reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(tile) + (((uint32_t)jl << 9) + b));
                if constexpr (kVS) {
                  // the per-pair walk's expressions: the same bits
                  const float4 a = __builtin_bit_cast(float4, R.a), d = __builtin_bit_cast(float4, R.d);
                  const float sp = __builtin_fmaf((float)column - __uint_as_float(r1.x), __uint_as_float(r1.z),
                                                  __uint_as_float(r1.y));
                  const float al = __builtin_fmaf(sp, d.w, a.w);
                  deposit2<T, kStride>(t, m, pack_q(__builtin_fmaf(sp, d.x, a.x), cs0),
                                       pack_q(__builtin_fmaf(sp, d.y, a.y), cs1),
                                       pack_q(__builtin_fmaf(sp, d.z, a.z), cs2), pack_q(al * al, cs3, q_top));
                } else {
                  deposit2<T, kStride>(t, m, r1.x, r1.y, r1.z, r1.w);
                }
              };
              const float m = __builtin_fmaf((float)col, __uint_as_float(r0.z), __uint_as_float(r0.y));
              const float m2 = __builtin_fmaf((float)(col + delta), __uint_as_float(r0.z), __uint_as_float(r0.y));
              const uint32_t base = ((uint32_t)p << 3) + r0.w;
              put(col, m, base);
              put(col + delta, p < (int)(r0.x & 0xfffu) ? m2 : (float)-kGuard, base + ((uint32_t)delta << 3));
            };
            // One step ahead: the records of step s + 1 are read while step s deposits; two
            // steps per trip with the record registers swapped, so that nothing read ahead is
            // copied (a copy would wait for its read). Scheduling barriers keep the reads ahead
            // of the deposits they overlap.
            StepRec ra{}, rb{};
            read_recs(0, ra);
            // zero adds into guard row -2: the loop is entered with the same LDS operations
            // in flight as it loops back with (two reads and four adds; more with
            // channels), so that the
            // compiler's wait counts inside the loop stay exact
            if constexpr (kRuns) {
              uint32_t zero = 0u;
              asm volatile("" : "+v"(zero));
              uint32_t* const g = tile32 + (-kGuard * T + lane);
              for (int k = 0; k < 2; k++) {
                atomicAdd(g, zero);
                atomicAdd(g + T, zero);
              }
            } else {
              unsigned long long zero = 0ull;
              asm volatile("" : "+v"(zero));  // an add the compiler cannot turn into a load
              unsigned long long* const g = tile + (-kGuard * T + lane);
              for (int k = 0; k < (kHues ? 1 : 2); k++) {
                atomicAdd(g, zero);
                atomicAdd(g + T, zero);
                atomicAdd(g + kStride, zero);
                atomicAdd(g + T + kStride, zero);
              }
            }
            __builtin_amdgcn_sched_barrier(0);
            for (int st = 0;; st += 2) {
              read_recs(st + 1, rb);
              __builtin_amdgcn_sched_barrier(0);
              deposit_step(st, ra);
              __builtin_amdgcn_sched_barrier(0);
              if (st + 1 >= steps) break;
              read_recs(st + 2, ra);
              __builtin_amdgcn_sched_barrier(0);
              deposit_step(st + 1, rb);
              __builtin_amdgcn_sched_barrier(0);
              if (st + 2 >= steps) break;
            }
            if (count_work)
              wave_samples += (unsigned long long)__builtin_amdgcn_readlane(wave_sum_incl(n_all), 63);
            wave_atomics += (kHues || kRuns ? 4u : 8u) * (unsigned)steps;
          }
          return;
        }
        // One pair per step: pair j's samples are columns jq0 .. jq0 + jn - 1 of the tile (jn <=
        // 64); lane t takes column jq0 + t. Four-channel deposits are exact 64-bit products:
        // (2^20 - wq) * c at minor pixel jl and wq * c at jl + 1, which add up to exactly c << 20
        // (f < 1 keeps wq = trunc(f * 2^20 + 1/2) <= 2^20).
        uint64_t todo = __ballot(packed != 0);
        while (todo) {
          const int j = __builtin_ctzll(todo);
          todo &= todo - 1;
          const int jp = bcast_i(packed, j);
          const int jn = jp & 0xff, jq0 = (jp >> 8) & 0xff, jvc = (jp >> 17) & 1;
          const int jneg = (jp >> 18) & 1;
          wave_samples += (unsigned long long)jn;
          wave_atomics += kHues ? 2u : two_ch ? 4u : 8u;
          const float jm = bcast_f(m_first, j), jsl = bcast_f(slope, j);
          // lane's sample: minor pixel jl, weights wl (pixel jl) and wq (jl + 1), and the entry
          // t of (jl, jq0 + lane) in plane 0 (t2 in plane 2); the row below and the next plane
          // are at fixed offsets from these. Every plane has two guard rows on either side and
          // jl is clamped to [-2, T]: a sample whose deposits fall outside the tile (rows -1 or
          // T, or farther off after the clamp) adds into guard rows, which are never read, so
          // only lanes past jn need masking.
          const int col = lane + jq0;
          const float m = __builtin_fmaf((float)col, jsl, jm);
          int jl;
          asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(jl) : "v"(m));
          jl = jl < -kGuard ? -kGuard : (jl > T ? T : jl);
          const int e0 = jl * T + col;
          const bool in = lane < jn;
          if constexpr (kHues) {
            const uint32_t qs = (uint32_t)bcast_i(cq0, j), qa = (uint32_t)bcast_i(cq1, j);
            const int plane = bcast_i(cq2, j);
            if (in) deposit1<T>(tile + e0 + plane, m, qs, qa);
            continue;
          }
          if (two_ch) {
            uint32_t q0, q1, q2, q3;
            if (!kVC || !jvc) {
              q0 = (uint32_t)bcast_i(cq0, j);
              q1 = (uint32_t)bcast_i(cq1, j);
              q2 = (uint32_t)bcast_i(cq2, j);
              q3 = (uint32_t)bcast_i(cq3, j);
            } else {
              const float jds = bcast_f(ds, j), jsa = bcast_f(s_first, j);
              const float a0 = bcast_f(ca.x, j), a1 = bcast_f(ca.y, j), a2 = bcast_f(ca.z, j), a3 = bcast_f(ca.w, j);
              const float d0 = bcast_f(dc.x, j), d1 = bcast_f(dc.y, j), d2 = bcast_f(dc.z, j), d3 = bcast_f(dc.w, j);
              const float sp = __builtin_fmaf(lane_f, jds, jsa);
              const float al = __builtin_fmaf(sp, d3, a3);
              q0 = pack_q(blend_value(bc0, __builtin_fmaf(sp, d0, a0), al, bk0), cs0, q_top);
              q1 = pack_q(blend_value(bc1, __builtin_fmaf(sp, d1, a1), al, bk1), cs1, q_top);
              q2 = pack_q(blend_value(bc2, __builtin_fmaf(sp, d2, a2), al, bk2), cs2, q_top);
              q3 = pack_q(blend_value(bc3, al, al, bk3), cs3, q_top);
            }
            if (in) deposit2<T, kStride>(tile + e0, m, q0, q1, q2, q3);
            continue;
          }
          const int wq = (int)__builtin_fmaf(__builtin_amdgcn_fractf(m), (float)kWOne, 0.5f);
          const int wl = kWOne - wq;
          // plane 2's entry as an opaque register: the deposits of planes 2 and 3 then address
          // it with the instruction's offset field instead of each adding 64 KB and more
          int e2 = e0 + 2 * kStride;
          asm volatile("" : "+v"(e2));
          unsigned long long* const t = tile + e0;
          unsigned long long* const t2 = tile + e2;
          if ((!kVC || !jvc) && !jneg) {
            // non-negative colour: unsigned 32x32 -> 64-bit products (one multiply per deposit)
            const unsigned jc0 = (unsigned)bcast_i(cq0, j), jc1 = (unsigned)bcast_i(cq1, j),
                           jc2 = (unsigned)bcast_i(cq2, j), jc3 = (unsigned)bcast_i(cq3, j);
            const unsigned ul = (unsigned)wl, uq = (unsigned)wq;
            if (in) {
              atomicAdd(t, (unsigned long long)ul * jc0);
              atomicAdd(t + kStride, (unsigned long long)ul * jc1);
              atomicAdd(t2, (unsigned long long)ul * jc2);
              atomicAdd(t2 + kStride, (unsigned long long)ul * jc3);
              atomicAdd(t + T, (unsigned long long)uq * jc0);
              atomicAdd(t + T + kStride, (unsigned long long)uq * jc1);
              atomicAdd(t2 + T, (unsigned long long)uq * jc2);
              atomicAdd(t2 + T + kStride, (unsigned long long)uq * jc3);
            }
          } else {
            int c0, c1, c2, c3;
            if (!kVC || !jvc) {
              c0 = bcast_i(cq0, j);
              c1 = bcast_i(cq1, j);
              c2 = bcast_i(cq2, j);
              c3 = bcast_i(cq3, j);
            } else {
              // per-vertex colours: the colour is interpolated along the segment at each sample
              const float jds = bcast_f(ds, j), jsa = bcast_f(s_first, j);
              const float a0 = bcast_f(ca.x, j), a1 = bcast_f(ca.y, j), a2 = bcast_f(ca.z, j), a3 = bcast_f(ca.w, j);
              const float d0 = bcast_f(dc.x, j), d1 = bcast_f(dc.y, j), d2 = bcast_f(dc.z, j), d3 = bcast_f(dc.w, j);
              const float sp = __builtin_fmaf(lane_f, jds, jsa);
              const float al = __builtin_fmaf(sp, d3, a3);
              c0 = fx(blend_value(bc0, __builtin_fmaf(sp, d0, a0), al, bk0), cs0);
              c1 = fx(blend_value(bc1, __builtin_fmaf(sp, d1, a1), al, bk1), cs1);
              c2 = fx(blend_value(bc2, __builtin_fmaf(sp, d2, a2), al, bk2), cs2);
              c3 = fx(blend_value(bc3, al, al, bk3), cs3);
            }
            if (in) {
              atomicAdd(t, (unsigned long long)((long long)wl * c0));
              atomicAdd(t + kStride, (unsigned long long)((long long)wl * c1));
              atomicAdd(t2, (unsigned long long)((long long)wl * c2));
              atomicAdd(t2 + kStride, (unsigned long long)((long long)wl * c3));
              atomicAdd(t + T, (unsigned long long)((long long)wq * c0));
              atomicAdd(t + T + kStride, (unsigned long long)((long long)wq * c1));
              atomicAdd(t2 + T, (unsigned long long)((long long)wq * c2));
              atomicAdd(t2 + T + kStride, (unsigned long long)((long long)wq * c3));
            }
          }
        }
      };
      // a wave's first two batches are fixed (wave, kWaves + wave); the counter hands out the
      // rest from 2 kWaves on
      uint32_t b0 = (uint32_t)__builtin_amdgcn_readfirstlane(wave);
      uint32_t e0 = entry(b0);
      uint32_t b1 = b0 + (uint32_t)kWaves;
      uint32_t e1 = entry(b1);
      float4 p0 = make_float4(0.f, 0.f, 0.f, 0.f), a0 = p0, c0v = p0, p1 = p0, a1 = p0, c1v = p0;
      fetch(e0, p0, a0, c0v);
      if (lane == 0) taken = atomicAdd(&s_batch[phase], 1u);
      // two batches per trip with the register sets swapped, so that every value loaded ahead is
      // written once per trip and none is copied (a copy would wait for its load)
      auto run = [&](auto mode_tag) {
        for (;;) {
          if (b0 >= n_batches) break;
          uint32_t b2, e2;
          step(mode_tag, e0, p0, a0, c0v, e1, p1, a1, c1v, b2, e2);
          if (b1 >= n_batches) break;
          uint32_t b3, e3;
          step(mode_tag, e1, p1, a1, c1v, e2, p0, a0, c0v, b3, e3);
          b0 = b2;
          e0 = e2;
          b1 = b3;
          e1 = e3;
        }
      };
      bool walked = RUNS;
      if constexpr (RUNS) run(std::integral_constant<int, WALK_RUNS>{});
      if constexpr (kHueKernel) {
        if (hues) {
          run(std::integral_constant<int, WALK_HUES>{});
          walked = true;
        }
      }
      if constexpr (RUNS) {
      } else if (walked) {
      } else if (kStreamKernel && col1 && bc == kBlendDefault) {
        run(std::integral_constant<int, kStreamKernel ? WALK_VERTEX_STREAM : WALK_VERTEX_COLORS>{});
      } else if (col1) {
        run(std::integral_constant<int, WALK_VERTEX_COLORS>{});
      } else {
        run(std::integral_constant<int, WALK_COLOR>{});
      }
      __syncthreads();
      if (phase == 0) {
        if constexpr (RUNS)
          transpose_tile<T, kStride, kWaves>(tile32, planes, wave, lane);
        else
          transpose_tile<T, kStride, kWaves>(tile, planes, wave, lane);
        __syncthreads();
      }
    }
    if constexpr (RUNS) {
      for (int f = 0; f < planes; f++) {
        const uint32_t q0 = s_run[f][0], q1 = s_run[f][1], q2 = s_run[f][2], q3 = s_run[f][3];
#pragma unroll
        for (int i = 0; i < T * T / BLOCK; i++) {
          const uint32_t w = tile32[f * kStride + i * BLOCK + (int)threadIdx.x];
          acc[i][0] += (unsigned long long)w * q0;
          acc[i][1] += (unsigned long long)w * q1;
          acc[i][2] += (unsigned long long)w * q2;
          acc[i][3] += (unsigned long long)w * q3;
        }
      }
      __syncthreads();  // the next layer writes s_run
    }
    }
    if (!claim_early) claim();
    const WorkItem wn = load_next();  // in flight during the flush
    if constexpr (RUNS) {
      unsigned long long* fx = split_fx + (size_t)W.slot * kSlotU64;
      double un[4];
#pragma unroll
      for (int c = 0; c < 4; c++) un[c] = __builtin_ldexp(1.0 / (double)wq, -K[c]);
#pragma unroll
      for (int i = 0; i < T * T / BLOCK; i++) {
        const int k = i * BLOCK + (int)threadIdx.x;
        if (split) {  // (the merge converts the tile's sums)
#pragma unroll
          for (int c = 0; c < 4; c++)
            if (acc[i][c]) atomicAdd(&fx[c * T * T + k], acc[i][c]);
          continue;
        }
        const int gx = x0 + k % T, gy = y0 + k / T;
        if (gx >= v.width || gy >= v.height) continue;
        const size_t px = (size_t)gy * v.width + gx;
        float4 o = accum[px];
        o.x += (float)((double)(long long)acc[i][0] * un[0]);
        o.y += (float)((double)(long long)acc[i][1] * un[1]);
        o.z += (float)((double)(long long)acc[i][2] * un[2]);
        o.w += (float)((double)(long long)acc[i][3] * un[3]);
        accum[px] = o;
      }
    } else if (split) {
      // exact partial sums into the tile's merge slot (integer atomics: order independent)
      unsigned long long* fx = split_fx + (size_t)W.slot * kSlotU64;
      const int n_fields = hues ? 2 * n_hues : 4;
      if (two_ch && slot_words(W.tile_pairs)) {
        for (int k = threadIdx.x; k < T * T; k += BLOCK)
          for (int f = 0; f < n_fields / 2; f++) {
            const unsigned long long val = tile[f * kStride + k];
            if (val) atomicAdd(&fx[f * T * T + k], val);
          }
      } else {
        for (int k = threadIdx.x; k < T * T; k += BLOCK) {
          for (int c = 0; c < n_fields; c++) {
            const unsigned long long val =
                two_ch ? (tile[(c >> 1) * kStride + k] >> (32 * (c & 1))) & 0xffffffffull : tile[c * kStride + k];
            if (val) atomicAdd(&fx[c * T * T + k], val);
          }
        }
      }
    } else {
      // the only item of its tile: fixed point -> FP32 accumulator
      const int wb = two_ch ? 0 : kWBits;
      const double un0 = __builtin_ldexp(1.0, -(G[0] + wb)), un1 = __builtin_ldexp(1.0, -(G[1] + wb));
      const double un2 = __builtin_ldexp(1.0, -(G[2] + wb)), un3 = __builtin_ldexp(1.0, -(G[3] + wb));
      // a 32-bit field w scaled by 2^-G (G <= 126) is a normal float or 0 or beyond the float
      // range: rounding w to FP32 and then scaling rounds the exact w * 2^-G once, as the FP64
      // product rounded to FP32 does (the merge of split tiles takes that route), bit for bit
      auto field = [](uint32_t w, int g) { return __builtin_ldexpf((float)w, -g); };
      for (int k = threadIdx.x; k < T * T; k += BLOCK) {
        int r = k / T, cc = k % T;
        int gx = x0 + cc, gy = y0 + r;
        if (gx >= v.width || gy >= v.height) continue;
        const int idx = k;  // row-major
        const size_t px = (size_t)gy * v.width + gx;
        float4 o = whole ? make_float4(0.f, 0.f, 0.f, 0.f) : accum[px];
        if (hues) {
          double p[4] = {0.0, 0.0, 0.0, 0.0};
          for (int f = 0; f < n_hues; f++) {
            const unsigned long long w = tile[f * kStride + idx];
            hue_add(p, s_hue[f], (uint32_t)w, w >> 32);
          }
          o.x += (float)p[0];
          o.y += (float)p[1];
          o.z += (float)p[2];
          o.w += (float)p[3];
        } else if (two_ch) {
          const unsigned long long w0 = tile[idx], w1 = tile[kStride + idx];
          o.x += field((uint32_t)w0, G[0]);
          o.y += field((uint32_t)(w0 >> 32), G[1]);
          o.z += field((uint32_t)w1, G[2]);
          o.w += field((uint32_t)(w1 >> 32), G[3]);
        } else {
          o.x += (float)((double)(long long)tile[idx] * un0);
          o.y += (float)((double)(long long)tile[kStride + idx] * un1);
          o.z += (float)((double)(long long)tile[2 * kStride + idx] * un2);
          o.w += (float)((double)(long long)tile[3 * kStride + idx] * un3);
        }
        accum[px] = o;
        if (whole) gen(D.out16)[px] = resolve_px(o);
      }
    }
    publish_next(wn);
    __syncthreads();
  }
  // Profiled frames: the walk's work, one global add per workgroup. (An add per wave to either
  // word in every frame held up the claims of the work items, 8192 adds of 12 ns to one line: the
  // tile walk of a 20k-ray frame took 90 us where it takes 62.)
  if (count_work) {
    __shared__ unsigned long long s_work[2];
    if (threadIdx.x < 2) s_work[threadIdx.x] = 0ull;
    __syncthreads();
    if (lane == 0 && wave_samples) {
      atomicAdd(&s_work[0], wave_samples);
      atomicAdd(&s_work[1], wave_atomics);
    }
    __syncthreads();
    if (threadIdx.x == 0 && s_work[0]) {
      atomicAdd(&ctl->samples, s_work[0]);
      atomicAdd(&ctl->lds_atomics, s_work[1]);
    }
  }
}

// Converts the merge slots of split tiles into the FP32 accumulator (the same expression as
// the unsplit flush) and leaves the slots zeroed for the next frame. Persistent over parts of 256
// pixels: a frame splits some tens to hundreds of tiles, and with a workgroup per slot the few
// that ran took the latency of 16 passes over it each (us: 1M-ray frame 104 -> 27, 1.6M segments at
// 4096x4096 299 -> 179, 20k-ray frame 20 -> 5).
constexpr int kMergeBlock = 256;
__global__ __launch_bounds__(kMergeBlock) void tile_merge_kernel(const SceneDesc* __restrict__ descs,
                                                        const uint32_t* __restrict__ tile_scene,
                                                        const uint32_t* __restrict__ row_start,
                                                        const uint32_t* __restrict__ split_tiles,
                                                        const BatchCtl* ctl, unsigned long long* split_fx,
                                                        uint32_t split_cap, int tile_px) {
  if (ctl->flags & kCtlStop) return;
  uint32_t n_split = ctl->n_split;
  n_split = n_split < split_cap ? n_split : split_cap;
  __shared__ HueScale s_hue[kMaxHues];
  const uint32_t parts = (uint32_t)tile_px / kMergeBlock;
  for (uint32_t u = blockIdx.x; u < n_split * parts; u += gridDim.x) {
    const uint32_t sl = u / parts;
    const int k = (int)(u % parts) * kMergeBlock + (int)threadIdx.x;
    const uint32_t g = split_tiles[sl];
    const SceneDesc& D = descs[tile_scene[g]];
    const AccumView v = D.view;
    const uint32_t t = g - (uint32_t)D.tile_base;
    const int T = v.tile, TT = tile_px;
    const int x0 = (int)(t % (uint32_t)v.tiles_x) * T, y0 = (int)(t / (uint32_t)v.tiles_x) * T;
    const bool hues = (D.flags & SCENE_HUES) != 0;
    const bool runs = (D.flags & SCENE_RUNS) != 0;
    const uint32_t nl = runs ? D.row_stride : 1u;
    const uint32_t nt = row_start[2u * nl * (g + 1u)] - row_start[2u * nl * g];
    const uint32_t np = nt < kPackedPiece ? nt : kPackedPiece;
    __syncthreads();  // (the slot before is done with the table)
    if (hues && threadIdx.x < kMaxHues) s_hue[threadIdx.x] = hue_scale(D, threadIdx.x, np);
    __syncthreads();
    double un[4] = {0.0, 0.0, 0.0, 0.0};
    if (!hues) {
#pragma unroll
      for (int c = 0; c < 4; c++)
        un[c] = runs ? __builtin_ldexp(1.0 / (double)run_weight(np), -run_color_bits(D, c, nt))
                     : __builtin_ldexp(1.0, (D.flags & SCENE_PACKED) ? -packed_fixed_bits(D, c, np)
                                                                     : -(scene_fixed_bits(D, c) + kWBits));
    }
    const int n_fields = hues ? 2 * D.n_hues : 4;
    const bool whole = (D.flags & SCENE_FRESH_IMAGE) != 0;  // the frame clears and resolves here
    unsigned long long* fx = split_fx + (size_t)sl * kSlotU64;
    unsigned long long a[2 * kMaxHues] = {}, any = 0ull;
    const bool words = (D.flags & SCENE_PACKED) && !runs && slot_words(np);
    const int n_slot = words ? n_fields / 2 : n_fields;
#pragma unroll
    for (int c = 0; c < 2 * kMaxHues; c++)
      if (c < n_slot) {
        a[c] = fx[c * TT + k];
        any |= a[c];
      }
    if (any == 0ull && !whole) continue;
#pragma unroll
    for (int c = 0; c < 2 * kMaxHues; c++)
      if (a[c]) fx[c * TT + k] = 0ull;
    if (words) {
#pragma unroll
      for (int f = kMaxHues - 1; f >= 0; f--) {
        const unsigned long long w = a[f];
        a[2 * f] = w & 0xffffffffull;
        a[2 * f + 1] = w >> 32;
      }
    }
    const int gx = x0 + (k % T), gy = y0 + (k / T);
    if (gx >= v.width || gy >= v.height) continue;
    const size_t px = (size_t)gy * v.width + gx;
    float4 o = whole ? make_float4(0.f, 0.f, 0.f, 0.f) : gen(D.accum)[px];
    if (hues) {
      double p[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int f = 0; f < kMaxHues; f++)
        if (2 * f < n_fields) hue_add(p, s_hue[f], a[2 * f], a[2 * f + 1]);
      o.x += (float)p[0];
      o.y += (float)p[1];
      o.z += (float)p[2];
      o.w += (float)p[3];
    } else {
      o.x += (float)((double)(long long)a[0] * un[0]);
      o.y += (float)((double)(long long)a[1] * un[1]);
      o.z += (float)((double)(long long)a[2] * un[2]);
      o.w += (float)((double)(long long)a[3] * un[3]);
    }
    gen(D.accum)[px] = o;
    if (whole) gen(D.out16)[px] = resolve_px(o);
  }
}

// ---- clear and resolve of one image (a frame's own are part of its tile flushes) ------------------
// Bound by HBM: 4096x4096 clear 268 MB in 34 us, resolve 403 MB in 72 us. They are launched by
// themselves: as frames of the pipeline, with its upload and readback, a call on a 1920x1080
// image took 36 to 46 us for 8 us of kernel (17 and 20 so).
template <int MODE>  // 0 clear, 1 resolve
__global__ __launch_bounds__(256) void pixels_kernel(float4* __restrict__ accum, ushort4* __restrict__ out16, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (MODE == 0)
    accum[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  else
    out16[i] = resolve_px(accum[i]);
}

// The issue ceiling of the tile walk's LDS atomics: workgroups shaped like the two-channel
// 64-pixel tile kernel's (512 threads, two 32 KB planes, two per compute unit), each wave adding
// into consecutive 64-bit words (no bank conflicts), four ds_add_u64 per loop trip as a walk
// step issues. A wave instruction costs the same however many lanes are active, so this rate in
// wave instructions per second is the roof the walk's atomic count is held against.
constexpr int kAtomicRateBlock = 512;
__global__ __launch_bounds__(kAtomicRateBlock) void lds_atomic_rate_kernel(uint32_t iters, unsigned long long* sink) {
  __shared__ unsigned long long s[2 * 4096];
  for (int k = threadIdx.x; k < 2 * 4096; k += kAtomicRateBlock) s[k] = 0ull;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long v = (unsigned long long)lane + 1ull;
  int r = wave * 7;  // wave-uniform row in [0, 62]: rows r and r + 1 of both planes stay inside s
  for (uint32_t i = 0; i < iters; i++) {
    const int e = r * 64 + lane;
    atomicAdd(&s[e], v);
    atomicAdd(&s[e + 64], v);
    atomicAdd(&s[e + 4096], v);
    atomicAdd(&s[e + 4096 + 64], v);
    r = (r + 2) % 63;
  }
  __syncthreads();
  if (threadIdx.x == 0) sink[blockIdx.x] = s[0] + s[4095];
}

hipError_t launch_lds_atomic_rate(int n_cu, uint32_t iters, unsigned long long* sink, hipStream_t st,
                                  uint64_t* wave_instructions) {
  const int grid = 2 * n_cu;
  hipLaunchKernelGGL(lds_atomic_rate_kernel, dim3(grid), dim3(kAtomicRateBlock), 0, st, iters, sink);
  *wave_instructions = (uint64_t)grid * (kAtomicRateBlock / 64) * iters * 4ull;
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void iota_u64_kernel(uint64_t* p, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = i;
}

__global__ void fill_u32_kernel(uint32_t* p, uint64_t n, uint32_t v) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// ---- host launchers ---------------------------------------------------------------------
bool tile_size_supported(int tile) { return tile == 32 || tile == 64; }
uint64_t merge_slot_u64() { return kSlotU64; }

uint64_t scan_scratch_elems(uint64_t n) {
  uint64_t total = 0;
  while (n > 1) {
    uint64_t nb = (n + kScanBlock - 1) / kScanBlock;
    total += nb;
    n = nb;
  }
  return total + 1;
}

hipError_t launch_scan_exclusive(const uint32_t* in, uint32_t* out, uint64_t n, uint32_t* scratch,
                                 hipStream_t st, unsigned long long* total) {
  if (n == 0) return hipSuccess;
  uint64_t nb = (n + kScanBlock - 1) / kScanBlock;
  uint32_t* sums = scratch;
  hipLaunchKernelGGL(scan_block_kernel, dim3((unsigned)nb), dim3(kScanThreads), 0, st, in, out, n, sums, total);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || nb == 1) return e;
  e = launch_scan_exclusive(sums, sums, nb, scratch + nb, st, total);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(scan_add_kernel, dim3((unsigned)nb), dim3(kScanThreads), 0, st, out, n, sums);
  return hipGetLastError();
}

hipError_t launch_iota_u64(uint64_t* p, uint64_t n, hipStream_t st) {
  hipLaunchKernelGGL(iota_u64_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, n);
  return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t st) {
  if (n == 0) return hipSuccess;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(fill_u32_kernel, dim3((unsigned)blocks), dim3(256), 0, st, p, n, v);
  return hipGetLastError();
}

hipError_t launch_bin_count(const SceneDesc* descs, int n_scenes, uint32_t chunk_min, uint32_t target,
                            uint32_t* chunk_pre, uint32_t* cbase, BatchCtl* ctl, uint32_t* places, uint32_t* row_count,
                            int max_tiles, int grid, hipStream_t st) {
  const BinPlan P{chunk_min, target, (uint32_t)grid, 2u * (uint32_t)max_tiles};
  if (n_scenes > kBinScenes) {
    hipLaunchKernelGGL(build_chunks_kernel, dim3(1), dim3(1024), 0, st, descs, n_scenes, P, chunk_pre, cbase, ctl);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  const size_t words = P.lds_counters + (n_scenes > kBinScenes ? 0u : bin_layout_words(n_scenes));
  hipLaunchKernelGGL(bin_kernel<0>, dim3(grid), dim3(256), words * sizeof(uint32_t), st, descs, n_scenes, P, chunk_pre,
                     cbase, ctl, places, row_count, nullptr, 0);
  return hipGetLastError();
}

hipError_t launch_bin_fill(const SceneDesc* descs, int n_scenes, uint32_t* chunk_pre, uint32_t* cbase, BatchCtl* ctl,
                           uint32_t* places, uint32_t* row_start, uint32_t* pairs, uint64_t pairs_cap, int max_tiles,
                           int grid, hipStream_t st) {
  hipLaunchKernelGGL(bin_kernel<1>, dim3(grid), dim3(256), (size_t)max_tiles * 2 * sizeof(uint32_t), st, descs, n_scenes,
                     BinPlan{}, chunk_pre, cbase, ctl, places, row_start, pairs, pairs_cap);
  return hipGetLastError();
}

uint64_t work_items_scratch_elems(int n_tiles_total) {
  return n_tiles_total <= kPlanTiles ? 1 : scan_scratch_elems(2 * (uint64_t)n_tiles_total + 1);
}

hipError_t launch_work_items(const SceneDesc* descs, const uint32_t* tile_scene, int n_tiles_total, int layers,
                             const uint32_t* row_count, uint32_t* row_start, uint32_t* scan_scratch, BatchCtl* ctl,
                             WorkItem* items, uint32_t items_cap, uint32_t* split_tiles, uint32_t split_cap,
                             uint64_t pairs_cap, uint32_t min_piece, uint32_t max_piece, uint32_t grid,
                             bool whole_images, hipStream_t st) {
  const PlanLimits L{pairs_cap, items_cap, split_cap, min_piece, max_piece, grid, whole_images ? 1u : 0u,
                     (uint32_t)layers};
  const int n = n_tiles_total;
  if (n <= kPlanTiles) {
    hipLaunchKernelGGL(plan_items_kernel, dim3(1), dim3(1024), 0, st, descs, tile_scene, n, row_count, ctl, row_start,
                       items, split_tiles, L);
    return hipGetLastError();
  }
  hipError_t e = launch_scan_exclusive(row_count, row_start, 2 * (uint64_t)n * layers + 1, scan_scratch, st, &ctl->total_pairs);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(tile_classes_kernel, dim3((n + 255) / 256), dim3(256), 0, st, n, row_start, ctl, L);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(write_items_kernel, dim3((n + 255) / 256), dim3(256), 0, st, descs, tile_scene, row_start, n, ctl,
                     items, split_tiles, L);
  return hipGetLastError();
}

// The tile kernel of a frame: tile edge 64 or 32; `packed_only` when every scene of the frame
// keeps two channels per LDS word. Workgroups per compute unit follow from the LDS: 64 with four
// planes 139.3 KB (one 1024-thread workgroup); 64 packed, with 1024 threads three planes and the
// streams' records and masks, 146.4 KB (one; so the kernel of runs too), with block = 512 two planes,
// 69.6 KB (two); 32 with four planes 36.9 KB and with two 18.4 KB (four of 256). The persistent
// grid fills every compute unit.
int tile_groups_per_cu(int tile, bool packed_only, int block, bool runs) {
  return tile == 32 ? 4 : packed_only && block == 512 && !runs ? 2 : 1;
}

hipError_t launch_tile_accum(const SceneDesc* descs, const uint32_t* pairs, const WorkItem* items,
                             const uint32_t* row_start, unsigned long long* split_fx, BatchCtl* ctl, int tile,
                             bool packed_only, int block, bool runs, bool count_work, int n_cu, hipStream_t st) {
  const int grid = n_cu * tile_groups_per_cu(tile, packed_only, block, runs);
#define LG_TILE_LAUNCH(T, P, B, ...)                                                                   \
  hipLaunchKernelGGL((tile_accum_kernel<T, P, B, bool(__VA_ARGS__ + 0)>), dim3(grid), dim3(B), 0, st, \
                     descs, pairs, items, row_start, split_fx, ctl, count_work ? 1u : 0u)
  if (runs) {
    LG_TILE_LAUNCH(64, true, 1024, 1);
  } else if (tile == 64) {
    if (packed_only && block == 512)
      LG_TILE_LAUNCH(64, true, 512);
    else if (packed_only)
      LG_TILE_LAUNCH(64, true, 1024);
    else
      LG_TILE_LAUNCH(64, false, 1024);
  } else {
    if (packed_only)
      LG_TILE_LAUNCH(32, true, 256);
    else
      LG_TILE_LAUNCH(32, false, 256);
  }
#undef LG_TILE_LAUNCH
  return hipGetLastError();
}

hipError_t launch_tile_merge(const SceneDesc* descs, const uint32_t* tile_scene, const uint32_t* row_start,
                             const uint32_t* split_tiles, const BatchCtl* ctl, unsigned long long* split_fx,
                             uint32_t split_cap, int tile, int n_cu, hipStream_t st) {
  static_assert(32 * 32 % kMergeBlock == 0, "a part is a whole number of blocks for both tile edges");
  hipLaunchKernelGGL(tile_merge_kernel, dim3(8 * n_cu), dim3(kMergeBlock), 0, st, descs, tile_scene, row_start,
                     split_tiles, ctl, split_fx, split_cap, tile * tile);
  return hipGetLastError();
}

hipError_t launch_pixels(int mode, float4* accum, ushort4* out16, uint64_t n, hipStream_t st) {
  const unsigned blocks = (unsigned)((n + 255) / 256);
  if (mode == 0)
    hipLaunchKernelGGL(pixels_kernel<0>, dim3(blocks), dim3(256), 0, st, accum, out16, n);
  else
    hipLaunchKernelGGL(pixels_kernel<1>, dim3(blocks), dim3(256), 0, st, accum, out16, n);
  return hipGetLastError();
}

}  // namespace lg
