// vt_render.hip -- fused primary + shadow render kernels for gfx950.
//
// One launch does what the reference splits into two dispatches plus a blit:
// raygen + traceMap + G-buffer store (primary.comp.glsl:23-69), shadow
// traceMap + traceEntities (secondary.comp.glsl:18-50) and the composite
// formula (blit.fragment.glsl:30-31).  The G-buffer round trip between the
// two passes stays in registers; the G-buffer images are only written when
// the caller asks for them.
//
// Launch shape: 256-thread blocks = 4 wave64s; each wave owns one tile of 64
// pixels (8x8, 16x4 or 32x2) for ray coherence, a block 2x2 tiles.  Block ids
// are remapped (xcd_remap) so that each XCD receives strips of neighbouring
// blocks spread over the whole image: its L2 working set stays local and
// no XCD is left with the costliest rows.  Each lane traces its primary ray,
// then (on a hit) its shadow ray.
//
// Rays end early where nothing is left to hit and cross clear space without
// lookups: with the clearance map (ClearMap in vt_trace.hpp) the line is
// followed from clear cube to clear cube first.  Lit shadow rays, which
// otherwise run to the edge of the grid, mostly end a few cells after their
// start, so the lanes of a wave finish close together.
#include "vt_pixel.hpp"

namespace vt {

// amdgpu_waves_per_eu: with the clearance map six waves per SIMD (80 VGPRs)
// -- six views of the 512^3 world at 1080p 290 us on average, 301 at seven
// (spills), 295 at five -- without it seven (72 VGPRs, no spills).
constexpr int kClearWaves = 6;
constexpr int kPlainWaves = 7;
// Launches without the clearance map of at most five waves per SIMD (96 VGPRs
// hold the iteration in flight) run ahead (dense_skip_ahead): all their waves
// are resident at once.
constexpr int kAheadWaves = 5;
// kSched: the launch order comes from the frame's tile schedule (`sched`);
// the kernels without it carry none of its code.
template <class L, bool kStats, int kShade, bool kSched>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(L::kClear ? kClearWaves : (L::kAhead ? kAheadWaves : kPlainWaves))))
void k_render_dense(
    DenseWorld w, ViewConsts v, ShadeConsts sc, FrameOut out, uint32_t* sched, uint32_t log2_tw,
    uint32_t blocks_x) {
  __shared__ SchedBlock sb;
  const uint32_t wave = threadIdx.x >> 6;
  uint32_t bid = xcd_remap(blockIdx.x, gridDim.x);
  if constexpr (kSched)
    bid = sched_begin(sched_geometry(sched, v.W, v.H, log2_tw, gridDim.x), bid, wave, sb);
  const uint32_t tw = 1u << log2_tw, th = 64u >> log2_tw;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t bx = bid % blocks_x, by = bid / blocks_x;
  const uint32_t px = bx * (2u * tw) + (wave & 1u) * tw + (lane & (tw - 1u));
  const uint32_t py = by * (2u * th) + (wave >> 1) * th + (lane >> log2_tw);
  Counters cnt = {0, 0, 0, 0, 0, 0, 0, 0};
  GradAcc gacc = grad_acc();
  if (px < v.W && py < v.H)
    trace_pixel_dense<L, kStats, kShade>(w, v, sc, out, px, py, cnt, gacc);
  if (kStats) flush_counters(out, cnt);
  if constexpr (kShade == kShadeLambertGrad) {
    flush_albedo(sc, gacc);
    flush_grad(sc, gacc);
  }
  if constexpr (kSched) sched_end(sb, lane);
}

// Seven waves per SIMD (72 VGPRs) without the clearance map; with it five (96
// VGPRs): the engine's map with long caps at 1600x900, six views, 245 us on
// average, 272 at six, 316 at seven; its own frame 138, 143 and 152 (fewer
// spills around its many literal-loop iterations).
// kClear: the empty-space runs take the clearance map.
// kSched: as k_render_dense.
template <bool kStats, bool kClear, bool kSched>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kClear ? 5 : 7))) void k_render_brickmap(
    BrickmapWorld w, ViewConsts v, ShadeConsts sc, FrameOut out, uint32_t* sched,
    uint32_t log2_tw, uint32_t blocks_x) {
  __shared__ SchedBlock sb;
  const uint32_t wave = threadIdx.x >> 6;
  uint32_t bid = xcd_remap(blockIdx.x, gridDim.x);
  if constexpr (kSched)
    bid = sched_begin(sched_geometry(sched, v.W, v.H, log2_tw, gridDim.x), bid, wave, sb);
  const uint32_t tw = 1u << log2_tw, th = 64u >> log2_tw;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t bx = bid % blocks_x, by = bid / blocks_x;
  const uint32_t px = bx * (2u * tw) + (wave & 1u) * tw + (lane & (tw - 1u));
  const uint32_t py = by * (2u * th) + (wave >> 1) * th + (lane >> log2_tw);
  const bool active = px < v.W && py < v.H;
  Counters cnt = {0, 0, 0, 0, 0, 0, 0, 0};
  if (active) {
    float d[3], e[3], inv[3];
    primary_ray(v, (float)w.dim, px, py, d, e, inv);
    GeneralHit g;
    if (!kStats && w.occ)
      trace_brickmap_fast<false, kClear, false>(w, e[0], e[1], e[2], d[0], d[1], d[2], inv,
                                                sc.max_primary, g);
    else
      trace_general<kStats>(w, e[0], e[1], e[2], d[0], d[1], d[2], sc.max_primary, g, cnt.l1f,
                            cnt.l0f);
    Primary p;
    p.hit = g.data != 0u;
    p.steps = g.steps;
    float sox = 0.f, soy = 0.f, soz = 0.f;
    bool shit = false;
    float shx = -1.0f, shy = -1.0f, shz = -1.0f;
    int ssteps = 0;
    if (p.hit) {
      p.face = g.face;
      p.voxel = (uint32_t)g.bx + w.dim * ((uint32_t)g.by + w.dim * (uint32_t)g.bz);
      p.data = g.data;
      p.material = bm_block(w, g.bx, g.by, g.bz) & 255u;
      p.sub = g.sub;
      p.hx = g.hx;
      p.hy = g.hy;
      p.hz = g.hz;
      shadow_origin(p, sc.flags, sox, soy, soz);
      store_hit_primary(v, sc, out, (size_t)py * v.W + px, p);
      const uint32_t data = p.data, info0 = hit_info(p.face, p.sub, p.material, false);
      const int psteps = p.steps;
      GeneralHit s;
      if (!kStats && w.occ) {
        // the sun is the same for every lane: a uniform branch
        if (sc.sun[0] >= 0.0f && sc.sun[1] >= 0.0f && sc.sun[2] >= 0.0f)
          trace_brickmap_fast<true, kClear, true>(w, sox, soy, soz, sc.sun[0], sc.sun[1],
                                                  sc.sun[2], sc.shadow.inv, sc.max_shadow, s);
        else
          trace_brickmap_fast<false, kClear, true>(w, sox, soy, soz, sc.sun[0], sc.sun[1],
                                                   sc.sun[2], sc.shadow.inv, sc.max_shadow, s);
      } else {
        trace_general<kStats>(w, sox, soy, soz, sc.sun[0], sc.sun[1], sc.sun[2], sc.max_shadow,
                              s, cnt.l1f, cnt.l0f);
      }
      shit = s.data != 0u;
      if (shit) {
        shx = s.hx;
        shy = s.hy;
        shz = s.hz;
      }
      ssteps = s.steps;
      store_hit_shadow_ref<kStats>(v, sc, out, px, py, data, info0, psteps, shit, shx, shy, shz, sox, soy,
                           soz, ssteps, cnt);
    }
    if (!p.hit) {  // a hit's stores are made above
      GradAcc gacc = grad_acc();
      write_pixel<kShadeRef, kStats>(v, sc, out, px, py, p, shit, shx, shy, shz, sox, soy, soz, ssteps,
                             cnt, nullptr, gacc);
    }
  }
  if (kStats) flush_counters(out, cnt);
  if constexpr (kSched) sched_end(sb, lane);
}

static void grid_shape(const ViewConsts& v, TileShape tile, uint32_t& blocks_x, uint32_t& nblocks) {
  uint32_t tw = 1u << tile.log2_w, th = 64u >> tile.log2_w;
  blocks_x = (v.W + 2u * tw - 1u) / (2u * tw);
  uint32_t blocks_y = (v.H + 2u * th - 1u) / (2u * th);
  nblocks = blocks_x * blocks_y;
}


template <class L, bool kStats, bool kSched>
static void launch_dense_shade(const DenseWorld& w, const ViewConsts& v, const ShadeConsts& sc,
                               const FrameOut& out, uint32_t* sd, uint32_t log2_w,
                               uint32_t blocks_x, dim3 grid, hipStream_t stream) {
  switch (shade_mode(sc.flags)) {
    case kShadeLambertGrad:
      hipLaunchKernelGGL((k_render_dense<L, kStats, kShadeLambertGrad, kSched>), grid, dim3(256),
                         0, stream, w, v, sc, out, sd, log2_w, blocks_x);
      break;
    case kShadeLambert:
      hipLaunchKernelGGL((k_render_dense<L, kStats, kShadeLambert, kSched>), grid, dim3(256), 0,
                         stream, w, v, sc, out, sd, log2_w, blocks_x);
      break;
    default:
      hipLaunchKernelGGL((k_render_dense<L, kStats, kShadeRef, kSched>), grid, dim3(256), 0,
                         stream, w, v, sc, out, sd, log2_w, blocks_x);
  }
}

// The traversal variant of a dense launch (kSched: as k_render_dense).
template <bool kSched>
static void launch_dense_select(const DenseWorld& w, uint32_t traversal, const ViewConsts& v,
                                const ShadeConsts& sc, const FrameOut& out, uint32_t* sd,
                                uint32_t lw, uint32_t blocks_x, dim3 grid, uint32_t compute_units,
                                hipStream_t stream) {
  const bool stats = out.stats != nullptr;
  if (traversal == VT_TRAVERSAL_BITMASK) {
    if (stats)
      launch_dense_shade<BitmaskLookup, true, kSched>(w, v, sc, out, sd, lw, blocks_x, grid, stream);
    else
      launch_dense_shade<BitmaskLookup, false, kSched>(w, v, sc, out, sd, lw, blocks_x, grid, stream);
  } else if (traversal == VT_TRAVERSAL_BITMASK8) {
    if (stats)
      launch_dense_shade<BitmaskLookup8, true, kSched>(w, v, sc, out, sd, lw, blocks_x, grid, stream);
    else
      launch_dense_shade<BitmaskLookup8, false, kSched>(w, v, sc, out, sd, lw, blocks_x, grid, stream);
  } else {
    const bool long_caps = sc.max_primary >= kLongCap || sc.max_shadow >= kLongCap;
    if (stats && w.clear_bytes)  // statistics of the steps executed
      launch_dense_shade<FlatLookupClear, true, kSched>(w, v, sc, out, sd, lw, blocks_x, grid, stream);
    else if (stats)
      launch_dense_shade<FlatLookup, true, kSched>(w, v, sc, out, sd, lw, blocks_x, grid, stream);
    else if (w.clear_bytes)
      launch_dense_shade<FlatLookupClear, false, kSched>(w, v, sc, out, sd, lw, blocks_x, grid, stream);
    else if (grid.x <= kAheadWaves * compute_units)
      launch_dense_shade<FlatLookupAhead, false, kSched>(w, v, sc, out, sd, lw, blocks_x, grid, stream);
    else if (long_caps)
      launch_dense_shade<FlatLookupLong, false, kSched>(w, v, sc, out, sd, lw, blocks_x, grid, stream);
    else
      launch_dense_shade<FlatLookup, false, kSched>(w, v, sc, out, sd, lw, blocks_x, grid, stream);
  }
}

// The tile schedule is taken for frames with a buffer and a step cap of at
// least kLongCap.  With the shaders' own caps (192 / 48) the blocks' costs
// are flat and the costliest-first order measured slower: the engine's frame
// +8.6% at 1280x720, +19% at 1920x1080, the 512^3 world +4% at 1280x720;
// with caps of 2048 it gains 7-25% on both worlds at 1280x720..2560x1440.
static bool sched_taken(const uint32_t* schedule, const ShadeConsts& sc) {
  return schedule && (sc.max_primary >= kLongCap || sc.max_shadow >= kLongCap);
}

hipError_t launch_render_dense(const DenseWorld& w_in, uint32_t traversal, const ViewConsts& v,
                               const ShadeConsts& sc_in, const FrameOut& out, uint32_t* schedule,
                               TileShape tile, uint32_t compute_units, hipStream_t stream) {
  DenseWorld w = w_in;
  // Where step counts are observed (stored, or counted as traceMap's by
  // statistics without the clearance map) no ray ends early, at the reach box
  // neither.
  if (out.steps) w.clear_bytes = 0;
  if (out.steps || (out.stats && !w.clear_bytes)) reach_everywhere(w.reach_lo, w.reach_hi);
  ShadeConsts sc = sc_in;
  sc.shadow = make_ray_consts(sc.sun[0], sc.sun[1], sc.sun[2], w.mx, w.my, w.mz);
  uint32_t blocks_x, nblocks;
  grid_shape(v, tile, blocks_x, nblocks);
  if (schedule && nblocks > VT_SCHEDULE_BLOCKS(v.W, v.H)) return hipErrorInvalidValue;
  const dim3 grid(nblocks);
  if (sched_taken(schedule, sc))
    launch_dense_select<true>(w, traversal, v, sc, out, schedule, tile.log2_w, blocks_x, grid,
                              compute_units, stream);
  else
    launch_dense_select<false>(w, traversal, v, sc, out, nullptr, tile.log2_w, blocks_x, grid,
                               compute_units, stream);
  return hipGetLastError();
}

template <bool kStats, bool kClear>
static void launch_brickmap(bool sched, const BrickmapWorld& w, const ViewConsts& v,
                            const ShadeConsts& sc, const FrameOut& out, uint32_t* schedule,
                            uint32_t lw, uint32_t blocks_x, dim3 grid, hipStream_t stream) {
  if (sched)
    hipLaunchKernelGGL((k_render_brickmap<kStats, kClear, true>), grid, dim3(256), 0, stream, w, v,
                       sc, out, schedule, lw, blocks_x);
  else
    hipLaunchKernelGGL((k_render_brickmap<kStats, kClear, false>), grid, dim3(256), 0, stream, w,
                       v, sc, out, nullptr, lw, blocks_x);
}

hipError_t launch_render_brickmap(const BrickmapWorld& w_in, const ViewConsts& v,
                                  const ShadeConsts& sc, const FrameOut& out, uint32_t* schedule,
                                  TileShape tile, hipStream_t stream) {
  BrickmapWorld w = w_in;
  // a map of fewer blocks a side than two empty-space iterations take steps
  // (8^3: one chunk) stays on the literal loop (dense_left_grid)
  if (w.dim < 2u * (uint32_t)kSkipLong) w.occ = nullptr;
  // step counts stored, or statistics (of traceMap's steps on this layout):
  // no early end of rays
  if (out.steps || out.stats) w.clear_bytes = 0;
  uint32_t blocks_x, nblocks;
  grid_shape(v, tile, blocks_x, nblocks);
  if (schedule && nblocks > VT_SCHEDULE_BLOCKS(v.W, v.H)) return hipErrorInvalidValue;
  const dim3 grid(nblocks);
  const bool sched = sched_taken(schedule, sc);
  const uint32_t lw = tile.log2_w;
  if (out.stats)
    launch_brickmap<true, false>(sched, w, v, sc, out, schedule, lw, blocks_x, grid, stream);
  else if (w.occ && w.clear_bytes)
    launch_brickmap<false, true>(sched, w, v, sc, out, schedule, lw, blocks_x, grid, stream);
  else
    launch_brickmap<false, false>(sched, w, v, sc, out, schedule, lw, blocks_x, grid, stream);
  return hipGetLastError();
}

}  // namespace vt
