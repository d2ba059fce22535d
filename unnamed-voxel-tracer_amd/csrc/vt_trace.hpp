// vt_trace.hpp -- device-side REF voxel traversal for gfx950.
//
// Restates traceMap (assets/shaders/map.glsl:83-168) and its callers
// (primary.comp.glsl:23-69, secondary.comp.glsl:18-50, blit.fragment.glsl:30-31)
// in binary32 with the same operation order as the CPU restatement: built with
// -ffp-contract=off and correctly rounded division/sqrt, every multiply and add
// rounds once, so hits are bit-exact.
//
// Two traversal loops:
//  * dense_begin + dense_run: worlds where one grid voxel is one reference
//    block whose atlas model is a solid cube.  After the first lookup
//    traceMap never leaves the block level (stepSize 3), so the block
//    coordinates G = gridsCoords >> 3 live in a Morton code while
//    withinGridCoords stays in x8 units; this is the same recurrence, with
//    pos >> 3 == G + (int(within) >> 3).
//  * The literal general loop (trace_general) with both levels, used for the
//    reference brickmap + atlas layout.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vt {

// ---------------------------------------------------------------------------
// binary32 helpers (same definitions as the CPU restatement)
// ---------------------------------------------------------------------------

// ivec3(float) at ray set-up: truncation toward zero, NaN -> 0, saturating,
// which is what the conversion instruction does (C++'s own conversion is
// undefined out of range).
__device__ __forceinline__ int f2i_sat(float x) {
  int i;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(i) : "v"(x));
  return i;
}

// Several quotients by one divisor share its reciprocal in binary64:
// recip64's is within 2^-52 of 1 / x (a hardware estimate good to 2^-22 and
// one third-order step), so a * recip64(x) is within 2^-51 of a / x, and no
// quotient of two binary32 numbers lies closer than 2^-50 to a midpoint of two
// binary32 numbers without being one -- which a normal one cannot be, as the
// midpoint's 25 bits would have to divide the 24 of a.  So rounding the
// product gives the correctly rounded quotient, at 3 instructions (and 6 once
// for the reciprocal) where a division takes 11.  For finite x of ordinary
// size (divisible) and quotients in the normal range; 0 / x keeps its sign.
// What a pixel costs besides its rays' steps came to 900 instructions of the
// 2600-6600 a wave takes; with the shared quotients, the constants of a
// launch's hits in ShadeConsts, may_meet_entities and sky_base it
// is under half of that (six views at 1080p 272 -> 252 us, an 853x479 frame with
// its G-buffer 30.8 -> 22.3, the engine's 720p frame 134 -> 122, a batch of 64
// views 2180 -> 1970).
__device__ __forceinline__ double recip64(float x) {
  const double d = (double)x, y = (double)__builtin_amdgcn_rcpf(x);
  const double e = fma(-d, y, 1.0);
  return fma(y, fma(e, e, e), y);
}
__host__ __device__ __forceinline__ float quotient(float a, double recip) {
  return (float)((double)a * recip);
}
__device__ __forceinline__ bool divisible(float x) {
  return fabsf(x) >= 0x1p-60f && fabsf(x) <= 0x1p60f;
}

// b / 255 for the integers 0 .. 255, correctly rounded: the product with the
// rounded reciprocal and one correction.
__host__ __device__ __forceinline__ float over255(float b) {
  const float q = b * (1.0f / 255.0f);
  return fmaf(fmaf(q, -255.0f, b), 1.0f / 255.0f, q);
}

__host__ __device__ __forceinline__ float len3(float x, float y, float z) {
  float s = x * x;
  s = s + y * y;
  s = s + z * z;
  return sqrtf(s);
}

// rgba8 UNORM store followed by a load (gbuffer.zig:10-13 formats).
__host__ __device__ __forceinline__ float unorm8(float x) {
  float c = fminf(fmaxf(x, 0.0f), 1.0f);
  float b = floorf(c * 255.0f + 0.5f);
  return over255(b);
}

// RGBA8 framebuffer store of a colour: per channel clamp to [0,1], round to
// nearest (the unorm8 rule), R in the low byte.
__device__ __forceinline__ uint32_t pack_unorm8(float4 c) {
  const float v[4] = {c.x, c.y, c.z, c.w};
  uint32_t r = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float k = fminf(fmaxf(v[i], 0.0f), 1.0f);
    r |= (uint32_t)floorf(k * 255.0f + 0.5f) << (8 * i);
  }
  return r;
}

// Present pass of one pixel (blit.fragment.glsl:32-35): texPos is the pixel
// centre of the full-screen quad, ((x+0.5)/W, (y+0.5)/H).
__device__ __forceinline__ float4 present_pixel(float4 c, uint32_t x, uint32_t y, uint32_t W,
                                                uint32_t H) {
  const float u = ((float)x + 0.5f) / (float)W;
  const float v = ((float)y + 0.5f) / (float)H;
  const float du = u - 0.5f, dv = v - 0.5f;
  float d2 = du * du;
  d2 = d2 + dv * dv;
  if (sqrtf(d2) <= 0.002f) {  // crosshair: mix(color, vec4(1,1,1,0.4), 0.5)
    c = make_float4(c.x * 0.5f + 0.5f, c.y * 0.5f + 0.5f, c.z * 0.5f + 0.5f,
                    c.w * 0.5f + 0.4f * 0.5f);
  }
  const float a = u * (1.0f - u), b = v * (1.0f - v);
  const float g = powf((a * b) * 15.0f, 0.6f * 0.3f);  // vignette
  return make_float4(g * c.x, g * c.y, g * c.z, g * c.w);
}

// normals[] (map.glsl:72-79), face id 1..6
__device__ __forceinline__ void face_normal(int face, float& nx, float& ny, float& nz) {
  nx = face == 1 ? -1.0f : (face == 2 ? 1.0f : 0.0f);
  ny = face == 3 ? -1.0f : (face == 4 ? 1.0f : 0.0f);
  nz = face == 5 ? -1.0f : (face == 6 ? 1.0f : 0.0f);
}

// ---------------------------------------------------------------------------
// per-view constants
// ---------------------------------------------------------------------------
struct ViewConsts {
  float pos[3];     // C_position.xyz
  float view[16];   // C_view, column-major
  float tan_half;   // tan(fov/2), evaluated once per view on the host
  uint32_t W, H;
  float aspect;         // H / W
  double inv_w, inv_h;  // 1 / W and 1 / H, for quotient()
};

// primary.comp.glsl:31-39
__device__ __forceinline__ void raygen(const ViewConsts& v, uint32_t px, uint32_t py, float& dx,
                                       float& dy, float& dz) {
  float u = quotient((float)px, v.inv_w);
  float w = quotient((float)py, v.inv_h);
  u = u * 2.0f - 1.0f;
  w = w * 2.0f - 1.0f;
  w = w * v.aspect;
  u = u * v.tan_half;
  w = w * v.tan_half;
  float r[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    float acc = v.view[0 * 4 + i] * u;
    acc = acc + v.view[1 * 4 + i] * w;
    acc = acc + v.view[2 * 4 + i] * 1.0f;
    acc = acc + v.view[3 * 4 + i] * 1.0f;
    r[i] = acc;
  }
  float s = r[0] * r[0];
  s = s + r[1] * r[1];
  s = s + r[2] * r[2];
  s = s + r[3] * r[3];
  float l = sqrtf(s);
  if (divisible(l)) {
    const double y = recip64(l);
    dx = quotient(r[0], y);
    dy = quotient(r[1], y);
    dz = quotient(r[2], y);
  } else {
    dx = r[0] / l;
    dy = r[1] / l;
    dz = r[2] / l;
  }
}

// intersectAABB (map.glsl:21-29)
__device__ __forceinline__ void intersect_aabb(float ox, float oy, float oz, float dx, float dy,
                                               float dz, float x0, float y0, float z0, float x1,
                                               float y1, float z1, float& tn, float& tf) {
  float ax = (x0 - ox) / dx, bx = (x1 - ox) / dx;
  float ay = (y0 - oy) / dy, by = (y1 - oy) / dy;
  float az = (z0 - oz) / dz, bz = (z1 - oz) / dz;
  float t1x = fminf(ax, bx), t2x = fmaxf(ax, bx);
  float t1y = fminf(ay, by), t2y = fmaxf(ay, by);
  float t1z = fminf(az, bz), t2z = fmaxf(az, bz);
  tn = fmaxf(fmaxf(t1x, t1y), t1z);
  tf = fminf(fminf(t2x, t2y), t2z);
}

// The primary ray of a pixel (primary.comp.glsl:31-43): its direction, where
// it enters the map's box [0, D]^3 (the eye if inside), less the 0.001 offset,
// and 1 / d after traceMap's zero substitution.  The nine quotients of the
// three components come from three reciprocals.
__device__ __forceinline__ void primary_ray(const ViewConsts& v, float D, uint32_t px, uint32_t py,
                                            float (&d)[3], float (&e)[3], float (&inv)[3]) {
  raygen(v, px, py, d[0], d[1], d[2]);
  float tn, tf;
  if (divisible(d[0]) && divisible(d[1]) && divisible(d[2])) {
    float t1[3], t2[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const double y = recip64(d[i]);
      const float a = quotient(0.0f - v.pos[i], y), b = quotient(D - v.pos[i], y);
      t1[i] = fminf(a, b);
      t2[i] = fmaxf(a, b);
      inv[i] = (float)y;
    }
    tn = fmaxf(fmaxf(t1[0], t1[1]), t1[2]);
    tf = fminf(fminf(t2[0], t2[1]), t2[2]);
  } else {
    intersect_aabb(v.pos[0], v.pos[1], v.pos[2], d[0], d[1], d[2], 0.0f, 0.0f, 0.0f, D, D, D, tn,
                   tf);
#pragma unroll
    for (int i = 0; i < 3; i++) inv[i] = 1.0f / (d[i] == 0.0f ? 0.001f : d[i]);
  }
  const float tc = fmaxf(tn, 0.0f);
#pragma unroll
  for (int i = 0; i < 3; i++) e[i] = (v.pos[i] + d[i] * tc) - 0.001f;
}

// Whether the line o + d t can meet one of traceEntities' boxes: the slab test
// of the box around all five, wider by 0.01 on each side.  inv = 1 / d,
// finite.  The widening outweighs the rounding of both tests (under 2e-3
// voxel for |o| up to 4096), so each slab interval here holds the ones that
// trace_entities computes, and a ray culled here meets none.  25
// instructions where the exact test of the five boxes (30 divisions) takes
// 400, which ran for every hit.
__device__ __forceinline__ bool may_meet_entities(float ox, float oy, float oz,
                                                  const float* inv) {
  const float ax = (250.99f - ox) * inv[0], bx = (258.01f - ox) * inv[0];
  const float ay = (20.99f - oy) * inv[1], by = (22.01f - oy) * inv[1];
  const float az = (255.99f - oz) * inv[2], bz = (262.01f - oz) * inv[2];
  const float tn = fmaxf(fmaxf(fminf(ax, bx), fminf(ay, by)), fminf(az, bz));
  const float tf = fminf(fminf(fmaxf(ax, bx), fmaxf(ay, by)), fmaxf(az, bz));
  return tn <= tf;
}

// traceEntities occlusion (map.glsl:172-201); the code after the return on
// map.glsl:201 is unreachable in the reference.
__device__ __forceinline__ bool trace_entities(float ox, float oy, float oz, float dx, float dy,
                                               float dz, float max_distance) {
  const float PX[5] = {256.f, 251.f, 253.f, 251.f, 257.f};
  const float PY[5] = {21.f, 21.f, 21.f, 21.f, 21.f};
  const float PZ[5] = {256.f, 259.f, 256.f, 256.f, 261.f};
  float prevD = __builtin_inff();
  int id = -1;
#pragma unroll
  for (int i = 0; i < 5; i++) {
    float dist = len3(ox - PX[i], oy - PY[i], oz - PZ[i]);
    if (dist >= max_distance) continue;
    float tn, tf;
    intersect_aabb(ox, oy, oz, dx, dy, dz, PX[i], PY[i], PZ[i], PX[i] + 1.0f, PY[i] + 1.0f,
                   PZ[i] + 1.0f, tn, tf);
    if (tf >= tn && prevD >= tf) {
      id = i;
      prevD = tf;
    }
  }
  return id >= 0;  // the re-test on map.glsl:199-200 repeats a test that passed
}

// SkyDome2 (camera.glsl:11-19) in two halves.  The clamped cosine between the
// normalised sun and the normalised ray, and the colour before the sun's
// glow, are the same for every hit of a launch, and made on the host (each
// operation rounded as on the device); the powers are taken on the device,
// whose pow the colour bytes have always been rounded from.
struct SkyBase {
  float sv;       // clamp(dot(sun, ray), 0, 1.2)
  float r, g, b;  // colour without the glow
};
__host__ __device__ inline SkyBase sky_base(const float* sun_n, float rnx, float rny, float rnz,
                                            float ry) {
  SkyBase s;
  float dt = sun_n[0] * rnx;
  dt = dt + sun_n[1] * rny;
  dt = dt + sun_n[2] * rnz;
  s.sv = fminf(fmaxf(dt, 0.0f), 1.2f);
  const float k = ry * 0.2f;
  s.r = ((0.6f - k * 1.0f) + 0.075f);
  s.g = ((0.71f - k * 0.5f) + 0.075f);
  s.b = ((0.75f - k * 1.0f) + 0.075f);
  return s;
}
// pow(0, y) = 0 exactly: the sky away from the sun needs no powers.
__device__ __forceinline__ void sky_glow(const SkyBase& s, float& r, float& g, float& b) {
  float p8 = s.sv, p3 = s.sv;
  if (s.sv != 0.0f) {
    p8 = powf(s.sv, 8.0f);
    p3 = powf(s.sv, 3.0f);
  }
  r = s.r + (0.4f * 1.0f) * p8;
  g = s.g + (0.4f * 0.6f) * p8;
  b = s.b + (0.4f * 0.1f) * p8;
  r = r + 0.2f * p3;
  g = g + 0.08f * p3;
  b = b + 0.04f * p3;
}

__device__ __forceinline__ void sky(const float* sun_n, float rx, float ry, float rz, float& r,
                                    float& g, float& b) {
  const float lr = len3(rx, ry, rz);
  float nx, ny, nz;
  if (divisible(lr)) {
    const double y = recip64(lr);
    nx = quotient(rx, y);
    ny = quotient(ry, y);
    nz = quotient(rz, y);
  } else {
    nx = rx / lr;
    ny = ry / lr;
    nz = rz / lr;
  }
  sky_glow(sky_base(sun_n, nx, ny, nz, ry), r, g, b);
}

// ---------------------------------------------------------------------------
// dense worlds: Morton-ordered voxels
// ---------------------------------------------------------------------------
// The material bytes are stored in Morton (Z) order: voxel (x,y,z) at
// code = interleave(x, y, z) (x in bits 0,3,6,..., y in 1,4,..., z in 2,5,...).
// A 128-byte cache line then holds a ~5^3 neighbourhood, a 4^3 brick is 64
// consecutive codes and a 16^3 region 4096, whatever direction a ray moves.
// The two occupancy levels fall out of the same order: L0 word code >> 6 has
// bit code & 63, L1 word code >> 12 has bit (code >> 6) & 63.
struct DenseWorld {
  const uint8_t* vox;       // material byte of voxel (x,y,z) at morton(x,y,z)
  const uint64_t* l0;       // 4^3 bricks: bit per voxel
  const uint64_t* l1;       // 16^3 regions: bit per nonempty 4^3 brick
  const uint64_t* l1b;      // 32^3 regions: bit per nonempty 8^3 brick
  const uint32_t* palette;  // RGBA8 colour of material k (the solid atlas cube)
  uint32_t dim;             // voxels per axis (MAP_DIMENSION), a power of two
  uint32_t log2dim;
  uint32_t mx, my, mz;      // dilated masks of x, y, z over 3*log2(dim) bits
  uint32_t nvox;            // dim^3 (bytes of vox)
  const uint32_t* prefix;   // compact albedo index: occupied voxels before each
                            // L0 word (null until built)
  // clearance map (see ClearMap below); clear_bytes 0 = not used
  const uint8_t* clear;
  uint32_t clear_bytes, clear_oct_bytes;
  // the box of the nonempty voxels widened by the traversal's reach
  // (line_meets_reach); the whole grid when the world is empty; everywhere
  // (reach_everywhere) when step counts are observed
  float reach_lo[3], reach_hi[3];
};

__device__ __forceinline__ uint32_t part1by2(uint32_t x) {
  x &= 0x000003FFu;
  x = (x | (x << 16)) & 0xFF0000FFu;
  x = (x | (x << 8)) & 0x0300F00Fu;
  x = (x | (x << 4)) & 0x030C30C3u;
  x = (x | (x << 2)) & 0x09249249u;
  return x;
}
__device__ __forceinline__ uint32_t compact1by2(uint32_t x) {
  x &= 0x09249249u;
  x = (x | (x >> 2)) & 0x030C30C3u;
  x = (x | (x >> 4)) & 0x0300F00Fu;
  x = (x | (x >> 8)) & 0xFF0000FFu;
  x = (x | (x >> 16)) & 0x000003FFu;
  return x;
}
__device__ __forceinline__ uint32_t morton3(uint32_t x, uint32_t y, uint32_t z) {
  return part1by2(x) | (part1by2(y) << 1) | (part1by2(z) << 2);
}

__device__ __forceinline__ bool in_dim(const DenseWorld& w, int bx, int by, int bz) {
  return ((uint32_t)bx < w.dim) & ((uint32_t)by < w.dim) & ((uint32_t)bz < w.dim);
}

// Steps per iteration of the empty-space phase (dense_skip_empty): 6 for
// frames with a step cap of at least 512, 5 below.  Measured on MI355X with
// the free-region test: C1 at 1080p 0.2740 / 0.2725 / 0.2710 ms at K = 6 /
// 7 / 8 against 0.2796 at 5; C3's views 0.1065 ms against 0.1117; the C1
// world in the reference layout 0.2858 (6) / 0.2892 (7) / 0.292 (8) against
// 0.2869 (5); the engine's own frame (caps 192/48, short runs between model
// blocks) 0.2747 at 5 against 0.2972 at 6 and 0.335 at 7.
// With the clearance map (near something only) 5: the batch 2.32 ms against
// 2.38 at 6, the engine's map with long caps 272 us against 275.
constexpr int kSkipShort = 5;
constexpr int kSkipLong = 6;
constexpr int kSkipClear = 5;
constexpr int kLongCap = 512;
// Steps per turn of the loop without lookups (clear_advance).
constexpr int kClearSteps = 4;

// Occupancy probe strategies (identical answers by contract).
struct FlatLookup {
  // one byte gather per probe; returns the material (0 = empty)
  static constexpr bool kPrefetch = true;  // probes have no state: run ahead
  static constexpr bool kClear = false;    // no clearance map
  static constexpr bool kAhead = false;    // no iteration ahead
  static constexpr int kSkip = kSkipShort;  // empty-space iteration length
  __device__ __forceinline__ void reset() {}
  template <bool kStats>
  __device__ __forceinline__ uint32_t probe(const DenseWorld& w, uint32_t code, uint32_t&,
                                            uint32_t&) {
    return w.vox[code];
  }
  __device__ __forceinline__ uint32_t material(const DenseWorld&, uint32_t, uint32_t v,
                                               uint32_t&) {
    return v;
  }
};

// The 2-level occupancy probe: a region word (one bit per brick) and the
// probed voxel's 64-bit leaf word, both kept in registers between probes.
//  kBrick = 4: 4^3 bricks in 16^3 regions -- region word l1[code >> 12],
//              bit (code >> 6) & 63; the brick is the leaf word l0[code >> 6].
//  kBrick = 8: 8^3 bricks in 32^3 regions -- region word l1b[code >> 15],
//              bit (code >> 9) & 63; an occupied 8^3 brick's voxels are the
//              8 leaf words l0[code >> 6], of which the one holding the
//              probed 4^3 sub-brick is fetched.
// A leaf word is fetched only when its brick is marked occupied, a region
// word only when the region changes.
template <uint32_t kBrick>
struct BitmaskLookupT {
  static_assert(kBrick == 4 || kBrick == 8, "4^3 or 8^3 bricks");
  static constexpr bool kPrefetch = false;
  static constexpr bool kClear = false;
  static constexpr bool kAhead = false;
  static constexpr int kSkip = kSkipShort;  // (the plain loop has no empty-space phase)
  static constexpr uint32_t kBrickShift = kBrick == 8 ? 9u : 6u;  // log2 codes per brick
  uint32_t brick, region, leaf;
  uint64_t bword, rword;
  bool bset;  // the current brick is marked occupied
  __device__ __forceinline__ void reset() {
    brick = 0xFFFFFFFFu;
    region = 0xFFFFFFFFu;
    leaf = 0xFFFFFFFFu;
    bword = 0;
    rword = 0;
    bset = false;
  }
  template <bool kStats>
  __device__ __forceinline__ uint32_t probe(const DenseWorld& w, uint32_t code, uint32_t& l1f,
                                            uint32_t& l0f) {
    const uint32_t lf = code >> 6;
    if (lf != leaf) {
      leaf = lf;
      const uint32_t bk = code >> kBrickShift;
      if (bk != brick) {
        brick = bk;
        const uint32_t rk = bk >> 6;
        if (rk != region) {
          region = rk;
          rword = kBrick == 8 ? w.l1b[rk] : w.l1[rk];
          if (kStats) l1f++;
        }
        bset = ((rword >> (bk & 63u)) & 1ull) != 0ull;
      }
      bword = 0;
      if (bset) {
        bword = w.l0[lf];
        if (kStats) l0f++;
      }
    }
    return (uint32_t)(bword >> (code & 63u)) & 1u;
  }
  __device__ __forceinline__ uint32_t material(const DenseWorld& w, uint32_t code, uint32_t,
                                               uint32_t& leaf_reads) {
    leaf_reads++;
    return w.vox[code];
  }
};
using BitmaskLookup = BitmaskLookupT<4>;
using BitmaskLookup8 = BitmaskLookupT<8>;

// The flat lookup with the clearance map (see ClearMap below): empty stretches
// of a ray are crossed without lookups, and a ray whose line meets nothing
// more ends.
struct FlatLookupClear : FlatLookup {
  static constexpr bool kClear = true;
  static constexpr int kSkip = kSkipClear;
};

// The flat lookup for frames with long step caps: the longer empty-space
// iteration, no clearance map.
struct FlatLookupLong : FlatLookup {
  static constexpr int kSkip = kSkipLong;
};

// For launches whose waves are all resident at once (dense_skip_ahead).
struct FlatLookupAhead : FlatLookup {
  static constexpr int kSkip = kSkipLong;
  static constexpr bool kAhead = true;
};

// Result of one traceMap call in a dense world.
struct DenseHit {
  bool hit;
  int face;             // 1..6
  int bx, by, bz;       // block coordinates (pos >> 3)
  uint32_t code;        // morton(bx, by, bz)
  uint32_t v;           // probe value at the hit (flat: the material byte)
  uint32_t sub;         // pos % 8 packed x + 8y + 64z
  float hx, hy, hz;     // hit_pos = gridsCoords + withinGridCoords
  int steps;
};

// Ray state at the block level.
struct DenseRay {
  float wx, wy, wz;   // withinGridCoords, x8 units
  float dx, dy, dz;   // rayDir after the zero substitution
  float ix, iy, iz;   // 1 / rayDir
  float Px, Py, Pz;   // float(rayPositivity << 3)
  float Ax, Ay, Az;   // float((1 - rayPositivity) << 3) * 0.999f
  int px, py, pz;     // rayPositivity
  uint32_t c;         // Morton code of G = gridsCoords >> 3, axes the ray
                      // travels negatively stored complemented
  uint32_t flip;      // the complemented axes' masks; address = c ^ flip
  int steps, max_steps;
  int blind;          // steps whose lookups can only read empty (blind_steps);
                      // after dense_run_prefetch, the steps taken without them
};

// The per-ray constants of traceMap's set-up (map.glsl:85-97): the 0.001
// substitution of zero direction components, positivity, 1/d, and the
// block-level crossing and re-anchoring constants.  A __host__ __device__
// function: the shadow rays' direction is the sun for every pixel, so their
// constants are computed once per launch on the host (binary32, correctly
// rounded division, like the device) and reach the kernels as arguments --
// scalar registers instead of per-lane copies of uniform values.
struct RayConsts {
  float d[3];    // rayDir after the zero substitution
  float inv[3];  // 1 / rayDir
  float P[3];    // float(rayPositivity << 3)
  float A[3];    // float((1 - rayPositivity) << 3) * 0.999f
  int pos[3];    // rayPositivity
  uint32_t flip; // masks of the axes the ray travels negatively
};

// The same with inv = 1 / d after the substitution at hand.
__host__ __device__ inline RayConsts ray_consts(const float* d, const float* inv, uint32_t mx,
                                                uint32_t my, uint32_t mz) {
  RayConsts k;
  const uint32_t m[3] = {mx, my, mz};
  k.flip = 0u;
  for (int i = 0; i < 3; i++) {
    k.d[i] = d[i] == 0.0f ? 0.001f : d[i];
    k.pos[i] = k.d[i] > 0.0f ? 1 : 0;
    k.inv[i] = inv[i];
    k.P[i] = k.pos[i] ? 8.0f : 0.0f;
    k.A[i] = k.pos[i] ? 0.0f : 8.0f * 0.999f;
    k.flip |= k.pos[i] ? 0u : m[i];
  }
  return k;
}

__host__ __device__ inline RayConsts make_ray_consts(float dx, float dy, float dz, uint32_t mx,
                                                     uint32_t my, uint32_t mz) {
  const float d[3] = {dx, dy, dz};
  const float inv[3] = {1.0f / (dx == 0.0f ? 0.001f : dx), 1.0f / (dy == 0.0f ? 0.001f : dy),
                        1.0f / (dz == 0.0f ? 0.001f : dz)};
  return ray_consts(d, inv, mx, my, mz);
}

__device__ __forceinline__ void dense_ray_from(DenseRay& r, const RayConsts& k) {
  r.dx = k.d[0];
  r.dy = k.d[1];
  r.dz = k.d[2];
  r.ix = k.inv[0];
  r.iy = k.inv[1];
  r.iz = k.inv[2];
  r.Px = k.P[0];
  r.Py = k.P[1];
  r.Pz = k.P[2];
  r.Ax = k.A[0];
  r.Ay = k.A[1];
  r.Az = k.A[2];
  r.px = k.pos[0];
  r.py = k.pos[1];
  r.pz = k.pos[2];
  r.flip = k.flip;
}

__device__ __forceinline__ void dense_ray_consts(DenseRay& r, const DenseWorld& w, float dx,
                                                 float dy, float dz) {
  dense_ray_from(r, make_ray_consts(dx, dy, dz, w.mx, w.my, w.mz));
}

// Can traceMap's block-level walk from e (voxel units) along d probe a
// nonempty voxel?  Only if the line e + d t, t >= 0, meets the box of the
// nonempty voxels widened by how far a probe can lie from that line:
//   * every step moves the position along d up to binary32 rounding (< 1e-6
//     sub-voxel per step: 0.01 voxel over 65,535 steps);
//   * a step across a negative axis re-anchors within at 8 x 0.999 instead
//     of 8, 0.001 voxel off the line per crossing, at most dim crossings per
//     axis inside the grid (the walk ends where it leaves it);
//   * the probed voxel is the position's, or the next one on a positive axis
//     whose within reached 8: within 2 voxels of the position;
// so the widening of 2.5 + dim / 1000 voxels (wide_margin) covers all three
// with room for the rounding of this test.  A ray whose line misses it ends
// as a miss; only its step count differs from traceMap's.
__host__ __device__ __forceinline__ float wide_margin(uint32_t dim) {
  return 2.5f + (float)dim / 1000.0f;
}
// A reach every line meets: for launches whose step counts are observed
// (stored per pixel, or statistics of traceMap's steps), where no ray may
// end before traceMap does.
__host__ __device__ inline void reach_everywhere(float* lo, float* hi) {
  for (int i = 0; i < 3; i++) {
    lo[i] = -1.0e30f;
    hi[i] = 1.0e30f;
  }
}
// The slab test of the line against [lo, hi] (inv = 1 / d after the zero
// substitution, so never infinite).
__device__ __forceinline__ bool line_meets_box(const float* lo, const float* hi, float ex,
                                               float ey, float ez, const float* inv) {
  const float e[3] = {ex, ey, ez};
  float tn = 0.0f, tf = 3.0e38f;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const float a = (lo[i] - e[i]) * inv[i], b = (hi[i] - e[i]) * inv[i];
    tn = fmaxf(tn, fminf(a, b));
    tf = fminf(tf, fmaxf(a, b));
  }
  return tn <= tf;
}
__device__ __forceinline__ bool line_meets_reach(const DenseWorld& w, float ex, float ey,
                                                 float ez, const RayConsts& k) {
  return line_meets_box(w.reach_lo, w.reach_hi, ex, ey, ez, k.inv);
}

// How many of traceMap's steps from e (voxel units) along k.d, whose line
// meets the reach box, come before the walk can probe a nonempty voxel: the
// blocks the line crosses before it enters the reach box, less a slack.
// Why the lookups of the first blind_steps steps read empty: after k steps
// the walk has crossed k block boundaries, c_i of them on axis i, and its
// position lies within the drift (< 1.03 voxel, see above) of a point
// L(s) of the line; the boundaries the line crosses up to s, n_i(s), differ
// from c_i by at most 4 (2 for the drift, 1 for a within that reached 8, 1
// for the binary32 floor below), so k <= n(t_enter) - 13 gives n(s) <
// n(t_enter), s < t_enter, L(s) outside the reach box, and the probe
// outside the box of the nonempty voxels (the reach box's argument).
__device__ __forceinline__ int blind_steps_box(const float* lo, const float* hi, float ex,
                                               float ey, float ez, const float* d,
                                               const float* inv) {
  const float e[3] = {ex, ey, ez};
  float tn = 0.0f;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const float a = (lo[i] - e[i]) * inv[i], b = (hi[i] - e[i]) * inv[i];
    tn = fmaxf(tn, fminf(a, b));
  }
  int n = 0;
#pragma unroll
  for (int i = 0; i < 3; i++) n += abs((int)floorf(e[i] + d[i] * tn) - (int)floorf(e[i]));
  return n - 13;
}
__device__ __forceinline__ int blind_steps(const DenseWorld& w, float ex, float ey, float ez,
                                           const RayConsts& k) {
  return blind_steps_box(w.reach_lo, w.reach_hi, ex, ey, ez, k.d, k.inv);
}

// Set-up (map.glsl:85-104) plus iteration 0 (stepSize 0).  Returns true when
// the ray already terminated (hit or miss) in iteration 0; otherwise the ray
// is at the block level, ready for the DDA step of iteration 0.
// dense_begin_k: the same with the direction's constants made beforehand.
template <bool kStats, class L>
__device__ __forceinline__ bool dense_begin_k(DenseRay& r, L& lk, const DenseWorld& w, float ox,
                                              float oy, float oz, const RayConsts& k,
                                              int max_steps, DenseHit& h, uint32_t& l1f,
                                              uint32_t& l0f);

template <bool kStats, class L>
__device__ __forceinline__ bool dense_begin(DenseRay& r, L& lk, const DenseWorld& w, float ox,
                                            float oy, float oz, float dx, float dy, float dz,
                                            int max_steps, DenseHit& h, uint32_t& l1f,
                                            uint32_t& l0f) {
  return dense_begin_k<kStats>(r, lk, w, ox, oy, oz, make_ray_consts(dx, dy, dz, w.mx, w.my, w.mz),
                               max_steps, h, l1f, l0f);
}

template <bool kStats, class L>
__device__ __forceinline__ bool dense_begin_k(DenseRay& r, L& lk, const DenseWorld& w, float ox,
                                              float oy, float oz, const RayConsts& k,
                                              int max_steps, DenseHit& h, uint32_t& l1f,
                                              uint32_t& l0f) {
  dense_ray_from(r, k);
  r.steps = 0;
  r.max_steps = max_steps;
  r.blind = 0;
  lk.reset();

  float s8x = ox * 8.0f, s8y = oy * 8.0f, s8z = oz * 8.0f;
  int gx = f2i_sat(s8x), gy = f2i_sat(s8y), gz = f2i_sat(s8z);
  float wx = s8x - (float)gx, wy = s8y - (float)gy, wz = s8z - (float)gz;

  h.hit = false;
  h.steps = 0;
  const int B = (int)(8u * w.dim);
  if (max_steps <= 0) return true;
  if (gx >= B || gy >= B || gz >= B || gx < 0 || gy < 0 || gz < 0) return true;
  // iteration 0, stepSize 0: pos = gridsCoords + int(within)
  int qx = gx + (int)wx, qy = gy + (int)wy, qz = gz + (int)wz;
  int bx = qx >> 3, by = qy >> 3, bz = qz >> 3;
  uint32_t v = 0;
  uint32_t code = 0;
  if (in_dim(w, bx, by, bz)) {
    code = morton3((uint32_t)bx, (uint32_t)by, (uint32_t)bz);
    v = lk.template probe<kStats>(w, code, l1f, l0f);
  }
  if (v != 0u) {
    h.hit = true;
    h.face = 2 - r.px;  // minIdx == 0 on the first iteration
    h.bx = bx;
    h.by = by;
    h.bz = bz;
    h.code = code;
    h.v = v;
    h.sub = (uint32_t)(qx & 7) | ((uint32_t)(qy & 7) << 3) | ((uint32_t)(qz & 7) << 6);
    h.hx = (float)gx + wx;
    h.hy = (float)gy + wy;
    h.hz = (float)gz + wz;
    h.steps = 1;
    return true;
  }
  // empty block: switch to the block level (map.glsl:140-144)
  int lx = gx & 7, ly = gy & 7, lz = gz & 7;
  r.wx = wx + (float)lx;
  r.wy = wy + (float)ly;
  r.wz = wz + (float)lz;
  r.c = morton3((uint32_t)(gx - lx) >> 3, (uint32_t)(gy - ly) >> 3, (uint32_t)(gz - lz) >> 3) ^
        r.flip;
  return false;
}

// Real-space increment of one axis of a Morton code (mask M); sets `out`
// when the coordinate was already dim - 1.
__device__ __forceinline__ uint32_t morton_inc(uint32_t a, uint32_t M, bool& out) {
  out |= (a & M) == M;
  return (((a | ~M) + 1u) & M) | (a & ~M);
}

// The block-level loop of traceMap (map.glsl:106-165 at stepSize 3) after
// iteration 0.  A step is the DDA arithmetic (map.glsl:157-162), one dilated
// increment of the crossed axis in the flipped Morton code and one probe:
//   M = mask of the crossed axis,  c' = ((c & M) - M) & M | (c & ~M)
// Leaving the grid is exactly the wrap of that increment, (c & M) == M,
// which is traceMap's bounds test.  The probed block is pos >> 3 =
// G + (int(within) >> 3): within reaches 8 on a positive axis the DDA did not
// cross when two crossing times tie exactly (frequent for rays started on
// lattice points, e.g. every shadow ray), so that correction is a short
// branch inside the loop rather than an exit from it.
// A wave-uniform value held in a VGPR for the length of a loop.  The step's
// mask select (two selects between the three axis masks) cannot read two
// SGPRs in one instruction, and the compiler re-creates VGPR copies of the
// masks with a v_mov at every step rather than keep three registers; an
// opaque copy cannot be re-created, so it is made once and stays.
__device__ __forceinline__ uint32_t in_vgpr(uint32_t s) {
  uint32_t v;
  asm("v_mov_b32 %0, %1" : "=v"(v) : "s"(s));
  return v;
}

// One block-level DDA step of traceMap (map.glsl:157-162) and the cell it
// lands in; the state after the step is what the next lookup probes.
struct DenseCell {
  float wx, wy, wz;  // withinGridCoords
  uint32_t c;        // flipped Morton code of gridsCoords >> 3
  uint32_t M;        // mask of the axis crossed by the step (minIdx)
  uint32_t a;        // Morton code of the probed block pos >> 3, or
                     // kOutside when the within >= 8 correction left the grid
  bool wrapped;      // the step left the grid (traceMap's bounds test)
};

// Beyond every grid (codes use at most 30 bits): a bounds-checked buffer load
// of it returns 0, i.e. "empty", as map_getChunkFlags does outside the map.
constexpr uint32_t kOutside = 0xFFFFFFFFu;

// Real-space increment of one axis of a Morton code; kOutside when the
// coordinate was already dim - 1 (kOutside stays kOutside).
__device__ __forceinline__ uint32_t morton_inc_or_out(uint32_t a, uint32_t M) {
  return (a & M) == M ? kOutside : ((((a | ~M) + 1u) & M) | (a & ~M));
}

// The step's ray constants are passed as scalars: the mask select below must
// stay a select of values (a struct here was turned into a dynamically
// indexed stack object, one scratch load per step).
__device__ __forceinline__ DenseCell dense_step(float Px, float Py, float Pz, float Ax, float Ay,
                                                float Az, float dx, float dy, float dz, float ix,
                                                float iy, float iz, uint32_t mx, uint32_t my,
                                                uint32_t mz, uint32_t flip, const DenseCell& s) {
  DenseCell n;
  const float tx = (Px - s.wx) * ix;
  const float ty = (Py - s.wy) * iy;
  const float tz = (Pz - s.wz) * iz;
  // minIdx = tx < ty ? (tx < tz ? 0 : 2) : (ty < tz ? 1 : 2): m1 = yz & !m0
  // is the same rule.  t is never NaN (d != 0 after the 0.001 substitution,
  // within is finite), so t[minIdx] is the smallest t; min3 can differ from
  // it only in the sign of a zero, which no later operation can see
  // (w + d * (+-0) = w, P - w, int(w) and hit_pos are unchanged).
  const bool xy = tx < ty, xz = tx < tz, yz = ty < tz;
  const bool m0 = xy & xz;
  const bool m1 = yz & !m0;
  const float tm = fminf(fminf(tx, ty), tz);
  const float nwx = s.wx + dx * tm;
  const float nwy = s.wy + dy * tm;
  const float nwz = s.wz + dz * tm;
  n.wx = m0 ? Ax : nwx;
  n.wy = m1 ? Ay : nwy;
  n.wz = (m0 | m1) ? nwz : Az;
  n.M = m0 ? mx : (m1 ? my : mz);
  const uint32_t cm = s.c & n.M;
  n.wrapped = cm == n.M;
  n.c = ((cm - n.M) & n.M) | (s.c & ~n.M);
  n.a = n.c ^ flip;
  if (fmaxf(fmaxf(n.wx, n.wy), n.wz) >= 8.0f) {  // pos >> 3 = G + (int(within) >> 3)
    if (n.wx >= 8.0f) n.a = morton_inc_or_out(n.a, mx);
    if (n.wy >= 8.0f) n.a = morton_inc_or_out(n.a, my);
    if (n.wz >= 8.0f) n.a = morton_inc_or_out(n.a, mz);
  }
  return n;
}

// Code c one block further on the axis of mask M (wrapping).
__device__ __forceinline__ uint32_t morton_step(uint32_t c, uint32_t M) {
  const uint32_t t = __builtin_amdgcn_bitop3_b32(c, M, 0u, 0xF3u) + 1u;  // (c | ~M) + 1
  return __builtin_amdgcn_bitop3_b32(t, M, c, 0xE2u);                    // (t & M) | (c & ~M)
}

// Whether every crossing time from this state on is an ordered number: the
// reciprocals are finite, and within starts finite (it stays within a few
// units of [0, 8]).
__device__ __forceinline__ bool dense_ordered(float ix, float iy, float iz, float wx, float wy,
                                              float wz) {
  return fmaxf(fmaxf(fabsf(ix), fabsf(iy)), fabsf(iz)) < 1.0e30f &&
         fabsf(wx) + fabsf(wy) + fabsf(wz) < 1.0e6f;
}

// minIdx of a step whose smallest crossing time is tm (dense_ordered rays).
// The masks are formed as lane masks: on booleans the compiler replaces the
// negated one by a third compare.
struct StepAxis {
  bool y, z, yz;  // the step crosses y; z; y or z
};
__device__ __forceinline__ StepAxis step_axis(float ty, float tz, float tm) {
  const uint64_t ey = __builtin_amdgcn_ballot_w64(ty == tm);
  const uint64_t ez = __builtin_amdgcn_ballot_w64(tz == tm);
  StepAxis a;
  a.y = __builtin_amdgcn_inverse_ballot_w64(ey & ~ez);
  a.z = __builtin_amdgcn_inverse_ballot_w64(ez);
  a.yz = __builtin_amdgcn_inverse_ballot_w64(ey | ez);
  return a;
}

// The same step without its lookup: the state alone.  Returns the crossing
// time the step took, which is <= 0 when within had reached 8 on a positive
// axis (t = (8 - within) / d there, and the smallest t is at most that one):
// the state before the step then probes the block after its own.
//
// For rays without NaN crossing times (dense_ordered): minIdx is then z when
// tz equals the smallest t, else y when ty does, else x -- traceMap's nested
// compares, whose ties go to the later axis -- which takes two compares and
// two mask operations a step (step_axis) instead of three and four.  The code of axis k
// is incremented with the other axes' bits set, so that the carry runs
// through them: (c | ~M) + 1, merged back under M.  A wave that runs alone on
// its SIMD issues one instruction every four cycles, scalar or vector, and the
// frames end with such waves, so the instructions of a step are their time: an
// iteration of 6 steps takes 193 instructions against 216 with the nested
// compares and (((c & M) - M) & M) | (c & ~M), and the kernels' spills are
// gone.  Six views of the 512^3 world at 1080p 290 -> 272 us, the engine's map
// with long caps 248 -> 231, its own frame 139 -> 134, a batch of 64 views
// 2260 -> 2170, 16 Lambert views of a 256^3 height field and their backward
// 1357 -> 1298.
__device__ __forceinline__ float dense_advance(float Px, float Py, float Pz, float Ax, float Ay,
                                               float Az, float dx, float dy, float dz, float ix,
                                               float iy, float iz, uint32_t mx, uint32_t my,
                                               uint32_t mz, float& wx, float& wy, float& wz,
                                               uint32_t& c) {
  const float tx = (Px - wx) * ix;
  const float ty = (Py - wy) * iy;
  const float tz = (Pz - wz) * iz;
  const float tm = fminf(fminf(tx, ty), tz);
  const StepAxis ax = step_axis(ty, tz, tm);
  const float nwx = wx + dx * tm;
  const float nwy = wy + dy * tm;
  const float nwz = wz + dz * tm;
  wx = ax.yz ? nwx : Ax;
  wy = ax.y ? Ay : nwy;
  wz = ax.z ? Az : nwz;
  c = morton_step(c, ax.z ? mz : (ax.y ? my : mx));
  return tm;
}

// Whether some axis left the grid between the flipped codes c0 and c, at
// most dim / 2 steps apart: a coordinate only grows, by one per crossing, so
// it wrapped exactly when its top bit went from 1 to 0.
__device__ __forceinline__ bool dense_left_grid(uint32_t c0, uint32_t c, uint32_t mx, uint32_t my,
                                                uint32_t mz) {
  const uint32_t all = mx | my | mz;
  return (c0 & ~c & (all & ~(all >> 3))) != 0u;
}

// The flat lookup's loop, software-pipelined: the byte of step k+1's block is
// requested before step k's byte is tested, so each gather's latency overlaps
// one step of DDA arithmetic; the run-ahead result is discarded when the ray
// stops at step k.  The bytes are read with bounds-checked buffer loads
// (base and size in a scalar resource, a 32-bit offset per lane): a wrapped
// code is still a code of the grid, and kOutside reads as 0.  Same steps,
// same stopping rule and same final state as the plain loop.
// Block-level steps from s0 (whose own lookup was empty, `steps0` steps
// done) over the byte array behind `bytes` until a step lands on a nonzero
// byte, leaves the grid or reaches max_steps.  Returns the stopping state
// field by field (a struct select would go through memory).
__device__ __forceinline__ void dense_loop_prefetch(
    float Px, float Py, float Pz, float Ax, float Ay, float Az, float dx, float dy, float dz,
    float ix, float iy, float iz, uint32_t mx, uint32_t my, uint32_t mz, uint32_t flip,
    const DenseCell& s0, int steps0, int max_steps, __amdgpu_buffer_rsrc_t bytes, float& fwx,
    float& fwy, float& fwz, uint32_t& fc, uint32_t& fM, uint32_t& fa, uint32_t& fv, int& sF,
    bool& wrappedF) {
#define VT_STEP(s) dense_step(Px, Py, Pz, Ax, Ay, Az, dx, dy, dz, ix, iy, iz, mx, my, mz, flip, s)
#define VT_LOAD(a) (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(bytes, (int)(a), 0, 0)
  DenseCell A = VT_STEP(s0), B;
  int sA = steps0 + 1, sB = 0;
  uint32_t vA = VT_LOAD(A.a), vB = 0u;
  bool useB;
  for (;;) {
    B = VT_STEP(A);
    vB = VT_LOAD(B.a);
    if (A.wrapped | (vA != 0u) | (sA >= max_steps)) {
      useB = false;
      break;
    }
    sB = sA + 1;
    A = VT_STEP(B);
    vA = VT_LOAD(A.a);
    if (B.wrapped | (vB != 0u) | (sB >= max_steps)) {
      useB = true;
      break;
    }
    sA = sB + 1;
  }
#undef VT_STEP
#undef VT_LOAD
  sF = useB ? sB : sA;
  wrappedF = useB ? B.wrapped : A.wrapped;
  fwx = useB ? B.wx : A.wx;
  fwy = useB ? B.wy : A.wy;
  fwz = useB ? B.wz : A.wz;
  fc = useB ? B.c : A.c;
  fM = useB ? B.M : A.M;
  fa = useB ? B.a : A.a;
  fv = useB ? vB : vA;
}

// How an empty-space run ended.
enum SkipStatus : int {
  kSkipLimit = 0,    // reached its step limit; every lookup so far empty
  kSkipBlocked = 1,  // an iteration met a nonzero byte or left the grid
  kSkipFree = 2,     // nothing ahead of the ray on all three axes: a miss
  kSkipOpen = 3,     // the wave's rays stand clear of everything: clear_advance
  kSkipPause = 4,    // most of the wave's rays wait for the others
};

// ---- ClearMap: the clearance map (built by k_maps_first, k_clear_planes and k_clear_cubes) ----
// Cells of 8^3 blocks, R = dim / 8 per axis.  A cell is near when the cell
// widened by 2 blocks a side holds a nonempty block.  For each direction
// octant (bit k = travelling negatively on axis k) the byte of a cell is the
// side m, in cells, of the largest cube of cells none of them near that has
// this cell as its corner and extends in the octant's travel direction (parts
// outside the grid count as clear): 0 = the cell is near; 255 = no near cell
// at or ahead of this one on all three axes.  Each octant's cells are
// numbered with its negative axes complemented, as the traversal's codes are,
// twice: in Morton order (8 planes of R^3 bytes, byte c >> 9 for a flipped
// block code c) and, after those, x + R (y + R z).
//
// What it is exact for.  A step of traceMap's block-level recurrence moves
// the position p = G + within / 8 along the direction by the crossing time tm
// (p += d tm / 8) up to binary32 rounding (< 1e-6 block), and a crossing of
// a negative axis re-anchors within at A = 8 x 0.999 instead of 8, 1 - A / 8 =
// 0.001 block ahead.  After crossing times summing to T the position is
// therefore p0 + d T / 8 to within 0.001 block per negative crossing (at most
// dim of them: 1.03 blocks) and the rounding of the sum (< 0.2 block over
// 3 x 1024 steps), and the block a lookup probes contains the position or
// touches it.  So while the line p0 + d T / 8 runs through cells that are not
// near, every probe is at least 2 - 1.3 blocks from the nearest nonempty
// block: the lookups read empty and need not be made.  Where the line leaves
// the grid through such cells, or the cell's byte is 255, the ray is a miss.
//
// clear_walk follows the line from cube to cube; the walk itself is then
// taken step by step (its float state must be traceMap's), without lookups
// and without tracking the block, until the sum of its crossing times says
// that the line comes near something: 19 VALU a step against 25 with its
// lookup, and no memory latency.  The block at the end follows from T: axis
// i crossed n_i = round(((within0 - within) + d T) / 8) boundaries (negative
// axes: / -A).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t clear_rsrc(const uint8_t* map, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)map, (short)0, (int)bytes, 0x00020000);
}

// Byte offset of the octant plane of a ray whose complemented (negative)
// axes are `flip`.
__device__ __forceinline__ uint32_t clear_octant_offset(uint32_t flip, uint32_t mx, uint32_t my,
                                                        uint32_t mz, uint32_t oct_bytes) {
  const uint32_t o = ((flip & mx) ? 1u : 0u) | ((flip & my) ? 2u : 0u) | ((flip & mz) ? 4u : 0u);
  return o * oct_bytes;
}

// The map's byte for the cell of flipped block code c.
__device__ __forceinline__ uint32_t clear_byte(__amdgpu_buffer_rsrc_t cm, uint32_t cofs,
                                               uint32_t c) {
  return (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(cm, (int)(cofs + (c >> 9)), 0, 0);
}

// Directions the line argument holds for: every component and reciprocal
// within 1e-30 .. 1e30 (no product of the walk overflows or turns NaN).
__device__ __forceinline__ bool clear_usable(float ix, float iy, float iz) {
  const float a = fabsf(ix), b = fabsf(iy), c = fabsf(iz);
  return fmaxf(fmaxf(a, b), c) < 1.0e30f && fminf(fminf(a, b), c) > 1.0e-30f;
}

// From the flipped cell (cx, cy, cz) of the point q (flipped, cell units),
// follows the line q + |d| T / 64 until it comes to a near cell: true, T =
// where (0: at once).  False: nothing near ahead.  Each turn takes the
// largest clear cube from the cell and moves on to the cell behind its far
// face: at least one axis moves on and none back, so the walk ends within 3 R
// turns.  Rounding can put the line in a cell next to its own, within 1e-3
// block of it: the 2-block widening has room for that.  Cell numbers are kept
// as floats (exact), the index by two fused multiply-adds: a turn is about
// 45 VALU and one load.
__device__ __forceinline__ bool clear_walk(__amdgpu_buffer_rsrc_t cm, uint32_t lofs, float R,
                                           float cx, float cy, float cz, float qx, float qy,
                                           float qz, float ax, float ay, float az, float bx,
                                           float by, float bz, float& T) {
  // a = |d| / 64, b = 64 / |d|
  T = 0.0f;
  for (;;) {
    const uint32_t i = (uint32_t)fmaf(R, fmaf(R, cz, cy), cx);
    const uint32_t m =
        (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(cm, (int)(lofs + i), 0, 0);
    if (m == 0u) return true;
    if (m == 255u) return false;
    const float side = (float)m;
    const float fx = cx + side, fy = cy + side, fz = cz + side;  // behind the far faces
    const float tx = (fx - qx) * bx, ty = (fy - qy) * by, tz = (fz - qz) * bz;
    const float t = fminf(fminf(tx, ty), tz);
    T = fmaxf(T, t);
    cx = tx > t ? fmaxf(floorf(qx + ax * T), cx) : fx;
    cy = ty > t ? fmaxf(floorf(qy + ay * T), cy) : fy;
    cz = tz > t ? fmaxf(floorf(qz + az * T), cz) : fz;
    if (!(fmaxf(fmaxf(cx, cy), cz) < R)) return false;
  }
}

// Takes the ray from state s as far as the clearance map shows its lookups
// to read empty (steps advanced by as many).  False: the ray is a miss --
// nothing near ahead, or the walk left the grid or reached max_steps
// meanwhile.  After crossing times summing to T the walk has crossed at least
// (|dx| + |dy| + |dz|) T / 8 - 3 boundaries, one a step (each axis at least its
// line's, the drift being ahead), so a line that comes near something only
// after max_steps + 5 of them does so past the cap.
template <int K>
__device__ __forceinline__ bool clear_advance(float Px, float Py, float Pz, float Ax, float Ay,
                                              float Az, float dx, float dy, float dz, float ix,
                                              float iy, float iz, uint32_t flip, uint32_t mx,
                                              uint32_t my, uint32_t mz, uint32_t dim,
                                              DenseCell& s, int& steps, int max_steps,
                                              __amdgpu_buffer_rsrc_t cm, uint32_t cofs,
                                              uint32_t oct_bytes) {
  const bool nx = (flip & mx) != 0u, ny = (flip & my) != 0u, nz = (flip & mz) != 0u;
  uint32_t hx = compact1by2(s.c), hy = compact1by2(s.c >> 1), hz = compact1by2(s.c >> 2);
  float T;
  if (!clear_walk(cm, 8u * oct_bytes + cofs, (float)(dim >> 3), (float)(hx >> 3),
                  (float)(hy >> 3), (float)(hz >> 3),
                  ((float)hx + (nx ? 8.0f - s.wx : s.wx) * 0.125f) * 0.125f,
                  ((float)hy + (ny ? 8.0f - s.wy : s.wy) * 0.125f) * 0.125f,
                  ((float)hz + (nz ? 8.0f - s.wz : s.wz) * 0.125f) * 0.125f,
                  fabsf(dx) * 0.015625f, fabsf(dy) * 0.015625f, fabsf(dz) * 0.015625f,
                  fabsf(ix) * 64.0f, fabsf(iy) * 64.0f, fabsf(iz) * 64.0f, T))
    return false;
  if ((fabsf(dx) + fabsf(dy) + fabsf(dz)) * T >= 8.0f * (float)(max_steps - steps + 5))
    return false;  // the cap comes first
  // K steps take at most K crossing times of the fastest axis
  const float lim = T - (8.0f * K) * fminf(fminf(fabsf(ix), fabsf(iy)), fabsf(iz));
  // The wave's rays go on together while all of them can (a wave-uniform
  // loop): a ray that could go further alone would have the others wait for
  // it now and wait for them later.
  if (__ballot(!(lim >= 0.0f)) != 0ull) return true;
  float wx = s.wx, wy = s.wy, wz = s.wz, t = 0.0f;
  do {
#pragma unroll
    for (int i = 0; i < K; ++i) {
      // dense_advance without the block (clear_usable directions are
      // dense_ordered)
      const float tx = (Px - wx) * ix;
      const float ty = (Py - wy) * iy;
      const float tz = (Pz - wz) * iz;
      const float tm = fminf(fminf(tx, ty), tz);
      const StepAxis ax = step_axis(ty, tz, tm);
      const float nwx = wx + dx * tm;
      const float nwy = wy + dy * tm;
      const float nwz = wz + dz * tm;
      wx = ax.yz ? nwx : Ax;
      wy = ax.y ? Ay : nwy;
      wz = ax.z ? Az : nwz;
      t += tm;
    }
  } while (__ballot(!(t <= lim)) == 0ull);
  const float kp = 0.125f, kn = -1.0f / (8.0f * 0.999f);
  const uint32_t cx = (uint32_t)(int)rintf(((s.wx - wx) + dx * t) * (nx ? kn : kp));
  const uint32_t cy = (uint32_t)(int)rintf(((s.wy - wy) + dy * t) * (ny ? kn : kp));
  const uint32_t cz = (uint32_t)(int)rintf(((s.wz - wz) + dz * t) * (nz ? kn : kp));
  hx += cx;
  hy += cy;
  hz += cz;
  steps += (int)(cx + cy + cz);
  if ((hx >= dim) | (hy >= dim) | (hz >= dim)) return false;  // left the grid, all empty
  s.wx = wx;
  s.wy = wy;
  s.wz = wz;
  s.c = morton3(hx, hy, hz);
  return true;
}

// Steps K at a time from s while steps + K <= lim without their lookups:
// the caller guarantees that they all read empty (blind_steps).  Stops
// before an iteration that leaves the grid; the state is traceMap's after
// `steps` steps, for the empty-space phase to continue from.
template <int K>
__device__ __forceinline__ void dense_skip_blind(float Px, float Py, float Pz, float Ax,
                                                 float Ay, float Az, float dx, float dy, float dz,
                                                 float ix, float iy, float iz, uint32_t mx,
                                                 uint32_t my, uint32_t mz, DenseCell& s,
                                                 int& steps, int lim) {
  float bx = s.wx, by = s.wy, bz = s.wz;
  uint32_t bc = s.c;
  int sb = steps;
  while (sb + K <= lim) {
    float wx = bx, wy = by, wz = bz;
    uint32_t c = bc;
#pragma unroll
    for (int i = 0; i < K; ++i)
      dense_advance(Px, Py, Pz, Ax, Ay, Az, dx, dy, dz, ix, iy, iz, mx, my, mz, wx, wy, wz, c);
    if (dense_left_grid(bc, c, mx, my, mz)) break;
    bx = wx;
    by = wy;
    bz = wz;
    bc = c;
    sb += K;
  }
  s.wx = bx;
  s.wy = by;
  s.wz = bz;
  s.c = bc;
  steps = sb;
}

// Empty-space phase of the flat loop.  An iteration takes K block-level steps
// from `s` (whose own lookup was empty, `steps` steps done) and requests all K
// bytes without testing any of them in between; only when all K are zero and
// no step left the grid does the state advance by K steps.  Otherwise `s` and
// `steps` are left at the start of that iteration and the exact loop
// (dense_loop_prefetch) replays it to the first stopping step.  The state
// after K empty, in-grid steps is exactly the exact loop's state after those
// steps, so the result is unchanged.  What this buys: one divergent exit per
// K steps instead of one per step, and with it none of the per-step copies of
// the exit state that a divergent exit costs.  An iteration only starts when
// steps + K < limit (limit <= max_steps), so the step cap falls inside the
// replay.  With kClear each iteration also requests the clearance map's byte
// of its start block (octant plane at `cofs` of `cm`): 255 ends the run with
// kSkipFree, the ray can hit nothing more; when the cells of all the wave's
// rays in the loop have clear neighbours ahead (>= 2) they leave together
// with kSkipOpen for clear_advance (one ray at a time would have the wave
// alternate between the loops).  With kPause the last quarter of the `entered`
// rays that began together leave with kSkipPause, to take the run up again
// later.  Returns kSkipBlocked when it stopped at an
// iteration that met a nonzero byte or left the grid, kSkipLimit at the
// limit; either way `s` is a state the exact loop (or another call)
// continues from.
//
// The lookup of a state with within >= 8 probes the next block.  Instead of
// a branch at every step the iteration is taken without that correction and
// taken again with it when a crossing time says that such a state was among
// them (4% of the rays of a terrain frame meet one): 29 VALU + 8 SALU a step
// against 39 + 19, and 25 + 3 with step_axis and morton_step.
template <int K, bool kClear, bool kPause = false>
__device__ __forceinline__ int dense_skip_empty(float Px, float Py, float Pz, float Ax, float Ay,
                                                float Az, float dx, float dy, float dz, float ix,
                                                float iy, float iz, uint32_t mx, uint32_t my,
                                                uint32_t mz, uint32_t flip, DenseCell& s,
                                                int& steps, int limit,
                                                __amdgpu_buffer_rsrc_t bytes,
                                                __amdgpu_buffer_rsrc_t cm, uint32_t cofs,
                                                bool usable, int entered = 0) {
  float bx = s.wx, by = s.wy, bz = s.wz;
  uint32_t bc = s.c;
  int sb = steps;
  int status = kSkipLimit;
  while (sb + K < limit) {
    const uint32_t m = kClear ? clear_byte(cm, cofs, bc) : 0u;
    float wx = bx, wy = by, wz = bz;
    uint32_t c = bc, any = 0u;
    float mn = 1.0f;  // smallest crossing time of the steps from S_1 .. S_K-1
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const float tm = dense_advance(Px, Py, Pz, Ax, Ay, Az, dx, dy, dz, ix, iy, iz, mx, my, mz,
                                     wx, wy, wz, c);
      if (i > 0) mn = fminf(mn, tm);
      any |= (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(bytes, (int)(c ^ flip), 0, 0);
    }
    if ((mn <= 0.0f) | (fmaxf(fmaxf(wx, wy), wz) >= 8.0f)) {
      // a state with within >= 8 (an exact tie): the same steps again, with
      // the corrected lookups
      DenseCell n;
      n.wx = bx;
      n.wy = by;
      n.wz = bz;
      n.c = bc;
      any = 0u;
#pragma unroll 1
      for (int i = 0; i < K; ++i) {
        n = dense_step(Px, Py, Pz, Ax, Ay, Az, dx, dy, dz, ix, iy, iz, mx, my, mz, flip, n);
        any |= (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(bytes, (int)n.a, 0, 0);
      }
    }
    if (kClear && m == 255u) {
      status = kSkipFree;
      break;
    }
    if (dense_left_grid(bc, c, mx, my, mz) | (any != 0u)) {
      status = kSkipBlocked;
      break;
    }
    bx = wx;
    by = wy;
    bz = wz;
    bc = c;
    sb += K;
    if (kClear && __ballot(!((m >= 2u) & usable)) == 0ull) {
      status = kSkipOpen;
      break;
    }
    if (kPause && 4 * __popcll(__ballot(true)) < entered) {
      status = kSkipPause;
      break;
    }
  }
  s.wx = bx;
  s.wy = by;
  s.wz = bz;
  s.c = bc;
  steps = sb;
  return status;
}

// The empty-space phase for rays whose direction is positive on every axis
// (after the zero substitution) -- the shadow rays of a sun with no negative
// component.  Then rayPositivity is 1 everywhere: the crossing position is
// 8, the re-anchored within is 0 and the Morton code is the address (no
// complemented axes).  Same contract as dense_skip_empty; what differs is how
// the lookup of a state S_i is made exact without a branch:
//   pos >> 3 = G + (int(within) >> 3) moves the probed block one step along
//   each axis k with within_k >= 8, and with positivity 1 that is exactly
//   t_k = (8 - within_k) / d_k <= 0 for the next step.  When one axis has
//   t <= 0 it is the smallest crossing time, so the next step crosses that
//   axis and lands in the very block the corrected lookup probes: the lookup
//   of S_i is the block of S_{i+1}.  Two or more axes at t <= 0 (the median
//   crossing time <= 0) stop the iteration, and the exact loop replays it.
// The lookup of an iteration's last state has no next step inside the
// iteration and takes the general branch (dense_step's).  Shadow rays start
// on lattice points, so this correction is frequent for them: as a branch it
// ran in about half of the wave-steps.
// The clearance map's part is dense_skip_empty's, on octant 0's plane.
template <int K, bool kClear, bool kPause = false>
__device__ __forceinline__ int dense_skip_positive(float dx, float dy, float dz, float ix,
                                                   float iy, float iz, uint32_t mx, uint32_t my,
                                                   uint32_t mz, DenseCell& s, int& steps,
                                                   int limit, __amdgpu_buffer_rsrc_t bytes,
                                                   __amdgpu_buffer_rsrc_t cm, bool usable,
                                                   int entered = 0) {
  float bx = s.wx, by = s.wy, bz = s.wz;
  uint32_t bc = s.c;
  int sb = steps;
  int status = kSkipLimit;
  while (sb + K < limit) {
    const uint32_t m = kClear ? clear_byte(cm, 0u, bc) : 0u;
    float wx = bx, wy = by, wz = bz;
    uint32_t c = bc;
    uint32_t any = 0u;
    float med = 1.0f;  // smallest median crossing time of the iteration
#pragma unroll
    for (int i = 0; i < K; ++i) {
      // the step from S_i (S_0 is the iteration's start, already probed)
      const float tx = (8.0f - wx) * ix;
      const float ty = (8.0f - wy) * iy;
      const float tz = (8.0f - wz) * iz;
      const float tm = fminf(fminf(tx, ty), tz);
      const StepAxis ax = step_axis(ty, tz, tm);
      const float nwx = wx + dx * tm;
      const float nwy = wy + dy * tm;
      const float nwz = wz + dz * tm;
      wx = ax.yz ? nwx : 0.0f;
      wy = ax.y ? 0.0f : nwy;
      wz = ax.z ? 0.0f : nwz;
      const uint32_t cn = morton_step(c, ax.z ? mz : (ax.y ? my : mx));
      if (i > 0) {  // the lookup of S_i
        any |= (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(bytes, (int)(tm <= 0.0f ? cn : c), 0,
                                                             0);
        med = fminf(med, __builtin_amdgcn_fmed3f(tx, ty, tz));
      }
      c = cn;
    }
    const bool stop = (med <= 0.0f) | dense_left_grid(bc, c, mx, my, mz);
    {  // the lookup of S_K
      uint32_t a = c;
      if (fmaxf(fmaxf(wx, wy), wz) >= 8.0f) {
        if (wx >= 8.0f) a = morton_inc_or_out(a, mx);
        if (wy >= 8.0f) a = morton_inc_or_out(a, my);
        if (wz >= 8.0f) a = morton_inc_or_out(a, mz);
      }
      any |= (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(bytes, (int)a, 0, 0);
    }
    if (kClear && m == 255u) {
      status = kSkipFree;
      break;
    }
    if (stop | (any != 0u)) {
      status = kSkipBlocked;
      break;
    }
    bx = wx;
    by = wy;
    bz = wz;
    bc = c;
    sb += K;
    if (kClear && __ballot(!((m >= 2u) & usable)) == 0ull) {
      status = kSkipOpen;
      break;
    }
    if (kPause && 4 * __popcll(__ballot(true)) < entered) {
      status = kSkipPause;
      break;
    }
  }
  s.wx = bx;
  s.wy = by;
  s.wz = bz;
  s.c = bc;
  steps = sb;
  return status;
}

// The two rules of an iteration for dense_skip_ahead: any direction
// (SkipGeneral, dense_skip_empty's) and directions positive on every axis
// (SkipPositive, dense_skip_positive's).
struct SkipState {
  float wx, wy, wz;
  uint32_t c;
};

template <int K>
struct SkipGeneral {
  float Px, Py, Pz, Ax, Ay, Az, dx, dy, dz, ix, iy, iz;
  uint32_t mx, my, mz, flip;
  __amdgpu_buffer_rsrc_t bytes;
  // The K steps from a: the state b after them; probe(i, address) for each.
  template <class P>
  __device__ __forceinline__ void run(const SkipState& a, SkipState& b, bool& tie,
                                      P probe) const {
    float wx = a.wx, wy = a.wy, wz = a.wz;
    uint32_t c = a.c;
    float mn = 1.0f;  // smallest crossing time of the steps from S_1 .. S_K-1
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const float tm = dense_advance(Px, Py, Pz, Ax, Ay, Az, dx, dy, dz, ix, iy, iz, mx, my, mz,
                                     wx, wy, wz, c);
      if (i > 0) mn = fminf(mn, tm);
      probe(i, c ^ flip);
    }
    tie = (mn <= 0.0f) | (fmaxf(fmaxf(wx, wy), wz) >= 8.0f);
    b.wx = wx;
    b.wy = wy;
    b.wz = wz;
    b.c = c;
  }
  // Whether the iteration from a to b ends the phase; any = its bytes or-ed.
  __device__ __forceinline__ bool stops(const SkipState& a, const SkipState& b, bool tie,
                                        uint32_t any) const {
    if (tie) {  // the same steps again, with the corrected lookups
      DenseCell n;
      n.wx = a.wx;
      n.wy = a.wy;
      n.wz = a.wz;
      n.c = a.c;
      any = 0u;
#pragma unroll 1
      for (int i = 0; i < K; ++i) {
        n = dense_step(Px, Py, Pz, Ax, Ay, Az, dx, dy, dz, ix, iy, iz, mx, my, mz, flip, n);
        any |= (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(bytes, (int)n.a, 0, 0);
      }
    }
    return dense_left_grid(a.c, b.c, mx, my, mz) | (any != 0u);
  }
};

template <int K>
struct SkipPositive {
  float dx, dy, dz, ix, iy, iz;
  uint32_t mx, my, mz;
  __amdgpu_buffer_rsrc_t bytes;
  template <class P>
  __device__ __forceinline__ void run(const SkipState& a, SkipState& b, bool& tie,
                                      P probe) const {
    float wx = a.wx, wy = a.wy, wz = a.wz;
    uint32_t c = a.c;
    float med = 1.0f;  // smallest median crossing time of the iteration
#pragma unroll
    for (int i = 0; i < K; ++i) {
      // the step from S_i (S_0 is the iteration's start, already probed)
      const float tx = (8.0f - wx) * ix;
      const float ty = (8.0f - wy) * iy;
      const float tz = (8.0f - wz) * iz;
      const float tm = fminf(fminf(tx, ty), tz);
      const StepAxis ax = step_axis(ty, tz, tm);
      const float nwx = wx + dx * tm;
      const float nwy = wy + dy * tm;
      const float nwz = wz + dz * tm;
      wx = ax.yz ? nwx : 0.0f;
      wy = ax.y ? 0.0f : nwy;
      wz = ax.z ? 0.0f : nwz;
      const uint32_t cn = morton_step(c, ax.z ? mz : (ax.y ? my : mx));
      if (i > 0) {  // the lookup of S_i
        probe(i - 1, tm <= 0.0f ? cn : c);
        med = fminf(med, __builtin_amdgcn_fmed3f(tx, ty, tz));
      }
      c = cn;
    }
    uint32_t q = c;
    if (fmaxf(fmaxf(wx, wy), wz) >= 8.0f) {  // the lookup of S_K
      if (wx >= 8.0f) q = morton_inc_or_out(q, mx);
      if (wy >= 8.0f) q = morton_inc_or_out(q, my);
      if (wz >= 8.0f) q = morton_inc_or_out(q, mz);
    }
    probe(K - 1, q);
    tie = med <= 0.0f;
    b.wx = wx;
    b.wy = wy;
    b.wz = wz;
    b.c = c;
  }
  __device__ __forceinline__ bool stops(const SkipState& a, const SkipState& b, bool tie,
                                        uint32_t any) const {
    return tie | dense_left_grid(a.c, b.c, mx, my, mz) | (any != 0u);
  }
};

// The empty-space phase without the clearance map, an iteration ahead: the
// steps of iteration i + 1 are taken while the bytes of iteration i are on
// their way, and thrown away when those end the phase.  Same contract as
// dense_skip_empty.  For launches whose waves are all resident at once
// (launch_dense_select): they last as long as their longest wave, which runs
// alone on its SIMD towards the end, and there the wait for an iteration's
// bytes cost as much as its steps.  16 frames of 128x128 of a 256^3 height
// field 1047 -> 851 us, of 512x512 with their backward 1257 -> 1162.  A full
// chip loses what is thrown away: the same world at 1080p 44.2 -> 47.2 us, a
// batch of 32 views 1060 -> 1140.
template <int K, class It>
__device__ __forceinline__ void dense_skip_ahead(const It& it, DenseCell& s, int& steps,
                                                 int limit) {
  int sb = steps;
  if (sb + K >= limit) return;
  SkipState x, y, z;
  x.wx = s.wx;
  x.wy = s.wy;
  x.wz = s.wz;
  x.c = s.c;
  uint32_t p[K], v[K];
  bool ty, tz;
  it.run(x, y, ty, [&](int i, uint32_t a) {
    v[i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(it.bytes, (int)a, 0, 0);
  });
  for (;;) {
    it.run(y, z, tz, [&](int i, uint32_t a) { p[i] = a; });
    uint32_t any = 0u;
#pragma unroll
    for (int i = 0; i < K; ++i) any |= v[i];
    // The next requests only after this iteration's bytes have arrived (the
    // asm orders them): on every path to the loop's head just these K are in
    // flight, into the registers the last K left, so nothing waits for them
    // before the `or` above.
#pragma unroll
    for (int i = 0; i < K; ++i) asm volatile("" : "+v"(any), "+v"(p[i]));
#pragma unroll
    for (int i = 0; i < K; ++i)
      v[i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(it.bytes, (int)p[i], 0, 0);
    if (it.stops(x, y, ty, any)) break;
    x = y;
    y = z;
    ty = tz;
    sb += K;
    if (sb + K >= limit) break;
  }
  s.wx = x.wx;
  s.wy = x.wy;
  s.wz = x.wz;
  s.c = x.c;
  steps = sb;
}

// The flat lookup's traversal from r's block-level state: the empty-space
// phase, then the exact loop to the ray's end.
// kShadow: the ray starts next to a nonempty voxel.  kPositive: the caller
// guarantees a direction positive on every axis (after the zero
// substitution), and the empty-space phase is dense_skip_positive.
template <class L, bool kPositive = false, bool kShadow = false>
__device__ __forceinline__ void dense_run_prefetch(DenseRay& r, L& lk, const DenseWorld& w,
                                                   DenseHit& h) {
  const uint32_t mx = in_vgpr(w.mx), my = in_vgpr(w.my), mz = in_vgpr(w.mz), flip = r.flip;
  const int max_steps = r.max_steps;
  // rays with unordered crossing times (a NaN or infinite direction or
  // origin) take the exact loop alone
  const bool ordered = dense_ordered(r.ix, r.iy, r.iz, r.wx, r.wy, r.wz);
  const int limit = ordered ? max_steps : 0;
  DenseCell s0;
  s0.wx = r.wx;
  s0.wy = r.wy;
  s0.wz = r.wz;
  s0.c = r.c;
  const __amdgpu_buffer_rsrc_t vox =
      __builtin_amdgcn_make_buffer_rsrc((void*)w.vox, (short)0, (int)w.nvox, 0x00020000);
  int steps0 = r.steps;
  int status;
  if constexpr (L::kClear) {
    // clear stretches without lookups and stretches near something with
    // them, in turn; a primary ray starts with the former, a shadow ray (it
    // starts at a nonempty voxel) with the latter
    const __amdgpu_buffer_rsrc_t cm = clear_rsrc(w.clear, w.clear_bytes);
    const uint32_t cofs =
        kPositive ? 0u : clear_octant_offset(flip, mx, my, mz, w.clear_oct_bytes);
    const bool usable = ordered && clear_usable(r.ix, r.iy, r.iz);
    bool open = !kShadow;
    int blind = 0;
    for (;;) {
      if (open & usable) {
        const int s1 = steps0;
        const bool on = clear_advance<kClearSteps>(
            r.Px, r.Py, r.Pz, r.Ax, r.Ay, r.Az, r.dx, r.dy, r.dz, r.ix, r.iy, r.iz, flip, mx, my,
            mz, w.dim, s0, steps0, max_steps, cm, cofs, w.clear_oct_bytes);
        blind += steps0 - s1;
        if (!on || steps0 >= max_steps) {
          status = kSkipFree;
          break;
        }
      }
      if constexpr (kPositive)
        status = dense_skip_positive<L::kSkip, true>(r.dx, r.dy, r.dz, r.ix, r.iy, r.iz, mx, my,
                                                     mz, s0, steps0, limit, vox, cm, usable);
      else
        status = dense_skip_empty<L::kSkip, true>(
            r.Px, r.Py, r.Pz, r.Ax, r.Ay, r.Az, r.dx, r.dy, r.dz, r.ix, r.iy, r.iz, mx, my, mz,
            flip, s0, steps0, limit, vox, cm, cofs, usable);
      if (status != kSkipOpen) break;
      open = true;
    }
    r.blind = blind;  // the steps taken without lookups
    if (status == kSkipFree) {  // a miss: no later lookup can be nonzero
      h.hit = false;
      h.steps = min(steps0, max_steps);
      return;
    }
  } else if constexpr (kPositive && L::kAhead) {
    const SkipPositive<L::kSkip> it = {r.dx, r.dy, r.dz, r.ix, r.iy, r.iz, mx, my, mz, vox};
    dense_skip_ahead<L::kSkip>(it, s0, steps0, limit);
  } else if constexpr (kPositive) {
    dense_skip_positive<L::kSkip, false>(r.dx, r.dy, r.dz, r.ix, r.iy, r.iz, mx, my, mz, s0,
                                         steps0, limit, vox, vox, false);
  } else {
    // the lookups that can only read empty first (primary rays), the
    // iteration that reaches the cap left to the loops below
    if (ordered && r.blind > steps0)
      dense_skip_blind<L::kSkip>(r.Px, r.Py, r.Pz, r.Ax, r.Ay, r.Az, r.dx, r.dy, r.dz, r.ix,
                                 r.iy, r.iz, mx, my, mz, s0, steps0,
                                 min(r.blind, max_steps - 1));
    if constexpr (L::kAhead) {
      const SkipGeneral<L::kSkip> it = {r.Px, r.Py, r.Pz, r.Ax, r.Ay, r.Az, r.dx, r.dy, r.dz,
                                        r.ix, r.iy, r.iz, mx,   my,   mz,   flip, vox};
      dense_skip_ahead<L::kSkip>(it, s0, steps0, limit);
    } else {
      dense_skip_empty<L::kSkip, false>(r.Px, r.Py, r.Pz, r.Ax, r.Ay, r.Az, r.dx, r.dy, r.dz, r.ix,
                                        r.iy, r.iz, mx, my, mz, flip, s0, steps0, limit, vox, vox,
                                        0u, false);
    }
  }
  float fwx, fwy, fwz;
  uint32_t fc, fM, fa, fv;
  int sF;
  bool wrappedF;
  dense_loop_prefetch(r.Px, r.Py, r.Pz, r.Ax, r.Ay, r.Az, r.dx, r.dy, r.dz, r.ix, r.iy, r.iz, mx,
                      my, mz, flip, s0, steps0, max_steps, vox, fwx, fwy, fwz, fc, fM, fa, fv,
                      sF, wrappedF);
  (void)lk;
  if (sF >= max_steps || wrappedF) {  // the loop cap, then the bounds test
    h.hit = false;
    h.steps = sF;
    return;
  }
  const uint32_t g = fc ^ flip;
  // faceId = 2 minIdx + 2 - rayPositivity[minIdx] (map.glsl:119-125)
  const bool fx = fM == mx, fy = fM == my;
  const int pm = (flip & fM) ? 0 : 1;  // the complemented axes are the negative ones
  h.hit = true;
  h.face = (fx ? 2 : (fy ? 4 : 6)) - pm;
  const uint32_t gx = compact1by2(g), gy = compact1by2(g >> 1), gz = compact1by2(g >> 2);
  h.bx = (int)gx;
  h.by = (int)gy;
  h.bz = (int)gz;
  if (fa != g) {  // a corrected lookup
    h.bx = (int)compact1by2(fa);
    h.by = (int)compact1by2(fa >> 1);
    h.bz = (int)compact1by2(fa >> 2);
  }
  h.code = fa;
  h.v = fv;
  h.sub = (uint32_t)((int)fwx & 7) | ((uint32_t)((int)fwy & 7) << 3) |
          ((uint32_t)((int)fwz & 7) << 6);
  h.hx = (float)(gx << 3) + fwx;
  h.hy = (float)(gy << 3) + fwy;
  h.hz = (float)(gz << 3) + fwz;
  h.steps = sF + 1;
}

// kStats with the clearance map keeps the fast loops: its statistics count
// the steps executed, rays ending early included.
template <bool kStats, class L>
__device__ __forceinline__ void dense_run(DenseRay& r, L& lk, const DenseWorld& w, DenseHit& h,
                                          uint32_t& l1f, uint32_t& l0f) {
  if constexpr (L::kPrefetch && (!kStats || L::kClear)) {
    dense_run_prefetch(r, lk, w, h);
    return;
  }
  const float Px = r.Px, Py = r.Py, Pz = r.Pz, Ax = r.Ax, Ay = r.Ay, Az = r.Az;
  const float dx = r.dx, dy = r.dy, dz = r.dz, ix = r.ix, iy = r.iy, iz = r.iz;
  const uint32_t mx = w.mx, my = w.my, mz = w.mz, flip = r.flip;
  const int max_steps = r.max_steps;
  float wx = r.wx, wy = r.wy, wz = r.wz;
  uint32_t c = r.c;
  uint32_t M = mx;
  uint32_t a;
  int steps = r.steps;
  uint32_t v;
  bool wrapped;
  do {
    float tx = (Px - wx) * ix;
    float ty = (Py - wy) * iy;
    float tz = (Pz - wz) * iz;
    bool xy = tx < ty, xz = tx < tz, yz = ty < tz;
    bool m0 = xy & xz;
    bool m1 = (!xy) & yz;
    float tm = m0 ? tx : (m1 ? ty : tz);
    float nwx = wx + dx * tm;
    float nwy = wy + dy * tm;
    float nwz = wz + dz * tm;
    wx = m0 ? Ax : nwx;
    wy = m1 ? Ay : nwy;
    wz = (m0 | m1) ? nwz : Az;
    M = m0 ? mx : (m1 ? my : mz);
    const uint32_t cm = c & M;
    wrapped = cm == M;
    c = ((cm - M) & M) | (c & ~M);
    steps++;
    a = c ^ flip;
    bool outside = false;
    if (fmaxf(fmaxf(wx, wy), wz) >= 8.0f) {  // pos >> 3 = G + (int(within) >> 3)
      if (wx >= 8.0f) a = morton_inc(a, mx, outside);
      if (wy >= 8.0f) a = morton_inc(a, my, outside);
      if (wz >= 8.0f) a = morton_inc(a, mz, outside);
    }
    v = outside ? 0u : lk.template probe<kStats>(w, a, l1f, l0f);
  } while (!wrapped & (v == 0u) & (steps < max_steps));

  if (steps >= max_steps || wrapped) {  // the loop cap, then the bounds test
    h.hit = false;
    h.steps = steps;
    return;
  }
  const uint32_t g = c ^ flip;
  h.hit = true;
  h.face = (M == mx ? 2 : (M == my ? 4 : 6)) - ((flip & M) ? 0 : 1);
  h.bx = (int)compact1by2(a);
  h.by = (int)compact1by2(a >> 1);
  h.bz = (int)compact1by2(a >> 2);
  h.code = a;
  h.v = v;
  h.sub = (uint32_t)((int)wx & 7) | ((uint32_t)((int)wy & 7) << 3) |
          ((uint32_t)((int)wz & 7) << 6);
  h.hx = (float)(compact1by2(g) << 3) + wx;
  h.hy = (float)(compact1by2(g >> 1) << 3) + wy;
  h.hz = (float)(compact1by2(g >> 2) << 3) + wz;
  h.steps = steps + 1;
}

// ---------------------------------------------------------------------------
// reference brickmap + atlas layout (literal two-level traceMap)
// ---------------------------------------------------------------------------
struct BrickmapWorld {
  const uint32_t* chunks;  // (dim/8)^3, 0 = empty else pool index + 1
  const uint32_t* pool;    // 512 u32 per block, in-block index x + 8y + 64z
  const uint32_t* atlas;   // 256^3 RGBA8 texels
  // nonzero texels of model m (8^3, a cache line): word 8 m + z, bit x + 8 y;
  // present with occ
  const uint64_t* masks;
  uint32_t dim;            // MAP_DIMENSION
  // block occupancy for the empty-space loop (power-of-two dim only, else
  // null): byte at morton(block) = (map_getVoxel(block) != 0)
  const uint8_t* occ;
  uint32_t nvox;           // dim^3
  uint32_t mx, my, mz;     // dilated Morton masks of x, y, z
  // clearance map of the occupancy bytes (as DenseWorld's); clear_bytes 0 =
  // not used
  const uint8_t* clear;
  uint32_t clear_bytes, clear_oct_bytes;
};

// map_getVoxel (map.glsl:38-47) of block coordinates b; counts the chunk-table
// and pool reads it makes.
template <bool kStats = false>
__device__ __forceinline__ uint32_t bm_block(const BrickmapWorld& w, int bx, int by, int bz,
                                             uint32_t* chunk_reads = nullptr,
                                             uint32_t* pool_reads = nullptr) {
  int M = (int)(w.dim >> 3);
  int cx = bx >> 3, cy = by >> 3, cz = bz >> 3;
  if (cx < 0 || cy < 0 || cz < 0 || cx >= M || cy >= M || cz >= M) return 0;
  uint32_t idx = w.chunks[cx + M * (cy + cz * M)];
  if (kStats) ++*chunk_reads;
  if (idx == 0) return 0;
  size_t o = (size_t)(idx - 1u) * 512u + (size_t)(bx % 8) + (size_t)(((bz % 8) * 8 + (by % 8)) * 8);
  if (kStats) ++*pool_reads;
  return w.pool[o];
}

// map_getSubVoxel (map.glsl:57-60)
__device__ __forceinline__ uint32_t bm_sub(const BrickmapWorld& w, uint32_t block, int sx, int sy,
                                           int sz) {
  // sx, sy, sz = pos % 8 lie in [0, 8) (pos >= 0 once the bounds check
  // passed); the & 255 only keeps the texel inside the 256^3 atlas by
  // construction.
  uint32_t id = block & 0xFFFFFFFu;
  uint32_t x = ((uint32_t)sx + (id & 31u) * 8u) & 255u;
  uint32_t y = ((uint32_t)sy + ((id / 32u) & 31u) * 8u) & 255u;
  uint32_t z = ((uint32_t)sz + ((id / 1024u) & 31u) * 8u) & 255u;
  return w.atlas[x + 256u * (y + 256u * z)];
}

struct GeneralHit {
  uint32_t data;
  int face;
  int bx, by, bz;
  uint32_t sub;
  float hx, hy, hz;
  int steps;
};

// traceMap (map.glsl:83-168) literally, both levels.
template <bool kStats>
__device__ bool trace_general(const BrickmapWorld& w, float ox, float oy, float oz, float dx,
                              float dy, float dz, int max_steps, GeneralHit& h,
                              uint32_t& chunk_reads, uint32_t& pool_atlas_reads) {
  if (dx == 0.0f) dx = 0.001f;
  if (dy == 0.0f) dy = 0.001f;
  if (dz == 0.0f) dz = 0.001f;
  const int B = (int)(8u * w.dim);
  int sgn[3] = {dx > 0.0f ? 1 : (dx < 0.0f ? -1 : 0), dy > 0.0f ? 1 : (dy < 0.0f ? -1 : 0),
                dz > 0.0f ? 1 : (dz < 0.0f ? -1 : 0)};
  int pv[3] = {(1 + sgn[0]) >> 1, (1 + sgn[1]) >> 1, (1 + sgn[2]) >> 1};
  float d[3] = {dx, dy, dz};
  float inv[3] = {1.0f / dx, 1.0f / dy, 1.0f / dz};
  int m = 0;
  float o8[3] = {ox * 8.0f, oy * 8.0f, oz * 8.0f};
  int g[3] = {f2i_sat(o8[0]), f2i_sat(o8[1]), f2i_sat(o8[2])};
  float wc[3] = {o8[0] - (float)g[0], o8[1] - (float)g[1], o8[2] - (float)g[2]};
  int s = 0;
  h.data = 0;
  h.hx = h.hy = h.hz = -1.0f;
  int step;
  for (step = 0; step < max_steps; step++) {
    if (g[0] >= B || g[1] >= B || g[2] >= B || g[0] < 0 || g[1] < 0 || g[2] < 0) break;
    int p[3] = {g[0] + (int)wc[0], g[1] + (int)wc[1], g[2] + (int)wc[2]};
    int b[3] = {p[0] >> 3, p[1] >> 3, p[2] >> 3};
    uint32_t block = bm_block<kStats>(w, b[0], b[1], b[2], &chunk_reads, &pool_atlas_reads);
    if (block != 0u) {
      uint32_t sub = bm_sub(w, block, p[0] % 8, p[1] % 8, p[2] % 8);
      if (kStats) pool_atlas_reads++;
      if (sub != 0u) {
        h.data = sub;
        h.face = m == 0 ? 2 - pv[0] : (m == 1 ? 4 - pv[1] : 6 - pv[2]);
        h.bx = b[0];
        h.by = b[1];
        h.bz = b[2];
        h.sub = (uint32_t)(p[0] & 7) | ((uint32_t)(p[1] & 7) << 3) | ((uint32_t)(p[2] & 7) << 6);
        h.hx = (float)g[0] + wc[0];
        h.hy = (float)g[1] + wc[1];
        h.hz = (float)g[2] + wc[2];
        h.steps = step + 1;
        return true;
      }
      if (s != 0) {
#pragma unroll
        for (int i = 0; i < 3; i++) {
          g[i] += (int)wc[i];
          wc[i] = wc[i] - floorf(wc[i]);
        }
        s = 0;
      }
    } else if (s != 3) {
#pragma unroll
      for (int i = 0; i < 3; i++) {
        int lo = g[i] & 7;
        wc[i] = wc[i] + (float)lo;
        g[i] -= lo;
      }
      s = 3;
    }
    float t[3];
#pragma unroll
    for (int i = 0; i < 3; i++) t[i] = ((float)(pv[i] << s) - wc[i]) * inv[i];
    m = t[0] < t[1] ? (t[0] < t[2] ? 0 : 2) : (t[1] < t[2] ? 1 : 2);
    float tm = m == 0 ? t[0] : (m == 1 ? t[1] : t[2]);
    int sm = m == 0 ? sgn[0] : (m == 1 ? sgn[1] : sgn[2]);
    int pm = m == 0 ? pv[0] : (m == 1 ? pv[1] : pv[2]);
    float am = (float)((1 - pm) << s) * 0.999f;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      float nw = wc[i] + d[i] * tm;
      wc[i] = (i == m) ? am : nw;
      g[i] += (i == m) ? sm * (1 << s) : 0;
    }
  }
  h.steps = step;
  return false;
}


// traceMap over the reference layout with the empty-space steps on the fast
// path: whenever the literal loop is at the block level (stepSize 3) and the
// block it just looked up is empty, the following block-level steps run in
// the pipelined Morton loop over the occupancy bytes (the same recurrence,
// the same stopping rule) until a step lands on a nonempty block, leaves the
// map or reaches the cap; the literal loop then resumes at that block's
// lookup with the same grid / within / minIdx / step count.  Same hits, steps
// and positions as trace_general.  The literal loop is an inner loop that a
// lane leaves when it reaches an empty block: a wave's lanes that leave a
// model block (or start inside one, as shadow rays do) after different
// numbers of sub-voxel steps then run their empty-space steps together
// instead of one group after another.
// kPositive: the caller guarantees a direction with no negative component (the
// zero substitution below makes it positive), and the empty-space steps take
// dense_skip_positive.
// kClear: the empty-space runs take the clearance map of the occupancy bytes.
// It holds here too: block-level lookups only descend into nonempty blocks,
// so a stretch whose block-level lookups all read empty is walked at the
// block level, and each run starts its line from the walk's own position.
// kShadow: the ray starts next to a nonempty block.
// inv = 1 / d after the zero substitution.
template <bool kPositive = false, bool kClear = false, bool kShadow = false>
__device__ bool trace_brickmap_fast(const BrickmapWorld& w, float ox, float oy, float oz, float dx,
                                    float dy, float dz, const float* inv, int max_steps,
                                    GeneralHit& h) {
  constexpr int kSkip = kClear ? kSkipClear : kSkipShort;
  if (dx == 0.0f) dx = 0.001f;
  if (dy == 0.0f) dy = 0.001f;
  if (dz == 0.0f) dz = 0.001f;
  const int B = (int)(8u * w.dim);
  int sgn[3] = {dx > 0.0f ? 1 : (dx < 0.0f ? -1 : 0), dy > 0.0f ? 1 : (dy < 0.0f ? -1 : 0),
                dz > 0.0f ? 1 : (dz < 0.0f ? -1 : 0)};
  int pv[3] = {(1 + sgn[0]) >> 1, (1 + sgn[1]) >> 1, (1 + sgn[2]) >> 1};
  float d[3] = {dx, dy, dz};
  // block-level constants of the fast loop (stepSize 3)
  const float P3[3] = {(float)(pv[0] << 3), (float)(pv[1] << 3), (float)(pv[2] << 3)};
  const float A3[3] = {(float)((1 - pv[0]) << 3) * 0.999f, (float)((1 - pv[1]) << 3) * 0.999f,
                       (float)((1 - pv[2]) << 3) * 0.999f};
  const uint32_t flip = (pv[0] ? 0u : w.mx) | (pv[1] ? 0u : w.my) | (pv[2] ? 0u : w.mz);
  const __amdgpu_buffer_rsrc_t occ =
      __builtin_amdgcn_make_buffer_rsrc((void*)w.occ, (short)0, (int)w.nvox, 0x00020000);
  int m = 0;
  float o8[3] = {ox * 8.0f, oy * 8.0f, oz * 8.0f};
  int g[3] = {f2i_sat(o8[0]), f2i_sat(o8[1]), f2i_sat(o8[2])};
  float wc[3] = {o8[0] - (float)g[0], o8[1] - (float)g[1], o8[2] - (float)g[2]};
  int s = 0;
  h.data = 0;
  h.hx = h.hy = h.hz = -1.0f;
  int step = 0;
  bool hit = false;
  // and of the walk inside a model block (stepSize 0): an eighth, exactly
  const float P1[3] = {P3[0] * 0.125f, P3[1] * 0.125f, P3[2] * 0.125f};
  const float A1[3] = {A3[0] * 0.125f, A3[1] * 0.125f, A3[2] * 0.125f};
  // rays with unordered crossing times take the exact loop alone
  const bool ordered = dense_ordered(inv[0], inv[1], inv[2], wc[0], wc[1], wc[2]);
  const int limit = ordered ? max_steps : 0;
  // the map's plane and whether the direction allows it; a primary ray's
  // first run starts with a stretch without lookups
  const __amdgpu_buffer_rsrc_t cm = clear_rsrc(w.clear, w.clear_bytes);
  const bool usable = kClear && ordered && clear_usable(inv[0], inv[1], inv[2]);
  bool open = kClear && !kShadow;
  bool paused = false;  // in the middle of an empty-space run
  for (;;) {
    // The literal loop (both levels) until the lane stands at an empty
    // block at the block level, hits, leaves the map or reaches the cap.
    // Lanes at an empty block wait here for the rest of the wave, so the
    // wave's empty-space runs below start together.
    bool fast = paused;
    paused = false;
    // The block of the last lookup, so that the lookup of a step inside it
    // makes no load.  Successive lookups are neighbours, so 11 bits an axis
    // tell their blocks apart.
    uint32_t key = 0xFFFFFFFFu, block = 0u;
    while (!fast) {
      if (step >= max_steps || g[0] >= B || g[1] >= B || g[2] >= B || g[0] < 0 || g[1] < 0 ||
          g[2] < 0)
        break;
      int p[3] = {g[0] + (int)wc[0], g[1] + (int)wc[1], g[2] + (int)wc[2]};
      int b[3] = {p[0] >> 3, p[1] >> 3, p[2] >> 3};
      const uint32_t k = (uint32_t)b[0] + ((uint32_t)b[1] << 11) + ((uint32_t)b[2] << 22);
      if (k != key) {
        key = k;
        block = bm_block(w, b[0], b[1], b[2]);
      }
      if (block != 0u) {
        // (a model's texels lie in 64 cache lines, its mask in one)
        const uint64_t layer = w.masks[(size_t)(block & 0x7FFFu) * 8u + ((uint32_t)p[2] & 7u)];
        if ((layer >> (((uint32_t)p[0] & 7u) | (((uint32_t)p[1] & 7u) << 3))) & 1u) {
          h.data = bm_sub(w, block, p[0] & 7, p[1] & 7, p[2] & 7);
          h.face = m == 0 ? 2 - pv[0] : (m == 1 ? 4 - pv[1] : 6 - pv[2]);
          h.bx = b[0];
          h.by = b[1];
          h.bz = b[2];
          h.sub = (uint32_t)(p[0] & 7) | ((uint32_t)(p[1] & 7) << 3) | ((uint32_t)(p[2] & 7) << 6);
          h.hx = (float)g[0] + wc[0];
          h.hy = (float)g[1] + wc[1];
          h.hz = (float)g[2] + wc[2];
          h.steps = step + 1;
          hit = true;
          break;
        }
        if (s != 0) {
#pragma unroll
          for (int i = 0; i < 3; i++) {
            g[i] += (int)wc[i];
            wc[i] = wc[i] - floorf(wc[i]);
          }
          s = 0;
        }
      } else {
        if (s != 3) {
#pragma unroll
          for (int i = 0; i < 3; i++) {
            int lo = g[i] & 7;
            wc[i] = wc[i] + (float)lo;
            g[i] -= lo;
          }
          s = 3;
        }
        fast = true;  // this iteration's step onwards run in the loop below
        break;
      }
      // Inside the model block: its voxels one by one (stepSize 0), until one
      // is solid or the ray leaves the block; the lookup above then takes that
      // step.  p is g here: a within of 1 or more (a tie) ends the walk too.
      // By the lookup above alone a step was 260 instructions and up to three
      // dependent loads (chunk table, pool, atlas): 2400 cycles in the waves a
      // frame ends with, where these steps took a third of the time.  Here it
      // is 50 and one load that hits the L1.  Six views of the engine's frame at
      // 1280x720 121 -> 104 us, of its map with long caps at 1600x900 230 ->
      // 200, at 320x180 163 -> 127.
      const uint64_t* model = w.masks + (size_t)(block & 0x7FFFu) * 8u;
      const int base[3] = {p[0] & ~7, p[1] & ~7, p[2] & ~7};
      bool on;
      do {
        const float tx = (P1[0] - wc[0]) * inv[0];
        const float ty = (P1[1] - wc[1]) * inv[1];
        const float tz = (P1[2] - wc[2]) * inv[2];
        const bool m0 = (tx < ty) & (tx < tz), m1 = !(tx < ty) & (ty < tz);
        const float tm = m0 ? tx : (m1 ? ty : tz);
        const float nx = wc[0] + d[0] * tm, ny = wc[1] + d[1] * tm, nz = wc[2] + d[2] * tm;
        wc[0] = m0 ? A1[0] : nx;
        wc[1] = m1 ? A1[1] : ny;
        wc[2] = (m0 | m1) ? nz : A1[2];
        g[0] += m0 ? sgn[0] : 0;
        g[1] += m1 ? sgn[1] : 0;
        g[2] += (m0 | m1) ? 0 : sgn[2];
        m = m0 ? 0 : (m1 ? 1 : 2);
        step++;
        const uint32_t out = (uint32_t)((g[0] ^ base[0]) | (g[1] ^ base[1]) | (g[2] ^ base[2]));
        const float wm = fmaxf(fmaxf(fabsf(wc[0]), fabsf(wc[1])), fabsf(wc[2]));
        const uint64_t word = model[g[2] & 7];
        const uint32_t bit = ((uint32_t)g[0] & 7u) | (((uint32_t)g[1] & 7u) << 3);
        on = (out < 8u) & (wm < 1.0f) & (step < max_steps) & !((word >> bit) & 1u);
      } while (on);
    }
    if (!fast) break;
    // empty block at the block level: the fast loop takes the next steps
    DenseCell s0;
    s0.wx = wc[0];
    s0.wy = wc[1];
    s0.wz = wc[2];
    s0.c = morton3((uint32_t)g[0] >> 3, (uint32_t)g[1] >> 3, (uint32_t)g[2] >> 3) ^ flip;
    const uint32_t mx = in_vgpr(w.mx), my = in_vgpr(w.my), mz = in_vgpr(w.mz);
    int s0steps = step;
    int status;
    const uint32_t cofs =
        kPositive || !kClear ? 0u : clear_octant_offset(flip, mx, my, mz, w.clear_oct_bytes);
    const int entered = __popcll(__ballot(true));
    for (;;) {
      if constexpr (kClear) {
        if (open & usable) {
          if (!clear_advance<kClearSteps>(P3[0], P3[1], P3[2], A3[0], A3[1], A3[2], d[0], d[1],
                                          d[2], inv[0], inv[1], inv[2], flip, mx, my, mz, w.dim,
                                          s0, s0steps, max_steps, cm, cofs, w.clear_oct_bytes) ||
              s0steps >= max_steps) {
            status = kSkipFree;
            break;
          }
        }
      }
      if constexpr (kPositive)
        status = dense_skip_positive<kSkip, kClear, kClear>(d[0], d[1], d[2], inv[0], inv[1], inv[2], mx,
                                                    my, mz, s0, s0steps, limit, occ, cm, usable,
                                                    entered);
      else
        status = dense_skip_empty<kSkip, kClear, kClear>(P3[0], P3[1], P3[2], A3[0], A3[1], A3[2], d[0],
                                                 d[1], d[2], inv[0], inv[1], inv[2], mx, my, mz,
                                                 flip, s0, s0steps, limit, occ, cm, cofs,
                                                 usable, entered);
      if (status != kSkipOpen) break;
      open = true;
    }
    open = false;  // the next run starts at a nonempty block
    if (kClear && status == kSkipPause) {
      // Three quarters of the rays that began this run wait for the rest, at
      // blocks of their own: those go on first, and this ray takes its run up
      // again with them, from the state it has reached.  Otherwise every run of
      // a wave lasts as long as its longest ray's, and a wave whose rays meet
      // model blocks at different depths pays the longest run once per block
      // (half of the cycles of a frame's last waves).  Six views of the engine's
      // map with long caps at 1600x900 203 -> 184 us, at 320x180 143 -> 135, an
      // edit with its frame 312 -> 296, the engine's frame 104.5 -> 104.6; at half
      // of the rays 175, 142, 290 and 107; at a sixth 194, 140, 300 and 105.
      paused = true;
      const uint32_t gc = s0.c ^ flip;
      g[0] = (int)(compact1by2(gc) << 3);
      g[1] = (int)(compact1by2(gc >> 1) << 3);
      g[2] = (int)(compact1by2(gc >> 2) << 3);
      wc[0] = s0.wx;
      wc[1] = s0.wy;
      wc[2] = s0.wz;
      step = s0steps;
      continue;
    }
    if (kClear && status == kSkipFree) {
      step = s0steps;
      break;
    }
    float fw[3];
    uint32_t fc, fM, fa, fv;
    int sF;
    bool wrappedF;
    dense_loop_prefetch(P3[0], P3[1], P3[2], A3[0], A3[1], A3[2], d[0], d[1], d[2], inv[0],
                        inv[1], inv[2], mx, my, mz, flip, s0, s0steps, max_steps, occ, fw[0],
                        fw[1], fw[2], fc, fM, fa, fv, sF, wrappedF);
    (void)fa;
    (void)fv;
    step = sF;  // iteration sF starts with its bounds test and lookup
    if (wrappedF) break;  // left the map: the bounds test of iteration sF
    const uint32_t gc = fc ^ flip;
    g[0] = (int)(compact1by2(gc) << 3);
    g[1] = (int)(compact1by2(gc >> 1) << 3);
    g[2] = (int)(compact1by2(gc >> 2) << 3);
    wc[0] = fw[0];
    wc[1] = fw[1];
    wc[2] = fw[2];
    m = fM == mx ? 0 : (fM == my ? 1 : 2);
  }
  if (!hit) h.steps = step;
  return hit;
}

}  // namespace vt
