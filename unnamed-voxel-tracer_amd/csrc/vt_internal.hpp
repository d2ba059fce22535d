// vt_internal.hpp -- host-side objects behind the C-ABI handles and the
// launchers each kernel translation unit exports.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "../../include/vt.h"
#include "vt_trace.hpp"

// Staging owned by a context, allocated once by vt_create: page-locked host
// memory that kernels read and write in place.  It carries the edit lists of
// vt_world_set_voxels (larger ones take device memory for the call), the
// coordinates and values of vt_world_get_voxels (in chunks of
// kCtxStageVoxels), the pick result, and what the host needs to know of a
// rebuilt free-region map, so that small calls make no copies and no
// allocations: a copy of a few bytes costs 11-13 us of its own, a kernel
// with a synchronisation 11 us with the bytes on either side.  Calls that use
// it return only after their stream work is done, so calls made one after
// another on the context's thread never overlap on it.
constexpr size_t kCtxStageBytes = 256u * 1024u;
constexpr uint32_t kCtxStageVoxels = (uint32_t)(kCtxStageBytes / 16u);  // 12 B xyz + 4 B value
constexpr size_t kCtxReportBytes = 256;  // after the staging: CtxReport

// What the map builders report to the host (written by the device into the
// context's staging, valid once the stream has synchronised).
struct CtxReport {
  uint32_t free_built;       // 0: no region had changed, the map was left as it is
  uint32_t free_regions[8];  // else: free regions of each octant
  uint32_t near_cells;       // near cells of the clearance map that are not filled
  uint32_t filled_cells;     // cells of it with something in every 2^3 sub-block
  int32_t box_lo[3], box_hi[3];  // box of the nonempty voxels; lo > hi: none
};
static_assert(sizeof(CtxReport) <= kCtxReportBytes, "CtxReport");

struct vt_ctx {
  int device;
  int compute_units;
  char name[256];
  void* stage;        // kCtxStageBytes + kCtxReportBytes of page-locked host memory
  void* stage_dev;    // its device address
  // (the report follows the staging)
  CtxReport* report() const {
    return reinterpret_cast<CtxReport*>(static_cast<char*>(stage) + kCtxStageBytes);
  }
  CtxReport* report_dev() const {
    return reinterpret_cast<CtxReport*>(static_cast<char*>(stage_dev) + kCtxStageBytes);
  }
};

enum class WorldKind { Dense, Brickmap };

struct vt_world {
  vt_ctx* ctx;
  WorldKind kind;
  uint32_t dim;
  size_t bytes;
  // dense (Morton order)
  uint8_t* vox;
  uint64_t* l0;
  uint64_t* l1;
  uint64_t* l1b;  // 8^3-brick level, l1b_words(dim) words
  uint32_t* palette;
  // brickmap
  uint32_t* chunks;
  uint32_t* pool;
  uint32_t* atlas;
  size_t pool_words;     // words of allocated blocks (512 per block)
  size_t pool_capacity;  // words the device pool holds
  uint32_t* chunk_mirror;  // host copy of the chunk table (edit allocation)
  uint8_t* occ;            // block occupancy in Morton order (power-of-two dim)
  uint64_t* masks;         // texel masks of the atlas's models (with occ)
  uint64_t* brick_bits;    // brickmap: bit per 4^3 brick of blocks, from occ
  // free-region map (dense worlds and power-of-two brickmap worlds)
  uint32_t* freemap;       // 8 octants x free_words_per_octant(dim) words, then
                           // the words edits set (maps_changed)
  // clearance map (the same worlds, dim >= 16)
  uint8_t* clear;          // 2 orders x 8 octants x clear_cells(dim) bytes
  uint8_t* clear_tmp;      // clear_tmp_bytes(dim): the sub-block bits of every
                           // 4^3 brick (kept current), then build scratch;
                           // dim >= 32
  bool maps_valid;         // both maps match the occupancy (finish_maps)
  float near_frac;         // share of near cells among the clearance map's cells
                           // that are not filled: of the space rays cross
  float free_frac;         // largest share of free regions over the 8 octants
  // the box of a dense world's nonempty voxels, inclusive; grown by edits,
  // never shrunk; box_any = false while the world has none
  int32_t box_lo[3], box_hi[3];
  bool box_any;
  // compact albedo index of a dense world (built on request)
  uint32_t* prefix;     // occupied voxels before each L0 word
  uint64_t n_occupied;
};

namespace vt {

// Error reporting shared by the C-ABI translation units: record a detail
// message for vt_last_error() and return the status.
int fail(int status, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
int hip_fail(hipError_t e, const char* what);
bool aligned(const void* p, size_t a);
void dev_free(void* p);

#define VT_HIP(call)                                       \
  do {                                                     \
    hipError_t e_ = (call);                                \
    if (e_ != hipSuccess) return ::vt::hip_fail(e_, #call); \
  } while (0)

// Per-launch shading constants.
struct ShadeConsts {
  float sun[3];
  RayConsts shadow;  // the shadow rays' direction constants (set by the dense launchers)
  // what every hit has in common (the illumination image holds the sun):
  float sun_n[3], sun_len;     // sun / |sun| and |sun|
  float illum[3];              // illumination.xyz, through rgba8 if the G-buffer is
  float illum_lit, illum_occ;  // illumination.w
  SkyBase sky;                 // of the sky along illumination.xyz
  bool cull_entities;          // may_meet_entities holds for the sun
  int max_primary, max_shadow;
  uint32_t flags;
  float ambient;
  const float* albedo;
  float* grad_albedo;  // VT_FLAG_GRAD_L2 accumulators
  float* grad_sun;
  float* loss;
};

// Output pointers (any may be null).
struct alignas(8) FrameOut {
  float4* shaded;
  uint32_t* hits;  // 3 words per pixel
  float4* color;
  float4* normal;
  float4* position;
  float4* illum;
  uint32_t* steps;
  unsigned long long* stats;
  const float4* target;  // VT_FLAG_GRAD_L2 input
  uint32_t* display;     // VT_FLAG_PRESENT RGBA8 output
};

// Wave tile: 64 lanes cover tile_w x (64 / tile_w) pixels; a 256-thread
// block covers 2 x 2 wave tiles.
struct TileShape {
  uint32_t log2_w;  // 3 (8x8), 4 (16x4) or 5 (32x2)
};

// Bit k = byte k of v is nonzero.
__device__ __forceinline__ uint32_t nonzero_bytes(uint64_t v) {
  uint64_t y = v | (v >> 4);
  y |= y >> 2;
  y |= y >> 1;
  y &= 0x0101010101010101ull;
  return (uint32_t)((y * 0x0102040810204080ull) >> 56);
}

DenseWorld dense_view(const vt_world* w);
void grow_box(vt_world* w, int32_t x, int32_t y, int32_t z);
void reach_of(const vt_world* w, float* lo, float* hi);
BrickmapWorld brickmap_view(const vt_world* w);

// Takes the device address of the no-allocation scratch array on `device`
// (the current device) once per device; called by vt_create.
int noalloc_init(int device);

// Host-side validation and translation of the C-ABI structs.
int check_image_size(uint32_t W, uint32_t H, const char* who);
int check_params(const vt_render_params& p, const vt_world* world, const char* who);
// The Lambert modes divide by |sun|: false when its binary32 squared length
// is 0 (or overflows), where that division has no finite result.
bool sun_normalizable(const float sun[3]);
int check_frame(const vt_frame* frame, uint32_t flags, const char* who);
ViewConsts view_consts(const vt_camera* camera, uint32_t W, uint32_t H);
ShadeConsts shade_consts(const vt_render_params& p);
FrameOut frame_out(const vt_frame* frame);

// `schedule`: the frame's tile schedule buffer (vt_frame.schedule) or null.
hipError_t launch_render_dense(const DenseWorld& w, uint32_t traversal, const ViewConsts& v,
                               const ShadeConsts& sc, const FrameOut& out, uint32_t* schedule,
                               TileShape tile, uint32_t compute_units, hipStream_t stream);
hipError_t launch_render_brickmap(const BrickmapWorld& w, const ViewConsts& v,
                                  const ShadeConsts& sc, const FrameOut& out, uint32_t* schedule,
                                  TileShape tile, hipStream_t stream);

// World construction kernels.
// occ[morton(b)] = (map_getVoxel(b) != 0) for every block b of a brickmap
// world (power-of-two dim) with y < y_end (0: all layers), and the brick
// bits of those layers' 4^3 bricks (bits of a partly covered word are set
// only, never cleared: the other layers' bits must be right already).
// sub (may be null): the clearance map's byte of each of those bricks.
// The texel masks of all 32^3 models of an atlas (BrickmapWorld::masks).
constexpr size_t kAtlasMaskWords = 32768u * 8u;
hipError_t launch_atlas_masks(const uint32_t* atlas, uint64_t* masks, hipStream_t stream);
hipError_t launch_build_occupancy(const BrickmapWorld& w, uint8_t* occ, uint64_t* brick_bits,
                                  uint8_t* sub, hipStream_t stream, uint32_t y_end = 0);
// Grows a brickmap world's block pool to at least `blocks` blocks by
// doubling (GpuBlockAllocator.alloc, gpu_block_allocator.zig:20-30), keeping
// the contents and zeroing the new blocks; `who` names the caller in errors.
int grow_pool(vt_world* w, uint64_t blocks, hipStream_t s, const char* who);
// The Morton-ordered voxels of a linear grid and their occupancy levels, and
// the box of the nonempty voxels into *report (which holds an empty box
// before); sub: the clearance map's byte of each 4^3 brick.
hipError_t launch_build_dense(const uint8_t* linear, uint32_t dim, uint8_t* vox, uint64_t* l0,
                              uint64_t* l1, uint64_t* l1b, uint8_t* sub, int32_t* box6,
                              CtxReport* report, hipStream_t stream);
// Words of the 8^3-brick level of a dim^3 world: one per 32^3 region (one
// partial word for dim 16).
inline uint64_t l1b_words(uint32_t dim) {
  const uint64_t n = (uint64_t)dim * dim * dim / 32768u;
  return n ? n : 1u;
}
// Rebuilds the listed L1b words (all l1b_words(dim) when words is null)
// from the L0 words, n0 of them.
hipError_t launch_build_l1b(const uint64_t* l0, uint64_t n0, const uint32_t* words,
                            uint32_t nwords, uint64_t* l1b, hipStream_t stream);
// Free-region map: regions of 16^3 blocks, R = free_regions(dim) per axis;
// bit r of octant o's bitmap (free_words_per_octant(dim) words) is set when
// no region at or ahead of r on every axis in o's travel direction holds a
// nonempty block.  Built from a dense world's L1b words or a brickmap world's
// brick_bits, unless *changed (device, may be null) is 0;
// reports whether it was and the free regions of each octant.
uint32_t free_regions(uint32_t dim);
uint32_t free_words_per_octant(uint32_t dim);
// Clearance map (ClearMap in vt_trace.hpp): 2 x 8 octant planes of
// clear_cells(dim) bytes, built from one byte per 4^3 brick (a bit per 2^3
// sub-block) at the start of tmp, unless *changed (device, may be null) is 0;
// reports the near cells.
uint32_t clear_cells(uint32_t dim);
size_t clear_tmp_bytes(uint32_t dim);
// Whether launches with these flags and step caps use the clearance map: it is
// valid and VT_FLAG_FREE_MAP_ON, or neither FREE_MAP flag and a world open
// enough for it to pay.
bool use_clear_map(const vt_world* w, uint32_t flags, int max_primary, int max_shadow);
// Whether vt_render uses it for this world, parameters and frame: no stored
// step counts (they would lack the steps of rays that end early); on dense
// worlds the flat traversal, and statistics only with VT_FLAG_FREE_MAP_ON
// (they then count the steps executed); on the reference layout occupancy
// bytes and no statistics.
bool render_clear_map(const vt_world* w, const vt_render_params& p, const vt_frame& f);
// To be called before the first kernel that changes a world's voxels is
// enqueued: from here until finish_maps the maps and the occupancy levels may
// differ from the voxels, and the renderers read neither map.  False: they
// did already (an earlier change failed midway), so the levels have to be
// made from all voxels and the maps rebuilt whatever this change does.
inline bool begin_occupancy_change(vt_world* w) {
  const bool current = w->maps_valid || !w->freemap;
  w->maps_valid = false;
  return current;
}
// Rebuilds a world's free-region and clearance maps from its current
// occupancy (L1b words or brick bits, and the sub-block bits); no-op without
// them.  `changed`: the words of maps_changed (null: rebuild everything).
// Leaves maps_valid false: the caller calls finish_maps once the stream has
// synchronised without error.
hipError_t rebuild_maps(vt_world* w, hipStream_t stream, const uint32_t* changed = nullptr);
// The words edits set: [0] a 16^3 region emptied or filled; [1 ..] bit z: a
// 2^3 sub-block did from which the near cells of layer z follow (cells of the
// clearance map, at most 128 layers).
constexpr uint32_t kChangedWords = 5;
inline uint32_t* maps_changed(const vt_world* w) {
  return w->freemap ? w->freemap + 8u * free_words_per_octant(w->dim) : nullptr;
}
// After a rebuild completed: takes what the context's report says (free_frac,
// near_frac) and marks the maps valid.
void finish_maps(vt_world* w);
// The free-region rule (vt.h): the map is valid and has a free region, and
// VT_FLAG_FREE_MAP_ON, or neither FREE_MAP flag, a step cap of at least
// VT_FREE_MIN_CAP and at least 1/VT_FREE_MIN_SHARE of the regions free in
// some octant.
bool use_free_map(const vt_world* w, const ShadeConsts& sc);
// vt_free_map_used: use_free_map, and no stored step counts; on dense worlds
// the flat traversal, and statistics only with VT_FLAG_FREE_MAP_ON (they
// then count the steps executed); on the reference layout occupancy bytes
// and no statistics.
bool render_free_map(const vt_world* w, const vt_render_params& p, const vt_frame& f);
// Words of a brickmap world's brick bits: one uint64 per 4096 codes.
uint32_t brick_bit_words(uint32_t dim);
// Exclusive prefix sum of popcount(l0[i]) into prefix[0..nwords); scratch
// holds ceil(nwords/1024) + 1 words; *total receives the sum (device).
hipError_t launch_compact_prefix(const uint64_t* l0, uint64_t nwords, uint32_t* prefix,
                                 uint32_t* scratch, hipStream_t stream);

// Lambert shading / backward from stored hit records.
hipError_t launch_present(const float4* composite, uint32_t W, uint32_t H, float4* out,
                          uint32_t* display, hipStream_t stream);
hipError_t launch_lambert_shade(const DenseWorld& w, const ShadeConsts& sc, const uint32_t* hits,
                                uint32_t npix, float4* out, hipStream_t stream);
hipError_t launch_lambert_backward(const DenseWorld& w, const ShadeConsts& sc,
                                   const uint32_t* hits, uint32_t npix, const float4* upstream,
                                   uint32_t kind, hipStream_t stream);

}  // namespace vt
