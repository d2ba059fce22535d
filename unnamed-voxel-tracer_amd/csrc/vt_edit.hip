// vt_edit.hip -- world edits, voxel reads and the centre-ray pick.
//
// Edits replace VoxelBrickmap.set (src/engine/voxel.zig:46-61, the CPU
// writing through a persistent mapping) and map_setVoxel (map.glsl:49-55);
// reads replace VoxelBrickmap.get / map_getVoxel (voxel.zig:63-70,
// map.glsl:38-47); the pick is terrain_edit.comp.glsl:11-17.
//
// A batch of edits means what calling set() once per edit, in order, means:
// chunks are allocated on first touch in edit order (pool block index =
// allocation count, voxel.zig:47-56), and of several edits of one voxel the
// last wins.  The host resolves that order (chunk allocation, last-writer
// dedup) and the device applies the surviving writes in one kernel that reads
// them from page-locked host memory:
//   brickmap: pool words and new chunk-table entries; the pool grows by
//             doubling like GpuBlockAllocator.alloc (gpu_block_allocator.zig:
//             20-30), new blocks zero;
//   dense:    Morton-ordered bytes, then the occupancy words of every touched
//             4^3 brick (one wave per brick: ballot over its 64 bytes) and
//             of every touched 16^3 region (ballot over its 64 brick words),
//             then the compact albedo index, when built, is recomputed in
//             place (its numbering changes with the occupancy).
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <new>
#include <unordered_map>
#include <vector>

#include "vt_internal.hpp"

namespace vt {

// The edits of a brickmap world.  data: n records (pool block, value, voxel's
// Morton code), then m records (chunk, its new entry).  The code's low 9 bits
// place the voxel in its pool block; a pool can hold more than 2^32 words.
__global__ __launch_bounds__(256) void k_edit_brickmap(uint32_t* __restrict__ pool,
                                                       uint8_t* __restrict__ occ,
                                                       uint32_t* __restrict__ chunks,
                                                       const uint32_t* __restrict__ data,
                                                       uint32_t n, uint32_t m,
                                                       uint32_t* __restrict__ changed) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < kChangedWords && changed) changed[i] = 0u;  // for the kernels that follow
  if (i < n) {
    const uint3 r = reinterpret_cast<const uint3*>(data)[i];
    pool[(size_t)r.x * 512u + (compact1by2(r.z) & 7u) + 8u * (compact1by2(r.z >> 1) & 7u) +
         64u * (compact1by2(r.z >> 2) & 7u)] = r.y;
    if (occ) occ[r.z] = r.y != 0u ? 1 : 0;
  }
  if (i < m) {
    const uint32_t* c = data + 3u * (size_t)n + 2u * (size_t)i;
    chunks[c[0]] = c[1];
  }
}

// The clearance map's byte of brick b (null: a world without the map), from
// its occupancy word; when it is another one, marks the brick's layer of cells
// and the one it faces (of two bricks a cell has along z).
__device__ __forceinline__ void put_sub(uint8_t* sub, uint32_t b, uint64_t word,
                                        uint32_t* changed) {
  if (!sub) return;
  const uint8_t v = (uint8_t)nonzero_bytes(word);
  if (sub[b] != v) {
    sub[b] = v;
    const uint32_t bz = compact1by2(b >> 2), z = bz >> 1, to = (bz & 1u) ? z + 1u : z - 1u;
    atomicOr(&changed[1u + (z >> 5)], 1u << (z & 31u));
    if (to < 128u) atomicOr(&changed[1u + (to >> 5)], 1u << (to & 31u));
  }
}

// The brick bits of the listed 4^3 bricks, from their 64 occupancy bytes
// (one wave per brick; several bricks of a word: atomics on its bits), and
// their sub-block bits.  Sets changed[0] when a word (a 16^3 region) stops
// or starts being zero.  A brick may be listed several times: its waves write
// the same bits.
__global__ __launch_bounds__(256) void k_edit_bricks(const uint8_t* __restrict__ occ,
                                                     const uint32_t* __restrict__ bricks,
                                                     uint32_t n,
                                                     unsigned long long* __restrict__ bits,
                                                     uint8_t* __restrict__ sub,
                                                     uint32_t* __restrict__ changed) {
  const uint32_t wave = (blockIdx.x * 256u + threadIdx.x) >> 6, lane = threadIdx.x & 63u;
  if (wave >= n) return;  // whole waves leave together
  const uint32_t b = bricks[wave];
  const uint64_t m = __ballot(occ[(size_t)b * 64u + lane] != 0);
  if (lane != 0u) return;
  put_sub(sub, b, m, changed);
  const unsigned long long bit = 1ull << (b & 63u);
  if (m) {
    if (atomicOr(bits + (b >> 6), bit) == 0ull) changed[0] = 1u;
  } else {
    const unsigned long long old = atomicAnd(bits + (b >> 6), ~bit);
    if (old != 0ull && (old & ~bit) == 0ull) changed[0] = 1u;
  }
}

// Undoes new chunk entries: data holds m records (chunk, entry).
__global__ __launch_bounds__(256) void k_unset_chunks(uint32_t* __restrict__ chunks,
                                                      const uint32_t* __restrict__ data,
                                                      uint32_t m) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < m) chunks[data[2u * (size_t)i]] = 0u;
}

// The edits of a dense world: n records (Morton code, material).
__global__ __launch_bounds__(256) void k_edit_dense(uint8_t* __restrict__ vox,
                                                    const uint32_t* __restrict__ data,
                                                    uint32_t n, uint32_t* __restrict__ changed) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < kChangedWords) changed[i] = 0u;  // for the kernels that follow
  if (i < n) vox[data[2u * (size_t)i]] = (uint8_t)data[2u * (size_t)i + 1u];
}

// The L0 words of the listed 4^3 bricks (one wave per word: ballot over its
// 64 bytes; no list: of the first n) and their sub-block bits.
__global__ __launch_bounds__(256) void k_edit_l0(const uint8_t* __restrict__ vox,
                                                 uint64_t* __restrict__ l0,
                                                 const uint32_t* __restrict__ bricks, uint32_t n,
                                                 uint8_t* __restrict__ sub,
                                                 uint32_t* __restrict__ changed) {
  const uint32_t wave = (blockIdx.x * 256u + threadIdx.x) >> 6, lane = threadIdx.x & 63u;
  if (wave >= n) return;  // whole waves leave together
  const uint32_t b = bricks ? bricks[wave] : wave;
  const uint64_t m = __ballot(vox[(size_t)b * 64u + lane] != 0);
  if (lane == 0) {
    l0[b] = m;
    put_sub(sub, b, m, changed);
  }
}

// The L1 words of the listed 16^3 regions (no list: of the first n), one wave
// per word: bit l = (l0[region * 64 + l] != 0).  Sets changed[0] when a word
// stops or starts being zero.
__global__ __launch_bounds__(256) void k_edit_l1(const uint64_t* __restrict__ l0,
                                                 uint64_t* __restrict__ l1,
                                                 const uint32_t* __restrict__ regions, uint32_t n,
                                                 uint32_t* __restrict__ changed) {
  const uint32_t wave = (blockIdx.x * 256u + threadIdx.x) >> 6, lane = threadIdx.x & 63u;
  if (wave >= n) return;  // whole waves leave together
  const uint32_t r = regions ? regions[wave] : wave;
  const uint64_t m = __ballot(l0[(size_t)r * 64u + lane] != 0ull);
  if (lane == 0) {
    if ((l1[r] == 0ull) != (m == 0ull)) changed[0] = 1u;
    l1[r] = m;
  }
}

__global__ void k_gather_dense(const DenseWorld w, const uint32_t* __restrict__ xyz, uint32_t n,
                               uint32_t* __restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] = w.vox[morton3(xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2])];
}

__global__ void k_gather_brickmap(const BrickmapWorld w, const uint32_t* __restrict__ xyz,
                                  uint32_t n, uint32_t* __restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] = bm_block(w, (int)xyz[3 * i], (int)xyz[3 * i + 1], (int)xyz[3 * i + 2]);
}

// terrain_edit.comp.glsl:11-17: rayUV = 0, then the primary ray's
// normalize(C_view * vec4(rayUV, 1, 1)).xyz (4 components), AABB entry and
// EPSILON offset.
__device__ __forceinline__ void centre_ray(const ViewConsts& v, uint32_t dim, float e[3],
                                           float d[3]) {
  float r[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    float s = v.view[i] * 0.0f;
    s = s + v.view[4 + i] * 0.0f;
    s = s + v.view[8 + i] * 1.0f;
    s = s + v.view[12 + i] * 1.0f;
    r[i] = s;
  }
  float q = r[0] * r[0];
  q = q + r[1] * r[1];
  q = q + r[2] * r[2];
  q = q + r[3] * r[3];
  const float len = sqrtf(q);
  d[0] = r[0] / len;
  d[1] = r[1] / len;
  d[2] = r[2] / len;
  float tn, tf;
  const float D = (float)dim;
  intersect_aabb(v.pos[0], v.pos[1], v.pos[2], d[0], d[1], d[2], 0.0f, 0.0f, 0.0f, D, D, D, tn,
                 tf);
  const float tc = fmaxf(tn, 0.0f);
#pragma unroll
  for (int i = 0; i < 3; i++) e[i] = (v.pos[i] + d[i] * tc) - 0.001f;
}

// HitInfo of the pick (map.glsl:127 on a hit, :167 on a miss) and the cells
// of the shader's disabled edit body (terrain_edit.comp.glsl:21,23).
__device__ __forceinline__ vt_pick_result pick_result(bool hit, uint32_t data, int face,
                                                      float hx, float hy, float hz, int steps) {
  vt_pick_result res = {};
  res.steps = (uint32_t)steps;
  if (hit) {
    res.data = data;
    res.face = (uint32_t)face;
    res.hit_pos[0] = hx;
    res.hit_pos[1] = hy;
    res.hit_pos[2] = hz;
    face_normal(face, res.normal[0], res.normal[1], res.normal[2]);
  } else {
    res.hit_pos[0] = res.hit_pos[1] = res.hit_pos[2] = -1.0f;
  }
  for (int i = 0; i < 3; i++) {
    res.place[i] = f2i_sat(res.hit_pos[i] + res.normal[i]) >> 3;
    res.remove[i] = f2i_sat(res.hit_pos[i]) >> 3;
  }
  return res;
}

__global__ void k_pick_dense(const DenseWorld w, ViewConsts v, int max_steps,
                             vt_pick_result* __restrict__ out) {
  if (threadIdx.x != 0) return;
  float e[3], d[3];
  centre_ray(v, w.dim, e, d);
  DenseRay ray;
  FlatLookup lk;
  DenseHit h;
  uint32_t l1f = 0, l0f = 0, leaf = 0;
  if (!dense_begin<false>(ray, lk, w, e[0], e[1], e[2], d[0], d[1], d[2], max_steps, h, l1f, l0f))
    dense_run<false>(ray, lk, w, h, l1f, l0f);
  const uint32_t data = h.hit ? w.palette[lk.material(w, h.code, h.v, leaf)] : 0u;
  *out = pick_result(h.hit, data, h.face, h.hx, h.hy, h.hz, h.steps);
}

__global__ void k_pick_brickmap(const BrickmapWorld w, ViewConsts v, int max_steps,
                                vt_pick_result* __restrict__ out) {
  if (threadIdx.x != 0) return;
  float e[3], d[3];
  centre_ray(v, w.dim, e, d);
  // one lane: bound by the latency of its lookups, so the empty blocks go
  // through the loop that keeps several in flight (same steps, same count)
  GeneralHit g;
  if (w.occ) {
    const float inv[3] = {1.0f / (d[0] == 0.0f ? 0.001f : d[0]),
                          1.0f / (d[1] == 0.0f ? 0.001f : d[1]),
                          1.0f / (d[2] == 0.0f ? 0.001f : d[2])};
    trace_brickmap_fast<false, false>(w, e[0], e[1], e[2], d[0], d[1], d[2], inv, max_steps, g);
  } else {
    uint32_t chunk_reads = 0, pool_reads = 0;
    trace_general<false>(w, e[0], e[1], e[2], d[0], d[1], d[2], max_steps, g, chunk_reads,
                         pool_reads);
  }
  *out = pick_result(g.data != 0u, g.data, g.face, g.hx, g.hy, g.hz, g.steps);
}

// Grows the block pool to at least `blocks` blocks (doubling), keeping the
// contents and zeroing the new blocks.
int grow_pool(vt_world* w, uint64_t blocks, hipStream_t s, const char* who) {
  const uint64_t cap = w->pool_capacity / 512u;
  if (blocks <= cap) return VT_OK;
  uint64_t ncap = cap ? cap : 1;
  while (ncap < blocks) ncap *= 2;
  // An optional budget for the block pool (bytes): a growth past it fails
  // like a failed allocation, before anything changes.
  if (const char* lim = std::getenv("VT_POOL_LIMIT_BYTES")) {
    const unsigned long long limit = std::strtoull(lim, nullptr, 10);
    if (limit && ncap * 512u * 4u > limit)
      return fail(VT_ERR_OUT_OF_MEMORY, "%s: the pool would grow to %llu bytes, past "
                  "VT_POOL_LIMIT_BYTES=%llu", who, (unsigned long long)(ncap * 512u * 4u), limit);
  }
  uint32_t* np = nullptr;
  hipError_t e = hipMalloc((void**)&np, ncap * 512u * 4u);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return hip_fail(e, who);
  }
  e = hipMemcpyAsync(np, w->pool, cap * 512u * 4u, hipMemcpyDeviceToDevice, s);
  if (e == hipSuccess) e = hipMemsetAsync(np + cap * 512u, 0, (ncap - cap) * 512u * 4u, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    dev_free(np);
    return hip_fail(e, who);
  }
  dev_free(w->pool);
  w->pool = np;
  w->bytes += (ncap - cap) * 512u * 4u;
  w->pool_capacity = ncap * 512u;
  return VT_OK;
}

}  // namespace vt

namespace {

using vt::fail;
using vt::hip_fail;

// The words of one call's lists where the device can read them: the
// context's staging, or device memory for the call when they are more.
// The destructor waits for the stream: the next call may use the staging.
struct Lists {
  vt_ctx* ctx;
  hipStream_t s;
  uint32_t* own = nullptr;
  const uint32_t* dev = nullptr;
  Lists(vt_ctx* c, hipStream_t st) : ctx(c), s(st) {}
  ~Lists() {
    if (dev) (void)hipStreamSynchronize(s);
    vt::dev_free(own);
  }
  hipError_t put(const std::vector<uint32_t>& words) {
    const size_t bytes = words.size() * 4u;
    if (bytes <= kCtxStageBytes) {
      std::memcpy(ctx->stage, words.data(), bytes);
      dev = (const uint32_t*)ctx->stage_dev;
      return hipSuccess;
    }
    hipError_t e = hipMalloc((void**)&own, bytes);
    if (e != hipSuccess) return e;
    e = hipMemcpyAsync(own, words.data(), bytes, hipMemcpyHostToDevice, s);
    dev = own;
    return e;
  }
};

// Sorted, each value once.
void sort_unique(std::vector<uint32_t>& v) {
  std::sort(v.begin(), v.end());
  v.erase(std::unique(v.begin(), v.end()), v.end());
}

uint32_t part1by2_host(uint32_t v) {
  v &= 0x3FFu;
  v = (v | (v << 16)) & 0xFF0000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  return (v | (v << 2)) & 0x09249249u;
}

uint32_t morton_code(uint32_t x, uint32_t y, uint32_t z) {
  return part1by2_host(x) | (part1by2_host(y) << 1) | (part1by2_host(z) << 2);
}

uint32_t blocks_for(uint64_t n, uint32_t per_block) {
  return (uint32_t)((n + per_block - 1) / per_block);
}

int check_coords(const vt_world* w, const uint32_t* xyz, uint32_t n, const char* who) {
  for (uint32_t i = 0; i < n; i++)
    for (int k = 0; k < 3; k++)
      if (xyz[3 * (size_t)i + k] >= w->dim)
        return fail(VT_ERR_INVALID_ARGUMENT, "%s: voxel %u coordinate %u outside [0, %u)", who, i,
                    xyz[3 * (size_t)i + k], w->dim);
  return VT_OK;
}

// The box of the nonempty voxels grows with every voxel set nonzero (a
// cleared voxel leaves it as it was: still a box around all of them).
static void grow_box_by(vt_world* w, const uint32_t* xyz, const uint32_t* values, uint32_t n) {
  for (uint32_t i = 0; i < n; i++)
    if (values[i] != 0u)
      vt::grow_box(w, (int32_t)xyz[3 * (size_t)i], (int32_t)xyz[3 * (size_t)i + 1],
                   (int32_t)xyz[3 * (size_t)i + 2]);
}

int set_brickmap(vt_world* w, const uint32_t* xyz, const uint32_t* values, uint32_t n,
                 hipStream_t s) {
  const uint32_t M = w->dim / 8u;
  std::unordered_map<uint64_t, uint32_t> last;  // pool word -> its record
  // chunks this call allocates: kept here and entered into the host chunk
  // table only once the device holds them, so a failed call leaves the
  // world as it was
  std::unordered_map<uint64_t, uint32_t> fresh;
  std::vector<uint32_t> words;  // records (pool block, value, Morton code), see k_edit_brickmap
  std::vector<uint32_t> chunks, bricks;
  uint64_t used = w->pool_words / 512u;
  last.reserve(n);
  words.reserve(3 * (size_t)n);
  for (uint32_t i = 0; i < n; i++) {
    const uint32_t x = xyz[3 * (size_t)i], y = xyz[3 * (size_t)i + 1], z = xyz[3 * (size_t)i + 2];
    const uint64_t ci = (uint64_t)(x / 8u) + M * ((uint64_t)(y / 8u) + (uint64_t)M * (z / 8u));
    uint32_t entry = w->chunk_mirror[ci];
    if (entry == 0) {
      auto f = fresh.find(ci);
      if (f != fresh.end()) {
        entry = f->second;
      } else {  // get_block_for_chunk: allocate on first touch
        // (after the blocks of the pool the world was made with, however many)
        if (used >= 0xFFFFFFFEull) return fail(VT_ERR_OUT_OF_MEMORY, "vt_world_set_voxels: pool");
        entry = (uint32_t)(++used);
        fresh.emplace(ci, entry);
        chunks.push_back((uint32_t)ci);
        chunks.push_back(entry);
      }
    }
    const uint64_t a = (uint64_t)(entry - 1u) * 512u + (x % 8u) + 8u * ((y % 8u) + 8u * (z % 8u));
    const uint32_t code = morton_code(x, y, z);
    auto it = last.find(a);
    if (it == last.end()) {
      last.emplace(a, (uint32_t)(words.size() / 3u));
      words.insert(words.end(), {entry - 1u, values[i], code});
      // (rows of voxels: neighbours share their brick)
      if (bricks.empty() || bricks.back() != code >> 6) bricks.push_back(code >> 6);
    } else {
      words[3 * (size_t)it->second + 1] = values[i];
    }
  }
  int st = vt::grow_pool(w, used, s, "vt_world_set_voxels: pool growth");
  if (st != VT_OK) return st;  // nothing written: the world is unchanged
  // (bricks may hold one more than once: sorting them took the host as long as
  // all the rest of a large call, 16,384 edits 1430 us against 920)
  const uint32_t nw = (uint32_t)(words.size() / 3u), nc = (uint32_t)(chunks.size() / 2u),
                 nb = (uint32_t)bricks.size();
  words.insert(words.end(), chunks.begin(), chunks.end());
  words.insert(words.end(), bricks.begin(), bricks.end());
  Lists lists(w->ctx, s);
  VT_HIP(lists.put(words));
  const uint32_t* d_chunks = lists.dev + 3 * (size_t)nw;
  const bool current = vt::begin_occupancy_change(w);
  hipLaunchKernelGGL(vt::k_edit_brickmap, dim3(blocks_for(std::max(nw, nc), 256)), dim3(256), 0, s,
                     w->pool, w->occ, w->chunks, lists.dev, nw, nc, vt::maps_changed(w));
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && w->occ) {
    if (current) {
      hipLaunchKernelGGL(vt::k_edit_bricks, dim3(blocks_for(nb, 4)), dim3(256), 0, s, w->occ,
                         d_chunks + 2 * (size_t)nc, nb, (unsigned long long*)w->brick_bits,
                         w->clear_tmp, vt::maps_changed(w));
      e = hipGetLastError();
    } else {  // an earlier change failed midway: everything from the pool
      e = vt::launch_build_occupancy(vt::brickmap_view(w), w->occ, w->brick_bits, w->clear_tmp, s);
    }
    if (e == hipSuccess) e = vt::rebuild_maps(w, s, current ? vt::maps_changed(w) : nullptr);
  }
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    // Undo what may have reached the device: new chunk entries back to 0
    // and the new blocks zero again (edits allocate zero blocks), so the
    // device agrees with the unchanged host chunk table and pool count.  The
    // occupancy bytes may stay set where the pool is zero again (a lookup
    // then reads the empty block) until the next change makes them anew.
    if (nc)
      hipLaunchKernelGGL(vt::k_unset_chunks, dim3(blocks_for(nc, 256)), dim3(256), 0, s, w->chunks,
                         d_chunks, nc);
    const uint64_t b0 = w->pool_words / 512u;
    if (used > b0)
      (void)hipMemsetAsync(w->pool + b0 * 512u, 0, (used - b0) * 512u * 4u, s);
    (void)hipStreamSynchronize(s);
    (void)hipGetLastError();
    return hip_fail(e, "vt_world_set_voxels: scatter");
  }
  for (uint32_t k = 0; k < nc; k++) w->chunk_mirror[chunks[2 * k]] = chunks[2 * k + 1];
  w->pool_words = used * 512u;
  if (w->occ) vt::finish_maps(w);
  return VT_OK;
}

int set_dense(vt_world* w, const uint32_t* xyz, const uint32_t* values, uint32_t n,
              hipStream_t s) {
  for (uint32_t i = 0; i < n; i++)
    if (values[i] > 255u)
      return fail(VT_ERR_INVALID_ARGUMENT, "vt_world_set_voxels: dense value %u > 255 (edit %u)",
                  values[i], i);
  std::unordered_map<uint64_t, uint32_t> last;
  std::vector<uint32_t> words, bricks, regions, regions8;
  last.reserve(n);
  words.reserve(2 * (size_t)n);
  grow_box_by(w, xyz, values, n);
  for (uint32_t i = 0; i < n; i++) {
    const uint32_t code =
        morton_code(xyz[3 * (size_t)i], xyz[3 * (size_t)i + 1], xyz[3 * (size_t)i + 2]);
    auto it = last.find(code);
    if (it == last.end()) {
      last.emplace(code, (uint32_t)(words.size() / 2u));
      words.insert(words.end(), {code, values[i]});
      bricks.push_back(code >> 6);
    } else {
      words[2 * (size_t)it->second + 1] = values[i];
    }
  }
  sort_unique(bricks);
  for (const uint32_t b : bricks) {  // sorted, so equal neighbours only
    if (regions.empty() || regions.back() != b >> 6) regions.push_back(b >> 6);
    if (regions8.empty() || regions8.back() != b >> 9) regions8.push_back(b >> 9);
  }
  const uint64_t nwords = (uint64_t)w->dim * w->dim * w->dim / 64u;
  const uint32_t nw = (uint32_t)(words.size() / 2u), nb = (uint32_t)bricks.size(),
                 nr = (uint32_t)regions.size(), nr8 = (uint32_t)regions8.size();
  words.insert(words.end(), bricks.begin(), bricks.end());
  words.insert(words.end(), regions.begin(), regions.end());
  words.insert(words.end(), regions8.begin(), regions8.end());
  Lists lists(w->ctx, s);
  VT_HIP(lists.put(words));
  const uint32_t* d_bricks = lists.dev + 2 * (size_t)nw;
  const bool current = vt::begin_occupancy_change(w);
  hipLaunchKernelGGL(vt::k_edit_dense, dim3(blocks_for(nw, 256)), dim3(256), 0, s, w->vox,
                     lists.dev, nw, vt::maps_changed(w));
  if (current) {
    hipLaunchKernelGGL(vt::k_edit_l0, dim3(blocks_for(nb, 4)), dim3(256), 0, s, w->vox, w->l0,
                       d_bricks, nb, w->clear_tmp, vt::maps_changed(w));
    hipLaunchKernelGGL(vt::k_edit_l1, dim3(blocks_for(nr, 4)), dim3(256), 0, s, w->l0, w->l1,
                       d_bricks + nb, nr, vt::maps_changed(w));
    VT_HIP(hipGetLastError());
    VT_HIP(vt::launch_build_l1b(w->l0, nwords, d_bricks + nb + nr, nr8, w->l1b, s));
  } else {  // an earlier change failed midway: every level from the voxels
    const uint32_t n0 = (uint32_t)nwords, n1 = (uint32_t)(nwords / 64u);
    hipLaunchKernelGGL(vt::k_edit_l0, dim3(blocks_for(n0, 4)), dim3(256), 0, s, w->vox, w->l0,
                       nullptr, n0, w->clear_tmp, vt::maps_changed(w));
    hipLaunchKernelGGL(vt::k_edit_l1, dim3(blocks_for(n1, 4)), dim3(256), 0, s, w->l0, w->l1,
                       nullptr, n1, vt::maps_changed(w));
    VT_HIP(hipGetLastError());
    VT_HIP(vt::launch_build_l1b(w->l0, nwords, nullptr, (uint32_t)vt::l1b_words(w->dim), w->l1b,
                                s));
  }
  VT_HIP(vt::rebuild_maps(w, s, current ? vt::maps_changed(w) : nullptr));
  if (w->prefix) {  // keep the compact index current
    const uint64_t ntiles = (nwords + 1023) / 1024;
    uint32_t* scratch = nullptr;
    VT_HIP(hipMalloc((void**)&scratch, (ntiles + 1) * 4));
    hipError_t e = vt::launch_compact_prefix(w->l0, nwords, w->prefix, scratch, s);
    uint32_t total = 0;
    if (e == hipSuccess)
      e = hipMemcpyAsync(&total, scratch + ntiles, 4, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    vt::dev_free(scratch);
    VT_HIP(e);
    w->n_occupied = total;
  }
  VT_HIP(hipStreamSynchronize(s));
  vt::finish_maps(w);
  return VT_OK;
}

}  // namespace

extern "C" {

int vt_world_set_voxels(vt_ctx* ctx, vt_world* world, const uint32_t* xyz,
                        const uint32_t* values, uint32_t n, void* stream) {
  if (!ctx || !world || (n && (!xyz || !values)))
    return fail(VT_ERR_NULL_POINTER, "vt_world_set_voxels: null argument");
  if (world->ctx != ctx) return fail(VT_ERR_WRONG_CONTEXT, "vt_world_set_voxels");
  int st = check_coords(world, xyz, n, "vt_world_set_voxels");
  if (st != VT_OK || n == 0) return st;
  VT_HIP(hipSetDevice(ctx->device));
  const hipStream_t s = (hipStream_t)stream;
  try {
    return world->kind == WorldKind::Dense ? set_dense(world, xyz, values, n, s)
                                           : set_brickmap(world, xyz, values, n, s);
  } catch (const std::bad_alloc&) {  // the host lists; nothing written yet
    return fail(VT_ERR_OUT_OF_MEMORY, "vt_world_set_voxels: host lists of %u edits", n);
  }
}

int vt_world_get_voxels(vt_ctx* ctx, const vt_world* world, const uint32_t* xyz, uint32_t n,
                        uint32_t* values, void* stream) {
  if (!ctx || !world || (n && (!xyz || !values)))
    return fail(VT_ERR_NULL_POINTER, "vt_world_get_voxels: null argument");
  if (world->ctx != ctx) return fail(VT_ERR_WRONG_CONTEXT, "vt_world_get_voxels");
  int st = check_coords(world, xyz, n, "vt_world_get_voxels");
  if (st != VT_OK || n == 0) return st;
  VT_HIP(hipSetDevice(ctx->device));
  const hipStream_t s = (hipStream_t)stream;
  // the context's staging: coordinates, then values, kCtxStageVoxels at a
  // time, read and written in place by the kernel
  char* host = (char*)ctx->stage;
  uint32_t* d_xyz = (uint32_t*)ctx->stage_dev;
  for (uint32_t i0 = 0; i0 < n; i0 += kCtxStageVoxels) {
    const uint32_t m = std::min(n - i0, kCtxStageVoxels);
    std::memcpy(host, xyz + 3 * (size_t)i0, 12 * (size_t)m);
    uint32_t* d_out = d_xyz + 3 * (size_t)m;
    if (world->kind == WorldKind::Dense)
      hipLaunchKernelGGL(vt::k_gather_dense, dim3(blocks_for(m, 256)), dim3(256), 0, s,
                         vt::dense_view(world), d_xyz, m, d_out);
    else
      hipLaunchKernelGGL(vt::k_gather_brickmap, dim3(blocks_for(m, 256)), dim3(256), 0, s,
                         vt::brickmap_view(world), d_xyz, m, d_out);
    VT_HIP(hipGetLastError());
    VT_HIP(hipStreamSynchronize(s));
    std::memcpy(values + i0, host + 12 * (size_t)m, 4 * (size_t)m);
  }
  return VT_OK;
}

int vt_world_read_brickmap(vt_ctx* ctx, const vt_world* world, uint32_t* chunks,
                           uint32_t* pool, size_t pool_capacity_words, size_t* pool_words,
                           void* stream) {
  if (!ctx || !world || !pool_words)
    return fail(VT_ERR_NULL_POINTER, "vt_world_read_brickmap: null argument");
  if (world->ctx != ctx) return fail(VT_ERR_WRONG_CONTEXT, "vt_world_read_brickmap");
  if (world->kind != WorldKind::Brickmap)
    return fail(VT_ERR_INVALID_ARGUMENT, "vt_world_read_brickmap: needs a brickmap world");
  *pool_words = world->pool_words;
  if (pool && pool_capacity_words < world->pool_words)
    return fail(VT_ERR_INVALID_ARGUMENT,
                "vt_world_read_brickmap: pool holds %zu words, the output room is %zu",
                world->pool_words, pool_capacity_words);
  VT_HIP(hipSetDevice(ctx->device));
  const hipStream_t s = (hipStream_t)stream;
  const size_t M = world->dim / 8u;
  if (chunks)
    VT_HIP(hipMemcpyAsync(chunks, world->chunks, M * M * M * 4, hipMemcpyDeviceToHost, s));
  if (pool && world->pool_words)
    VT_HIP(hipMemcpyAsync(pool, world->pool, world->pool_words * 4, hipMemcpyDeviceToHost, s));
  VT_HIP(hipStreamSynchronize(s));
  return VT_OK;
}

int vt_world_read_free_map(vt_ctx* ctx, const vt_world* world, uint32_t* words,
                           size_t capacity_words, uint32_t* words_per_octant, int* valid,
                           void* stream) {
  if (!ctx || !world || !words_per_octant || !valid)
    return fail(VT_ERR_NULL_POINTER, "vt_world_read_free_map: null argument");
  if (world->ctx != ctx) return fail(VT_ERR_WRONG_CONTEXT, "vt_world_read_free_map");
  const uint32_t wpo = vt::free_words_per_octant(world->dim);
  *words_per_octant = wpo;
  *valid = world->freemap && world->maps_valid ? 1 : 0;
  if (!words || !world->freemap) return VT_OK;
  if (capacity_words < 8u * (size_t)wpo)
    return fail(VT_ERR_INVALID_ARGUMENT,
                "vt_world_read_free_map: the map holds %u words, the output room is %zu",
                8u * wpo, capacity_words);
  VT_HIP(hipSetDevice(ctx->device));
  const hipStream_t s = (hipStream_t)stream;
  VT_HIP(hipMemcpyAsync(words, world->freemap, 8u * (size_t)wpo * 4u, hipMemcpyDeviceToHost, s));
  VT_HIP(hipStreamSynchronize(s));
  return VT_OK;
}

int vt_pick(vt_ctx* ctx, const vt_world* world, const vt_camera* camera, int32_t max_steps,
            vt_pick_result* result, void* stream) {
  if (!ctx || !world || !camera || !result)
    return fail(VT_ERR_NULL_POINTER, "vt_pick: null argument");
  if (world->ctx != ctx) return fail(VT_ERR_WRONG_CONTEXT, "vt_pick");
  if (max_steps < 0 || max_steps > 65535)
    return fail(VT_ERR_INVALID_ARGUMENT, "vt_pick: max_steps %d outside [0, 65535]", max_steps);
  VT_HIP(hipSetDevice(ctx->device));
  const hipStream_t s = (hipStream_t)stream;
  const vt::ViewConsts v = vt::view_consts(camera, 1, 1);
  vt_pick_result* d = (vt_pick_result*)ctx->stage_dev;  // the context's staging
  if (world->kind == WorldKind::Dense) {
    vt::DenseWorld dw = vt::dense_view(world);
    dw.clear_bytes = 0;  // the result reports traceMap's step count
    hipLaunchKernelGGL(vt::k_pick_dense, dim3(1), dim3(64), 0, s, dw, v, (int)max_steps, d);
  } else {
    vt::BrickmapWorld bw = vt::brickmap_view(world);
    if (bw.dim < 2u * (uint32_t)vt::kSkipLong) bw.occ = nullptr;  // as launch_render_brickmap
    hipLaunchKernelGGL(vt::k_pick_brickmap, dim3(1), dim3(64), 0, s, bw, v, (int)max_steps, d);
  }
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return hip_fail(e, "vt_pick");
  std::memcpy(result, ctx->stage, sizeof *result);
  return VT_OK;
}

}  // extern "C"
