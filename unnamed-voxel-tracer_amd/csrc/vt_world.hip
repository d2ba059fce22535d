// vt_world.hip -- device-side construction of dense world layouts.
//
// The caller hands over a linear uint8 grid (x fastest).  On the device it is
// re-laid in Morton order (voxel (x,y,z) at interleave(x,y,z)), and the
// occupancy levels are built from it: L0 = one uint64 per 64 consecutive
// codes (a 4^3 brick, bit = code & 63), L1 = one uint64 per 4096 codes (a
// 16^3 region, bit = brick index & 63 set when the brick has a solid voxel),
// L1b = one uint64 per 32768 codes (a 32^3 region, bit per 8^3 brick).
#include <algorithm>

#include "vt_internal.hpp"

namespace vt {

// The 64 Morton bytes of a 4^3 brick from its 16 rows of 4 voxels (row
// [4 z + y], x in the byte order).  Byte code bits are x0 y0 z0 x1 y1 z1, so
// the 32-bit word (z0, x1, y1, z1) takes two half words of rows 2 y1 and
// 2 y1 + 1 of layer 2 z1 + z0.  Returns the brick's occupancy word.
__device__ __forceinline__ uint64_t morton_brick(const uint32_t row[16], uint32_t out[16]) {
  uint64_t mask = 0;
#pragma unroll
  for (uint32_t w = 0; w < 16u; w++) {
    const uint32_t z = (w & 1u) | ((w >> 3) << 1), x1 = (w >> 1) & 1u, y1 = (w >> 2) & 1u;
    const uint32_t a = row[4u * z + 2u * y1], b = row[4u * z + 2u * y1 + 1u];
    const uint32_t v = x1 ? (a >> 16) | (b & 0xFFFF0000u) : (a & 0xFFFFu) | (b << 16);
    out[w] = v;
    uint32_t y = v | (v >> 4);  // bit k = byte k is nonzero
    y |= y >> 2;
    y |= y >> 1;
    y &= 0x01010101u;
    mask |= (uint64_t)((y | (y >> 7) | (y >> 14) | (y >> 21)) & 15u) << (4u * w);
  }
  return mask;
}

// One thread per 4^3 brick: 16 rows of 4 voxels in (a wave's rows are
// contiguous along x), 64 Morton bytes and the L0 word out (two bricks a
// 128-byte line).  Bound by HBM: 2 bytes a voxel and 1/8 byte of L0.  512^3:
// 262 us as one thread per 4 codes (4-byte gathers of bytes) with a second
// pass for L0, 64 us here.
__global__ __launch_bounds__(256) void k_build_bricks(const uint8_t* __restrict__ lin,
                                                      uint32_t log2n, uint8_t* __restrict__ vox,
                                                      uint64_t* __restrict__ l0,
                                                      uint8_t* __restrict__ sub) {
  const uint32_t n = 1u << log2n;  // bricks per axis
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= 1u << (3u * log2n)) return;
  const uint32_t bx = i & (n - 1u), by = (i >> log2n) & (n - 1u), bz = i >> (2u * log2n);
  const size_t dim = 4u * (size_t)n;
  const uint8_t* src = lin + 4u * bx + dim * (4u * by + dim * (4u * (size_t)bz));
  uint32_t row[16], out[16];
#pragma unroll
  for (uint32_t k = 0; k < 16u; k++)
    row[k] = *reinterpret_cast<const uint32_t*>(src + dim * ((k & 3u) + dim * (k >> 2)));
  const uint64_t mask = morton_brick(row, out);
  const uint32_t c = morton3(bx, by, bz);
  uint4* dst = reinterpret_cast<uint4*>(vox + 64u * (size_t)c);
#pragma unroll
  for (uint32_t q = 0; q < 4u; q++)
    dst[q] = make_uint4(out[4 * q], out[4 * q + 1], out[4 * q + 2], out[4 * q + 3]);
  l0[c] = mask;
  if (sub) sub[c] = (uint8_t)nonzero_bytes(mask);
}

// The box of the nonempty voxels from the L0 words: grid-stride, a sum over
// the block first, so that the atomics on box6 (lo, then hi) stay few.
__global__ __launch_bounds__(256) void k_box(const uint64_t* __restrict__ l0, uint32_t nwords,
                                             int32_t* __restrict__ box6) {
  // bits of a word whose voxel has x / y / z = k (x in code bits 0 and 3)
  constexpr uint64_t X0 = 0x0055005500550055ull, Y0 = 0x0000333300003333ull,
                     Z0 = 0x000000000F0F0F0Full;
  constexpr uint64_t at[3][4] = {{X0, X0 << 1, X0 << 8, X0 << 9},
                                 {Y0, Y0 << 2, Y0 << 16, Y0 << 18},
                                 {Z0, Z0 << 4, Z0 << 32, Z0 << 36}};
  int lo[3] = {1 << 20, 1 << 20, 1 << 20}, hi[3] = {-1, -1, -1};
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < nwords; i += gridDim.x * 256u) {
    const uint64_t w = l0[i];
    if (w == 0ull) continue;
    const int base[3] = {4 * (int)compact1by2(i), 4 * (int)compact1by2(i >> 1),
                         4 * (int)compact1by2(i >> 2)};
#pragma unroll
    for (int a = 0; a < 3; a++) {
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (w & at[a][k]) {
          lo[a] = min(lo[a], base[a] + k);
          hi[a] = max(hi[a], base[a] + k);
        }
    }
  }
  __shared__ int32_t part[6];
  if (threadIdx.x < 6u) part[threadIdx.x] = threadIdx.x < 3u ? 1 << 20 : -1;
  __syncthreads();
#pragma unroll
  for (int a = 0; a < 3; a++) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      lo[a] = min(lo[a], __shfl_xor(lo[a], off, 64));
      hi[a] = max(hi[a], __shfl_xor(hi[a], off, 64));
    }
    if ((threadIdx.x & 63u) == 0u && hi[a] >= 0) {
      atomicMin(&part[a], lo[a]);
      atomicMax(&part[3 + a], hi[a]);
    }
  }
  __syncthreads();
  if (threadIdx.x < 6u && part[3] >= 0) {
    if (threadIdx.x < 3u)
      atomicMin(&box6[threadIdx.x], part[threadIdx.x]);
    else
      atomicMax(&box6[threadIdx.x], part[threadIdx.x]);
  }
}

__global__ void k_box_clear(int32_t* __restrict__ box6) {
  if (threadIdx.x < 6u) box6[threadIdx.x] = threadIdx.x < 3u ? 1 << 20 : -1;
}

__global__ void k_box_report(const int32_t* __restrict__ box6, CtxReport* __restrict__ report) {
  if (threadIdx.x < 3u) {
    report->box_lo[threadIdx.x] = box6[threadIdx.x];
    report->box_hi[threadIdx.x] = box6[3u + threadIdx.x];
  }
}

// One thread per L1 word: 64 consecutive L0 words.
__global__ __launch_bounds__(256) void k_build_l1(const uint64_t* __restrict__ l0, uint64_t nwords,
                                                  uint64_t* __restrict__ l1) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nwords) return;
  uint64_t mask = 0;
  for (uint32_t j = 0; j < 64; j++)
    if (l0[i * 64u + j]) mask |= 1ull << j;
  l1[i] = mask;
}

// The 8^3-brick level: one uint64 per 32^3 region (32768 codes), bit j set
// when 8^3 brick 64 i + j (L0 words 8 (64 i + j) .. + 7) holds a solid
// voxel.  A 16^3 world has one partial word (8 bricks).  One wave per word.
__global__ __launch_bounds__(256) void k_build_l1b(const uint64_t* __restrict__ l0, uint64_t n0,
                                                   const uint32_t* __restrict__ words,
                                                   uint32_t nwords, uint64_t* __restrict__ l1b) {
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t lane = threadIdx.x & 63u;
  if (wave >= nwords) return;  // whole waves leave together
  const uint32_t word = words ? words[wave] : wave;
  const uint64_t first = ((uint64_t)word * 64u + lane) * 8u;
  uint64_t any = 0;
  if (first < n0)
#pragma unroll
    for (uint32_t k = 0; k < 8; k++) any |= l0[first + k];
  const uint64_t m = __ballot(any != 0ull);
  if (lane == 0) l1b[word] = m;
}

hipError_t launch_build_l1b(const uint64_t* l0, uint64_t n0, const uint32_t* words,
                            uint32_t nwords, uint64_t* l1b, hipStream_t stream) {
  if (nwords == 0) return hipSuccess;
  hipLaunchKernelGGL(k_build_l1b, dim3((nwords + 3u) / 4u), dim3(256), 0, stream, l0, n0, words,
                     nwords, l1b);
  return hipGetLastError();
}

// ---- compact albedo index: exclusive prefix sum of popcount(L0 word) ----
// Three passes: per-tile sums (1024 words per 256-thread block), one block
// scanning the tile sums, then each tile scanning its own words.
constexpr uint32_t kScanTile = 1024;

__device__ __forceinline__ uint32_t block_exclusive_scan_256(uint32_t v, uint32_t* sh,
                                                             uint32_t& total) {
  const uint32_t t = threadIdx.x;
  sh[t] = v;
  __syncthreads();
  for (uint32_t off = 1; off < 256; off <<= 1) {
    const uint32_t a = t >= off ? sh[t - off] : 0u;
    __syncthreads();
    sh[t] += a;
    __syncthreads();
  }
  total = sh[255];
  const uint32_t incl = sh[t];
  __syncthreads();
  return incl - v;
}

__global__ __launch_bounds__(256) void k_popc_tile_sums(const uint64_t* __restrict__ l0,
                                                        uint64_t nwords,
                                                        uint32_t* __restrict__ sums) {
  __shared__ uint32_t sh[256];
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + threadIdx.x * 4u;
  uint32_t s = 0;
  for (uint32_t k = 0; k < 4; k++)
    if (base + k < nwords) s += (uint32_t)__popcll(l0[base + k]);
  uint32_t total;
  (void)block_exclusive_scan_256(s, sh, total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(1024) void k_scan_tile_sums(uint32_t* __restrict__ sums,
                                                         uint32_t ntiles,
                                                         uint32_t* __restrict__ total) {
  __shared__ uint32_t buf[1024];
  const uint32_t t = threadIdx.x;
  uint32_t carry = 0;
  for (uint32_t c = 0; c < ntiles; c += 1024u) {
    const uint32_t i = c + t;
    const uint32_t v = i < ntiles ? sums[i] : 0u;
    buf[t] = v;
    __syncthreads();
    for (uint32_t off = 1; off < 1024u; off <<= 1) {
      const uint32_t a = t >= off ? buf[t - off] : 0u;
      __syncthreads();
      buf[t] += a;
      __syncthreads();
    }
    if (i < ntiles) sums[i] = carry + buf[t] - v;
    carry += buf[1023];
    __syncthreads();
  }
  if (t == 0) *total = carry;
}

__global__ __launch_bounds__(256) void k_prefix_words(const uint64_t* __restrict__ l0,
                                                      uint64_t nwords,
                                                      const uint32_t* __restrict__ tile_off,
                                                      uint32_t* __restrict__ prefix) {
  __shared__ uint32_t sh[256];
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + threadIdx.x * 4u;
  uint32_t pc[4], s = 0;
  for (uint32_t k = 0; k < 4; k++) {
    pc[k] = base + k < nwords ? (uint32_t)__popcll(l0[base + k]) : 0u;
    s += pc[k];
  }
  uint32_t total;
  uint32_t run = tile_off[blockIdx.x] + block_exclusive_scan_256(s, sh, total);
  for (uint32_t k = 0; k < 4; k++) {
    if (base + k < nwords) prefix[base + k] = run;
    run += pc[k];
  }
}

hipError_t launch_compact_prefix(const uint64_t* l0, uint64_t nwords, uint32_t* prefix,
                                 uint32_t* scratch, hipStream_t stream) {
  const uint32_t ntiles = (uint32_t)((nwords + kScanTile - 1) / kScanTile);
  hipLaunchKernelGGL(k_popc_tile_sums, dim3(ntiles), dim3(256), 0, stream, l0, nwords, scratch);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_scan_tile_sums, dim3(1), dim3(1024), 0, stream, scratch, ntiles,
                     scratch + ntiles);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_prefix_words, dim3(ntiles), dim3(256), 0, stream, l0, nwords, scratch,
                     prefix);
  return hipGetLastError();
}

hipError_t launch_build_dense(const uint8_t* linear, uint32_t dim, uint8_t* vox, uint64_t* l0,
                              uint64_t* l1, uint64_t* l1b, uint8_t* sub, int32_t* box6,
                              CtxReport* report, hipStream_t stream) {
  const uint64_t n = (uint64_t)dim * dim * dim;  // a power of two >= 4096
  const uint32_t n0 = (uint32_t)(n / 64u), n1 = (uint32_t)(n / 4096u);
  uint32_t log2n = 0;
  while ((4u << log2n) < dim) log2n++;
  hipLaunchKernelGGL(k_build_bricks, dim3((n0 + 255u) / 256u), dim3(256), 0, stream, linear, log2n,
                     vox, l0, sub);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_build_l1, dim3((n1 + 255u) / 256u), dim3(256), 0, stream, l0, (uint64_t)n1,
                     l1);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_box_clear, dim3(1), dim3(64), 0, stream, box6);
  hipLaunchKernelGGL(k_box, dim3(std::min((n0 + 255u) / 256u, 256u)), dim3(256), 0, stream, l0, n0,
                     box6);
  hipLaunchKernelGGL(k_box_report, dim3(1), dim3(64), 0, stream, box6, report);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_build_l1b(l0, n0, nullptr, (uint32_t)l1b_words(dim), l1b, stream);
}

// ---- free-region map: where a ray's remaining path is provably empty ----
// Regions are 16^3 blocks (one L1 word; R = max(dim / 16, 1) per axis).  For
// each of the 8 direction octants o, free_o(r) = no region r' at or ahead of
// r on every axis in o's travel direction (the forward orthant, r itself
// included) holds a nonempty block.  Bit r (region Morton code) of octant
// o's bitmap is free_o(r).  vt_free_map_used decides by its largest share.

// Threads of a block of the maps' first launch.
constexpr uint32_t kMapBlock = 1024;

// One block per octant, the regions as bit rows along x in LDS (R = 1 << lg,
// at most 64 rows of 64 bits a layer, 32 KiB).  A row's bit x becomes the OR
// of the regions at or ahead of x by shifts; along y and z the rows take the
// OR of rows 1, 2, 4, ... ahead.  Then bit j of word w of the octant's bitmap
// = the region with Morton code 32 w + j is free.  Bound by the one CU a block
// has: 14 us at 512^3 (five kernels over byte planes: 36), 49 at 1024^3 (59
// with a word of 8 bytes a region instead of a byte).  An edit rarely
// empties or fills a whole region, so it passes `changed` (device word: a
// region did) and the launch ends at once, in 3 us, when none did.
struct FreeMapArgs {
  const uint64_t* l1b;    // a dense world's 8^3-brick level
  const uint64_t* words;  // else: a word per region
  uint32_t lg, nwords;
  uint32_t* fm;
  const uint32_t* changed;
  CtxReport* report;
};
__device__ __forceinline__ void free_map_block(const FreeMapArgs& a, uint64_t* row,
                                               uint32_t& total) {
  const uint32_t lg = a.lg, words = a.nwords;
  uint32_t* __restrict__ fm = a.fm;
  CtxReport* __restrict__ report = a.report;
  const bool run = !a.changed || *a.changed != 0u;
  if (blockIdx.x == 0u && threadIdx.x == 0u) report->free_built = run ? 1u : 0u;
  if (!run) return;  // the same for every thread
  const uint32_t R = 1u << lg, rows = R << lg, n = rows << lg;
  const uint32_t o = blockIdx.x, t = threadIdx.x;
  if (t == 0u) total = 0u;
  const uint64_t full = R == 64u ? ~0ull : (1ull << R) - 1ull;
  for (uint32_t r = t; r < rows; r += 1024u) row[r] = 0ull;
  __syncthreads();
  // eight consecutive codes (2^3 regions) a thread: two bits of four rows.  A
  // region is a byte of the 8^3-brick level's words (dense worlds) or a word of
  // the brick bits.
  uint32_t* half = reinterpret_cast<uint32_t*>(row);
  for (uint32_t g = t; g < (n >= 8u ? n / 8u : 1u); g += 1024u) {
    uint32_t any = 0u;
    if (a.l1b) {
      any = nonzero_bytes(a.l1b[g]);
    } else if (n >= 8u) {
      const uint4* p = reinterpret_cast<const uint4*>(a.words + 8u * (size_t)g);
#pragma unroll
      for (uint32_t k = 0; k < 4u; k++) {
        const uint4 q = p[k];
        any |= ((q.x | q.y) ? 1u : 0u) << (2u * k) | ((q.z | q.w) ? 2u : 0u) << (2u * k);
      }
    } else {
      any = a.words[0] != 0ull ? 1u : 0u;  // R = 1
    }
    if (any == 0u) continue;
    const uint32_t x = 2u * compact1by2(g), y = 2u * compact1by2(g >> 1),
                   z = 2u * compact1by2(g >> 2);
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++) {
      const uint32_t two = (any >> (2u * k)) & 3u;
      if (two) {
        const uint32_t r = (y + (k & 1u)) + ((z + (k >> 1)) << lg);
        atomicOr(&half[2u * r + (x >> 5)], two << (x & 31u));
      }
    }
  }
  __syncthreads();
  // along x: each row by itself
  for (uint32_t r = t; r < rows; r += 1024u) {
    uint64_t v = row[r];
#pragma unroll
    for (uint32_t s = 1; s < 64u; s <<= 1) v |= (o & 1u) ? v << s : v >> s;
    row[r] = v & full;
  }
  __syncthreads();
  for (uint32_t axis = 1; axis < 3u; axis++) {
    const uint32_t sh = axis == 1u ? 0u : lg;  // log2 of the row stride
    const bool neg = ((o >> axis) & 1u) != 0u;
    for (uint32_t s = 1; s < R; s <<= 1) {
      uint64_t v[4] = {0, 0, 0, 0};
#pragma unroll
      for (uint32_t k = 0; k < 4u; k++) {
        const uint32_t r = t + 1024u * k, c = (r >> sh) & (R - 1u);
        if (r < rows && (neg ? c >= s : c + s < R))
          v[k] = row[neg ? r - (s << sh) : r + (s << sh)];
      }
      __syncthreads();
#pragma unroll
      for (uint32_t k = 0; k < 4u; k++)
        if (t + 1024u * k < rows) row[t + 1024u * k] |= v[k];
      __syncthreads();
    }
  }
  uint32_t sum = 0;
  for (uint32_t w = t; w < words; w += 1024u) {
    // 32 regions: x 4, y 4, z 2 of them (code bits x0 y0 z0 x1 y1); fewer in
    // the one word of a map with R < 4
    const uint32_t c = w * 32u;
    const uint32_t x = compact1by2(c), y = compact1by2(c >> 1), z = compact1by2(c >> 2);
    uint32_t bits = 0;
#pragma unroll
    for (uint32_t k = 0; k < 8u; k++) {
      const uint32_t dy = (k & 1u) | (k & 2u), dz = k >> 2;
      if (y + dy >= R || z + dz >= R) continue;
      const uint32_t q = (uint32_t)(~row[(y + dy) + ((z + dz) << lg)] >> x);
#pragma unroll
      for (uint32_t dx = 0; dx < 4u; dx++)
        if (x + dx < R)
          bits |= ((q >> dx) & 1u)
                  << ((dx & 1u) | ((dy & 1u) << 1) | (dz << 2) | ((dx >> 1) << 3) | ((dy >> 1) << 4));
    }
    fm[o * words + w] = bits;
    sum += (uint32_t)__popc(bits);
  }
  if (sum) atomicAdd(&total, sum);
  __syncthreads();
  if (t == 0u) report->free_regions[o] = total;
}

uint32_t free_regions(uint32_t dim) { return dim >= 16u ? dim / 16u : 1u; }

uint32_t free_words_per_octant(uint32_t dim) {
  const uint32_t R = free_regions(dim);
  return (R * R * R + 31u) / 32u;
}

// ---- clearance map: how far a ray's line stays clear of everything ----
// Cells of 8^3 blocks, R = dim / 8 per axis (a power of two, 4 .. 128; 2:
// k_clear_16).  A
// cell is near when the cell widened by 2 blocks a side holds a nonempty
// block.  For each of the 8 direction octants, the byte of a cell is the
// Chebyshev distance in cells to the first near cell of its forward orthant:
// the side of the largest cube of clear cells with this one as its corner (0:
// near itself; 255: no near cell in the orthant).
//
// The cells are tested at 2-block resolution: byte b of `sub` holds, for 4^3
// brick b, one bit per 2^3 sub-block, so the 8 bytes of a cell are one word
// with a bit per sub-block in Morton order.  The distance is separable: along
// x the distance to the first near cell of the row, along y min over j of
// max(j, that of the row j ahead), along z the same of those planes -- 2, 4
// and 8 direction variants.  Bound by the search (at most the distance itself
// per cell): four cells a thread, as 16-bit pairs.  512^3, with the rows
// alone: 12 + 9 + 12 us (one cell a thread: 32 + 21 + 57), 1024^3 about 8
// times that.

// Whether the cell is near: its own word, and of each neighbour the
// sub-blocks that face it.  Neighbours' codes by dilated increments; a
// neighbour outside the grid repeats the cell itself.  filled: every sub-block
// of the cell holds something.
__device__ __forceinline__ bool cell_near(const uint64_t* __restrict__ words, uint32_t R,
                                          uint32_t x, uint32_t y, uint32_t z, bool& filled) {
  // sub-blocks of a word with x coordinate 0 / 3 (bits 0 and 3 of the code)
  constexpr uint64_t X0 = 0x0055005500550055ull, X3 = X0 << 9;
  constexpr uint64_t Y0 = 0x0000333300003333ull, Y3 = Y0 << 18;
  constexpr uint64_t Z0 = 0x000000000F0F0F0Full, Z3 = Z0 << 36;
  const uint32_t cx[3] = {part1by2(x ? x - 1u : x), part1by2(x), part1by2(min(x + 1u, R - 1u))};
  const uint32_t cy[3] = {part1by2(y ? y - 1u : y) << 1, part1by2(y) << 1,
                          part1by2(min(y + 1u, R - 1u)) << 1};
  const uint32_t cz[3] = {part1by2(z ? z - 1u : z) << 2, part1by2(z) << 2,
                          part1by2(min(z + 1u, R - 1u)) << 2};
  uint64_t any = 0;
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int i = 0; i < 3; i++) {
        uint64_t mask = ~0ull;
        if (i != 1) mask &= i == 0 ? X3 : X0;
        if (j != 1) mask &= j == 0 ? Y3 : Y0;
        if (k != 1) mask &= k == 0 ? Z3 : Z0;
        any |= words[cx[i] | cy[j] | cz[k]] & mask;
      }
  filled = words[cx[1] | cy[1] | cz[1]] == ~0ull;
  return any != 0ull;
}

// The layers of cells whose near cells an edit may have changed, bit z of 128
// (maps_changed).  A rebuild after an edit makes the rows and planes of these
// alone: the scratch holds the others'.  1024^3, a brush of 4^3 blocks: the
// rebuild's launches 49 + 9 + 58 us where all layers take 83 + 26 + 82, the
// edit 147 us against 223; 64 blocks anywhere (most layers) 176 against 220.
struct Layers {
  uint64_t lo, hi;
};
__device__ __forceinline__ Layers changed_layers(const uint32_t* __restrict__ changed) {
  return {changed[0] | (uint64_t)changed[1] << 32, changed[2] | (uint64_t)changed[3] << 32};
}
// Whether one of layers z0 .. z1 is among them.
__device__ __forceinline__ bool some_layer(const Layers& l, uint32_t z0, uint32_t z1) {
  for (uint32_t z = z0; z <= z1; z++)
    if ((z < 64u ? l.lo >> z : l.hi >> (z - 64u)) & 1u) return true;
  return false;
}
// Layers from z on (z itself: 0) to the first of them upwards or downwards;
// 255: none.
__device__ __forceinline__ uint32_t next_layer(const Layers& l, uint32_t z, bool down) {
  uint64_t near, far;  // `near` the half that z lies in, from z on
  uint32_t to_far;
  if (down) {
    near = z < 64u ? l.lo << (63u - z) : l.hi << (127u - z);
    far = z < 64u ? 0ull : l.lo;
    to_far = z - 63u;
    if (near) return (uint32_t)__builtin_clzll(near);
    return far ? to_far + (uint32_t)__builtin_clzll(far) : 255u;
  }
  near = z < 64u ? l.lo >> z : l.hi >> (z - 64u);
  far = z < 64u ? l.hi : 0ull;
  to_far = 64u - z;
  if (near) return (uint32_t)__builtin_ctzll(near);
  return far ? to_far + (uint32_t)__builtin_ctzll(far) : 255u;
}

// Rows of cells along x, one thread per cell: the distance along +x (plane 0)
// and -x (plane 1) to the first near cell of the row.  A block takes kMapBlock
// cells (whole rows), finds the rows' near cells by ballot and notes how many
// of them are not filled (low half of its count) and how many are (high half).
struct ClearRowsArgs {
  const uint64_t* words;
  uint32_t lg;
  uint8_t* rows;
  uint32_t* near_count;
  const uint32_t* changed;
};
__device__ __forceinline__ void clear_rows_block(const ClearRowsArgs& a, uint32_t block,
                                                 uint64_t* bits) {
  const uint64_t* __restrict__ words = a.words;
  uint8_t* __restrict__ rows = a.rows;
  const uint32_t lg = a.lg;
  const uint32_t R = 1u << lg, n = 1u << (3u * lg), i0 = block * kMapBlock;
  if (a.changed &&  // the same for every thread
      !some_layer(changed_layers(a.changed), i0 >> (2u * lg),
                  min(i0 + kMapBlock - 1u, n - 1u) >> (2u * lg)))
    return;
  const uint32_t i = i0 + threadIdx.x, x = i & (R - 1u);
  bool near = false, filled = false;
  if (i < n) near = cell_near(words, R, x, (i >> lg) & (R - 1u), i >> (2u * lg), filled);
  const uint64_t b = __ballot(near), f = __ballot(filled);
  if ((threadIdx.x & 63u) == 0u) {
    bits[threadIdx.x >> 6] = b;
    bits[kMapBlock / 64u + (threadIdx.x >> 6)] = f;
  }
  __syncthreads();
  if (threadIdx.x == 0u) {
    uint32_t count = 0u;  // (a filled cell is near)
#pragma unroll
    for (uint32_t k = 0; k < kMapBlock / 64u; k++) {
      const uint32_t full = (uint32_t)__popcll(bits[kMapBlock / 64u + k]);
      count += (uint32_t)__popcll(bits[k]) - full + (full << 16);
    }
    a.near_count[block] = count;
  }
  if (i >= n) return;
  // the row's bits, as one or two words (R <= 64: part of the wave's)
  const uint32_t first = threadIdx.x - x, w0 = first >> 6, sh = first & 63u;
  const uint64_t full = R >= 64u ? ~0ull : (1ull << R) - 1ull;
  const uint64_t lo = (bits[w0] >> sh) & full, hi = R > 64u ? bits[w0 + 1u] : 0ull;
  const uint64_t up_lo = x < 64u ? lo >> x : 0ull;
  const uint64_t up_hi = x < 64u ? hi : hi >> (x - 64u);
  uint32_t up = 255u, down = 255u;
  if (up_lo)
    up = (uint32_t)__builtin_ctzll(up_lo);
  else if (up_hi)
    up = (uint32_t)__builtin_ctzll(up_hi) + (x < 64u ? 64u - x : 0u);
  const uint64_t dn_lo = x < 63u ? lo & ((2ull << x) - 1ull) : lo;
  const uint64_t dn_hi = x < 64u ? 0ull : (x < 127u ? hi & ((2ull << (x - 64u)) - 1ull) : hi);
  if (dn_hi)
    down = x - 64u - (63u - (uint32_t)__builtin_clzll(dn_hi));
  else if (dn_lo)
    down = x - (63u - (uint32_t)__builtin_clzll(dn_lo));
  rows[i] = (uint8_t)up;
  rows[(size_t)n + i] = (uint8_t)down;
}

// The free-region map and the clearance map's first pass in one launch: they
// read different words and neither waits for the other, and each was a
// launch of 12-15 us with most of the chip idle (8 blocks; 262,144 threads of
// one wave's latency).  The first 8 blocks take the octants' bitmaps, the
// others the rows of cells.  A rebuild at 512^3 37 us instead of 48, after an
// edit of a few layers 28 (this launch 14 of them; the octants' blocks, one CU
// each, bound it).
__global__ __launch_bounds__(1024) void k_maps_first(FreeMapArgs fa, ClearRowsArgs ca) {
  __shared__ uint64_t row[4096];
  __shared__ uint32_t total;
  if (blockIdx.x < 8u)
    free_map_block(fa, row, total);
  else
    clear_rows_block(ca, blockIdx.x - 8u, row);
}

// Four bytes as two pairs of 16 bits, and back.
typedef unsigned short us2 __attribute__((ext_vector_type(2)));
struct Cells4 {
  us2 even, odd;  // cells 0, 2 and 1, 3
};
__device__ __forceinline__ Cells4 cells4(uint32_t v) {
  Cells4 c;
  const uint32_t e = v & 0x00FF00FFu, o = (v >> 8) & 0x00FF00FFu;
  __builtin_memcpy(&c.even, &e, 4);
  __builtin_memcpy(&c.odd, &o, 4);
  return c;
}
__device__ __forceinline__ uint32_t cells4_word(const Cells4& c) {
  uint32_t e, o;
  __builtin_memcpy(&e, &c.even, 4);
  __builtin_memcpy(&o, &c.odd, 4);
  return e | (o << 8);
}

// min over j >= 0 of max(j, p[j * stride]) of four cells side by side, `len`
// words; 255 = none.  Four words in flight: the search waits on its loads.
__device__ __forceinline__ uint32_t ahead(const uint8_t* __restrict__ p, ptrdiff_t stride,
                                          uint32_t len) {
  Cells4 best = cells4(*reinterpret_cast<const uint32_t*>(p));
  for (uint32_t j = 1; j < len; j += 4u) {
    const us2 most = __builtin_elementwise_max(best.even, best.odd);
    if (j >= (uint32_t)max((int)most.x, (int)most.y)) break;
    uint32_t word[4];
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++)
      word[k] = *reinterpret_cast<const uint32_t*>(p + (ptrdiff_t)min(j + k, len - 1u) * stride);
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++) {  // (past the end: the last word, further off)
      const Cells4 v = cells4(word[k]);
      const us2 jj = (us2)((unsigned short)(j + k));
      best.even = __builtin_elementwise_min(best.even, __builtin_elementwise_max(v.even, jj));
      best.odd = __builtin_elementwise_min(best.odd, __builtin_elementwise_max(v.odd, jj));
    }
  }
  return cells4_word(best);
}

// Planes: variant v = x direction | y direction << 1.  The first block also
// sums up the near cells for the report.
__global__ __launch_bounds__(256) void k_clear_planes(const uint8_t* __restrict__ rows,
                                                      uint32_t lg, uint8_t* __restrict__ planes,
                                                      const uint32_t* __restrict__ near_count,
                                                      const uint32_t* __restrict__ changed,
                                                      CtxReport* __restrict__ report) {
  const uint32_t R = 1u << lg, n = 1u << (3u * lg);
  if (blockIdx.x == 0u) {
    __shared__ uint32_t total[2];
    if (threadIdx.x < 2u) total[threadIdx.x] = 0u;
    __syncthreads();
    uint32_t open = 0, full = 0;
    for (uint32_t b = threadIdx.x; b < (n + kMapBlock - 1u) / kMapBlock; b += 256u) {
      open += near_count[b] & 0xFFFFu;
      full += near_count[b] >> 16;
    }
    if (open) atomicAdd(&total[0], open);
    if (full) atomicAdd(&total[1], full);
    __syncthreads();
    if (threadIdx.x == 0u) {
      report->near_cells = total[0];
      report->filled_cells = total[1];
    }
  }
  const uint32_t t = 4u * (blockIdx.x * 256u + threadIdx.x);
  if (t >= 4u * n) return;
  const uint32_t v = t >> (3u * lg), i = t & (n - 1u), y = (i >> lg) & (R - 1u);
  const uint32_t layer = i >> (2u * lg);
  if (changed && !some_layer(changed_layers(changed), layer, layer)) return;
  const bool neg = (v & 2u) != 0u;
  *reinterpret_cast<uint32_t*>(planes + t) =
      ahead(rows + (size_t)(v & 1u) * n + i, neg ? -(ptrdiff_t)R : (ptrdiff_t)R,
            neg ? y + 1u : R - y);
}

// The map: octant plane o with its negative axes complemented, in Morton
// order and (8 planes on) in linear order.  A byte m follows from the layers
// up to m ahead (a near cell further on is further off), so after an edit it
// stays what it is when none of those changed.
__global__ __launch_bounds__(256) void k_clear_cubes(const uint8_t* __restrict__ planes,
                                                     uint32_t lg, uint8_t* __restrict__ map,
                                                     const uint32_t* __restrict__ changed) {
  const uint32_t R = 1u << lg, n = 1u << (3u * lg);
  const uint32_t t = 4u * (blockIdx.x * 256u + threadIdx.x);
  if (t >= 8u * n) return;
  const uint32_t o = t >> (3u * lg), i = t & (n - 1u);
  const uint32_t x = i & (R - 1u), y = (i >> lg) & (R - 1u), z = i >> (2u * lg);
  const ptrdiff_t layer = (ptrdiff_t)R * R;
  const bool neg = (o & 4u) != 0u;
  const uint32_t fx = (o & 1u) ? R - 4u - x : x, fy = (o & 2u) ? R - 1u - y : y,
                 fz = (o & 4u) ? R - 1u - z : z;
  uint8_t* plane = map + (size_t)o * n;
  uint32_t* linear =
      reinterpret_cast<uint32_t*>(plane + 8u * (size_t)n + fx + (size_t)R * (fy + (size_t)R * fz));
  if (changed) {
    const uint32_t next = next_layer(changed_layers(changed), z, neg);
    if (next == 255u) return;  // nothing ahead
    const uint32_t old = *linear;
    const uint32_t most = max(max(old & 255u, (old >> 8) & 255u), max((old >> 16) & 255u, old >> 24));
    if (next > most) return;
  }
  uint32_t m = ahead(planes + (size_t)(o & 3u) * n + i, neg ? -layer : layer,
                     neg ? z + 1u : R - z);
  if (o & 1u) m = __builtin_bswap32(m);
  // cells fx .. fx + 3 have Morton codes c, c + 1, c + 8, c + 9
  uint16_t* mor = reinterpret_cast<uint16_t*>(plane + morton3(fx, fy, fz));
  mor[0] = (uint16_t)m;
  mor[4] = (uint16_t)(m >> 16);
  *linear = m;
}

// A 16^3 map has 2 cells a side and is one region: clear all round (255) when
// it holds nothing, else all of it near, so that no ray is asked to walk 2
// cells.
__global__ __launch_bounds__(128) void k_clear_16(const uint64_t* __restrict__ word,
                                                  uint8_t* __restrict__ map,
                                                  CtxReport* __restrict__ report) {
  const bool empty = word[0] == 0ull;
  map[threadIdx.x] = empty ? 255 : 0;
  if (threadIdx.x == 0u) {
    report->near_cells = empty ? 0u : 8u;
    report->filled_cells = 0u;
  }
}

uint32_t clear_cells(uint32_t dim) {
  const uint32_t R = dim / 8u;
  return R * R * R;
}

size_t clear_tmp_bytes(uint32_t dim) {
  const size_t n = clear_cells(dim);
  return 14u * n + 4u * ((n + 255u) / 256u);
}

// The rebuild of a world's maps; without a clearance map (map null, dim < 16)
// the free-region map alone.  changed: the words of maps_changed; null =
// rebuild both.
static hipError_t launch_build_maps(const uint64_t* l1b, const uint64_t* words, uint32_t dim,
                                    uint32_t* fm, uint8_t* tmp, uint8_t* map,
                                    const uint32_t* changed, CtxReport* report,
                                    hipStream_t stream) {
  FreeMapArgs fa = {l1b, words, 0u, free_words_per_octant(dim), fm, changed, report};
  while ((1u << fa.lg) < free_regions(dim)) fa.lg++;
  if (dim < 32u) {
    hipLaunchKernelGGL(k_maps_first, dim3(8), dim3(kMapBlock), 0, stream, fa, ClearRowsArgs{});
    if (map) hipLaunchKernelGGL(k_clear_16, dim3(1), dim3(128), 0, stream, l1b ? l1b : words, map,
                                report);
    return hipGetLastError();
  }
  const uint32_t n = clear_cells(dim);
  uint32_t lg = 0;
  while ((8u << lg) < dim) lg++;
  uint8_t *rows = tmp + 8u * (size_t)n, *planes = rows + 2u * (size_t)n;
  uint32_t* near_count = reinterpret_cast<uint32_t*>(planes + 4u * (size_t)n);
  const uint32_t* moved = changed ? changed + 1 : nullptr;
  const ClearRowsArgs ca = {reinterpret_cast<const uint64_t*>(tmp), lg, rows, near_count, moved};
  hipLaunchKernelGGL(k_maps_first, dim3(8u + (n + kMapBlock - 1u) / kMapBlock), dim3(kMapBlock), 0,
                     stream, fa, ca);
  hipLaunchKernelGGL(k_clear_planes, dim3((n + 255u) / 256u), dim3(256), 0, stream, rows, lg,
                     planes, near_count, moved, report);
  hipLaunchKernelGGL(k_clear_cubes, dim3((2u * n + 255u) / 256u), dim3(256), 0, stream, planes,
                     lg, map, moved);
  return hipGetLastError();
}

uint32_t brick_bit_words(uint32_t dim) {
  const uint64_t n = (uint64_t)dim * dim * dim;
  return n >= 4096u ? (uint32_t)(n / 4096u) : 1u;
}

hipError_t rebuild_maps(vt_world* w, hipStream_t stream, const uint32_t* changed) {
  w->maps_valid = false;
  if (!w->freemap) return hipSuccess;
  return launch_build_maps(w->l1b, w->brick_bits, w->dim, w->freemap, w->clear_tmp, w->clear,
                           changed, w->ctx->report_dev(), stream);
}

void finish_maps(vt_world* w) {
  w->maps_valid = false;
  if (!w->freemap) return;
  const CtxReport* r = w->ctx->report();
  if (r->free_built) {
    const double R = free_regions(w->dim);
    w->free_frac = 0.0f;
    for (uint32_t o = 0; o < 8; o++)
      w->free_frac = std::max(w->free_frac, (float)((double)r->free_regions[o] / (R * R * R)));
  }
  if (w->clear) {
    const uint32_t open = clear_cells(w->dim) - r->filled_cells;
    w->near_frac = open ? (float)((double)r->near_cells / (double)open) : 1.0f;
  }
  w->maps_valid = true;
}

bool use_free_map(const vt_world* w, const ShadeConsts& sc) {
  if (!w->freemap || !w->maps_valid || w->free_frac <= 0.0f) return false;
  if (sc.flags & VT_FLAG_FREE_MAP_OFF) return false;
  if (sc.flags & VT_FLAG_FREE_MAP_ON) return true;
  return (sc.max_primary >= VT_FREE_MIN_CAP || sc.max_shadow >= VT_FREE_MIN_CAP) &&
         w->free_frac * VT_FREE_MIN_SHARE >= 1.0f;
}

// The map pays where rays cross clear space, so the rule counts the cells they
// can cross: a filled cell (solid ground) says nothing.  Microseconds with the
// map and without, 256^3 at 1280x720 with caps of 2048 (of 192 / 48), by the
// near share of what is not filled:
//   scattered blocks, no sky    0.12 126, 177 (75, 95)    0.27 163, 168 (109, 107)
//                               0.40 175, 165 (116, 106)  0.59 195, 175 (118, 106)
//   terrain, blocks up to the top (0.50) 124, 120 (84, 78)
//   ground with open sky        0.08 58, 96 (44, 49)      0.18 76, 131 (65, 87)
// and worlds of 512^3 with open ground to 55% of their height 73, 165, in the
// reference layout 81, 262.  Above the line the space between things is too
// small to cross, but a ray that leaves it for the sky still ends at once with
// the map and otherwise takes every step to the edge of the grid.  By the
// largest share of free regions, blocks below an empty sky, caps of 2048:
//   near 0.44, free 0.3: 162, 183     near 0.62, free 0.38: 81, 115
//   near 0.71, free 0.25: 74, 84      near 0.80, free 0.19: 74, 74
//   near 0.56, free 0.06: 213, 198
// Caps of 192 / 48 end most such rays themselves, and it takes a sky of half
// the world: near 0.49, free 0.5: 61, 79 at 512^3 and 44, 94 in the reference
// layout; free 0.38: 65, 72, and at 256x256 32, 27; free 0.3: 105, 98.
constexpr float kClearNearShare = 1.0f / 3.0f;
constexpr float kClearFreeShare = 0.25f, kClearFreeShareShort = 0.45f;

bool use_clear_map(const vt_world* w, uint32_t flags, int max_primary, int max_shadow) {
  if (!w->clear || !w->maps_valid || (flags & VT_FLAG_FREE_MAP_OFF)) return false;
  if ((flags & VT_FLAG_FREE_MAP_ON) || w->near_frac <= kClearNearShare) return true;
  const bool long_caps = max_primary >= VT_FREE_MIN_CAP || max_shadow >= VT_FREE_MIN_CAP;
  return w->free_frac >= (long_caps ? kClearFreeShare : kClearFreeShareShort);
}

// The texel masks of an atlas: a thread makes one word (layer z of a model)
// from 64 texels, lanes along x, so that a wave reads whole rows of the atlas
// (64 MiB once: 16 us).
__global__ __launch_bounds__(256) void k_atlas_masks(const uint4* __restrict__ atlas,
                                                     uint64_t* __restrict__ masks) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  const uint32_t mx = i & 31u, z = (i >> 5) & 7u, my = (i >> 8) & 31u, mz = i >> 13;
  uint64_t m = 0u;
#pragma unroll
  for (uint32_t y = 0; y < 8u; ++y) {
    const uint4* row = atlas + (((mz * 8u + z) * 256u + my * 8u + y) * 256u + mx * 8u) / 4u;
    const uint4 a = row[0], b = row[1];
    const uint32_t t[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (uint32_t x = 0; x < 8u; ++x) m |= (uint64_t)(t[x] != 0u) << (x + 8u * y);
  }
  masks[(mx + 32u * (my + 32u * mz)) * 8u + z] = m;
}

hipError_t launch_atlas_masks(const uint32_t* atlas, uint64_t* masks, hipStream_t stream) {
  hipLaunchKernelGGL(k_atlas_masks, dim3((uint32_t)(kAtlasMaskWords / 256)), dim3(256), 0, stream,
                     reinterpret_cast<const uint4*>(atlas), masks);
  return hipGetLastError();
}

// One thread per 4^3 brick of the layers y < 4 ny: a brick lies in one chunk,
// so one chunk-table read and 16 rows of 4 pool words make its 64 occupancy
// bytes (Morton order).  A whole 512^3 map, mostly empty chunks: 384 us as
// one thread per block, 45 us here.
__global__ __launch_bounds__(256) void k_build_occupancy(BrickmapWorld w, uint8_t* __restrict__ occ,
                                                         uint64_t* __restrict__ brick_bits,
                                                         uint8_t* __restrict__ sub, uint32_t ny) {
  const uint32_t nb = w.dim / 4u;
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (uint64_t)nb * ny * nb) return;
  const uint32_t bx = (uint32_t)(i % nb), by = (uint32_t)(i / nb % ny),
                 bz = (uint32_t)(i / ((uint64_t)nb * ny));
  const uint32_t M = w.dim / 8u;
  const uint32_t c = morton3(bx, by, bz);
  const uint32_t e = w.chunks[bx / 2u + M * (by / 2u + (size_t)(bz / 2u) * M)];
  uint32_t out[16] = {};
  uint64_t mask = 0;
  if (e != 0u) {
    const uint32_t* src = w.pool + (size_t)(e - 1u) * 512u + 4u * (bx & 1u) + 32u * (by & 1u) +
                          256u * (bz & 1u);
    uint32_t row[16];
#pragma unroll
    for (uint32_t k = 0; k < 16u; k++) {
      const uint4 v = *reinterpret_cast<const uint4*>(src + 8u * (k & 3u) + 64u * (k >> 2));
      row[k] = (v.x ? 1u : 0u) | (v.y ? 0x100u : 0u) | (v.z ? 0x10000u : 0u) |
               (v.w ? 0x1000000u : 0u);
    }
    mask = morton_brick(row, out);
  }
  uint4* dst = reinterpret_cast<uint4*>(occ + 64u * (size_t)c);
#pragma unroll
  for (uint32_t q = 0; q < 4u; q++)
    dst[q] = make_uint4(out[4 * q], out[4 * q + 1], out[4 * q + 2], out[4 * q + 3]);
  if (sub) sub[c] = (uint8_t)nonzero_bytes(mask);
  if (mask)
    atomicOr(reinterpret_cast<unsigned long long*>(brick_bits + (c >> 6)), 1ull << (c & 63u));
}

__global__ __launch_bounds__(256) void k_clear_words(uint64_t* __restrict__ p, uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) p[i] = 0ull;
}

hipError_t launch_build_occupancy(const BrickmapWorld& w, uint8_t* occ, uint64_t* brick_bits,
                                  uint8_t* sub, hipStream_t stream, uint32_t y_end) {
  if (y_end == 0 || y_end > w.dim) y_end = w.dim;
  if (y_end == w.dim) {
    const uint32_t nwords = brick_bit_words(w.dim);
    hipLaunchKernelGGL(k_clear_words, dim3((nwords + 255u) / 256u), dim3(256), 0, stream,
                       brick_bits, nwords);
  }
  const uint32_t ny = (y_end + 3u) / 4u;
  const uint64_t n = (uint64_t)(w.dim / 4u) * ny * (w.dim / 4u);
  hipLaunchKernelGGL(k_build_occupancy, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, stream, w,
                     occ, brick_bits, sub, ny);
  return hipGetLastError();
}

}  // namespace vt
