// Marching-cubes mesh extraction: the reference's MeshEngine
// (RGBDFusion/src/MeshEngine.cu:7-339, tables RGBDFusion/utils/TriangleTable.h).
//
// MI355X design: one wavefront per allocated block.  The +1 corners of a
// block's voxels live in up to seven neighbour blocks, whose pool indices are
// resolved once per block (seven hash probes) and recorded.  Extraction is a
// count pass over two bits per voxel, a scan of the per-block counts and an
// emission pass through lists, so every block's output is contiguous and
// ordered by voxel index, then table order: the output is deterministic,
// unlike the reference's atomic triangle counter (MeshEngine.cu:246).
//
// Two output forms share the count pass:
//   * the reference's triangle soup (9 positions + 9 face-normal floats per
//     triangle, MeshEngine.cu:246-264), bit-identical to the scalar
//     restatement;
//   * an indexed mesh (float32 xyz vertices, int32 triangle corners).  Each
//     voxel owns the three cube edges leaving its corner along +x, +y, +z;
//     an owned edge with a sign change between two observed end voxels gets
//     one vertex, placed by the reference's interpolation evaluated from the
//     lower end.  Triangles of a cube reference the owners' vertices, so a
//     vertex is shared by every triangle that touches its edge.

#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

#include "yas_internal.hpp"

using namespace yas;

MapView yas_map_view(yas_map* map);
yas_ctx* yas_map_ctx(yas_map* map);
int yas_map_get_stats(yas_map* m, yas_map_stats* st);

namespace {

// Triangulation table: bits 0-3 = triangle count, then 4 bits per edge.
__constant__ uint64_t kTriTable[256] = {
#include "mc_tables.inc"
};

// MeshEngine.cu:76-112 corner order: corner c lies at x + (0x66 >> c & 1),
// y + (0xCC >> c & 1), z + (c >> 2).
__device__ inline int corner_step(int c, int sx, int sy, int sz) {
  return ((0x66 >> c) & 1) * sx + ((0xCC >> c) & 1) * sy + (c >> 2) * sz;
}
// MeshEngine.cu:150-224: cube edge e runs from corner edge_a(e) to edge_b(e).
__device__ inline int edge_a(int e) { return (int)((0x321076543210ull >> (4 * e)) & 7); }
__device__ inline int edge_b(int e) { return (int)((0x765447650321ull >> (4 * e)) & 7); }

// MeshEngine.cu:114-123.  The reference compares with the double 1e-6; the
// largest float below it is 1e-6f, so |v| < 1e-6 is |v| <= 1e-6f.
__device__ inline float edge_t(float v1, float v2) {
  if (fabsf(0.0f - v1) <= 1e-6f) return 0.0f;
  if (fabsf(0.0f - v2) <= 1e-6f) return 1.0f;
  if (fabsf(v1 - v2) <= 1e-6f) return 0.0f;
  return (0.0f - v1) / (v2 - v1);
}

// Edge e's point at parameter t in the unit cube: along x for edges 0, 2, 4,
// 6 (2 and 6 backwards), along y for 1, 3, 5, 7 (3 and 7 backwards), along z
// for 8 to 11.
__device__ inline void edge_offset(int e, float t, float& ox, float& oy, float& oz) {
  const float u = ((0x0CC >> e) & 1) ? 1.f - t : t;
  ox = ((0x055 >> e) & 1) ? u : ((0x622 >> e) & 1) ? 1.f : 0.f;
  oy = ((0x0AA >> e) & 1) ? u : ((0xC44 >> e) & 1) ? 1.f : 0.f;
  oz = e >= 8 ? t : ((0x0F0 >> e) & 1) ? 1.f : 0.f;
}
// Owner of cube edge e: the voxel at the edge's lower end, an offset from
// the cube's corner 0, and the edge's axis (0 = x, 1 = y, 2 = z).
__device__ inline int owner_x(int e) { return (0x622 >> e) & 1; }
__device__ inline int owner_y(int e) { return (0xC44 >> e) & 1; }
__device__ inline int owner_z(int e) { return (0x0F0 >> e) & 1; }
__device__ inline int owner_axis(int e) { return (0xAA4444 >> (2 * e)) & 3; }

// One wavefront takes one block at a time, four a workgroup: they share a copy
// of the triangulation table in LDS and meet at one barrier, after which the
// wavefronts go on by themselves.
constexpr int kMcWaves = 4;
constexpr int kMcThreads = 64 * kMcWaves;
constexpr int kMcCube = 9 * 9 * 9;  // a block and its +1 halo, index (z*9 + y)*9 + x

// The volume's blocks, or none when they are more than the records' `cap`:
// the host launches for the capacity, without asking for the count first,
// and repeats the extraction with more room when it did not suffice.
__device__ inline int mc_num_blocks(const MapView& m, int cap) {
  int n = m.ctr[kCtrAlloc];
  n = n < m.num_blocks ? n : m.num_blocks;
  return n <= cap ? n : 0;
}
// The block of this thread's wavefront.
__device__ inline int mc_block() {
  return __builtin_amdgcn_readfirstlane((int)blockIdx.x * kMcWaves + (int)(threadIdx.x >> 6));
}

__device__ inline int mc_cube_at(int x, int y, int z) { return (z * 9 + y) * 9 + x; }

// A staged word's sdf; every NaN as the quiet one.
template <class VT>
__device__ inline float mc_sdf(uint32_t w) {
  const float f = VT::word_sdf(w);
  return f != f ? __uint_as_float(0x7FC00000u) : f;
}

// Lanes of one wavefront exchanging values through LDS.
__device__ inline void mc_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A value per voxel of a block's +1 halo as a wavefront holds it: of the up
// to seven neighbour blocks (pool index nb of lane k for the
// offset (k&1, k>>1&1, k>>2&1), -1 absent: zeros) the faces x = 8 (lane (z,
// y)), y = 8 (lane (z, x)), z = 8 (lane (y, x)), and in `e` the edges: lanes
// 0-7 x = y = 8 (z = lane), 8-15 x = z = 8 (y = lane - 8), 16-23 y = z = 8
// (x = lane - 16), 24 the corner.
template <class T>
struct McHalo {
  T fx, fy, fz, e;
};
__device__ inline bool mc_bit(unsigned m, int i) { return (m >> i) & 1u; }
template <class T>
__device__ inline T mc_load(const T* src, bool wanted, int blk, int at) {
  T v = {};
  if (wanted && blk >= 0) v = src[(size_t)blk * 512 + at];
  return v;
}
// The layers z = 0..8 whose bit of `layers` is set; zeros for the others.
template <class T>
__device__ inline void mc_load_halo(const T* src, int nb, unsigned layers, McHalo<T>& v) {
  const int lane = threadIdx.x & 63, a = lane & 7, b = lane >> 3;
  const bool mine = mc_bit(layers, b), top = mc_bit(layers, 8);
  v.fx = mc_load(src, mine, __builtin_amdgcn_readlane(nb, 1), lane * 8);
  v.fy = mc_load(src, mine, __builtin_amdgcn_readlane(nb, 2), b * 64 + a);
  v.fz = mc_load(src, top, __builtin_amdgcn_readlane(nb, 4), lane);
  v.e = mc_load(src, lane < 8 ? mc_bit(layers, a) : lane < 25 && top, __shfl(nb, b == 0 ? 3 : b == 1 ? 5 : b == 2 ? 6 : 7),
                b == 0 ? a * 64 : b == 1 ? a * 8 : a);
}
// The halo's values written to LDS as f(value), index mc_cube_at.
template <class T, class S, class F>
__device__ inline void mc_stage_halo(const McHalo<T>& v, S* cube, F f) {
  const int lane = threadIdx.x & 63, a = lane & 7, b = lane >> 3;
  cube[mc_cube_at(8, a, b)] = f(v.fx);
  cube[mc_cube_at(a, 8, b)] = f(v.fy);
  cube[mc_cube_at(a, b, 8)] = f(v.fz);
  if (lane < 25) cube[mc_cube_at(b == 2 ? a : 8, b == 1 ? a : 8, b == 0 ? a : 8)] = f(v.e);
}

// Inclusive scan of v over the wavefront.
__device__ inline unsigned mc_scan(unsigned v) {
  int x = (int)v;
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31
  return (unsigned)x;
}
// The value of the next lane of 16 (the last: 0).
__device__ inline unsigned mc_next_lane(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x101, 0xF, 0xF, false);  // row_shl:1
}
// Bits i, 8 + i, .., 56 + i of m to bits 0..7.
__device__ inline unsigned mc_gather(unsigned long long m, int i) {
  const unsigned lo = ((unsigned)m >> i) & 0x01010101u, hi = ((unsigned)(m >> 32) >> i) & 0x01010101u;
  return ((lo * 0x01020408u) >> 24) | (((hi * 0x01020408u) >> 24) << 4);
}
// Bits 0..7 of v to bits 0, 4, .., 28.
__device__ inline unsigned mc_spread4(unsigned v) {
  v &= 0xFFu;
  v = (v | (v << 12)) & 0x000F000Fu;
  v = (v | (v << 6)) & 0x03030303u;
  return (v | (v << 3)) & 0x11111111u;
}
// Bits 0..3 of v to bits 0, 8, 16, 24.
__device__ inline unsigned mc_spread8(unsigned v) { return ((v & 0xFu) * 0x00204081u) & 0x01010101u; }

__device__ inline int block_excl_scan(int v, int* wsum, int& total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  int before = 0;
  total = 0;
  for (int i = 0; i < nw; ++i) {
    const int x = wsum[i];
    before += i < w ? x : 0;
    total += x;
  }
  __syncthreads();
  return before + inc - v;
}

// Count pass: per block, triangles and owned vertices; per voxel, the cube
// index (MeshEngine.cu:76-112; -1 unless all 8 corners are observed) and
// (local vertex prefix << 3 | owned edge mask).  It needs two bits of a
// voxel, its sign and whether it is observed.  A lane packs those of its
// column of voxels z = 0..8 into one word, signs in bits 0-8 and observed in
// bits 16-24; with the columns at x + 1, y + 1 and both, fetched from the next
// lanes, the tests of a column's 8 cubes are bit operations on 4 words, and
// the 8 slices' vertex prefixes are two scans of bytes (a slice owns at most
// 192 vertices).  Bound by memory: 58k float32 blocks, some 380 MB with the
// neighbours' faces, in 85 us.  (121 us with the block in LDS, each voxel
// reading its 8 corners there; 107 us with a slice's planes as 64-bit scalar
// masks, some 850 scalar instructions a block for a CU's one scalar unit.)
template <class VT>
__global__ void __launch_bounds__(kMcThreads) k_mc_count(MapView m, int cap, int2* counts, int16_t* cases,
                                                         uint16_t* vinfo, int* nbr) {
  __shared__ unsigned char tri_n[256];
  const int nblocks = mc_num_blocks(m, cap);
  // room left by a larger volume (463 blocks after 58k: 30.9 -> 29.5 us, by an
  // engine of its own 28.7; the same in the other passes gave nothing)
  if ((int)blockIdx.x * kMcWaves >= nblocks) return;
  if (threadIdx.x < 256) tri_n[threadIdx.x] = (unsigned char)(kTriTable[threadIdx.x] & 0xF);
  __syncthreads();
  const int blk = mc_block();
  if (blk >= nblocks) return;
  const int lane = threadIdx.x & 63, a = lane & 7, b = lane >> 3;
  const typename VT::T* vox = (const typename VT::T*)m.voxels;
  typename VT::T own[8];
  McHalo<typename VT::T> v;
#pragma unroll
  for (int z = 0; z < 8; ++z) own[z] = vox[(size_t)blk * 512 + z * 64 + lane];
  int nb = -1;
  if (lane < 8) {
    int bx, by, bz;
    unpack_key(m.block_keys[blk], bx, by, bz);
    nb = lane == 0 ? blk : find_block_xyz(m, bx + (lane & 1), by + ((lane >> 1) & 1), bz + ((lane >> 2) & 1));
    nbr[(size_t)blk * 8 + lane] = nb;
  }
  mc_load_halo(vox, nb, 0x1FFu, v);
  unsigned c0 = 0;  // this lane's column
#pragma unroll
  for (int z = 0; z < 9; ++z) {
    typename VT::T w = v.fz;
    if (z < 8) w = own[z];
    c0 |= (VT::negative(w) ? 1u << z : 0u) | (VT::observed(w) ? 0x10000u << z : 0u);
  }
  // the columns (8, y = b), (x = a, 8) and (8, 8)
  const unsigned en = (unsigned)__ballot(VT::negative(v.e)), eo = (unsigned)__ballot(VT::observed(v.e));
  const unsigned hx = mc_gather(__ballot(VT::negative(v.fx)), b) | (((en >> (8 + b)) & 1u) << 8) |
                      (mc_gather(__ballot(VT::observed(v.fx)), b) | (((eo >> (8 + b)) & 1u) << 8)) << 16;
  const unsigned hy = mc_gather(__ballot(VT::negative(v.fy)), a) | (((en >> (16 + a)) & 1u) << 8) |
                      (mc_gather(__ballot(VT::observed(v.fy)), a) | (((eo >> (16 + a)) & 1u) << 8)) << 16;
  const unsigned hxy = ((en & 0xFFu) | ((en >> 16) & 0x100u)) | ((eo & 0xFFu) | ((eo >> 16) & 0x100u)) << 16;
  // the columns at the cube's corners 1 (x + 1), 2 (x + 1, y + 1), 3 (y + 1)
  const unsigned n0 = mc_next_lane(c0), nhy = mc_next_lane(hy);
  const unsigned c1 = a == 7 ? hx : n0;
  const unsigned u0 = (unsigned)__shfl_down((int)c0, 8, 64), u1 = (unsigned)__shfl_down((int)c1, 8, 64);
  const unsigned c3 = b == 7 ? hy : u0;
  const unsigned c2 = b < 7 ? u1 : a == 7 ? hxy : nhy;
  unsigned all = c0 & c1 & c2 & c3, any = c0 | c1 | c2 | c3;
  all &= all >> 1;
  any |= any >> 1;
  const unsigned valid = (all >> 16) & 0xFFu;
  const unsigned mixed = valid & any & ~all;  // cubes with both signs: the others have no triangles
  const unsigned lo = mc_spread4(c0) | mc_spread4(c1) << 1 | mc_spread4(c2) << 2 | mc_spread4(c3) << 3;
  const unsigned hi = ((c0 >> 8) & 1u) | ((c1 >> 7) & 2u) | ((c2 >> 6) & 4u) | ((c3 >> 5) & 8u);
  const unsigned long long corners = (unsigned long long)hi << 32 | lo;
  const size_t at = (size_t)blk * 512 + lane;
  int tri = 0;
#pragma unroll
  for (int z = 0; z < 8; ++z) {
    const int cube = (int)(corners >> (4 * z)) & 0xFF;
    cases[at + z * 64] = (int16_t)((valid >> z) & 1u ? cube : -1);
    if ((mixed >> z) & 1u) tri += (int)tri_n[cube];
  }
  // owned edges: both ends observed, with a sign change
  const unsigned ex = (c0 ^ c1) & (c0 >> 16) & (c1 >> 16) & 0xFFu;
  const unsigned ey = (c0 ^ c3) & (c0 >> 16) & (c3 >> 16) & 0xFFu;
  const unsigned ez = (c0 ^ (c0 >> 1)) & (c0 >> 16) & (c0 >> 17) & 0xFFu;
  const unsigned edges = mc_spread4(ex) | mc_spread4(ey) << 1 | mc_spread4(ez) << 2;
  int vert = 0;  // vertices of the slices below
  if (__ballot(edges != 0u) != 0ull) {
    const unsigned nlo = mc_spread8(ex) + mc_spread8(ey) + mc_spread8(ez);
    const unsigned nhi = mc_spread8(ex >> 4) + mc_spread8(ey >> 4) + mc_spread8(ez >> 4);
    const unsigned slo = mc_scan(nlo), shi = mc_scan(nhi);
    const unsigned tlo = (unsigned)__builtin_amdgcn_readlane((int)slo, 63);
    const unsigned thi = (unsigned)__builtin_amdgcn_readlane((int)shi, 63);
#pragma unroll
    for (int z = 0; z < 8; ++z) {
      const int sh = 8 * (z & 3);
      const int pre = vert + (int)(((z < 4 ? slo - nlo : shi - nhi) >> sh) & 0xFFu);
      vinfo[at + z * 64] = (uint16_t)((pre << 3) | ((edges >> (4 * z)) & 7u));
      vert += (int)(((z < 4 ? tlo : thi) >> sh) & 0xFFu);
    }
  } else {
#pragma unroll
    for (int z = 0; z < 8; ++z) vinfo[at + z * 64] = 0;
  }
  tri = (int)mc_scan((unsigned)tri);
  if (lane == 63) counts[blk] = make_int2(tri, vert);
}

// Exclusive scan of the blocks' counts: 1024-block chunks scanned in parallel
// into `out`, and the chunks' totals, by the workgroup that ends last, into
// `chunk`; block i's prefix is out[i] + chunk[i >> kMcChunkShift], which its
// readers add.  (As three launches, local scan, chunk scan and addition, it
// cost 14 us of a 284 us extraction.)  `done` is 0 before and after.
struct McTotals {
  int tri, vert, blocks;
};
constexpr int kMcChunkShift = 10, kMcChunk = 1 << kMcChunkShift;
__device__ inline unsigned long long mc_pack2(int x, int y) {
  return (unsigned long long)(unsigned)x | (unsigned long long)(unsigned)y << 32;
}
__global__ void __launch_bounds__(kMcChunk) k_mc_scan(MapView m, int cap, const int2* in, int2* out,
                                                      unsigned long long* chunk, McTotals* total, unsigned* done) {
  __shared__ int wsum[16];
  __shared__ int carry[2];
  __shared__ int last;
  const int i = blockIdx.x * kMcChunk + threadIdx.x, nchunks = gridDim.x, n = mc_num_blocks(m, cap);
  const int2 v = i < n ? in[i] : make_int2(0, 0);
  int tx, ty;
  const int ex = block_excl_scan(v.x, wsum, tx);
  const int ey = block_excl_scan(v.y, wsum, ty);
  if (i < n) out[i] = make_int2(ex, ey);
  if (threadIdx.x == 0) {
    __hip_atomic_store(&chunk[blockIdx.x], mc_pack2(tx, ty), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = __hip_atomic_fetch_add(done, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)nchunks - 1u;
    carry[0] = carry[1] = 0;
  }
  __syncthreads();
  if (!last) return;
  for (int base = 0; base < nchunks; base += kMcChunk) {
    const int c = base + threadIdx.x;
    unsigned long long w = 0;
    if (c < nchunks) w = __hip_atomic_load(&chunk[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int cx = block_excl_scan((int)(unsigned)w, wsum, tx);
    const int cy = block_excl_scan((int)(unsigned)(w >> 32), wsum, ty);
    if (c < nchunks) chunk[c] = mc_pack2(carry[0] + cx, carry[1] + cy);
    __syncthreads();
    if (threadIdx.x == 0) {
      carry[0] += tx;
      carry[1] += ty;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    *total = McTotals{carry[0], carry[1], m.ctr[kCtrAlloc] < m.num_blocks ? m.ctr[kCtrAlloc] : m.num_blocks};
    *done = 0;
  }
}
// The scan's result for block `blk`.
struct McOffsets {
  const int2* local;
  const unsigned long long* chunk;
  __device__ inline int tri(int blk) const { return local[blk].x + (int)(unsigned)chunk[blk >> kMcChunkShift]; }
  __device__ inline int vert(int blk) const { return local[blk].y + (int)(unsigned)(chunk[blk >> kMcChunkShift] >> 32); }
};

// The emission passes.  A wavefront takes blocks in turn; lane l holds row
// (y, z) = (l & 7, l >> 3) of the count pass's records, voxels 8 l + x, so one
// 16-byte load brings each, a lane's entries are consecutive in voxel order
// and one scan places them.  The records of its next block are loaded while
// it works on the present one; of the sdf, the slices that this block's
// triangles or vertices need.
// The triangles and vertices are first listed in LDS and then taken from the
// list one per lane: only one voxel in five of a surface block has triangles,
// and those up to five, so emitting them voxel by voxel left most lanes idle,
// and the lanes of a list write consecutive entries.  A list holds entries
// done .. done + its size of the block; a block with more is listed again.
// 58k float32 blocks, 6.0 M indexed triangles: 110 us (246 us voxel by voxel,
// with the cubes formed again from a staged block); 2.1k int16 blocks, 232k
// triangles of the soup: 18 us (86 us).  About as much instruction issue as
// memory; 5 waves a SIMD instead of 4 (96 registers, some spilled) 115 us.
//   triangle entry: voxel (9 bits) | which of its triangles << 9
//   vertex entry:   voxel (9 bits) | axis << 9
constexpr int kTriList = 512, kVertList = 320;

struct McTables {
  uint64_t word[256];       // kTriTable
  unsigned char count[256]; // triangles
};
__device__ inline void mc_fill_tables(McTables& T) {
  T.word[threadIdx.x] = kTriTable[threadIdx.x];
  T.count[threadIdx.x] = (unsigned char)(kTriTable[threadIdx.x] & 0xF);
}
static_assert(kMcThreads == 256, "mc_fill_tables: a thread per case");

// A lane's row of a per-voxel 16-bit record.
struct McRow {
  unsigned w[4];
  __device__ inline unsigned at(int x) const { return (w[x >> 1] >> (16 * (x & 1))) & 0xFFFFu; }
};
__device__ inline McRow mc_load_row(const void* records, int blk) {
  const uint4 v = ((const uint4*)records)[(size_t)blk * 64 + (threadIdx.x & 63)];
  return McRow{{v.x, v.y, v.z, v.w}};
}
// Triangles of the row's voxels, 4 bits each.
__device__ inline unsigned mc_row_triangles(const McTables& T, const McRow& cases) {
  unsigned nt = 0;
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    const unsigned c = cases.at(x);  // 0xFFFF: not all corners observed
    nt |= (c - 1u < 254u ? (unsigned)T.count[c] : 0u) << (4 * x);
  }
  return nt;
}
__device__ inline int mc_nibble_sum(unsigned v) {  // of eight values, 40 at most
  v = (v & 0x0F0F0F0Fu) + ((v >> 4) & 0x0F0F0F0Fu);
  return (int)((v * 0x01010101u) >> 24);
}
// Slices with a lane for which `has` holds.
__device__ inline unsigned mc_slices(bool has) {
  unsigned long long m = __ballot(has);
  m |= m >> 4;
  m |= m >> 2;
  m |= m >> 1;
  return mc_gather(m, 0);
}
// The lane's triangles, at block positions first .. first + their number, put
// where the list's window [done, done + kTriList) holds them; last first.
__device__ inline void mc_list_triangles(uint16_t* list, unsigned nt, int end, int done) {
  const unsigned row = (threadIdx.x & 63) * 8;
  while (nt) {
    const int x4 = (31 - __clz((int)nt)) & ~3;
    const unsigned i = (nt >> x4) - 1u;
    nt -= 1u << x4;
    const unsigned at = (unsigned)(--end - done);
    if (at < (unsigned)kTriList) list[at] = (uint16_t)(row | (unsigned)(x4 >> 2) | (i << 9));
  }
}
__device__ inline void mc_list_vertices(uint16_t* list, unsigned edges, int first, int done) {
  const unsigned row = (threadIdx.x & 63) * 8;
  while (edges) {
    const int bit = __ffs((int)edges) - 1;
    edges &= edges - 1u;
    const unsigned at = (unsigned)(first++ - done);
    if (at < (unsigned)kVertList) list[at] = (uint16_t)(row | (unsigned)(bit >> 2) | (unsigned)(bit & 3) << 9);
  }
}
// A block's sdf and its halo's, layers z of the set bits, as 32-bit words.
template <class VT>
struct McSdf {
  static constexpr int kPer = 16 / (int)sizeof(typename VT::T);  // voxels of one load
  static constexpr int kLoads = 8 / kPer;
  uint4 own[kLoads];
  McHalo<typename VT::T> halo;
  __device__ inline void load(const typename VT::T* vox, int blk, int nb, unsigned layers) {
    const int lane = threadIdx.x & 63;
    const uint4* src = (const uint4*)(vox + (size_t)blk * 512);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      own[i] = make_uint4(0, 0, 0, 0);
      if (mc_bit(layers, (i * 64 + lane) * kPer >> 6)) own[i] = src[i * 64 + lane];
    }
    mc_load_halo(vox, nb, layers, halo);
  }
  __device__ inline void stage(uint32_t* cube) const {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int l = (i * 64 + lane) * kPer, at = mc_cube_at(l & 7, (l >> 3) & 7, l >> 6);
      if constexpr (kPer == 2) {
        cube[at] = own[i].x;  // {sdf, weight} twice
        cube[at + 1] = own[i].z;
      } else {
        cube[at] = own[i].x;
        cube[at + 1] = own[i].y;
        cube[at + 2] = own[i].z;
        cube[at + 3] = own[i].w;
      }
    }
    mc_stage_halo(halo, cube, [](const typename VT::T& w) { return VT::sdf_word(w); });
  }
};

__device__ inline void mc_voxel_xyz(int l, int& x, int& y, int& z) {
  x = l & 7;
  y = (l >> 3) & 7;
  z = l >> 6;
}

// Emit, reference form: triangle slot = block offset + exclusive prefix (in
// voxel index order) of the per-voxel counts.
struct McSoupLds {
  uint32_t sdf[kMcCube];
  alignas(16) uint16_t cases[512];
  uint16_t tri[kTriList];
};
template <class VT>
__device__ inline void mc_soup_flush(const McSoupLds& S, const McTables& T, int bx, int by, int bz, float vs,
                                     int first, int n, float* tris, float* normals, int cap) {
  for (int t = threadIdx.x & 63; t < n && first + t < cap; t += 64) {
    const unsigned ent = S.tri[t];
    int x, y, z;
    mc_voxel_xyz((int)(ent & 511u), x, y, z);
    const unsigned edges = (unsigned)(T.word[S.cases[ent & 511u]] >> (4 + 12 * (ent >> 9)));
    const int at = mc_cube_at(x, y, z);
    const float px = (float)(bx * 8 + x), py = (float)(by * 8 + y), pz = (float)(bz * 8 + z);
    float p[3][3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      // MeshEngine.cu:114-224: corner A + t * (edge direction), scaled by vs
      const int e = (int)((edges >> (4 * k)) & 0xF);
      const float sa = mc_sdf<VT>(S.sdf[at + corner_step(edge_a(e), 1, 9, 81)]);
      const float sb = mc_sdf<VT>(S.sdf[at + corner_step(edge_b(e), 1, 9, 81)]);
      float ox, oy, oz;
      edge_offset(e, edge_t(sa, sb), ox, oy, oz);
      p[k][0] = (px + ox) * vs;
      p[k][1] = (py + oy) * vs;
      p[k][2] = (pz + oz) * vs;
    }
    const float u0 = p[1][0] - p[0][0], u1 = p[1][1] - p[0][1], u2 = p[1][2] - p[0][2];
    const float w0 = p[2][0] - p[0][0], w1 = p[2][1] - p[0][1], w2 = p[2][2] - p[0][2];
    float n0 = u1 * w2 - u2 * w1, n1 = u2 * w0 - u0 * w2, n2 = u0 * w1 - u1 * w0;
    const float q = n0 * n0 + n1 * n1 + n2 * n2;
    if (q > 0.0f) {
      const float nn = sqrtf(q);
      n0 = n0 / nn; n1 = n1 / nn; n2 = n2 / nn;
    }
    float* P = tris + (size_t)(first + t) * 9;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      P[3 * k] = p[k][0]; P[3 * k + 1] = p[k][1]; P[3 * k + 2] = p[k][2];
    }
    if (normals) {
      float* N = normals + (size_t)(first + t) * 9;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        N[3 * k] = n0; N[3 * k + 1] = n1; N[3 * k + 2] = n2;
      }
    }
  }
}
template <class VT>
__global__ void __launch_bounds__(kMcThreads) k_mc_emit(MapView m, int cap_blocks, McOffsets offsets,
                                                        const int16_t* cases, float* tris, float* normals, int cap,
                                                        const int* nbr) {
  __shared__ McTables T;
  __shared__ McSoupLds lds[kMcWaves];
  mc_fill_tables(T);
  __syncthreads();
  const int nblocks = mc_num_blocks(m, cap_blocks);
  const int lane = threadIdx.x & 63, stride = gridDim.x * kMcWaves;
  McSoupLds& S = lds[threadIdx.x >> 6];
  int blk = mc_block(), nb = -1;
  McRow row = {};
  if (blk < nblocks) {
    row = mc_load_row(cases, blk);
    if (lane < 8) nb = nbr[(size_t)blk * 8 + lane];
  }
  while (blk < nblocks) {
    const int next = blk + stride;
    const McRow cur = row;
    const int cur_nb = nb;
    const unsigned nt = mc_row_triangles(T, cur), slices = mc_slices(nt != 0u), layers = slices | slices << 1;
    McSdf<VT> v;
    if (slices) v.load((const typename VT::T*)m.voxels, blk, cur_nb, layers);
    if (next < nblocks) {
      row = mc_load_row(cases, next);
      if (lane < 8) nb = nbr[(size_t)next * 8 + lane];
    }
    if (slices) {
      const int sum = mc_nibble_sum(nt), end = (int)mc_scan((unsigned)sum);
      const int total = __builtin_amdgcn_readlane(end, 63), first = offsets.tri(blk);
      int bx, by, bz;
      unpack_key(m.block_keys[blk], bx, by, bz);
      __builtin_memcpy(&S.cases[lane * 8], cur.w, 16);
      mc_list_triangles(S.tri, nt, end, 0);
      v.stage(S.sdf);
      for (int done = 0; done < total; done += kTriList) {
        if (done > 0) mc_list_triangles(S.tri, nt, end, done);
        mc_wave_sync();
        mc_soup_flush<VT>(S, T, bx, by, bz, m.voxel_size, first + done, min(kTriList, total - done), tris, normals, cap);
        mc_wave_sync();
      }
    }
    blk = next;
  }
}

// Emit, indexed form: the voxels' owned vertices, and their triangles as
// indices of the owners' vertices.
struct McIndexedLds {
  uint32_t sdf[kMcCube];
  uint16_t vi[kMcCube];    // the count pass's vertex info
  uint16_t vert[kVertList];
  uint16_t tri[kTriList];
  alignas(16) uint16_t cases[512];
  int vbase[8];            // first vertex of the block and its neighbours
};
// Owned vertices, interpolated from the voxel towards +x, +y, +z.
template <class VT>
__device__ inline void mc_vertex_flush(const McIndexedLds& S, int bx, int by, int bz, float vs, int first, int n,
                                       float* verts, int vcap) {
  for (int t = threadIdx.x & 63; t < n && first + t < vcap; t += 64) {
    const int ent = S.vert[t], a = ent >> 9;
    int x, y, z;
    mc_voxel_xyz(ent & 511, x, y, z);
    const int at = mc_cube_at(x, y, z);
    const float f = edge_t(mc_sdf<VT>(S.sdf[at]), mc_sdf<VT>(S.sdf[at + (a == 0 ? 1 : a == 1 ? 9 : 81)]));
    const float px = (float)(bx * 8 + x), py = (float)(by * 8 + y), pz = (float)(bz * 8 + z);
    float* V = verts + (size_t)(first + t) * 3;
    V[0] = (px + (a == 0 ? f : 0.0f)) * vs;
    V[1] = (py + (a == 1 ? f : 0.0f)) * vs;
    V[2] = (pz + (a == 2 ? f : 0.0f)) * vs;
  }
}
__device__ inline void mc_index_flush(const McIndexedLds& S, const McTables& T, int first, int n, int* tris,
                                      int tcap) {
  for (int t = threadIdx.x & 63; t < n && first + t < tcap; t += 64) {
    const unsigned ent = S.tri[t];
    int x, y, z;
    mc_voxel_xyz((int)(ent & 511u), x, y, z);
    const unsigned edges = (unsigned)(T.word[S.cases[ent & 511u]] >> (4 + 12 * (ent >> 9)));
    const int at = mc_cube_at(x, y, z);
    const unsigned xyz = (unsigned)(x | (y << 4) | (z << 8));  // 4 bits a coordinate: 8 is the neighbour's 0
    int id[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int e = (int)((edges >> (4 * k)) & 0xF);
      const int ox = owner_x(e), oy = owner_y(e), oz = owner_z(e);
      // the owner's block is present: every corner of an emitting cube is observed
      const unsigned oi = S.vi[at + mc_cube_at(ox, oy, oz)];
      const unsigned over = (xyz + (unsigned)(ox | (oy << 4) | (oz << 8))) & 0x888u;
      id[k] = S.vbase[((over * 0x49u) >> 9) & 7u] + (int)(oi >> 3) + __popc(oi & ((1u << owner_axis(e)) - 1u));
    }
    int* P = tris + (size_t)(first + t) * 3;
    P[0] = id[0]; P[1] = id[1]; P[2] = id[2];
  }
}
template <class VT>
__global__ void __launch_bounds__(kMcThreads) k_mc_emit_indexed(MapView m, int cap_blocks, McOffsets offsets,
                                                                const int16_t* cases, const uint16_t* vinfo,
                                                                float* verts, int vcap, int* tris, int tcap,
                                                                const int* nbr) {
  __shared__ McTables T;
  __shared__ McIndexedLds lds[kMcWaves];
  mc_fill_tables(T);
  __syncthreads();
  const int nblocks = mc_num_blocks(m, cap_blocks);
  const int lane = threadIdx.x & 63, stride = gridDim.x * kMcWaves;
  McIndexedLds& S = lds[threadIdx.x >> 6];
  int blk = mc_block(), nb = -1;
  McRow row = {}, irow = {};
  if (blk < nblocks) {
    row = mc_load_row(cases, blk);
    irow = mc_load_row(vinfo, blk);
    if (lane < 8) nb = nbr[(size_t)blk * 8 + lane];
  }
  while (blk < nblocks) {
    const int next = blk + stride;
    const McRow cur = row, info = irow;
    const int cur_nb = nb;
    const unsigned nt = mc_row_triangles(T, cur);
    unsigned edges = 0;
#pragma unroll
    for (int x = 0; x < 8; ++x) edges |= (info.at(x) & 7u) << (4 * x);
    const unsigned slices = mc_slices((nt | edges) != 0u), layers = slices | slices << 1;
    McSdf<VT> v;
    McHalo<uint16_t> ih;
    int vb = 0;
    if (slices) {
      v.load((const typename VT::T*)m.voxels, blk, cur_nb, layers);
      mc_load_halo(vinfo, cur_nb, layers, ih);
      if (lane < 8 && cur_nb >= 0) vb = offsets.vert(cur_nb);
    }
    if (next < nblocks) {
      row = mc_load_row(cases, next);
      irow = mc_load_row(vinfo, next);
      if (lane < 8) nb = nbr[(size_t)next * 8 + lane];
    }
    if (slices) {
      const int sum = mc_nibble_sum(nt), end = (int)mc_scan((unsigned)sum), vfirst = (int)(info.at(0) >> 3);
      const int ntri = __builtin_amdgcn_readlane(end, 63);
      const int nvert = __builtin_amdgcn_readlane(vfirst + __popc(edges), 63);
      const int tfirst = offsets.tri(blk), vbase = __builtin_amdgcn_readlane(vb, 0);
      int bx, by, bz;
      unpack_key(m.block_keys[blk], bx, by, bz);
      __builtin_memcpy(&S.cases[lane * 8], cur.w, 16);
      mc_list_triangles(S.tri, nt, end, 0);
      mc_list_vertices(S.vert, edges, vfirst, 0);
      if (lane < 8) S.vbase[lane] = vb;
#pragma unroll
      for (int x = 0; x < 8; ++x) S.vi[mc_cube_at(x, lane & 7, lane >> 3)] = (uint16_t)info.at(x);
      mc_stage_halo(ih, S.vi, [](uint16_t w) { return w; });
      v.stage(S.sdf);
      for (int done = 0; done < nvert; done += kVertList) {
        if (done > 0) mc_list_vertices(S.vert, edges, vfirst, done);
        mc_wave_sync();
        mc_vertex_flush<VT>(S, bx, by, bz, m.voxel_size, vbase + done, min(kVertList, nvert - done), verts, vcap);
        mc_wave_sync();
      }
      for (int done = 0; done < ntri; done += kTriList) {
        if (done > 0) mc_list_triangles(S.tri, nt, end, done);
        mc_wave_sync();
        mc_index_flush(S, T, tfirst + done, min(kTriList, ntri - done), tris, tcap);
        mc_wave_sync();
      }
    }
    blk = next;
  }
}

}  // namespace

struct yas_mesher {
  yas_ctx* ctx;
  int max_tri;
  float* tris;      // soup: 9 floats per triangle; indexed: 3 ints per triangle
  float* normals;   // soup: 9 floats per triangle; indexed: 3 floats per vertex
  char* records;    // the arrays below to nbr, in one allocation
  int2* counts;     // per block {triangles, vertices}
  int2* offsets;    // exclusive prefix of counts within a chunk
  unsigned long long* chunk;  // exclusive prefix of 1024-block chunks, {triangles, vertices}
  int16_t* cases;   // per voxel cube index
  uint16_t* vinfo;  // per voxel (local vertex prefix << 3 | owned edges)
  int* nbr;         // per block, pool indices of it and its 7 +x/+y/+z neighbours (-1 absent)
  int block_cap;
  unsigned* done;   // the scan's finished workgroups
  McTotals* total;  // host memory
  int num_blocks;
  int num_tri;
  int num_vert;
  int indexed;
  yas_map* map;
};

// The records' arrays for n blocks in one allocation from `base` (or its size
// alone, for a null base).
static size_t carve_records(yas_mesher* me, char* base, int n) {
  size_t at = 0;
  auto take = [&](auto*& p, size_t bytes) {
    p = base ? (std::remove_reference_t<decltype(p)>)(base + at) : nullptr;
    at += (bytes + 255) & ~(size_t)255;
  };
  take(me->counts, sizeof(int2) * n);
  take(me->offsets, sizeof(int2) * n);
  take(me->chunk, sizeof(*me->chunk) * ((n + kMcChunk - 1) / kMcChunk));
  take(me->cases, sizeof(int16_t) * 512 * (size_t)n);
  take(me->vinfo, sizeof(uint16_t) * 512 * (size_t)n);
  take(me->nbr, sizeof(int) * 8 * (size_t)n);
  return at;
}
// Records for `need` blocks; where an engine outgrows those that it has, for a
// quarter more, at most `most`, if there is room for them.  A new engine's
// first extraction of 58k blocks takes 0.27 ms, 0.21 ms of it the passes (0.35
// ms with six allocations and the quarter more from the start).
static int ensure_block_cap(yas_mesher* me, int need, int most) {
  if (need <= me->block_cap) return YAS_OK;
  int n = me->block_cap ? (int)std::min<long long>(most, (long long)need + need / 4) : need;
  hipFree(me->records);
  me->records = nullptr;
  me->block_cap = 0;
  hipError_t e = hipMalloc((void**)&me->records, carve_records(me, nullptr, n));
  if (e != hipSuccess && n > need) {
    (void)hipGetLastError();
    n = need;
    e = hipMalloc((void**)&me->records, carve_records(me, nullptr, n));
  }
  if (e != hipSuccess) {
    yas_set_error("yas_mesh_extract: the records of %d blocks: %s", n, hipGetErrorString(e));
    return YAS_E_HIP;
  }
  carve_records(me, me->records, n);
  me->block_cap = n;
  return YAS_OK;
}

// Workgroups of an emission pass: as many as the device holds at once, each
// wavefront taking blocks in turn, for the records' capacity.
static int emit_groups(yas_mesher* me, const void* kernel, int* groups) {
  int per = 0;
  YAS_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, kMcThreads, 0));
  const int all = (me->block_cap + kMcWaves - 1) / kMcWaves, fit = std::max(1, per) * me->ctx->cus;
  *groups = std::min(all, fit);
  return YAS_OK;
}

template <class VT>
static int launch_extract(yas_mesher* me, const MapView& v) {
  hipStream_t s = me->ctx->stream;
  const int cap = me->block_cap;
  const McOffsets off = {me->offsets, me->chunk};
  int groups = 0, rc;
  hipLaunchKernelGGL(k_mc_count<VT>, dim3((cap + kMcWaves - 1) / kMcWaves), dim3(kMcThreads), 0, s, v, cap, me->counts, me->cases, me->vinfo,
                     me->nbr);
  YAS_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_mc_scan, dim3((cap + kMcChunk - 1) / kMcChunk), dim3(kMcChunk), 0, s, v, cap,
                     (const int2*)me->counts, me->offsets, me->chunk, me->total, me->done);
  YAS_LAUNCH_CHECK();
  if (me->indexed) {
    // triangle indices in the soup buffer (3 of its 9 floats per triangle),
    // vertices in the normal buffer (capacity max_tri * 3 vertices)
    if ((rc = emit_groups(me, (const void*)k_mc_emit_indexed<VT>, &groups))) return rc;
    hipLaunchKernelGGL(k_mc_emit_indexed<VT>, dim3(groups), dim3(kMcThreads), 0, s, v, cap, off,
                       (const int16_t*)me->cases, (const uint16_t*)me->vinfo, me->normals, me->max_tri * 3,
                       (int*)me->tris, me->max_tri, (const int*)me->nbr);
  } else {
    if ((rc = emit_groups(me, (const void*)k_mc_emit<VT>, &groups))) return rc;
    hipLaunchKernelGGL(k_mc_emit<VT>, dim3(groups), dim3(kMcThreads), 0, s, v, cap, off, (const int16_t*)me->cases,
                       me->tris, me->normals, me->max_tri, (const int*)me->nbr);
  }
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}

// Extraction of every allocated block of `map`, waited for: num_blocks,
// num_tri and num_vert.  The passes read the block count themselves and write
// the totals to host memory, so one wait serves for both (asking for the
// count first cost some 25 us); a volume that outgrew the records is extracted
// again.
static int extract(yas_mesher* me, yas_map* map, bool indexed) {
  YAS_REQUIRE(me && map, "yas_mesh_extract: null argument");
  YAS_REQUIRE_ACTIVE(map);
  YAS_REQUIRE(yas_map_ctx(map)->stream == me->ctx->stream, "yas_mesh_extract: map and mesher must share a stream");
  YAS_HIP(hipSetDevice(me->ctx->device));
  me->num_blocks = me->num_tri = me->num_vert = 0;
  me->map = map;
  me->indexed = indexed;
  const MapView v = yas_map_view(map);
  int rc;
  if (me->block_cap == 0) {
    yas_map_stats st;
    if ((rc = yas_map_get_stats(map, &st))) return rc;
    if (st.num_allocated == 0) return YAS_OK;
    if ((rc = ensure_block_cap(me, st.num_allocated, v.num_blocks))) return rc;
  }
  for (;;) {
    switch (v.format) {
      case YAS_VOXEL_I16_U8: rc = launch_extract<VoxI16>(me, v); break;
      case YAS_VOXEL_F16_U16: rc = launch_extract<VoxF16>(me, v); break;
      default: rc = launch_extract<VoxF32>(me, v);
    }
    if (rc) return rc;
    YAS_HIP(hipStreamSynchronize(me->ctx->stream));
    if (me->total->blocks <= me->block_cap) break;
    if ((rc = ensure_block_cap(me, me->total->blocks, v.num_blocks))) return rc;
  }
  me->num_blocks = me->total->blocks;
  me->num_tri = me->total->tri;
  me->num_vert = me->total->vert;
  return YAS_OK;
}

// Host copies of the last indexed extraction (for file writers).
int yas_mesher_indexed_host(yas_mesher* me, std::vector<float>& verts, std::vector<int32_t>& tris) {
  YAS_REQUIRE(me && me->indexed, "no indexed extraction to write");
  const int nv = me->num_vert < me->max_tri * 3 ? me->num_vert : me->max_tri * 3;
  const int nt = me->num_tri < me->max_tri ? me->num_tri : me->max_tri;
  verts.resize((size_t)nv * 3);
  tris.resize((size_t)nt * 3);
  if (nv > 0) YAS_HIP(hipMemcpy(verts.data(), me->normals, sizeof(float) * 3 * (size_t)nv, hipMemcpyDeviceToHost));
  if (nt > 0) YAS_HIP(hipMemcpy(tris.data(), me->tris, sizeof(int32_t) * 3 * (size_t)nt, hipMemcpyDeviceToHost));
  return YAS_OK;
}

extern "C" {

int yas_mesher_create(yas_ctx* ctx, int max_triangles, yas_mesher** out) {
  YAS_REQUIRE(ctx && out && max_triangles > 0, "yas_mesher_create: bad argument");
  YAS_HIP(hipSetDevice(ctx->device));
  yas_mesher* me = new yas_mesher();
  std::memset(me, 0, sizeof(*me));
  me->ctx = yas_ctx_retain(ctx);
  me->max_tri = max_triangles;
  hipError_t e = hipMalloc((void**)&me->tris, sizeof(float) * 9 * (size_t)max_triangles);
  if (e == hipSuccess) e = hipMalloc((void**)&me->normals, sizeof(float) * 9 * (size_t)max_triangles);
  if (e == hipSuccess) e = hipHostMalloc((void**)&me->total, sizeof(McTotals), hipHostMallocDefault);
  if (e == hipSuccess) e = hipMalloc((void**)&me->done, sizeof(unsigned));
  // on the context's stream, which the null stream need not be in order with
  if (e == hipSuccess) e = hipMemsetAsync(me->done, 0, sizeof(unsigned), ctx->stream);
  if (e != hipSuccess) {
    yas_set_error("yas_mesher_create: %s", hipGetErrorString(e));
    yas_mesher_destroy(me);
    return YAS_E_HIP;
  }
  *me->total = McTotals{0, 0, 0};
  *out = me;
  return YAS_OK;
}

int yas_mesher_destroy(yas_mesher* me) {
  if (!me) return YAS_OK;
  hipSetDevice(me->ctx->device);
  hipStreamSynchronize(me->ctx->stream);
  hipFree(me->tris);
  hipFree(me->normals);
  hipFree(me->records);
  hipHostFree(me->total);
  hipFree(me->done);
  yas_ctx_release(me->ctx);
  delete me;
  return YAS_OK;
}

int yas_mesh_extract(yas_mesher* me, yas_map* map, int* num_triangles) {
  if (num_triangles) *num_triangles = 0;
  int rc = extract(me, map, false);
  if (rc) return rc;
  if (num_triangles) *num_triangles = me->num_tri;
  if (me->num_tri > me->max_tri) {
    yas_set_error("yas_mesh_extract: %d triangles exceed the capacity %d", me->num_tri, me->max_tri);
    return YAS_E_CAPACITY;
  }
  return YAS_OK;
}

int yas_mesh_extract_indexed(yas_mesher* me, yas_map* map, int* num_vertices, int* num_triangles) {
  if (num_vertices) *num_vertices = 0;
  if (num_triangles) *num_triangles = 0;
  int rc = extract(me, map, true);
  if (rc) return rc;
  const int vcap = me->max_tri * 3;
  if (num_vertices) *num_vertices = me->num_vert;
  if (num_triangles) *num_triangles = me->num_tri;
  if (me->num_tri > me->max_tri || me->num_vert > vcap) {
    yas_set_error("yas_mesh_extract_indexed: %d triangles / %d vertices exceed the capacity %d / %d", me->num_tri,
                  me->num_vert, me->max_tri, vcap);
    return YAS_E_CAPACITY;
  }
  return YAS_OK;
}

int yas_mesher_download(yas_mesher* me, float* vertices, float* normals, int capacity) {
  YAS_REQUIRE(me, "null mesher");
  YAS_REQUIRE(!me->indexed, "yas_mesher_download: the last extraction was indexed");
  int n = me->num_tri < me->max_tri ? me->num_tri : me->max_tri;
  if (n > capacity) n = capacity;
  if (n <= 0) return YAS_OK;
  if (vertices) YAS_HIP(hipMemcpy(vertices, me->tris, sizeof(float) * 9 * (size_t)n, hipMemcpyDeviceToHost));
  if (normals) YAS_HIP(hipMemcpy(normals, me->normals, sizeof(float) * 9 * (size_t)n, hipMemcpyDeviceToHost));
  return YAS_OK;
}

int yas_mesher_download_indexed(yas_mesher* me, float* vertices, int32_t* triangles, int vertex_capacity,
                                int triangle_capacity) {
  YAS_REQUIRE(me, "null mesher");
  YAS_REQUIRE(me->indexed, "yas_mesher_download_indexed: the last extraction was not indexed");
  int nv = me->num_vert < me->max_tri * 3 ? me->num_vert : me->max_tri * 3;
  int nt = me->num_tri < me->max_tri ? me->num_tri : me->max_tri;
  if (nv > vertex_capacity) nv = vertex_capacity;
  if (nt > triangle_capacity) nt = triangle_capacity;
  if (vertices && nv > 0) YAS_HIP(hipMemcpy(vertices, me->normals, sizeof(float) * 3 * (size_t)nv, hipMemcpyDeviceToHost));
  if (triangles && nt > 0) YAS_HIP(hipMemcpy(triangles, me->tris, sizeof(int32_t) * 3 * (size_t)nt, hipMemcpyDeviceToHost));
  return YAS_OK;
}

int yas_mesher_indexed_device(yas_mesher* me, const float** vertices, const int32_t** triangles) {
  YAS_REQUIRE(me && me->indexed, "yas_mesher_indexed_device: no indexed extraction");
  if (vertices) *vertices = me->normals;
  if (triangles) *triangles = (const int32_t*)me->tris;
  return YAS_OK;
}

int yas_mesher_blocks(yas_mesher* me, int32_t* keys, int32_t* first, int32_t* count, int16_t* cases, int capacity,
                      int* num_blocks) {
  YAS_REQUIRE(me, "null mesher");
  if (num_blocks) *num_blocks = me->num_blocks;
  int n = me->num_blocks < capacity ? me->num_blocks : capacity;
  if (n <= 0 || !me->map) return YAS_OK;
  YAS_HIP(hipStreamSynchronize(me->ctx->stream));
  if (keys) {
    MapView v = yas_map_view(me->map);
    std::vector<unsigned long long> k(n);
    YAS_HIP(hipMemcpy(k.data(), v.block_keys, sizeof(unsigned long long) * n, hipMemcpyDeviceToHost));
    for (int i = 0; i < n; ++i) unpack_key(k[i], keys[3 * i], keys[3 * i + 1], keys[3 * i + 2]);
  }
  if (first || count) {
    std::vector<int2> o(n), c(n);
    std::vector<unsigned long long> chunk((n + kMcChunk - 1) / kMcChunk);
    YAS_HIP(hipMemcpy(chunk.data(), me->chunk, sizeof(chunk[0]) * chunk.size(), hipMemcpyDeviceToHost));
    YAS_HIP(hipMemcpy(o.data(), me->offsets, sizeof(int2) * n, hipMemcpyDeviceToHost));
    YAS_HIP(hipMemcpy(c.data(), me->counts, sizeof(int2) * n, hipMemcpyDeviceToHost));
    for (int i = 0; i < n; ++i) {
      if (first) first[i] = o[i].x + (int)(unsigned)chunk[i >> kMcChunkShift];
      if (count) count[i] = c[i].x;
    }
  }
  if (cases) YAS_HIP(hipMemcpy(cases, me->cases, sizeof(int16_t) * 512 * (size_t)n, hipMemcpyDeviceToHost));
  return YAS_OK;
}

}  // extern "C"
