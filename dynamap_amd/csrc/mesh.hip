// Marching cubes over the allocated blocks of a volume
// (include/geometry/mesh/meshExtractor/meshExtractor.cu:22-242, 364-402).
//
// Output order is canonical: blocks in hash (bucket, slot) order, the 512
// cells of a block in x-major local order, the triangles of a cell in table
// order -- the order of the CPU restatement, independent of scheduling.
//
// Passes (all on the volume's stream):
//   1. gather the per-bucket occupancy counts, exclusive-scan them, and write
//      the pool index of every occupied slot at its canonical position;
//   2. k_mc_count: one wavefront per block.  The block's voxels plus a
//      one-voxel halo (10^3 sdf values, and bit rows of observed and sign) are
//      staged in LDS; cells that can hold a surface are listed, take their 8
//      strict trilinear corner samples from there and store their cube index
//      (0 = no triangles), and the block's triangles are summed;
//   3. exclusive scan of the per-block counts;
//   4. k_mc_emit: blocks with triangles recompute the corner samples of their
//      cells, scan the cells' counts, and write positions, colours and edge ids
//      at their canonical offset.
// Cell rules (K): cell centre g * vs, corners at +-vs/2, strict trilinear
// samples (any corner voxel of weight 0 gives no sample), the reference's
// corner-bit convention, Bourke's tables, the 1e-5 snaps of
// VertexInterpolation, the centre voxel's colour.  The float operations are
// those of the restatement in the same order, so positions are bit-identical.
#include <string.h>
#include <algorithm>
#include <mutex>
#include <vector>
#include "dm_device.h"
#include "dm_session.h"
#include "mc_table.h"
#include "dm_scan.h"

namespace dm {

__constant__ uint64_t c_mc_tri[256] = {DM_MC_TRI_TABLE};
static const uint64_t h_mc_tri[256] = {DM_MC_TRI_TABLE};

// corner index ci = 4a + 2b + c for the offset (a, b, c) in {-, +}^3; edge
// endpoints and the cube-index bit of each corner (meshExtractor.cu:181-189)
__constant__ int8_t c_edge_a[12] = {2, 6, 4, 0, 3, 7, 5, 1, 2, 6, 4, 0};
__constant__ int8_t c_edge_b[12] = {6, 4, 0, 2, 7, 5, 1, 3, 3, 7, 5, 1};
__constant__ int8_t c_edge_axis[12] = {0, 1, 0, 1, 0, 1, 0, 1, 2, 2, 2, 2};
__constant__ uint8_t c_corner_bit[8] = {8, 128, 1, 16, 4, 64, 2, 32};

constexpr int kHalo = 10;         // block edge + one voxel each side

__global__ __launch_bounds__(256) void k_gather_counts(const DmView *__restrict__ vp, int *__restrict__ counts) {
  const DmView &v = *vp;
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b < v.num_buckets) counts[b] = bucket_count(v, bucket_ptr(v, b));
}

// pool index of every occupied slot at its (bucket, slot) rank
__global__ __launch_bounds__(256) void k_block_list(const DmView *__restrict__ vp, const long long *__restrict__ offs,
                                                   int *__restrict__ list) {
  const DmView &v = *vp;
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b >= v.num_buckets) return;
  const uint8_t *bk = bucket_ptr(v, b);
  const int cnt = bucket_count(v, bk);
  const int32_t *ptrs = (const int32_t *)(bk + 8 * v.bucket_size);
  const long long o = offs[b];
  for (int s = 0; s < cnt; ++s) list[o + s] = ptrs[s];
}

// ---------------------------------------------------------------- cells
struct BoxArg {
  int use;
  double lo[3], hi[3];
};

// Each corner sample is TrilinearInterpolation (meshExtractor.cu:22-93), strict:
// none when any of its 8 voxels is unobserved.  The samples sit at c +- vs/2 per
// axis, and every per-axis quantity of the interpolation (the voxel indices of
// dual = p - vs/2 and dual + vs, the weight p/vs - floor(p/vs)) depends only
// on the axis, the cell's coordinate on it and the sign: 48 values per block,
// evaluated once by 48 lanes, where each cell combines 6 of them with the same
// arithmetic as interpolating each corner on its own.
struct AxisCorner {
  float p;     // corner coordinate c +- vs/2
  int i0, i1;  // voxel indices of dual + 0 and dual + vs
  float w;     // trilinear weight
};
__device__ __forceinline__ AxisCorner axis_corner(float c, float off, float vs) {
  AxisCorner a;
  a.p = c + off;
  const float dual = a.p - vs / 2.f;
  a.i0 = world_to_voxel(dual + 0.f, vs);
  a.i1 = world_to_voxel(dual + vs, vs);
  const float vp = a.p / vs;
  a.w = vp - floorf(vp);
  return a;
}

// A wavefront holds one block: its voxels and a one-voxel halo, the per-axis
// corner values, and the list of cells that are worth evaluating.  rows[r] has,
// for the 10 voxels of row r = (x + 1) * 10 + (y + 1), observed in bits 0..9,
// sdf >= 0 in 10..19 and sdf <= -1e-30 in 20..29.
constexpr uint32_t kRowObs = 1u, kRowPos = 1u << 10, kRowNeg = 1u << 20;
struct Cells {
  float sdf[kHalo * kHalo * kHalo];
  uint32_t rows[kHalo * kHalo];
  AxisCorner ax[3][8][2];  // [axis][cell][sign]
  uint16_t list[kBlockVox];
};
constexpr int kMcWaves = 4;  // wavefronts per workgroup

// Loads the block.  False when no cell can give a triangle: on every axis one of a
// cell's corner indices lies in the cell's block (regular or not, at any block
// key), so some sample reads a voxel of the block, and a block without an observed
// voxel is left before its halo is read.  `regular`: every cell samples exactly its own
// voxel and the 26 around it, with weights in [0.25, 0.75] (true but for
// coordinates so large that rounding moves them).
__device__ __forceinline__ bool load_cells(const DmView &v, int ptr, Cells &C, bool &regular) {
  const int lane = threadIdx.x & 63;
  const int4 key = v.block_key[ptr];
  const uint64_t *own = v.vox + (size_t)ptr * kBlockVox;
  uint64_t w[8];
#pragma unroll
  for (int x = 0; x < 8; ++x) w[x] = ldg(own + 64 * x + lane);
  int nb = -1;
  if (lane < 27) nb = find_block(v, key.x + lane % 3 - 1, key.y + (lane / 3) % 3 - 1, key.z + lane / 9 - 1);
  bool any = false;
#pragma unroll
  for (int x = 0; x < 8; ++x) any |= (w[x] >> 56) != 0;
  if (!__ballot(any)) return false;
  // the halo: 128 ends of the block's own rows, then 36 whole rows of 10
  uint64_t hw[8];
  int hr[8], hz[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int e = min(64 * k + lane, 487);
    int x, y, z;
    if (k < 2) {
      x = 1 + (e >> 4);
      y = 1 + ((e >> 1) & 7);
      z = (e & 1) * 9;
    } else {
      const int q = (e - 128) / 10;
      z = (e - 128) - 10 * q;
      x = q < 20 ? (q < 10 ? 0 : 9) : 1 + ((q - 20) >> 1);
      y = q < 20 ? (q < 10 ? q : q - 10) : (q & 1) * 9;
    }
    const int o = (x + 7) / 8 + 3 * ((y + 7) / 8) + 9 * ((z + 7) / 8);
    const int hp = __shfl(nb, o, 64);
    const uint64_t word = ldg(v.vox + ((size_t)(hp >= 0 ? hp : ptr) * kBlockVox + ((x + 7) & 7) * 64 +
                                       ((y + 7) & 7) * 8 + ((z + 7) & 7)));
    hw[k] = hp >= 0 ? word : 0ull;
    hr[k] = x * 10 + y;
    hz[k] = z;
  }
  const float vs = v.voxel_size;
  bool ok = true;
  if (lane < 48) {
    const int axis = lane >> 4, l = (lane >> 1) & 7, sign = lane & 1;
    const int g = (axis == 0 ? key.x : axis == 1 ? key.y : key.z) * 8 + l;
    const float P = vs / 2.f;
    const AxisCorner a = axis_corner((float)g * vs + 0.f, sign ? P : -P, vs);
    C.ax[axis][l][sign] = a;
    ok = a.i0 == g - 1 + sign && a.i1 == g + sign && a.w >= 0.25f && a.w <= 0.75f;
  }
  regular = __ballot(!ok) == 0;
  for (int r = lane; r < kHalo * kHalo; r += 64) C.rows[r] = 0;
  wave_lds();
  // the block's own rows: lane = 8 y + z, so a ballot's byte y is a row
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    const float s = vox_sdf(w[x]);
    const int sh = lane & 56;
    const uint32_t o = (uint32_t)(__ballot((w[x] >> 56) != 0) >> sh) & 0xFF;
    const uint32_t p = (uint32_t)(__ballot(s >= 0.f) >> sh) & 0xFF;
    const uint32_t n = (uint32_t)(__ballot(s <= -1e-30f) >> sh) & 0xFF;
    const int r = (x + 1) * 10 + (lane >> 3) + 1;
    C.sdf[r * 10 + (lane & 7) + 1] = s;
    if ((lane & 7) == 0) C.rows[r] = (o << 1) | (p << 11) | (n << 21);
  }
  wave_lds();
#pragma unroll
  for (int k = 0; k < 8; ++k)
    if (64 * k + lane < 488) {
      const float s = vox_sdf(hw[k]);
      C.sdf[hr[k] * 10 + hz[k]] = s;
      const uint32_t bits = ((hw[k] >> 56) ? kRowObs : 0u) | (s >= 0.f ? kRowPos : 0u) | (s <= -1e-30f ? kRowNeg : 0u);
      atomicOr(&C.rows[hr[k]], bits << hz[k]);
    }
  wave_lds();
  return true;
}

// Lists the block's cells whose 27 voxels are all observed and neither all
// >= 0 (every corner sample is then >= 0: cube 0) nor all below zero (cube
// 255), in cell order; all cells of a block that is not regular.
__device__ __forceinline__ int list_cells(Cells &C, bool regular) {
  const int lane = threadIdx.x & 63, y = lane >> 3, z = lane & 7;
  uint32_t m[kHalo];
#pragma unroll
  for (int x = 0; x < kHalo; ++x) m[x] = C.rows[x * 10 + y] & C.rows[x * 10 + y + 1] & C.rows[x * 10 + y + 2];
  const uint64_t below = ((uint64_t)1 << lane) - 1;
  int n = 0;
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    const uint32_t t = (m[x] & m[x + 1] & m[x + 2]) >> z;
    const bool take = !regular || ((t & 7) == 7 && ((t >> 10) & 7) != 7 && ((t >> 20) & 7) != 7);
    const uint64_t b = __ballot(take);
    if (take) C.list[n + __popcll(b & below)] = (uint16_t)(64 * x + lane);
    n += __popcll(b);
  }
  wave_lds();
  return n;
}

// The 8 corner samples of a listed cell of a regular block.
__device__ __forceinline__ int cell_samples(const Cells &C, int li, float *d) {
  const int lx = li >> 6, ly = (li >> 3) & 7, lz = li & 7;
  float s[27];
#pragma unroll
  for (int k = 0; k < 27; ++k) s[k] = C.sdf[(lx + k / 9) * 100 + (ly + (k / 3) % 3) * 10 + lz + k % 3];
  const float wx[2] = {C.ax[0][lx][0].w, C.ax[0][lx][1].w}, wy[2] = {C.ax[1][ly][0].w, C.ax[1][ly][1].w},
              wz[2] = {C.ax[2][lz][0].w, C.ax[2][lz][1].w};
  // sample k: offsets (0,0,0) (1,0,0) (0,1,0) (0,0,1) (1,1,0) (0,1,1) (1,0,1) (1,1,1)
  constexpr uint8_t cxm = 0xD2, cym = 0xB4, czm = 0xE8;
  int cube = 0;
#pragma unroll
  for (int ci = 0; ci < 8; ++ci) {
    const int cx = (ci >> 2) & 1, cy = (ci >> 1) & 1, cz = ci & 1;
    float dd = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int ox = (cxm >> k) & 1, oy = (cym >> k) & 1, oz = (czm >> k) & 1;
      const float a = ox ? wx[cx] : 1.f - wx[cx];
      const float b = oy ? wy[cy] : 1.f - wy[cy];
      const float g = oz ? wz[cz] : 1.f - wz[cz];
      dd += a * b * g * s[(cx + ox) * 9 + (cy + oy) * 3 + cz + oz];
    }
    d[ci] = dd;
    if (dd < 0.f) cube += c_corner_bit[ci];
  }
  return cube;
}

// Voxel at global index g: from the halo when inside it, else from the table.
__device__ __forceinline__ bool halo_voxel(const DmView &v, const Cells &C, int4 key, int gx, int gy, int gz,
                                           float &sdf) {
  const int hx = gx - 8 * key.x + 1, hy = gy - 8 * key.y + 1, hz = gz - 8 * key.z + 1;
  if ((unsigned)hx < kHalo && (unsigned)hy < kHalo && (unsigned)hz < kHalo) {
    sdf = C.sdf[hx * 100 + hy * 10 + hz];
    return (C.rows[hx * 10 + hy] >> hz) & 1;
  }
  BlockCache bc;
  bc.init();
  const uint64_t w = voxel_at(v, gx, gy, gz, bc);
  sdf = vox_sdf(w);
  return (w >> 56) != 0;
}

// The same samples for any indices and weights; -1 when a sample is missing.
__device__ __noinline__ int cell_samples_any(const DmView &v, const Cells &C, int4 key, int li, float *d, int stride) {
  const AxisCorner *X = C.ax[0][li >> 6], *Y = C.ax[1][(li >> 3) & 7], *Z = C.ax[2][li & 7];
  constexpr uint8_t cxm = 0xD2, cym = 0xB4, czm = 0xE8;
  int cube = 0;
#pragma unroll 1
  for (int ci = 0; ci < 8; ++ci) {
    const AxisCorner ax = X[(ci >> 2) & 1], ay = Y[(ci >> 1) & 1], az = Z[ci & 1];
    float dd = 0.f;
#pragma unroll 1
    for (int k = 0; k < 8; ++k) {
      const bool ox = (cxm >> k) & 1, oy = (cym >> k) & 1, oz = (czm >> k) & 1;
      float sv;
      if (!halo_voxel(v, C, key, ox ? ax.i1 : ax.i0, oy ? ay.i1 : ay.i0, oz ? az.i1 : az.i0, sv)) return -1;
      const float a = ox ? ax.w : 1.f - ax.w;
      const float b = oy ? ay.w : 1.f - ay.w;
      const float g = oz ? az.w : 1.f - az.w;
      dd += a * b * g * sv;
    }
    if (d) d[ci * stride] = dd;
    if (dd < 0.f) cube += c_corner_bit[ci];
  }
  return cube;
}

__device__ __forceinline__ bool outside_box(const BoxArg &box, int gx, int gy, int gz, float vs) {
  const f3 c = mk((float)gx * vs + 0.f, (float)gy * vs + 0.f, (float)gz * vs + 0.f);
  return (double)c.x < box.lo[0] || (double)c.y < box.lo[1] || (double)c.z < box.lo[2] ||
         (double)c.x > box.hi[0] || (double)c.y > box.hi[1] || (double)c.z > box.hi[2];
}

// Bound by memory latency (the block's key, its neighbours' pool entries,
// then their voxels), so a block takes one wavefront with all its loads in
// flight, and as many blocks as registers and LDS allow are resident.  Cells
// without a sign change or with an unobserved voxel, nearly all, are dropped
// on bit masks; the others are packed into full wavefronts.  Room at 8 mm 353 ->
// 43 us, at 2 cm 42 -> 10 (against 512 threads per block evaluating every cell).
__global__ __launch_bounds__(64 * kMcWaves) void k_mc_count(const DmView *__restrict__ vp, const int *__restrict__ list,
                                                           int n, BoxArg box, uint8_t *__restrict__ cubes,
                                                           int *__restrict__ block_tri) {
  __shared__ Cells S[kMcWaves];
  __shared__ uint64_t out[kMcWaves][kBlockVox / 8];
  const DmView &v = *vp;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int blk = blockIdx.x * kMcWaves + wave;
  if (blk >= n) return;
  Cells &C = S[wave];
  const int ptr = list[blk];
  bool regular;
  int cells = 0;
  if (load_cells(v, ptr, C, regular)) cells = list_cells(C, regular);
  int ntri = 0;
  if (cells) {
    const int4 key = v.block_key[ptr];
    uint8_t *cb = (uint8_t *)out[wave];
    out[wave][lane] = 0;
    wave_lds();
    for (int k = lane; k < cells; k += 64) {
      const int li = C.list[k];
      if (box.use &&
          outside_box(box, key.x * 8 + (li >> 6), key.y * 8 + ((li >> 3) & 7), key.z * 8 + (li & 7), v.voxel_size))
        continue;
      float d[8];
      const int cube = regular ? cell_samples(C, li, d) : cell_samples_any(v, C, key, li, nullptr, 0);
      const int nt = cube > 0 ? mc_num_tri(c_mc_tri[cube]) : 0;
      if (nt) cb[li] = (uint8_t)cube;
      ntri += nt;
    }
    wave_lds();
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ntri += __shfl_xor(ntri, o, 64);
    if (ntri) ((uint64_t *)(cubes + (size_t)blk * kBlockVox))[lane] = out[wave][lane];  // else never read
  }
  if (lane == 0) block_tri[blk] = ntri;
}

// VertexInterpolation at isolevel 0 (meshExtractor.cu:95-123)
__device__ __forceinline__ f3 vertex_interp(f3 p1, f3 p2, float d1, float d2) {
  const float eps = 0.00001f;
  if (fabsf(0.f - d1) < eps) return p1;
  if (fabsf(0.f - d2) < eps) return p2;
  if (fabsf(d1 - d2) < eps) return p1;
  const float mu = (0.f - d1) / (d2 - d1);
  return mk(p1.x + mu * (p2.x - p1.x), p1.y + mu * (p2.y - p1.y), p1.z + mu * (p2.z - p1.z));
}

__device__ __forceinline__ uint64_t edge_id(int gx, int gy, int gz, int e) {
  const int a = c_edge_a[e], b = c_edge_b[e];
  const int lo = a < b ? a : b;
  const int cx = gx + ((lo >> 2) & 1), cy = gy + ((lo >> 1) & 1), cz = gz + (lo & 1);
  const uint64_t off = 1u << 19, m = (1u << 20) - 1;
  return ((uint64_t)c_edge_axis[e] << 60) | ((((uint64_t)(cx + (int)off)) & m) << 40) |
         ((((uint64_t)(cy + (int)off)) & m) << 20) | (((uint64_t)(cz + (int)off)) & m);
}

// A wavefront per block with triangles.  64 of its cells at a time leave their
// corner samples in LDS; then a lane takes a vertex, so that neighbouring
// lanes write neighbouring vertices.  At 8 mm 82 -> 33 us, at 2 cm 36 -> 20
// (against a lane per cell writing its triangles one by one).
__global__ __launch_bounds__(64 * kMcWaves) void k_mc_emit(const DmView *__restrict__ vp, const int *__restrict__ list,
                                                          int n, const uint8_t *__restrict__ cubes,
                                                          const int *__restrict__ block_tri,
                                                          const long long *__restrict__ block_off, long long cap,
                                                          float *__restrict__ pos, float *__restrict__ col,
                                                          uint64_t *__restrict__ eid) {
  __shared__ Cells S[kMcWaves];
  __shared__ float D[kMcWaves][8][64];       // [corner][cell of this pass]
  __shared__ uint16_t tri[kMcWaves][64 * 5];  // triangle -> cell of this pass | number in the cell << 8
  const DmView &v = *vp;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int blk = blockIdx.x * kMcWaves + wave;
  if (blk >= n || block_tri[blk] == 0 || block_off[blk] >= cap) return;
  Cells &C = S[wave];
  const int ptr = list[blk];
  const int4 key = v.block_key[ptr];
  const uint8_t *cb = cubes + (size_t)blk * kBlockVox;
  uint8_t cube_of[8];
#pragma unroll
  for (int x = 0; x < 8; ++x) cube_of[x] = ldg(cb + 64 * x + lane);
  bool regular;
  if (!load_cells(v, ptr, C, regular)) return;  // the count pass saw observed voxels
  const uint64_t below = ((uint64_t)1 << lane) - 1;
  int cells = 0;
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    const uint64_t b = __ballot(cube_of[x] != 0);
    if (cube_of[x]) C.list[cells + __popcll(b & below)] = (uint16_t)(64 * x + lane);
    cells += __popcll(b);
  }
  wave_lds();
  long long t0 = block_off[blk];
  for (int c0 = 0; c0 < cells; c0 += 64) {
    const bool have = c0 + lane < cells;
    int nt = 0;
    if (have) {
      const int li = C.list[c0 + lane];
      nt = mc_num_tri(c_mc_tri[cb[li]]);
      if (regular) {
        float d[8];
        cell_samples(C, li, d);
#pragma unroll
        for (int k = 0; k < 8; ++k) D[wave][k][lane] = d[k];
      } else {
        cell_samples_any(v, C, key, li, &D[wave][0][lane], 64);
      }
    }
    int incl = nt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(incl, o, 64);
      if (lane >= o) incl += u;
    }
    for (int k = 0; k < nt; ++k) tri[wave][incl - nt + k] = (uint16_t)(lane | k << 8);
    const int total = __shfl(incl, 63, 64);
    wave_lds();
    const int lim = (int)min((long long)total, cap - t0);  // triangles past cap are not written
    for (int q = lane; q < 3 * lim; q += 64) {
      const int e3 = tri[wave][q / 3], c = e3 & 0xFF, li = C.list[c0 + c];
      const int e = mc_tri_edge(c_mc_tri[cb[li]], 3 * (e3 >> 8) + q % 3);
      const int ea = c_edge_a[e], eb = c_edge_b[e];
      const int lx = li >> 6, ly = (li >> 3) & 7, lz = li & 7;
      const size_t o = (size_t)t0 * 3 + q;
      if (pos) {
        const f3 pa = mk(C.ax[0][lx][(ea >> 2) & 1].p, C.ax[1][ly][(ea >> 1) & 1].p, C.ax[2][lz][ea & 1].p);
        const f3 pb = mk(C.ax[0][lx][(eb >> 2) & 1].p, C.ax[1][ly][(eb >> 1) & 1].p, C.ax[2][lz][eb & 1].p);
        const f3 p = vertex_interp(pa, pb, D[wave][ea][c], D[wave][eb][c]);
        pos[3 * o] = p.x;
        pos[3 * o + 1] = p.y;
        pos[3 * o + 2] = p.z;
      }
      if (col) {
        const uint32_t rgbw = vox_rgbw(v.vox[(size_t)ptr * kBlockVox + li]);
        col[3 * o] = (float)(rgbw & 0xFF) / 255.f;
        col[3 * o + 1] = (float)((rgbw >> 8) & 0xFF) / 255.f;
        col[3 * o + 2] = (float)((rgbw >> 16) & 0xFF) / 255.f;
      }
      if (eid) eid[o] = edge_id(8 * key.x + lx, 8 * key.y + ly, 8 * key.z + lz, e);
    }
    wave_lds();
    t0 += total;
    if (t0 >= cap) break;
  }
}

// ---------------------------------------------------------------- host

// Scratch of dm_mesh_extract_noalloc: one fixed array per device, resident
// until the process ends.  Segments (bytes, each 256-aligned):
//   counts  int32 per bucket            (kNaMaxBuckets)
//   offs    int64 per bucket            (kNaMaxBuckets)
//   wsum1   scan workspace of the buckets
//   list    pool index per allocated block (kNaMaxBlocks)
//   cubes   cube index per cell of a chunk of kNaChunk blocks
//   btri    triangles per block of the chunk
//   boff    triangle offset per block of the chunk
//   wsum2   scan workspace of the chunk
// Every segment is written before it is read within one call, so nothing
// needs clearing between calls.
constexpr int kNaMaxBuckets = 1 << 20;
constexpr int kNaMaxBlocks = 1 << 21;
constexpr int kNaChunk = 1 << 14;
constexpr size_t na_align(size_t b) { return (b + 255) & ~(size_t)255; }
constexpr size_t kNaOffCounts = 0;
constexpr size_t kNaOffOffs = kNaOffCounts + na_align((size_t)kNaMaxBuckets * 4);
constexpr size_t kNaOffWsum1 = kNaOffOffs + na_align((size_t)kNaMaxBuckets * 8);
constexpr size_t kNaOffList = kNaOffWsum1 + na_align((size_t)(kNaMaxBuckets / kScanItems + 2) * 8);
constexpr size_t kNaOffCubes = kNaOffList + na_align((size_t)kNaMaxBlocks * 4);
constexpr size_t kNaOffBtri = kNaOffCubes + na_align((size_t)kNaChunk * kBlockVox);
constexpr size_t kNaOffBoff = kNaOffBtri + na_align((size_t)kNaChunk * 4);
constexpr size_t kNaOffWsum2 = kNaOffBoff + na_align((size_t)kNaChunk * 8);
constexpr size_t kNaScratchBytes = kNaOffWsum2 + na_align((size_t)(kNaChunk / kScanItems + 2) * 8);

static __device__ __align__(256) uint8_t scratch[kNaScratchBytes];

// Device address of `scratch` per device, taken once with that device
// current.  The host-side name of the array is not a device address.
constexpr int kNaMaxDevices = 64;
static std::mutex g_na_mutex;
static uint8_t *g_na_ptr[kNaMaxDevices];

static int na_scratch(int device, uint8_t **out) {
  if (device < 0 || device >= kNaMaxDevices) {
    set_error("dm_mesh_extract_noalloc: device index out of range");
    return DM_E_INVALID;
  }
  std::lock_guard<std::mutex> lock(g_na_mutex);
  if (!g_na_ptr[device]) {
    void *p = nullptr;
    DM_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_na_ptr[device] = (uint8_t *)p;
  }
  *out = g_na_ptr[device];
  return DM_OK;
}

// Makes `device` current for the scope and restores the previous one.
struct DeviceScope {
  int prev = -1;
  int enter(int device) {
    DM_HIP(hipGetDevice(&prev));
    if (prev != device) DM_HIP(hipSetDevice(device));
    return DM_OK;
  }
  ~DeviceScope() {
    int cur = -1;
    if (prev >= 0 && hipGetDevice(&cur) == hipSuccess && cur != prev) (void)hipSetDevice(prev);
  }
};

}  // namespace dm

using namespace dm;
struct dm_volume : Sess {};

extern "C" {

int dm_mc_tri_table(uint64_t *out) {
  if (!out) { set_error("null argument"); return DM_E_INVALID; }
  memcpy(out, h_mc_tri, sizeof h_mc_tri);
  return DM_OK;
}

int dm_mesh_extract(dm_volume *vol, const double *box_lo, const double *box_hi, int64_t cap, float *pos, float *col,
                    uint64_t *edge_ids, int64_t *ntri_out) {
  if (!vol || !ntri_out || cap < 0 || (!box_lo) != (!box_hi)) {
    set_error("dm_mesh_extract: invalid argument");
    return DM_E_INVALID;
  }
  hipStream_t st = vol->stream;
  const int nb = vol->h.num_buckets;
  BoxArg box{};
  box.use = box_lo != nullptr;
  for (int k = 0; k < 3 && box.use; ++k) { box.lo[k] = box_lo[k]; box.hi[k] = box_hi[k]; }
  DevBuf counts, offs, wsum1, list, cubes, btri, boff, wsum2, dpos, dcol, deid;
  if (int rc = dev_alloc(counts, (size_t)nb * 4)) return rc;
  if (int rc = dev_alloc(offs, (size_t)nb * 8)) return rc;
  hipLaunchKernelGGL(k_gather_counts, dim3((nb + 255) / 256), dim3(256), 0, st, vol->d_view, counts.as<int>());
  long long *d_nblk = nullptr;
  if (int rc = scan_ints(counts.as<int>(), nb, offs.as<long long>(), wsum1, st, &d_nblk)) return rc;
  long long nblk = 0;
  DM_HIP(hipMemcpyAsync(&nblk, d_nblk, 8, hipMemcpyDeviceToHost, st));
  DM_HIP(hipStreamSynchronize(st));
  *ntri_out = 0;
  if (nblk == 0) return DM_OK;
  if (nblk > vol->h.num_blocks) {
    set_error("dm_mesh_extract: hash table holds more entries than the pool");
    return DM_E_HIP;
  }
  const int n = (int)nblk;
  if (int rc = dev_alloc(list, (size_t)n * 4)) return rc;
  if (int rc = dev_alloc(cubes, (size_t)n * kBlockVox)) return rc;
  if (int rc = dev_alloc(btri, (size_t)n * 4)) return rc;
  if (int rc = dev_alloc(boff, (size_t)n * 8)) return rc;
  hipLaunchKernelGGL(k_block_list, dim3((nb + 255) / 256), dim3(256), 0, st, vol->d_view, offs.as<long long>(),
                     list.as<int>());
  hipLaunchKernelGGL(k_mc_count, dim3((n + kMcWaves - 1) / kMcWaves), dim3(64 * kMcWaves), 0, st, vol->d_view,
                     list.as<int>(), n, box,
                     cubes.as<uint8_t>(), btri.as<int>());
  DM_HIP(hipGetLastError());
  long long *d_ntri = nullptr;
  if (int rc = scan_ints(btri.as<int>(), n, boff.as<long long>(), wsum2, st, &d_ntri)) return rc;
  long long T = 0;
  DM_HIP(hipMemcpyAsync(&T, d_ntri, 8, hipMemcpyDeviceToHost, st));
  DM_HIP(hipStreamSynchronize(st));
  *ntri_out = T;
  const long long m = std::min<long long>(T, cap);
  if (m == 0 || (!pos && !col && !edge_ids)) return DM_OK;
  if (pos) { if (int rc = dev_alloc(dpos, (size_t)m * 36)) return rc; }
  if (col) { if (int rc = dev_alloc(dcol, (size_t)m * 36)) return rc; }
  if (edge_ids) { if (int rc = dev_alloc(deid, (size_t)m * 24)) return rc; }
  hipLaunchKernelGGL(k_mc_emit, dim3((n + kMcWaves - 1) / kMcWaves), dim3(64 * kMcWaves), 0, st, vol->d_view,
                     list.as<int>(), n,
                     cubes.as<uint8_t>(), btri.as<int>(), boff.as<long long>(), m, dpos.as<float>(),
                     dcol.as<float>(), deid.as<uint64_t>());
  DM_HIP(hipGetLastError());
  if (pos) DM_HIP(hipMemcpyAsync(pos, dpos.p, (size_t)m * 36, hipMemcpyDeviceToHost, st));
  if (col) DM_HIP(hipMemcpyAsync(col, dcol.p, (size_t)m * 36, hipMemcpyDeviceToHost, st));
  if (edge_ids) DM_HIP(hipMemcpyAsync(edge_ids, deid.p, (size_t)m * 24, hipMemcpyDeviceToHost, st));
  DM_HIP(hipStreamSynchronize(st));
  return DM_OK;
}

int dm_mesh_extract_noalloc(dm_volume *vol, const double *box_lo, const double *box_hi, int64_t cap, float *dev_pos,
                            float *dev_col, uint64_t *dev_edge_ids, int64_t *ntri_out) {
  if (!vol || !ntri_out || cap < 0 || (!box_lo) != (!box_hi)) {
    set_error("dm_mesh_extract_noalloc: invalid argument");
    return DM_E_INVALID;
  }
  const int nb = vol->h.num_buckets;
  if (nb > kNaMaxBuckets) {
    set_error("dm_mesh_extract_noalloc: the volume has more than 2^20 hash buckets (use dm_mesh_extract)");
    return DM_E_CAPACITY;
  }
  DeviceScope scope;
  DM_TRY(scope.enter(vol->device));
  uint8_t *base = nullptr;
  DM_TRY(na_scratch(vol->device, &base));
  int *counts = (int *)(base + kNaOffCounts);
  long long *offs = (long long *)(base + kNaOffOffs), *wsum1 = (long long *)(base + kNaOffWsum1);
  int *list = (int *)(base + kNaOffList);
  uint8_t *cubes = base + kNaOffCubes;
  int *btri = (int *)(base + kNaOffBtri);
  long long *boff = (long long *)(base + kNaOffBoff), *wsum2 = (long long *)(base + kNaOffWsum2);

  hipStream_t st = vol->stream;
  BoxArg box{};
  box.use = box_lo != nullptr;
  for (int k = 0; k < 3 && box.use; ++k) { box.lo[k] = box_lo[k]; box.hi[k] = box_hi[k]; }
  hipLaunchKernelGGL(k_gather_counts, dim3((nb + 255) / 256), dim3(256), 0, st, vol->d_view, counts);
  long long *d_total = nullptr;
  DM_TRY(scan_ints_ws(counts, nb, offs, wsum1, st, &d_total));
  long long nblk = 0;
  DM_HIP(hipMemcpyAsync(&nblk, d_total, 8, hipMemcpyDeviceToHost, st));
  DM_HIP(hipStreamSynchronize(st));
  *ntri_out = 0;
  if (nblk == 0) return DM_OK;
  if (nblk > vol->h.num_blocks) {
    set_error("dm_mesh_extract_noalloc: hash table holds more entries than the pool");
    return DM_E_HIP;
  }
  if (nblk > kNaMaxBlocks) {
    set_error("dm_mesh_extract_noalloc: more than 2^21 allocated blocks (use dm_mesh_extract)");
    return DM_E_CAPACITY;
  }
  const int n = (int)nblk;
  hipLaunchKernelGGL(k_block_list, dim3((nb + 255) / 256), dim3(256), 0, st, vol->d_view, offs, list);
  const bool want = dev_pos || dev_col || dev_edge_ids;
  long long T = 0;
  for (int c0 = 0; c0 < n; c0 += kNaChunk) {
    const int cn = std::min(kNaChunk, n - c0);
    hipLaunchKernelGGL(k_mc_count, dim3((cn + kMcWaves - 1) / kMcWaves), dim3(64 * kMcWaves), 0, st, vol->d_view,
                       list + c0, cn, box, cubes, btri);
    DM_HIP(hipGetLastError());
    DM_TRY(scan_ints_ws(btri, cn, boff, wsum2, st, &d_total));
    long long Tc = 0;
    DM_HIP(hipMemcpyAsync(&Tc, d_total, 8, hipMemcpyDeviceToHost, st));
    DM_HIP(hipStreamSynchronize(st));
    const long long m = std::min<long long>(Tc, cap - std::min<long long>(T, cap));
    if (want && m > 0) {
      hipLaunchKernelGGL(k_mc_emit, dim3((cn + kMcWaves - 1) / kMcWaves), dim3(64 * kMcWaves), 0, st, vol->d_view,
                         list + c0, cn, cubes, btri,
                         boff, m, dev_pos ? dev_pos + (size_t)T * 9 : nullptr,
                         dev_col ? dev_col + (size_t)T * 9 : nullptr,
                         dev_edge_ids ? dev_edge_ids + (size_t)T * 3 : nullptr);
      DM_HIP(hipGetLastError());
    }
    T += Tc;
  }
  DM_HIP(hipStreamSynchronize(st));
  *ntri_out = T;
  return DM_OK;
}

}  // extern "C"
