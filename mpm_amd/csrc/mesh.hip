// mesh.hip -- surface mesh of the particles on the GPU: the reference's
// MeshBuilder::computeMesh (include/mesh_builder.h:181-211) with its
// distance field (fillVoxelGrid_distance, mesh_builder.h:103-149).
//
// 1. Distance field on a side^3 voxel grid (voxel_dx = N dx / side): every
//    voxel starts at the cut-off (r + 1) voxel_dx and takes the minimum of
//    |x_p - x_node| over the particles whose box of voxels, truncated as the
//    reference truncates it, reaches it. The particles are binned by blocks of
//    4^3 voxels, and a wavefront per block looks for the nearest one of each
//    of its voxels. A minimum does not depend on the order of the particles.
// 2. The iso-surface S = r voxel_dx - d = 0 (S in FP64 as the reference
//    forms it) by marching cubes. The case table is generated at compile time
//    from the cube's faces: on each face, seen from outside, a segment runs
//    from every edge crossing where the corners go outside -> inside (counter-
//    clockwise) to the next crossing; on a face with four crossings this cuts
//    off each inside corner, and the neighbouring cube, which sees the face
//    from the other side, makes the same cut, so the surface is closed. The
//    segments chain into loops around the inside corners, and each loop is
//    cut into a fan from the first of its vertices whose diagonals do not
//    lie in a face of the cube (a diagonal in a face could meet the
//    neighbour's). Vertices lie on grid edges, linearly interpolated from the
//    edge's lower-index end, so the cubes that share an edge give the same
//    bits; the triangles wind with their normals out of the inside (S > 0).
//    The reference runs libigl's marching cubes (its own case table) on the
//    same field.
// Two passes over the rows of cubes: count the triangles, scan, write them.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_math.hpp"
#include "engine_types.hpp"
#include "kernels.hpp"
#include "mc_table.hpp"

namespace {

// Small boxes or crowded bins (mesh_distance_field has the rule): one thread
// per particle over the voxels of its box, the minimum as an
// integer atomic on the float bits (all distances are >= 0).
__global__ void __launch_bounds__(256)
    k_sdf_scatter(ParticlesDev P, int side, float vdx, float cutoff, uint32_t* __restrict__ sdf) {
#pragma clang fp contract(off)  // the reference's separate roundings, no fused multiply-adds
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P.n) return;
  float x[3];
  int beg[3], end[3];
  const float rg = cutoff / vdx;  // r_gridpoints, mesh_builder.h:124
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    x[a] = P.f[(PL_X + a) * P.stride + p];
    const float xg = x[a] / vdx;
    // (x - r).cast<int>() and (x + r + 1).cast<int>(): truncation, mesh_builder.h:128-129
    beg[a] = max(0, (int)(xg - rg));
    end[a] = min(side, (int)(xg + (rg + 1.0f)));
  }
  // |x - x_node| = sqrt(dx^2 + (dy^2 + dz^2)): Eigen's norm() sums the three
  // squares of a fixed-size vector as e0 + (e1 + e2); x_node = i * voxel_dx
  for (int i = beg[0]; i < end[0]; ++i) {
    const float dx = x[0] - (float)(uint32_t)i * vdx;
    const float dx2 = dx * dx;
    // rows and planes whose nearest voxel is at the cut-off or beyond change
    // nothing: rounding is monotonic, so d^2 >= fl(dx^2 + dy^2) >= dx^2 in
    // float as well
    if (sqrtf(dx2) >= cutoff) continue;
    for (int j = beg[1]; j < end[1]; ++j) {
      const float dy = x[1] - (float)(uint32_t)j * vdx;
      const float dy2 = dy * dy;
      if (sqrtf(dx2 + dy2) >= cutoff) continue;
      const size_t row = ((size_t)i * side + (size_t)j) * side;
      for (int k = beg[2]; k < end[2]; ++k) {
        const float dz = x[2] - (float)(uint32_t)k * vdx;
        const float d = sqrtf(dx2 + (dy2 + dz * dz));
        const uint32_t bits = __float_as_uint(d);
        uint32_t* const cell = sdf + row + (size_t)k;
        if (bits < *cell) atomicMin(cell, bits);
      }
    }
  }
}

constexpr int kBinEdge = 4;  // voxels per bin edge
constexpr double kGatherMaxBox = 36.0;  // box edge, in voxels, up to which the gather runs
// particles in an occupied bin from which on 4 and 16 wavefronts share a block
constexpr double kGatherFew = 100.0, kGatherMany = 1000.0;

__device__ __forceinline__ int voxel_of(float x, float vdx, int side) {  // clamped to the grid (NaN: 0)
  return max(0, min(side - 1, (int)(x / vdx)));
}

constexpr uint32_t kNoBin = 0xffffffffu;

// Bin of 4^3 voxels that holds particle p, the nearest one for a particle past
// the grid; none for one too far off to matter (the hundredth is for rounding),
// or whose position is not a number: a simulation that has come apart would
// crowd the bins at the faces with them (half of 1,000,000 particles: 60 ms).
__device__ __forceinline__ uint32_t bin_of(const ParticlesDev& P, int64_t p, int side, float vdx, float cutoff,
                                           int nb) {
  const float lo = -1.01f * cutoff, hi = (float)(side - 1) * vdx - lo;
  int b[3];
  bool near = true;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float x = P.f[(PL_X + a) * P.stride + p];
    near = near && x >= lo && x <= hi;
    b[a] = voxel_of(x, vdx, side) / kBinEdge;
  }
  return near ? (uint32_t)((b[0] * nb + b[1]) * nb + b[2]) : kNoBin;  // (at most 256^3 bins)
}

// Neighbouring particles mostly share bins (they are in cell order), and the
// atomics of one bin run one after the other (0.2 us each, 5 ms for 1,000,000
// particles in 50 bins): one lane adds for all lanes of its wavefront that
// hold its bin.
__global__ void __launch_bounds__(256)
    k_bin_count(ParticlesDev P, int side, float vdx, float cutoff, int nb, uint32_t* __restrict__ count,
                uint32_t* __restrict__ bins, uint32_t* __restrict__ rank) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const uint32_t bin = p < P.n ? bin_of(P, p, side, vdx, cutoff, nb) : kNoBin;
  const bool valid = bin != kNoBin;
  if (p < P.n) bins[p] = bin;
  uint64_t mine = 0ull, left = __ballot(valid);
  while (left) {
    const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)bin, __ffsll((long long)left) - 1);
    const uint64_t m = __ballot(valid && bin == b);
    if (bin == b) mine = m;
    left &= ~m;
  }
  if (!valid) return;
  const int first = __ffsll((long long)mine) - 1;
  uint32_t base = 0;
  if (lane == first) base = atomicAdd(count + bin, (uint32_t)__popcll(mine));
  base = (uint32_t)__shfl((int)base, first);
  rank[p] = base + (uint32_t)__popcll(mine & ((1ull << lane) - 1ull));
}

// the positions in bin order, as 3 planes of `stride` floats. (The bin is the
// one that was counted: found again from the position it could be another,
// and its place past the arrays, if an advance that the caller did not order
// with this call moves the particle in between.)
__global__ void __launch_bounds__(256)
    k_bin_scatter(ParticlesDev P, const uint32_t* __restrict__ start, const uint32_t* __restrict__ bins,
                  const uint32_t* __restrict__ rank, float* __restrict__ pos, size_t stride) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= P.n) return;
  const uint32_t bin = bins[p];
  if (bin == kNoBin) return;
  const size_t at = start[bin] + rank[p];
#pragma unroll
  for (int a = 0; a < 3; ++a) pos[a * stride + at] = P.f[(PL_X + a) * P.stride + p];
}

// the reference's truncated box of voxels on one axis (mesh_builder.h:124-129):
// (x - r).cast<int>() and (x + r + 1).cast<int>()
__device__ __forceinline__ bool in_box(float x, int i, float vdx, float rg, int side) {
#pragma clang fp contract(off)
  const float xg = x / vdx;
  return i >= max(0, (int)(xg - rg)) && i < min(side, (int)(xg + (rg + 1.0f)));
}

// One wavefront per block of 4^3 voxels, one voxel a lane; start[b] ..
// start[b + 1] are the particles of bin b (the block's own bins and blocks
// coincide). The lanes keep the least squared distance so far, and R2, the
// largest of them over the block, bounds what can still matter: the bins
// around are taken shell by shell until a shell lies beyond it, a bin's
// particles 64 at a time, and only those nearer to the block than R2 are
// given to all lanes (their coordinates through v_readlane). Inside a body a
// block looks at its own and the 26 bins around and evaluates some 40
// particles; a bin is a contiguous range, a shell's ranges are read one a
// lane, and a block with no particle in reach leaves after two loads.
// Pruning changes nothing: every rounding here is monotonic, so a particle's
// squared distance to a voxel is never below the one to the voxels' box, in
// float as well; and the square root of the least is the least square root.
// Bound by the latency of the shells' loads. One thread per particle over the
// ~2,000 voxels of its box with a read and an atomic minimum each took 9.2 ms
// for 1,000,000 particles on 250^3 voxels at radius 5; this takes 0.34 ms and
// the bins 0.1 ms.
// W > 1: W wavefronts take turns with a bin's runs of 64 particles and put
// their minima together at the end (bins of thousands of particles, few
// blocks). The bound of any of them holds for the block, so they share the
// least.
template <int W>
__global__ void __launch_bounds__(W == 1 ? 256 : 64 * W)
    k_sdf_gather(const float* __restrict__ pos, size_t stride, const uint32_t* __restrict__ start, int side, int nb,
                 float vdx, float cutoff, uint32_t* __restrict__ sdf) {
#pragma clang fp contract(off)  // the reference's separate roundings, no fused multiply-adds
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6, turn = W == 1 ? 0 : wave;
  const uint32_t unb = (uint32_t)nb;  // (at most 256^3 blocks)
  const uint32_t blk = W == 1 ? blockIdx.x * 4u + (uint32_t)wave : blockIdx.y * (unb * unb) + blockIdx.x;
  if (blk >= unb * unb * unb) return;  // uniform for the wavefront (W = 1), else for the workgroup
  __shared__ uint32_t bound;
  __shared__ float least[W == 1 ? 1 : W][64];
  const int bz = (int)(blk % unb), by = (int)(blk / unb % unb), bx = (int)(blk / (unb * unb));
  const int v0 = bx * kBinEdge + (lane >> 4), v1 = by * kBinEdge + ((lane >> 2) & 3), v2 = bz * kBinEdge + (lane & 3);
  const bool in_grid = v0 < side && v1 < side && v2 < side;
  // x_node = i * voxel_dx
  const float n0 = (float)(uint32_t)v0 * vdx, n1 = (float)(uint32_t)v1 * vdx, n2 = (float)(uint32_t)v2 * vdx;
  float lo[3], hi[3];
  {
    const int b[3] = {bx, by, bz};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      lo[a] = (float)(uint32_t)(b[a] * kBinEdge) * vdx;
      hi[a] = (float)(uint32_t)min(b[a] * kBinEdge + kBinEdge - 1, side - 1) * vdx;
    }
  }
  const float rg = cutoff / vdx;  // r_gridpoints, mesh_builder.h:124
  const float near2 = (0.99f * cutoff) * (0.99f * cutoff);
  float best = in_grid ? cutoff * cutoff * 1.01f : 0.0f;  // beyond the cut-off: taken back at the end
  float R2 = cutoff * cutoff * 1.01f;
  if (W > 1) {
    if (threadIdx.x == 0) bound = __float_as_uint(R2);
    __syncthreads();
  }
  const int reach = (int)(rg / kBinEdge) + 1;  // bins beyond it lie 4 reach > rg voxels away
  // anything in reach? a row of bins along z is one range of `start`
  {
    const int w = 2 * reach + 1;
    const int z0 = max(0, bz - reach), z1 = min(nb, bz + reach + 1);
    bool any = false;
    for (int r = lane; r < w * w; r += 64) {
      const int x = bx + r / w - reach, y = by + r % w - reach;
      if (x < 0 || x >= nb || y < 0 || y >= nb) continue;
      const uint32_t* const row = start + ((size_t)x * nb + y) * nb;
      any = any || row[z1] > row[z0];
    }
    if (__ballot(any) == 0ull) {  // (the same for all W wavefronts)
      if (in_grid) sdf[((size_t)v0 * side + v1) * side + v2] = __float_as_uint(cutoff);
      return;
    }
  }
  for (int s = 0; s <= reach; ++s) {
    // bins of shell s lie at least 4 (s - 1) voxels off (less a rounding of x / vdx)
    const float gap = ((float)(kBinEdge * (s - 1)) - 0.01f) * vdx;
    if (s > 1 && gap * gap >= R2) break;
    const int w = 2 * s + 1, all = w * w * w;
    for (int c = 0; c < all; c += 64) {
      const int q = c + lane;
      const int ox = q / (w * w) - s, oy = q / w % w - s, oz = q % w - s;
      uint32_t from = 0, to = 0;
      float near = 0.0f;
      if (q < all && max(abs(ox), max(abs(oy), abs(oz))) == s) {
        const int x = bx + ox, y = by + oy, z = bz + oz;
        if (x >= 0 && x < nb && y >= 0 && y < nb && z >= 0 && z < nb) {
          // voxels between the block's nodes and the bin's cells, per axis
          const auto off = [&](int o) {
            return o == 0 ? 0.0f : fmaxf(0.0f, (float)(o > 0 ? kBinEdge * o - (kBinEdge - 1) : -kBinEdge * (o + 1)) - 0.01f) * vdx;
          };
          const float dx = off(ox), dy = off(oy), dz = off(oz);
          near = dx * dx + dy * dy + dz * dz;
          const size_t b = ((size_t)x * nb + y) * nb + z;
          from = start[b];
          to = start[b + 1];
        }
      }
      uint64_t bins = __ballot(to > from && near < R2);
      while (bins) {
        const int l = __ffsll((long long)bins) - 1;
        bins &= bins - 1;
        if (__uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(near), l)) >= R2) continue;
        const uint32_t p0 = __builtin_amdgcn_readlane(from, l), p1 = __builtin_amdgcn_readlane(to, l);
        bool changed = false;
        for (uint32_t p = p0 + 64u * (uint32_t)turn; p < p1; p += 64u * W) {
          const uint32_t i = p + lane;
          float x = 0.f, y = 0.f, z = 0.f;
          bool keep = false;
          if (i < p1) {
            x = pos[i];
            y = pos[stride + i];
            z = pos[2 * stride + i];
            const float e0 = fmaxf(fmaxf(lo[0] - x, x - hi[0]), 0.0f), e1 = fmaxf(fmaxf(lo[1] - y, y - hi[1]), 0.0f),
                        e2 = fmaxf(fmaxf(lo[2] - z, z - hi[2]), 0.0f);
            keep = e0 * e0 + (e1 * e1 + e2 * e2) < R2;
          }
          uint64_t m = __ballot(keep);
          changed = changed || m != 0ull;
          while (m) {
            const int j = __ffsll((long long)m) - 1;
            m &= m - 1;
            const float px = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), j));
            const float py = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(y), j));
            const float pz = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(z), j));
            // |x - x_node|^2 = dx^2 + (dy^2 + dz^2): Eigen's norm() sums the
            // three squares of a fixed-size vector as e0 + (e1 + e2)
            const float dx = px - n0, dy = py - n1, dz = pz - n2;
            const float d2 = dx * dx + (dy * dy + dz * dz);
            bool closer = d2 < best;
            // near the cut-off the reference's box, truncated in float, decides
            if (__ballot(closer && d2 > near2) != 0ull && closer && d2 > near2)
              closer = in_box(px, v0, vdx, rg, side) && in_box(py, v1, vdx, rg, side) && in_box(pz, v2, vdx, rg, side);
            best = closer ? d2 : best;
          }
        }
        // (non-negative floats order like their bits)
        uint32_t r2 = __float_as_uint(R2);
        if (changed) r2 = (uint32_t)__builtin_amdgcn_readlane(mpmdev::wave_max_scan((int)__float_as_uint(best)), 63);
        if (W > 1) {
          if (changed && lane == 0) atomicMin(&bound, r2);
          r2 = min(r2, *(volatile uint32_t*)&bound);
        }
        R2 = __uint_as_float(__builtin_amdgcn_readfirstlane(r2));
      }
    }
  }
  if (W > 1) {
    least[wave][lane] = best;
    __syncthreads();
    if (wave > 0) return;
    for (int q = 1; q < W; ++q) best = fminf(best, least[q][lane]);
  }
  if (in_grid) sdf[((size_t)v0 * side + v1) * side + v2] = __float_as_uint(fminf(sqrtf(best), cutoff));
}

// ---- the case table, generated at compile time (mc_table.hpp) ----
__constant__ mc::Table kMc = mc::make_table();
__constant__ int kMcEdge[12][2] = {{0, 4}, {1, 5}, {2, 6}, {3, 7}, {0, 2}, {1, 3},
                                   {4, 6}, {5, 7}, {0, 1}, {2, 3}, {4, 5}, {6, 7}};

// A row of cubes (i, j, 0 .. side - 2) belongs to one wavefront, 63 cubes at a
// time: lane l holds the nodes k = c + l of the row's four node rows, and the
// ballots of their inside flags give every cube its case. Stretches with all
// nodes inside or all outside, most of them, end there.
constexpr int kRowCubes = 63;

// The cases of the cubes c .. c + 62 of row (i, j), one a lane (bit q: corner q
// inside, S = rv - d > 0); returns whether any of them holds triangles.
__device__ __forceinline__ bool row_cases(const uint32_t* __restrict__ sdf, int side, double rv, int i, int j, int c,
                                          int lane, int* m) {
  const int k = c + lane;
  uint64_t in[4];
  bool all = true, none = true;
  const uint64_t valid = __ballot(k < side);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const size_t n = ((size_t)(i + (q >> 1)) * side + (size_t)(j + (q & 1))) * side + (size_t)k;
    const bool inside = k < side && rv - (double)__uint_as_float(sdf[n]) > 0.0;
    in[q] = __ballot(inside);
    all = all && in[q] == valid;
    none = none && in[q] == 0ull;
  }
  *m = 0;
  if (all || none) return false;  // uniform
  if (lane < kRowCubes && k < side - 1) {
#pragma unroll
    for (int q = 0; q < 4; ++q) *m |= (int)((in[q] >> lane) & 3ull) << (2 * q);
  }
  return true;
}

__global__ void __launch_bounds__(256)
    k_mc_count(const uint32_t* __restrict__ sdf, int side, double rv, uint32_t* __restrict__ count) {
  const int lane = threadIdx.x & 63;
  const uint32_t s1 = (uint32_t)side - 1u, row = blockIdx.x * 4u + (threadIdx.x >> 6);
  if (row >= s1 * s1) return;  // uniform for the wavefront
  const int i = (int)(row / s1), j = (int)(row % s1);
  int sum = 0;
  for (int c = 0; c < (int)s1; c += kRowCubes) {
    int m;
    if (row_cases(sdf, side, rv, i, j, c, lane, &m)) sum += kMc.ntri[m];
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) sum += __shfl_xor(sum, o);
  if (lane == 0) count[row] = (uint32_t)sum;
}

// grid position of node n
__device__ __forceinline__ void node_pos(uint32_t n, int side, double p[3]) {
  p[2] = (double)(n % (uint32_t)side);
  p[1] = (double)((n / (uint32_t)side) % (uint32_t)side);
  p[0] = (double)(n / ((uint32_t)side * (uint32_t)side));
}

// the iso-point on the edge between nodes na and nb, from the lower node
__device__ __forceinline__ void edge_point(const uint32_t* __restrict__ sdf, uint32_t na, uint32_t nb, int side,
                                           double rv, double vdx, float* out, uint64_t* key) {
#pragma clang fp contract(off)  // one rounding per operation, as the test's restatement forms it
  if (nb < na) { const uint32_t t = na; na = nb; nb = t; }
  const double Sa = rv - (double)__uint_as_float(sdf[na]), Sb = rv - (double)__uint_as_float(sdf[nb]);
  const double t = Sa / (Sa - Sb);
  double pa[3], pb[3];
  node_pos(na, side, pa);
  node_pos(nb, side, pb);
#pragma unroll
  for (int a = 0; a < 3; ++a) out[a] = (float)((pa[a] + t * (pb[a] - pa[a])) * vdx);
  *key = ((uint64_t)na << 32) | (uint64_t)nb;
}

// The vertices of a row's triangles, one a lane: a stretch's triangles are
// listed in LDS first, so that its lanes share the work however few of its
// cubes are cut, and neighbouring lanes store neighbouring vertices. (One
// thread per cube, with its up to 15 vertices in turn: 344 us for the 454,000
// triangles of the 1,000,000-particle dam break on 250^3, and 205 us to count
// and scan 15.4 million cubes; rows: 51 and 70 us.)
__global__ void __launch_bounds__(256)
    k_mc_emit(const uint32_t* __restrict__ sdf, int side, double rv, double vdx, const uint32_t* __restrict__ offset,
              float* __restrict__ xyz, uint64_t* __restrict__ keys) {
  __shared__ uint16_t list[4][5 * 64];  // of each triangle: its cube's lane, and its number there (above 8 bits)
  __shared__ uint8_t cases[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t s1 = (uint32_t)side - 1u, row = blockIdx.x * 4u + (uint32_t)wave;
  if (row >= s1 * s1) return;  // uniform for the wavefront, as what follows
  uint32_t at = offset[row];
  if (offset[row + 1] == at) return;
  const int i = (int)(row / s1), j = (int)(row % s1);
  const uint64_t below = (1ull << lane) - 1ull;
  for (int c = 0; c < (int)s1; c += kRowCubes) {
    int m;
    if (!row_cases(sdf, side, rv, i, j, c, lane, &m)) continue;
    const int nt = kMc.ntri[m];
    int first = 0, total = 0;
#pragma unroll
    for (int b = 0; b < 3; ++b) {  // (at most 5 triangles a cube)
      const uint64_t bit = __ballot((nt >> b) & 1);
      first += __popcll(bit & below) << b;
      total += __popcll(bit) << b;
    }
    cases[wave][lane] = (uint8_t)m;
    for (int t = 0; t < nt; ++t) list[wave][first + t] = (uint16_t)(lane | (t << 8));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int e = lane; e < 3 * total; e += 64) {
      const int t = e / 3, q = e - 3 * t;
      const int cube = list[wave][t] & 255, nth = list[wave][t] >> 8;
      const int edge = kMc.tri[cases[wave][cube]][3 * nth + q];
      const auto node = [&](int corner) {
        return ((uint32_t)(i + ((corner >> 2) & 1)) * (uint32_t)side + (uint32_t)(j + ((corner >> 1) & 1))) *
                   (uint32_t)side + (uint32_t)(c + cube + (corner & 1));
      };
      float v[3];
      uint64_t key;
      edge_point(sdf, node(kMcEdge[edge][0]), node(kMcEdge[edge][1]), side, rv, vdx, v, &key);
      const size_t o = (size_t)at * 3 + (size_t)e;
#pragma unroll
      for (int a = 0; a < 3; ++a) xyz[3 * o + a] = v[a];
      if (keys) keys[o] = key;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    at += (uint32_t)total;
  }
}

}  // namespace

namespace mpmk {

int mesh_bins(int side) { return (side + kBinEdge - 1) / kBinEdge; }

hipError_t mesh_distance_field(const ParticlesDev& P, int side, float vdx, float cutoff, double fill,
                               const MeshScratch& w, uint32_t* sdf, hipStream_t s) {
  const int64_t nv = (int64_t)side * side * side;
  const dim3 gp((unsigned)((P.n + 255) / 256));
  // Scatter or gather, in microseconds as measured on scenes of 10,000 to
  // 1,000,000 particles, 24 to 250 voxels a side and radii 1 to 5. Scatter: a
  // thread's box takes 0.35 us a voxel, and all boxes 2e-6 us a voxel. Gather:
  // 60 for the bins' launches, 1e-5 a voxel of the grid, and a block's turn
  // through its bins, 0.06 a particle of an occupied bin. (1,000,000 particles
  // on 250^3, radius 5: 9,200 against 440; on 24^3, radius 2: 500 against 650;
  // 100,000 on 60^3, radius 1: 70 against 190.)
  const int nb = mesh_bins(side);
  const int64_t bins = (int64_t)nb * nb * nb;
  const double box = 2.0 * (double)(cutoff / vdx) + 1.0;
  const double held = (double)P.n / std::max(1.0, fill * (double)bins);  // particles of an occupied bin
  const double scatter = box * box * box * (0.35 + 2e-6 * (double)P.n);
  const double gather = 60.0 + 1e-5 * (double)nv + 0.06 * held;
  if (!w.pos || P.n <= 0 || box > kGatherMaxBox || scatter < gather) {
    const hipError_t e = fill_u32(sdf, nv, __builtin_bit_cast(uint32_t, cutoff), s);
    if (e != hipSuccess || P.n <= 0) return e;
    hipLaunchKernelGGL(k_sdf_scatter, gp, dim3(256), 0, s, P, side, vdx, cutoff, sdf);
    return hipGetLastError();
  }
  if (!w.count || !w.start || !w.scan || !w.bins || !w.rank || w.pos_stride < (size_t)P.n) return hipErrorInvalidValue;
  hipError_t e = fill_u32(w.count, bins, 0u, s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_bin_count, gp, dim3(256), 0, s, P, side, vdx, cutoff, nb, w.count, w.bins, w.rank);
  e = exclusive_scan(w.count, w.start, bins, w.scan, w.start + bins, s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_bin_scatter, gp, dim3(256), 0, s, P, w.start, w.bins, w.rank, w.pos, w.pos_stride);
  if (held < kGatherFew)
    hipLaunchKernelGGL(k_sdf_gather<1>, dim3((unsigned)((bins + 3) / 4)), dim3(256), 0, s, w.pos, w.pos_stride,
                       w.start, side, nb, vdx, cutoff, sdf);
  else {
    // (by planes of blocks: a dimension of a launch has less than 2^32 threads, and
    // 1024 for each of the blocks of 700^3 voxels are more)
    const dim3 g((unsigned)nb * (unsigned)nb, (unsigned)nb);
    if (held < kGatherMany)
      hipLaunchKernelGGL(k_sdf_gather<4>, g, dim3(256), 0, s, w.pos, w.pos_stride, w.start, side, nb, vdx, cutoff, sdf);
    else
      hipLaunchKernelGGL(k_sdf_gather<16>, g, dim3(1024), 0, s, w.pos, w.pos_stride, w.start, side, nb, vdx, cutoff,
                         sdf);
  }
  return hipGetLastError();
}

hipError_t mesh_count(const uint32_t* sdf, int side, double rv, uint32_t* count, hipStream_t s) {
  const int64_t rows = (int64_t)(side - 1) * (side - 1);
  hipLaunchKernelGGL(k_mc_count, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, sdf, side, rv, count);
  return hipGetLastError();
}

hipError_t mesh_emit(const uint32_t* sdf, int side, double rv, double vdx, const uint32_t* offset, float* xyz,
                     uint64_t* keys, hipStream_t s) {
  const int64_t rows = (int64_t)(side - 1) * (side - 1);
  hipLaunchKernelGGL(k_mc_emit, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, sdf, side, rv, vdx, offset, xyz,
                     keys);
  return hipGetLastError();
}

}  // namespace mpmk
