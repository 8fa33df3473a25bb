// adjoint.hip -- a differentiable MLS-MPM substep and its hand-written adjoint
// (gfx950). No reference counterpart: the reference has no gradients.
//
// The substep is the engine's (P2G, grid update, G2P: reference src/mpm.cu:
// 14-178) for the fixed-corotated model (MMFixedCorotated, MaterialModel.cuh:
// 56-61) with J = det F, per-particle Lame parameters mu_p, lambda_p, no
// plasticity, and the stencil clipped at the grid faces (N - base). State
// planes (24 x n floats, plane-major): x(3) v(3) C(9) F(9), 3x3 row-major.
// The forward records a grid tape per node that the backward replays: the
// velocity and mass after the update (N^3 float4, read by G2P), then the
// velocity before the walls and the wall flags (N^3 float4).
//
// Kernels, 64 particles and four wavefronts per workgroup (a particle is lane i
// of each):
//   k_diff_step<G2P, P2G>   grid update and G2P of substep n (gather of its
//                           sums, F and x update), fused with the P2G of
//                           substep n+1 (stress through the polar rotation of
//                           F, scatter); further workgroups write the grid
//                           update into the tape
//   k_adj_step<P2G', G2P'>  the adjoint of the P2G of substep s (gather of the
//                           momentum and mass adjoints, stress adjoint, mu and
//                           lambda adjoints) fused with the adjoint of the G2P
//                           of substep s-1 (scatter of the grid velocity
//                           adjoint)
//   k_adj_grid              grid update backward: momentum and mass adjoints
// so a substep is one launch forward and two backward, and a run of
// substeps is enqueued from one host call (diff_forward_steps /
// diff_backward_steps).
//
// What bounds them is latency: the elastic cube of 32,768 particles is 512
// workgroups on 256 CUs, a small one 35, and the state that a substep moves
// (200 bytes a particle, 6.5 MB) takes 1.3 us at the copy rate. So three
// wavefronts take an x-plane of the stencil each and run what needs a whole
// particle (stress, F) side by side, a fourth takes what does not wait for
// them (storing the state, the cells of the scatter, mu's adjoint).
// A wavefront has its SIMD nearly to itself and runs its code once: short code
// without branches, in which an LDS or memory round trip is waited for once, is
// what counts. For a jittered cube of 32,768 particles under shear
// (perf/cases.py's rollouts) k_diff_step and k_adj_step took 26 and 38 us with
// one wavefront per 64 particles, now 12.4 and 13.6, the grid update of 3 to 5 us
// in the first (2,197 particles: 19 and 29, now 9.6 and 11.4); for bench.py's
// cube, which falls freely in lattice order, 18.8 and 29.8, now 11.4 and 12.4.
// Where the chip is full the wavefronts' repeated work still costs less than the
// shorter chain saves: a substep forward and its adjoint 77 + 104 -> 56 + 80 us for
// 262,144 particles in cell order, 541 + 690 -> 374 + 580 for 2,097,152. (In
// random order the atomics bound both: 91 + 98 -> 79 + 82 us for 32,768, 284 + 379
// -> 311 + 327 for 262,144 on 64^3, 1,149 + 1,150 -> 1,068 + 1,063 for 1,000,000.)
// The SVD's serial chain is 2 us of each launch. Newton's iteration for the
// rotation takes 0.6, but the position's adjoint is what is left of momenta
// that cancel: the last bits by which the rotations differ come out as 1e-3 of
// its root mean square in sparse cells.
//
// The stress adjoint differentiates the polar rotation R of F = U S V^T:
// with Rbar the adjoint of R and M = V^T skew(R^T Rbar) V,
// Fbar += 2 U N V^T, N_ij = M_ij / (s_i + s_j).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "device_math.hpp"
#include "engine_types.hpp"
#include "kernels.hpp"

using namespace mpmdev;

namespace {

enum : int { DX = 0, DV = 3, DC = 6, DF = 15 };

constexpr int kWave = 64;            // particles per workgroup
constexpr int kPlanes = 3;           // wavefronts per workgroup: one per x-plane of the stencil, and a
constexpr int kThreads = 4 * kWave;  // fourth for what does not wait for the planes
constexpr int kNodes = 27;           // of a stencil
constexpr int kRunsAhead = 8;        // runs whose sums are loaded together
constexpr int kNowhere = 1 << 20;    // a cell that no node is next to
// Workgroups of a launch at most, in 2^30 threads: a dimension of a launch has
// less than 2^32, and more wrap around without an error (1,073,741,824
// particles; 1024^3 nodes are 2^22 workgroups by themselves). Kernels get the
// number of their launch's first one.
constexpr unsigned kMaxBlocks = 1u << 22;

struct DiffK {
  StepConsts k;
  float mass, volume;
  int wall_lo, wall_hi;  // a node index below wall_lo or from wall_hi on is a wall's
  int64_t n;
};

// One axis of a particle's stencil: quadratic B-spline weights and their
// derivatives (InterpolationKernel.cuh), node offsets and node indices. A node
// outside the grid has weight 0 and the index of the nearest node inside, so
// that a load of it is in range (plane_sums takes 0 for what it loads there).
struct Axis {
  int base;
  int node[3];
  float w[3], dw[3], dp[3];
};

struct Stencil {
  Axis ax[3];
  bool clipped;  // a node of the stencil is not in the grid
  bool outside;  // past the grid: the particle is left as it is
};

__device__ __forceinline__ Stencil make_stencil(const float x[3], const StepConsts& k) {
  Stencil s;
  s.clipped = s.outside = false;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    Axis& t = s.ax[a];
    const float xg = x[a] * k.dx_inv;
    t.base = (int)(xg - 0.5f);
    const float f = xg - (float)t.base;
    const float t0 = 1.5f - f, t1 = f - 1.0f, t2 = f - 0.5f;
    const float w[3] = {0.5f * (t0 * t0), 0.75f - t1 * t1, 0.5f * (t2 * t2)};
    const float dw[3] = {-t0 * k.dx_inv, -2.0f * t1 * k.dx_inv, t2 * k.dx_inv};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int node = t.base + i;
      const bool ok = (unsigned)node < (unsigned)k.N;
      t.w[i] = ok ? w[i] : 0.0f;
      t.dw[i] = ok ? dw[i] : 0.0f;
      t.dp[i] = (float)node * k.dx - x[a];
      t.node[i] = min(max(node, 0), k.N - 1);
    }
    s.clipped |= (unsigned)t.base >= (unsigned)max(k.N - 2, 0);
    s.outside |= t.base + 3 < 0 || t.base >= k.N;  // mpm.cu:31-35,129-133
  }
  return s;
}

// the entry of an x-axis array that a wavefront's plane has
template <typename T>
__device__ __forceinline__ T of_plane3(T a, T b, T c, int plane) {
  return plane == 0 ? a : plane == 1 ? b : c;
}
template <typename T>
__device__ __forceinline__ T of_plane(const T (&v)[3], int plane) {
  return of_plane3(v[0], v[1], v[2], plane);
}

// the base cell of a particle inside the domain (base in [-3, N) per axis)
// as one non-negative integer
__device__ __forceinline__ int cell_key(const Stencil& s, int N) {
  const int M = N + 3;
  return ((s.ax[0].base + 3) * M + (s.ax[1].base + 3)) * M + (s.ax[2].base + 3);
}

template <int PLANES>
__device__ __forceinline__ void load_planes(const float* st, int64_t n, int64_t p, int first, float* out) {
#pragma unroll
  for (int a = 0; a < PLANES; ++a) out[a] = st[(first + a) * n + p];
}

template <int PLANES>
__device__ __forceinline__ void store_planes(float* st, int64_t n, int64_t p, int first, const float* in) {
#pragma unroll
  for (int a = 0; a < PLANES; ++a) st[(first + a) * n + p] = in[a];
}

// a particle's 24 values, shared out to the three wavefronts that hold them
__device__ __forceinline__ void store_state(float* st, int64_t n, int64_t p, int plane, const float x[3],
                                            const float v[3], const float C[9], const float F[9]) {
  if (plane == 0) {
    store_planes<3>(st, n, p, DX, x);
    store_planes<3>(st, n, p, DV, v);
  } else if (plane == 1) {
    store_planes<9>(st, n, p, DC, C);
  } else if (plane == 2) {
    store_planes<9>(st, n, p, DF, F);
  }
}

// tau = 2 mu (F - R) F^T + lambda (J - 1) J I, J = det F
__device__ __forceinline__ void fc_stress(const float F[9], const float R[9], float mu, float lam,
                                          float tau[9]) {
  float FmR[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) FmR[i] = 2.0f * mu * (F[i] - R[i]);
  mul_abt(FmR, F, tau);
  const float J = det3(F);
  const float vol = lam * ((J - 1.0f) * J);
  tau[0] += vol;
  tau[4] += vol;
  tau[8] += vol;
}

// the affine momentum matrix of P2G is A = sc tau + m C, sc = -Dinv dt V
__device__ __forceinline__ float stress_scale(const DiffK& d) {
  return ((-d.k.dinv) * d.k.dt) * d.volume;
}

// ---------------------------------------------------------------- plane of a stencil
// One x-plane (9 nodes) of a particle's stencil, as tensor products of the y
// and z axes: each of the sums over the nodes is taken over z, then over y, so
// a node costs 6 (velocity and its first moments), 15 (with the gradient) or 8
// (a row) multiply-adds where the node by node form had 30 to 60.

// the q-vector q0 + M dp of the plane's nodes: at (plane, b) and at node c
__device__ __forceinline__ void q_start(const float q0[3], const float M[9], float dpa, float qa[3]) {
#pragma unroll
  for (int r = 0; r < 3; ++r) qa[r] = __builtin_fmaf(M[3 * r], dpa, q0[r]);
}

// The velocity of a node from its momentum and mass (w > 0) before the walls:
// the quotients, and gravity on y (mpm.cu:76-91). The quotients are c / w to the
// last bit but in rare cases (q + (c - q w) / w with the reciprocal of a Newton
// step: Markstein, 1990): with the divisions of the language, each with a
// serial chain of its own, the 27 of a gather took 2.1 us, these 0.95. The scale
// keeps a vanishing or a huge mass's reciprocal in range.
__device__ __forceinline__ void free_velocity(const float4& c, const StepConsts& k, float u[3]) {
  const float scale = c.w < 0x1p-96f ? 0x1p64f : c.w > 0x1p96f ? 0x1p-64f : 1.0f;
  const float w = c.w * scale, p[3] = {c.x * scale, c.y * scale, c.z * scale};
  float r = __builtin_amdgcn_rcpf(w);
  r = w < __builtin_inff() ? __builtin_fmaf(__builtin_fmaf(-w, r, 1.0f), r, r) : r;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float q = p[a] * r;
    u[a] = fabsf(q) < __builtin_inff() ? __builtin_fmaf(__builtin_fmaf(-w, q, p[a]), r, q) : q;
  }
  u[1] = __builtin_fmaf(k.dt, k.gravity, u[1]);
}

// the walls of a node (mpm.cu:92-105): sticky on five sides, a floor
struct NodeWalls {
  bool sticky, floor_;
};
__device__ __forceinline__ NodeWalls node_walls(int i, int j, int k, const DiffK& d) {
  NodeWalls w;
  w.sticky = i < d.wall_lo || i >= d.wall_hi || j >= d.wall_hi || k < d.wall_lo || k >= d.wall_hi;
  w.floor_ = j < d.wall_lo;
  return w;
}
__device__ __forceinline__ void apply_walls(const NodeWalls& w, float u[3]) {
#pragma unroll
  for (int a = 0; a < 3; ++a) u[a] = w.sticky ? 0.0f : u[a];
  u[1] = w.floor_ ? fmaxf(0.0f, u[1]) : u[1];
}

__device__ __forceinline__ float4 node_velocity(const float4& sum, int i, int j, int k, const DiffK& d) {
  float u[3];
  free_velocity(sum, d.k, u);
  apply_walls(node_walls(i, j, k, d), u);
  const bool has = sum.w > 0.0f;
  return make_float4(has ? u[0] : 0.0f, has ? u[1] : 0.0f, has ? u[2] : 0.0f, 0.0f);
}

// Sums over the plane of the 4-vectors g = grid[node]:
//   s[0..2]    sum w g              s[3 + 3 r + q]  sum w g_r dp_q
// and with GRAD, val = g . (q0 + M dp) + m g.w (m = 0 without MASS),
//   s[12 + q]  sum (dw/dx_q) val
// With ROWS the plane's rows w (q0 + M dp) go to `row`.
// With UPDATE grid holds the momentum and mass sums, updated to velocities here.
template <bool UPDATE, bool GRAD, bool MASS, bool ROWS>
__device__ __forceinline__ void plane_sums(const float4* __restrict__ grid, const Stencil& sn, int plane,
                                           const DiffK& d, const float q0[3], const float M[9], float m, float4* row,
                                           float s[16]) {
  const Axis &ay = sn.ax[1], &az = sn.ax[2];
  const float wa = of_plane(sn.ax[0].w, plane), dpa = of_plane(sn.ax[0].dp, plane);
  const int na = of_plane(sn.ax[0].node, plane);
  const StepConsts& k = d.k;
  float4 g[9];
#pragma unroll
  for (int b = 0; b < 3; ++b)
#pragma unroll
    for (int c = 0; c < 3; ++c)
      g[3 * b + c] = grid[((size_t)na * k.N + (size_t)ay.node[b]) * k.N + (size_t)az.node[c]];
  if (__builtin_expect(__ballot(sn.clipped) != 0ull, 0)) {
    // a weight of 0 would not do: it makes NaN of a value that is not finite
    const auto in_grid = [&](int node) { return (unsigned)node < (unsigned)k.N; };
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int c = 0; c < 3; ++c)
        if (!(in_grid(sn.ax[0].base + plane) && in_grid(ay.base + b) && in_grid(az.base + c)))
          g[3 * b + c] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  if (UPDATE) {
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int c = 0; c < 3; ++c) g[3 * b + c] = node_velocity(g[3 * b + c], na, ay.node[b], az.node[c], d);
  }
  float qa[3];
  if (GRAD) q_start(q0, M, dpa, qa);
  float S0[3] = {0.f, 0.f, 0.f}, S1[3] = {0.f, 0.f, 0.f}, S2[3] = {0.f, 0.f, 0.f};
  float u0 = 0.f, u1 = 0.f, u2 = 0.f;
#pragma unroll
  for (int b = 0; b < 3; ++b) {
    float T0[3] = {0.f, 0.f, 0.f}, T2[3] = {0.f, 0.f, 0.f}, t0 = 0.f, t2 = 0.f;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float4 gc = g[3 * b + c];
      const float gv[3] = {gc.x, gc.y, gc.z};
      const float wc = az.w[c], wd = az.w[c] * az.dp[c];
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        T0[r] += wc * gv[r];
        T2[r] += wd * gv[r];
      }
      if (GRAD) {
        float q[3], val = MASS ? m * gc.w : 0.0f;
#pragma unroll
        for (int r = 0; r < 3; ++r) {
          q[r] = qa[r] + M[3 * r + 1] * ay.dp[b] + M[3 * r + 2] * az.dp[c];
          val += gv[r] * q[r];
        }
        t0 += wc * val;
        t2 += az.dw[c] * val;
        if (ROWS) {
          const float wt = (wa * ay.w[b]) * wc;
          row[3 * b + c] = make_float4(wt * q[0], wt * q[1], wt * q[2], 0.0f);
        }
      }
    }
    const float wb = ay.w[b], wbd = ay.w[b] * ay.dp[b];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      S0[r] += wb * T0[r];
      S1[r] += wbd * T0[r];
      S2[r] += wb * T2[r];
    }
    if (GRAD) {
      u0 += wb * t0;
      u1 += ay.dw[b] * t0;
      u2 += wb * t2;
    }
  }
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    s[r] = wa * S0[r];
    s[3 + 3 * r] = (wa * dpa) * S0[r];
    s[3 + 3 * r + 1] = wa * S1[r];
    s[3 + 3 * r + 2] = wa * S2[r];
  }
  s[12] = GRAD ? of_plane(sn.ax[0].dw, plane) * u0 : 0.f;
  s[13] = GRAD ? wa * u1 : 0.f;
  s[14] = GRAD ? wa * u2 : 0.f;
  s[15] = 0.f;
}

// Adds up the planes' parts of the first 4 V4 values of s, in the planes'
// order: every wavefront of the workgroup ends with the same bits. put_plane
// by the planes' wavefronts, a barrier, sum_planes by all. `part` has
// 3 V4 kWave float4.
template <int V4>
__device__ __forceinline__ void put_plane(float4* part, int plane, int lane, const float s[16]) {
#pragma unroll
  for (int j = 0; j < V4; ++j)
    part[(plane * V4 + j) * kWave + lane] = make_float4(s[4 * j], s[4 * j + 1], s[4 * j + 2], s[4 * j + 3]);
}
template <int V4>
__device__ __forceinline__ void sum_planes(const float4* part, int lane, float s[16]) {
#pragma unroll
  for (int j = 0; j < V4; ++j) {
    const float4 a = part[j * kWave + lane], b = part[(V4 + j) * kWave + lane],
                 c = part[(2 * V4 + j) * kWave + lane];
    s[4 * j] = (a.x + b.x) + c.x;
    s[4 * j + 1] = (a.y + b.y) + c.y;
    s[4 * j + 2] = (a.z + b.z) + c.z;
    s[4 * j + 3] = (a.w + b.w) + c.w;
  }
}

// ---------------------------------------------------------------- scatter
// largest value over the wavefront's lanes (v >= 0), the same in every lane
__device__ __forceinline__ int wave_max(int v) { return __builtin_amdgcn_readlane(wave_max_scan(v), kWave - 1); }

// What the wavefronts of a scatter share in LDS.
struct ScatterShared {
  float4 rows[kWave * kNodes + kWave];  // a run's 27 node sums, and a zero for each lane
  int4 cell[kWave];                     // a run's base cell, and packed, its place in the box
  int lo[3], hi[3];                     // box of the base cells
  int runs;
  float4 sum[kThreads];                 // a wavefront's nodes on their way to the grid
  int node[kThreads];
};

// Adds a workgroup's rows (VPN values for each of the 27 nodes of each of 64
// particles) to `grid` (4 floats per node). Many workgroups aim at the same
// few nodes, so the rows are summed twice before the FP32 atomics:
//   scatter_runs   each plane's wavefront sums its 9 nodes over the runs of
//                  particles of one cell (cut every 16 lanes), a segmented
//                  scan over the lanes in registers, and puts the runs' sums
//                  into LDS
//   scatter_nodes  after a barrier, a lane takes a node of the box that the
//                  workgroup's particles reach, adds up the runs that touch it
//                  and sends the sum to `grid`
// 32,768 particles at 25 a cell have 4 runs in a workgroup at the start of a
// rollout and 19 (of 8 cells) after 100 substeps, and reach 49 and 74 nodes,
// where an atomic per run and node makes 100 and 520: 100 substeps took 2.86
// ms with the runs' atomics alone and 1.72 summed by node. Tried besides: a
// walk over the 64 rows (50 cycles a row unrolled, 200 in a loop: 5 us and
// more), and LDS atomics into the box, run by run (a wavefront's 64 lanes take
// 130 cycles or more per instruction: 14.9 us for the kernel, this 12.6).
// A box of more nodes than the workgroup has threads (particles in no order,
// or from the end of one row of cells and the start of the next) goes run by
// run to `grid`: a second pass over the runs costs more than the atomics saved
// (4,096 particles in rows of the lattice: a substep and its adjoint 49 us
// with up to 384 nodes, 43 with one pass; 32,768 in order: no difference).
//
// A lane's place among the runs; `inside`: its particle reaches the grid (the
// same in every wavefront). Every lane of the wavefront calls it.
struct Runs {
  uint64_t ends;  // the last lane of each run
  int depth;      // lanes of the run before this one
  int run;        // its number
};
__device__ __forceinline__ Runs find_runs(bool inside, const Stencil& sn, int N) {
  const int lane = threadIdx.x & (kWave - 1);
  const int key = inside ? cell_key(sn, N) : -1;
  const int prev = __shfl_up(key, 1);
  const uint64_t starts = __ballot((lane & 15) == 0 || key != prev);
  Runs r;
  r.ends = (starts >> 1) | (1ull << 63);
  r.depth = lane - (63 - __clzll((long long)(starts & ((2ull << lane) - 1ull))));
  r.run = (int)__popcll(r.ends & ((1ull << lane) - 1ull));
  return r;
}

// by the planes' wavefronts, all lanes
template <int VPN>
__device__ __forceinline__ void scatter_runs(ScatterShared& sh, float4 row[9], bool inside, const Stencil& sn,
                                             int plane, int N) {
  const int lane = threadIdx.x & (kWave - 1);
  const Runs runs = find_runs(inside, sn, N);
  const int depth = runs.depth;
  float* v = &row[0].x;
  // lane i adds lane i - n of its run (a DPP shift within 16 lanes); the mask
  // drops what belongs to another run, whatever it is
#define MPM_RUN_STEP(n)                                                                              \
  {                                                                                                  \
    int keep = depth >= n ? -1 : 0;                                                                  \
    __asm__("" : "+v"(keep)); /* (a mask, not a select: one instruction with the shift) */           \
    _Pragma("unroll") for (int i = 0; i < 36; ++i) if (VPN == 4 || (i & 3) != 3) {                   \
      const int t = __builtin_amdgcn_update_dpp(0, __float_as_int(v[i]), 0x110 + n, 0xf, 0xf, true); \
      v[i] += __int_as_float(t & keep);                                                              \
    }                                                                                                \
  }
  MPM_RUN_STEP(1)
  MPM_RUN_STEP(2)
  MPM_RUN_STEP(4)
  MPM_RUN_STEP(8)
#undef MPM_RUN_STEP
  if ((runs.ends >> lane) & 1ull) {
#pragma unroll
    for (int o = 0; o < 9; ++o) sh.rows[runs.run * kNodes + 9 * plane + o] = row[o];
  }
}

// by the fourth wavefront, all lanes: the runs' cells and the box of nodes they reach
__device__ __forceinline__ void scatter_cells(ScatterShared& sh, bool inside, const Stencil& sn, int N) {
  const int lane = threadIdx.x & (kWave - 1);
  const Runs runs = find_runs(inside, sn, N);
  const int count = (int)__popcll(runs.ends);
  int lo[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {  // (no particle inside: lo = N, hi = -3)
    const int base = sn.ax[a].base;
    const int hi = wave_max(inside ? base + 3 : 0) - 3;
    lo[a] = N - wave_max(inside ? N - base : 0);
    if (lane == 0) {
      sh.lo[a] = lo[a];
      sh.hi[a] = hi;
    }
  }
  if ((runs.ends >> lane) & 1ull) {
    const int b0 = sn.ax[0].base, b1 = sn.ax[1].base, b2 = sn.ax[2].base;
    // (in a box that is summed by node the offsets are below 2^8)
    sh.cell[runs.run] = inside ? make_int4(b0, b1, b2, (b0 - lo[0]) | (b1 - lo[1]) << 10 | (b2 - lo[2]) << 20)
                               : make_int4(kNowhere, 0, 0, 0x3fffffff);
  }
  sh.rows[kWave * kNodes + lane] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (lane == 0) sh.runs = count;
}

// Adds component lane & 3 of node lane >> 2 of 16 nodes with one instruction:
// atomics that lie side by side go out together (a component of 64 nodes at a
// time, a node's four 16 bytes apart in turn, took 4 times as long).
__device__ __forceinline__ void add_component(float* __restrict__ grid, int node, int comp, float sum) {
  if (node >= 0 && sum != 0.0f) unsafeAtomicAdd(grid + 4 * (size_t)(unsigned)node + comp, sum);
}

// the index of a node of the grid (N <= 1024: below 2^30), -1 outside
__device__ __forceinline__ int node_index(int i, int j, int k, int N) {
  return ((unsigned)i < (unsigned)N) & ((unsigned)j < (unsigned)N) & ((unsigned)k < (unsigned)N)
             ? (i * N + j) * N + k
             : -1;
}

// by all wavefronts, a barrier after the two above
template <int VPN>
__device__ __forceinline__ void scatter_nodes(ScatterShared& sh, int wave, int N, float* __restrict__ grid) {
  const int lane = threadIdx.x & (kWave - 1);
  const int runs = __builtin_amdgcn_readfirstlane(sh.runs);
  const int lo0 = sh.lo[0], lo1 = sh.lo[1], lo2 = sh.lo[2];
  const int e0 = sh.hi[0] - lo0 + 3, e1 = sh.hi[1] - lo1 + 3, e2 = sh.hi[2] - lo2 + 3;  // nodes per axis
  if (e0 <= 0) return;
  // (N <= 1024, so two extents' product is below 2^21)
  if (e0 * e1 <= kThreads && e0 * e1 * e2 <= kThreads) {
    const int count = __builtin_amdgcn_readfirstlane(e0 * e1 * e2);
    const float r1 = __builtin_amdgcn_rcpf((float)e1), r2 = __builtin_amdgcn_rcpf((float)e2);
    if (wave * kWave < count) {
      const int node = threadIdx.x;
      const int ij = (int)(((float)node + 0.5f) * r2);  // (exact: node < 2^8)
      const int i = (int)(((float)ij + 0.5f) * r1);
      const int j = ij - i * e1, k = node - ij * e2;
      const int cells = sh.cell[lane].w;  // run r's, in lane r
      float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 1
      for (int r = 0; r < runs; r += kRunsAhead) {
        float4 v[kRunsAhead];
#pragma unroll
        for (int q = 0; q < kRunsAhead; ++q) {
          const int cell = __builtin_amdgcn_readlane(cells, (r + q) & (kWave - 1));
          const int a = i - (cell & 0x3ff), b = j - ((cell >> 10) & 0x3ff), c = k - (cell >> 20);
          const bool mine = (max(max((unsigned)a, (unsigned)b), (unsigned)c) < 3u) & (r + q < runs);
          int at = (r + q) * kNodes + 9 * a + 3 * b + c;
          at = mine ? at : kWave * kNodes + lane;
          v[q] = sh.rows[at];
        }
#pragma unroll
        for (int q = 0; q < kRunsAhead; ++q) {
          sum.x += v[q].x;
          sum.y += v[q].y;
          sum.z += v[q].z;
          if (VPN == 4) sum.w += v[q].w;
        }
      }
      // (the wavefront's own: its LDS accesses are in order)
      sh.sum[threadIdx.x] = sum;
      sh.node[threadIdx.x] = node < count ? node_index(lo0 + i, lo1 + j, lo2 + k, N) : -1;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int at = wave * kWave + 16 * q + (lane >> 2), comp = lane & 3;
        const float part = (&sh.sum[at].x)[comp];
        if (VPN == 4 || comp != 3) add_component(grid, sh.node[at], comp, part);
      }
    }
  } else {
    // a thread keeps its node and component, of every other run
    constexpr int kValues = 4 * kNodes;
    if (threadIdx.x >= 2 * kValues) return;
    const int comp = lane & 3, part = threadIdx.x / kValues, o = (threadIdx.x - part * kValues) >> 2;
    if (VPN == 3 && comp == 3) return;
    const int a = o / 9, b = (o / 3) % 3, c = o % 3;
#pragma unroll 1
    for (int r = part; r < runs; r += 8) {
      int4 cell[4];
      float sum[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int at = min(r + 2 * q, runs - 1);
        cell[q] = sh.cell[at];
        sum[q] = (&sh.rows[at * kNodes + o].x)[comp];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (r + 2 * q < runs)  // (a cell of kNowhere is outside the grid)
          add_component(grid, node_index(cell[q].x + a, cell[q].y + b, cell[q].z + c, N), comp, sum[q]);
    }
  }
}

// ---------------------------------------------------------------- forward
// What the node blocks of a forward launch do, 256 nodes each: the grid update
// of the substep's momentum and mass `sums` into the tape, tv = (velocity,
// mass) after the update, tw = (velocity before the walls, wall flags: 1
// sticky, 2 floor), and the clearing of a later substep's sums. Either may be
// null.
struct NodeWork {
  const float4* sums;
  float4 *tv, *tw, *clear;
};

__device__ __forceinline__ void node_block(const NodeWork& w, const DiffK& d, unsigned block) {
  const int N = d.k.N;
  const size_t nodes = (size_t)N * N * N;
  const size_t t = (size_t)block * kThreads + threadIdx.x;
  if (t >= nodes) return;
  if (w.clear) w.clear[t] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (!w.tv) return;
  const float4 c = w.sums[t];
  float4 o0 = make_float4(0.f, 0.f, 0.f, c.w), o1 = make_float4(0.f, 0.f, 0.f, 0.f);
  if (c.w > 0.0f) {
    // (32-bit: N <= 1024, so a node index is below 2^30)
    const uint32_t ti = (uint32_t)t, n = (uint32_t)N;
    const int zi = (int)(ti % n), yi = (int)((ti / n) % n), xi = (int)(ti / (n * n));
    float u[3];
    free_velocity(c, d.k, u);
    const NodeWalls walls = node_walls(xi, yi, zi, d);
    o1 = make_float4(u[0], u[1], u[2], (float)((walls.sticky ? 1 : 0) | (walls.floor_ ? 2 : 0)));
    apply_walls(walls, u);
    o0 = make_float4(u[0], u[1], u[2], c.w);
  }
  w.tv[t] = o0;
  w.tw[t] = o1;
}

// G2P of substep n from `st` into `out` (particles outside the grid are
// copied), fused with the P2G of substep n+1 of the new state into `grid`.
// Without G2P: the P2G of `st`. Without P2G: the G2P only. The first `blocks`
// workgroups hold the particles, those past them the nodes; `first` is the
// launch's first one.
// The G2P updates the nodes that it gathers by itself, from substep n's sums: 27
// times as many updates as there are nodes, for 0.95 us of 12.2 (32,768
// particles), where the grid update as a launch of its own took 3.3 us, a gap
// and 4 us of the host.
template <bool G2P, bool P2G>
__global__ void __launch_bounds__(kThreads)
    k_diff_step(const float* __restrict__ st, float* __restrict__ out, const float4* __restrict__ sums,
                const float* __restrict__ mu, const float* __restrict__ lam, DiffK d,
                float* __restrict__ grid, unsigned blocks, NodeWork nodes, unsigned first) {
  __shared__ float4 part[G2P ? kPlanes * 3 * kWave : 1];
  __shared__ ScatterShared sh;  // (unused without P2G, then it takes no LDS)
  const StepConsts& k = d.k;
  const unsigned block = first + blockIdx.x;
  if (block >= blocks) {
    node_block(nodes, d, block - blocks);
    return;
  }
  const int lane = threadIdx.x & (kWave - 1);
  const int plane = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t p = (int64_t)block * kWave + lane, n = d.n;
  const bool valid = p < n;
  float x[3] = {0.f, 0.f, 0.f}, v[3] = {0.f, 0.f, 0.f}, C[9], F[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) C[i] = F[i] = 0.f;
  float mup = 0.f, lamp = 0.f;
  if (valid) {
    load_planes<3>(st, n, p, DX, x);
    load_planes<9>(st, n, p, DF, F);
    if (P2G) {
      mup = mu[p];
      lamp = lam[p];
    }
    if (!G2P) {
      load_planes<3>(st, n, p, DV, v);
      load_planes<9>(st, n, p, DC, C);
    }
  }
  Stencil sn = make_stencil(x, k);
  bool inside = valid && !sn.outside;
  if (G2P) {
    float s[16];
    if (plane < kPlanes) {
      plane_sums<true, false, false, false>(sums, sn, plane, d, nullptr, nullptr, 0.f, nullptr, s);
      put_plane<3>(part, plane, lane, s);
    }
    __syncthreads();
    sum_planes<3>(part, lane, s);
    if (inside) {
      float A[9];
#pragma unroll
      for (int i = 0; i < 9; ++i) {
        C[i] = k.dinv * s[3 + i];
        A[i] = ((i % 4 == 0) ? 1.0f : 0.0f) + k.dt * C[i];
      }
      mul_ab(A, F, F);
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        v[a] = s[a];
        x[a] = x[a] + k.dt * s[a];
      }
    } else if (valid) {
      load_planes<3>(st, n, p, DV, v);
      load_planes<9>(st, n, p, DC, C);
    }
    if (valid && plane == kPlanes) {
      store_planes<3>(out, n, p, DX, x);
      store_planes<3>(out, n, p, DV, v);
      store_planes<9>(out, n, p, DC, C);
      store_planes<9>(out, n, p, DF, F);
    }
    if (P2G) {
      sn = make_stencil(x, k);
      inside = valid && !sn.outside;
    }
  }
  if (!P2G) return;
  if (plane == kPlanes) {
    scatter_cells(sh, inside, sn, k.N);
  } else {
    float U[9], sv[3], V[9], R[9], tau[9], A[9];
    svd3_robust(F, U, sv, V);
    mul_abt(U, V, R);
    fc_stress(F, R, mup, lamp, tau);
    const float sc = stress_scale(d);
    float q0[3], qa[3];
#pragma unroll
    for (int i = 0; i < 9; ++i) A[i] = sc * tau[i] + d.mass * C[i];
#pragma unroll
    for (int r = 0; r < 3; ++r) q0[r] = d.mass * v[r];
    q_start(q0, A, of_plane(sn.ax[0].dp, plane), qa);
    const float wa = of_plane(sn.ax[0].w, plane);
    float4 row[9];
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const float wt = (wa * sn.ax[1].w[b]) * sn.ax[2].w[c];
        float q[3];
#pragma unroll
        for (int r = 0; r < 3; ++r) q[r] = qa[r] + A[3 * r + 1] * sn.ax[1].dp[b] + A[3 * r + 2] * sn.ax[2].dp[c];
        row[3 * b + c] = make_float4(wt * q[0], wt * q[1], wt * q[2], wt * d.mass);
      }
    scatter_runs<4>(sh, row, inside, sn, plane, k.N);
  }
  __syncthreads();
  scatter_nodes<4>(sh, plane, k.N, grid);
}

// ---------------------------------------------------------------- backward
// The adjoint of the P2G of substep s (P2GA: the momentum and mass adjoints
// `gm` of that substep, gathered) fused with the adjoint of the G2P of
// substep s-1 (G2PA: the grid velocity adjoint scattered into `gv_out`).
//   adj_src   P2GA: the partial adjoint of X_s the previous G2PA left (x and F
//             parts; the whole adjoint for particles outside the grid);
//             otherwise the full adjoint of X_s.
//   adj_dst   G2PA: the partial adjoint of X_{s-1} (may be adj_src);
//             otherwise the full adjoint of X_s.
// X_s = st_s (state before substep s), X_{s-1} = st_prev with tape velocities
// vel_prev. The mu and lambda adjoints are added into adj_mu, adj_lam.
//
// The fourth wavefront takes the mu and lambda adjoints off the others.
template <bool P2GA, bool G2PA>
__global__ void __launch_bounds__(kThreads)
    k_adj_step(const float* __restrict__ st_s, const float* __restrict__ mu, const float* __restrict__ lam,
               const float4* __restrict__ gm, const float* adj_src, const float* __restrict__ st_prev,
               const float4* __restrict__ vel_prev, float* adj_dst, float* __restrict__ adj_mu,
               float* __restrict__ adj_lam, float* __restrict__ gv_out, DiffK d, unsigned first) {
  __shared__ float4 part_p[P2GA ? kPlanes * 4 * kWave : 1];
  __shared__ float4 part_g[G2PA ? kPlanes * 4 * kWave : 1];
  __shared__ ScatterShared sh;  // (unused without G2PA)
  const int lane = threadIdx.x & (kWave - 1);
  const int plane = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t p = (int64_t)(first + blockIdx.x) * kWave + lane, n = d.n;
  const StepConsts& k = d.k;
  const bool valid = p < n;
  // adjoint of X_s
  float xb[3] = {0.f, 0.f, 0.f}, vb[3] = {0.f, 0.f, 0.f}, Cb[9], Fb[9];
  float xp[3] = {0.f, 0.f, 0.f}, Fp[9];  // of X_{s-1}
#pragma unroll
  for (int i = 0; i < 9; ++i) Cb[i] = Fb[i] = Fp[i] = 0.f;
  if (valid) {
    load_planes<3>(adj_src, n, p, DX, xb);
    load_planes<9>(adj_src, n, p, DF, Fb);
    if (!P2GA) {
      load_planes<3>(adj_src, n, p, DV, vb);
      load_planes<9>(adj_src, n, p, DC, Cb);
    }
    if (G2PA) {
      load_planes<3>(st_prev, n, p, DX, xp);
      load_planes<9>(st_prev, n, p, DF, Fp);
    }
  }

  if (P2GA) {
    float x[3] = {0.f, 0.f, 0.f}, v[3] = {0.f, 0.f, 0.f}, C[9], F[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) C[i] = F[i] = 0.f;
    float mup = 0.f, lamp = 0.f;
    if (valid) {
      load_planes<3>(st_s, n, p, DX, x);
      load_planes<9>(st_s, n, p, DF, F);
      load_planes<3>(st_s, n, p, DV, v);
      load_planes<9>(st_s, n, p, DC, C);
      mup = mu[p];
      lamp = lam[p];
    }
    const Stencil sn = make_stencil(x, k);
    const bool inside = valid && !sn.outside;
    float U[9], sv[3], V[9], R[9], tau[9], A[9], q0[3];
    const float sc = stress_scale(d);
    float s[16];
    svd3_robust(F, U, sv, V);
    mul_abt(U, V, R);
    if (plane < kPlanes) {
      fc_stress(F, R, mup, lamp, tau);
#pragma unroll
      for (int i = 0; i < 9; ++i) A[i] = sc * tau[i] + d.mass * C[i];
#pragma unroll
      for (int r = 0; r < 3; ++r) q0[r] = d.mass * v[r];
      // per node, pb . (m v + A dp) + mb m is what its weight multiplies
      plane_sums<false, true, true, false>(gm, sn, plane, d, q0, A, d.mass, nullptr, s);
      put_plane<4>(part_p, plane, lane, s);
    }
    __syncthreads();
    sum_planes<4>(part_p, lane, s);
    if (inside && plane == kPlanes) {
      const float* Ab = s + 3;
      float FmR[9], FmRFt[9];
#pragma unroll
      for (int i = 0; i < 9; ++i) FmR[i] = F[i] - R[i];
      mul_abt(FmR, F, FmRFt);
      float dmu = 0.f;
#pragma unroll
      for (int i = 0; i < 9; ++i) dmu += FmRFt[i] * (sc * Ab[i]);
      const float J = det3(F);
      adj_mu[p] += 2.0f * dmu;
      adj_lam[p] += ((J - 1.0f) * J) * (sc * Ab[0] + sc * Ab[4] + sc * Ab[8]);
    } else if (inside) {
      const float *pb = s, *Ab = s + 3;  // sum w pb, sum w pb dp^T
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        vb[q] = d.mass * pb[q];
        xb[q] += s[12 + q] - (A[q] * pb[0] + A[3 + q] * pb[1] + A[6 + q] * pb[2]);
      }
      // stress adjoint tb = sc Ab
      float tb[9];
#pragma unroll
      for (int i = 0; i < 9; ++i) tb[i] = sc * Ab[i];
      const float J = det3(F);
      float FmR[9];
#pragma unroll
      for (int i = 0; i < 9; ++i) FmR[i] = F[i] - R[i];
      const float trt = tb[0] + tb[4] + tb[8];
      // with R held: d/dF of 2 mu (F - R) F^T contracted with tb = 2 mu (tb F + tb^T (F - R))
      float tbF[9], tbtFmR[9];
      mul_ab(tb, F, tbF);
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c)
          tbtFmR[3 * r + c] = tb[r] * FmR[c] + tb[3 + r] * FmR[3 + c] + tb[6 + r] * FmR[6 + c];
#pragma unroll
      for (int i = 0; i < 9; ++i) Fb[i] += 2.0f * mup * (tbF[i] + tbtFmR[i]);
      // through R: Rbar = -2 mu tb F, M = R^T Rbar
      float M[9];
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c)
          M[3 * r + c] = -2.0f * mup * (R[r] * tbF[c] + R[3 + r] * tbF[3 + c] + R[6 + r] * tbF[6 + c]);
      float Sk[9], T1[9], Nm[9], UN[9], UNVt[9];
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) Sk[3 * r + c] = 0.5f * (M[3 * r + c] - M[3 * c + r]);
      mul_ab(Sk, V, T1);  // skew(M) V
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const float mt = V[r] * T1[c] + V[3 + r] * T1[3 + c] + V[6 + r] * T1[6 + c];
          const float den = sv[r] + sv[c];
          Nm[3 * r + c] = (r == c || den == 0.0f) ? 0.0f : mt / den;
        }
      mul_ab(U, Nm, UN);
      mul_abt(UN, V, UNVt);
#pragma unroll
      for (int i = 0; i < 9; ++i) Fb[i] += 2.0f * UNVt[i];
      // volumetric: lambda (2J - 1) tr(tb) dJ/dF, dJ/dF = cof(F)
      const float cv = lamp * (2.0f * J - 1.0f) * trt;
      const float cof[9] = {F[4] * F[8] - F[5] * F[7], F[5] * F[6] - F[3] * F[8], F[3] * F[7] - F[4] * F[6],
                            F[2] * F[7] - F[1] * F[8], F[0] * F[8] - F[2] * F[6], F[1] * F[6] - F[0] * F[7],
                            F[1] * F[5] - F[2] * F[4], F[2] * F[3] - F[0] * F[5], F[0] * F[4] - F[1] * F[3]};
#pragma unroll
      for (int i = 0; i < 9; ++i) Fb[i] += cv * cof[i];
#pragma unroll
      for (int i = 0; i < 9; ++i) Cb[i] = d.mass * Ab[i];
    } else if (valid) {  // the partial already holds the identity map
      load_planes<3>(adj_src, n, p, DV, vb);
      load_planes<9>(adj_src, n, p, DC, Cb);
    }
  }
  // (xb, vb, Cb, Fb) is the adjoint of X_s
  if (!G2PA) {
    // (adj_dst may be adj_src: no wavefront stores before all have read)
    __syncthreads();
    if (valid) store_state(adj_dst, n, p, plane, xb, vb, Cb, Fb);
    return;
  }
  // G2P of substep s-1: X_s = G2P(X_{s-1}); the adjoint of X_s flows back
  // to x and F of X_{s-1} and to the grid velocities of substep s-1:
  // x' = x + dt v', F' = (I + dt C') F, adjoints of v' and C' through them
  const Stencil sn = make_stencil(xp, k);
  const bool inside = valid && !sn.outside;
  float vbt[3], D[9], FbFt[9];  // D: Dinv times the adjoint of C'
#pragma unroll
  for (int a = 0; a < 3; ++a) vbt[a] = vb[a] + k.dt * xb[a];
  mul_abt(Fb, Fp, FbFt);
#pragma unroll
  for (int i = 0; i < 9; ++i) D[i] = k.dinv * (Cb[i] + k.dt * FbFt[i]);
  // per node, g . (vbt + D dp) is what its weight multiplies, and w (vbt + D dp)
  // the adjoint of its velocity
  float s[16];
  if (plane < kPlanes) {
    float4 row[9];
    plane_sums<false, true, false, true>(vel_prev, sn, plane, d, vbt, D, 0.f, row, s);
    put_plane<4>(part_g, plane, lane, s);
    scatter_runs<3>(sh, row, inside, sn, plane, k.N);
  } else {
    scatter_cells(sh, inside, sn, k.N);
  }
  __syncthreads();  // (also: all have read adj_src before any stores)
  sum_planes<4>(part_g, lane, s);
  if (inside) {
    if (plane == 0) {
#pragma unroll
      for (int q = 0; q < 3; ++q)
        xb[q] += s[12 + q] - (D[q] * s[0] + D[3 + q] * s[1] + D[6 + q] * s[2]);
      store_planes<3>(adj_dst, n, p, DX, xb);
    } else if (plane == 1) {
      float Fo[9];
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          // ((I + dt C')^T Fb')_rc
          float acc = 0.f;
#pragma unroll
          for (int q = 0; q < 3; ++q)
            acc += (((q == r) ? 1.0f : 0.0f) + (k.dt * k.dinv) * s[3 + 3 * q + r]) * Fb[3 * q + c];
          Fo[3 * r + c] = acc;
        }
      store_planes<9>(adj_dst, n, p, DF, Fo);
    }
  } else if (valid) {
    store_state(adj_dst, n, p, plane, xb, vb, Cb, Fb);  // the identity map
  }
  scatter_nodes<3>(sh, plane, k.N, gv_out);
}

// adjoint of the updated velocity (gadj.xyz) -> adjoints of the P2G momentum
// and mass (gadj, in place); clears `clear` (the next scatter's target)
__global__ void __launch_bounds__(256)
    k_adj_grid(float4* __restrict__ gadj, float4* __restrict__ clear, const float4* __restrict__ tv,
               const float4* __restrict__ tw, StepConsts k) {
  const size_t nodes = (size_t)k.N * k.N * k.N;
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nodes) return;
  if (clear) clear[t] = make_float4(0.f, 0.f, 0.f, 0.f);
  const float4 t0 = tv[t];
  const float4 t1 = tw[t];
  const float m = t0.w;
  float4 out = make_float4(0.f, 0.f, 0.f, 0.f);
  if (m > 0.0f) {
    const float4 g = gadj[t];
    float b0 = g.x, b1 = g.y, b2 = g.z;
    const int flags = (int)t1.w;
    if (flags & 1) { b0 = 0.f; b1 = 0.f; b2 = 0.f; }
    if ((flags & 2) && !(t1.y > 0.0f)) b1 = 0.f;  // max(0, v_y) is flat where it clamps
    // v = P / m + dt g e_y: dP = b / m, dm = -b . (P / m) / m
    const float py = t1.y - k.dt * k.gravity;
    out.x = b0 / m;
    out.y = b1 / m;
    out.z = b2 / m;
    out.w = -(b0 * t1.x + b1 * py + b2 * t1.z) / m;
  }
  gadj[t] = out;
}

__global__ void __launch_bounds__(256) k_zero4(float4* __restrict__ g, size_t n) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) g[t] = make_float4(0.f, 0.f, 0.f, 0.f);
}

DiffK diff_consts(const StepConsts& k, float mass, float volume, int64_t n) {
  DiffK d;
  d.k = k;
  d.mass = mass;
  d.volume = volume;
  // wall_flags' comparisons as node indices: i / N grows with i
  d.wall_lo = k.bcells;
  d.wall_hi = k.N - k.bcells;
  if (k.boundary_mode != MPM_BOUNDARY_CELLS) {
    auto first = [&](auto past) {
      int lo = 0, hi = k.N;
      while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if (past((float)mid / (float)k.N)) hi = mid;
        else lo = mid + 1;
      }
      return lo;
    };
    const float top = 1.0f - k.bfrac;
    d.wall_lo = first([&](float f) { return !(f < k.bfrac); });
    d.wall_hi = first([&](float f) { return f > top; });
  }
  d.n = n;
  return d;
}

size_t nodes_of(const StepConsts& k) { return (size_t)k.N * k.N * k.N; }
unsigned node_blocks(const StepConsts& k) { return (unsigned)((nodes_of(k) + 255) / 256); }
unsigned particle_blocks(int64_t n) { return (unsigned)((n + kWave - 1) / kWave); }

// launch(workgroups, first one) for all of `blocks`
template <class Launch>
void launch_blocks(unsigned blocks, const Launch& launch) {
  for (unsigned first = 0; first < blocks; first += kMaxBlocks) launch(dim3(std::min(blocks - first, kMaxBlocks)), first);
}

// the two halves of a tape slot: velocities (read by G2P), then the rest
const float4* tape_v(const float* tape) { return reinterpret_cast<const float4*>(tape); }
const float4* tape_w(const float* tape, const StepConsts& k) {
  return reinterpret_cast<const float4*>(tape) + nodes_of(k);
}
float4* tape_v(float* tape) { return reinterpret_cast<float4*>(tape); }
float4* tape_w(float* tape, const StepConsts& k) { return reinterpret_cast<float4*>(tape) + nodes_of(k); }

}  // namespace

// ---------------------------------------------------------------- no-allocation forward
// The scatter grid of the forward (4 floats per node) for callers that cannot
// allocate: one array per device, sized for grids up to kNoAllocMaxN^3 nodes,
// held until the process ends. Host code never uses the array's name (a
// host-side stand-in, not a device address): the device address comes from
// hipGetSymbolAddress, once per device with that device current.
static __device__ __align__(256) float4 scratch[(size_t)mpmk::kNoAllocMaxN * mpmk::kNoAllocMaxN *
                                                mpmk::kNoAllocMaxN];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float4* g_scratch_ptr[kMaxDevices] = {};

// The device address of the current device's copy of `scratch`.
hipError_t scratch_address(float4** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    g_scratch_ptr[dev] = static_cast<float4*>(p);
  }
  *out = g_scratch_ptr[dev];
  return hipSuccess;
}
}  // namespace

namespace mpmk {

hipError_t diff_forward_noalloc(const StepConsts& k, float mass, float volume, int64_t n,
                                const float* st, float* out, const float* mu, const float* lam,
                                float* tape, hipStream_t s) {
  if (k.N < 1 || k.N > kNoAllocMaxN) return hipErrorInvalidValue;
  float4* grid = nullptr;
  const hipError_t e = scratch_address(&grid);
  if (e != hipSuccess) return e;
  // diff_forward clears the first 4 N^3 floats with a kernel before the
  // scatter, whatever the last call left there
  return diff_forward(k, mass, volume, n, st, out, mu, lam, grid, tape, s);
}


// A substep's launch reads the sums of its own scatter, adds up the next
// substep's and clears those of the one after: three grids are in use at a
// time. With a tape for each substep, the sums of substep j lie in the tape of
// substep j + 1, which is written after they were read (the last substep's in
// `grid`); with one tape for all, in `grid` and its two halves in turn, and
// only the last substep, whose sums are in `grid`, writes it.
hipError_t diff_forward_steps(const StepConsts& k, float mass, float volume, int64_t n, int32_t steps,
                              const float* st0, float* states, int64_t state_stride, const float* mu,
                              const float* lam, float4* grid, float* tapes, int64_t tape_stride,
                              hipStream_t s) {
  const DiffK d = diff_consts(k, mass, volume, n);
  const unsigned gp = particle_blocks(n), gn = node_blocks(k);
  auto tape = [&](int32_t j) { return tapes + (size_t)j * (size_t)tape_stride; };
  auto sums = [&](int32_t j) -> float4* {
    if (j >= steps) return nullptr;
    const int32_t left = steps - 1 - j;
    if (tape_stride > 0) return left == 0 ? grid : tape_v(tape(j + 1));
    return left % 3 == 0 ? grid : left % 3 == 1 ? tape_v(tapes) : tape_w(tapes, k);
  };
  if (steps < 1) return hipGetLastError();
  hipLaunchKernelGGL(k_zero4, dim3(gn), dim3(256), 0, s, sums(0), nodes_of(k));
  if (n > 0 || steps > 1) {
    const NodeWork w = {nullptr, nullptr, nullptr, sums(1)};
    launch_blocks(gp + (steps > 1 ? gn : 0u), [&](dim3 g, unsigned first) {
      hipLaunchKernelGGL((k_diff_step<false, true>), g, dim3(kThreads), 0, s, st0, (float*)nullptr,
                         (const float4*)nullptr, mu, lam, d, (float*)sums(0), gp, w, first);
    });
  }
  for (int32_t j = 0; j < steps; ++j) {
    const float* in = j == 0 ? st0 : states + (size_t)(j - 1) * (size_t)state_stride;
    float* out = states + (size_t)j * (size_t)state_stride;
    const bool last = j + 1 == steps, taped = last || tape_stride > 0;
    const NodeWork w = {sums(j), taped ? tape_v(tape(j)) : nullptr, taped ? tape_w(tape(j), k) : nullptr, sums(j + 2)};
    launch_blocks(gp + (w.tv || w.clear ? gn : 0u), [&](dim3 g, unsigned first) {
      if (!last)
        hipLaunchKernelGGL((k_diff_step<true, true>), g, dim3(kThreads), 0, s, in, out, (const float4*)w.sums, mu, lam,
                           d, (float*)sums(j + 1), gp, w, first);
      else
        hipLaunchKernelGGL((k_diff_step<true, false>), g, dim3(kThreads), 0, s, in, out, (const float4*)w.sums, mu, lam,
                           d, (float*)nullptr, gp, w, first);
    });
  }
  return hipGetLastError();
}

hipError_t diff_forward(const StepConsts& k, float mass, float volume, int64_t n, const float* st,
                        float* out, const float* mu, const float* lam, float4* grid, float* tape,
                        hipStream_t s) {
  return diff_forward_steps(k, mass, volume, n, 1, st, out, 0, mu, lam, grid, tape, 0, s);
}

hipError_t diff_backward_steps(const StepConsts& k, float mass, float volume, int64_t n, int32_t steps,
                               const float* states, int64_t state_stride, const float* mu,
                               const float* lam, const float* tapes, int64_t tape_stride,
                               const float* adj_out, float* adj_in, float* adj_mu, float* adj_lam,
                               float4* grid2, float* work, hipStream_t s) {
  const DiffK d = diff_consts(k, mass, volume, n);
  const unsigned gp = particle_blocks(n), gn = node_blocks(k);
  const size_t nodes = nodes_of(k);
  float4* ga = grid2;
  float4* gb = steps > 1 ? grid2 + nodes : nullptr;  // a single substep needs one grid
  auto state = [&](int32_t j) { return states + (size_t)j * (size_t)state_stride; };
  auto tape = [&](int32_t j) { return tapes + (size_t)j * (size_t)tape_stride; };
  hipLaunchKernelGGL(k_zero4, dim3(gn), dim3(256), 0, s, ga, nodes);
  // the G2P adjoint of the last substep, from the caller's adjoint
  launch_blocks(gp, [&](dim3 g, unsigned first) {
    hipLaunchKernelGGL((k_adj_step<false, true>), g, dim3(kThreads), 0, s, (const float*)nullptr, (const float*)nullptr,
                       (const float*)nullptr, (const float4*)nullptr, adj_out, state(steps - 1),
                       tape_v(tape(steps - 1)), work, (float*)nullptr, (float*)nullptr, (float*)ga, d, first);
  });
  for (int32_t j = steps - 1; j >= 0; --j) {
    hipLaunchKernelGGL(k_adj_grid, dim3(gn), dim3(256), 0, s, ga, j > 0 ? gb : (float4*)nullptr,
                       tape_v(tape(j)), tape_w(tape(j), k), k);
    if (n == 0) continue;
    if (j > 0) {
      launch_blocks(gp, [&](dim3 g, unsigned first) {
        hipLaunchKernelGGL((k_adj_step<true, true>), g, dim3(kThreads), 0, s, state(j), mu, lam, (const float4*)ga,
                           (const float*)work, state(j - 1), tape_v(tape(j - 1)), work, adj_mu, adj_lam, (float*)gb, d,
                           first);
      });
      float4* t = ga;
      ga = gb;
      gb = t;
    } else {
      launch_blocks(gp, [&](dim3 g, unsigned first) {
        hipLaunchKernelGGL((k_adj_step<true, false>), g, dim3(kThreads), 0, s, state(0), mu, lam, (const float4*)ga,
                           (const float*)work, (const float*)nullptr, (const float4*)nullptr, adj_in, adj_mu, adj_lam,
                           (float*)nullptr, d, first);
      });
    }
  }
  return hipGetLastError();
}

hipError_t diff_backward(const StepConsts& k, float mass, float volume, int64_t n, const float* st,
                         const float* mu, const float* lam, const float* tape, const float* adj_out,
                         float* adj_in, float* adj_mu, float* adj_lam, float4* grid_adj, hipStream_t s) {
  // one substep: one grid, and adj_in holds the partial adjoint in between
  return diff_backward_steps(k, mass, volume, n, 1, st, 0, mu, lam, tape, 0, adj_out, adj_in, adj_mu,
                             adj_lam, grid_adj, adj_in, s);
}

}  // namespace mpmk
