// Rigid-body kernels of a dense 3D solve (gfx950).
//   k_rigid_force     momentum exchange on the bounce-back links with
//                     Ladd's moving-wall term at the local wall density, and
//                     the swept-cell term (common_d3_force.wgsl:171-222),
//                     over a box around the body; FP64 partials per block,
//                     summed in block order by the last block, which then
//                     appends the force record and integrates the body
//                     (d3_physics.wgsl:56-158, d3-body.mjs:234-297)
//   k_rigid_classify  solid bit and pull-link mask of every cell near the
//                     body at its new pose, over the union of the old and new
//                     neighbourhoods, so that cells the body left are cleared
// Cells farther than rc + 2 from the centre can be neither solid nor next to
// the body (a link is at most sqrt(3) long), so both kernels leave them out.
#include <hip/hip_runtime.h>
#include "dense.h"
#include "device_common.h"
#include "lattice_tables.h"
#include "rigid.h"
#include "rigid_device.h"

namespace lbm {

namespace {

// Cell coordinate k of a box edge of `edge` cells starting `half` below
// floor(c) on an axis of n cells (the whole axis when edge >= n).
__device__ __forceinline__ int box_coord(double c, int half, int edge, int n, int k) {
  if (edge >= n) return k;
  int x = (int)floor(c) - half + k;
  x %= n;
  return x < 0 ? x + n : x;
}

template <class ST, int Q>
__device__ __forceinline__ const typename ST::T* cell_block(const typename ST::T* f, uint32_t cell) {
  return f + (size_t)(cell / kLatBlock) * (Q * kLatBlock);
}

__device__ __forceinline__ void omega_from_L(const RigidBody* B, const double q[4], const double L[3], double w[3]) {
#pragma clang fp contract(off)
  double Lb[3];
  q_rot_inv(q, L, Lb);
  const double t[3] = {Lb[0] / B->I[0], Lb[1] / B->I[1], Lb[2] / B->I[2]};
  q_rot(q, t, w);
}

__device__ __forceinline__ void q_normalize(double q[4]) {
#pragma clang fp contract(off)
  const double n = sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
  if (!(n > 1e-12)) { q[0] = 1.0; q[1] = q[2] = q[3] = 0.0; return; }
  for (int k = 0; k < 4; k++) q[k] = q[k] / n;
}

// One integrator step with the measured force and torque.
__device__ void rigid_physics(RigidBody* B, const double F[3], const double T[3]) {
#pragma clang fp contract(off)
  for (int k = 0; k < 3; k++) { B->force[k] = F[k]; B->torque[k] = T[k]; }
  if (B->pinned) return;
  const double use = B->no_fluid ? 0.0 : 1.0;
  const double m = B->mass;
  double v[3];
  for (int k = 0; k < 3; k++) v[k] = B->v[k] + (use * F[k] / m + B->g[k]);
  if (B->planar) v[2] = 0.0;
  const double vmag = len3(v[0], v[1], v[2]);
  if (vmag > B->v_max) for (int k = 0; k < 3; k++) v[k] = v[k] * (B->v_max / vmag);
  double L[3];
  for (int k = 0; k < 3; k++) L[k] = B->L[k] + use * T[k];
  if (B->planar) { L[0] = 0.0; L[1] = 0.0; }
  double q[4] = {B->q[0], B->q[1], B->q[2], B->q[3]};
  double w[3];
  omega_from_L(B, q, L, w);
  if (B->planar) { w[0] = 0.0; w[1] = 0.0; }
  const double wmag = len3(w[0], w[1], w[2]);
  if (wmag > B->o_max) {
    const double s = B->o_max / wmag;
    for (int k = 0; k < 3; k++) { w[k] = w[k] * s; L[k] = L[k] * s; }
  }
  double e[4], qh[4];
  exp_map(w, 0.5, e);
  q_mul(e, q, qh);
  q_normalize(qh);
  double wh[3];
  omega_from_L(B, qh, L, wh);
  if (B->planar) { wh[0] = 0.0; wh[1] = 0.0; }
  double qn[4];
  exp_map(wh, 1.0, e);
  q_mul(e, q, qn);
  q_normalize(qn);
  for (int k = 0; k < 3; k++) {
    B->d[k] = B->d[k] + v[k];
    B->c[k] = win_wrap_pos(B->c[k] + v[k], B->win_n[k]);
    B->v[k] = v[k];
    B->L[k] = L[k];
    B->w[k] = wh[k];
  }
  for (int k = 0; k < 4; k++) B->q[k] = qn[k];
}

}  // namespace

// Cells of a force block, which has a wave more (the pose ahead).
constexpr uint32_t kForceCells = 256;

// 8000 box cells for a body of radius 6: a chain of latencies, not work.  All
// of a cell's populations are loaded at once (a load per link, each waited for,
// took 14.2 us where this takes 12.0).
template <int Q, class ST>
__global__ void __launch_bounds__(kForceCells + 64) k_rigid_force(const typename ST::T* __restrict__ f, RigidArgs a) {
  using L = Lattice<Q>;
  using T = typename ST::T;
  __shared__ double lds[16 * 6];
  __shared__ bool last;
  __shared__ double ahead[7];  // the pose one step ahead: centre, orientation
  const RigidBody* B = a.body;
  const int tid = threadIdx.x;
  const bool swept = B->swept;
  // a wave of its own, beside the links of the others
  if (tid == kForceCells && swept) {
    // by v and the cached omega (common_d3_geometry.wgsl get_phi3Ahead)
    const double w[3] = {B->w[0], B->w[1], B->w[2]};
    const double q[4] = {B->q[0], B->q[1], B->q[2], B->q[3]};
    double e[4], qa[4];
    exp_map(w, 1.0, e);
    q_mul(e, q, qa);
    for (int k = 0; k < 3; k++) ahead[k] = B->c[k] + B->v[k];
    for (int k = 0; k < 4; k++) ahead[3 + k] = qa[k];
  }
  double fv[6] = {0, 0, 0, 0, 0, 0};
  const uint32_t t = blockIdx.x * kForceCells + tid;
  const uint32_t nbox = (uint32_t)a.fbox[0] * a.fbox[1] * a.fbox[2];
  const bool mine = tid < (int)kForceCells && t < nbox;
  double r[3] = {0, 0, 0}, fx = 0, fy = 0, fz = 0;
  int x = 0, y = 0, z = 0;
  bool close = false, solid_now = false;
  double fi[Q];  // the cell's populations, unshifted: all loads at once
  if (mine) {
    const int kx = t % a.fbox[0], ky = (t / a.fbox[0]) % a.fbox[1], kz = t / (a.fbox[0] * a.fbox[1]);
    x = box_coord(B->c[0], a.half, a.fbox[0], a.nx, kx);
    y = box_coord(B->c[1], a.half, a.fbox[1], a.ny, ky);
    z = box_coord(B->c[2], a.half, a.fbox[2], a.nz, kz);
    body_delta(B, x, y, z, r);
    close = len3(r[0], r[1], r[2]) <= B->rc + 2.0;
  }
  if (close) {
    const uint32_t cell = (uint32_t)((z * a.ny + y) * a.nx + x);
    const T* blk = cell_block<ST, Q>(f, cell);
    const uint32_t lo = cell % kLatBlock;
    solid_now = a.cls[cell] & 1;
    const uint32_t lm = a.links[cell];
    float g[Q];
#pragma unroll
    for (int i = 0; i < Q; i++) g[i] = ST::load(blk + i * kLatBlock, lo);
#pragma unroll
    for (int i = 0; i < Q; i++) fi[i] = (double)g[i] + (double)L::w[i];
    if (!solid_now && lm) {
      double us[3];
      body_velocity(B, x, y, z, us);
      double rho_w = 1.0;
      if (B->rho_w_local) {
        rho_w = 0.0;
#pragma unroll
        for (int i = 0; i < Q; i++) rho_w += fi[i];
      }
#pragma unroll
      for (int i = 1; i < Q; i++) {
        if (!((lm >> i) & 1u)) continue;
        const double eu = L::ex[i] * us[0] + L::ey[i] * us[1] + L::ez[i] * us[2];
        const double m = 2.0 * fi[L::opp[i]] + 2.0 * (double)L::w[i] * rho_w * eu * 3.0;
        fx -= L::ex[i] * m;
        fy -= L::ey[i] * m;
        fz -= L::ez[i] * m;
      }
    }
  }
  __syncthreads();
  if (close && swept) {
    const double ca[3] = {ahead[0], ahead[1], ahead[2]};
    const double qa[4] = {ahead[3], ahead[4], ahead[5], ahead[6]};
    if (solid_now != (body_phi(B, ca, qa, x, y, z) < 0.0)) {
      double mx = 0, my = 0, mz = 0;
#pragma unroll
      for (int i = 0; i < Q; i++) {
        mx += fi[i] * L::ex[i];
        my += fi[i] * L::ey[i];
        mz += fi[i] * L::ez[i];
      }
      const double s = solid_now ? -1.0 : 1.0;
      fx += s * mx;
      fy += s * my;
      fz += s * mz;
    }
  }
  if (close) {
    fv[0] = fx; fv[1] = fy; fv[2] = fz;
    fv[3] = r[1] * fz - r[2] * fy;
    fv[4] = r[2] * fx - r[0] * fz;
    fv[5] = r[0] * fy - r[1] * fx;
  }
  block_sum<6>(fv, lds);
  const unsigned nblocks = gridDim.x;
  if (tid == 0) {
    for (int k = 0; k < 6; k++) a.partials[(size_t)blockIdx.x * 6 + k] = fv[k];
    __threadfence();
    last = atomicAdd(a.counter, 1u) == nblocks - 1;
  }
  __syncthreads();
  if (!last) return;
  __threadfence();
  // wave 0: lane l sums blocks l, l + 64, ... in order, then a fixed
  // butterfly, so the totals repeat bit for bit
  if (tid >= 64) return;
  double tot[6] = {0, 0, 0, 0, 0, 0};
  for (unsigned j = tid; j < nblocks; j += 64) {
    double v[6];
#pragma unroll
    for (int k = 0; k < 6; k++)
      v[k] = __hip_atomic_load(&a.partials[(size_t)j * 6 + k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int k = 0; k < 6; k++) tot[k] += v[k];
  }
#pragma unroll
  for (int k = 0; k < 6; k++) tot[k] = wave_sum(tot[k]);
  if (tid == 0) {
    *a.counter = 0u;
    const unsigned long long n = *a.written;
    for (int k = 0; k < 6; k++) a.history[(size_t)(n % a.hist_cap) * 6 + k] = tot[k];
    *a.written = n + 1;
    const double F[3] = {tot[0], tot[1], tot[2]}, Tq[3] = {tot[3], tot[4], tot[5]};
    rigid_physics(a.body, F, Tq);
  }
}

// Half a wave evaluates a cell's links, a lane a direction, where a thread a
// cell goes through up to Q - 1 sources one after the other.  A small box has
// half a wave per cell from the start (WIDE false); in a large one, most of
// whose cells are far from the surface, a lane first takes each cell's own
// distance and the half waves then go through the cells next to it.
template <int Q, bool WIDE>
__global__ void __launch_bounds__(256) k_rigid_classify(RigidArgs a) {
  using L = Lattice<Q>;
  const RigidBody* B = a.body;
  const uint32_t t = WIDE ? blockIdx.x * blockDim.x + threadIdx.x : blockIdx.x * (blockDim.x >> 5) + (threadIdx.x >> 5);
  const int i = threadIdx.x & 31, half = threadIdx.x & 32;
  const uint32_t nbox = (uint32_t)a.cbox[0] * a.cbox[1] * a.cbox[2];
  const bool inside = t < nbox;
  const double c[3] = {B->c[0], B->c[1], B->c[2]};
  const double q[4] = {B->q[0], B->q[1], B->q[2], B->q[3]};
  int x = 0, y = 0, z = 0;
  bool solid = false, near = false;
  if (inside) {
    const int kx = t % a.cbox[0], ky = (t / a.cbox[0]) % a.cbox[1], kz = t / (a.cbox[0] * a.cbox[1]);
    // the box starts below both the new centre and the previous one (c - v)
    x = box_coord(fmin(c[0], c[0] - B->v[0]), a.half, a.cbox[0], a.nx, kx);
    y = box_coord(fmin(c[1], c[1] - B->v[1]), a.half, a.cbox[1], a.ny, ky);
    z = box_coord(fmin(c[2], c[2] - B->v[2]), a.half, a.cbox[2], a.nz, kz);
    double r[3];
    body_delta(B, x, y, z, r);
    if (len3(r[0], r[1], r[2]) <= B->rc + 2.0) {
      const double phi = body_phi(B, c, q, x, y, z);
      solid = phi < 0.0;
      // a signed distance is 1-Lipschitz and a link at most sqrt(3) long, so
      // only cells this close can pull from a solid cell
      near = !solid && phi < 1.75;
    }
  }
  int ex = 0, ey = 0, ez = 0;  // this lane's direction
#pragma unroll
  for (int k = 1; k < Q; k++)
    if (i == k) ex = L::ex[k], ey = L::ey[k], ez = L::ez[k];
  const bool moving = i >= 1 && i < Q;
  // the half wave's links of the cell (sx, sy, sz)
  auto links_of = [&](bool wanted, int sx, int sy, int sz) {
    const bool link = wanted && moving && body_phi(B, c, q, sx - ex, sy - ey, sz - ez) < 0.0;
    return (uint32_t)(__ballot(link) >> half);
  };
  uint32_t lm = 0;
  if constexpr (WIDE) {
    for (uint32_t todo = (uint32_t)(__ballot(near) >> half); todo; todo &= todo - 1) {
      const int lane = __ffs(todo) - 1;
      const uint32_t m = links_of(true, __shfl(x, lane, 32), __shfl(y, lane, 32), __shfl(z, lane, 32));
      if (i == lane) lm = m;
    }
  } else {
    lm = links_of(near, x, y, z);
  }
  if (inside && (WIDE || i == 0)) {
    const uint32_t cell = (uint32_t)((z * a.ny + y) * a.nx + x);
    a.cls[cell] = solid ? 1 : (lm ? 2 : 0);
    a.links[cell] = lm;
  }
}

uint32_t rigid_force_blocks(const RigidArgs& a) {
  return ((uint32_t)a.fbox[0] * a.fbox[1] * a.fbox[2] + kForceCells - 1) / kForceCells;
}

template <int Q>
static hipError_t force_q(int storage, const void* f, const RigidArgs& a, hipStream_t s) {
  const dim3 grid(rigid_force_blocks(a)), block(kForceCells + 64);
  if (storage == kF32) hipLaunchKernelGGL((k_rigid_force<Q, StoreF32>), grid, block, 0, s, (const float*)f, a);
  else if (storage == kF16)
    hipLaunchKernelGGL((k_rigid_force<Q, StoreF16>), grid, block, 0, s, (const uint16_t*)f, a);
  else hipLaunchKernelGGL((k_rigid_force<Q, StoreBF16>), grid, block, 0, s, (const uint16_t*)f, a);
  return hipGetLastError();
}

hipError_t launch_rigid_force(int q, int storage, const void* f, const RigidArgs& a, hipStream_t s) {
  return q == 19 ? force_q<19>(storage, f, a, s) : force_q<27>(storage, f, a, s);
}

// Largest box, in cells, that takes half a wave a cell.  Beyond, most of its
// cells need one distance only, and 32 threads for each of 2^27 cells would be
// more than a launch's 2^32.  us, half a wave a cell and WIDE (a thread a cell
// that also goes through its own links, before either): 14k cells 6.8, 12.0
// (15.8); 22k 9.6, 11.0 (16.0); 33k 13.4, 10.3 (15.7); 64k 21.6, 11.4 (14.2);
// 373k 108, 22.4 (33.6); 2.3M 634, 66 (132).
constexpr uint32_t kSmallBox = 24000;

template <int Q>
static hipError_t classify_q(const RigidArgs& a, hipStream_t s) {
  const uint32_t nbox = (uint32_t)a.cbox[0] * a.cbox[1] * a.cbox[2];
  if (nbox <= kSmallBox) hipLaunchKernelGGL((k_rigid_classify<Q, false>), dim3((nbox + 7) / 8), dim3(256), 0, s, a);
  else hipLaunchKernelGGL((k_rigid_classify<Q, true>), dim3((nbox + 255) / 256), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_rigid_classify(int q, const RigidArgs& a, hipStream_t s) {
  return q == 19 ? classify_q<19>(a, s) : classify_q<27>(a, s);
}

}  // namespace lbm
