// One cell of the dense step, shared by the one-step kernels
// (dense_step.h) and the multi-step ones (dense_pair.hip, dense_multi.hip): halfway
// bounce-back with the momentum it exchanges, the sponge weight, and the
// BGK/TRT relaxation in pair form.  Every kernel runs the same arithmetic
// here, so a step's result does not depend on which of them took it.
#pragma once
#include <hip/hip_runtime.h>
#include "collide.h"
#include "dense.h"
#include "device_common.h"
#include "lattice_pairs.h"
#include "lattice_tables.h"

namespace lbm {

// Sum of force slots [first, last) of step `rec`.  The order is that of 256
// lanes whatever the block: lane l takes slots l, l + 256, ... in order, a
// butterfly folds each 64 lanes, and the four results are added in order.  This
// is one of the four waves' worth, into out[6] (all 64 lanes of the wave active).
// With `cells` a slot holds a boundary cell's force alone (3 doubles), and its
// torque is taken here; otherwise a slot is a tile's force and torque (6
// doubles).  The slots come from other XCDs' caches, so a wave's time is the
// latency of its loads: those of two slots are in flight together (more would
// cost the step kernels this is part of their occupancy).
template <bool PERIODIC, bool CELLS>
__device__ __forceinline__ void sum_force_wave(const ForceSum& f, int rec, uint32_t first, uint32_t last, int part,
                                               int lane, double* out) {
  const double* p = f.partials + (size_t)rec * f.stride;
  double v[6] = {0, 0, 0, 0, 0, 0};
  if (CELLS && f.cells) {
    constexpr int B = PERIODIC ? 1 : 2;
    for (uint32_t s0 = first + part * 64 + lane; s0 < last; s0 += B * 256) {
      uint32_t c[B];
      double F[B][3];
#pragma unroll
      for (int k = 0; k < B; k++) {
        const uint32_t s = min(s0 + k * 256, last - 1);
        c[k] = f.cells[s];
#pragma unroll
        for (int j = 0; j < 3; j++) F[k][j] = p[(size_t)s * 3 + j];
      }
#pragma unroll
      for (int k = 0; k < B; k++) {
        if (k > 0 && s0 + k * 256 >= last) break;
        const uint32_t row = div_invariant(c[k], f.div_nx), z = div_invariant(row, f.div_ny);
        double rx = (double)(c[k] - row * f.nx) - f.centre[0], ry = (double)(row - z * f.ny) - f.centre[1],
               rz = (double)z - f.centre[2];
        if constexpr (PERIODIC) {  // 2D: nearest periodic image
          rx -= f.nx * rint(rx / f.nx);
          ry -= f.ny * rint(ry / f.ny);
          rz = 0.0;
        }
        const double fx = F[k][0], fy = F[k][1], fz = F[k][2];
        v[0] += fx;
        v[1] += fy;
        v[2] += fz;
        v[3] += ry * fz - rz * fy;
        v[4] += rz * fx - rx * fz;
        v[5] += rx * fy - ry * fx;
      }
    }
  } else {
    for (uint32_t s = first + part * 64 + lane; s < last; s += 256) {
#pragma unroll
      for (int k = 0; k < 6; k++) v[k] += p[(size_t)s * 6 + k];
    }
  }
#pragma unroll
  for (int k = 0; k < 6; k++) {
    const double t = wave_sum(v[k]);
    if (lane == 0) out[k] = t;
  }
}
// Appends the records of a launch of up to MAX steps to the history, or this
// block's share of it: block `block` of `blocks` sums chunks block, block +
// blocks, ..., and the last of them to end adds up the chunks.  None waits for
// another.  The whole block (64 threads or more) takes part.
// One block alone takes 2 us per 512 slots, which a large body's launches waited
// for: us a step, one block and shared, D3Q19 120^3 with radius 30 79.4 and 56,
// 96^3 with 24 35.3 and 26.7, f16 27.2 and 21.2.
// CELLS false: f holds no boundary cells, one chunk.
template <bool PERIODIC, int MAX, bool CELLS = true>
__device__ __forceinline__ void append_force_records(const ForceSum& f, uint32_t block, uint32_t blocks) {
  constexpr int ITEMS = MAX * 4 > 16 ? MAX * 4 : 16;
  __shared__ double part[ITEMS][6];
  __shared__ bool last_block;
  const int tid = threadIdx.x + threadIdx.y * blockDim.x, waves = (blockDim.x * blockDim.y) >> 6;
  const int n = MAX == 1 ? 1 : f.steps;
  const bool whole = !CELLS || f.chunks == 1;
  const uint32_t size = whole ? f.nslots : kForceChunk;
  const int batch = max(1, waves / (4 * n));  // chunks at a time
  for (uint32_t c0 = block; c0 < (CELLS ? f.chunks : 1u); c0 += batch * blocks) {
    for (int w = tid >> 6; w < batch * 4 * n; w += waves) {
      const uint32_t c = c0 + (w / (4 * n)) * blocks;
      if (c >= (CELLS ? f.chunks : 1u)) break;
      sum_force_wave<PERIODIC, CELLS>(f, (w >> 2) % n, c * size, min(f.nslots, (c + 1) * size), w & 3, tid & 63, part[w]);
    }
    __syncthreads();
    if (tid < batch * 6 * n && c0 + (tid / (6 * n)) * blocks < (CELLS ? f.chunks : 1u)) {
      const int q = tid / 6, k = tid - q * 6;
      const uint32_t c = c0 + (q / n) * blocks;
      const double v = ((part[q * 4][k] + part[q * 4 + 1][k]) + part[q * 4 + 2][k]) + part[q * 4 + 3][k];
      if (whole) f.history[(size_t)((*f.written + q % n) % f.capacity) * 6 + k] = v;
      else __hip_atomic_store(&f.chunk_sums[((size_t)c * n + q % n) * 6 + k], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
  }
  if (whole) {
    if (tid == 0) *f.written += n;
    return;
  }
  // The chunk sums are the only data that pass between blocks, written and read
  // at agent scope past the XCDs' caches, by the first wave (at most 48 lanes);
  // its wait orders them before the count.  A release and an acquire here would
  // write back and drop whole caches in the middle of a step (D3Q27 112^3: 63.5
  // us a step for 60).
  if (tid == 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    last_block = __hip_atomic_fetch_add(f.arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == blocks - 1;
  }
  __syncthreads();
  if (!last_block) return;
  // lane l takes chunks l, l + 64, ... in order, then a butterfly
  const unsigned long long at = *f.written;
  for (int w = tid >> 6; w < 6 * n; w += waves) {
    double v = 0.0;
    for (uint32_t c = tid & 63; c < f.chunks; c += 64)
      v += __hip_atomic_load(&f.chunk_sums[(size_t)c * n * 6 + w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v = wave_sum(v);
    if ((tid & 63) == 0) f.history[(size_t)((at + w / 6) % f.capacity) * 6 + w % 6] = v;
  }
  __syncthreads();
  if (tid == 0) {
    *f.arrived = 0u;
    *f.written = at + n;
  }
}

// Slot of a boundary cell: the cells' ascending rank, from a bit mask and a
// base count per 64 cells.
__device__ __forceinline__ uint32_t boundary_slot(const BoundaryRank* r, uint32_t cell) {
  const BoundaryRank b = r[cell / 64];
  return b.base + (uint32_t)__popcll(b.mask & ((1ull << (cell % 64)) - 1ull));
}

// Signed distance of the pinned body at cell (x, y, z), binary32 with one
// rounding per operation (no contraction), the same value k_classify and the
// oracle compute:
//   sphere  phi = sqrt((x-cx)^2 + (y-cy)^2 + (z-cz)^2) - a
//           (common_d3_geometry.wgsl:119, :174-187)
//   circle  nearest periodic image of (x-cx, y-cy), then length - a
//           (common_geometry.wgsl:94-108)
__device__ __forceinline__ float body_phi(int shape, float radius, float cx, float cy, float cz, int nx, int ny,
                                          int x, int y, int z) {
  float dx = sub_rn((float)x, cx);
  float dy = sub_rn((float)y, cy);
  if (shape == 2) {
    const float W = (float)nx, H = (float)ny;
    dx = sub_rn(dx, mul_rn(W, rintf(div_rn(dx, W))));
    dy = sub_rn(dy, mul_rn(H, rintf(div_rn(dy, H))));
    return sub_rn(sqrt_rn(add_rn(mul_rn(dx, dx), mul_rn(dy, dy))), radius);
  }
  const float dz = sub_rn((float)z, cz);
  const float s = add_rn(add_rn(mul_rn(dx, dx), mul_rn(dy, dy)), mul_rn(dz, dz));
  return sub_rn(sqrt_rn(s), radius);
}

// Is the cell on a face with a halfway wall.
__device__ __forceinline__ bool on_wall_face(const StepArgs& a, int x, int y, int z) {
  return (a.wall_mask & 1 && (x == 0 || x == a.nx - 1)) || (a.wall_mask & 2 && (y == 0 || y == a.ny - 1)) ||
         (a.wall_mask & 4 && (z == 0 || z == a.nz - 1));
}

// Bit i set for the directions whose component on `axis` is v.
template <int Q>
__host__ __device__ constexpr uint32_t dirs_with(int axis, int v) {
  uint32_t m = 0;
  for (int i = 0; i < Q; i++) {
    const int e = axis == 0 ? Lattice<Q>::ex[i] : (axis == 1 ? Lattice<Q>::ey[i] : Lattice<Q>::ez[i]);
    if (e == v) m |= 1u << i;
  }
  return m;
}

// Halfway bounce-back of a cell next to the body (link mask `lm`) or on a
// wall face: the body first, then the walls (common_d3_step.wgsl:250-276).
// w_i = w_opp(i), so a reflected population keeps its shift.  own(j) is the
// cell's own pre-stream population j; link(i) what a moving body's surface
// adds to the reflected population (0 for a body at rest).  F accumulates the
// momentum exchange on the body of a fluid cell, -e_i (2 f_opp).
template <int Q, class Own, class Link>
__device__ __forceinline__ void reflect_cell(const StepArgs& a, int x, int y, int z, bool solid, uint32_t lm, bool face,
                                             float (&g)[Q], double (&F)[3], Own own, Link link) {
  using L = Lattice<Q>;
  const int nx = a.nx, ny = a.ny, nz = a.nz;
#pragma unroll
  for (int i = 1; i < Q; i++) {
    const int ex = L::ex[i], ey = L::ey[i], ez = L::ez[i];
    if ((lm >> i) & 1u) {
      g[i] = own(L::opp[i]);
      link(i, g[i]);
      if (!solid) {
        const double m = 2.0 * ((double)g[i] + (double)L::w[i]);
        if (ex == 1) F[0] -= m; else if (ex == -1) F[0] += m;
        if (ey == 1) F[1] -= m; else if (ey == -1) F[1] += m;
        if (ez == 1) F[2] -= m; else if (ez == -1) F[2] += m;
      }
    } else if (face) {
      const bool xo = (ex == 1 && x == 0) || (ex == -1 && x == nx - 1);
      const bool yo = (ey == 1 && y == 0) || (ey == -1 && y == ny - 1);
      const bool zo = (ez == 1 && z == 0) || (ez == -1 && z == nz - 1);
      const bool yWall = (a.wall_mask & 2) && yo;
      if (((a.wall_mask & 1) && xo) || yWall || ((a.wall_mask & 4) && zo)) {
        float corr = 0.f;
        if (ex != 0 && yWall) {
          // moving y-wall (common_walls.wgsl:27-31): 2 w e_x u_wall / cs2
          const float uw = (ey == 1) ? a.wall_u0 : a.wall_u1;
          corr = 2.f * L::w[i] * (float)ex * uw / (1.0f / 3.0f);
        }
        g[i] = own(L::opp[i]) + corr;
      }
    }
  }
}

// The same for directions given as masks, links `lm` and wall crossings
// `wall`, without a branch per direction (a wave takes it whole, and a
// two-step block waits for its slowest wave): own(i) is the value direction i
// reflects to before a moving wall's term; ylo, yhi: the cell lies on the
// wall at y = 0, at y = ny - 1.
template <int Q, class Own>
__device__ __forceinline__ void reflect_masked(const StepArgs& a, bool ylo, bool yhi, bool solid, uint32_t lm, uint32_t wall,
                                               float (&g)[Q], double (&F)[3], Own own) {
  using L = Lattice<Q>;
  const uint32_t back = lm | wall;
  const bool fluid = !solid;
#pragma unroll
  for (int i = 1; i < Q; i++) {
    const int ex = L::ex[i], ey = L::ey[i], ez = L::ez[i];
    const bool link = (lm >> i) & 1u;
    float v = own(i);
    if (ex != 0 && ey != 0) {
      // moving y-wall (common_walls.wgsl:27-31): 2 w e_x u_wall / cs2
      const float uw = (ey == 1) ? a.wall_u0 : a.wall_u1;
      const float corr = (ey == 1 ? ylo : yhi) ? 2.f * L::w[i] * (float)ex * uw / (1.0f / 3.0f) : 0.f;
      v = link ? v : v + corr;
    }
    g[i] = ((back >> i) & 1u) ? v : g[i];
    // a link's exchange, half of it: doubling is exact, so it is left to the end
    const double m = link && fluid ? (double)g[i] + (double)L::w[i] : 0.0;
    if (ex == 1) F[0] -= m; else if (ex == -1) F[0] += m;
    if (ey == 1) F[1] -= m; else if (ey == -1) F[1] += m;
    if (ez == 1) F[2] -= m; else if (ez == -1) F[2] += m;
  }
#pragma unroll
  for (int k = 0; k < 3; k++) F[k] *= 2.0;
}

// rho - 1 and the momentum of a cell from its pair sums.  D2Q9's f32 weights
// do not sum to 1 (wsum_m1); the 3D sets' do exactly.  The momentum sums start
// from -0, the identity of floating-point addition, so that their first term
// costs no instruction (0 + x is not x when x is -0).
template <int Q>
__device__ __forceinline__ void cell_sums(const StepArgs& a, float g0, const float (&S)[Pairs<Q>::NP],
                                          const float (&D)[Pairs<Q>::NP], float& drho, float& mx, float& my, float& mz) {
  using L = Lattice<Q>;
  drho = Q == 9 ? g0 + a.wsum_m1 : g0;
  mx = my = mz = -0.f;
#pragma unroll
  for (int k = 0; k < Pairs<Q>::NP; k++) {
    const int i = Pairs<Q>::lo(k);
    drho += S[k];
    if (L::ex[i] == 1) mx += D[k]; else if (L::ex[i] == -1) mx -= D[k];
    if (L::ey[i] == 1) my += D[k]; else if (L::ey[i] == -1) my -= D[k];
    if (L::ez[i] == 1) mz += D[k]; else if (L::ez[i] == -1) mz -= D[k];
  }
}

// rho - 1, rho, the velocity (momentum with the Guo half-force over rho) and
// u.u, u.F of a cell, with a uniform body force (FRC) or none.  The velocity's
// products stay out of later contractions: a sum of two components would
// otherwise take one of them unrounded into an FMA wherever the compiler sees
// both together, and the kernels would differ by a rounding.
template <int Q, bool FRC>
__device__ __forceinline__ void cell_moments(const StepArgs& a, float g0, const float (&S)[Pairs<Q>::NP],
                                             const float (&D)[Pairs<Q>::NP], float& drho, float& rho, float& ux,
                                             float& uy, float& uz, float& usq, float& uF) {
  float mx, my, mz;
  cell_sums<Q>(a, g0, S, D, drho, mx, my, mz);
  rho = 1.f + drho;
  const float rinv = recip_nr(fmaxf(rho, 1e-6f));
  // Guo: u = u* + F / (2 rho); half of F is exact
  if constexpr (FRC) {
    mx += 0.5f * a.F[0];
    my += 0.5f * a.F[1];
    mz += 0.5f * a.F[2];
  }
  {
#pragma clang fp contract(off)
    ux = mx * rinv;
    uy = my * rinv;
    uz = mz * rinv;
  }
  usq = ux * ux + uy * uy + uz * uz;
  uF = FRC ? ux * a.F[0] + uy * a.F[1] + uz * a.F[2] : 0.f;
}

// Blend weight of the sponge: d is the distance to the nearest face of the
// masked axes, position p of n cells away from an axis' faces by
// sponge_distance.
__device__ __forceinline__ float sponge_distance(bool masked, float p, int n) {
  return masked ? fminf(p, (float)(n - 1) - p) : 1e30f;
}
__device__ __forceinline__ float sponge_weight(const StepArgs& a, float d) {
  float sp = 0.f;
  // beyond the band d / w >= 1 rounds to >= 1, so t clamps to 0 there:
  // only cells inside the band pay for the division
  if (a.sponge_w > 0.f && d < a.sponge_w) {
    float t = 1.f - d / a.sponge_w;
    t = fminf(fmaxf(t, 0.f), 1.f);
    sp = t * t * (3.f - 2.f * t);
  }
  return sp;
}

// Collides pair by pair.  With g+ = (g_i + g_j)/2, g- = (g_i - g_j)/2
// (j = opp i) and the equilibrium split into its even part
//   A = w (rho - 1 + rho (4.5 (e.u)^2 - 1.5 u.u))
// and odd part B = 3 w rho (e.u), BGK/TRT with Guo forcing reads
//   P = g+ - omega   (g+ - A) + (1 - omega/2)   w (9 (e.u)(e.F) - 3 u.F)
//   M = g- - omega_m (g- - B) + (1 - omega_m/2) 3 w (e.F)
//   g_i' = P + M,  g_j' = P - M,
// which is the BGK line plus the TRT delta terms of plans/TRT.md:333-349
// regrouped (omega_m = omega gives BGK).  The sponge blends P and M
// toward the even and odd parts of feq(1, U_far) - w (SP).
//
// It is evaluated doubled: P2 = 2P and M2 = 2M from S = 2 g+ and D = 2 g-
// with 2w in place of w (and the host's pair constants doubled), then
// g_i' = fma(1/2, P2, M2/2), g_j' = fma(1/2, P2, -M2/2).  Scaling by two
// commutes with rounding, so every intermediate is exactly twice its
// undoubled value and the outputs are bit for bit P + M and P - M, without
// the two halvings per pair.
//
// Rounding: every relaxation keeps the form h - omega (h - eq), and the exact
// f32 weight w is the LAST factor of A and B.  A pre-rounded constant such as
// f32(3 w) or f32((1 - omega_m)/2) would carry the same relative bias (~1e-8)
// into every cell and every step, which breaks mass/momentum conservation
// systematically: the error then grows linearly in time instead of as a
// random walk.
//
// rest(g_0', r) and pair(k, i, j, g_i', g_j', r_i, r_j) take the results with
// their dither bits (hsh: this cell and step's hash).
template <int Q, class ST, bool SP, bool FRC, bool DIFF, class Rest, class Pair>
__device__ __forceinline__ void relax_cell(const StepArgs& a, float g0, const float (&S)[Pairs<Q>::NP],
                                           const float (&D)[Pairs<Q>::NP], float drho, float rho, float ux, float uy,
                                           float uz, float usq, float uF, float Fx, float Fy, float Fz, float sp,
                                           uint32_t hsh, Rest rest, Pair pair) {
  using L = Lattice<Q>;
  const float om = a.omega, omm = a.omega_m;
  const float c0 = drho - 1.5f * rho * usq;
  const float g3uF2 = FRC ? 6.f * a.guo * uF : 0.f;  // 2 (3 (1 - omega/2) u.F)
  {
    const float w = L::w[0];
    float p = g0 - om * (g0 - w * c0);
    if constexpr (FRC) p -= w * (0.5f * g3uF2);
    if constexpr (SP) p += sp * (a.ae[13] - p);
    rest(p, ST::dither(hsh, 0));
  }
#pragma unroll
  for (int k = 0; k < Pairs<Q>::NP; k++) {
    const int i = Pairs<Q>::lo(k);
    const int j = L::opp[i];
    const float w = L::w[i], w2 = 2.f * L::w[i];
    const float eu = edot<Q>(i, ux, uy, uz);
    const float t = rho * eu;
    const float X = c0 + 4.5f * (t * eu);
    float P2 = S[k] - om * (S[k] - w2 * X);
    float M2 = D[k] - omm * (D[k] - w2 * (3.f * t));
    if constexpr (FRC) {
      // Guo source, even and odd parts (doubled): (1 - omega/2) w (9
      // (e.u)(e.F) - 3 u.F) and (1 - omega_m/2) 3 w (e.F); a uniform F
      // has them per pair
      float c1k = a.c1[k], sok = a.so[k];
      if constexpr (DIFF) {
        const float eF = edot<Q>(i, Fx, Fy, Fz);
        c1k = 18.f * a.guo * w * eF;
        sok = (1.f - 0.5f * omm) * 6.f * w * eF;
      }
      P2 += c1k * eu - w * g3uF2;
      M2 += sok;
    }
    if constexpr (SP) {
      P2 += sp * (a.ae[k] - P2);
      M2 += sp * (a.bo[k] - M2);
    }
    const float hM = 0.5f * M2;
    pair(k, i, j, __builtin_fmaf(0.5f, P2, hM), __builtin_fmaf(0.5f, P2, -hM), ST::dither(hsh, (11 * (2 * k + 1)) % 17),
         ST::dither(hsh, (11 * (2 * k + 2)) % 17));
  }
}

}  // namespace lbm
