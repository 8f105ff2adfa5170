// The dense step kernels for gfx950: fused pull-stream + collide (D2Q9, D3Q19,
// D3Q27; BGK or TRT; Guo forcing; halfway bounce-back on walls and a pinned
// body; ALBC sponge; SOLID_EQ) with the FP64 momentum-exchange force fused
// in, and their launches: a template per lattice, instantiated by
// dense_step_q9.hip, dense_step_q19.hip and dense_step_q27.hip.
//
// Semantics follow the reference kernels
//   shaders/common_d3_step.wgsl:224-400 (step)
//   shaders/lbm_step.wgsl:137-270 (D2Q9 main)
//   plans/TRT.md:333-349 (TRT delta form)
//   shaders/common_d3_force.wgsl:171-216, shaders/lbm_force.wgsl:128-147 (MEM)
// The arithmetic is rewritten in shifted variables g_i = f_i - w_i:
//   rho - 1 = sum g_i (+ (sum w_i - 1), nonzero only for D2Q9's weights)
//   rho u   = sum g_i e_i + F/2          (sum w_i e_i = 0 exactly)
//   g_eq    = w_i ((rho - 1) + rho (3 e.u + 4.5 (e.u)^2 - 1.5 u.u))
// which is the same collision with the large constant w_i taken out before
// rounding.
//
// Layout: blocks of kLatBlock (64) consecutive cells, each holding its Q
// populations as Q runs of 64 elements (dense.h kLatBlock, lat_elem).
// One thread owns one cell; a wave covers 64 consecutive x, so every plane
// load and store of a wave is one contiguous 256 B (f32) or 128 B (16-bit)
// span, shifted by at most one element for the x-moving directions.  All Q
// loads are issued back to back (no branch between them); the rare cells next
// to a wall or the body then patch their reflected directions.
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>
#include "collide.h"
#include "dense.h"
#include "dense_cell.h"
#include "device_common.h"
#include "lattice_pairs.h"
#include "lattice_tables.h"
#include "rigid_device.h"

namespace lbm {

// Lattice offset of cell x of a row, relative to the row's first element
// (rows are whole layout blocks).
template <int Q>
__device__ __forceinline__ uint32_t row_off(int x) {
  // a 24-bit multiply is full rate (a 32-bit one a quarter); x < 2^24
  return (uint32_t)__umul24((uint32_t)x / kLatBlock, Q * kLatBlock) + (uint32_t)x % kLatBlock;
}

// One step of tile b of a solve: every thread of the block pulls, collides
// and stores its cell; a tile with a force slot leaves its FP64 force there.
// `salt` seeds the dither of 16-bit stores; `mac` (or null) receives the
// macroscopic field.  Shared by the single-solve and the batched kernels.
// ROW (step_row_mode): each wave lies in one row, so y, z and every source
// row's base address are wave-uniform and only the x part of an address is
// per lane; otherwise each lane locates its sources' blocks itself.
// RIGID (with GEN): a moving rigid body, a.rigid (its own instantiations, so
// that the kernels without one keep their register budget).
// BODY (with GEN): the solve has a body; a general solve without one (walls,
// sponge or an AMR level's covered cells) runs instantiations without class
// bytes, links and force records (D2Q9 channel 517x203, bf16: 5.1 -> 4.7 us a step).
// DIFF (with GEN): the pinned body's diffuse penalty coupling in place of
// bounce-back (common_d3_step.wgsl:288-300; the reference's default without
// ?bounceback): every cell takes the Guo force F + rho chi (0 - u*), u* = m /
// rho, chi = 1/2 (1 - tanh(clamp(phi / eps, -20, 20))), and a cell with chi >=
// 1e-6 adds rho chi u* to the body's force (common_d3_force.wgsl:242-268).
template <int Q, class ST, bool GEN, bool NT, bool ROW, bool RIGID = false, bool DIFF = false, bool FRC = true,
          bool BODY = GEN>
__device__ __forceinline__ void step_tile(const typename ST::T* __restrict__ gin, typename ST::T* __restrict__ gout,
                                          const StepArgs& a, uint32_t b, uint32_t salt, float* mac) {
  static_assert(!DIFF || FRC, "the diffuse coupling forces every cell");
  using L = Lattice<Q>;
  const int nx = a.nx, ny = a.ny, nz = a.nz;
  int x, y, z;
  bool active;
  if (a.linear) {
    const uint32_t c = b * (blockDim.x * blockDim.y) + threadIdx.y * blockDim.x + threadIdx.x;
    const uint32_t row = div_invariant(c, a.div_nx);
    x = (int)(c - row * nx);
    const uint32_t r = ROW ? __builtin_amdgcn_readfirstlane(row) : row;
    z = (int)div_invariant(r, a.div_ny);
    y = (int)(r - (uint32_t)z * ny);
    active = c < a.ncells;
  } else {
    const int tx = b % a.ntx;
    const int rest = b / a.ntx;
    const int ty = rest % a.nty;
    z = rest / a.nty;
    x = tx * blockDim.x + threadIdx.x;
    y = ty * blockDim.y + threadIdx.y;
    if constexpr (ROW) y = __builtin_amdgcn_readfirstlane(y);
    active = x < nx && y < ny;
  }
  if constexpr (GEN) {
    if (active && a.cover)
      active = a.cover[((z / a.cover_rb) * a.cover_nby + y / a.cover_rb) * a.cover_nbx + x / a.cover_rb] < 0;
  }
  double fv[6] = {0, 0, 0, 0, 0, 0};  // diffuse coupling: this cell's force/torque on the body

  if (active) {
    const uint32_t cell = (uint32_t)((z * ny + y) * nx + x);

    // This cell's populations: population i at self + i * kLatBlock, lane
    // offset self_lo.
    using T = typename ST::T;
    size_t self;
    uint32_t self_lo;
    if constexpr (ROW) {
      self = (size_t)(z * ny + y) * nx * Q;
      self_lo = row_off<Q>(x);
    } else {
      self = (size_t)(cell / kLatBlock) * (Q * kLatBlock);
      self_lo = cell % kLatBlock;
    }

    // 1. periodic pull-stream, all Q loads straight-line.  The source of
    // direction i is cell - e_i, wrapping only on the domain faces.
    float g[Q];
    if constexpr (ROW) {
      const int xm = x == 0 ? nx - 1 : x - 1, xp = x == nx - 1 ? 0 : x + 1;
      const uint32_t lo_m = row_off<Q>(xm), lo_p = row_off<Q>(xp);
      const int ym = y == 0 ? ny - 1 : y - 1, yp = y == ny - 1 ? 0 : y + 1;
      const int zm = z == 0 ? nz - 1 : z - 1, zp = z == nz - 1 ? 0 : z + 1;
#pragma unroll
      for (int i = 0; i < Q; i++) {
        const int ex = L::ex[i], ey = L::ey[i], ez = L::ez[i];
        const int sy = ey == 1 ? ym : (ey == -1 ? yp : y);
        const int sz = ez == 1 ? zm : (ez == -1 ? zp : z);
        const T* src = gin + (size_t)(sz * ny + sy) * nx * Q + i * kLatBlock;
        g[i] = ld<ST, NT>(src, ex == 1 ? lo_m : (ex == -1 ? lo_p : self_lo));
      }
    } else {
      const int nxy = nx * ny;
      const int ox_m = x == 0 ? nx - 1 : -1, ox_p = x == nx - 1 ? 1 - nx : 1;
      const int oy_m = y == 0 ? (ny - 1) * nx : -nx, oy_p = y == ny - 1 ? (1 - ny) * nx : nx;
      const int oz_m = z == 0 ? (nz - 1) * nxy : -nxy, oz_p = z == nz - 1 ? (1 - nz) * nxy : nxy;
#pragma unroll
      for (int i = 0; i < Q; i++) {
        const int ex = L::ex[i], ey = L::ey[i], ez = L::ez[i];
        const int o = (ex == 1 ? ox_m : (ex == -1 ? ox_p : 0)) + (ey == 1 ? oy_m : (ey == -1 ? oy_p : 0)) +
                      (ez == 1 ? oz_m : (ez == -1 ? oz_p : 0));
        const uint32_t sc = (uint32_t)((int)cell + o);
        const T* src = gin + (size_t)(sc / kLatBlock) * (Q * kLatBlock) + i * kLatBlock;
        g[i] = ld<ST, NT>(src, sc % kLatBlock);
      }
    }
    const T* in_self = gin + self;
    T* out_self = gout + self;

    uint8_t c = 0;
    if constexpr (GEN) {
      // under the diffuse coupling the body has no links and no solid cells
      if (BODY && !DIFF && a.cls) c = a.cls[cell];
      const bool onFace = on_wall_face(a, x, y, z);
      if ((BODY && (c & 2)) || onFace) {
        // 1b. halfway bounce-back.  Which sources are solid comes from the
        // cell's precomputed link mask (one load instead of a class byte per
        // neighbour, which would keep Q addresses live in this rare branch and
        // cost the whole kernel occupancy).
        double F[3] = {0, 0, 0};
        const uint32_t lm = BODY && (c & 2) ? a.links[cell] : 0u;
        // a moving body's velocity here and the wall density: this cell's
        // own pre-stream density (common_d3_step.wgsl:236-242)
        float wux = 0.f, wuy = 0.f, wuz = 0.f, rho_w = 1.f;
        if (RIGID && lm) {
          body_velocity_f(a.rigid, x, y, z, wux, wuy, wuz);
          if (a.rigid->rho_w_local) {
            rho_w = 0.f;
            for (int i = 0; i < Q; i++) rho_w += ST::load(in_self + i * kLatBlock, self_lo) + L::w[i];
          }
        }
        reflect_cell<Q>(
            a, x, y, z, c & 1, lm, onFace, g, F,
            [&](int j) { return ST::load(in_self + j * kLatBlock, self_lo); },
            [&](int i, float& gi) {
              // Ladd's moving-wall term 2 w rho_w (e . u_body) / cs2
              if constexpr (RIGID)
                gi += 2.f * L::w[i] * rho_w *
                      ((float)L::ex[i] * wux + (float)L::ey[i] * wuy + (float)L::ez[i] * wuz) * 3.f;
            });
        if (BODY && !RIGID && a.boundary && lm && !(c & 1)) {
          double* slot = a.force_partials + (size_t)boundary_slot(a.boundary, cell) * 3;
#pragma unroll
          for (int k = 0; k < 3; k++) slot[k] = F[k];
        }
      }
    }

    // 2. pair sums and differences; moments from them
    constexpr int NP = Pairs<Q>::NP;
    float S[NP], D[NP], drho, rho, ux, uy, uz, usq, uF;
    pair_sums<Q>(g, S, D);
    float Fx = 0.f, Fy = 0.f, Fz = 0.f;
    if constexpr (!DIFF) {
      // FRC false: no body force (F = 0), so every Guo term vanishes
      cell_moments<Q, FRC>(a, g[0], S, D, drho, rho, ux, uy, uz, usq, uF);
    } else {
      float mx, my, mz;
      cell_sums<Q>(a, g[0], S, D, drho, mx, my, mz);
      rho = 1.f + drho;
      const float rinv = recip_nr(fmaxf(rho, 1e-6f));
      const float phi = body_phi(a.body_shape, a.body_r, a.body_cf[0], a.body_cf[1], a.body_cf[2], nx, ny, x, y, z);
      const float chi = 0.5f * (1.f - tanhf(fminf(fmaxf(phi / a.chi_eps, -20.f), 20.f)));
      const float usx = mx * rinv, usy = my * rinv, usz = mz * rinv;
      const float rc = rho * chi;
      Fx = a.F[0] + rc * (0.f - usx);
      Fy = a.F[1] + rc * (0.f - usy);
      Fz = a.F[2] + rc * (0.f - usz);
      if (a.force_slot && chi >= 1e-6f) {
        // the body feels the penalty's negative, rho chi (u* - U_s)
        const double fx = (double)rc * usx, fy = (double)rc * usy, fz = (double)rc * usz;
        double rx = x - a.body_c[0], ry = y - a.body_c[1], rz = z - a.body_c[2];
        if (a.periodic_arm) {
          rx -= nx * rint(rx / nx);
          ry -= ny * rint(ry / ny);
          rz = 0.0;
        }
        fv[0] = fx; fv[1] = fy; fv[2] = fz;
        fv[3] = ry * fz - rz * fy;
        fv[4] = rz * fx - rx * fz;
        fv[5] = rx * fy - ry * fx;
      }
      // Guo: u = u* + F / (2 rho)
      ux = (mx + 0.5f * Fx) * rinv;
      uy = (my + 0.5f * Fy) * rinv;
      uz = (mz + 0.5f * Fz) * rinv;
      usq = ux * ux + uy * uy + uz * uz;
      uF = ux * Fx + uy * Fy + uz * Fz;
    }

    bool solid = false;
    if constexpr (BODY) solid = a.solid_eq && (c & 1);
    // a moving body's interior velocity (zero for a pinned body)
    float sux = 0.f, suy = 0.f, suz = 0.f;
    if constexpr (RIGID) {
      if (solid) body_velocity_f(a.rigid, x, y, z, sux, suy, suz);
    }

    if (mac) {
      float4 m = make_float4(rho, ux, uy, uz);
      if (solid && a.solid_mac_rest) m = make_float4(1.f, sux, suy, suz);
      reinterpret_cast<float4*>(mac)[cell] = m;
    }

    if (solid) {
      // SOLID_EQ: feq(1, u_body), g = feq - w; for a pinned body g = 0,
      // exact in every format
      const float uu = sux * sux + suy * suy + suz * suz;
#pragma unroll
      for (int i = 0; i < Q; i++) {
        const float eu = (float)L::ex[i] * sux + (float)L::ey[i] * suy + (float)L::ez[i] * suz;
        st<ST, NT>(out_self + i * kLatBlock, self_lo, L::w[i] * (3.f * eu + 4.5f * eu * eu - 1.5f * uu));
      }
    } else {
      float sp = 0.f;
      if constexpr (GEN) {
        // under a moving window, distances in window coordinates
        // (common_d3_step.wgsl:332-337)
        float px = (float)x, py = (float)y, pz = (float)z;
        if constexpr (RIGID) {
          if (a.sponge_w > 0.f) {
            const RigidBody* B = a.rigid;
            px = (float)win_coord(x, B->c[0], B->win_a[0], B->win_n[0]);
            py = (float)win_coord(y, B->c[1], B->win_a[1], B->win_n[1]);
            pz = (float)win_coord(z, B->c[2], B->win_a[2], B->win_n[2]);
          }
        }
        sp = sponge_weight(a, fminf(sponge_distance(a.sponge_mask & 1, px, nx),
                                    fminf(sponge_distance(a.sponge_mask & 2, py, ny),
                                          sponge_distance(a.sponge_mask & 4, pz, nz))));
      }
      // 3. collide pair by pair (relax_cell); random bits of this cell and
      // step for the 16-bit stores
      const uint32_t hsh = ST::kBytes == 2 ? cell_hash(cell, salt) : 0u;
      relax_cell<Q, ST, GEN, FRC, DIFF>(
          a, g[0], S, D, drho, rho, ux, uy, uz, usq, uF, Fx, Fy, Fz, sp, hsh,
          [&](float p, uint32_t r) { st_sr<ST, NT>(out_self, self_lo, p, r); },
          [&](int, int i, int j, float gi, float gj, uint32_t ri, uint32_t rj) {
            st_sr_pair<ST, NT>(out_self + i * kLatBlock, out_self + j * kLatBlock, self_lo, gi, gj, ri, rj);
          });
    }
  }

  if constexpr (DIFF) {
    // Tiles in the coupling's band reduce their cells' force in FP64 and park
    // it in the tile's slot; the next launch sums the slots in order.
    if (a.force_slot) {
      const int slot = a.force_slot[b];
      if (slot >= 0) {
        __shared__ double lds[16 * 6];
        block_sum<6>(fv, lds);
        if (threadIdx.x == 0 && threadIdx.y == 0) {
#pragma unroll
          for (int k = 0; k < 6; k++) a.force_partials[(size_t)slot * 6 + k] = fv[k];
        }
      }
    }
  }
}

template <int Q, class ST, bool GEN, bool NT, bool ROW, bool RIGID = false, bool DIFF = false, bool FRC = true,
          bool BODY = GEN>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(Q == 27 ? 6 : 8)))
k_step(const typename ST::T* __restrict__ gin, typename ST::T* __restrict__ gout, StepArgs a) {
  // a moving body's records are k_rigid_force's; the diffuse coupling's slots
  // are one chunk
  if constexpr (BODY && !RIGID) {
    if (a.finalize_prev && blockIdx.x < (DIFF ? 1u : force_blocks(a.prev)))
      append_force_records<Q == 9, 1, !DIFF>(a.prev, blockIdx.x, DIFF ? 1u : force_blocks(a.prev));
  }
  uint32_t b = blockIdx.x;
  if (a.swizzle) {
    // Hardware hands block b to XCD b % 8.  Re-number so each XCD walks one
    // contiguous eighth of the tiles: neighbouring rows then share an L2.
    const uint32_t per = a.nblocks >> 3;
    if (b < per * 8u) b = (b & 7u) * per + (b >> 3);
  }
  uint32_t salt = 0;
  if constexpr (ST::kBytes == 2) {
    salt = *a.salt_in;
    if (blockIdx.x == 0 && threadIdx.x == 0 && threadIdx.y == 0) *a.salt_out = salt + 1;
  }
  step_tile<Q, ST, GEN, NT, ROW, RIGID, DIFF, FRC, BODY>(gin, gout, a, b, salt, a.mac);
}

// Many solves in one launch (the serve loop's packed pool): block k steps
// tile tiles[k].tile of solve tiles[k].solve.  A solve steps while
// launch < remaining; its lattice parity is its base parity flipped by the
// launch index, so every launch of a captured chunk is one step of every
// active solve.
// Tile k of the batch table at launch `launch` of the chunk.
template <int Q, class ST, bool GEN, bool NT, bool ROW, bool FRC>
__device__ __forceinline__ void batch_tile(const BatchArgs& B, uint32_t k, int32_t launch) {
  // The tables are written before the launch and only read during it: read
  // them through the constant address space, so their fields are scalar loads
  // that may be repeated at will instead of values held in registers.
  using CSolve = const __attribute__((address_space(4))) BatchSolve;
  using CTile = const __attribute__((address_space(4))) BatchTile;
  CTile* tp = ((CTile*)B.tiles) + k;
  const uint32_t tile = tp->tile;
  CSolve* sp = ((CSolve*)B.solves) + tp->solve;
  CSolve& S = *sp;
  if (launch >= S.remaining) return;
  const int p = S.parity ^ (launch & 1);
  const StepArgs& a = *(const StepArgs*)(&sp->args[p]);
  if constexpr (GEN) {
    if (a.boundary && tile < force_blocks(a.prev) && (launch > 0 || S.pending))
      append_force_records<Q == 9, 1>(a.prev, tile, force_blocks(a.prev));
  }
  // the dither counter of the solve is its step count
  const uint32_t salt = S.step0 + launch;
  float* mac = launch + 1 == S.remaining ? S.mac : nullptr;
  step_tile<Q, ST, GEN, NT, ROW, false, false, FRC>(static_cast<const typename ST::T*>(S.f[p]),
                                                    static_cast<typename ST::T*>(S.f[p ^ 1]), a, tile, salt, mac);
}

template <int Q, class ST, bool GEN, bool NT, bool ROW, bool FRC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(Q == 27 ? 6 : 8))) k_step_batch(BatchArgs B) {
  batch_tile<Q, ST, GEN, NT, ROW, FRC>(B, blockIdx.x, B.launch);
}

// Grid barrier of the persistent chunk, with a bounded wait.  Arrivals count
// up monotonically in one word (the host zeroes it before the launch):
// barrier j is passed when it reaches (j + 1) * gridDim.x.  Each block's
// first thread, after the block's own barrier, arrives with an agent-scope
// release (its XCD's L2 writes the block's populations back, so other XCDs
// can read them) and polls the same word with relaxed loads; an agent-scope
// acquire after the wait drops this XCD's stale lines.  A wait that exceeds
// kBarrierSpins polls (seconds, far beyond any step) sets the word's top bit,
// which ends every block's wait and fails every later barrier: the launch
// always ends, and the host reports the failure.
constexpr uint32_t kBarrierSpins = 1u << 20;
constexpr uint32_t kBarrierFailed = 1u << 31;

__device__ __forceinline__ bool grid_barrier(PersistBarrier* bar, uint32_t target) {
  __shared__ uint32_t ok;
  __syncthreads();
  if (threadIdx.x == 0 && threadIdx.y == 0) {
    uint32_t v = __hip_atomic_fetch_add(&bar->arrived, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT) + 1u;
    for (uint32_t spins = 0; v < target; spins++) {
      if (spins >= kBarrierSpins) {
        __hip_atomic_fetch_or(&bar->arrived, kBarrierFailed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        v = kBarrierFailed;
        break;
      }
      __builtin_amdgcn_s_sleep(8);
      v = __hip_atomic_load(&bar->arrived, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    ok = (v & kBarrierFailed) ? 0u : 1u;
  }
  __syncthreads();
  return ok != 0u;
}

// The persistent form of a chunk: one cooperative launch whose blocks stay
// resident for all `steps` launches of the chunk.  Block b steps tiles b, b +
// gridDim.x, ... of the batch table, then the grid meets at grid_barrier
// before the next step (the step reads every neighbour's populations of the
// previous one).  Every block runs the same `steps` iterations, so each
// barrier is reached by all; the cooperative launch keeps them all resident.
template <int Q, class ST, bool GEN, bool NT, bool ROW, bool FRC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(Q == 27 ? 6 : 8)))
k_step_persistent(BatchArgs B, uint32_t ntiles, int32_t steps, PersistBarrier* bar) {
  for (int32_t j = 0; j < steps; j++) {
    for (uint32_t k = blockIdx.x; k < ntiles; k += gridDim.x) batch_tile<Q, ST, GEN, NT, ROW, FRC>(B, k, j);
    if (j + 1 < steps && !grid_barrier(bar, (uint32_t)(j + 1) * gridDim.x)) return;
  }
}

// Dynamic LDS for a launch of kernel K under the cap: its share minus the
// kernel's own static LDS (queried once per kernel).
template <auto K>
static size_t occ_dynamic_lds(int occ, int threads) {
  const size_t A = occ_share(occ, threads);
  if (!A) return 0;
  static const size_t static_bytes = [] {
    hipFuncAttributes fa{};
    return hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(K)) == hipSuccess ? fa.sharedSizeBytes
                                                                                     : (size_t)0;
  }();
  return A > static_bytes ? A - static_bytes : 0;
}

// Runtime flags -> template arguments of the step kernels.
template <class F>
static void with_flags(bool general, bool nt, bool rows, F f) {
  auto r = [&](auto G, auto N) {
    if (rows) f(G, N, std::true_type{});
    else f(G, N, std::false_type{});
  };
  auto n = [&](auto G) {
    if (nt) r(G, std::true_type{});
    else r(G, std::false_type{});
  };
  if (general) n(std::true_type{});
  else n(std::false_type{});
}

template <int Q, class ST> struct OpStep {
  static hipError_t run(bool general, bool nt, int occ, const void* fin, void* fout, StepArgs a, int bx, int by,
                        hipStream_t s, bool diffuse) {
    using T = typename ST::T;
    const bool rows = step_row_mode(a.nx, a.linear != 0, bx, by);
    if (diffuse) {
      // the pinned body's diffuse coupling runs its own general instantiation
      with_flags(true, nt, rows, [&](auto, auto N, auto R) {
        constexpr auto k = k_step<Q, ST, true, decltype(N)::value, decltype(R)::value, false, true>;
        hipLaunchKernelGGL(k, dim3(a.nblocks), dim3(bx, by), occ_dynamic_lds<k>(occ, bx * by), s, (const T*)fin,
                           (T*)fout, a);
      });
      return hipGetLastError();
    }
    if constexpr (Q != 9) {
      if (a.rigid) {
        // a moving body runs the general kernel's rigid instantiation
        with_flags(true, nt, rows, [&](auto, auto N, auto R) {
          constexpr auto k = k_step<Q, ST, true, decltype(N)::value, decltype(R)::value, true>;
          hipLaunchKernelGGL(k, dim3(a.nblocks), dim3(bx, by), occ_dynamic_lds<k>(occ, bx * by), s, (const T*)fin,
                             (T*)fout, a);
        });
        return hipGetLastError();
      }
    }
    // a solve without a body force runs the instantiation without Guo terms
    const bool frc = a.F[0] != 0.f || a.F[1] != 0.f || a.F[2] != 0.f;
    const bool body = a.cls != nullptr;
    with_flags(general, nt, rows, [&](auto G, auto N, auto R) {
      auto go = [&](auto F, auto B) {
        constexpr bool g = decltype(G)::value;
        constexpr auto k = k_step<Q, ST, g, decltype(N)::value, decltype(R)::value, false, false, decltype(F)::value,
                                  g && decltype(B)::value>;
        hipLaunchKernelGGL(k, dim3(a.nblocks), dim3(bx, by), occ_dynamic_lds<k>(occ, bx * by), s, (const T*)fin,
                           (T*)fout, a);
      };
      auto forced = [&](auto B) {
        if (frc) go(std::true_type{}, B);
        else go(std::false_type{}, B);
      };
      if (body) forced(std::true_type{});
      else forced(std::false_type{});
    });
    return hipGetLastError();
  }
};
template <int Q, class ST> struct OpStepBatch {
  static hipError_t run(bool general, bool nt, int occ, bool rows, bool force, BatchArgs b, uint32_t ntiles, int bx,
                        int by, int persistent_steps, PersistBarrier* bar, hipStream_t s) {
    hipError_t err = hipSuccess;
    with_flags(general, nt, rows, [&](auto G, auto N, auto R) {
      auto go = [&](auto F) {
        constexpr bool g = decltype(G)::value, n = decltype(N)::value, r = decltype(R)::value, f = decltype(F)::value;
        if (persistent_steps <= 0) {
          constexpr auto k = k_step_batch<Q, ST, g, n, r, f>;
          hipLaunchKernelGGL(k, dim3(ntiles), dim3(bx, by), occ_dynamic_lds<k>(occ, bx * by), s, b);
          err = hipGetLastError();
          return;
        }
        // at most 4 blocks per CU (and never more than the device holds at
        // once: the cooperative launch requires every block resident), at
        // most one per tile.  Each block's arrival at the grid barrier is an
        // agent-scope atomic on one word, so the barrier grows with the block
        // count: on a 192^3 f16 request the step took 0.432, 0.293, 0.287 and
        // 0.366 ms at 8, 4, 2 and 1 blocks per CU (0.110 ms as a graph of
        // batched launches).
        constexpr auto k = k_step_persistent<Q, ST, g, n, r, f>;
        const size_t lds = occ_dynamic_lds<k>(occ, bx * by);
        int per_cu = 0, dev = 0, cus = 0;
        if ((err = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(k), bx * by,
                                                                lds)) != hipSuccess ||
            (err = hipGetDevice(&dev)) != hipSuccess ||
            (err = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess)
          return;
        if (per_cu <= 0) {
          err = hipErrorInvalidConfiguration;
          return;
        }
        per_cu = std::min(per_cu, 4);
        const uint32_t grid = std::min<uint32_t>(ntiles, (uint32_t)per_cu * (uint32_t)cus);
        uint32_t nt_arg = ntiles;
        int32_t steps_arg = persistent_steps;
        if ((err = hipMemsetAsync(bar, 0, sizeof(PersistBarrier), s)) != hipSuccess) return;
        void* args[] = {&b, &nt_arg, &steps_arg, &bar};
        err = hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k), dim3(grid), dim3(bx, by), args, lds, s);
      };
      if (force) go(std::true_type{});
      else go(std::false_type{});
    });
    return err;
  }
};

template <int Q, class... A>
static hipError_t step_of_storage(int storage, A... args) {
  if (storage == kF32) return OpStep<Q, StoreF32>::run(args...);
  if (storage == kF16) return OpStep<Q, StoreF16>::run(args...);
  return OpStep<Q, StoreBF16>::run(args...);
}
template <int Q, class... A>
static hipError_t batch_of_storage(int storage, A... args) {
  if (storage == kF32) return OpStepBatch<Q, StoreF32>::run(args...);
  if (storage == kF16) return OpStepBatch<Q, StoreF16>::run(args...);
  return OpStepBatch<Q, StoreBF16>::run(args...);
}

template <int Q>
hipError_t DenseStep<Q>::step(int storage, bool general, bool nt, int occ, const void* fin, void* fout,
                              const StepArgs& a, int bx, int by, hipStream_t s, bool diffuse) {
  return step_of_storage<Q>(storage, general, nt, occ, fin, fout, a, bx, by, s, diffuse);
}
template <int Q>
hipError_t DenseStep<Q>::batch(int storage, bool general, bool nt, int occ, bool rows, bool force, const BatchArgs& b,
                               uint32_t ntiles, int bx, int by, int persistent_steps, PersistBarrier* bar,
                               hipStream_t s) {
  return batch_of_storage<Q>(storage, general, nt, occ, rows, force, b, ntiles, bx, by, persistent_steps, bar, s);
}

}  // namespace lbm
