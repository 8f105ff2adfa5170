// Two dense 3D steps in one launch (gfx950).
//
// A one-step launch reads and writes every population once: 2 Q elements per
// cell and step, and it runs at HBM's rate.  Here a block takes a column of
// 64 x rows cells through z and computes two steps on the way, so a pair of
// steps reads and writes the lattice once.
//
// At plane k a block pulls the lattice at t and collides its column and a
// one-cell frame around it (step 1), then takes plane k - 1 through step 2.
// Step 2 at plane k - 1 pulls populations with e_z = -1 from plane k, 0 from
// k - 1 and +1 from k - 2, so each thread keeps its cell's e_z = 0
// populations for one plane and its e_z = +1 ones for two, and LDS holds one
// plane's worth of what its neighbours pull: 16 of 19 (24 of 27) populations,
// the other three being the cell's own.  Two LDS buffers take turns, which
// leaves one barrier per plane, and the loads of plane k + 1 are issued before
// step 2 of plane k - 1, so they are in flight while it computes.
//
// A wave owns one row of 64 cells (one layout block where nx is a multiple of
// 64, so every store fills whole cache lines).  rows + 2 waves hold the
// column's rows and the frame's two; one more wave holds the frame's two
// columns.  The frame is recomputed by every block that touches it, as are
// the first and last plane of a chunk along z: (rows + 3) / rows times
// (planes + 2) / planes step-1 cells per step-2 cell.
//
// The cell arithmetic is dense_cell.h's, so the result is the one-step
// kernel's bit for bit.  fp32 storage only: in the 16-bit formats the
// conversions and the dither of the intermediate state take what the halved
// traffic gives back (256x128x128 sphere, f16: 54.8 us a step one by one,
// 58.4 in pairs).
//
// Measured (MI355X, us per step, one by one -> in pairs): D3Q19 256x128x128
// periodic 106.0 -> 70.8, with the sphere and sponge 105.9 -> 76.0; 256^3 436
// -> 259; D3Q27 128^3 77.4 -> 58.9.  At 256x128x128 a pair reads 370 MB (with
// the sphere 406) and writes 322 MB, 1.16 (1.28) and 1.01 times the lattice; it
// is bound by the block's own latency (load, barrier, LDS, store of a plane: 4.4
// us a plane with 40 blocks on the chip, 6.2 with 240) rather than by HBM (three
// quarters of a copy's rate) or its VALU (under half busy).  Smaller columns (4 to 6 rows, two blocks per CU) measured slower,
// 83-93 us: their frames are read and computed too often.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <atomic>
#include <cmath>
#include <vector>
#include "dense.h"
#include "dense_cell.h"

namespace lbm {

namespace {

constexpr int kTileX = 64, kPitch = kTileX + 2;

// LDS slot of direction i (one that a neighbour's cell pulls), or -1.
template <int Q>
__host__ __device__ constexpr int lds_slot(int i) {
  using L = Lattice<Q>;
  if (L::ex[i] == 0 && L::ey[i] == 0) return -1;
  int n = 0;
  for (int k = 0; k < i; k++) n += (L::ex[k] != 0 || L::ey[k] != 0) ? 1 : 0;
  return n;
}
template <int Q>
constexpr int lds_slots() {
  return Q - 3;  // all but (0, 0, -1), (0, 0, 0), (0, 0, 1)
}
// Most rows of a block's column: 16 waves with the frame's, and two LDS buffers
// of lds_slots directions of rows + 2 rows within the CU's 160 KiB.
template <int Q>
__host__ __device__ constexpr int pair_rows() {
  return Q == 19 ? 13 : 9;
}
// Rank of direction i among those with its e_z.
template <int Q>
__host__ __device__ constexpr int rank_z(int i) {
  int n = 0;
  for (int k = 0; k < i; k++) n += Lattice<Q>::ez[k] == Lattice<Q>::ez[i] ? 1 : 0;
  return n;
}
template <int Q>
constexpr int count_z(int v) {
  int n = 0;
  for (int k = 0; k < Q; k++) n += Lattice<Q>::ez[k] == v ? 1 : 0;
  return n;
}

__device__ __forceinline__ int wrap_one(int v, int n) { return v < 0 ? v + n : (v >= n ? v - n : v); }

}  // namespace

template <int Q, bool GEN, bool FRC, bool ALIGNED>
__global__ void __launch_bounds__(64 * (pair_rows<Q>() + 3))
k_step_pair(const float* __restrict__ gin, float* __restrict__ gout, StepArgs a, PairArgs p) {
  using L = Lattice<Q>;
  constexpr int NP = Pairs<Q>::NP, N0 = count_z<Q>(0), N1 = count_z<Q>(1);
  extern __shared__ float lds[];

  uint32_t b = blockIdx.x;
  if constexpr (GEN) {
    // a block of its own for the previous launch's force records: in one that
    // also steps cells it would hold up all of that block's waves
    if (p.finalize_prev) {
      if (b == 0) {
        append_force_records<false, 2>(a.prev, 0, 1);
        return;
      }
      b--;
    }
  }
  // hardware hands block b to XCD b % 8: neighbouring columns to one XCD
  const uint32_t per = p.nblocks >> 3;
  if (b < per * 8u) b = (b & 7u) * per + (b >> 3);
  const int nx = a.nx, ny = a.ny, nz = a.nz;
  const PairBlock blk = p.blocks[b];
  const int x0 = blk.x0, y0 = blk.y0, z0 = blk.z0, D = blk.planes;
  const int W = min(kTileX, nx - x0), H = min(p.rows, ny - y0);

  // this thread's cell of every plane: row r of the frame, column lane of a
  // main wave, or one of the frame's two columns in the last wave
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const bool side = wave == p.rows + 2;
  bool live = true;  // computes step 1
  int r = wave, cx = lane;
  if (side) {
    const int right = lane >= H + 2 ? 1 : 0;
    live = lane < 2 * (H + 2);
    r = live ? lane - right * (H + 2) : 0;
    cx = right ? W : -1;
  } else {
    live = lane < W && wave < H + 2;
    if (lane >= W) cx = 0;
    if (wave >= H + 2) r = 0;
  }
  const bool own_row = !side && wave >= 1 && wave <= H;  // wave-uniform
  const bool owned = own_row && lane < W;
  const int x = wrap_one(x0 + cx, nx), y = wrap_one(y0 - 1 + r, ny);
  const int xm = x == 0 ? nx - 1 : x - 1, xp = x == nx - 1 ? 0 : x + 1;
  const int pos = r * kPitch + cx + 1;
  constexpr int plane = (pair_rows<Q>() + 2) * kPitch;  // LDS elements per direction

  // Addresses.  A plane's cells start s = (z nx ny) % 64 cells into a layout
  // block; the cell c cells from that block's first lies at element
  // c + (c / 64) (Q - 1) 64 of it.  Where planes are whole blocks (ALIGNED)
  // that offset is the same in every plane, so the nine pulled cells of a
  // plane cost nine registers for the whole march and a load no address
  // arithmetic; otherwise the nine in-plane indices are kept.
  const uint32_t nxy = (uint32_t)nx * (uint32_t)ny;
  auto element = [&](uint32_t c) { return (uint32_t)__umul24(c / kLatBlock, (Q - 1) * kLatBlock) + c; };
  uint32_t at9[3][3];  // [e_y + 1][e_x + 1]: the cell at (x - e_x, y - e_y)
#pragma unroll
  for (int ey = -1; ey <= 1; ey++)
#pragma unroll
    for (int ex = -1; ex <= 1; ex++) {
      const int sy = ey == 1 ? (y == 0 ? ny - 1 : y - 1) : (ey == -1 ? (y == ny - 1 ? 0 : y + 1) : y);
      const uint32_t c = (uint32_t)sy * (uint32_t)nx + (uint32_t)(ex == 1 ? xm : (ex == -1 ? xp : x));
      at9[ey + 1][ex + 1] = ALIGNED ? element(c) : c;
    }
  auto plane_base = [&](int z) { return (size_t)((uint32_t)z * nxy / kLatBlock) * (Q * kLatBlock); };
  auto plane_skew = [&](int z) { return ALIGNED ? 0u : (uint32_t)z * nxy % kLatBlock; };
  auto offset = [&](uint32_t skew, uint32_t at) { return ALIGNED ? at : element(skew + at); };
  float g[Q];
  const uint32_t cell0 = (uint32_t)y * nx + x;  // in-plane index
  const bool ylo = (a.wall_mask & 2) && y == 0, yhi = (a.wall_mask & 2) && y == ny - 1;
  const float dxy = fminf(sponge_distance(a.sponge_mask & 1, (float)x, nx), sponge_distance(a.sponge_mask & 2, (float)y, ny));
  // Directions whose source lies behind a wall: of this thread's x and y, and
  // of plane z.
  uint32_t wall_xy = 0;
  if constexpr (GEN) {
    if (a.wall_mask & 1) wall_xy |= (x == 0 ? dirs_with<Q>(0, 1) : 0u) | (x == nx - 1 ? dirs_with<Q>(0, -1) : 0u);
    if (a.wall_mask & 2) wall_xy |= (y == 0 ? dirs_with<Q>(1, 1) : 0u) | (y == ny - 1 ? dirs_with<Q>(1, -1) : 0u);
  }
  auto walls = [&](int z) {
    if (!GEN) return 0u;
    uint32_t m = wall_xy;
    if (a.wall_mask & 4) m |= (z == 0 ? dirs_with<Q>(2, 1) : 0u) | (z == nz - 1 ? dirs_with<Q>(2, -1) : 0u);
    return m;
  };
  // Pulls plane z of the lattice at t.  A direction whose source is solid or
  // behind a wall (mask `back`, general kernel) takes the address of the
  // cell's own opposite population instead: bounce-back without a load of its
  // own, which a whole block would wait for at the plane's barrier.
  auto pull = [&](int z, uint32_t back) {
    const int zz[3] = {z == nz - 1 ? 0 : z + 1, z, z == 0 ? nz - 1 : z - 1};  // [e_z + 1]
    if constexpr (!GEN) {
#pragma unroll
      for (int i = 0; i < Q; i++) {
        const int zi = zz[L::ez[i] + 1];
        g[i] = *at(gin + plane_base(zi) + i * kLatBlock, offset(plane_skew(zi), at9[L::ey[i] + 1][L::ex[i] + 1]));
      }
    } else {
      // one base and 32-bit element offsets (the lattice is below 4 GiB)
      uint32_t o[Q];
#pragma unroll
      for (int i = 0; i < Q; i++) {
        const int zi = zz[L::ez[i] + 1];
        o[i] = (uint32_t)plane_base(zi) + i * kLatBlock + offset(plane_skew(zi), at9[L::ey[i] + 1][L::ex[i] + 1]);
      }
      if (__any(back != 0)) {
        const uint32_t self = (uint32_t)plane_base(z) + offset(plane_skew(z), at9[1][1]);
#pragma unroll
        for (int i = 1; i < Q; i++)
          if ((back >> i) & 1u) o[i] = self + L::opp[i] * kLatBlock;
      }
#pragma unroll
      for (int i = 0; i < Q; i++) g[i] = *at(gin, o[i]);
    }
  };
  // A plane's pull needs its link masks, and those its class bytes.  Memory
  // operations complete in order, stores included, so each is loaded one plane
  // earlier still, ahead of that plane's pull: waiting for the pull then covers
  // it, and nothing waits for the stores of step 2.
  auto class_of = [&](int z) { return GEN && a.cls ? (uint32_t)a.cls[(uint32_t)z * nxy + cell0] : 0u; };
  auto links_of = [&](int z, uint32_t c) {
    return GEN && (c & 2) ? a.links[(uint32_t)z * nxy + cell0] : 0u;
  };
  auto next = [&](int z) { return z == nz - 1 ? 0 : z + 1; };

  float h0[N0] = {}, hp1[N1] = {}, hp2[N1] = {};  // e_z = 0 of plane k - 1; e_z = +1 of k - 1 and k - 2
  float hz1 = 0.f;                                // (0, 0, -1) of plane k - 1; its other e_z = -1 stay in LDS
  uint32_t solid1 = 0, lm1 = 0;               // plane k - 1's solid bit and links
  float sp1 = 0.f;                            // and sponge weight
  int z = wrap_one(z0 - 1, nz);
  int z1 = 0;  // plane k - 1
  uint32_t c = class_of(z), lm = links_of(z, c);                  // plane k
  uint32_t cn = class_of(next(z)), lmn = links_of(next(z), cn);   // plane k + 1
  uint32_t cnn = class_of(next(next(z)));                         // plane k + 2
  pull(z, lm | walls(z));
  for (int k = 0; k < D + 2; k++) {
    const uint32_t cell = (uint32_t)z * nxy + cell0;
    const int zn = next(z);
    // --- step 1 at plane k (z) ------------------------------------------
    float h[Q];
    float sp = 0.f;
    uint32_t lmnn = 0, cnnn = 0;
    {
      if constexpr (GEN) {
        const uint32_t wall = walls(z);
        if (__any((lm | wall) != 0)) {
          // reflected by the pull: the moving walls' terms, and the body's force
          double F[3] = {0, 0, 0};
          reflect_masked<Q>(a, ylo, yhi, c & 1, lm, wall, g, F, [&](int i) { return g[i]; });
          if (a.boundary && lm && !(c & 1) && owned && k >= 1 && k <= D) {
            double* slot = a.force_partials + (size_t)boundary_slot(a.boundary, cell) * 3;
#pragma unroll
            for (int m = 0; m < 3; m++) slot[m] = F[m];
          }
        }
        sp = sponge_weight(a, fminf(dxy, sponge_distance(a.sponge_mask & 4, (float)z, nz)));
      }
      float S[NP], Df[NP], drho, rho, ux, uy, uz, usq, uF;
      pair_sums<Q>(g, S, Df);
      const float g0 = g[0];
      // the next plane's loads, in flight through both steps' arithmetic; the
      // general kernel has no registers to spare for them here and issues them
      // after step 1
      if (!GEN && k < D + 1) pull(zn, 0);
      cell_moments<Q, FRC>(a, g0, S, Df, drho, rho, ux, uy, uz, usq, uF);
      relax_cell<Q, StoreF32, GEN, FRC, false>(
          a, g0, S, Df, drho, rho, ux, uy, uz, usq, uF, 0.f, 0.f, 0.f, sp, 0u,
          [&](float v, uint32_t) { h[0] = v; },
          [&](int, int i, int j, float gi, float gj, uint32_t, uint32_t) {
            h[i] = gi;
            h[j] = gj;
          });
      if constexpr (GEN) {
        if (a.solid_eq && (c & 1)) {
#pragma unroll
          for (int i = 0; i < Q; i++) h[i] = 0.f;  // feq(1, 0) - w
        }
      }
    }
    // --- what step 2 at plane k - 1 pulls, to LDS --------------------------
    float* const buf = lds + (k & 1) * (lds_slots<Q>() * plane);
    if (live) {
#pragma unroll
      for (int i = 0; i < Q; i++) {
        const int s = lds_slot<Q>(i);
        if (s < 0) continue;
        const float v = L::ez[i] == -1 ? h[i] : (L::ez[i] == 0 ? h0[rank_z<Q>(i)] : hp2[rank_z<Q>(i)]);
        buf[s * plane + pos] = v;
      }
    }
    if (GEN && k < D + 1) {
      lmnn = links_of(next(zn), cnn);
      cnnn = class_of(next(next(zn)));
      pull(zn, lmn | walls(zn));
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    // --- step 2 at plane k - 1 ----------------------------------------------
    if (k >= 2 && own_row) {
      const uint32_t cell1 = (uint32_t)z1 * nxy + cell0;
      float q[Q];
#pragma unroll
      for (int i = 0; i < Q; i++) {
        const int s = lds_slot<Q>(i);
        if (s >= 0) q[i] = (buf[s * plane + pos - L::ey[i] * kPitch - L::ex[i]]);
        else q[i] = (L::ez[i] == -1 ? h[i] : (L::ez[i] == 0 ? h0[rank_z<Q>(i)] : hp2[rank_z<Q>(i)]));
      }
      if constexpr (GEN) {
        const uint32_t wall = walls(z1);
        if (__any((lm1 | wall) != 0)) {
          // plane k - 1's e_z = -1 populations are still in the other buffer
          const float* const last = lds + ((k + 1) & 1) * (lds_slots<Q>() * plane);
          double F[3] = {0, 0, 0};
          reflect_masked<Q>(a, ylo, yhi, solid1, lm1, wall, q, F, [&](int i) {
            const int j = L::opp[i];
            if (L::ez[j] == 0) return (h0[rank_z<Q>(j)]);
            if (L::ez[j] == 1) return (hp1[rank_z<Q>(j)]);
            return lds_slot<Q>(j) < 0 ? (hz1) : (last[lds_slot<Q>(j) * plane + pos]);
          });
          if (a.boundary && lm1 && !solid1 && owned) {
            double* slot = p.force2 + (size_t)boundary_slot(a.boundary, cell1) * 3;
#pragma unroll
            for (int m = 0; m < 3; m++) slot[m] = F[m];
          }
        }
      }
      float S[NP], Df[NP], drho, rho, ux, uy, uz, usq, uF;
      pair_sums<Q>(q, S, Df);
      cell_moments<Q, FRC>(a, q[0], S, Df, drho, rho, ux, uy, uz, usq, uF);
      const bool solid = GEN && a.solid_eq && solid1;
      if (owned) {
        if (a.mac) {
          float4 m = make_float4(rho, ux, uy, uz);
          if (solid && a.solid_mac_rest) m = make_float4(1.f, 0.f, 0.f, 0.f);
          reinterpret_cast<float4*>(a.mac)[cell1] = m;
        }
        float* const out = gout + plane_base(z1);
        const uint32_t lo = offset(plane_skew(z1), at9[1][1]);
        if (solid) {
#pragma unroll
          for (int i = 0; i < Q; i++) st<StoreF32, true>(out + i * kLatBlock, lo, 0.f);
        } else {
          relax_cell<Q, StoreF32, GEN, FRC, false>(
              a, q[0], S, Df, drho, rho, ux, uy, uz, usq, uF, 0.f, 0.f, 0.f, sp1, 0u,
              [&](float v, uint32_t) { st<StoreF32, true>(out, lo, v); },
              [&](int, int i, int j, float gi, float gj, uint32_t, uint32_t) {
                st<StoreF32, true>(out + i * kLatBlock, lo, gi);
                st<StoreF32, true>(out + j * kLatBlock, lo, gj);
              });
        }
      }
    }
#pragma unroll
    for (int i = 0; i < Q; i++) {
      if (L::ez[i] == 0) h0[rank_z<Q>(i)] = h[i];
      if (L::ez[i] == 1) {
        hp2[rank_z<Q>(i)] = hp1[rank_z<Q>(i)];
        hp1[rank_z<Q>(i)] = h[i];
      }
      if (GEN && L::ez[i] == -1 && lds_slot<Q>(i) < 0) hz1 = h[i];
    }
    solid1 = c & 1;
    lm1 = lm;
    c = cn;
    lm = lmn;
    cn = cnn;
    lmn = lmnn;
    cnn = cnnn;
    sp1 = sp;
    z1 = z;
    z = zn;
  }
}

// ---------------------------------------------------------------------------
// shapes and dispatch
// ---------------------------------------------------------------------------
// Compute units of the current device (256 on MI355X).
static int device_cus() {
  static const int n = [] {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 1)
      v = 256;
    return v;
  }();
  return n;
}

template <int Q>
static constexpr size_t pair_lds() {
  return (size_t)2 * lds_slots<Q>() * (pair_rows<Q>() + 2) * kPitch * sizeof(float);
}

PairPlan pair_plan(int q, int storage, bool general, int nx, int ny, int nz, const std::vector<uint32_t>& boundary,
                   bool always) {
  PairPlan plan;
  const double cells = (double)nx * ny * nz, bytes = cells * 2 * q * 4;
  // the kernel's 32-bit in-plane byte offsets and, with walls or a body, its
  // 32-bit lattice ones
  if (q == 9 || storage != kF32 || (double)nx * ny * q * 4 >= 4.0e9 || (general && bytes / 2 >= 4.0e9)) return plan;
  // lanes past the end of a row idle: a narrow last column costs a whole one
  if (!always && nx < 0.7 * kTileX * ((nx + kTileX - 1) / kTileX)) return plan;
  const int most = q == 19 ? pair_rows<19>() : pair_rows<27>();
  const int nty = (ny + most - 1) / most, rows = (ny + nty - 1) / nty, ntx = (nx + kTileX - 1) / kTileX;
  const int cols = ntx * nty;
  // A column's work along z: 1 a plane, and more where it holds boundary
  // cells, whose reflection its block's other waves wait for.  Measured on the
  // 256x128x128 sphere with even chunks, such a plane took 1.25 times one
  // without (the step 87.8 us; 76.0 with this plan).
  const float extra = 0.25f;
  std::vector<float> work((size_t)cols * nz, 1.f);
  for (uint32_t c : boundary) {
    const int x = c % nx, y = (c / nx) % ny, z = c / (nx * ny);
    work[((size_t)(y / rows) * ntx + x / kTileX) * nz + z] = 1.f + extra;
  }
  std::vector<double> total(cols, 0.0);
  for (int k = 0; k < cols; k++)
    for (int z = 0; z < nz; z++) total[k] += work[(size_t)k * nz + z];
  // One block per CU at a time (its LDS and registers), one CU left for the
  // force records.  `r` rounds of blocks, each block at most `most_work` and
  // the two planes of its frame: the cheapest r.
  const int cus = device_cus() - (boundary.empty() ? 0 : 1);
  double best = 1e300;
  std::vector<int> chunks(cols), c2(cols);
  for (int r = 1; r <= 8; r++) {
    double lo = 1.0, hi = (double)nz * 2;
    auto fits = [&](double w) {
      long n = 0;
      for (int k = 0; k < cols; k++) n += c2[k] = std::max(1, std::min(nz, (int)std::ceil(total[k] / w)));
      return n <= (long)r * cus;
    };
    if (!fits(hi)) continue;
    for (int it = 0; it < 30; it++) {
      const double mid = 0.5 * (lo + hi);
      if (fits(mid)) hi = mid;
      else lo = mid;
    }
    fits(hi);
    double longest = 0;
    for (int k = 0; k < cols; k++) longest = std::max(longest, std::ceil(total[k] / c2[k]));
    if (r * (longest + 2.0) < best * 0.99) {
      best = r * (longest + 2.0);
      chunks = c2;
    }
  }
  if (best >= 1e300) {  // more columns than eight rounds: whole columns
    std::fill(chunks.begin(), chunks.end(), 1);
    best = (nz + 2.0) * cols / cus;
  }
  // Pairs where their estimate is the shorter one: a pair takes the longest
  // block's planes at a plane's latency and the traffic at the rate it reaches,
  // less where planes are not whole layout blocks (address arithmetic) or rows
  // are not (split lines); a one-step launch the traffic, at the rate of the
  // last-level cache as long as both lattices fit it.  Fitted to 51 grids from
  // 32^3 to 240^3 of either lattice, each periodic, with walls and with a body:
  // the form chosen is 0.3% off the faster one on average, 14% at most.  us a
  // step, one by one and in pairs: D3Q19 96^3 20.6 and 17.9, 100^3 23.0 and 27.6,
  // 64x32x32 3.6 and 4.5, 140^3 with a body 78.0 and 82.8, 160^3 107 and 83;
  // D3Q27 with walls 190x99x99 80 and 64, 150x75x50 22.7 and 26.0.
  const bool whole = (uint64_t)nx * ny % kLatBlock == 0, row = nx % (int)kLatBlock == 0, body = !boundary.empty();
  const double mb = 1e-6 * bytes;
  const double plane_us = (general ? (q == 19 ? 2.9 : 3.3) : 2.1) + (whole ? 0.0 : 0.8);
  const double mb_us = (row ? 0.15 : 0.165) - (general && q == 27 ? 0.03 : 0.0) + (body ? 0.02 : 0.0);
  const double pair_us = plane_us * best + mb_us * mb;
  const double step_us = std::max(3.8, mb <= 270.0 ? mb / 7.1 + (body ? 6.0 : (general ? 3.0 : 2.0))
                                                   : mb / (row ? 6.0 : 5.4) + 2.0);
  if (!always && pair_us > 2.0 * step_us) return plan;
  plan.rows = rows;
  // chunk by chunk over the columns, so that neighbouring columns march the
  // same planes at the same time on one XCD
  std::vector<std::vector<int>> cuts(cols);
  int deepest = 0;
  for (int k = 0; k < cols; k++) {
    double acc = 0;
    int n = 0;
    cuts[k].push_back(0);
    for (int z = 0; z < nz; z++) {
      acc += work[(size_t)k * nz + z];
      if (n + 1 < chunks[k] && acc >= total[k] * (n + 1) / chunks[k] - 1e-6) {
        cuts[k].push_back(z + 1);
        n++;
      }
    }
    if (cuts[k].back() != nz) cuts[k].push_back(nz);
    deepest = std::max(deepest, (int)cuts[k].size() - 1);
  }
  for (int n = 0; n < deepest; n++)
    for (int k = 0; k < cols; k++)
      if (n + 1 < (int)cuts[k].size())
        plan.blocks.push_back({(k % ntx) * kTileX, (k / ntx) * rows, cuts[k][n], cuts[k][n + 1] - cuts[k][n]});
  return plan;
}

template <int Q>
static hipError_t run_pair(bool general, const float* fin, float* fout, const StepArgs& a, const PairArgs& p,
                           hipStream_t s) {
  constexpr size_t lds = pair_lds<Q>();
  const bool frc = a.F[0] != 0.f || a.F[1] != 0.f || a.F[2] != 0.f;
  const bool aligned = (uint64_t)a.nx * a.ny % kLatBlock == 0;
  hipError_t err = hipSuccess;
  auto go = [&](auto G, auto F, auto A) {
    constexpr auto k = k_step_pair<Q, decltype(G)::value, decltype(F)::value, decltype(A)::value>;
    // gfx950 has 160 KiB of LDS per CU; a launch above 64 KiB asks for it, once
    // on each GPU
    static std::atomic<uint64_t> grown{0};
    int dev = 0;
    if ((err = hipGetDevice(&dev)) != hipSuccess) return;
    const uint64_t bit = 1ull << (dev & 63);
    if (!(grown.load() & bit)) {
      err = hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (err != hipSuccess) return;
      grown.fetch_or(bit);
    }
    hipLaunchKernelGGL(k, dim3(p.nblocks + (p.finalize_prev ? 1 : 0)), dim3(64 * (p.rows + 3)), lds, s, fin, fout, a, p);
    err = hipGetLastError();
  };
  auto with = [&](bool v, auto f) { v ? f(std::true_type{}) : f(std::false_type{}); };
  with(general, [&](auto G) { with(frc, [&](auto F) { with(aligned, [&](auto A) { go(G, F, A); }); }); });
  return err;
}

hipError_t launch_step_pair(int q, bool general, const void* fin, void* fout, const StepArgs& a, const PairArgs& p,
                            hipStream_t s) {
  const float* in = static_cast<const float*>(fin);
  float* out = static_cast<float*>(fout);
  return q == 19 ? run_pair<19>(general, in, out, a, p, s) : run_pair<27>(general, in, out, a, p, s);
}

}  // namespace lbm
