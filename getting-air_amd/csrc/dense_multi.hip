// Several D2Q9 steps in one launch (gfx950).
//
// A one-step launch of a 2D grid is short: 460k cells take 9 us and 4k cells
// 2.7, most of it launching, filling and draining the chip, and each step goes
// through memory.  Here a block reads a tile of cells and a frame around it as
// wide as the launch has steps, and steps them in LDS: step s computes the tile
// grown by (steps - s) cells on each side, and the tile alone is stored.  Frames
// are recomputed by the tiles they overlap.
//
// Populations sit in LDS in the storage format, one plane per direction.  A
// thread keeps up to C cells for the whole launch, so that a cell's position,
// links, walls and sponge weight are worked out once; cells are dealt out tile
// first and ring by ring, which leaves whole waves idle as the frame shrinks.
// Per step a thread pulls and collides its cells into registers, the block
// meets, writes them back in place, and meets again.  A block none of whose
// cells has a wall, a link or a sponge weight takes the plain step.
//
// The cell arithmetic is dense_cell.h's and each step's dither its own, so the
// result is the one-step kernel's bit for bit.
//
// Vector arithmetic bounds it: about 150 instructions a cell and step, 1.3 times
// for a 32 x 16 tile's frames of four steps.  Dealing the cells out anew each
// step (no ring order, positions per step) took 7.9 us a step where this takes
// 6.2, with body and sponge at 724^2; storing from inside the step loop kept
// every store address in registers across it and spilled, 11.3 us.
#include <hip/hip_runtime.h>
#include "dense.h"
#include "dense_cell.h"

namespace lbm {

namespace {

// Tile TX x TY, at most T steps, N threads, B blocks a CU (three with a body,
// whose code spills in the 64 registers four leave it).
template <int TX_, int TY_, int T_, int N_, int B_>
struct Shape {
  static constexpr int TX = TX_, TY = TY_, T = T_, N = N_, B = B_;
  // LDS rows hold the tile and its frame, on a pitch that spreads both a row
  // and a column of cells over the banks.
  static constexpr int FX = TX + 2 * T, FY = TY + 2 * T;
  static constexpr int PX = TX == 16 ? (FX + 31 - 17) / 32 * 32 + 17 : FX | 1, CELLS = PX * FY;
  static constexpr int C = (FX * FY + N - 1) / N;
};

__device__ __forceinline__ int wrap_one(int v, int n) { return v < 0 ? v + n : (v >= n ? v - n : v); }

// Position of cell j of a W x H tile and its frame, from the tile's origin:
// the tile row by row, then ring after ring of the frame, so that the cells of
// a step with frame h are the first (W + 2 h)(H + 2 h).
__device__ __forceinline__ void position(int j, int W, int H, int steps, int& x, int& y) {
  // j < 4096: floor(j / W) = (j ceil(2^20 / W)) >> 20
  const int row = (int)(((uint32_t)j * (((1u << 20) + (uint32_t)W - 1u) / (uint32_t)W)) >> 20);
  x = j - row * W;
  y = row;
  int k = j - W * H;
  if (k < 0) return;
  x = y = 0;  // past the frame
  for (int r = 1; r <= steps; r++) {
    const int w = W + 2 * r, v = H + 2 * r - 2, ring = 2 * (w + v);
    if (k < ring) {
      if (k < 2 * w) {
        x = (k < w ? k : k - w) - r;
        y = k < w ? -r : H - 1 + r;
      } else {
        k -= 2 * w;
        x = k < v ? -r : W - 1 + r;
        y = (k < v ? k : k - v) + 1 - r;
      }
      return;
    }
    k -= ring;
  }
}

}  // namespace

template <class ST, class S, bool GEN, bool BODY, bool FRC>
__global__ void __launch_bounds__(S::N, (BODY && S::B > 3 ? 3 : S::B) * S::N / 256)
k_step_multi(const typename ST::T* __restrict__ gin, typename ST::T* __restrict__ gout, StepArgs a, MultiArgs p) {
  constexpr int Q = 9, NP = Pairs<Q>::NP, C = S::C;
  using L = Lattice<Q>;
  using T = typename ST::T;
  __shared__ T pop[Q * S::CELLS];
  __shared__ uint32_t vote[GEN ? S::N / 64 : 1];

  uint32_t b = blockIdx.x;
  if constexpr (BODY) {
    // a block of its own for the previous launch's force records
    if (p.finalize_prev) {
      if (b == 0) {
        append_force_records<true, kMaxLaunchSteps>(a.prev, 0, 1);
        return;
      }
      b--;
    }
  }
  uint32_t salt = 0;
  if constexpr (ST::kBytes == 2) {
    salt = *a.salt_in;
    if (b == 0 && threadIdx.x == 0) *a.salt_out = salt + p.steps;
  }
  // hardware hands block b to XCD b % 8: neighbouring tiles to one XCD
  const uint32_t per = p.nblocks >> 3;
  if (b < per * 8u) b = (b & 7u) * per + (b >> 3);
  const int nx = a.nx, ny = a.ny, steps = p.steps;
  const int x0 = (int)(b % p.ntx) * S::TX, y0 = (int)(b / p.ntx) * S::TY;
  const int W = min(S::TX, nx - x0), H = min(S::TY, ny - y0);
  auto element = [](uint32_t c) { return (size_t)(c / kLatBlock) * (Q * kLatBlock) + c % kLatBlock; };
  auto area = [&](int h) { return (W + 2 * h) * (H + 2 * h); };

  // 1. the tile and its frame into LDS
  uint32_t pos[C], cell[C];
  uint32_t near[C];  // bits 1-8 links, 9 in the body, 10 and 11 on the walls y = 0 and ny - 1, 17-24 wall crossings
  float sp[C];
  {
    T v[C][Q];
#pragma unroll
    for (int c = 0; c < C; c++) {
      const int j = threadIdx.x + c * S::N;
      int x, y;
      position(j, W, H, steps, x, y);
      pos[c] = (uint32_t)((y + S::T) * S::PX + x + S::T);
      x = wrap_one(x0 + x, nx);
      y = wrap_one(y0 + y, ny);
      cell[c] = (uint32_t)(y * nx + x);
      const T* const src = gin + element(cell[c]);
#pragma unroll
      for (int i = 0; i < Q; i++) v[c][i] = src[i * kLatBlock];
      if constexpr (GEN) {
        uint32_t n = 0;
        if constexpr (BODY) {
          const uint32_t k = a.cls[cell[c]];
          n = ((k & 2) ? a.links[cell[c]] & 0x1feu : 0u) | (k & 1) << 9;
        }
        if (a.wall_mask & 1) n |= ((x == 0 ? dirs_with<Q>(0, 1) : 0u) | (x == nx - 1 ? dirs_with<Q>(0, -1) : 0u)) << 16;
        if (a.wall_mask & 2)
          n |= (y == 0 ? dirs_with<Q>(1, 1) << 16 | 0x400u : 0u) | (y == ny - 1 ? dirs_with<Q>(1, -1) << 16 | 0x800u : 0u);
        near[c] = n;
        sp[c] = sponge_weight(a, fminf(sponge_distance(a.sponge_mask & 1, (float)x, nx),
                                       sponge_distance(a.sponge_mask & 2, (float)y, ny)));
      }
    }
    const int all = area(steps);
    if constexpr (GEN) {
      bool special = false;
#pragma unroll
      for (int c = 0; c < C; c++) special |= (near[c] & 0x1fe03feu) || sp[c] > 0.f;
      const bool any = __any(special);
      if ((threadIdx.x & 63) == 0) vote[threadIdx.x >> 6] = any;
    }
#pragma unroll
    for (int c = 0; c < C; c++) {
      if (threadIdx.x + c * S::N >= all) continue;
#pragma unroll
      for (int i = 0; i < Q; i++) pop[i * S::CELLS + pos[c]] = v[c][i];
    }
  }
  __syncthreads();

  // s = 1 .. steps, then the store; General: some cell is not a plain one
  auto run = [&](auto General) {
    constexpr bool G = decltype(General)::value;
    T out[C][Q];
    for (int s = 1;; s++) {
      const int active = area(steps - s);
#pragma unroll
      for (int c = 0; c < C; c++) {
        if (threadIdx.x + c * S::N >= active) continue;
        // 2. pull, and next to a wall or the body bounce back
        float g[Q];
#pragma unroll
        for (int i = 0; i < Q; i++) g[i] = ST::load(pop, pos[c] + i * S::CELLS - (L::ey[i] * S::PX + L::ex[i]));
        bool solid = false;
        if constexpr (G) {
          if (near[c] & 0x1fe01feu) {
            const uint32_t lm = near[c] & 0x1feu, wall = near[c] >> 16;
            const bool in_body = near[c] & 0x200u;
            double F[3] = {0, 0, 0};
            reflect_masked<Q>(a, near[c] & 0x400u, near[c] & 0x800u, in_body, lm, wall, g, F,
                              [&](int i) { return ST::load(pop, pos[c] + L::opp[i] * S::CELLS); });
            if (BODY && a.boundary && lm && !in_body && threadIdx.x + c * S::N < area(0)) {
              double* slot = a.force_partials + (size_t)(s - 1) * p.force_stride +
                             (size_t)boundary_slot(a.boundary, cell[c]) * 3;
#pragma unroll
              for (int k = 0; k < 3; k++) slot[k] = F[k];
            }
          }
          solid = BODY && a.solid_eq && (near[c] & 0x200u);
        }
        // 3. collide
        float Sm[NP], Df[NP], drho, rho, ux, uy, uz, usq, uF;
        pair_sums<Q>(g, Sm, Df);
        cell_moments<Q, FRC>(a, g[0], Sm, Df, drho, rho, ux, uy, uz, usq, uF);
        if (a.mac && s == steps) {
          float4 m = make_float4(rho, ux, uy, uz);
          if (solid && a.solid_mac_rest) m = make_float4(1.f, 0.f, 0.f, 0.f);
          *at(reinterpret_cast<float4*>(a.mac), cell[c]) = m;
        }
        const uint32_t hsh = ST::kBytes == 2 ? cell_hash(cell[c], salt + (uint32_t)(s - 1)) : 0u;
        relax_cell<Q, ST, G, FRC, false>(
            a, g[0], Sm, Df, drho, rho, ux, uy, uz, usq, uF, 0.f, 0.f, 0.f, G ? sp[c] : 0.f, hsh,
            [&](float v, uint32_t r) { out[c][0] = ST::round_sr(v, r); },
            [&](int, int i, int k, float gi, float gk, uint32_t ri, uint32_t rk) {
              round_sr_pair<ST>(gi, gk, ri, rk, out[c][i], out[c][k]);
            });
        if (solid) {
#pragma unroll
          for (int i = 0; i < Q; i++) out[c][i] = T(0);  // feq(1, 0) - w
        }
      }
      // 4. keep: in LDS for the next step, in the lattice after the last
      if (s == steps) break;
      __syncthreads();  // every pull of this step is done
#pragma unroll
      for (int c = 0; c < C; c++) {
        if (threadIdx.x + c * S::N >= active) continue;
#pragma unroll
        for (int i = 0; i < Q; i++) pop[i * S::CELLS + pos[c]] = out[c][i];
      }
      __syncthreads();
    }
#pragma unroll
    for (int c = 0; c < C; c++) {
      if (threadIdx.x + c * S::N >= area(0)) continue;
      T* const dst = gout + element(cell[c]);
#pragma unroll
      for (int i = 0; i < Q; i++) dst[i * kLatBlock] = out[c][i];
    }
  };
  if constexpr (GEN) {
    uint32_t any = 0;
#pragma unroll
    for (int w = 0; w < S::N / 64; w++) any |= vote[w];
    if (__builtin_amdgcn_readfirstlane(any)) {
      run(std::true_type{});
      return;
    }
  }
  run(std::false_type{});
}

// ---------------------------------------------------------------------------
// shapes and dispatch
// ---------------------------------------------------------------------------
// A block's time is its busiest SIMD's arithmetic, so small grids take small
// tiles, frames and all, as long as the chip has room for more blocks; the
// frames of eight steps then cost less than the launches they save.  Grids
// beyond that take the tile with the least frame.
using Small = Shape<8, 8, 8, 576, 3>;
using Deep = Shape<16, 16, 8, 1024, 2>;
using Wide = Shape<32, 16, 4, 512, 4>;

// us a step, D2Q9 fp32 (16-bit storage within 8%), one-step launches, Small,
// Deep, Wide; plain periodic and, after the bar, with body and sponge:
//     64^2   2.73  0.96  1.31  1.65 | 5.20  1.35  1.82  3.00
//    160^2   3.08  1.34  1.41  1.89 | 5.07  1.72  1.96  3.14
//    192^2   3.13  1.84  1.38  1.89 | 5.20  2.18  1.95  3.22
//    352^2   4.37  4.56  2.05  2.02 | 5.94  5.13  2.66  3.46
//    384^2   4.63  5.38  2.58  2.42 | 6.13  5.94  3.03  3.83
//    724^2   8.83   -    6.38  4.86 | 9.79   -    6.63  5.6
//   4096^2 199      -     -   108   | 213    -     -   121
// Small to 400 tiles, Deep to 512, then Wide.  A grid too narrow for Wide, or
// one that leaves its tiles less than 0.7 full (36 x 20000: 10.1 us with body
// against the one-step launch's 8.5 in f16, half its blocks a sliver), takes
// Deep, then Small, while those stay ahead of the one-step launch (35 x 4001:
// 3.2 against 5.6; 16 x 4000, beyond Small's 900 tiles, 3.2).
MultiPlan multi_plan(int q, int nx, int ny) {
  // 32-bit byte offsets into the macroscopic field
  if (q != 9 || (double)nx * ny >= (double)(1u << 28)) return MultiPlan{};
  // tiles of shape S, 0 where a frame would wrap around the grid twice
  auto tiles = [&](auto shape) {
    using S = decltype(shape);
    if (nx < S::TX + S::T || ny < S::TY + S::T) return 0.0;
    return (double)((nx + S::TX - 1) / S::TX) * ((ny + S::TY - 1) / S::TY);
  };
  const double small = tiles(Small{}), deep = tiles(Deep{});
  double wide = tiles(Wide{});
  if ((double)nx * ny < 0.7 * wide * (Wide::TX * Wide::TY)) wide = 0;
  if (small > 0 && small <= 400) return {kMultiSmall, Small::T};
  if (deep > 0 && (deep <= 512 || (wide == 0 && deep <= 1600))) return {kMultiDeep, Deep::T};
  if (wide > 0) return {kMultiWide, Wide::T};
  return small > 0 && small <= 900 ? MultiPlan{kMultiSmall, Small::T} : MultiPlan{};
}

template <class ST, class S>
static hipError_t run_multi(bool general, const void* fin, void* fout, const StepArgs& a, MultiArgs p, hipStream_t s) {
  using T = typename ST::T;
  p.ntx = (a.nx + S::TX - 1) / S::TX;
  p.nblocks = (uint32_t)p.ntx * ((a.ny + S::TY - 1) / S::TY);
  p.finalize_prev = a.finalize_prev;
  const bool frc = a.F[0] != 0.f || a.F[1] != 0.f || a.F[2] != 0.f, body = a.cls != nullptr;
  auto go = [&](auto G, auto B, auto F) {
    constexpr auto k = k_step_multi<ST, S, decltype(G)::value, decltype(B)::value, decltype(F)::value>;
    hipLaunchKernelGGL(k, dim3(p.nblocks + (p.finalize_prev ? 1 : 0)), dim3(S::N), 0, s, (const T*)fin, (T*)fout, a, p);
  };
  auto of = [&](auto G, auto B) { frc ? go(G, B, std::true_type{}) : go(G, B, std::false_type{}); };
  if (body) of(std::true_type{}, std::true_type{});
  else if (general) of(std::true_type{}, std::false_type{});
  else of(std::false_type{}, std::false_type{});
  return hipGetLastError();
}

template <class ST>
static hipError_t of_shape(int shape, bool general, const void* fin, void* fout, const StepArgs& a, const MultiArgs& p,
                           hipStream_t s) {
  switch (shape) {
    case kMultiSmall: return run_multi<ST, Small>(general, fin, fout, a, p, s);
    case kMultiDeep: return run_multi<ST, Deep>(general, fin, fout, a, p, s);
    default: return run_multi<ST, Wide>(general, fin, fout, a, p, s);
  }
}

hipError_t launch_step_multi(int storage, int shape, bool general, const void* fin, void* fout, const StepArgs& a,
                             const MultiArgs& p, hipStream_t s) {
  if (storage == kF32) return of_shape<StoreF32>(shape, general, fin, fout, a, p, s);
  if (storage == kF16) return of_shape<StoreF16>(shape, general, fin, fout, a, p, s);
  return of_shape<StoreBF16>(shape, general, fin, fout, a, p, s);
}

}  // namespace lbm
