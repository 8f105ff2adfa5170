// Dense-lattice kernels for gfx950 beside the step itself (dense_step.h,
// dense_pair.hip): equilibrium initialisation, the wire format, FP64 population
// totals, force records, classification and the copy probe; and the dispatch
// of the step's launches.
//
// initEq follows shaders/common_d3_step.wgsl:206-222.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>
#include "collide.h"
#include "dense.h"
#include "dense_cell.h"
#include "device_common.h"
#include "lattice_tables.h"

namespace lbm {

// First element of the block holding cell c (its population i is then at
// element i * kLatBlock + c % kLatBlock of the block).
template <int Q, class T>
__device__ __forceinline__ T* block_of(T* g, uint32_t c) {
  return g + (size_t)(c / kLatBlock) * (Q * kLatBlock);
}

__global__ void __launch_bounds__(512) k_force_finalize(ForceSum a) {
  if (a.periodic_arm) append_force_records<true, kMaxLaunchSteps>(a, blockIdx.x, gridDim.x);
  else append_force_records<false, kMaxLaunchSteps>(a, blockIdx.x, gridDim.x);
}

template <int Q, class ST>
__global__ void __launch_bounds__(256)
k_init_eq(const float* __restrict__ mac, typename ST::T* __restrict__ g, uint32_t N) {
  using L = Lattice<Q>;
  const uint32_t cell = blockIdx.x * blockDim.x + threadIdx.x;
  if (cell >= N) return;
  const float4 m = reinterpret_cast<const float4*>(mac)[cell];
  const float usq = m.y * m.y + m.z * m.z + m.w * m.w;
  const float drho = m.x - 1.f;
#pragma unroll
  for (int i = 0; i < Q; i++) {
    const float eu = (float)L::ex[i] * m.y + (float)L::ey[i] * m.z + (float)L::ez[i] * m.w;
    const float geq = L::w[i] * (drho + m.x * (3.f * eu + 4.5f * eu * eu - 1.5f * usq));
    ST::store(block_of<Q>(g, cell) + i * kLatBlock, cell % kLatBlock, geq);
  }
}

// Wire format (f32 plane-major f) <-> storage (shifted g), f-pack.mjs:93-124.
template <int Q, class ST>
__global__ void __launch_bounds__(256)
k_pack(const float* __restrict__ wire, typename ST::T* __restrict__ g, uint32_t N) {
  using L = Lattice<Q>;
  const uint32_t cell = blockIdx.x * blockDim.x + threadIdx.x;
  if (cell >= N) return;
#pragma unroll
  for (int i = 0; i < Q; i++)
    ST::store(block_of<Q>(g, cell) + i * kLatBlock, cell % kLatBlock, wire[(size_t)i * N + cell] - L::w[i]);
}

template <int Q, class ST>
__global__ void __launch_bounds__(256)
k_unpack(const typename ST::T* __restrict__ g, float* __restrict__ wire, uint32_t N) {
  using L = Lattice<Q>;
  const uint32_t cell = blockIdx.x * blockDim.x + threadIdx.x;
  if (cell >= N) return;
#pragma unroll
  for (int i = 0; i < Q; i++)
    wire[(size_t)i * N + cell] = ST::load(block_of<Q>(g, cell) + i * kLatBlock, cell % kLatBlock) + L::w[i];
}

template <int Q, class ST>
__global__ void __launch_bounds__(256)
k_totals(const typename ST::T* __restrict__ g, TotalsArgs a) {
  using L = Lattice<Q>;
  __shared__ double lds[16 * 4];
  double v[4] = {0, 0, 0, 0};
  for (uint32_t cell = blockIdx.x * blockDim.x + threadIdx.x; cell < a.ncells; cell += gridDim.x * blockDim.x) {
#pragma unroll
    for (int i = 0; i < Q; i++) {
      const double fi = (double)ST::load(block_of<Q>(g, cell) + i * kLatBlock, cell % kLatBlock) + (double)L::w[i];
      v[0] += fi;
      v[1] += L::ex[i] * fi;
      v[2] += L::ey[i] * fi;
      v[3] += L::ez[i] * fi;
    }
  }
  block_sum<4>(v, lds);
  partials_then_fixed_order_sum<4>(v, a.partials, a.counter, [&](int j, double s) { a.out[j] = s; });
}

// Per-cell class byte from the signed distance of the pinned body (body_phi),
// which the host oracle reproduces exactly.
__global__ void __launch_bounds__(256) k_classify(ClassifyArgs a) {
  const uint32_t n = (uint32_t)a.nx * a.ny * a.nz;
  const uint32_t cell = blockIdx.x * blockDim.x + threadIdx.x;
  if (cell >= n) return;
  const int x = cell % a.nx;
  const int y = (cell / a.nx) % a.ny;
  const int z = cell / (a.nx * a.ny);
  const float phi = body_phi(a.shape, a.radius, a.cx, a.cy, a.cz, a.nx, a.ny, x, y, z);
  uint8_t c = 0;
  if (phi < 0.f) c |= kClsSolid;
  if (phi < 2.f) c |= kClsNear;
  if (phi < a.band) c |= kClsBand;
  a.cls[cell] = c;
}

// Link masks for the bounce-back branch of the step: bit i of a cell next to
// the body is set when its pull source cell - e_i (periodic) is solid.
template <int Q>
__global__ void __launch_bounds__(256) k_links(ClassifyArgs a) {
  using L = Lattice<Q>;
  const int nx = a.nx, ny = a.ny, nz = a.nz;
  const uint32_t n = (uint32_t)nx * ny * nz;
  const uint32_t cell = blockIdx.x * blockDim.x + threadIdx.x;
  if (cell >= n) return;
  uint32_t m = 0;
  if (a.cls[cell] & 2) {
    const int x = cell % nx, y = (cell / nx) % ny, z = cell / (nx * ny);
#pragma unroll
    for (int i = 1; i < Q; i++) {
      const int sx = x - L::ex[i], sy = y - L::ey[i], sz = z - L::ez[i];
      const int wx = sx < 0 ? sx + nx : (sx >= nx ? sx - nx : sx);
      const int wy = sy < 0 ? sy + ny : (sy >= ny ? sy - ny : sy);
      const int wz = sz < 0 ? sz + nz : (sz >= nz ? sz - nz : sz);
      if (a.cls[(uint32_t)((wz * ny + wy) * nx + wx)] & 1) m |= 1u << i;
    }
  }
  a.links[cell] = m;
}

// 16-byte streaming copy, one element per thread with non-temporal loads and
// stores: the practical HBM ceiling the roofline fraction is read against.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__global__ void __launch_bounds__(256) k_copy_probe(const u32x4* __restrict__ src, u32x4* __restrict__ dst, size_t n) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i < n) __builtin_nontemporal_store(__builtin_nontemporal_load(src + i), dst + i);
}

// ---------------------------------------------------------------------------
// dispatch: one Op<Q, Storage>::run per kernel family
// ---------------------------------------------------------------------------
template <template <int, class> class Op, class... A>
static hipError_t dispatch(int q, int storage, A... args) {
  switch (q) {
    case 9:
      if (storage == kF32) return Op<9, StoreF32>::run(args...);
      if (storage == kF16) return Op<9, StoreF16>::run(args...);
      return Op<9, StoreBF16>::run(args...);
    case 19:
      if (storage == kF32) return Op<19, StoreF32>::run(args...);
      if (storage == kF16) return Op<19, StoreF16>::run(args...);
      return Op<19, StoreBF16>::run(args...);
    default:
      if (storage == kF32) return Op<27, StoreF32>::run(args...);
      if (storage == kF16) return Op<27, StoreF16>::run(args...);
      return Op<27, StoreBF16>::run(args...);
  }
}

static inline dim3 cells_grid(uint32_t n) { return dim3((n + 255) / 256); }

// LDS bytes per CU of the current device (160 KiB on gfx950).
static size_t lds_per_cu() {
  static const size_t bytes = [] {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) != hipSuccess || v <= 0)
      v = 160 * 1024;
    return (size_t)v;
  }();
  return bytes;
}

// Blocks per CU that give `occ` waves on each of the CU's 4 SIMDs, and the
// LDS share A = L / blocks that admits exactly that many: blocks * A <= L <
// (blocks + 1) * A.  A is a multiple of 1 KiB for the shapes used here, so
// the hardware's allocation granule does not round it up.
size_t occ_share(int occ, int threads) {
  const int wpb = threads / 64;
  if (occ <= 0 || wpb <= 0 || (4 * occ) % wpb) return 0;
  const size_t blocks = (size_t)(4 * occ / wpb), L = lds_per_cu();
  const size_t A = L / blocks / 1024 * 1024;
  if (A == 0 || (blocks + 1) * A <= L) return 0;
  return A;
}
bool occupancy_cap_ok(int occ, int threads) { return occ == 0 || occ_share(occ, threads) != 0; }

template <int Q, class ST> struct OpInit {
  static hipError_t run(const float* mac, void* f, uint32_t N, hipStream_t s) {
    hipLaunchKernelGGL((k_init_eq<Q, ST>), cells_grid(N), dim3(256), 0, s, mac, (typename ST::T*)f, N);
    return hipGetLastError();
  }
};
template <int Q, class ST> struct OpPack {
  static hipError_t run(const float* wire, void* f, uint32_t N, hipStream_t s) {
    hipLaunchKernelGGL((k_pack<Q, ST>), cells_grid(N), dim3(256), 0, s, wire, (typename ST::T*)f, N);
    return hipGetLastError();
  }
};
template <int Q, class ST> struct OpUnpack {
  static hipError_t run(const void* f, float* wire, uint32_t N, hipStream_t s) {
    hipLaunchKernelGGL((k_unpack<Q, ST>), cells_grid(N), dim3(256), 0, s, (const typename ST::T*)f, wire, N);
    return hipGetLastError();
  }
};
template <int Q, class ST> struct OpTotals {
  static hipError_t run(const void* f, TotalsArgs a, int nblocks, hipStream_t s) {
    hipLaunchKernelGGL((k_totals<Q, ST>), dim3(nblocks), dim3(256), 0, s, (const typename ST::T*)f, a);
    return hipGetLastError();
  }
};

template <class F>
static hipError_t of_lattice(int q, F f) {
  if (q == 9) return f(DenseStep<9>{});
  if (q == 19) return f(DenseStep<19>{});
  return f(DenseStep<27>{});
}
hipError_t launch_step(int q, int storage, bool general, bool nontemporal, int occ, const void* fin, void* fout,
                       const StepArgs& a, int bx, int by, hipStream_t s, bool diffuse) {
  return of_lattice(q, [&](auto d) {
    return d.step(storage, general, nontemporal, occ, fin, fout, a, bx, by, s, diffuse);
  });
}
hipError_t launch_step_batch(int q, int storage, bool general, bool nontemporal, int occ, bool rows, bool force,
                             const BatchArgs& b, uint32_t ntiles, int bx, int by, hipStream_t s) {
  return launch_step_persistent(q, storage, general, nontemporal, occ, rows, force, b, ntiles, bx, by, -1, nullptr, s);
}
hipError_t launch_step_persistent(int q, int storage, bool general, bool nontemporal, int occ, bool rows, bool force,
                                  const BatchArgs& b, uint32_t ntiles, int bx, int by, int steps, PersistBarrier* bar,
                                  hipStream_t s) {
  if (ntiles == 0 || steps == 0) return hipSuccess;
  return of_lattice(q, [&](auto d) {
    return d.batch(storage, general, nontemporal, occ, rows, force, b, ntiles, bx, by, steps, bar, s);
  });
}
hipError_t launch_init_eq(int q, int storage, const float* mac, void* f, uint32_t N, hipStream_t s) {
  return dispatch<OpInit>(q, storage, mac, f, N, s);
}
hipError_t launch_pack(int q, int storage, const float* wire, void* f, uint32_t N, hipStream_t s) {
  return dispatch<OpPack>(q, storage, wire, f, N, s);
}
hipError_t launch_unpack(int q, int storage, const void* f, float* wire, uint32_t N, hipStream_t s) {
  return dispatch<OpUnpack>(q, storage, f, wire, N, s);
}
hipError_t launch_totals(int q, int storage, const void* f, const TotalsArgs& a, int nblocks, hipStream_t s) {
  return dispatch<OpTotals>(q, storage, f, a, nblocks, s);
}
hipError_t launch_force_finalize(const ForceSum& a, hipStream_t s) {
  hipLaunchKernelGGL(k_force_finalize, dim3(force_blocks(a)), dim3(a.steps > 1 ? 512 : 256), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_classify(const ClassifyArgs& a, hipStream_t s) {
  const uint32_t n = (uint32_t)a.nx * a.ny * a.nz;
  hipLaunchKernelGGL(k_classify, dim3((n + 255) / 256), dim3(256), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_links(int q, const ClassifyArgs& a, hipStream_t s) {
  const uint32_t n = (uint32_t)a.nx * a.ny * a.nz;
  const dim3 grid((n + 255) / 256);
  if (q == 9) hipLaunchKernelGGL(k_links<9>, grid, dim3(256), 0, s, a);
  else if (q == 19) hipLaunchKernelGGL(k_links<19>, grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL(k_links<27>, grid, dim3(256), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_copy_probe(const void* src, void* dst, size_t bytes, hipStream_t s) {
  const size_t n = bytes / 16;
  hipLaunchKernelGGL(k_copy_probe, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (const u32x4*)src, (u32x4*)dst, n);
  return hipGetLastError();
}

}  // namespace lbm
