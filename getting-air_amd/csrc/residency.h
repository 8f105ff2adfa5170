// Whether lattices stay in the 256 MB of last-level cache from step to step:
// ordinary loads and stores, and neighbouring tiles on one XCD, in place of
// non-temporal access.  Host rules, in MB of population lattices.
#pragma once

namespace lbm {

// A dense solve's default one-step launches.  us a step, non-temporal and
// ordinary: D3Q19 fp32 200x100x19 (60 MB) 13.0 and 10.1, 200x100x78 (240 MB)
// 44.8 and 34.3, x88 (270 MB) 50.2 and 39.0, x98 (300 MB) 54.9 and 52.1, x115
// (350 MB) 63.9 and 65.4; f16 with walls 200x100x157 (240 MB) 50.6 and 43.4;
// D2Q9 400x5208 (150 MB) 28.4 and 22.3.  Rows of whole 256-cell tiles gain less
// (256x128x48, 240 MB: 41.8 and 34.7) and small ones nothing (10 MB: f16 5.56
// and 5.70; D3Q27 with walls, 60 MB: 12.5 and 13.4).
//
// Grids of about as many bytes as the XCDs' own caches hold are an exception
// where a few blocks are slow, those next to a body and, in rows of whole
// layout blocks, to walls.  Measured, not explained: ordinary loads with
// non-temporal stores are slower than both there (64^3 1.2 times), so neither
// alone is it.  Ordinary over non-temporal, two sizes of body: D3Q19 fp32 64^3 1.18, 1.08, 128x70x37 1.11, 1.02, 96^3 0.91, 0.91;
// D3Q27 56^3 1.02, 1.07, 64^3 1.40, 1.25, 96x64x64 1.11, 1.03, 80^3 0.95, 0.84;
// f16 D3Q19 64^3 0.99, 0.94, 128x64x64 1.18, 1.17, 80^3 1.12, 1.14, 100^3 0.97,
// 0.94; D3Q27 64^3 1.13, 1.12, 128x64x64 1.22, 1.18, 80^3 1.12, 1.09, 100^3
// 0.97, 0.95; D2Q9 768^2 1.07, f16 1024^2 1.2.  Walls: D3Q19 fp32 64^3 1.18,
// 72^3 0.86, f16 64^3 1.10.
inline bool cache_resident(double lattice_mb, double cells, int nx, int q, int elem, bool general, bool body) {
  const double least = nx % 256 ? 0.0 : (q == 27 && general ? 100.0 : 30.0);
  if (lattice_mb < least || lattice_mb > 270.0) return false;
  const bool rows = nx % 64 == 0;
  double lo = 0.0, hi = 0.0;  // the exception, million cells
  if (body && elem == 4) {
    if (q == 9) lo = 0.55, hi = 0.8;
    else if (q == 27 || rows) lo = q == 27 ? 0.15 : 0.22, hi = 0.42;
  } else if (body) {
    lo = q == 9 ? 0.9 : (q == 19 ? 0.44 : (rows ? 0.22 : 0.28));
    hi = q == 9 || rows ? 1.2 : 0.9;
  } else if (general && rows && q != 9) {
    lo = 0.22, hi = 0.3;
  }
  return 1e-6 * cells < lo || 1e-6 * cells >= hi;
}

// Such lattices under a refined solve, which passes through the active tiles'
// lattices between their steps: `mb` is everything a macro-step goes through,
// all lattices and macroscopic fields.  us a macro-step, L0 non-temporal and
// ordinary: D3Q27 96^3 with 0.01 and 0.04 of its blocks refined (240, 333 MB)
// 75.0 and 65.5, 100.0 and 109.4; 80^3, 0.06 and 0.1 (231, 305 MB) 79.6 and
// 73.2, 100.4 and 108; D2Q9 1024^2, 0.25 and 0.4 (235, 321 MB) 72.3 and 70.5,
// 102 and 117.  At 260 to 270 MB the two meet.
inline bool cache_resident_refined(double mb) { return mb <= 260.0; }

}  // namespace lbm
