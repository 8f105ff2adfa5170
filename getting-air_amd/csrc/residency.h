// Whether lattices stay in the 256 MB of last-level cache from step to step:
// ordinary loads and stores, and neighbouring tiles on one XCD, in place of
// non-temporal access.  Host rules, in MB of population lattices.
#pragma once

namespace lbm {

// A dense solve's default launches (both lattices).  us a step, non-temporal
// and ordinary, one step a launch: D3Q19 fp32 200x100x19 (60 MB) 13.0 and 10.1,
// 200x100x78 (240 MB) 44.8 and 34.3, x88 (270 MB) 50.2 and 39.0, x98 (300 MB)
// 54.9 and 52.1, x115 (350 MB) 63.9 and 65.4; f16 with walls 200x100x157 (240 MB)
// 50.6 and 43.4; D2Q9 400x5208 (150 MB) 28.4 and 22.3.  Rows of whole 256-cell
// tiles gain less (256x128x48, 240 MB: 41.8 and 34.7) and small ones nothing
// (10 MB: f16 5.56 and 5.70; D3Q27 with walls, 60 MB: 12.5 and 13.4).
inline bool cache_resident(double lattice_mb, int nx, int q, bool general) {
  const double least = nx % 256 ? 0.0 : (q == 27 && general ? 100.0 : 30.0);
  return lattice_mb >= least && lattice_mb <= 270.0;
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
