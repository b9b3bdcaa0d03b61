// Rules on sizes that choose a launch, free of HIP so that a host compiler
// builds them alone (tests/test_dispatch_rules.py).
#pragma once

#include <algorithm>
#include <cstdint>

namespace csahca {

// Slots per wavefront of the split-KV attention: the caller's tile, or a
// multiple of it where more slots per wavefront are better.  A tile is a hint
// for the split, and the partials of several of the caller's tiles are one
// partial of their union, so the workspace the caller sized for its own tile
// holds them.  `vec`: the vectorised kernel runs (esz: bytes per element).
//
// The smallest multiple that, for the vectorised kernel,
//   * fills one batch of row loads (16 slots at 16-bit head_dim 128, 32 at 64;
//     a smaller tile re-reads its last row);
//   * leaves a head at most 64 tiles, the one-round-trip merge, as long as that
//     makes tiles of at most 128 slots;
//   * leaves the call at most 8192 wavefronts (32 per CU): more only write and
//     merge more partials.
// Measured (graph period, us, tile 8 as called / split chosen): B1 H8 D128
// top-8 5.31 / 5.06, top-32 49.3 / 7.3; B8 top-16 16.4 / 10.3, top-32 60.6 /
// 15.3; B32 top-32 104.7 / 56.7; B4 H12 D64 f16 480 slots 7.3 / 6.4; f32 D256
// 512 slots 9.4 (kept at 8).
//
// Generic kernel: its wavefronts take 4 slots per round trip, 0.23 us a slot at
// D 40 to 0.39 at D 320 f32, so long tiles are a long serial chain, and the
// merge of more than 64 partials is the cheaper side until the rows themselves
// take that long to stream: the same line, with 12800 wavefronts for rows below
// 1 KiB, but no multiple above 16 slots, 32 from 100 MiB of rows, any from 200
// MiB of rows of at least 384 bytes.  Measured, us, with tiles of 8 / 16 / 32 /
// 64 (and by the vectorised kernel's line): D40 bf16 B1 H8 3200 slots 12.7 /
// 11.6 / 13.1 / 19.4 (16.7); D96 bf16 B1 1600 slots 9.6 / 10.1 / 13.2 / 21.2
// (12.1), B4 6400 35.7 / 32.3 / 32.8 / 38.9 (41.4), B32 1600 53.4 / 50.1 / 49.3
// / 55.2 (52.4), 3200 102.7 / 92.7 / 90.1 / 92.5 (94.7); D192 B32 800 37.0 /
// 34.6 / 36.6 / 45.0 (38.8), 3200 150 / 140 / 137 / 137 (134.5); D320 f32 B4
// 6400 115 / 108 / 106 / 105 (95.9).
inline int64_t csa_split_tile(int64_t tile, int64_t total, int64_t bh, int64_t D, int64_t esz, bool vec) {
  constexpr int64_t kLanes = 64, kOneTripTiles = 64;
  const auto ceil_of = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const int64_t batch = vec ? 4 * (kLanes / (D * esz / 16)) : 4;
  const int64_t waves = vec || D * esz >= 1024 ? 8192 : 12800;
  int64_t want = std::max({batch, std::min<int64_t>(ceil_of(total, kOneTripTiles), 128), ceil_of(total * bh, waves)});
  int64_t most = INT64_MAX;
  if (!vec) {
    const double mib = 2.0 * static_cast<double>(total) * static_cast<double>(bh * D * esz) / (1 << 20);
    if (mib < 200.0 || D * esz < 384) most = mib < 100.0 ? 16 : 32;
    want = std::min(want, most);
  }
  int64_t t = tile;
  if (tile < want) t = std::min(ceil_of(want, tile), most / tile) * tile;
  return std::min<int64_t>(t, std::max<int64_t>(total, 1));
}

}  // namespace csahca
