// Rules on sizes that choose a launch, free of HIP so that a host compiler
// builds them alone (tests/test_dispatch_rules.py).
#pragma once

#include <algorithm>
#include <cstdint>

namespace csahca {

// Slots per wavefront of the split-KV attention: the caller's tile, or more
// where that is better.  A tile is a hint for the split, and larger tiles are
// fewer partials, so the workspace the caller sized for its own tile holds
// them.  `vec`: the vectorised kernel runs (esz: bytes per element).
//
// The least number of whole load batches that, for the vectorised kernel,
//   * fills one batch of row loads (16 slots at 16-bit head_dim 128, 32 at 64;
//     a smaller tile re-reads its last row);
//   * leaves a head at most 64 tiles, the one-round-trip merge, as long as that
//     makes tiles of at most 128 slots;
//   * leaves the call at most 8192 wavefronts (32 per CU): more only write and
//     merge more partials.
// Measured (graph period, us, tile 8 as called / split chosen): B1 H8 D128
// top-8 5.31 / 5.06, top-32 49.3 / 7.3; B8 top-16 16.4 / 10.3, top-32 60.6 /
// 15.3; B32 top-32 104.7 / 56.7; B4 H12 D64 f16 480 slots 7.3 / 6.4; f32 D256
// 512 slots 9.4 (kept at 8).  Multiples of the caller's tile would pass the line
// by up to a tile, a serial chain twice as long: f32 D128 H12 4352 slots, tile
// 64, with tiles of 64 / 72 / 128 20.0 / 17.0 / 24.4; f32 D64 H8 6000, tile 80, of
// 80 / 96 / 160 14.2 / 11.6 / 15.5.
//
// Generic kernel: its wavefronts take 4 slots per round trip, 0.23 us a slot at
// D 40 to 0.39 at D 320 f32, so long tiles are a long serial chain, and the
// merge of more than 64 partials is the cheaper side until the rows themselves
// take that long to stream: the same line, with 12800 wavefronts for rows below
// 1 KiB, but at most 16 slots, 32 from 100 MiB of rows, any number from 200 MiB
// of rows of at least 384 bytes.  Measured, us, with tiles of 8 / 16 / 32 /
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
  if (!vec) {
    const double mib = 2.0 * static_cast<double>(total) * static_cast<double>(bh * D * esz) / (1 << 20);
    if (mib < 200.0 || D * esz < 384) want = std::min<int64_t>(want, mib < 100.0 ? 16 : 32);
  }
  const int64_t t = std::max(tile, ceil_of(want, batch) * batch);
  return std::min<int64_t>(t, std::max<int64_t>(total, 1));
}

// The largest selection that the register path takes of C <= 2048 chunks (up to
// 16 heads: few_heads).  It fails where more than 64 keys reach its threshold,
// the k-th largest of the 64 lanes' maxima: never for k + C <= 128 distinct keys
// (C - 64 lanes hold a second one), and of many independent keys 64 ln(64 / (64
// - k)) reach it (44 for k = 32, 53 for 36, 63 for 40), fewer of few per lane.
// The radix select behind it costs 6-20 us, and one head of the call that takes
// it costs the call that.  So the line is where a call of all its heads still
// rarely fails.  Simulated, failures a head: 96 chunks k = 43, 45 1e-4, 3e-3;
// 128 k = 41, 43 5e-5, 2e-3; 144 k = 39, 41 2e-4, 2e-3; 192 k = 37, 39 5e-5, 1e-3;
// 256 k = 36, 38, 40 9e-5, 2.6e-3, 2.7e-2; 512 k = 34, 36, 38 5e-5, 2.9e-3,
// 2.6e-2; 2048 k = 34, 36, 38 1.1e-3, 1.3e-2, 7.9e-2.  Measured, registers (not
// failing) against block_topk, us a step, B1 H8 D128 chunk 16: top-33 of 256,
// 512, 1024, 2048: 9.4 / 10.1, 9.5 / 10.5, 11.6 / 11.7, 12.9 / 13.5; top-36 of 256,
// 512: 9.4 / 10.1, 9.6 / 10.5; top-40 of 64, 128: 9.3 / 10.0, 9.3 / 9.8, and
// failing, of 384: 17.6 / 10.5; top-64 of 64, 128, 512, 2048: 9.6 / 10.2, 18.3 /
// 10.7, 21.4 / 11.5, 36.2 / 13.7; 48 heads of 64, top-37 of 132 12.9 / 13.9; 16
// heads of 256, the selection op, top-50 of 65 6.3 / 6.7.
inline int64_t csa_topk_regs_most(int64_t C, bool few_heads) {
  if (C <= 64) return 64;
  if (C <= 84) return 128 - C;
  const int64_t most = C <= 96 ? 43 : C <= 128 ? 41 : C <= 144 ? 39 : C <= 192 ? 37 : C <= 256 ? 36 : C <= 512 ? 34 : 32;
  return most + (few_heads ? 2 : 0);
}

// Register-path size for the fused step's selection of k of C chunks: keys per
// lane M (C <= 64 * M), or 0 for block_topk (k <= 64) or the radix select.
// Kernels take M as a template parameter so each instantiation carries exactly
// one of them.
// The fewest keys per lane that hold C: `fine` where the kernels with 2 and 16
// exist (head_dim 128 in 16 bits; bf16 us a step, top-8: 128 chunks with 8 and
// with 2 7.92 / 7.59, 1024 with 32 and with 16 10.0 / 9.15).
inline int csa_step_topk_regs(int64_t C, int64_t k, int64_t bh, bool fine) {
  if (C > 2048 || k > csa_topk_regs_most(C, bh <= 16)) return 0;
  if (fine && C <= 128) return 2;
  if (C <= 512) return 8;
  return fine && C <= 1024 ? 16 : 32;
}

// The same for the selection op: keys per lane of its one-wavefront kernel, or 0
// for the workgroup's.  Measured, 8 heads, registers against block_topk, us a
// call with the scores: top-32 of 64, 128: 4.5 / 5.1, 5.0 / 5.4; top-40, 48 of
// 128: 5.2 / 5.4, 11.7 / 5.3; top-8 of 129, 160, 192: 4.94 / 5.32, 5.18 / 5.30,
// 5.11 / 5.27; top-36 of 129, 192: 5.32 / 5.76, 5.56 / 5.72; top-16 level.
inline int csa_select_topk_regs(int64_t C, int64_t k) {
  if (C > 192 || k > csa_topk_regs_most(C, false)) return 0;
  return C <= 128 ? 2 : 4;
}

// Whether the hybrid op reads K once for the summaries and the HCA chunk pass
// (`items` HCA chunks of hca_chunk rows over all heads).  A wavefront walks a
// whole HCA chunk of one tensor, and is the longer chain where few others run
// beside it, the more so the fewer row groups (4096 bytes of K) lie in a CSA
// chunk, whose end it stops to reduce: there long chunks go in two reads.  With
// head_dim 128 in 16 bits the other route runs the step beside the HCA pass,
// which hides it: there the second read of K has to cost more than the step,
// from about 64 MiB of K (48 for short chunks).  One read / two, time ratio by
// HCA chunk, row groups a CSA chunk (g) and items, 8 heads and 64:
//   32 KiB: bf16 D64 g1 of 32, 128, 192, 256 1.06, 1.04, 1.03, 1.00, g2 .95, .94,
//   .93, .88; f32 D64 g1 .97 of 16 to 128; D256 bf16 .92-.97;
//   64 KiB: bf16 D64 g1 of 64, 128, 256, 512 1.26, 1.16, 1.04, .87, g2 1.07, .96,
//   .93, .78, g4 1.02, 1.01, .94, .80; bf16 D256 g2 of 64, 128, 192, 256 1.08, .99,
//   .99, .95, g4 1.10, 1.03, 1.01, .97, g8 1.06, .98, .97, .94; f32 D64 g1 1.09,
//   1.06, .98, .93, g2 .98, .89; f32 D128 .95-1.02 of 16 to 128; f32 D256 of 64,
//   128 1.07, .97;
//   128 KiB: bf16 D64 g1 of 128, 256, 512 1.40, 1.15, .84, g2 1.15, .95, .79, g4
//   1.08, .93; bf16 D256 g2 of 128, 192, 256 1.15, 1.12, .95, g8 1.05, .99, .92; f32
//   D64 g1 of 128, 192, 256 1.15, 1.05, .96, g2 of 32, 64 1.12, .97; f32 D128 g4
//   of 64, 128 1.07, .98; f32 D256 1.10, .98;
//   512 KiB: f32 D256 of 64, 1024 1.06, .71;
//   bf16 D128, 48 MiB of K in chunks of 16 KiB .95; of 64 KiB g1 1.05, g4 1.03; of
//   128 KiB g1 1.23, g4 1.01; 64 MiB of 96 KiB g3 .97, 128 KiB g1 1.06, g4 .93; 79
//   MiB of 64 KiB g1 .88.
inline bool csa_hybrid_one_read(int64_t esz, int64_t head_dim, int64_t csa_chunk, int64_t hca_chunk, int64_t items) {
  constexpr int64_t KiB = 1024, MiB = 1024 * 1024;
  const int64_t bytes = hca_chunk * head_dim * esz, groups = csa_chunk * head_dim * esz / 4096;
  if (bytes > 128 * KiB && items < 512) return false;
  if (esz == 2 && head_dim == 128)
    return items * bytes >= (bytes <= 16 * KiB ? 48 * MiB : groups <= 1 && bytes > 64 * KiB ? 80 * MiB : 64 * MiB);
  int64_t fewest = 1;
  if (bytes > 64 * KiB)
    fewest = esz == 4 ? (groups <= 1 ? 256 : 128) : groups <= 1 ? 512 : groups >= 8 ? 192 : 256;
  else if (bytes > 32 * KiB)
    fewest = esz == 4 ? (groups <= 1 ? 192 : head_dim == 256 ? 128 : 1)
                      : groups <= 1 ? 512 : head_dim == 64 || groups >= 8 ? 128 : 256;
  else if (bytes > 16 * KiB && esz == 2 && groups <= 1)
    fewest = 256;
  return items >= fewest;
}

}  // namespace csahca
