// hca.hip -- heavily compressed attention (HCA) decode and the CSA/HCA hybrid
// blend, for gfx950.
//
// hca_reference (hybrid_attention/reference.py:87-92): K and V are mean-pooled
// per chunk (fp32 mean, then rounded to the storage type) and the query
// attends to all C = S/chunk summary rows with full softmax attention whose
// probabilities are rounded to the storage type before the PV product
// (reference.py:31-37).  hybrid_reference (reference.py:95-108) blends
// w*csa + (1-w)*hca with each product and the sum rounded to the storage type.
//
// Kernels:
//   hca_chunk_kernel  one workgroup per (b, h, chunk) streams the chunk's K and
//                     V rows with 16-byte lane loads (the whole op is one pass
//                     over K and V: HBM-bound), reduces them to the two rounded
//                     means, scores the K mean against q and writes the
//                     score (scores[b,h,c]) and the V mean (means[b,h,c,:])
//                     to the workspace;
//   hybrid_chunk_kernel  the chunk pass above and the CSA summaries of the same
//                     K rows, from one read of K (the hybrid op that builds its
//                     own summaries): one wavefront per chunk and tensor;
//   hca_merge_kernel  one workgroup per (b, h, block of 32 output columns):
//                     softmax over the C scores, probabilities rounded to the
//                     storage type, sum of its columns of the V means,
//                     optional blend with a CSA output.  Spreading a head's
//                     columns over workgroups keeps each one to a single round
//                     trip of ~C x 128 bytes even at batch 1.
#include "csa_device.hpp"
#include "dispatch.hpp"
#include "hca_device.hpp"

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdlib>

namespace csahca {
namespace {

constexpr int kHcaProbChunk = 2048;  // probabilities staged in LDS per pass

// Parameter order: the inputs of the first loads (q, K, V and the sizes that
// place them) lead, so they fit the 14 dwords preloaded into SGPRs at wave
// launch (the library builds this file with -amdgpu-kernarg-preload-count);
// the outputs and the scale, needed at the end, follow.
template <typename T, bool kVec>
__global__ __launch_bounds__(kHcaThreads) void hca_chunk_kernel(const T* __restrict__ q,
                                                              const T* __restrict__ k,
                                                              const T* __restrict__ v, int64_t S,
                                                              int64_t C, int D, int chunk,
                                                              float* __restrict__ scores,
                                                              float* __restrict__ means, float scale) {
  hca_chunk_body<T, kVec>(q, k, v, scores, means, S, D, chunk, C, scale, blockIdx.x);
}

// The HCA chunk pass and the CSA chunk summaries from one read of K and V.
// Wavefront 2i of the grid takes K of HCA chunk i, wavefront 2i + 1 its V, in
// the summary kernel's lane split: lane (grp, col) takes rows grp, grp + RPL,
// ... of VEC columns.  Of the rows one lane adds, every fourth belongs to the
// same row group of hca_chunk_body (256 / LPR = 4 RPL groups), so it keeps 4
// group sums, in that body's order, beside the running sum of the CSA chunk:
// both results have the bits of the separate kernels.  HBM-bound: kHybridRows
// 16-byte loads in flight per lane, no barrier.  (Measured, B2 H8 S32768 D128
// bf16, chunks 64 and 256, us a hybrid call: the summary kernel, then the step
// beside the HCA pass, 71.2; this kernel, then the step, 64.4.  8 loads: level
// where wavefronts fill the chip, 20% slower where they do not, 256 of them on
// 128 MiB.)
constexpr int kHybridRows = 16;
constexpr int kHybridWaves = 4;

template <typename T, int D>
__global__ __launch_bounds__(kHybridWaves * kWave) void hybrid_chunk_kernel(
    const T* __restrict__ k, const T* __restrict__ v, int64_t items, int hca_chunk, int csa_chunk,
    float* __restrict__ summary, const T* __restrict__ q, uint32_t hca_chunks, float* __restrict__ scores,
    float* __restrict__ means, float scale) {
  using L = AttendLayout<T, D>;
  constexpr int VEC = L::VEC, LPR = L::LPR, RPL = L::RPL;
  constexpr int G = 4;                // group sums per lane
  constexpr int R = G * RPL;          // row groups of hca_chunk_body
  constexpr int U = kHybridRows;
  static_assert(R * LPR == kHcaThreads && U % G == 0, "the row groups of hca_chunk_body");
  __shared__ __align__(16) float sums[kHybridWaves][R * D];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int grp = lane / LPR, col = lane % LPR;
  const int64_t item = static_cast<int64_t>(blockIdx.x) * (kHybridWaves / 2) + wave / 2;
  if (item >= items) return;
  const bool is_k = (wave & 1) == 0;
  // S is a multiple of both chunk sizes: chunks lie end to end over all heads.
  const T* __restrict__ base = (is_k ? k : v) + item * hca_chunk * D + col * VEC;
  float* __restrict__ dst = summary + item * (hca_chunk / csa_chunk) * D + col * VEC;
  const float fc = static_cast<float>(csa_chunk);
  float hs[G][VEC], acc[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) {
    acc[e] = 0.f;
#pragma unroll
    for (int g = 0; g < G; ++g) hs[g][e] = 0.f;
  }
  int left = csa_chunk;  // rows of the open CSA chunk not yet added
  for (int r0 = 0; r0 < hca_chunk; r0 += U * RPL) {
    uint4 x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {  // (rows past the chunk read its last rows again)
      const int r = r0 + (u / G) * R < hca_chunk ? r0 + u * RPL : hca_chunk - R + (u % G) * RPL;
      x[u] = load_global_u4(base + static_cast<int64_t>(r + grp) * D);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < U / G; ++b) {
      if (r0 + b * R < hca_chunk) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
          float f[VEC];
          widen16<T>(x[b * G + g], f);
#pragma unroll
          for (int e = 0; e < VEC; ++e) {
            hs[g][e] += f[e];
            acc[e] += f[e];
          }
        }
        left -= R;
        if (left == 0) {
          left = csa_chunk;
          if (is_k) {
#pragma unroll
            for (int off = LPR; off < kWave; off <<= 1)
#pragma unroll
              for (int e = 0; e < VEC; ++e) acc[e] += xor_lanes(acc[e], off);
            if (grp == 0) {
#pragma unroll
              for (int e = 0; e < VEC; ++e) dst[e] = acc[e] / fc;
            }
            dst += D;
          }
#pragma unroll
          for (int e = 0; e < VEC; ++e) acc[e] = 0.f;
        }
      }
    }
  }
  float* s = sums[wave];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int e = 0; e < VEC; ++e) s[(grp + g * RPL) * D + col * VEC + e] = hs[g][e];
  wave_lds_sync();
  const float inv_n = 1.f / static_cast<float>(hca_chunk);
  const T* qp = q + static_cast<int64_t>(static_cast<uint32_t>(item) / hca_chunks) * D;
  float dot = 0.f;
#pragma unroll
  for (int d0 = 0; d0 < D; d0 += kWave) {
    const int d = d0 + lane;
    float a = 0.f;
#pragma unroll
    for (int g = 0; g < R; ++g) a += s[g * D + d];
    const float m = round_to<T>(a * inv_n);
    if (is_k) {
      const float part = wave_sum(fmaf(to_f32(qp[d]), m, 0.f));
      dot = d0 == 0 ? part : dot + part;
    } else {
      means[item * D + d] = m;
    }
  }
  if (is_k && lane == 0) scores[item] = dot * scale;
}

// Merge thread layout: 32 columns x 8 row groups; a wavefront reads 2 rows of
// 128 contiguous bytes per load.  When C <= 256 every score and every V-mean
// value a thread needs is requested before the first wait (one round trip);
// larger C runs in passes of kHcaProbChunk rows, kMergeRows rows per batch.
constexpr int kMergeCols = 32;
constexpr int kMergeRowGroups = kHcaThreads / kMergeCols;  // 8
constexpr int kMergeRows = 32;                             // rows per thread per batch
constexpr int kMergeFastRows = kMergeRows * kMergeRowGroups;  // 256
static_assert(kMergeFastRows <= kHcaThreads, "one score per thread in the one-round-trip path");

template <typename T>
__global__ __launch_bounds__(kHcaThreads) void hca_merge_kernel(const float* __restrict__ scores,
                                                              const float* __restrict__ means,
                                                              const T* __restrict__ blend,
                                                              float w_csa, T* __restrict__ out,
                                                              int64_t C, int D, int col_blocks) {
  __shared__ float s_p[kHcaProbChunk];
  __shared__ float s_sum[kHcaThreads];
  __shared__ float red[kHcaThreads / kWave];
  const int tid = threadIdx.x;
  const int64_t bh = blockIdx.x / col_blocks;
  const int cb = static_cast<int>(blockIdx.x - bh * col_blocks);
  const int rg = tid / kMergeCols, cl = tid % kMergeCols;
  const int d = cb * kMergeCols + cl;
  const bool has_col = d < D;
  const float* sb = scores + bh * C;
  const float* col = means + bh * C * D + (has_col ? d : 0);  // column 0 stands in: loads stay in bounds

  float a = 0.f;
  if (C <= kMergeFastRows) {
    const int n = static_cast<int>(C);
    // Unconditional loads (clamped indices, values dropped after the load):
    // the score and the V-mean column values are one batch in flight.
    const float sraw = load_global_raw<float>(sb + (tid < n ? tid : 0));
    float x[kMergeRows];
#pragma unroll
    for (int i = 0; i < kMergeRows; ++i) {
      const int r = rg + i * kMergeRowGroups;
      x[i] = load_global_raw<float>(col + static_cast<int64_t>(r < n ? r : 0) * D);
    }
    const float sc = tid < n ? sraw : -INFINITY;
    const float M = block_reduce(sc, red, true);
    const float e = (tid < n && M != -INFINITY) ? fast_exp2((sc - M) * kLog2e) : 0.f;
    const float L = block_reduce(e, red, false);
    const float iv = L > 0.f ? 1.f / L : 0.f;
    // softmax in fp32, then the cast of the probabilities to the V dtype
    if (tid < n) s_p[tid] = round_to<T>(e * iv);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kMergeRows; ++i) {
      const int r = rg + i * kMergeRowGroups;
      if (r < n) a = fmaf(s_p[r], x[i], a);
    }
  } else {
    float mx = -INFINITY;
    for (int64_t c = tid; c < C; c += kHcaThreads) mx = fmaxf(mx, sb[c]);
    mx = block_reduce(mx, red, true);
    float L = 0.f;
    if (mx != -INFINITY)
      for (int64_t c = tid; c < C; c += kHcaThreads) L += fast_exp2((sb[c] - mx) * kLog2e);
    L = block_reduce(L, red, false);
    const float inv = L > 0.f ? 1.f / L : 0.f;
    for (int64_t p0 = 0; p0 < C; p0 += kHcaProbChunk) {
      const int pn = static_cast<int>(std::min<int64_t>(kHcaProbChunk, C - p0));
      for (int c = tid; c < pn; c += kHcaThreads)
        s_p[c] = mx != -INFINITY ? round_to<T>(fast_exp2((sb[p0 + c] - mx) * kLog2e) * inv) : 0.f;
      __syncthreads();
      const float* cp = col + p0 * D;
      for (int r0 = rg; r0 < pn; r0 += kMergeRows * kMergeRowGroups) {
        float x[kMergeRows];
#pragma unroll
        for (int i = 0; i < kMergeRows; ++i) {
          const int r = r0 + i * kMergeRowGroups;
          x[i] = cp[static_cast<int64_t>(r < pn ? r : r0) * D];
        }
#pragma unroll
        for (int i = 0; i < kMergeRows; ++i) {
          const int r = r0 + i * kMergeRowGroups;
          if (r < pn) a = fmaf(s_p[r], x[i], a);
        }
      }
      __syncthreads();
    }
  }
  s_sum[tid] = a;
  __syncthreads();
  if (rg == 0 && has_col) {
    float o = 0.f;
#pragma unroll
    for (int g = 0; g < kMergeRowGroups; ++g) o += s_sum[g * kMergeCols + cl];
    o = round_to<T>(o);
    if (blend) {
      // w*csa + (1-w)*hca with each product and the sum rounded to T
      const float ab = round_to<T>(w_csa * to_f32(blend[bh * D + d]));
      const float bb = round_to<T>((1.f - w_csa) * o);
      o = ab + bb;
    }
    out[bh * D + d] = from_f32<T>(o);
  }
}

}  // namespace
}  // namespace csahca

using namespace csahca;

namespace {
// Workspace: scores f32[B*H*C], then (256-byte aligned) means f32[B*H*C*D].
size_t hca_means_offset(int64_t n_scores) {
  return (static_cast<size_t>(n_scores) * sizeof(float) + 255) & ~size_t{255};
}

// CSAHCA_HYBRID_ONE_READ=0 / 1 turns hybrid_chunk_kernel off / on wherever it
// applies (read per call); unset (-1): the rule of csa_hybrid_one_read.
int env_one_read() {
  const char* s = std::getenv("CSAHCA_HYBRID_ONE_READ");
  return s ? (std::atoi(s) != 0 ? 1 : 0) : -1;
}

// Whether the hybrid op that builds its own summaries reads K once
// (hybrid_chunk_kernel): whole CSA chunks of whole row groups, and the measured
// rule (csa_hybrid_one_read).
bool hybrid_one_read(int dtype, int64_t head_dim, int64_t csa_chunk, int64_t hca_chunk, int64_t items) {
  if (dtype == CSAHCA_F64 || (head_dim != 64 && head_dim != 128 && head_dim != 256)) return false;
  const int64_t esz = dtype == CSAHCA_F32 ? 4 : 2;
  if (hca_chunk % csa_chunk != 0 || csa_chunk % (kHcaThreads * (16 / esz) / head_dim) != 0) return false;
  const int env = env_one_read();
  if (env >= 0) return env == 1;
  return csa_hybrid_one_read(esz, head_dim, csa_chunk, hca_chunk, items);
}
}  // namespace

extern "C" size_t csahca_hca_decode_workspace_bytes(int64_t batch, int64_t heads, int64_t seq_len,
                                                   int64_t head_dim, int64_t chunk_size) {
  if (batch < 0 || heads < 0 || seq_len < 0 || head_dim < 0 || chunk_size <= 0) return 0;
  const int64_t C = seq_len / chunk_size;
  return hca_means_offset(batch * heads * C) + static_cast<size_t>(batch * heads * C * head_dim) * sizeof(float);
}

extern "C" int csahca_hca_decode_forward(const void* q, const void* k_cache, const void* v_cache,
                                         const void* blend_src, double blend_weight, void* out,
                                         int dtype, int64_t batch, int64_t heads, int64_t seq_len,
                                         int64_t head_dim, int64_t chunk_size, void* workspace,
                                         size_t workspace_bytes, void* stream_ptr) {
  clear_error();
  CSAHCA_REQUIRE(valid_dtype(dtype), "q, k_cache and v_cache must be float32, float64, float16 or bfloat16");
  CSAHCA_REQUIRE(batch >= 0 && heads >= 0 && seq_len >= 0 && head_dim >= 0, "negative dimension");
  CSAHCA_REQUIRE(chunk_size > 0 && chunk_size <= INT_MAX, "chunk_size must be positive");
  CSAHCA_REQUIRE(seq_len % chunk_size == 0, "seq length must be divisible by chunk_size");
  CSAHCA_REQUIRE(head_dim <= 1024, "head_dim > 1024 is not supported");
  const int64_t bh = batch * heads;
  if (bh == 0 || head_dim == 0) return CSAHCA_OK;
  CSAHCA_REQUIRE(q && k_cache && v_cache && out, "null tensor pointer");
  const int64_t C = seq_len / chunk_size;
  if (C == 0) return fail(CSAHCA_ERR_ARGUMENT, "seq length must be at least chunk_size");
  CSAHCA_REQUIRE(bh * C <= INT32_MAX, "too many chunks in one call");
  const size_t need = csahca_hca_decode_workspace_bytes(batch, heads, seq_len, head_dim, chunk_size);
  if (workspace == nullptr || workspace_bytes < need)
    return fail(CSAHCA_ERR_WORKSPACE, "workspace too small for hca decode");
  hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
  float* scores = static_cast<float*>(workspace);
  float* means = reinterpret_cast<float*>(static_cast<char*>(workspace) + hca_means_offset(bh * C));
  const float scale = static_cast<float>(1.0 / std::sqrt(static_cast<double>(head_dim)));
  const int D = static_cast<int>(head_dim);
  return dispatch_dtype(dtype, [&](auto tag) -> int {
    using T = decltype(tag);
    constexpr int VEC = Vec16<T>::N;
    const bool vec = D % VEC == 0 &&
                     ((reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache)) % 16) == 0;
    const int nvc = vec ? D / VEC : D;
    const int R = kHcaThreads / std::min(nvc, kHcaThreads);
    const size_t lds = 2 * static_cast<size_t>(R) * D * sizeof(float);
    const dim3 grid(static_cast<uint32_t>(bh * C));
    const T* qp = static_cast<const T*>(q);
    const T* kp = static_cast<const T*>(k_cache);
    const T* vp = static_cast<const T*>(v_cache);
    const int rc =
        vec ? launch("hca_chunk_kernel", hca_chunk_kernel<T, true>, grid, dim3(kHcaThreads), lds, stream, qp,
                     kp, vp, seq_len, C, D, static_cast<int>(chunk_size), scores, means, scale)
            : launch("hca_chunk_kernel", hca_chunk_kernel<T, false>, grid, dim3(kHcaThreads), lds, stream, qp,
                     kp, vp, seq_len, C, D, static_cast<int>(chunk_size), scores, means, scale);
    if (rc != CSAHCA_OK) return rc;
    const int col_blocks = (D + kMergeCols - 1) / kMergeCols;
    CSAHCA_REQUIRE(bh * col_blocks <= INT32_MAX, "too many heads in one call");
    return launch("hca_merge_kernel", hca_merge_kernel<T>, dim3(static_cast<uint32_t>(bh * col_blocks)),
                  dim3(kHcaThreads), 0, stream, static_cast<const float*>(scores),
                  static_cast<const float*>(means), static_cast<const T*>(blend_src),
                  static_cast<float>(blend_weight), static_cast<T*>(out), C, D, col_blocks);
  });
}

namespace csahca {

// The HCA merge (+ optional blend) from a workspace a chunk pass of shape
// (bh, C, D) filled; used by the hybrid step, which runs the chunk pass inside
// its own kernel.
int hca_merge_launch(int dtype, void* workspace, const void* blend_src, double blend_weight, void* out,
                     int64_t bh, int64_t C, int D, hipStream_t stream) {
  const float* scores = static_cast<const float*>(workspace);
  const float* means =
      reinterpret_cast<const float*>(static_cast<const char*>(workspace) + hca_means_offset(bh * C));
  const int col_blocks = (D + kMergeCols - 1) / kMergeCols;
  CSAHCA_REQUIRE(bh * col_blocks <= INT32_MAX, "too many heads in one call");
  return dispatch_dtype(dtype, [&](auto tag) -> int {
    using T = decltype(tag);
    return launch("hca_merge_kernel", hca_merge_kernel<T>, dim3(static_cast<uint32_t>(bh * col_blocks)),
                  dim3(kHcaThreads), 0, stream, scores, means, static_cast<const T*>(blend_src),
                  static_cast<float>(blend_weight), static_cast<T*>(out), C, D, col_blocks);
  });
}

// Byte offset of the V means in an HCA workspace holding n chunk scores.
size_t hca_workspace_means_offset(int64_t n_scores) { return hca_means_offset(n_scores); }

}  // namespace csahca

extern "C" int csahca_hybrid_decode_forward_build(const void* q, const void* k_cache, const void* v_cache,
                                                  float* summary, void* csa_out, int32_t* csa_indices, void* out,
                                                  int dtype, int64_t batch, int64_t heads, int64_t seq_len,
                                                  int64_t head_dim, int64_t csa_chunk_size, int64_t top_k,
                                                  int64_t hca_chunk_size, double csa_weight, void* step_workspace,
                                                  size_t step_workspace_bytes, void* hca_workspace,
                                                  size_t hca_workspace_bytes, void* stream_ptr) {
  clear_error();
  CSAHCA_REQUIRE(valid_dtype(dtype), "q, k_cache and v_cache must be float32, float64, float16 or bfloat16");
  CSAHCA_REQUIRE(batch >= 0 && heads >= 0 && seq_len >= 0 && head_dim >= 0, "negative dimension");
  CSAHCA_REQUIRE(csa_chunk_size > 0 && csa_chunk_size <= INT_MAX, "chunk_size must be positive");
  CSAHCA_REQUIRE(hca_chunk_size > 0 && hca_chunk_size <= INT_MAX, "chunk_size must be positive");
  CSAHCA_REQUIRE(seq_len % csa_chunk_size == 0 && seq_len % hca_chunk_size == 0,
                 "seq length must be divisible by chunk_size");
  const int64_t bh = batch * heads, C = seq_len / csa_chunk_size, Ch = seq_len / hca_chunk_size;
  const size_t need = csahca_hca_decode_workspace_bytes(batch, heads, seq_len, head_dim, hca_chunk_size);
  const bool one_read = bh > 0 && Ch > 0 && bh * Ch <= INT32_MAX && q && k_cache && v_cache && out && csa_out && summary &&
                  hca_workspace != nullptr && hca_workspace_bytes >= need &&
                  ((reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache)) % 16) == 0 &&
                  hybrid_one_read(dtype, head_dim, csa_chunk_size, hca_chunk_size, bh * Ch);
  if (!one_read) {
    const int rc = csahca_csa_chunk_summary(k_cache, summary, dtype, batch, heads, seq_len, head_dim, csa_chunk_size,
                                            C, 0, C, stream_ptr);
    if (rc != CSAHCA_OK) return rc;
    return csahca_hybrid_decode_forward(q, k_cache, v_cache, summary, csa_out, csa_indices, out, dtype, batch, heads,
                                        seq_len, head_dim, C, csa_chunk_size, top_k, hca_chunk_size, csa_weight,
                                        step_workspace, step_workspace_bytes, hca_workspace, hca_workspace_bytes,
                                        stream_ptr);
  }
  hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
  float* scores = static_cast<float*>(hca_workspace);
  float* means = reinterpret_cast<float*>(static_cast<char*>(hca_workspace) + hca_means_offset(bh * Ch));
  const float scale = static_cast<float>(1.0 / std::sqrt(static_cast<double>(head_dim)));
  auto run = [&](auto tag, auto dim) -> int {
    using T = decltype(tag);
    constexpr int D = decltype(dim)::value;
    return launch("hybrid_chunk_kernel", hybrid_chunk_kernel<T, D>,
                  dim3(static_cast<uint32_t>(ceil_div(bh * Ch, int64_t{kHybridWaves / 2}))),
                  dim3(kHybridWaves * kWave), 0, stream, static_cast<const T*>(k_cache),
                  static_cast<const T*>(v_cache), bh * Ch, static_cast<int>(hca_chunk_size),
                  static_cast<int>(csa_chunk_size), summary, static_cast<const T*>(q), static_cast<uint32_t>(Ch),
                  scores, means, scale);
  };
  auto with_dim = [&](auto tag) -> int {
    if (head_dim == 64) return run(tag, std::integral_constant<int, 64>{});
    if (head_dim == 128) return run(tag, std::integral_constant<int, 128>{});
    return run(tag, std::integral_constant<int, 256>{});
  };
  int rc = dtype == CSAHCA_BF16 ? with_dim(bf16{}) : dtype == CSAHCA_F16 ? with_dim(f16{}) : with_dim(0.0f);
  if (rc != CSAHCA_OK) return rc;
  rc = csahca_csa_decode_step(q, k_cache, v_cache, summary, csa_out, csa_indices, dtype, batch, heads, seq_len,
                              head_dim, C, csa_chunk_size, top_k, step_workspace, step_workspace_bytes, stream_ptr);
  if (rc != CSAHCA_OK) return rc;
  return hca_merge_launch(dtype, hca_workspace, csa_out, csa_weight, out, bh, Ch, static_cast<int>(head_dim), stream);
}
