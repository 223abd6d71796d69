// Shared device helpers for butterfly_amd HIP kernels (gfx950 / CDNA4 only).
//
// Conventions used by every kernel in csrc/kernels:
//   * bf16 storage is `__bf16`; arithmetic is f32; f32->bf16 uses the plain cast,
//     which hipcc lowers to v_cvt_pk_bf16_f32 (RNE, NaN-preserving).
//   * Memory-bound kernels move 16 B per lane (8 x bf16) per access.
//   * Wave width is 64; the code hard-codes it (warpSize folds to 64 on gfx950).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bfly {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWave = 64;

__device__ __forceinline__ float bf2f(bf16 x) { return (float)x; }
__device__ __forceinline__ bf16 f2bf(float x) { return (bf16)x; }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// Inclusive sum over the lanes up to this one
__device__ __forceinline__ int lane_scan(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);     // row_shr 1, 2, 4, 8
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);     // row_bcast 15, 31
  return x + __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);
}

// Which sequence takes the pos-th place of a launch whose workgroups run down a sequence each, two of them on a compute unit: the
// longer first where `round` sequences fill the units once. Where the others are second workgroups there, those of the first `round`
// come from the shortest up, so that the longest run alone and the shortest beside the others. 16 heads of 128 x 128, in the order given
// and so, us: 11 sequences of 200 to 700 rows 195 and 136 (delta rule), 142 and 108 (gated), 14 to 500 140 and 97, 105 and 81, 20 to
// 400 157 and 131, 144 and 138. Steps of one length keep their order, and a rank is three instructions per sequence, of which the compiler
// sees sixteen at a time: short sequences notice either (gated, 8 heads, 64 of 32 rows 39 us, 45 with ranks in a loop; 40 of 5 to 95 with
// 16 heads 76 and 80). With more sequences the places even out: 40 to 200 178 and 170, 123 and 120, 60 to 130 194 and 195, 113 and 121.
__device__ __forceinline__ int by_length(const int* __restrict__ row_cu, int nseq, int pos, int round) {
  if (nseq <= round || nseq > min(64, 5 * round)) return pos;
  const int lane = threadIdx.x & 63, n = lane < nseq ? row_cu[lane + 1] - row_cu[lane] : -1;
  if (!__any(lane < nseq && n != __builtin_amdgcn_readfirstlane(n))) return pos;
  const int key = 64 * n + 63 - lane;      // (all different: of one length the first comes first)
  int before = 0;
  for (int j = 0; j < nseq; j += 16)
#pragma unroll
    for (int i = 0; i < 16; ++i) before += __builtin_amdgcn_readlane(key, j + i) > key;
  const int want = nseq <= 2 * round && pos < round ? round - 1 - pos : pos;
  return __builtin_ctzll(__ballot(lane < nseq && before == want));
}

// Maximum / sum over the four lanes l, l ^ 16, l ^ 32, l ^ 48 (one column of a 16x16 MFMA result) without LDS traffic
__device__ __forceinline__ float row4_max(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float row4_sum(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Block-wide sum for blocks of up to 1024 threads. `red` must hold >= 16 floats.
__device__ __forceinline__ float block_sum(float v, float* red) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nw = (blockDim.x + 63) >> 6;
  v = wave_sum(v);
  if (lane == 0) red[wid] = v;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < nw; ++i) t += red[i];
  __syncthreads();
  return t;
}

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Non-temporal 16-byte load for once-read streams (decode weights, KV pages).
__device__ __forceinline__ bf16x8 ld_nt(const bf16x8* p) {
  return __builtin_nontemporal_load(p);
}

// Bijective XCD-aware remap of a linear workgroup id: blocks that the dispatcher deals
// round-robin over the 8 XCDs (b % 8 share an L2) are renumbered so that each XCD gets a
// contiguous range of logical tiles (cdna_hip_programming.md §5 "XCD swizzle must be bijective").
__device__ __forceinline__ int xcd_remap(int orig, int nwg) {
  const int q = nwg >> 3, r = nwg & 7, xcd = orig & 7;
  return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
}

// MoE routing of token t from one wave holding expert `lane`'s router logit (E <= 64 experts,
// `live` = lane < E): softmax over all experts, top-K by probability (ties to the lowest
// expert id), the selected weights renormalised to sum 1. Writes gates[t][E] (0 for unselected
// experts), topk_ids[t][K] and topk_w[t][K]. Shared by moe_route_kernel and the add+RMSNorm
// that routes the rows it normalises (norm.hip).
__device__ __forceinline__ void moe_select_topk(float logit, bool live, int lane, int t, int E, int K,
                                                float* __restrict__ gates, int* __restrict__ topk_ids,
                                                float* __restrict__ topk_w) {
  logit = live ? logit : -INFINITY;
  const float mx = wave_max(logit);
  float p = live ? __expf(logit - mx) : 0.f;
  const float den = wave_sum(p);
  float g = 0.f, sel_sum = 0.f;
  int my_rank = -1;                     // this expert's position in the top-k (-1: not selected)
  for (int k = 0; k < K; ++k) {
    float bv = live ? p : -1.f;
    int bi = lane;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
    }
    sel_sum += bv / den;
    if (lane == bi) { my_rank = k; g = p / den; p = -1.f; }
  }
  if (!live) return;
  const float w = my_rank >= 0 ? g / sel_sum : 0.f;
  gates[(long)t * E + lane] = w;
  if (my_rank >= 0) {
    topk_ids[(long)t * K + my_rank] = lane;
    topk_w[(long)t * K + my_rank] = w;
  }
}

// a GLU's gate g sigmoid(alpha g), whose limit for alpha = inf is relu(g) (e = exp(-alpha g), unused then)
__device__ __forceinline__ float glu_gate(float g, float alpha, float e) {
  return alpha < INFINITY ? g / (1.f + e) : (g < 0.f ? 0.f : g);
}
__device__ __forceinline__ float silu(float x) { return x / (1.f + __expf(-x)); }
__device__ __forceinline__ float gelu_tanh(float x) {
  const float k0 = 0.7978845608028654f, k1 = 0.044715f;
  return 0.5f * x * (1.f + tanhf(k0 * (x + k1 * x * x * x)));
}

// Grouped expert GEMMs of the score-routed experts (gemm_big4_kernel GROUPED 2 / 3): moe_sort's groups and what the
// epilogues need
struct ExpertArgs {
  const int* perm = nullptr;        // row -> (token, choice) pair
  const int* offsets = nullptr;     // [E + 1] group bounds
  const int* tiles = nullptr;       // [..][2] (expert, first row)
  const float* topk_w = nullptr;    // up: the pair's score scales the row (nullptr: 1)
  int choices = 1, plain = 0;       // choices per token; plain: squared ReLU without a gate
  float limit = 0.f, alpha = 0.f, up_offset = 0.f;
  float* y = nullptr;               // down: f32 rows in pair order
};

// Scans over packed rows that come row by row and in chunks of 16 rows: which form takes which sequences of a step. Chunks take the
// time of `first` single rows and of `each` more per chunk, padded or not (chunk_cost): a sequence runs in chunks where that is no
// more than its rows. The host knows only the sum of the rows, so a step that may hold both kinds launches both forms, and every
// workgroup looks at its own sequence. The second launch (2 to 5 us) is saved where no sequence is long enough (max_rows, where the
// caller knows it) or repays it (six times the rows of the shortest sequence in chunks, or those of one chunk, beyond one each, none
// of them empty), and for steps of prompts where the shorter sequences cost the chunk form no more than that: `wgs` workgroups per
// sequence, at 11 to 25 ns for one with a single row.
struct ScanForms {
  bool rows, chunks;
};
__host__ __device__ constexpr int chunk_cost(int first, int each) { return first << 8 | each; }
__host__ __device__ inline bool scan_in_chunks(long n, int cost) { return (cost >> 8) + (cost & 255) * ((n + 15) >> 4) <= n; }
inline ScanForms scan_forms(long T, long nseq, int cost, long wgs, long max_rows) {
  if (nseq == 1) return {!scan_in_chunks(T, cost), scan_in_chunks(T, cost)};
  long least = 1;
  while (least < 256 && !scan_in_chunks(least, cost)) ++least;
  if (T - nseq < 6 * (least < 16 ? least : 16) || (max_rows > 0 && max_rows < least)) return {true, false};
  return {!(scan_in_chunks(T / nseq, cost) && nseq * wgs <= 512), true};
}
// (`cost` 0 in a kernel: it takes every sequence)

}  // namespace bfly

#define BFLY_HIP_CHECK(expr)                                                  \
  do {                                                                        \
    hipError_t _e = (expr);                                                   \
    if (_e != hipSuccess) {                                                   \
      fprintf(stderr, "HIP error %s at %s:%d\n", hipGetErrorString(_e),       \
              __FILE__, __LINE__);                                            \
    }                                                                         \
  } while (0)
