// MFMA GEMMs for every linear layer (K1 prefill GEMM, K2 decode skinny GEMM, K13 expert GEMM).
//
//   Y[M, N] = X[M, K] . W[N, K]^T        (W in nn.Linear [out, in] layout: both operands are
//                                          K-contiguous, the natural MFMA "NT" layout)
// Epilogues (fused, so the activation never makes an extra HBM round trip):
//   EPI_NONE  : Y = acc
//   EPI_BIAS  : Y = acc + bias[n]
//   EPI_RELU2 : Y = max(acc, 0)^2
//   EPI_SILU  : W's rows are gate/up interleaved in 16-row groups (g0 u0 g1 u1 ...);
//               Y[M, N/2] = silu(gate) * up  (the SwiGLU FFN's first half in one kernel)
//   EPI_GLU   : the same row layout; Y[M, N/2] = g sigmoid(alpha g) (u + offset) with g = min(gate
//               + bias, limit), u = clamp(up + bias, +-limit); bias and the three constants come
//               in one block (bfly_kernels.h)
//
// Kernels, picked by M on the host (gemm_stream_kernel, gemm_dec_kernel, gemm_mid*_kernel and gemm_big4_kernel have their own notes):
//  * gemm_skinny (M <= 64, decode): weight-streaming. Each wave streams 16*NT rows of W
//    straight into VGPRs with non-temporal 16-B loads (no LDS round trip for an operand that is
//    read exactly once: cdna_hip_programming.md §5 table, "GEMV / M <= 16" row), X fragments
//    come from L2. W is the MFMA A operand (16 weight rows per mfma_f32_16x16x32_bf16) and the
//    tokens are the B operand, so one weight fragment feeds MT token tiles. The K loop is
//    split over the 4 waves of a workgroup and, for narrow N, over workgroups (split-K with
//    f32 partial slabs and a reduce kernel that applies the epilogue).
//    K permutation: per 128-wide K chunk, sub-step s, lane group g = lane>>4 and element j
//    hold physical k = 32s + 8g + j, so each load instruction reads 64 contiguous bytes per
//    row; the same map is used for both operands, so every product pairs matching k.
//  * gemm_tile (M > 64, prefill / large-batch decode): BMx128x64 LDS-tiled, 4 waves (2x2),
//    both operands staged global->LDS by global_load_lds_dwordx4 (no VGPR round trip) into
//    two buffers (load of tile t+1 overlaps MFMAs on tile t), XOR-swizzled LDS image
//    (slot = chunk ^ ((row >> 1) & 7), applied on the per-lane SOURCE address because the
//    DMA writes lane-linearly; rule 21) which makes every ds_read_b128 lane group hit 16
//    distinct bank slots; bijective XCD-aware tile remap (T1).
#include "bfly_common.h"

#include <algorithm>
#include <cstdio>
#include <string>
#include <vector>
#include "bfly_kernels.h"
#include "bfly_kv.h"

namespace bfly {

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Non-temporal weight policy switch (BFLY_GEMM_NT_WEIGHTS=0 disables it; A/B measurements).
__constant__ int g_tile_w_nt = 1;
typedef __attribute__((address_space(1))) void* gbl_ptr_t;

// ---------------------------------------------------------------------------------------
// Epilogue helpers
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ void store_out(bf16* out, long ldo, int m, int n, float v) {
  out[(long)m * ldo + n] = f2bf(v);
}

// EPI_GLU: the constants behind the N bias values, and the activation of a (gate, up) pair.
struct GluPar {
  float limit, alpha, offset;
};
__device__ __forceinline__ GluPar glu_par(const bf16* bias, int N) {
  const float* f = reinterpret_cast<const float*>(bias + N);
  return GluPar{f[0], f[1], f[2]};
}
__device__ __forceinline__ float glu_clamped(float g, float u, const GluPar& p) {
  g = fminf(g, p.limit);
  u = fminf(fmaxf(u, -p.limit), p.limit);
  return glu_gate(g, p.alpha, __expf(-p.alpha * g)) * (u + p.offset);
}

// Four consecutive output columns of one row (the tile / decode-ring accumulators hold 4
// consecutive n per lane: W is their MFMA A operand). 8-B store when the row start allows it.
__device__ __forceinline__ void store_out4(bf16* out, long ldo, int m, int n, f32x4 v, bool vec) {
  bf16* p = out + (long)m * ldo + n;
  if (vec) {
    bf16x4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = f2bf(v[r]);
    *reinterpret_cast<bf16x4*>(p) = o;
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] = f2bf(v[r]);
  }
}

// Split-K partial slabs: 16 B per lane through a buffer descriptor, plain (write-back) stores.
// Measured and dropped: write-through (`sc1`) slab stores, meant to spare the consumer the
// write-back of MBs of dirty f32 lines (MI355X_MICROARCH.md 'boundary'), made the whole decode
// step SLOWER: Llama-3-70B 30.28-30.32 vs 29.99-30.02 ms, Llama-3-8B 5.58 vs 5.49 ms
// (profiles/r2_slab_writethrough_ab.log).

__device__ __forceinline__ __amdgpu_buffer_rsrc_t slab_rsrc(float* base, long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0,
                                           (int)(bytes < 0x7fffffffL ? bytes : 0x7fffffffL), 0x00020000);
}

__device__ __forceinline__ void store_slab4(__amdgpu_buffer_rsrc_t r, int off, f32x4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, 0, 0);
}

// Reduce split-K partial slabs [SK][M][N] (f32) and apply the epilogue.
__global__ void gemm_splitk_reduce_kernel(const float* __restrict__ part, int SK, int M, int N,
                                          int epi, const bf16* __restrict__ bias,
                                          bf16* __restrict__ out, long ldo) {
  const bool halves = epi == EPI_SILU || epi == EPI_GLU;
  const int nout = halves ? N / 2 : N;
  const long total = (long)M * nout;
  const long slab = (long)M * N;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total;
       e += (long)gridDim.x * blockDim.x) {
    const int m = (int)(e / nout), f = (int)(e % nout);
    if (halves) {
      const int g = f >> 4, w = f & 15;
      const long gi = (long)m * N + g * 32 + w, ui = gi + 16;
      float gs = 0.f, us = 0.f;
      for (int s = 0; s < SK; ++s) {
        gs += part[s * slab + gi];
        us += part[s * slab + ui];
      }
      if (epi == EPI_GLU)
        store_out(out, ldo, m, f, glu_clamped(gs + bf2f(bias[g * 32 + w]), us + bf2f(bias[g * 32 + w + 16]), glu_par(bias, N)));
      else
        store_out(out, ldo, m, f, silu(gs) * us);
    } else {
      const long i = (long)m * N + f;
      float acc = 0.f;
      for (int s = 0; s < SK; ++s) acc += part[s * slab + i];
      if (epi == EPI_BIAS) acc += bf2f(bias[f]);
      if (epi == EPI_RELU2) acc = fmaxf(acc, 0.f) * fmaxf(acc, 0.f);
      store_out(out, ldo, m, f, acc);
    }
  }
}

// Workspace head: kCounterBytes reserved ahead of the split-K slabs (the slab offset every
// consumer of deferred slabs uses, gemm_slab_offset_floats). Measured and removed: an in-kernel
// "last arriver reduces" fixup on these words; it only paid when sk x slab bytes per tile were
// a few tens of KB, and the decode plans write 256 KB per tile.
constexpr int kSplitCounters = 16384;
constexpr size_t kCounterBytes = kSplitCounters * sizeof(int);

// ---------------------------------------------------------------------------------------
// Skinny (decode) GEMM
// ---------------------------------------------------------------------------------------
constexpr int kSkThreads = 256;

template <int MT, int NT>
__device__ __forceinline__ void skinny_load(const bf16* __restrict__ W, const bf16* __restrict__ X,
                                            long ldw, long ldx, int n0, int kc, int lane, int M,
                                            bf16x8 (&a)[NT][4], bf16x8 (&b)[MT][4]) {
  // physical k of (lane group g, sub-step s, element j) = 32 s + 8 g + j: in each load
  // instruction the 4 lane groups of a row read 64 contiguous bytes.
  const int g = lane >> 4, r = lane & 15;
  const long kofs = (long)kc * 128 + 8 * g;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const bf16* p = W + (long)(n0 + 16 * t + r) * ldw + kofs;
#pragma unroll
    for (int s = 0; s < 4; ++s) a[t][s] = ld_nt(reinterpret_cast<const bf16x8*>(p + 32 * s));
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    int m = 16 * mt + r;
    m = m < M ? m : M - 1;
    const bf16* p = X + (long)m * ldx + kofs;
#pragma unroll
    for (int s = 0; s < 4; ++s) b[mt][s] = *reinterpret_cast<const bf16x8*>(p + 32 * s);
  }
}

template <int MT, int NT>
__device__ __forceinline__ void skinny_mma(const bf16x8 (&a)[NT][4], const bf16x8 (&b)[MT][4],
                                           f32x4 (&acc)[NT][MT]) {
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[t][mt] = mfma16(a[t][s], b[mt][s], acc[t][mt]);
}

// WK = waves of a workgroup that split K (their partials are summed through LDS); the other
// 4 / WK waves split N and share the same K range (their X fragments hit the same L1 lines).
template <int MT, int NT, int WK>
__global__ void __launch_bounds__(kSkThreads)
gemm_skinny_kernel(const bf16* __restrict__ X, long ldx, const bf16* __restrict__ W, long ldw,
                   int M, int N, int K, int epi, const bf16* __restrict__ bias,
                   bf16* __restrict__ out, long ldo, float* __restrict__ part) {
  constexpr int WN = 4 / WK;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int wk = wid % WK, wn = wid / WK;
  const int nb0 = blockIdx.x * 16 * NT * WN;
  const int n0 = nb0 + wn * 16 * NT;
  const int nchunks = K / 128;
  const int S = gridDim.y * WK;
  const int s_idx = blockIdx.y * WK + wk;
  const int c0 = (int)(((long)nchunks * s_idx) / S), c1 = (int)(((long)nchunks * (s_idx + 1)) / S);

  f32x4 acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

  bf16x8 a0[NT][4], b0[MT][4], a1[NT][4], b1[MT][4];
  int c = c0;
  if (c < c1) skinny_load<MT, NT>(W, X, ldw, ldx, n0, c, lane, M, a0, b0);
  // Two named register sets (runtime-indexed arrays would go to scratch: rule 20).
  while (c < c1) {
    if (c + 1 < c1) skinny_load<MT, NT>(W, X, ldw, ldx, n0, c + 1, lane, M, a1, b1);
    skinny_mma<MT, NT>(a0, b0, acc);
    ++c;
    if (c >= c1) break;
    if (c + 1 < c1) skinny_load<MT, NT>(W, X, ldw, ldx, n0, c + 1, lane, M, a0, b0);
    skinny_mma<MT, NT>(a1, b1, acc);
    ++c;
  }

  // Cross-wave reduction through LDS: red[wave][t][mt][i][lane], summed over the WK waves.
  constexpr int E = NT * MT * 4 * 64;
  __shared__ float red[4 * E];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wid * E + ((t * MT + mt) * 4 + i) * 64 + lane] = acc[t][mt][i];
  __syncthreads();

  const bool silu_epi = epi == EPI_SILU || epi == EPI_GLU;
  for (int idx = threadIdx.x; idx < WN * E; idx += kSkThreads) {
    const int vn = idx / E, e = idx % E;
    const int l = e & 63, i = (e >> 6) & 3, tm = e >> 8;
    const int t = tm / MT, mt = tm % MT;
    const int m = 16 * mt + (l & 15);
    if (m >= M) continue;
    const int nw0 = nb0 + vn * 16 * NT;
    const int n = nw0 + 16 * t + (l >> 4) * 4 + i;
    float v = 0.f;
#pragma unroll
    for (int k = 0; k < WK; ++k) v += red[(vn * WK + k) * E + e];
    if (part) {
      part[(long)blockIdx.y * M * N + (long)m * N + n] = v;
    } else if (silu_epi) {
      if (t & 1) continue;  // the gate tile's thread combines with its up partner
      const int eu = e + MT * 4 * 64;  // same (mt, i, lane), tile t + 1
      float u = 0.f;
#pragma unroll
      for (int k = 0; k < WK; ++k) u += red[(vn * WK + k) * E + eu];
      const int f = nw0 / 2 + 16 * (t / 2) + (l >> 4) * 4 + i;
      if (epi == EPI_GLU)
        store_out(out, ldo, m, f, glu_clamped(v + bf2f(bias[n]), u + bf2f(bias[n + 16]), glu_par(bias, N)));
      else
        store_out(out, ldo, m, f, silu(v) * u);
    } else {
      store_out(out, ldo, m, n, epi == EPI_BIAS ? v + bf2f(bias[n]) : epi == EPI_RELU2 ? fmaxf(v, 0.f) * fmaxf(v, 0.f) : v);
    }
  }
}

// ---------------------------------------------------------------------------------------
// Streamed product of few rows (kind 8)
// ---------------------------------------------------------------------------------------
// Workgroup = RB NT columns and all of K: NW waves take chunks of K in turn (chunk c: wave c % NW), straight into MFMA operands with
// U chunks in flight, and sum their parts in LDS: nothing staged, no partial sums in memory, no launch behind it.
// FOLD > 1 (up to RB = 16 / FOLD rows of X): the operands' 16 rows hold RB rows of FOLD neighbouring pieces of K, and the sum of the
// FOLD diagonal blocks is the product. A compute unit takes in 26 KB of weights a microsecond wherever they come from, which is what
// memory gives 256 of them together, so time goes by the unit with the most rows: folded tiles deal them out in fours and
// eights. 16-row tiles (gemm_skinny_kernel: 32 of them a workgroup) leave most units idle on narrow results and a last round nearly
// empty on others, and split products pay for their sums. One row, us, weights from memory: 1024 x 1024 5.0 -> 2.8, 2048 x 2048 7.9 ->
// 4.3, 4096 x 4096 9.3 -> 7.8, 6144 x 4096 14.5 -> 10.3, 8320 x 2048 13.4 -> 8.1, 28672 x 4096 41.5 -> 35.7 (6.6 TB/s), 128256 x
// 4096 172 -> 143; eight rows: 2048 x 2048 7.3 -> 4.6, 3072 x 2048 9.3 -> 6.0.
template <int MT, int NT, int U, int FOLD, bool LAST>
__device__ __forceinline__ void stream_step(f32x4 (&acc)[NT][MT], const bf16* const (&w)[NT], const bf16* const (&x)[MT], int c, int nw,
                                            long ktile, int left) {
  bf16x8 a[U][NT][2], b[U][MT][2];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (LAST && u >= left) break;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        a[u][t][h] = ld_nt(reinterpret_cast<const bf16x8*>(w[t] + (FOLD * (c + u * nw) + FOLD / 2 * h) * ktile + (FOLD == 1 ? 32 * h : 0)));
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (LAST && u >= left) break;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < MT; ++t)
        b[u][t][h] = *reinterpret_cast<const bf16x8*>(x[t] + 64L * FOLD * (c + u * nw) + 32 * FOLD * h);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (LAST && u >= left) break;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[t][m] = mfma16(a[u][t][h], b[u][m][h], acc[t][m]);
  }
}

// Element k of a weight row: k / 64 * ktile + k % 64, with ktile = 64 in rows of ldw, or (packed: [N / 256][K / 64][256][64]) ldw = 64 and
// ktile = 256 * 64. (For rows alone, with constants in its place, the loads are issued closer together: one sequence of 8B 909 -> 916 us a step.)
template <int MT, int NT, int NW, int U, int FOLD>
__global__ void __launch_bounds__(64 * NW)
gemm_stream_kernel(const bf16* __restrict__ X, long ldx, const bf16* __restrict__ W, long ldw, long ktile, int M, int N, int K, int epi,
                   const bf16* __restrict__ bias, bf16* __restrict__ out, long ldo) {
  static_assert(MT == 1 || FOLD == 1, "folded tiles hold one row tile");
  constexpr int RB = 16 / FOLD, KC = 64 * FOLD;
  __shared__ f32x4 parts[NW * NT * MT * 64];
  // (the wave as a scalar: matrix products run whatever lanes are masked off, so the last step has to branch around them)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int chunks = K / KC, r = lane & 15, ko = 8 * (lane >> 4) + 32 * (r / RB), tile0 = (int)blockIdx.x * NT;
  const bool halves = epi == EPI_SILU || epi == EPI_GLU;
  // weight row of a tile's row i; with gate and up halves the tile's first half are gate rows, the other their up rows
  const auto wrow = [&](int t, int i) {
    if (!halves) return (tile0 + t) * RB + i;
    const int f = (tile0 + t) * (RB / 2) + i % (RB / 2);
    return f + (f & ~15) + (i >= RB / 2 ? 16 : 0);
  };
  const bf16 *w[NT], *x[MT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int n = wrow(t, r % RB);
    w[t] = W + (ktile == 64 ? n * ldw : (long)(n >> 8) * 256 * K + (n & 255) * ldw) + ko / 64 * ktile + ko % 64;
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) x[t] = X + (long)min(16 * t + r % RB, M - 1) * ldx + ko;
  f32x4 acc[NT][MT] = {};
  int c = wave;
  for (; c + (U - 1) * NW < chunks; c += U * NW) stream_step<MT, NT, U, FOLD, false>(acc, w, x, c, NW, ktile, U);
  if (c < chunks) stream_step<MT, NT, U, FOLD, true>(acc, w, x, c, NW, ktile, (chunks - c + NW - 1) / NW);
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) parts[((wave * NT + t) * MT + m) * 64 + lane] = acc[t][m];
  __syncthreads();
  const bool vec = (ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0;
  constexpr int Q = RB / 4;      // groups of four rows of a tile
  for (int i = threadIdx.x; i < NT * MT * Q * RB; i += 64 * NW) {
    const int row = i % RB + RB * (i / (RB * Q) % MT), q = i / RB % Q, t = i / (RB * Q * MT);
    if (row >= M) continue;
    const auto sum = [&](int q) {      // over waves and pieces of K
      f32x4 v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < NW; ++k)
#pragma unroll
        for (int f = 0; f < FOLD; ++f) v += parts[((k * NT + t) * MT + row / 16) * 64 + 16 * (Q * f + q) + RB * f + row % RB];
      return v;
    };
    const int n = wrow(t, 4 * q);
    f32x4 v = sum(q);
    if (halves) {
      // four gates here and their ups Q / 2 groups on, or (tiles of four rows) two of each
      constexpr int C = RB == 4 ? 2 : 4;
      if (q >= (Q + 1) / 2) continue;
      const f32x4 up = RB == 4 ? f32x4{v[2], v[3], 0.f, 0.f} : sum(q + Q / 2);
      bf16* o = out + (long)row * ldo + (tile0 + t) * (RB / 2) + 4 * q;
#pragma unroll
      for (int e = 0; e < C; ++e) {
        if (epi == EPI_GLU) v[e] = glu_clamped(v[e] + bf2f(bias[n + e]), up[e] + bf2f(bias[n + 16 + e]), glu_par(bias, N));
        else v[e] = silu(v[e]) * up[e];
      }
      if constexpr (RB == 4) {
        o[0] = f2bf(v[0]);
        o[1] = f2bf(v[1]);
      } else {
        store_out4(o, 0, 0, 0, v, vec);
      }
      continue;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (epi == EPI_BIAS) v[e] += bf2f(bias[n + e]);
      if (epi == EPI_RELU2) v[e] = fmaxf(v[e], 0.f) * fmaxf(v[e], 0.f);
    }
    store_out4(out, ldo, row, n, v, vec);
  }
}

// ---------------------------------------------------------------------------------------
// LDS-tiled GEMM
// ---------------------------------------------------------------------------------------
constexpr int kTileThreads = 256;
constexpr int kBK = 64;

// Loads per wave per stage for a ROWS x 64 tile: every wave issues the same count (small
// tiles re-issue a piece another wave also loads: identical bytes to the same LDS address),
// so one compile-time `vmcnt` count is valid for every wave.
template <int ROWS>
constexpr int stage_loads() { return (ROWS / 8 + 3) / 4; }

// `nt`: stream the operand with the non-temporal policy (aux = 2) — for weights that exactly
// one workgroup reads once (decode, a single M tile): issued->landed ~18 % shorter and 5-10 %
// per decode layer on MI355X (MI355X_MICROARCH.md 'nt-weights'); never for re-read panels.
// PACKED: `src` is a weight in the K-tile-blocked layout [N/256][K/64][256][64] (pack_w256):
// a 256-row x 64-column block is 32 KiB of contiguous memory, so a 128-row stage reads 16 KiB
// in one run instead of 128 runs of 128 B one row pitch apart; `ld` then carries K.
template <int ROWS, bool GATHER = false, bool PACKED = false>
__device__ __forceinline__ void tile_stage(const bf16* __restrict__ src, long ld, int row0,
                                           int row_max, int k0, char* lds, int wid, int lane,
                                           const int* __restrict__ rows = nullptr, bool nt = false) {
  // ROWS x 64 bf16 = ROWS x 8 chunks of 16 B; one wave-instruction writes 8 rows (1 KiB).
  constexpr int kBlocks = ROWS / 8;
  constexpr int kInstr = stage_loads<ROWS>();
#pragma unroll
  for (int i = 0; i < kInstr; ++i) {
    int blk = i * 4 + wid;             // 8-row block index
    if (kBlocks % 4 != 0) blk %= kBlocks;
    const int row = blk * 8 + (lane >> 3);
    const int slot = lane & 7;
    const int chunk = slot ^ ((row >> 1) & 7);
    int gr = row0 + row;
    gr = gr < row_max ? gr : row_max - 1;
    if constexpr (GATHER) {
      if (rows) gr = rows[gr];   // grouped GEMM: row slot -> source token
    }
    const bf16* g = PACKED ? src + (((long)(gr >> 8) * (ld >> 6) + (k0 >> 6)) << 14) + (gr & 255) * 64 + chunk * 8
                           : src + (long)gr * ld + k0 + chunk * 8;
    if (nt)
      __builtin_amdgcn_global_load_lds((gbl_ptr_t)g, (lds_ptr_t)(lds + blk * 1024), 16, 0, 2);
    else
      __builtin_amdgcn_global_load_lds((gbl_ptr_t)g, (lds_ptr_t)(lds + blk * 1024), 16, 0, 0);
  }
}

template <int N>
__device__ __forceinline__ void vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ bf16x8 lds_frag(const char* lds, int row, int chunk) {
  const int slot = chunk ^ ((row >> 1) & 7);
  return *reinterpret_cast<const bf16x8*>(lds + row * 128 + slot * 16);
}

// Epilogue of the tile and decode-ring GEMMs. W is their MFMA A operand, so the accumulators
// hold C^T: acc[i][j][r] = C[m = mw + 16i + (lane&15)][n = nw + 16j + 4(lane>>4) + r] — four
// consecutive columns per lane, stored as one 16-B slab write or one 8-B bf16 write.
// `pslab`: this workgroup's split-K slab from row m0 on (nullptr: apply the epilogue).
// `rsc`: RMSNorm row scale of a consumer GEMM (RowScale, ss == nullptr: none), applied to the
// accumulators first, so split-K slabs, the bias and the SiLU all see the normalised rows.
template <int TI, int TJ>
__device__ __forceinline__ void tile_epilogue(const f32x4 (&acc)[TI][TJ], int mw, int nw, int lane,
                                              int M, int N, int epi, const bf16* __restrict__ bias,
                                              bf16* __restrict__ out, long ldo, float* __restrict__ pslab,
                                              int m0, const RowScale& rsc) {
  const int lr = lane & 15, lc = 4 * (lane >> 4);
  const auto rs = slab_rsrc(pslab, pslab ? (long)(M - m0) * N * 4 : 0);
  const bool vec = (ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0;
  float sc[TI];
#pragma unroll
  for (int i = 0; i < TI; ++i) sc[i] = 1.f;
  if (rsc.ss != nullptr) {
    // sum of the row's partial sums of squares: the 4 lanes of a row (lane >> 4) take every
    // 4th group of 4 chunks as 16-B loads, all in flight together, then two shuffles (a norm
    // norm leaves a chunk per 1024 columns, but a serial loop of dependent loads over many
    // chunks cost ~20 us per consumer GEMM); chunks % 4 != 0: one chunk per lane and step
    const int q = lane >> 4, nc = rsc.chunks;
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      const int m = min(mw + 16 * i + lr, M - 1);
      const float* sp = rsc.ss + (long)m * nc;
      float t = 0.f;
      if ((nc & 3) == 0) {
#pragma unroll 4
        for (int c = 4 * q; c < nc; c += 16) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(sp + c);
          t += (v[0] + v[1]) + (v[2] + v[3]);
        }
      } else {
        for (int c = q; c < nc; c += 4) t += sp[c];
      }
      t += __shfl_xor(t, 16, 64);
      t += __shfl_xor(t, 32, 64);
      sc[i] = rsqrtf(t * rsc.inv_dim + rsc.eps);
    }
  }
#pragma unroll
  for (int i = 0; i < TI; ++i) {
    const int m = mw + 16 * i + lr;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      const int n = nw + 16 * j + lc;
      if (pslab) {
        store_slab4(rs, ((m - m0) * N + n) * 4, acc[i][j] * sc[i]);
      } else if (epi == EPI_SILU || epi == EPI_SILU_GATE || epi == EPI_GLU) {
        if constexpr (TJ % 2 == 0) {   // gate/up 16-row groups pair up inside the wave
          if (j & 1) continue;
          f32x4 h;
          if (epi == EPI_GLU) {
            const GluPar gp = glu_par(bias, N);
#pragma unroll
            for (int r = 0; r < 4; ++r)
              h[r] = glu_clamped(acc[i][j][r] * sc[i] + bf2f(bias[n + r]), acc[i][j + 1][r] * sc[i] + bf2f(bias[n + 16 + r]), gp);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) h[r] = silu(acc[i][j][r] * sc[i]) * (acc[i][j + 1][r] * sc[i]);
          }
          const int f = nw / 2 + 16 * (j / 2) + lc;
          if (epi == EPI_SILU_GATE) {   // the 4 columns share an expert (gF % 16 == 0)
            const float g = rsc.gate[(long)m * rsc.gld + rsc.ge0 + f / rsc.gF];
#pragma unroll
            for (int r = 0; r < 4; ++r) h[r] = bf2f(f2bf(h[r])) * g;
          }
          store_out4(out, ldo, m, f, h, vec);
        }
      } else {
        f32x4 v = acc[i][j] * sc[i];
        if (epi == EPI_BIAS) {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] += bf2f(bias[n + r]);
        }
        if (epi == EPI_RELU2) {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = fmaxf(v[r], 0.f) * fmaxf(v[r], 0.f);
        }
        store_out4(out, ldo, m, n, v, vec);
      }
    }
  }
}

// STAGES-deep glds pipeline: K-tiles kt+1 .. kt+STAGES-1 stay in flight (LDS-DMA) while the
// MFMAs consume tile kt. Each iteration waits with a COUNTED vmcnt (only tile kt must have
// landed) and a raw s_barrier (a __syncthreads() would drain every in-flight DMA:
// cdna_hip_programming.md §5 "Pipelining across barriers"); the buffer refilled in an
// iteration is the one every wave finished reading in the previous iteration (WAR safe).
//
// GROUPED (MoE expert GEMM, K13): blockIdx.x indexes a device-built tile list
// gtiles[i] = {expert, first row slot, end row slot} (count in *gcount; excess workgroups
// exit), blockIdx.z the N tile; the expert selects W + expert * w_estride and A rows are
// gathered through grows[slot] (nullptr: slots are rows). Output rows are row slots.
template <int BM, int BN, int WMW, int STAGES, bool GROUPED = false, bool PACKW = false>
__global__ void __launch_bounds__(kTileThreads)
gemm_tile_kernel(const bf16* __restrict__ X, long ldx, const bf16* __restrict__ W, long ldw,
                 int M, int N, int K, int epi, const bf16* __restrict__ bias,
                 bf16* __restrict__ out, long ldo, float* __restrict__ part,
                 const int* __restrict__ grows = nullptr,
                 const int4* __restrict__ gtiles = nullptr, const int* __restrict__ gcount = nullptr,
                 long w_estride = 0, RowScale rsc = RowScale{nullptr, 0, 0.f, 0.f}) {
  constexpr int WNW = 4 / WMW;                // waves along M x waves along N
  constexpr int WM = BM / WMW, WN = BN / WNW; // per-wave output tile
  constexpr int TI = WM / 16, TJ = WN / 16;  // MFMA tiles per wave
  constexpr int A_BYTES = BM * kBK * 2, B_BYTES = BN * kBK * 2;
  constexpr int LPW = stage_loads<BM>() + stage_loads<BN>();  // glds per wave per stage
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int STAGE_BYTES = A_BYTES + B_BYTES;  // one buffer = [A tile | B tile]

  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int wm = wid / WNW, wn = wid % WNW;
  int tile, m0, n0, ksplit = 0;
  const int m_slab = M;             // split-K slab row stride (grouped: all row slots)
  bool single = false;              // grouped: this expert has one row tile (W read once)
  if constexpr (GROUPED) {
    if ((int)blockIdx.x >= *gcount) return;
    const int4 info = gtiles[blockIdx.x];
    W += (long)info.x * w_estride;
    m0 = info.y;
    M = info.z;                     // rows [m0, M) of the permuted slot space
    single = info.w != 0;
    n0 = blockIdx.z * BN;
    tile = 0;
  } else {
    const int mtiles = (M + BM - 1) / BM, ntiles = N / BN;
    tile = xcd_remap((int)blockIdx.x, mtiles * ntiles);
    const int tn = tile / mtiles, tm = tile % mtiles;  // consecutive tiles share a W panel
    m0 = tm * BM;
    n0 = tn * BN;
  }
  ksplit = (int)blockIdx.y;
  const int nsplit = (int)gridDim.y;

  const int ktiles = K / kBK;
  const int kt0 = (int)(((long)ktiles * ksplit) / nsplit);
  const int kt1 = (int)(((long)ktiles * (ksplit + 1)) / nsplit);
  // each W byte read by one workgroup: stream it non-temporally
  const bool w_nt = (GROUPED ? single : M <= BM) && g_tile_w_nt;

  f32x4 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) {
    if (kt0 + s < kt1) {
      char* b = smem + s * STAGE_BYTES;
      tile_stage<BM, GROUPED>(X, ldx, m0, M, (kt0 + s) * kBK, b, wid, lane, grows);
      tile_stage<BN, false, PACKW>(W, ldw, n0, N, (kt0 + s) * kBK, b + A_BYTES, wid, lane, nullptr, w_nt);
    }
  }
  int buf = 0;
  for (int kt = kt0; kt < kt1; ++kt) {
    // tiles issued after kt: min(STAGES - 2, kt1 - 1 - kt); wait until only those are pending
    const int after = min(STAGES - 2, kt1 - 1 - kt);
    if (STAGES >= 4 && after >= 2) vm_wait<(STAGES >= 4 ? 2 : 0) * LPW>();
    else if (STAGES >= 3 && after >= 1) vm_wait<LPW>();
    else vm_wait<0>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (kt + STAGES - 1 < kt1) {
      int nbuf = buf + STAGES - 1;
      if (nbuf >= STAGES) nbuf -= STAGES;
      char* nb = smem + nbuf * STAGE_BYTES;
      tile_stage<BM, GROUPED>(X, ldx, m0, M, (kt + STAGES - 1) * kBK, nb, wid, lane, grows);
      tile_stage<BN, false, PACKW>(W, ldw, n0, N, (kt + STAGES - 1) * kBK, nb + A_BYTES, wid, lane, nullptr, w_nt);
    }
    const char* As = smem + buf * STAGE_BYTES;
    const char* Bs = As + A_BYTES;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 af[TI], bfr[TJ];
#pragma unroll
      for (int i = 0; i < TI; ++i) af[i] = lds_frag(As, wm * WM + 16 * i + (lane & 15), ks * 4 + (lane >> 4));
#pragma unroll
      for (int j = 0; j < TJ; ++j) bfr[j] = lds_frag(Bs, wn * WN + 16 * j + (lane & 15), ks * 4 + (lane >> 4));
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = mfma16(bfr[j], af[i], acc[i][j]);   // C^T tile
    }
    if (++buf == STAGES) buf = 0;
  }
  tile_epilogue<TI, TJ>(acc, m0 + wm * WM, n0 + wn * WN, lane, M, N, epi, bias, out, ldo,
                        part ? part + (long)ksplit * m_slab * N + (long)m0 * N : nullptr, m0, rsc);
}

// ---------------------------------------------------------------------------------------
// Decode ring GEMM (kind 3; decode batches of 65-256 rows, e.g. TP2 replicas at 128 rows).
//
// Measured on MI355X (tools/exp_dec.py, N 57344 x K 8192): gemm_tile at BM = 128 streams
// weights at ~4.9-5.3 TB/s for ANY M (the time is flat in M: the kernel shape, not the
// arithmetic, is the limit), while 64-row tiles at two 4-wave workgroups per CU reach
// ~6.0 TB/s — but only for M <= 64 (a second row tile re-reads W through the per-CU load
// path: 3.9 TB/s at M = 128). The per-CU LDS-DMA stream scales with the number of waves
// issuing it, and X staged per K-tile competes with W for it. So this kernel:
//  * runs 8 waves per workgroup (NWM along M x NWN along N), one workgroup per CU;
//  * keeps X and W in separate LDS rings: X (L2-resident) needs 3 slots, W gets SW slots
//    (up to 160 KiB in all), so SW-1 weight K-tiles stream while the MFMAs consume tile kt;
//  * uses wide N tiles (BN up to 256: 224 makes N = 57344 exactly 256 tiles) so X is at most
//    half of the staged bytes at BM = 128.
// Issue order per iteration is W(kt+SW-1) then X(kt+2), so X(kt) is always the later of the
// two loads tile kt needs and one counted vmcnt covers both: LW + LX loads were issued after
// X(kt) in steady state; in the tail the wait is exact or conservative.
// ---------------------------------------------------------------------------------------
template <int ROWS, int NW>
constexpr int ring_loads() { return (ROWS / 8 + NW - 1) / NW; }

template <int ROWS, int NW>
__device__ __forceinline__ void ring_stage(const bf16* __restrict__ src, long ld, int row0, int row_max,
                                           int k0, char* lds, int wid, int lane, bool nt) {
  constexpr int kBlocks = ROWS / 8;   // 8-row blocks of 1 KiB; one wave-instruction each
#pragma unroll
  for (int i = 0; i < ring_loads<ROWS, NW>(); ++i) {
    int blk = i * NW + wid;
    if (kBlocks % NW != 0) blk %= kBlocks;   // surplus lanes re-load a block (same bytes)
    const int row = blk * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ ((row >> 1) & 7);
    int gr = row0 + row;
    gr = gr < row_max ? gr : row_max - 1;
    const bf16* g = src + (long)gr * ld + k0 + chunk * 8;
    if (nt)
      __builtin_amdgcn_global_load_lds((gbl_ptr_t)g, (lds_ptr_t)(lds + blk * 1024), 16, 0, 2);
    else
      __builtin_amdgcn_global_load_lds((gbl_ptr_t)g, (lds_ptr_t)(lds + blk * 1024), 16, 0, 0);
  }
}

constexpr int kDecThreads = 512;

template <int BM, int BN, int NWM, int NWN, int SW>
__global__ void __launch_bounds__(kDecThreads)
gemm_dec_kernel(const bf16* __restrict__ X, long ldx, const bf16* __restrict__ W, long ldw,
                int M, int N, int K, int epi, const bf16* __restrict__ bias,
                bf16* __restrict__ out, long ldo, float* __restrict__ part, RowScale rsc) {
  constexpr int SX = 3, NW = NWM * NWN;
  static_assert(NW * 64 <= kDecThreads && SW >= SX, "decode ring configuration");
  constexpr int WM = BM / NWM, WN = BN / NWN;   // per-wave output block
  constexpr int TI = WM / 16, TJ = WN / 16;
  static_assert(WM % 16 == 0 && WN % 16 == 0, "per-wave block must be whole MFMA tiles");
  constexpr int XB = BM * kBK * 2, WB = BN * kBK * 2;
  constexpr int LX = ring_loads<BM, NW>(), LW = ring_loads<BN, NW>();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* const xs = smem;
  char* const wsm = smem + SX * XB;

  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int wm = wid / NWN, wn = wid % NWN;
  const int mtiles = (M + BM - 1) / BM, ntiles = N / BN;
  const int tile = xcd_remap((int)blockIdx.x, mtiles * ntiles);
  const int ksplit = (int)blockIdx.y;
  const int tn = tile / mtiles, tm = tile % mtiles;
  const int m0 = tm * BM, n0 = tn * BN;
  const int nsplit = (int)gridDim.y;
  const int ktiles = K / kBK;
  const int kt0 = (int)(((long)ktiles * ksplit) / nsplit);
  const int kt1 = (int)(((long)ktiles * (ksplit + 1)) / nsplit);
  const bool w_nt = mtiles == 1 && g_tile_w_nt;   // each weight byte read by one workgroup

  f32x4 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // prologue = the issue pattern of virtual iterations kt0-SW+1 .. kt0-1: W(kt0 .. kt0+SW-2)
  // and, lagging by SW-SX, X(kt0 .. kt0+1). Slot of K-tile t: (t - kt0) mod S.
#pragma unroll
  for (int v = 0; v < SW - 1; ++v) {
    if (kt0 + v < kt1) ring_stage<BN, NW>(W, ldw, n0, N, (kt0 + v) * kBK, wsm + v * WB, wid, lane, w_nt);
    const int xv = v - (SW - SX);
    if (xv >= 0 && kt0 + xv < kt1) ring_stage<BM, NW>(X, ldx, m0, M, (kt0 + xv) * kBK, xs + xv * XB, wid, lane, false);
  }
  int xslot = 0, wslot = 0;
  for (int kt = kt0; kt < kt1; ++kt) {
    // loads issued after X(kt): iteration kt-1's W(kt+SW-2) (if any) and X(kt+1) (if any)
    if (kt + SW - 2 < kt1) vm_wait<LW + LX>();
    else if (kt + 1 < kt1) vm_wait<LX>();
    else vm_wait<0>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    // refill the slots every wave finished reading in iteration kt-1
    const int wfill = wslot == 0 ? SW - 1 : wslot - 1;
    const int xfill = xslot == 0 ? SX - 1 : xslot - 1;
    if (kt + SW - 1 < kt1) ring_stage<BN, NW>(W, ldw, n0, N, (kt + SW - 1) * kBK, wsm + wfill * WB, wid, lane, w_nt);
    if (kt + SX - 1 < kt1) ring_stage<BM, NW>(X, ldx, m0, M, (kt + SX - 1) * kBK, xs + xfill * XB, wid, lane, false);
    const char* As = xs + xslot * XB;
    const char* Bs = wsm + wslot * WB;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 af[TI];
#pragma unroll
      for (int i = 0; i < TI; ++i) af[i] = lds_frag(As, wm * WM + 16 * i + (lane & 15), ks * 4 + (lane >> 4));
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const bf16x8 b = lds_frag(Bs, wn * WN + 16 * j + (lane & 15), ks * 4 + (lane >> 4));
#pragma unroll
        for (int i = 0; i < TI; ++i) acc[i][j] = mfma16(b, af[i], acc[i][j]);   // C^T tile
      }
    }
    if (++xslot == SX) xslot = 0;
    if (++wslot == SW) wslot = 0;
  }
  tile_epilogue<TI, TJ>(acc, m0 + wm * WM, n0 + wn * WN, lane, M, N, epi, bias, out, ldo,
                        part ? part + (long)ksplit * M * N + (long)m0 * N : nullptr, m0, rsc);
}

// Prefill tiles are walked in GROUP_M super-rows inside each XCD's contiguous range, so the
// 32 CUs of an XCD share X and W panels in their L2.
constexpr int kBigGroupM = 8;

// ---------------------------------------------------------------------------------------
// 8-phase big-tile GEMM (prefill): 256x256 tile, BK = 64, two K-tile LDS buffers (128 KiB),
// 8 waves (2 along M x 4 along N, 128x64 outputs each) in two groups staggered by one barrier
// (group wr = 1 starts one s_barrier later), so on every SIMD one wave runs a 16-MFMA segment
// while its partner reads fragments and issues DMA (cdna_hip_programming.md §5 "The 256²
// 8-phase template", T3+T4+T5).
//
// A K-tile is consumed in 4 phases, one C-quadrant of the wave's 128x64 block each:
//   q0: rows 0-63 x cols 0-31   reads A-lo (8 ds_read_b128) + B-lo (4)
//   q1: rows 0-63 x cols 32-63  reads B-hi (4)            (A-lo kept in registers)
//   q2: rows 64-127 x cols 32-63 reads A-hi (8)           (B-hi kept)
//   q3: rows 64-127 x cols 0-31  no reads                 (A-hi, B-lo kept)
// so each of the K-tile's four half-tiles (A-lo = rows {0-63, 128-191}, A-hi = {64-127,
// 192-255}, B-lo = cols {0-31, 64-95, ...}, B-hi = the other 32-column groups; 16 KiB each) is
// read completely in ONE phase. Every phase issues one half-tile of DMA (2 glds per wave) into
// a half that was fully read (and retired by lgkmcnt(0) before a barrier every reader passed)
// in an earlier phase: K-tile k's halves go out at phases 4(k-2)+{2,3,4,5} (A-lo, B-lo, B-hi,
// A-hi), i.e. one phase after the same half of K-tile k-2 was read. The counted wait is in
// phase 4k only (the K-tile's last phase): vmcnt(6) leaves the 3 half-tiles issued after A-hi(k)
// in flight and retires all of K-tile k, which is read from phase 4k+1 on (one phase after the
// wait, behind a barrier both groups pass: the template's RAW rule). Raw s_barrier only: a
// __syncthreads() would drain the DMA in flight (§5 "Pipelining across barriers").
// The fragment schedule on top of that (the prefill kernel for every M > 256, plan kind 4):
//  * early LDS release: A-lo is the one half restaged one phase after its read, so only its
//    reads must retire before a phase's barrier (lgkmcnt(4) after A first, B last); every
//    other read completes inside the wave's own MFMA segment;
//  * lookahead: the A-lo fragments of K-tile k+1 are read in phase q3 of K-tile k (whose read
//    segment is otherwise empty), and its B-lo fragments right behind q3's MFMAs (b_lo(k)'s
//    last use), so q0 reads nothing and no read latency sits behind a barrier. A counted wait
//    in q2 retires this wave's A-lo / B-lo(k+1) DMA, and the barrier ending q2 of group 0 (=
//    the one starting q2's MFMAs of group 1) is passed by both groups before either reads;
//  * buffer-descriptor staging: the tile's A / B rows start at an SGPR base (the descriptor),
//    the K offset and the hi-half row shift ride in the scalar soffset (A-hi = A-lo + 64 rows,
//    B-hi = B-lo + 32 rows: the same XOR pattern, which depends on row bits 1-3 only), each lane
//    keeps 4 constant byte offsets, and A rows past M read as zeros instead of a clamped
//    re-read (VALU per K-tile 49 -> 24).
// 1.39-1.40 PF at M = 8192 on the 70B projections, +4.6-5.2 % over the schedule without the
// lookahead and descriptors (profiles/r4_gemm_prefill_la.log, r4_gemm_prefill_lb.log).
// Measured and dropped (profiles/r3_gemm_prefill_pmc.md, r4_gemm_prefill_{bal,lh}.log):
//  - the round-2 5-slot BK-32 ring kernel (8 waves, one 16x16x32 K-step per barrier):
//    2-7 % slower at M = 8192, within -3..+32 % at M = 256/512;
//  - one wave per SIMD, 4 waves x 128x128 per wave (hipBLASLt's shape: MT256x256x64, 256
//    threads): 32x32x16 with a 4/5-slot BK-32 glds ring 1.07-1.10 PF; 16x16x32 with buffer
//    loads to LDS and the second MFMA half deferred behind the next K-tile's reads 1.13-1.23
//    PF; the same with BK 64 in a 2-slot ring 1.00-1.12 PF (WAIT_ANY x3: one K-tile of lead
//    does not cover HBM latency). All at 49-52 % MFMA-busy cycles against hipBLASLt's 87 %;
//  - the 24 reads spread 6 / 6 / 6 / 6 over the four read segments (0.7-1.5 % slower), A-hi
//    read in q0's empty segment (1.5-2.8 % slower), and the plain / early-release-only
//    schedules (plan mt 0-3 of round 4).
// ---------------------------------------------------------------------------------------
constexpr int kB8Threads = 512;
constexpr int kB8LdsBytes = 2 * 2 * 256 * 128;   // 2 buffers x (A, B) x 256 rows x 128 B

// LDS row-block (8 rows x 128 B = 1 KiB) of the h-th DMA instruction of half-tile `half`
// (0 A-lo / 1 B-lo / 2 B-hi / 3 A-hi; h in 0..15: instruction 2*wave + {0,1}).
__device__ __forceinline__ int b8_block(int half, int h) {
  if (half == 0 || half == 3) {            // A: rows {0-63,128-191} (lo) or {64-127,192-255} (hi)
    const int base = half == 0 ? 0 : 8;
    return (h < 8 ? base + h : 16 + base + (h - 8));
  }
  // B: 32-row groups g (0..3) at rows 64g + (hi ? 32 : 0); 4 blocks per group
  const int g = h >> 2, b = h & 3;
  return g * 8 + (half == 2 ? 4 : 0) + b;
}

struct B8Dma {
  int a[2], b[2];
};

__device__ __forceinline__ B8Dma b8_dma_offsets(long ldx, long ldw, int wid, int lane) {
  B8Dma d;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int ra = b8_block(0, 2 * wid + i) * 8 + (lane >> 3);
    const int rb = b8_block(1, 2 * wid + i) * 8 + (lane >> 3);
    d.a[i] = (int)((ra * ldx + (((lane & 7) ^ ((ra >> 1) & 7)) * 8)) * 2);
    d.b[i] = (int)((rb * ldw + (((lane & 7) ^ ((rb >> 1) & 7)) * 8)) * 2);
  }
  return d;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t b8_rsrc(const bf16* base, long rows, long ld) {
  const long bytes = rows * ld * 2;
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)(bytes < 0x7fffffffL ? bytes : 0x7fffffffL),
                                           0x00020000);
}

__device__ __forceinline__ void b8_stage_buf(__amdgpu_buffer_rsrc_t ra, __amdgpu_buffer_rsrc_t rb, long ldx,
                                             long ldw, int k0, char* buf, int half, int wid, const B8Dma& d) {
  const bool isA = half == 0 || half == 3;
  char* lds = buf + (isA ? 0 : 256 * 128);
  const int shift = half == 3 ? (int)(64 * ldx * 2) : half == 2 ? (int)(32 * ldw * 2) : 0;
  const int soff = k0 * 2 + shift;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int blk = b8_block(half, 2 * wid + i);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(isA ? ra : rb, (lds_ptr_t)(lds + blk * 1024), 16, isA ? d.a[i] : d.b[i],
                                             soff, 0, 0);
  }
}

// GROUPED (MoE expert GEMM at prefill scale, K13): the M tiles are the entries of a device-built
// tile list gtiles[i] = {expert, first row slot, end row slot, -} (count in *gcount, up to
// `M` = the list's capacity; excess workgroups exit): the expert selects W + expert *
// w_estride, and the A rows of slot s are the token rows grows[s] (nullptr: slot s itself),
// gathered by per-lane LDS-DMA addresses (rows past the tile's end re-read its last row; their
// outputs are not stored). Output rows are slots. Consecutive list entries are mostly tiles of
// one expert, so the GROUP_M walk shares the expert's weight panels in an XCD's L2.
__device__ __forceinline__ void b8_stage_gather(const bf16* const (&arow)[4], int k0, char* buf, int half, int wid) {
  const int base = half == 3 ? 2 : 0;   // A-lo: pointers 0, 1; A-hi: 2, 3
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int blk = b8_block(half, 2 * wid + i);
    __builtin_amdgcn_global_load_lds((gbl_ptr_t)(arow[base + i] + k0), (lds_ptr_t)(buf + blk * 1024), 16, 0, 0);
  }
}

template <bool GROUPED = false>
__global__ void __launch_bounds__(kB8Threads)
gemm_big8_kernel(const bf16* __restrict__ X, long ldx, const bf16* __restrict__ W, long ldw,
                 int M, int N, int K, int epi, const bf16* __restrict__ bias,
                 bf16* __restrict__ out, long ldo, float* __restrict__ part,
                 const int* __restrict__ grows = nullptr, const int4* __restrict__ gtiles = nullptr,
                 const int* __restrict__ gcount = nullptr, long w_estride = 0) {
  constexpr int BM = 256, BN = 256;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int wr = wid >> 2, wc = wid & 3;
  const int mtiles = (M + BM - 1) / BM, ntiles = N / BN;   // GROUPED: M = tile-list capacity x BM
  const int t = xcd_remap(blockIdx.x, mtiles * ntiles);
  const int per_group = kBigGroupM * ntiles;
  const int grp = t / per_group, first_m = grp * kBigGroupM;
  const int gsize = min(mtiles - first_m, kBigGroupM);
  int m0 = (first_m + (t % per_group) % gsize) * BM;
  const int n0 = ((t % per_group) / gsize) * BN;
  const bf16* arow[4] = {};
  if constexpr (GROUPED) {
    const int ti = m0 / BM;
    if (ti >= *gcount) return;
    const int4 info = gtiles[ti];
    W += (long)info.x * w_estride;
    m0 = info.y;
    M = info.z;                    // rows [m0, M) of the slot space
    // this lane's A rows: the 4 row blocks it DMAs (A-lo: b8_block(0, 2 wid + i), A-hi: (3, ...))
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = b8_block(i < 2 ? 0 : 3, 2 * wid + (i & 1)) * 8 + (lane >> 3);
      const int chunk = (lane & 7) ^ ((row >> 1) & 7);
      int slot = m0 + row;
      slot = slot < M ? slot : M - 1;
      const long src = grows != nullptr ? grows[slot] : slot;
      arow[i] = X + src * ldx + chunk * 8;
    }
  }
  const int ktiles = K / 64;
  const int kt0 = (int)(((long)ktiles * blockIdx.y) / gridDim.y);
  const int kt1 = (int)(((long)ktiles * (blockIdx.y + 1)) / gridDim.y);
  const int nk = kt1 - kt0;   // >= 2 (host check)

  f32x4 acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto bufp = [&](int k) -> char* { return smem + (k & 1) * (2 * 256 * 128); };
  // descriptors at the tile's first A / B row (SGPRs), 4 per-lane offsets
  const auto rsa = b8_rsrc(X + (long)m0 * ldx, M - m0, ldx);
  const auto rsb = b8_rsrc(W + (long)n0 * ldw, N - n0, ldw);
  const B8Dma dma = b8_dma_offsets(ldx, ldw, wid, lane);
  auto stage = [&](int k, int half) {
    if (GROUPED && (half == 0 || half == 3))
      b8_stage_gather(arow, (kt0 + k) * 64, bufp(k), half, wid);
    else
      b8_stage_buf(rsa, rsb, ldx, ldw, (kt0 + k) * 64, bufp(k), half, wid, dma);
  };
  // prologue: all of K-tile 0, then A-lo, B-lo, B-hi of K-tile 1 (the load stream's order)
  stage(0, 0); stage(0, 1); stage(0, 2); stage(0, 3);
  stage(1, 0); stage(1, 1); stage(1, 2);
  vm_wait<6>();                          // K-tile 0 landed (this wave's part)
  __builtin_amdgcn_s_barrier();          // every wave's part
  if (wr == 1) __builtin_amdgcn_s_barrier();

  const int ar = wr * 128 + (lane & 15);  // A fragment row of block i: ar + 16 i
  const int bc = wc * 64 + (lane & 15);   // B fragment row (output column) of block j
  bf16x8 a_lo[4][2], a_hi[4][2], b_lo[2][2], b_hi[2][2];
  auto read_a_lo = [&](const char* As) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) a_lo[i][ks] = lds_frag(As, ar + 16 * i, ks * 4 + (lane >> 4));
  };
  auto read_b_lo = [&](const char* Bs) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) b_lo[j][ks] = lds_frag(Bs, bc + 16 * j, ks * 4 + (lane >> 4));
  };
  read_a_lo(bufp(0));
  read_b_lo(bufp(0) + 256 * 128);
  for (int k = 0; k < nk; ++k) {
    const char* As = bufp(k);
    const char* Bs = As + 256 * 128;
    const bool more = k + 1 < nk, more2 = k + 2 < nk;
    // ---- q0: (A-lo, B-lo read ahead); DMA A-hi(k+1)
    if (more) stage(k + 1, 3);
    asm volatile("s_waitcnt lgkmcnt(4)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma16(b_lo[j][ks], a_lo[i][ks], acc[i][j]);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_s_barrier();
    // ---- q1: read B-hi; DMA A-lo(k+2) (A-lo(k) was read in q3 of k-1)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) b_hi[j][ks] = lds_frag(Bs, bc + 32 + 16 * j, ks * 4 + (lane >> 4));
    if (more2) stage(k + 2, 0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][2 + j] = mfma16(b_hi[j][ks], a_lo[i][ks], acc[i][2 + j]);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_s_barrier();
    // ---- q2: read A-hi; DMA B-lo(k+2)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) a_hi[i][ks] = lds_frag(As, ar + 64 + 16 * i, ks * 4 + (lane >> 4));
    if (more2) stage(k + 2, 1);
    // this wave's A-lo / B-lo(k+1) DMA retired (left in flight: B-hi, A-hi(k+1) and, while
    // K-tile k+2 exists, A-lo / B-lo(k+2))
    if (more2) vm_wait<8>();
    else if (more) vm_wait<4>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[4 + i][2 + j] = mfma16(b_hi[j][ks], a_hi[i][ks], acc[4 + i][2 + j]);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_s_barrier();
    // ---- q3: read A-lo(k+1); DMA B-hi(k+2); retire K-tile k+1
    // a_lo(k) is dead since q1; q3's MFMAs use a_hi / b_lo. Unconditional (past the last K-tile
    // it reads the other buffer's stale image, never used), and pinned here: under a branch the
    // scheduler sank the reads behind q3's MFMAs and barrier, i.e. back into q0
    read_a_lo(bufp(k + 1));
    __builtin_amdgcn_sched_barrier(0);
    if (more2) stage(k + 2, 2);
    if (more2) vm_wait<6>();   // A-hi(k+1) and older landed; A-lo/B-lo/B-hi(k+2) fly
    else vm_wait<0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[4 + i][j] = mfma16(b_lo[j][ks], a_hi[i][ks], acc[4 + i][j]);
    __builtin_amdgcn_s_setprio(0);
    // B-lo(k+1) behind q3's MFMAs, so its latency is spent in the barrier and q0's read segment
    // instead of after q0's barrier (its DMA retired with q2's wait)
    read_b_lo(bufp(k + 1) + 256 * 128);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
  }
  if (wr == 0) __builtin_amdgcn_s_barrier();   // re-align the groups' barrier counts
  tile_epilogue<8, 4>(acc, m0 + wr * 128, n0 + wc * 64, lane, M, N, epi, bias, out, ldo,
                      part ? part + (long)blockIdx.y * M * N + (long)m0 * N : nullptr, m0,
                      RowScale{nullptr, 0, 0.f, 0.f});
}

// ---------------------------------------------------------------------------------------
// One wave per SIMD, 256x256 tile (plan kind 6, "big4"): 4 waves in 2 x 2, each owning a 128 x
// 128 output block (8 x 8 mfma_16x16x32 accumulators, 256 registers: the AGPR half of the
// 512-register file a lone wave gets). Per K-tile (BK = 64) a wave reads 32 fragments (16 KiB
// of A and B rows) for 128 MFMAs: a third fewer LDS bytes per FLOP than big8's 128 x 64 wave
// tile, whose fragment reads plus DMA writes fill the LDS port.
// LDS (160 KiB, all of it): LDS-DMA rings of whole K-tile halves, 3 slots of A (activation
// rows) and 2 of B (weight rows), 32 KiB each: no staging registers (those pushed the allocator
// into moving accumulators every K-tile). A gets the deeper ring: an XCD's 32 resident tiles
// are 8 row tiles x 4 column tiles (GROUP_M walk), so A misses its L2 twice as often as B.
// One barrier per K-tile, between its two k-steps (ks):
//   ks 0 of K-tile t: MFMAs on the ks-0 fragments; read the ks-1 fragments of t; DMA A(t+2)
//     into A slot (t+2) % 3, which K-tile t-1 left before the previous barrier;
//   own DMA of A(t+1), B(t+1) retired (vmcnt 8: A(t+2) flies), lgkmcnt(0), s_barrier;
//   ks 1: MFMAs on the ks-1 fragments; read the ks-0 fragments of t+1; DMA B(t+2) into B slot
//     t % 2 — K-tile t's last reads (its ks-1 fragments) are before this barrier in every wave.
// Source order is the schedule: each k-step is 16 slots of {4 MFMAs, 1 fragment read, a DMA
// every other slot} fenced by sched_barrier(0) (cdna_hip_programming.md T19: left alone, the
// scheduler clusters the memory operations, and a lone wave has nothing to hide the stall
// behind). A lane's fragments of one (slot, ks) share one address VGPR (immediate offsets: 4
// VALU per K-tile). No guards: past the last K-tile the DMA takes the next tile's first ones, or
// this tile's once more for nobody (a guard made hipcc wait vmcnt(0) per slot: 3.5x slower).
// Measured (profiles/r5_gemm_big4/): 1.52-1.55 PF at M = 8192 on the Llama-3-70B projections
// against 1.39-1.47 for gemm_big8_kernel and 1.53-1.64 for hipBLASLt on the same box. Steps that
// got it there from 1.0 PF: LDS-DMA rings instead of register staging (no accumulator moves),
// one loop with no peeled iterations, one fragment read per slot (not two), the loop rotated to
// end on the barrier, A's DMA moved into ks 0, immediate-offset fragment addresses.
// ---------------------------------------------------------------------------------------
constexpr int kB4Threads = 256;
constexpr int kB4Parts = -2;                       // in place of an epilogue: the sums of a part of K, in f32
constexpr int kB4Slot = 256 * 128;                 // one operand half of a K-tile: 32 KiB
constexpr int kB4LdsBytes = 5 * kB4Slot;           // A slots 0-2, B slots 3-4: 160 KiB

__device__ __forceinline__ void b4_dma(__amdgpu_buffer_rsrc_t r, char* lds, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)lds, 16, voff, soff, 0, 0);
}

// GROUPED 1 (MoE expert GEMM at prefill scale): as gemm_big8_kernel<true> — M tiles are the
// entries of the device tile list {expert, first row slot, end slot}, W is offset by the expert,
// A rows are gathered through grows[slot] by per-lane LDS-DMA offsets from X (rows past the
// tile's end re-read its last row; their outputs are not stored).
// GROUPED 2 / 3 (ExpertArgs, the score-routed experts of the heterogeneous stacks): the up / gate-and-up
// projection and the down projection over the row groups of moe_sort. A gate's 64 rows and the up rows of the same
// 64 columns are the two halves of a wave's 128 columns (the weight DMA picks the rows: the stored panels stay
// [gate | up]), so the clamped GLU runs on a lane's own accumulators; an expert that runs on (score x row) scales
// the accumulators by the score instead of rounding scaled rows. The down projection leaves f32 rows at their
// (token, choice) pair. Measured beside the smaller tiles: moe_tile_rows.
// E: the epilogue, or kB4Parts, in instances of their own because the branches of the others cost each of them up to 3 us, and
// with every epilogue added more (8192 x 57344 x 8192 SwiGLU 5050 us with four of them, 5066 with five, 5028 alone); two that share
// one also spill. EPI_BIAS reads the columns' values once for all rows (row by row, each load waited for by the only wave of its
// SIMD, they took 13 to 50 us of a product).
// The results leave through LDS: an MFMA leaves a lane 4 columns of a row, so that a store straight from the accumulators writes 16 rows
// of 32 bytes (64 in f32), and the last level's cache reads a line it does not hold before it takes a part of it. A wave puts its
// rows into its own piece of the rings (free behind the last K-tile) and stores them as whole lines, 16 bytes a lane. Before and
// after, us: 8192 x 8192 x 512 88 and 76, x 2048 214 and 204, 8192 x 16384 x 2048 (268 MB of results) 580 and 410, with SwiGLU 407
// and 390, 6184 x 8448 x 2048 184 and 170, 937 x 6144 x 4096 53 and 50. Non-temporal stores from there: 8192 x 8192 x 512 75 -> 86,
// the others level.
typedef unsigned u32x4_b4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x8_b4 __attribute__((ext_vector_type(8)));

// A wave's piece is 8 KB. Rows of RB bytes, their 16-byte chunks turned by the row so that both ways meet every bank alike.
template <int RB>
__device__ __forceinline__ int b4_place(int row, int chunk) {
  return row * RB + 16 * (chunk ^ (RB == 128 ? (row >> 1) & 7 : row & 15));
}

// What a lane holds of the piece's rows: 16 bytes at chunk lane % LPR of row lane / LPR + q RPI
template <int RB>
struct B4Rows {
  static constexpr int LPR = RB / 16, RPI = 64 / LPR;      // lanes of a row, rows of an instruction
  f32x4 v[8];
  __device__ __forceinline__ B4Rows(const char* piece, int lane) {
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = *reinterpret_cast<const f32x4*>(piece + b4_place<RB>(lane / LPR + q * RPI, lane % LPR));
  }
  // at base + row * stride bytes, rows below left: branches over the last ones would be taken 32 times. `whole`: rows that are
  // aligned to 16 bytes.
  __device__ __forceinline__ void out(__amdgpu_buffer_rsrc_t to, int lane, int row0, int left, int stride, bool whole) const {
    int off[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int r = row0 + lane / LPR + q * RPI;
      off[q] = r < left ? r * stride + 16 * (lane % LPR) : -1;      // (past every bound)
    }
    if (whole) {
#pragma unroll
      for (int q = 0; q < 8; ++q) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_b4, v[q]), to, off[q], 0, 0);
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q)
#pragma unroll
        for (int x = 0; x < 8; ++x)
          __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(u16x8_b4, v[q])[x], to, off[q] < 0 ? -1 : off[q] + 2 * x, 0, 0);
    }
  }
  // the same of bf16 rows too far apart for 32-bit offsets
  __device__ __forceinline__ void out_far(bf16* dst, long ldo, int lane, int row0, int left) const {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int r = row0 + lane / LPR + q * RPI;
      bf16* o = dst + r * ldo + 8 * (lane % LPR);
      const bf16x8 e = __builtin_bit_cast(bf16x8, v[q]);
      if (r < left)
#pragma unroll
        for (int x = 0; x < 8; ++x) o[x] = e[x];
    }
  }
};

// RI x NJ blocks of 16 x 16 results, value(i, j) a lane's four of one, as bf16 rows from dst on
template <int RI, int NJ, class Value>
__device__ __forceinline__ void b4_out(char* piece, int lane, int left, bf16* dst, long ldo, Value&& value) {
  constexpr int RB = 32 * NJ, RP = 8192 / RB / 16;      // row blocks of a piece
  const bool whole = (ldo & 7) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15) == 0;
  const auto to = __builtin_amdgcn_make_buffer_rsrc((void*)dst, (short)0, 0x7fffffff, 0x00020000);
#pragma unroll
  for (int h = 0; h < RI; h += RP) {
#pragma unroll
    for (int i = 0; i < RP; ++i) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const f32x4 v = value(h + i, j);
        bf16x4 w;
#pragma unroll
        for (int x = 0; x < 4; ++x) w[x] = f2bf(v[x]);
        *reinterpret_cast<bf16x4*>(piece + b4_place<RB>(16 * i + (lane & 15), 2 * j + (lane >> 5)) + 8 * (lane >> 4 & 1)) = w;
        if (j & 1) __builtin_amdgcn_sched_barrier(0);      // (a few values at a time: together they do not fit)
      }
    }
    const B4Rows<RB> rows(piece, lane);
    if (__builtin_expect(ldo < 1 << 20, 1)) rows.out(to, lane, 16 * h, left, (int)(ldo * 2), whole);
    else rows.out_far(dst, ldo, lane, 16 * h, left);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Row block i of f32 results into the piece
template <int RI>
__device__ __forceinline__ B4Rows<512> b4_rows_f32(char* piece, int lane, const f32x4 (&acc)[RI][8], int i) {
#pragma unroll
  for (int j = 0; j < 8; ++j) *reinterpret_cast<f32x4*>(piece + b4_place<512>(lane & 15, 4 * j + (lane >> 4))) = acc[i][j];
  return B4Rows<512>(piece, lane);
}

// What a workgroup runs: lane i holds its i-th tile, rows [m0, end) and columns from n0 on, of expert e (GROUPED)
struct B4Items {
  int m0, end, n0, e;
};

// The results of a wave's block, rows [mw, end) and 128 columns from nw on, through its piece of LDS. GROUPED 2 / 3: of row
// mw + 64 q + lane the score, the pair.
template <int GROUPED, int E, int RI>
__device__ __forceinline__ void big4_results(const f32x4 (&acc)[RI][8], char* piece, int lane, int mw, int end, int nw, int M, int N,
                                             const bf16* __restrict__ bias, bf16* __restrict__ out, long ldo,
                                             float* __restrict__ part, const ExpertArgs& ex, const int (&pairs)[RI / 4],
                                             const float (&scores)[RI / 4]) {
  int el = lane;
  asm volatile("" : "+v"(el));        // (nothing of what follows is computed ahead of the K loop)
  const int left = end - mw;
  // (read where it is used: copies of many sums ahead of their use are registers that the next tile's fragments need)
  auto sum = [&](int i, int j) {
    f32x4 v = acc[i][j];
    asm volatile("" : "+a"(v));
    return v;
  };
  if constexpr (GROUPED == 3) {
#pragma unroll
    for (int i = 0; i < RI; ++i) {
      const auto rows = b4_rows_f32<RI>(piece, el, acc, i);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int r = 16 * (i & 3) + (el >> 5) + 2 * q;
        float* yr = ex.y + (long)__shfl(pairs[i / 4], r, 64) * ldo + nw + 4 * (el & 31);      // (by all lanes)
        if (64 * (i / 4) + r < left) *reinterpret_cast<f32x4*>(yr) = rows.v[q];
      }
    }
    return;
  } else if constexpr (GROUPED == 2) {
    float sc[RI];
#pragma unroll
    for (int i = 0; i < RI; ++i) sc[i] = __shfl(scores[i / 4], 16 * (i & 3) + (el & 15), 64);
    if constexpr (E == EPI_RELU2)
      b4_out<RI, 8>(piece, el, left, out + (long)mw * ldo + nw, ldo, [&](int i, int j) {
        f32x4 v;
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = fmaxf(acc[i][j][x] * sc[i], 0.f);
        return v * v;
      });
    else
      b4_out<RI, 4>(piece, el, left, out + (long)mw * ldo + (nw >> 1), ldo, [&](int i, int j) {
        f32x4 v;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const float g = fminf(acc[i][j][x] * sc[i], ex.limit);
          const float u = fminf(fmaxf(acc[i][j + 4][x] * sc[i], -ex.limit), ex.limit);
          v[x] = glu_gate(g, ex.alpha, __expf(-ex.alpha * g)) * (u + ex.up_offset);
        }
        return v;
      });
    return;
  }
  if (nw >= N) return;     // the columns past N of a half tile (their weight rows read zeros)
  if constexpr (E == kB4Parts) {
    float* slab = part + ((long)blockIdx.y * M + mw) * N + nw;
    const auto to = __builtin_amdgcn_make_buffer_rsrc((void*)slab, (short)0, 0x7fffffff, 0x00020000);
#pragma unroll
    for (int i = 0; i < RI; ++i) b4_rows_f32<RI>(piece, el, acc, i).out(to, el, 16 * i, left, N * 4, true);
  } else if constexpr (E == EPI_SILU || E == EPI_GLU) {      // the wave's column blocks are gate and up in turn
    const GluPar gp = E == EPI_GLU ? glu_par(bias, N) : GluPar{};
    b4_out<RI, 4>(piece, el, left, out + (long)mw * ldo + (nw >> 1), ldo, [&](int i, int j) {
      const f32x4 g = sum(i, 2 * j), u = sum(i, 2 * j + 1);
      f32x4 v;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        if constexpr (E == EPI_GLU) {
          const bf16* b = bias + nw + 32 * j + 4 * (el >> 4) + x;
          v[x] = glu_clamped(g[x] + bf2f(b[0]), u[x] + bf2f(b[16]), gp);
        } else {
          v[x] = silu(g[x]) * u[x];
        }
      }
      return v;
    });
  } else {
    f32x4 b[8] = {};
    if constexpr (E == EPI_BIAS) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int x = 0; x < 4; ++x) b[j][x] = bf2f(bias[nw + 16 * j + 4 * (el >> 4) + x]);
    }
    b4_out<RI, 8>(piece, el, left, out + (long)mw * ldo + nw, ldo, [&](int i, int j) {
      f32x4 v = acc[i][j];
      if constexpr (E == EPI_BIAS) v += b[j];
      if constexpr (E == EPI_RELU2) {
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = fmaxf(v[x], 0.f) * fmaxf(v[x], 0.f);
      }
      return v;
    });
  }
}

// A run of tiles from the at-th item on: of 256 rows (BM 256) while each has more than 128, one of 128 or less. Returns the item behind it.
// The rings run on from a tile to the next: its first K-tiles are on their way through the last two of the one before, the slot
// that the last K-tile's A leaves holds the results on their way out (a wave's quarter of it is the part that its own next DMA
// fills, so nobody waits for anybody), and the stores go on under the next products. With a workgroup per tile and walked, us:
// 5000 x 5120 x 1024 54 and 51, 8192 x 8192 x 512 76 and 70, x 1024 117 and 111, x 2560 250 and 244, x 4096 374 and 374, 6184 x 8448
// x 1024 102 and 95, x 2048 175 and 169, 4000 x 28672 x 2048 (SwiGLU) 350 and 340; longer K, where power bounds the step, level
// (8192 x 10240 x 8192 928 and 927, 8192 x 57344 x 8192 SwiGLU 5143 and 5178).
template <int GROUPED, int BM, int E>
__device__ __forceinline__ int big4_run(const bf16* __restrict__ X, long ldx, const bf16* __restrict__ W, long ldw, long w_estride,
                                        const B4Items& items, int at, int count, int M, int N, int K,
                                        const bf16* __restrict__ bias, bf16* __restrict__ out, long ldo,
                                        float* __restrict__ part, const int* __restrict__ grows, const ExpertArgs& ex) {
  constexpr int RI = BM / 32;      // a wave's row blocks of 16, and its DMA instructions for a slot of A
  // Slots of the rings and their places: a half tile's products cover half of the latency only, and its smaller slots leave room
  // for one more of each.
  constexpr int SA = BM == 256 ? 3 : 4, SB = BM == 256 ? 2 : 3, kSlotA = BM * 128, kRingB = SA * kSlotA;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // wave index in an SGPR: the DMA's LDS destinations (M0) and the fragment row bases are then
  // scalar (a VGPR wave index cost a readfirstlane + s_nop per DMA instruction)
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wid >> 1, wc = wid & 1;
  const int ktiles = K / 64;
  const int kt0 = (int)(((long)ktiles * blockIdx.y) / gridDim.y);
  const int kt1 = (int)(((long)ktiles * (blockIdx.y + 1)) / gridDim.y);
  const int nk = kt1 - kt0;   // >= 2 (host check)

  // DMA: instruction s (0..7) of wave w fills LDS row block 8 w + s (8 rows x 128 B, lane-
  // linear); lane L supplies row 8 (8 w + s) + (L >> 3) at the chunk lds_frag expects in
  // position L & 7: chunk = (L & 7) ^ ((row >> 1) & 7) = (L & 7) ^ ((L >> 4) + 4 (s & 1)) & 7
  constexpr bool glu = GROUPED == 2 && E == EPI_GLU;
  const int drow = 64 * wid + (lane >> 3), arow = 8 * RI * wid + (lane >> 3);
  // weight row of LDS row drow: with a gate, waves 0 / 2 stage gate rows and 1 / 3 the up rows of the same columns
  const int brow = glu ? (wid & 1) * (N >> 1) + (wid >> 1) * 64 + (lane >> 3) : drow;
  int va[2], vb[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int ch = (lane & 7) ^ (((lane >> 4) + 4 * e) & 7);
    va[e] = (int)((arow * ldx + ch * 8) * 2);
    vb[e] = (int)((brow * ldw + ch * 8) * 2);
  }
  // Where an item's rows come from: the base and the bytes behind it (A rows past the tile's end and weight rows past N read
  // zeros). GROUPED 1 / 2: byte offsets of this lane's rows (at its chunk), from X where they are gathered (X has less than 2 GB:
  // grouped_on_big4, moe_big_ok), from the tile's first row where they follow one another (slots know no such bound)
  constexpr bool kRows = GROUPED == 1 || GROUPED == 2;
  const bool gather = GROUPED == 2 || grows != nullptr;
  struct Side {
    const char* base;
    int bytes;
  };
  auto item = [&](int v, int i) { return __builtin_amdgcn_readlane(v, i); };
  auto side = [](const bf16* base, long rows, long ld) {
    const long bytes = rows * ld * 2;
    return Side{reinterpret_cast<const char*>(base), (int)(bytes < 0x7fffffffL ? bytes : 0x7fffffffL)};
  };
  auto side_a = [&](int i) {
    const int m0 = item(items.m0, i);
    if (kRows) return side(gather ? X : X + (long)m0 * ldx, 1L << 30, 1);
    return side(X + (long)m0 * ldx, item(items.end, i) - m0, ldx);
  };
  auto side_b = [&](int i) {
    const int n = glu ? item(items.n0, i) >> 1 : item(items.n0, i);
    return side(W + (GROUPED ? (long)item(items.e, i) * w_estride : 0) + (long)n * ldw, N - n, ldw);
  };
  auto rows_of = [&](int i, int (&g)[RI]) {      // an item's rows (grows) or pairs (perm) ...
    if constexpr (kRows) {
      const int m0 = item(items.m0, i), end = item(items.end, i);
#pragma unroll
      for (int q = 0; q < RI; ++q) g[q] = min(m0 + arow + 8 * q, end - 1) - (gather ? 0 : m0);
      if (gather) {
        const int* from = GROUPED == 2 ? ex.perm : grows;
#pragma unroll
        for (int q = 0; q < RI; ++q) g[q] = from[g[q]];
      }
    }
  };
  auto offsets_of = [&](int (&g)[RI]) {      // ... and where they lie
    if constexpr (kRows) {
#pragma unroll
      for (int q = 0; q < RI; ++q) {
        const long src = GROUPED == 2 ? g[q] / ex.choices : g[q];
        g[q] = (int)((src * ldx + (((lane & 7) ^ (((lane >> 4) + 4 * (q & 1)) & 7)) * 8)) * 2);
        asm volatile("" : "+v"(g[q]));      // (here: behind the stores the wait for them would be one for those too)
      }
    }
  };
  auto rsrc = [](const Side& f) { return __builtin_amdgcn_make_buffer_rsrc((void*)f.base, (short)0, f.bytes, 0x00020000); };
  Side fa = side_a(at), fb = side_b(at);      // what the rings take next: tile and K-tile (bytes into a row)
  int ga[RI] = {}, oa = kt0 * 128, ob = kt0 * 128;
  auto dma_a = [&](int slot, int s) {
    if constexpr (kRows)
      b4_dma(rsrc(fa), smem + slot * kSlotA + (RI * wid + s) * 1024, ga[s], oa);
    else
      b4_dma(rsrc(fa), smem + slot * kSlotA + (RI * wid + s) * 1024, va[s & 1], oa + (int)(8 * s * ldx * 2));
  };
  auto dma_b = [&](int slot, int s) {
    b4_dma(rsrc(fb), smem + kRingB + slot * kB4Slot + (8 * wid + s) * 1024, vb[s & 1], ob + (int)(8 * s * ldw * 2));
  };
  const int fr = lane & 15, fq = lane >> 4;
  // fragment idx 0-7: B rows (output columns) 16 idx, 8-15: A rows 16 (idx - 8), of k-step ks.
  // lds_frag's swizzle depends on row bits 1-3 = fr bits 1-3 only, so a lane's fragments of one
  // (slot, ks) share one VGPR address and differ by immediates of 2048 B (16 rows)
  int lo[2][2];   // [operand A / B][ks] lane byte offset inside a slot
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int ch = ((ks * 4 + fq) ^ ((fr >> 1) & 7)) * 16;
    lo[0][ks] = (wr * (BM / 2) + fr) * 128 + ch;
    lo[1][ks] = (wc * 128 + fr) * 128 + ch;
  }
  auto rd1 = [&](int sa_, int sb_, int ks, int idx, bf16x8 (&f)[8 + RI]) {
    const char* p = idx < 8 ? smem + kRingB + sb_ * kB4Slot + lo[1][ks] + 2048 * idx
                            : smem + sa_ * kSlotA + lo[0][ks] + 2048 * (idx - 8);
    f[idx] = *reinterpret_cast<const bf16x8*>(p);
  };
  // store instructions of a full tile's results, at least
  constexpr int kStores = GROUPED == 3 || E == kB4Parts ? 8 * RI : E == EPI_SILU || E == EPI_GLU ? 2 * RI : 4 * RI;
  f32x4 acc[RI][8];
  // MFMA group n (0 .. 2 RI - 1): output row block i = n / 2, column blocks 4 (n & 1) .. + 3
  auto mf4 = [&](int n, const bf16x8 (&f)[8 + RI], bool first) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = n >> 1, j = 4 * (n & 1) + q;
      acc[i][j] = mfma16(f[j], f[8 + i], first ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[i][j]);
    }
  };
  bf16x8 f0[8 + RI], f1[8 + RI];   // all fragments of k-step 0 / k-step 1

  rows_of(at, ga);
  offsets_of(ga);
  // the next item goes on in the rings (BM 256): a whole tile whose rows are known before its first K-tile is due
  auto follows = [&](int i) { return BM == 256 && i < count && nk >= 4 && item(items.end, i) - item(items.m0, i) > 128; };
  bool more = follows(at + 1);
  int gn[RI] = {};      // the rows of the next item, or of this one where none follows: its first K-tiles once more, for nobody
  Side na = side_a(more ? at + 1 : at), nb = side_b(more ? at + 1 : at);
  // Ahead of the barrier in K-tile k: to the next item behind the last K-tile. One branch that the others fall through: a lone wave
  // waits for every jump (three of them took 2 % of a long K), and selects at the DMA would stand before the next products.
  auto turn = [&](int k) {
    oa += 128;
    if (__builtin_expect(k + SA >= nk, 0)) {
      asm volatile("");
      if (k + SA == nk) {
        fa = na;
        oa -= nk * 128;
#pragma unroll
        for (int q = 0; q < RI; ++q) ga[q] = gn[q];
      }
      if (k + SB == nk) {
        fb = nb;
        ob -= nk * 128;
      }
    }
  };

  // prologue: A(0), B(0), A(1), B(1), A(2) (the ring's load order: B(t+2) then A(t+3))
#pragma unroll
  for (int t = 0; t < SB; ++t) {
#pragma unroll
    for (int s = 0; s < RI; ++s) dma_a(t, s);
#pragma unroll
    for (int s = 0; s < 8; ++s) dma_b(t, s);
    oa = t + 1 < nk || nk >= SA ? oa + 128 : kt0 * 128;      // (fewer K-tiles than slots: nobody turns)
    ob = t + 1 < nk || nk >= SB ? ob + 128 : kt0 * 128;
  }
  rows_of(more ? at + 1 : at, gn);
  offsets_of(gn);
  vm_wait<(SB - 1) * (8 + RI)>();     // K-tile 0 landed (own part); A(1), B(1) (and A(2), B(2)) fly
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int idx = 0; idx < 8 + RI; ++idx) rd1(0, 0, 0, idx, f0);

  // The loop is rotated so its back edge sits right after the barrier (the compiler puts a
  // conservative lgkmcnt(0) at a loop header: there it finds nothing outstanding): iteration k =
  // ks 1 of K-tile k, then ks 0 of K-tile k + 1, then the barrier; the last ks 1 is peeled.
  auto next_b = [](int sb_) { return SB == 2 ? sb_ ^ 1 : sb_ == SB - 1 ? 0 : sb_ + 1; };
  auto ks0 = [&](int k, int sa_, int sb_, bool first, bool stores) {   // ks 0 of K-tile k: its ks-1 fragments read
#pragma unroll
    for (int n = 0; n < 2 * RI; ++n) {
      mf4(n, f0, first);
      // into the slot K-tile k-1 left (its last reads precede the previous barrier)
      if (n & 1) dma_a(sa_ == 0 ? SA - 1 : sa_ - 1, n >> 1);
      rd1(sa_, sb_, 1, n, f1);
      if (RI == 4 && n < 4) rd1(sa_, sb_, 1, 8 + n, f1);      // (twelve fragments in eight slots)
      __builtin_amdgcn_sched_barrier(0);
    }
    turn(k);
    // A(k+1), B(k+1) landed; A(k+2) (B(k+2), A(k+3)) may fly, and behind a tile the stores of its results (kStores or more)
    if (stores) vm_wait<RI + kStores < 63 ? RI + kStores : 63>();
    else vm_wait<RI + (SB - 2) * (8 + RI)>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
  };
  auto ks1 = [&](int k, int sa_, int sb_, int sa1_) {   // ks 1 of K-tile k: next ks-0 read, DMA
#pragma unroll
    for (int n = 0; n < 2 * RI; ++n) {
      mf4(n, f1, false);
      rd1(sa1_, next_b(sb_), 0, n, f0);
      if (RI == 4 && n < 4) rd1(sa1_, next_b(sb_), 0, 8 + n, f0);
      if (RI == 4) dma_b(sb_, n);      // B(k + SB) into the slot K-tile k just left
      else if (n & 1) dma_b(sb_, n >> 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    ob += 128;
  };
  int sa = 0, sb = 0;   // slots of K-tile k: those of a stream's K-tiles in turn
  bool stores = false;
  for (;;) {
    int pairs[RI / 4] = {};
    float scores[RI / 4];
    if constexpr (GROUPED >= 2) {
#pragma unroll
      for (int q = 0; q < RI / 4; ++q)
        pairs[q] = ex.perm[min(item(items.m0, at) + wr * (BM / 2) + 64 * q + lane, item(items.end, at) - 1)];
    }
    ks0(0, sa, sb, true, stores);
    for (int k = 0; k + 1 < nk; ++k) {
      const int sa1 = sa == SA - 1 ? 0 : sa + 1;
      ks1(k, sa, sb, sa1);
      sb = next_b(sb);
      ks0(k + 1, sa1, sb, false, false);
      sa = sa1;
    }
    const int last = sa;
    sa = sa == SA - 1 ? 0 : sa + 1;
    const bool again = more && follows(at + 2);
    rows_of(again ? at + 2 : more ? at + 1 : at, gn);       // (the next tile's own have become ga)
#pragma unroll
    for (int q = 0; q < RI / 4; ++q) scores[q] = 1.f;
    if (GROUPED == 2 && ex.topk_w) {
#pragma unroll
      for (int q = 0; q < RI / 4; ++q) scores[q] = ex.topk_w[pairs[q]];
    }
    ks1(nk - 1, last, sb, sa);
    offsets_of(gn);
    sb = next_b(sb);
    if (!more) {
      vm_wait<0>();                       // no LDS-DMA may outlive the workgroup, none lands where results wait
      if (BM == 128) __builtin_amdgcn_s_barrier();       // (its smaller slots: pieces over several of them)
    }
    big4_results<GROUPED, E, RI>(acc, smem + (BM == 256 ? last * kSlotA : 0) + 8192 * wid, lane, item(items.m0, at) + wr * (BM / 2),
                                 item(items.end, at), item(items.n0, at) + wc * 128, M, N, bias, out, ldo, part, ex, pairs, scores);
    stores = item(items.end, at) - item(items.m0, at) >= BM && item(items.n0, at) + 256 <= N;
    ++at;
    if (!more) return at;
    more = again;
    if (more) {
      na = side_a(at + 1);
      nb = side_b(at + 1);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // the piece is read: the next A may land in it
  }
}

// Tiles at the end of the walk that run as two halves of 128 rows each: those of a last round of 256 workgroups that would leave
// half of the compute units or more idle. A half tile takes 0.6 to 0.7 of a whole one's time (its K step is bound by LDS reads and
// latency, 0.7 us beside 1.15), so a last round of more tiles, whose halves come in two rounds, would gain nothing. Before and
// after, us: 2870 x 6144 x 4096 (288 tiles) 175 and 149, 520 x 28672 x 4096 (336, a third of them with 8 rows) 171 and 148, 8192 x
// 8448 x 2048 (1056) 250 and 236, 6184 x 10752 x 2048 (1050) 244 and 228. Tiles whose rows end in their first half run as half
// tiles everywhere.
__host__ __device__ __forceinline__ int big4_halved(int tiles) { return tiles % 256 <= 128 ? tiles % 256 : 0; }

template <int GROUPED, int E>
__global__ void __launch_bounds__(kB4Threads) __attribute__((amdgpu_waves_per_eu(1, 1)))
gemm_big4_kernel(const bf16* __restrict__ X, long ldx, const bf16* __restrict__ W, long ldw,
                 int M, int N, int K, const bf16* __restrict__ bias,
                 bf16* __restrict__ out, long ldo, float* __restrict__ part, int halved = 0,
                 const int* __restrict__ grows = nullptr, const int4* __restrict__ gtiles = nullptr,
                 const int* __restrict__ gcount = nullptr, long w_estride = 0, ExpertArgs ex = ExpertArgs()) {
  constexpr int BM = 256, BN = 256;
  const int mtiles = GROUPED ? __builtin_amdgcn_readfirstlane(*gcount) : (M + BM - 1) / BM;
  const int ntiles = (N + BN - 1) / BN;      // (N % 256 == 128: half a last column tile)
  const int tiles = mtiles * ntiles;
  if constexpr (GROUPED != 0) halved = big4_halved(tiles);
  const int whole = tiles - halved, all = whole + 2 * halved;
  const int count = (int)blockIdx.x < all ? (all - 1 - (int)blockIdx.x) / (int)gridDim.x + 1 : 0;
  B4Items items{0, 0, 0, 0};      // lane i: tile blockIdx.x + i gridDim.x of the walk
  {
    int t = (int)blockIdx.x + (int)(threadIdx.x & 63) * (int)gridDim.x, half = -1;
    if (t < all) {
      if (t < whole) {
        t = xcd_remap(t, whole);
      } else {
        t = xcd_remap(t - whole, 2 * halved);
        half = t & 1;
        t = whole + (t >> 1);
      }
      const int per_group = kBigGroupM * ntiles;
      const int grp = t / per_group, first_m = grp * kBigGroupM;
      const int gsize = min(mtiles - first_m, kBigGroupM);
      const int ti = first_m + (t % per_group) % gsize;
      items.n0 = ((t % per_group) / gsize) * BN;
      if constexpr (GROUPED == 0) {
        items.m0 = ti * BM;
        items.end = min(M, items.m0 + BM);
      } else if constexpr (GROUPED == 1) {
        const int4 info = gtiles[ti];      // rows [y, z) of the slot space
        items.e = info.x;
        items.m0 = info.y;
        items.end = min(info.z, info.y + BM);
      } else {
        items.e = ex.tiles[2 * ti];
        items.m0 = ex.tiles[2 * ti + 1];
        items.end = min(ex.offsets[items.e + 1], items.m0 + BM);      // rows of the expert's group
      }
      if (half >= 0) {      // rows [m0, m0 + 128) or the 128 behind them
        items.m0 += half * (BM / 2);
        items.end = min(items.end, items.m0 + BM / 2);
      }
    }
  }
  for (int i = 0; i < count;) {
    const int rows = __builtin_amdgcn_readlane(items.end, i) - __builtin_amdgcn_readlane(items.m0, i);
    if (rows <= 0) {
      ++i;
      continue;
    }
    if (rows <= BM / 2)
      i = big4_run<GROUPED, BM / 2, E>(X, ldx, W, ldw, w_estride, items, i, count, M, N, K, bias, out, ldo, part, grows, ex);
    else
      i = big4_run<GROUPED, BM, E>(X, ldx, W, ldw, w_estride, items, i, count, M, N, K, bias, out, ldo, part, grows, ex);
    __builtin_amdgcn_s_barrier();      // (the rings are everybody's again)
  }
}

// Workgroups for `tiles` tiles: one per compute unit, which walks them; more where a wave's lanes could not hold its list
static int big4_grid(long tiles) { return (int)std::min(tiles, 256 * ((tiles + 256 * 64 - 1) / (256 * 64))); }

// ---------------------------------------------------------------------------------------
// Mid-M GEMM (plan kind 5): the tensor-parallel shard projections at M = 128-512 rows (tp2-tp8
// decode at 64 sequences per GPU, large single-GPU batches), where a 256x256 tile grid leaves
// most of the 256 CUs idle (tp8 QKV at M = 512: 10 tiles) and the 4-wave tile kernel keeps the
// matrix pipe ~25 % busy (one wave per SIMD, every K-tile behind one barrier).
//
// 8 waves in two groups of 4 staggered by one s_barrier (big8's scheme): each wave owns a
// 64 x WN output block (WN = 64 for 256x128 / 128x256 tiles, 32 for 128x128), and every
// K-tile (BK = 64) is two k-steps of 32. Per k-step a wave has a READ segment (its A and B
// fragments of that k-step, TI + TJ ds_read_b128, and half of its share of the LDS-DMA) and an
// MFMA segment (TI x TJ mfma_16x16x32). Group 1 runs one barrier behind group 0, so on every
// SIMD one wave's MFMA segment overlaps its partner's read segment:
//     global segment:  4k     4k+1   4k+2   4k+3   (k = K-tile)
//     group 0:         R0(k)  M0(k)  R1(k)  M1(k)
//     group 1:         M1(k-1) R0(k) M0(k)  R1(k)
// LDS: two rings of K-tile images (128-B rows, XOR-swizzled like lds_frag): SX slots of the
// activation rows X (BM x 64, mostly L2 hits: short latency) and SW >= SX slots of the weight
// rows W (BN x 64, streamed from HBM: the deep one). Iteration k issues X(k + SX - 1) in its
// first read segment and W(k + SW - 1) in its second, each into the slot of K-tile k - 1,
// whose last reader (group 1's R1(k-1), global segment 4k-1) retired its reads (lgkmcnt(0))
// before the barrier opening segment 4k. RAW: K-tile k+1 is first read in global segment 4k+4
// (group 0's R0(k+1)), so every wave retires its own DMA of K-tile k+1 before the barrier that
// closes segment 4k+3: group 0 at the end of M1(k), group 1 at the end of R1(k); the counted
// wait leaves exactly the loads issued after the later of X(k+1) / W(k+1) in flight (counted
// at run time near the tail, where the load stream thins out).
// DMA through buffer descriptors based at the tile's first row (A rows past M read zeros);
// weights streamed non-temporally when one row tile covers M (each byte read by one workgroup).
// Grid: 1-D, split-major then N-tile then M-tile, XCD-remapped, so an XCD's consecutive
// workgroups share a weight panel (and K range) across the M tiles in its L2.
// Measured (profiles/r5_gemm): one ring of whole K-tiles (SX = SW = 3) kept the matrix pipe
// 29 % busy on the tp8 down projection at M = 512, the waves parked on the DMA wait (SQ_WAIT_ANY
// 35 %) with 75 % L2 hits: the weight stream's latency, not the MFMA or LDS issue, bounds it.
// ---------------------------------------------------------------------------------------
constexpr int kMidThreads = 512;

template <int BM, int BN, int SX, int SW>
struct MidCfg {
  static constexpr int WM = 64;                          // wave rows
  static constexpr int WN = (BM * BN) / (8 * WM);        // wave columns: 8 waves cover the tile
  static constexpr int WGN = BN / WN, WGM = BM / WM;     // wave grid
  static constexpr int TI = WM / 16, TJ = WN / 16;
  static constexpr int XB = BM * 128, WB = BN * 128;     // bytes per X / W slot
  static constexpr int LX = BM / 64, LW = BN / 64;       // DMA instructions per wave per K-tile
  static constexpr int LDS = SX * XB + SW * WB;
  static_assert(WGM * WGN == 8 && WN % 16 == 0, "mid tile shape");
  static_assert(SX >= 2 && SW >= SX, "mid rings");
  static_assert(LDS <= 160 * 1024, "mid rings exceed the LDS");
};

// One 1-KiB LDS-DMA block through a buffer descriptor (a __device__ helper: the builtin's LDS
// address-space cast inside the kernel template's lambda left the template uninstantiable on
// the host side, i.e. no launch stub was emitted)
template <int AUX>
__device__ __forceinline__ void mid_dma1(__amdgpu_buffer_rsrc_t r, char* lds, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)lds, 16, voff, soff, 0, AUX);
}

// s_waitcnt vmcnt(n) for a run-time n (the count is an immediate): a jump over constants;
// n above the largest case waits for less than allowed, i.e. is clamped to a safe (longer) wait
__device__ __forceinline__ void vm_wait_dyn(int n) {
  switch (n) {
    case 0: vm_wait<0>(); break;   case 1: vm_wait<1>(); break;   case 2: vm_wait<2>(); break;
    case 3: vm_wait<3>(); break;   case 4: vm_wait<4>(); break;   case 5: vm_wait<5>(); break;
    case 6: vm_wait<6>(); break;   case 7: vm_wait<7>(); break;   case 8: vm_wait<8>(); break;
    case 9: vm_wait<9>(); break;   case 10: vm_wait<10>(); break; case 11: vm_wait<11>(); break;
    case 12: vm_wait<12>(); break; case 13: vm_wait<13>(); break; case 14: vm_wait<14>(); break;
    case 15: vm_wait<15>(); break; case 16: vm_wait<16>(); break; case 17: vm_wait<17>(); break;
    case 18: vm_wait<18>(); break; case 19: vm_wait<19>(); break; case 20: vm_wait<20>(); break;
    case 21: vm_wait<21>(); break; case 22: vm_wait<22>(); break; case 23: vm_wait<23>(); break;
    default: vm_wait<24>(); break;
  }
}

template <int BM, int BN, int SX, int SW, bool PK = false>
__global__ void __launch_bounds__(kMidThreads)
gemm_mid8_kernel(const bf16* __restrict__ X, long ldx, const bf16* __restrict__ W, long ldw,
                 int M, int N, int K, int epi, const bf16* __restrict__ bias,
                 bf16* __restrict__ out, long ldo, float* __restrict__ part, int nsplit,
                 RowScale rsc) {
  using C = MidCfg<BM, BN, SX, SW>;
  constexpr int TI = C::TI, TJ = C::TJ, LX = C::LX, LW = C::LW;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* const xs = smem;
  char* const wsm = smem + SX * C::XB;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int grp = wid >> 2;
  const int wm = wid / C::WGN, wn = wid % C::WGN;
  const int mtiles = (M + BM - 1) / BM, ntiles = N / BN;
  const int t = xcd_remap((int)blockIdx.x, mtiles * ntiles * nsplit);
  const int tm = t % mtiles, tn = (t / mtiles) % ntiles, ksplit = t / (mtiles * ntiles);
  const int m0 = tm * BM, n0 = tn * BN;
  const int ktiles = K / kBK;
  const int kt0 = (int)(((long)ktiles * ksplit) / nsplit);
  const int nk = (int)(((long)ktiles * (ksplit + 1)) / nsplit) - kt0;

  // DMA: wave w moves the 1-KiB blocks w, w + 8, ... of an X / W slot (BM / 8, BN / 8 blocks)
  const auto rsa = b8_rsrc(X + (long)m0 * ldx, M - m0, ldx);
  // PK: W in the K-tile-blocked layout [N/256][K/64][256][64] (pack_w256): the tile's BN rows
  // lie in one 256-row block (BN divides 256), a row is 128 B and a K-tile 32 KiB further on
  const long wpitch = PK ? 64 : ldw;
  const auto rsb = PK ? b8_rsrc(W + ((long)(n0 >> 8) * K << 8) + (n0 & 255) * 64, 1, (long)K * 256 - (n0 & 255) * 64)
                      : b8_rsrc(W + (long)n0 * ldw, N - n0, ldw);
  const bool wnt = mtiles == 1 && g_tile_w_nt;
  int vx[LX], vw[LW];
#pragma unroll
  for (int i = 0; i < LX; ++i) {
    const int row = (wid + 8 * i) * 8 + (lane >> 3);
    vx[i] = (int)((row * ldx + (((lane & 7) ^ ((row >> 1) & 7)) * 8)) * 2);
  }
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int row = (wid + 8 * i) * 8 + (lane >> 3);
    vw[i] = (int)((row * wpitch + (((lane & 7) ^ ((row >> 1) & 7)) * 8)) * 2);
  }
  auto dma_x = [&](int k) {
    char* s = xs + (k % SX) * C::XB;
    const int soff = (kt0 + k) * kBK * 2;
#pragma unroll
    for (int i = 0; i < LX; ++i) mid_dma1<0>(rsa, s + (wid + 8 * i) * 1024, vx[i], soff);
  };
  auto dma_w = [&](int k) {
    char* s = wsm + (k % SW) * C::WB;
    const int soff = (kt0 + k) * (PK ? 256 * kBK * 2 : kBK * 2);
    if (wnt) {
#pragma unroll
      for (int i = 0; i < LW; ++i) mid_dma1<2>(rsb, s + (wid + 8 * i) * 1024, vw[i], soff);
    } else {
#pragma unroll
      for (int i = 0; i < LW; ++i) mid_dma1<0>(rsb, s + (wid + 8 * i) * 1024, vw[i], soff);
    }
  };
  // Loads issued (in order X(j + SX - 1), W(j + SW - 1) per iteration j; the prologue is the
  // virtual iterations 1 - SW .. -1) after the later of X(k+1) / W(k+1): what may stay in
  // flight once K-tile k+1 must have landed (k = -1: the prologue's wait for K-tile 0).
  auto after = [&](int k) {
    const int kt = k + 1;
    const int jx = kt - SX + 1, jw = kt - SW + 1;   // iterations that issued X(kt), W(kt)
    int n = 0;
    if (jw == jx) {   // SW == SX: W(kt) is the later one
      // nothing else of iteration jx after it
    } else if (kt + SW - SX < nk) {
      n += LW;        // W(jx + SW - 1) of the same iteration, behind X(kt)
    }
    for (int j = jx + 1; j <= k; ++j) {
      if (j + SX - 1 < nk) n += LX;
      if (j + SW - 1 < nk) n += LW;
    }
    return n;
  };

  f32x4 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // prologue = virtual iterations 1-SW .. -1: W(0 .. SW-2), X(0 .. SX-2) in issue order
#pragma unroll
  for (int v = 1 - SW; v <= -1; ++v) {
    if (v + SX - 1 >= 0 && v + SX - 1 < nk) dma_x(v + SX - 1);
    if (v + SW - 1 < nk) dma_w(v + SW - 1);
  }
  vm_wait_dyn(after(-1));
  __builtin_amdgcn_s_barrier();
  if (grp == 1) __builtin_amdgcn_s_barrier();

  const int ar = wm * C::WM + (lane & 15), bc = wn * C::WN + (lane & 15);
  bf16x8 af[TI], bfr[TJ];
  for (int k = 0; k < nk; ++k) {
    const char* As = xs + (k % SX) * C::XB;
    const char* Bs = wsm + (k % SW) * C::WB;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      // ---- read segment: this k-step's fragments; X(k + SX - 1) / W(k + SW - 1) DMA
#pragma unroll
      for (int i = 0; i < TI; ++i) af[i] = lds_frag(As, ar + 16 * i, ks * 4 + (lane >> 4));
#pragma unroll
      for (int j = 0; j < TJ; ++j) bfr[j] = lds_frag(Bs, bc + 16 * j, ks * 4 + (lane >> 4));
      if (ks == 0) {
        if (k + SX - 1 < nk) dma_x(k + SX - 1);
      } else {
        if (k + SW - 1 < nk) dma_w(k + SW - 1);
        if (grp == 1) vm_wait_dyn(after(k));
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      // ---- MFMA segment
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = mfma16(bfr[j], af[i], acc[i][j]);   // C^T tile
      __builtin_amdgcn_s_setprio(0);
      if (ks == 1 && grp == 0) vm_wait_dyn(after(k));
      __builtin_amdgcn_s_barrier();
    }
  }
  if (grp == 0) __builtin_amdgcn_s_barrier();   // re-align the groups' barrier counts
  tile_epilogue<TI, TJ>(acc, m0 + wm * C::WM, n0 + wn * C::WN, lane, M, N, epi, bias, out, ldo,
                        part ? part + (long)ksplit * M * N + (long)m0 * N : nullptr, m0, rsc);
}

// ---------------------------------------------------------------------------------------
// Host dispatch
// ---------------------------------------------------------------------------------------
// ---------------------------------------------------------------------------------------
// Mid-M one-wave-per-SIMD GEMM (plan kind 7, "mid4"): big4's structure on 128x128 / 256x128 /
// 128x256 tiles for the TP-shard and large-batch decode projections (M = 128-512), where
// split-K fills the chip and each workgroup walks only 8-30 K-tiles. 4 waves in 2 x 2, each
// owning a (BM/2) x (BN/2) block; per K-tile a wave runs TI x TJ MFMAs per k-step in slots of 4
// (sched_barrier-fenced, fragment reads and LDS-DMA spread over the slots); LDS-DMA rings of SA
// activation and SB weight K-tiles (the whole 160 KiB: up to 5 weight K-tiles of lead for the
// HBM stream); one barrier per K-tile; the loop rotated to end on it (see gemm_big4_kernel).
// The DMA wait count at the barrier follows the fixed issue order
//   prologue A(0), B(0), A(1 .. SA-2), B(1 .. SB-1); iteration t: A(t+SA-1) in k-step 0,
//   B(t+SB) in k-step 1
// and is computed per iteration (scalar), exact in the first iterations as in the steady state.
// ---------------------------------------------------------------------------------------
constexpr int kMid4Threads = 256;

template <int BM, int BN, int SA, int SB>
struct Mid4Cfg {
  static constexpr int WM = BM / 2, WN = BN / 2, TI = WM / 16, TJ = WN / 16;
  static constexpr int NS = TI * TJ / 4;            // MFMA slots per k-step
  static constexpr int NF = TI + TJ;                // fragments per k-step
  static constexpr int NA = BM / 32, NB = BN / 32;  // DMA instructions per thread per K-tile
  static constexpr int ASLOT = BM * 128, BSLOT = BN * 128;
  static constexpr int LDS = SA * ASLOT + SB * BSLOT;
  static_assert(TJ % 4 == 0 && NA % 2 == 0 && NB % 2 == 0, "mid4 tile shape");
  static_assert(SA >= 2 && SB >= 2 && LDS <= 160 * 1024, "mid4 rings");
};

template <int BM, int BN, int SA, int SB, bool PK = false>
__global__ void __launch_bounds__(kMid4Threads) __attribute__((amdgpu_waves_per_eu(1, 1)))
gemm_mid4_kernel(const bf16* __restrict__ X, long ldx, const bf16* __restrict__ W, long ldw,
                 int M, int N, int K, int epi, const bf16* __restrict__ bias,
                 bf16* __restrict__ out, long ldo, float* __restrict__ part, RowScale rsc) {
  using C = Mid4Cfg<BM, BN, SA, SB>;
  constexpr int TI = C::TI, TJ = C::TJ, NS = C::NS, NF = C::NF, NA = C::NA, NB = C::NB;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wid >> 1, wc = wid & 1;
  const int mtiles = (M + BM - 1) / BM, ntiles = N / BN;
  const int t = xcd_remap(blockIdx.x, mtiles * ntiles);
  const int per_group = kBigGroupM * ntiles;
  const int grp = t / per_group, first_m = grp * kBigGroupM;
  const int gsize = min(mtiles - first_m, kBigGroupM);
  const int m0 = (first_m + (t % per_group) % gsize) * BM;
  const int n0 = ((t % per_group) / gsize) * BN;
  const int ktiles = K / 64;
  const int kt0 = (int)(((long)ktiles * blockIdx.y) / gridDim.y);
  const int kt1 = (int)(((long)ktiles * (blockIdx.y + 1)) / gridDim.y);
  const int nk = kt1 - kt0;   // >= 1 (host check)

  // DMA: instruction s of wave w fills LDS row block NA w + s (A; NB w + s for B), 8 rows x
  // 128 B lane-linear, lane L supplying row 8 (block) + (L >> 3) at lds_frag's swizzled chunk
  // (L & 7) ^ ((L >> 4) + 4 (s & 1)) & 7 (NA, NB even)
  const auto rsa = b8_rsrc(X + (long)m0 * ldx, M - m0, ldx);   // A rows past M read zeros
  // PK: W in the pack_w256 layout (see gemm_mid8_kernel): 128-B rows, 32-KiB K-tiles
  const long wpitch = PK ? 64 : ldw;
  const int kstep = PK ? 256 * 128 : 128;
  const auto rsb = PK ? b8_rsrc(W + ((long)(n0 >> 8) * K << 8) + (n0 & 255) * 64, 1, (long)K * 256 - (n0 & 255) * 64)
                      : b8_rsrc(W + (long)n0 * ldw, N - n0, ldw);
  int va[2], vb[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int ch = (lane & 7) ^ (((lane >> 4) + 4 * e) & 7);
    va[e] = (int)(((8 * NA * wid + (lane >> 3)) * ldx + ch * 8) * 2);
    vb[e] = (int)(((8 * NB * wid + (lane >> 3)) * wpitch + ch * 8) * 2);
  }
  char* const bbase = smem + SA * C::ASLOT;
  auto dma_a = [&](int k, int slot, int s) {
    b4_dma(rsa, smem + slot * C::ASLOT + (NA * wid + s) * 1024, va[s & 1], (kt0 + k) * 128 + (int)(8 * s * ldx * 2));
  };
  auto dma_b = [&](int k, int slot, int s) {
    b4_dma(rsb, bbase + slot * C::BSLOT + (NB * wid + s) * 1024, vb[s & 1], (kt0 + k) * kstep + (int)(8 * s * wpitch * 2));
  };
  const int fr = lane & 15, fq = lane >> 4;
  int lo[2][2];   // [A / B][ks] lane byte offset inside a slot (fragments differ by 2048 B)
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int ch = ((ks * 4 + fq) ^ ((fr >> 1) & 7)) * 16;
    lo[0][ks] = (wr * C::WM + fr) * 128 + ch;
    lo[1][ks] = (wc * C::WN + fr) * 128 + ch;
  }
  // fragment idx 0 .. TJ-1: B (output columns 16 idx), TJ .. NF-1: A (rows 16 (idx - TJ))
  auto rd1 = [&](int sa_, int sb_, int ks, int idx, bf16x8 (&f)[NF]) {
    const char* p = idx < TJ ? bbase + sb_ * C::BSLOT + lo[1][ks] + 2048 * idx
                             : smem + sa_ * C::ASLOT + lo[0][ks] + 2048 * (idx - TJ);
    f[idx] = *reinterpret_cast<const bf16x8*>(p);
  };
  f32x4 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto mf4 = [&](int n, const bf16x8 (&f)[NF]) {   // slot n: row block i, 4 column blocks
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = n / (TJ / 4), j = 4 * (n % (TJ / 4)) + q;
      acc[i][j] = mfma16(f[j], f[TJ + i], acc[i][j]);
    }
  };
  bf16x8 f0[NF], f1[NF];

  // issue-order bookkeeping (per-thread load counts, see the header)
  constexpr int P = (SA - 1) * NA + SB * NB;
  auto idx_a = [&](int j) {
    return j == 0 ? NA : j <= SA - 2 ? NA + NB + j * NA : P + (j - SA + 1) * (NA + NB) + NA;
  };
  auto idx_b = [&](int j) {
    return j == 0 ? NA + NB : j <= SB - 1 ? NA + NB + (SA - 2) * NA + j * NB : P + (j - SB) * (NA + NB) + NA + NB;
  };
#pragma unroll
  for (int s = 0; s < NA; ++s) dma_a(0, 0, s);
#pragma unroll
  for (int s = 0; s < NB; ++s) dma_b(0, 0, s);
#pragma unroll
  for (int j = 1; j <= SA - 2; ++j)
#pragma unroll
    for (int s = 0; s < NA; ++s) dma_a(min(j, nk - 1), j, s);
#pragma unroll
  for (int j = 1; j <= SB - 1; ++j)
#pragma unroll
    for (int s = 0; s < NB; ++s) dma_b(min(j, nk - 1), j, s);
  vm_wait<P - NA - NB>();            // K-tile 0 landed (own part)
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int idx = 0; idx < NF; ++idx) rd1(0, 0, 0, idx, f0);

  auto ks0 = [&](int k, int sa_, int sb_) {   // k-step 0 of K-tile k; DMA A(k+SA-1); barrier
    const int ka = min(k + SA - 1, nk - 1), slot = sa_ == 0 ? SA - 1 : sa_ - 1;
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      mf4(n, f0);
#pragma unroll
      for (int q = n * NA / NS; q < (n + 1) * NA / NS; ++q) dma_a(ka, slot, q);
#pragma unroll
      for (int idx = n * NF / NS; idx < (n + 1) * NF / NS; ++idx) rd1(sa_, sb_, 1, idx, f1);
      __builtin_amdgcn_sched_barrier(0);
    }
    // A(k+1), B(k+1) landed (own part): the loads issued after the later of them may fly
    const int total = P + k * (NA + NB) + NA;
    vm_wait_dyn(total - max(idx_a(k + 1), idx_b(k + 1)));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
  };
  auto ks1 = [&](int k, int sa_, int sb_, int sa1_, int sb1_) {   // k-step 1; DMA B(k+SB)
    const int kb = min(k + SB, nk - 1);
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      mf4(n, f1);
#pragma unroll
      for (int idx = n * NF / NS; idx < (n + 1) * NF / NS; ++idx) rd1(sa1_, sb1_, 0, idx, f0);
#pragma unroll
      for (int q = n * NB / NS; q < (n + 1) * NB / NS; ++q) dma_b(kb, sb_, q);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int sa = 0, sb = 0;
  ks0(0, 0, 0);
  for (int k = 0; k + 1 < nk; ++k) {
    const int sa1 = sa == SA - 1 ? 0 : sa + 1, sb1 = sb == SB - 1 ? 0 : sb + 1;
    ks1(k, sa, sb, sa1, sb1);
    ks0(k + 1, sa1, sb1);
    sa = sa1;
    sb = sb1;
  }
  ks1(nk - 1, sa, sb, sa == SA - 1 ? 0 : sa + 1, sb == SB - 1 ? 0 : sb + 1);
  vm_wait<0>();                       // no LDS-DMA may outlive the workgroup
  tile_epilogue<TI, TJ>(acc, m0 + wr * C::WM, n0 + wc * C::WN, lane, M, N, epi, bias, out, ldo,
                        part ? part + (long)blockIdx.y * M * N + (long)m0 * N : nullptr, m0, rsc);
}

static int num_cus() { return 256; }

// Workspace layout: [kCounterBytes reserved head | SK x M x N f32 partials].
static float* splitk_part(float* ws) { return ws + kCounterBytes / sizeof(float); }



template <int MT, int NT, int WK>
static void run_skinny(const bf16* X, long ldx, const bf16* W, long ldw, int M, int N, int K,
                       int epi, const bf16* bias, bf16* out, long ldo, float* ws, int sk,
                       hipStream_t stream) {
  dim3 grid(N / (16 * NT * (4 / WK)), sk);
  gemm_skinny_kernel<MT, NT, WK><<<grid, kSkThreads, 0, stream>>>(
      X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, sk > 1 ? splitk_part(ws) : nullptr);
}

template <int MT, int NT, int NW, int U, int FOLD>
static void run_stream(const bf16* X, long ldx, const bf16* W, long ldw, int M, int N, int K, int epi, const bf16* bias,
                       bf16* out, long ldo, hipStream_t stream, bool packed) {
  gemm_stream_kernel<MT, NT, NW, U, FOLD><<<N / (16 / FOLD * NT), 64 * NW, 0, stream>>>(
      X, ldx, W, packed ? 64 : ldw, packed ? 256 * 64 : 64, M, N, K, epi, bias, out, ldo);
}

static void init_nt_policy() {
  static bool done = false;
  if (done) return;
  done = true;
  const int zero = 0;
  const char* e = getenv("BFLY_GEMM_NT_WEIGHTS");
  if (e && e[0] == '0') (void)hipMemcpyToSymbol(HIP_SYMBOL(g_tile_w_nt), &zero, sizeof(int));
}

template <int BM, int BN, int WMW, int STAGES, bool PACKW = false>
static void run_tile(const bf16* X, long ldx, const bf16* W, long ldw, int M, int N, int K,
                     int epi, const bf16* bias, bf16* out, long ldo, float* ws, int sk,
                     hipStream_t stream, const RowScale& rsc) {
  init_nt_policy();
  const int tiles = ((M + BM - 1) / BM) * (N / BN);
  const size_t lds = (size_t)STAGES * (BM + BN) * kBK * 2;
  const dim3 grid(tiles, sk);
  static bool attr_set = false;  // > 64 KiB of dynamic LDS must be opted into once per kernel
  if (!attr_set && lds > 65536) {
    hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_tile_kernel<BM, BN, WMW, STAGES, false, PACKW>),
                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    attr_set = true;
  }
  gemm_tile_kernel<BM, BN, WMW, STAGES, false, PACKW><<<grid, kTileThreads, lds, stream>>>(
      X, ldx, W, PACKW ? (long)K : ldw, M, N, K, epi, bias, out, ldo, sk > 1 ? splitk_part(ws) : nullptr,
      nullptr, nullptr, nullptr, 0, rsc);
}

template <int BM, int BN, int NWM, int NWN, int SW>
static void run_dec(const bf16* X, long ldx, const bf16* W, long ldw, int M, int N, int K,
                    int epi, const bf16* bias, bf16* out, long ldo, float* ws, int sk,
                    hipStream_t stream, const RowScale& rsc) {
  init_nt_policy();
  const int tiles = ((M + BM - 1) / BM) * (N / BN);
  constexpr size_t lds = (size_t)(3 * BM + SW * BN) * kBK * 2;
  static_assert(lds <= 160 * 1024, "decode GEMM rings exceed the 160 KiB LDS");
  static bool attr_set = false;
  if (!attr_set && lds > 65536) {
    hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_dec_kernel<BM, BN, NWM, NWN, SW>),
                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    attr_set = true;
  }
  const dim3 grid(tiles, sk);
  gemm_dec_kernel<BM, BN, NWM, NWN, SW><<<grid, NWM * NWN * 64, lds, stream>>>(
      X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, sk > 1 ? splitk_part(ws) : nullptr, rsc);
}

static void run_big8(const bf16* X, long ldx, const bf16* W, long ldw, int M, int N, int K,
                     int epi, const bf16* bias, bf16* out, long ldo, float* ws, int sk, hipStream_t stream) {
  static bool attr = false;
  if (!attr) {
    hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_big8_kernel<false>),
                        hipFuncAttributeMaxDynamicSharedMemorySize, kB8LdsBytes);
    attr = true;
  }
  const int tiles = ((M + 255) / 256) * (N / 256);
  dim3 grid(tiles, sk);
  float* part = sk > 1 ? splitk_part(ws) : nullptr;
  gemm_big8_kernel<false><<<grid, kB8Threads, kB8LdsBytes, stream>>>(X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, part);
}

static void run_big4(const bf16* X, long ldx, const bf16* W, long ldw, int M, int N, int K,
                     int epi, const bf16* bias, bf16* out, long ldo, float* ws, int sk, hipStream_t stream) {
  const int tiles = ((M + 255) / 256) * ((N + 255) / 256), halved = sk > 1 ? 0 : big4_halved(tiles);
  dim3 grid(sk > 1 ? tiles : big4_grid(tiles + halved), sk);
  float* part = sk > 1 ? splitk_part(ws) : nullptr;
#define BFLY_BIG4(E)                                                                                                     \
  {                                                                                                                      \
    static bool attr_set = false;                                                                                        \
    if (!attr_set) {                                                                                                     \
      hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_big4_kernel<0, E>),                                        \
                          hipFuncAttributeMaxDynamicSharedMemorySize, kB4LdsBytes);                                      \
      attr_set = true;                                                                                                   \
    }                                                                                                                    \
    gemm_big4_kernel<0, E><<<grid, kB4Threads, kB4LdsBytes, stream>>>(X, ldx, W, ldw, M, N, K, bias, out, ldo, part, \
                                                                      halved);                                           \
  }
  if (sk > 1) BFLY_BIG4(kB4Parts)      // (the reduce applies the epilogue)
  else if (epi == EPI_NONE) BFLY_BIG4(EPI_NONE)
  else if (epi == EPI_SILU) BFLY_BIG4(EPI_SILU)
  else if (epi == EPI_BIAS) BFLY_BIG4(EPI_BIAS)
  else if (epi == EPI_RELU2) BFLY_BIG4(EPI_RELU2)
  else BFLY_BIG4(EPI_GLU)
#undef BFLY_BIG4
}

template <int BM, int BN, int SA, int SB, bool PK = false>
static void run_mid4(const bf16* X, long ldx, const bf16* W, long ldw, int M, int N, int K, int epi,
                     const bf16* bias, bf16* out, long ldo, float* ws, int sk, hipStream_t stream,
                     const RowScale& rsc) {
  using C = Mid4Cfg<BM, BN, SA, SB>;
  static bool attr_set = false;
  if (!attr_set) {
    hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_mid4_kernel<BM, BN, SA, SB, PK>),
                        hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
    attr_set = true;
  }
  dim3 grid(((M + BM - 1) / BM) * (N / BN), sk);
  float* part = sk > 1 ? splitk_part(ws) : nullptr;
  gemm_mid4_kernel<BM, BN, SA, SB, PK><<<grid, kMid4Threads, C::LDS, stream>>>(X, ldx, W, ldw, M, N, K, epi, bias,
                                                                         out, ldo, part, rsc);
}

template <int BM, int BN, int SX, int SW, bool PK = false>
static void run_mid8(const bf16* X, long ldx, const bf16* W, long ldw, int M, int N, int K, int epi,
                     const bf16* bias, bf16* out, long ldo, float* ws, int sk, hipStream_t stream,
                     const RowScale& rsc) {
  init_nt_policy();
  constexpr size_t lds = (size_t)MidCfg<BM, BN, SX, SW>::LDS;
  static bool attr = false;
  if (!attr) {
    hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_mid8_kernel<BM, BN, SX, SW, PK>),
                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    attr = true;
  }
  const int tiles = ((M + BM - 1) / BM) * (N / BN);
  gemm_mid8_kernel<BM, BN, SX, SW, PK><<<tiles * sk, kMidThreads, lds, stream>>>(
      X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, sk > 1 ? splitk_part(ws) : nullptr, sk, rsc);
}

// Plan selection, from the tools/bench_gemm.py sweep on MI355X (Llama-3-70B TP1/TP8 shapes,
// weights streamed from HBM): the LDS-tiled kernel with a small BM and split-K beats the
// register-streaming skinny kernel for every M >= 8 (e.g. down-proj M=64: 90 us = 5.2 TB/s vs
// 186 us) and ties or beats hipBLASLt; the skinny kernel stays for M <= 4 (GEMV regime).
// Split-K is sized so the grid has ~448 workgroups (1.75 per CU) with >= 4 K-tiles each.
// Measured plan table (tools/gen_gemm_table.py from the profiles/gemm_tune_*.json sweeps of
// tools/bench_gemm.py --sweep on MI355X): the fastest plan per model projection shape and
// token-count bucket (entries exist only where the sweep beat the heuristic by > 3%).
struct TunedPlan { int N, K, M, kind, mt, nt, wk, bm, bn, sk; };
static const TunedPlan kTuned[] = {
#include "gemm_tuned.inc"
};

static GemmPlan plan_gemm_heuristic(int M, int N, int K);

static bool tuned_enabled() {   // BFLY_GEMM_TUNED=0: heuristic plans only (A/B runs)
  static const bool on = [] {
    const char* e = getenv("BFLY_GEMM_TUNED");
    return !(e && e[0] == '0');
  }();
  return on;
}

// BFLY_GEMM_PLAN="N,K,Mbucket:kind,mt,nt,wk,bm,bn,sk;..." forces plans for whole-model A/B runs
// (a shape's plan measured inside the decode step, where the neighbouring kernels and the
// cache state differ from an isolated sweep). Parsed once.
struct PlanOverride { int N, K, M; GemmPlan p; };
static const std::vector<PlanOverride>& plan_overrides() {
  static const std::vector<PlanOverride> v = [] {
    std::vector<PlanOverride> out;
    const char* e = getenv("BFLY_GEMM_PLAN");
    if (!e) return out;
    std::string s(e);
    size_t pos = 0;
    while (pos < s.size()) {
      size_t end = s.find(';', pos);
      if (end == std::string::npos) end = s.size();
      PlanOverride o{};
      if (sscanf(s.substr(pos, end - pos).c_str(), "%d,%d,%d:%d,%d,%d,%d,%d,%d,%d", &o.N, &o.K, &o.M, &o.p.kind,
                 &o.p.mt, &o.p.nt, &o.p.wk, &o.p.bm, &o.p.bn, &o.p.sk) == 10)
        out.push_back(o);
      pos = end + 1;
    }
    return out;
  }();
  return v;
}

// token-count buckets of the sweep: M uses the entry of its bucket, or the heuristic plan when the sweep found nothing better there
static bool tuned_plan(int M, int N, int K, GemmPlan& p) {
  if (!tuned_enabled()) return false;
  static const int kBuckets[] = {1, 16, 32, 64, 128, 256, 512};
  int bucket = 0;
  for (int b : kBuckets)
    if (b >= M) { bucket = b; break; }
  if (bucket == 0) return false;
  for (const TunedPlan& t : kTuned)
    if (t.N == N && t.K == K && t.M == bucket) {   // 256x256 entries (swept on big8) run big4: >= big8 at every swept M / sk
      p = t.kind == 4 ? GemmPlan{6, 0, 0, 0, 256, 256, t.sk} : GemmPlan{t.kind, t.mt, t.nt, t.wk, t.bm, t.bn, t.sk};
      return true;
    }
  return false;
}

GemmPlan plan_gemm(int M, int N, int K) {
  if (!plan_overrides().empty()) {
    static const int kB[] = {1, 16, 32, 64, 128, 256, 512};
    int bucket = 0;
    for (int b : kB)
      if (b >= M) { bucket = b; break; }
    for (const PlanOverride& o : plan_overrides())
      if (o.N == N && o.K == K && o.M == bucket) return o.p;
  }
  GemmPlan p;
  return tuned_plan(M, N, K, p) ? p : plan_gemm_heuristic(M, N, K);
}

// LDS-tiled kernel: 16 to 128 rows per tile, K split in two until there are 448 workgroups. Where that fills the chip with more than 16 column
// tiles, up to 64 rows (a weight stream) take the split with the least of the stream (all of it at 6.3 TB/s or the busiest compute unit's
// at 40 KB a microsecond, rows of X at 0.6 of the weights' cost, and half of the latter again; 1.2 of it with one workgroup a unit whose splits
// begin whole 4 KB apart, since their reads then meet in the same memory channels) and the sums (2 us, 0.2 a split, 0.65 per MB). Over 476 M x N x K of 6
// to 64 rows with weights from memory that is 1.3 % off the best of 16 splits on average, where 448 workgroups were 20 % off (a few past a round
// of 256, or sums for nothing). us, 448 workgroups -> here: 8320 x 2048 by 32 rows 19.0 -> 13.3, by 48 21.9 -> 15.3, 16384 x 2048 by 16 18.2 -> 15.9,
// 12416 x 4096 by 32 31.1 -> 26, 5120 x 6144 by 6 21.7 -> 17.4; 15360 x 4096 by 6 and 32 stay at 24.7 and 29.5 (two splits 30.9 and 33.5).
// More than 32 rows: four stages where a compute unit has one workgroup, three where it has two (32768 x 4096 by 64 in four up to 1.24 of that).
// Packed weights have no such channels and cheaper ends: the stream alone, the sums at 1 us less (14336 x 4096 by 8 and 32 rows in two splits 22.7 and
// 24.9, in the four of row-major weights 24.7 and 28.2).
static GemmPlan plan_tile(int M, int N, int K, bool packed = false) {
  GemmPlan p{};
  const int target = 448;
  p.kind = 1;
  const bool stream = M <= 64 && 2. * N * K <= 300e6;      // (what the estimate was fitted to; 8192 x 28672 stays at eight splits)
  p.mt = M >= 512 ? 2 : stream ? 4 : 3;   // tile plans: `mt` = pipeline depth (K-tiles in flight + 1)
  if (M <= 16) { p.bm = 16; p.wk = 1; }
  else if (M <= 32) { p.bm = 32; p.wk = 1; }
  else if (M <= 64) { p.bm = 64; p.wk = 2; }
  else { p.bm = 128; p.wk = 2; }
  p.bn = 128;
  const int tiles = ((M + p.bm - 1) / p.bm) * (N / p.bn);
  int sk = 1;
  const int ktiles = K / kBK;
  while (tiles * sk < target && sk * 2 * 4 <= ktiles && sk < 16) sk *= 2;
  if (stream && tiles * sk >= 256 && tiles > 16) {
    double least = 0;
    for (int n = 1; n <= 16 && (n == 1 || ktiles >= 4 * n); ++n) {
      const int rounds = (tiles * n + 255) / 256;
      const double unit = rounds * (K / (double)n) * (256 + 1.2 * M) / 40e3;
      const double most = std::max(2. * N * K / 6.3e6, unit), sums = n > 1 ? 1 + 0.2 * n + 2.6e-6 * n * M * N : 0;
      const double us = packed ? most + sums
                               : (most + 0.5 * unit) * (rounds == 1 && 2 * K % (4096 * n) == 0 ? 1.2 : 1) + (n > 1 ? 1 + sums : 0);
      if (n == 1 || us < least) least = us, sk = n;
    }
  }
  if (M > 32 && stream && (packed ? tiles : tiles * sk) > 256) p.mt = 3;
  p.sk = sk;
  return p;
}

// The mid-M tile (gemm_mid4_kernel) that takes least, in us: rounds of 256 workgroups of 128 x 128, 128 x 256 or (half column tiles) 256 x
// 128 at 0.5, 0.7 and 0.75 a K step (0.56, 0.88 and 0.75 from 2048 channels on, where more of a step's rows meet in a memory channel) and 4 for
// the pipeline's ends, and 2 + 0.5 per MB for the sums of a split K. Over 325 M x N x K of 65 to 2000 rows what the planner takes is within 2.2 % of the
// best tile on average (33 % at most: 1500 x 4096 x 4096 on the 256 x 256 tile).
static GemmPlan plan_mid(int M, int N, int K, double& least) {
  static const struct { int bm, bn, sa, sb; double step, long_k; } kTiles[] = {{128, 128, 3, 7, 0.5, 0.56}, {128, 256, 4, 3, 0.7, 0.88}, {256, 128, 3, 4, 0.75, 0.75}};
  GemmPlan p{};
  const int steps = K / 64;
  least = 0;
  for (const auto& t : kTiles) {
    if (N % t.bn != 0 || (t.bm == 256 && N % 256 == 0)) continue;
    const long tiles = (long)((M + t.bm - 1) / t.bm) * (N / t.bn);
    for (int sk = 1; sk <= 8 && (sk == 1 || (steps >= 4 * sk && tiles * sk <= 256)); sk *= 2) {
      const double us = (double)((tiles * sk + 255) / 256) * ((K >= 2048 ? t.long_k : t.step) * steps / sk + 4) + (sk > 1 ? 2 + 2e-6 * sk * M * N : 0);
      if (least != 0 && us >= least) continue;
      least = us;
      p = GemmPlan{7, t.sa, t.sb, 0, t.bm, t.bn, sk};
    }
  }
  return p;
}

static GemmPlan plan_gemm_heuristic(int M, int N, int K) {
  GemmPlan p{};
  const int target = 448;
  const bool skinny_ok = K % 128 == 0 && N % 128 == 0;
  // (one to four rows: for the gate epilogue, and what stream_plan compares with; the products themselves stream)
  // register-streaming kernel: GEMV-like M, and short-K shapes (row-parallel projections
  // after TP splits K) where the LDS pipeline cannot fill before the K loop ends
  // (not where the results are wide: there the tiles fill the chip without splitting K, and a row of X is read once per 128 columns
  // where it was once per 32. us, skinny -> tile: 24576 x 1024 by 16 rows 14.3 -> 11.2, by 64 30 -> 13.4, 10240 x 1024 by 32 12.4 -> 10.5, 32000 x
  // 1024 by 64 40 -> 14.5, 50304 x 768 by 16 23 -> 16; 16384 x 1024 by 16 rows 10.3 and 10.5, 8192 x 1024 by 32 8.0 and 10.4)
  if (skinny_ok && M > 4 && M <= 64 && K <= 1024 && N > (M <= 16 ? 16384 : 8192)) {
    p = plan_tile(M, N, K);
    p.sk = 1;
    return p;
  }
  if (skinny_ok && (M <= 4 || (M <= 64 && K <= 1024))) {
    p.kind = 0;
    p.mt = (M + 15) / 16;
    const bool long_k = K > 4096;
    p.nt = M <= 4 ? (long_k ? 4 : 2) : 2;   // even: the SiLU epilogue pairs gate/up groups
    p.wk = long_k ? 2 : 4;
    const int blocks = N / (16 * p.nt * (4 / p.wk));
    int sk = 1;
    const int nchunks = K / 128;
    while (long_k && blocks * sk < target && sk * 2 * p.wk <= nchunks && sk < 16) sk *= 2;
    p.sk = sk;
    return p;
  }
  // 65 to 256 rows: mid-M tiles, whose rings keep K steps in flight that the 128-row tiles of plan_tile wait for, split or not.
  // us, before -> here: 100 x 2048 x 2048 12.4 -> 11.9, 256 x 2688 x 1024 17.9 -> 12.8, 65 x 6272 x 2048 22.7 -> 14.4, 256 rows 42.6 ->
  // 20.8, 128 x 8320 x 2048 35.5 -> 20.0, 180 x 12416 x 4096 71.7 -> 35.3; not where few rows split a long K in 16 and fit one round of workgroups (65 and
  // 128 x 2048 x 6144 13.6 and 16.9, on mid-M tiles 17.1 and 19.8, 65 x 1024 x 8192 18.0 and 21.1, 65 x 2048 x 4096 12.6 and 14.6; 65 x 1408 x 4096 16.1 and 15.3, two rounds
  // 65 x 4096 x 6144 28.6 and 21.1, 128 x 3072 x 8192 32.5 and 24.7).
  double mid = 0;
  const bool mid_ok = M > 64 && N % 128 == 0 && K % 64 == 0 && K >= 256;
  const GemmPlan pm = mid_ok ? plan_mid(M, N, K, mid) : GemmPlan{};
  if (mid_ok && M <= 256 && !(M <= 128 && N <= 2048 && (long)N * K >= 8 << 20 && plan_tile(M, N, K).sk == 16)) return pm;
  // 256 x 256 tile from two K steps on (its pipeline's least)
  if (M > 256 && N % 128 == 0 && K % 64 == 0 && K >= 128 && (N % 256 == 0 || (N > 1024 && K >= 256))) {
    // prefill / large batch: the 256x256 one-wave-per-SIMD tile (gemm_big4_kernel: 1.52-1.55 PF at M = 8192 on the 70B
    // projections, 6-10 % over the 8-phase gemm_big8_kernel and ahead of it at M = 256-2048 too, profiles/r5_gemm_big4/). Split
    // K where that pays for the partial sums it writes and reads, in units of a K step of 64 (1.15 us): rounds of 256
    // workgroups times (steps + 8 for the pipeline's ends), plus 5 and 0.07 per tile and split for the sums, twice that beyond
    // 512 of them (128 MB no longer stay in the cache); unsplit, a last round of at most 128 tiles runs as half tiles
    // (big4_halved) in 0.62 of the steps, behind other rounds in 0.75. Unsplit, two, four and eight splits, us: 425 x 1024 x
    // 1024 (8 tiles) 17, 24; 1190 x 1024 x 2048 (20) 26, 33, 29; 999 x 2048 x 8192 (32) 82, 83, 56, 53; 724 x 4096 x 4096 (48)
    // 45, 54, 43, 65; 942 x 4096 x 4096 (64) 48, 56, 49, 71; 275 x 10240 x 8192 (80) 98, 87, 102; 753 x 8192 x 8192 (96) 109,
    // 106, 131; 756 x 10752 x 2048 (126) 38, 55, 77; 2991 x 4096 x 14336 (192) 261, 322, 320; 2585 x 6144 x 4096 (264) 138,
    // 181; 2265 x 8192 x 28672 (288) 927, 918; 2838 x 8192 x 8192 (384) 275, 376. At most 1024 tiles of partial sums: 256 MB of
    // workspace, and a need that grows with whole tiles only (ops.reserve_workspace).
    p.kind = 6;
    p.mt = 0;
    p.bm = p.bn = 256;
    const int tiles = ((M + 255) / 256) * ((N + 255) / 256), steps = K / 64;
    p.sk = 1;
    double best = 0, whole = 0;      // (whole: with the last round as whole tiles)
    for (int sk = 1; sk <= 8 && (sk == 1 || (steps >= sk * 8 && tiles * sk <= 1024)); sk *= 2) {
      const double sums = sk == 1 ? 0 : 5 + (tiles * sk <= 512 ? 0.07 : 0.14) * tiles * sk;
      const int halved = sk == 1 ? big4_halved(tiles) : 0;
      const double t = (double)(((tiles - halved) * sk + 255) / 256) * ((double)steps / sk + 8) +
                       (halved ? (tiles > 256 ? 0.75 : 0.62) * steps + 8 : 0) + sums;
      const double tw = (double)((tiles * sk + 255) / 256) * ((double)steps / sk + 8) + sums;
      if (sk == 1 || tw < whole) whole = tw;
      if (sk == 1 || t < best) {
        best = t;
        p.sk = sk;
      }
    }
    // The mid-M tiles where they take 15 % less (what the estimates are off by), this tile's time in us: 1.13 a K step (half tiles
    // 0.72 or, behind other rounds, 0.85) and 5 a round, sums as theirs. Few rows or columns leave it most compute units idle or many sums. us, before -> here: 937 x 4096 x 4096 49.5
    // -> 37.7, 1000 x 2048 x 2048 25.5 -> 20.3, 500 rows 23.9 -> 17.4, 700 x 3072 x 2048 25.7 -> 20.4, 1400 x 2048 x 4096 42 -> 36, 700 x 1024 x 4096
    // 27.2 -> 20.9, 400 x 2688 x 1024 25.4 -> 12.9, 257 x 2688 x 1024 17.8 -> 12.6, 300 x 1152 x 4096 24.7 -> 16.4, 320 x 8320 x 2048 41.6 -> 28.3, 1000 x 8192 x
    // 8192 stays (102 and 105). Where a reader took a split's sums as they are a step saves less: with the norm behind 850 and 1000 x 4096 x 4096 49.1 -> 46.6
    // and 52.8 -> 48.9. With a row kernel behind that sums the splits: 300 rows of 1024 x 1024 19.5 -> 13.9, 2048 x 2048 24.7 -> 18.9, 4096 x 2048
    // 45.6 -> 25.3, 2048 x 4096 26.7 -> 24.0, 4096 x 6144 40.9 -> 39.2.
    if (mid_ok) {
      const int halved = p.sk == 1 ? big4_halved(tiles) : 0;
      const double big = (double)(((long)(tiles - halved) * p.sk + 255) / 256) * (1.13 * steps / p.sk + 5) +
                         (halved ? (tiles > 256 ? 0.85 : 0.72) * steps + 5 : 0) + (p.sk > 1 ? 2 + 2e-6 * p.sk * M * N : 0);
      if (mid < 0.85 * big) return pm;
    }
    if (N % 256 == 0) return p;
    // N % 256 == 128: half of the last column tile is wasted and 128 x 128 tiles have four times as many workgroups, two of
    // them per compute unit. Their time in us, by rounds of 512 workgroups: (steps per split + 5) a round, and 6 + 0.02 per
    // tile and split for the sums of a split K; the unit above is 1.22 us here. Over 324 shapes of 300 to 8192 rows the choice
    // takes at most 9 % more than the 128 x 128 tiles. 128 x 128 and 256 x 256 tiles, us: 8192 x 8320 x 2048 348 and 253, 6200 x
    // 6272 x 2048 200 and 153, 1000 x 4224 x 1024 37 and 30; 300 x 1408 x 1024 15 and 24, 1838 x 4224 x 1024 24 and 31, 1838 x 8320
    // x 4096 139 and 164. Below 256 channels the small tiles are ahead nearly everywhere (4000 x 1152 x 128 10 and 15).
    const GemmPlan q = plan_tile(M, N, K);
    const long wgs = (long)((M + 127) / 128) * (N / 128) * q.sk;
    const double tq = (double)((wgs + 511) / 512) * ((double)steps / q.sk + 5) + (q.sk > 1 ? 6 + 0.02 * wgs : 0);
    return tq <= 1.22 * whole ? q : p;
  }
  return plan_tile(M, N, K);
}

static size_t plan_ws_bytes(const GemmPlan& p, int M, int N) {
  return p.sk > 1 ? kCounterBytes + (size_t)p.sk * M * N * sizeof(float) : 0;
}

// A row scale with a half column tile: the 256 x 256 tile's epilogue has none, the 128-row tiles' has
static bool rowscale_on_tile(const GemmPlan& p, int N) { return p.kind == 6 && N % 256 != 0; }

// Packed weights of up to 64 rows take the split of their own estimate where no entry of the table has the shape
static bool packed_tile(const GemmPlan& p, int M, int N, int K) {
  GemmPlan t;
  return p.kind == 1 && p.sk > 1 && M <= 64 && N % 256 == 0 && plan_overrides().empty() && !tuned_plan(M, N, K, t);
}

// Enough for the tuned plan, for the plans it may fall back to (below), for packed weights' splits and for the plan of five rows where those take it.
size_t gemm_workspace_bytes(int M, int N, int K) {
  const GemmPlan h = plan_gemm_heuristic(M, N, K);
  const size_t a = plan_ws_bytes(plan_gemm(M, N, K), M, N), b = plan_ws_bytes(h, M, N);
  return std::max({a, b, rowscale_on_tile(h, N) ? plan_ws_bytes(plan_tile(M, N, K), M, N) : 0,
                   packed_tile(h, M, N, K) ? plan_ws_bytes(plan_tile(M, N, K, true), M, N) : 0,
                   gemm_packed_first(M, N, K) ? gemm_workspace_bytes(5, N, K) : 0});
}

// The most that any number of rows up to M asks for. Each is asked: fewer rows may split K more inside a row tile (2048 x 1024 4 MB at 256
// rows, 8 at 244), and tiles change between any two (1 ms for 8192 rows). Beyond 512 tiles of 256 x 256 nothing is split.
size_t gemm_workspace_bound(int M, int N, int K) {
  const long split = 256L * std::max(2, 512 / ((N + 255) / 256));
  size_t need = 0;
  for (int m = 1; m <= (int)std::min<long>(M, split); ++m) need = std::max(need, gemm_workspace_bytes(m, N, K));
  return need;
}

// `dry`: validate only (the plan is supported for this shape/epilogue) without launching.
static int run_plan(const GemmPlan& p, const bf16* X, long ldx, const bf16* W, long ldw, int M,
                    int N, int K, int epi, const bf16* bias, bf16* out, long ldo, float* ws,
                    hipStream_t stream, bool dry = false, bool defer = false,
                    const RowScale* rs = nullptr, bool packed = false) {
  const RowScale rsc = rs ? *rs : RowScale{nullptr, 0, 0.f, 0.f};
  if (rs != nullptr && p.kind != 1 && p.kind != 3 && p.kind != 5 && p.kind != 7) return -4;   // row scale: tile / ring / mid epilogues
  if (epi == EPI_SILU_GATE && (p.kind != 1 || p.sk != 1)) return -4;   // gate: tile epilogue, no slabs
  // packed (pack_w256) weights: the tile plans mark it with nt = 1, the others take it here
  if (packed && p.kind != 5 && p.kind != 7 && p.kind != 8) return -5;
  if (p.kind == 4) {
    // 8-phase big tile: every split needs >= 2 K-tiles of 64
    if (N % 256 != 0 || K % 64 != 0 || K / 64 < 2 * p.sk) return -1;
    if (!dry) run_big8(X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, ws, p.sk, stream);
  } else if (p.kind == 7) {
    // mid-M one-wave-per-SIMD tile: plan {7, SA (activation ring), SB (weight ring), 0, BM, BN, sk}
    if (N % p.bn != 0 || K % 64 != 0 || K / 64 < p.sk) return -1;
    bool done = false;
#define MID4_CASE(BM_, BN_, SA_, SB_)                                                               \
  if (!done && p.bm == BM_ && p.bn == BN_ && p.mt == SA_ && p.nt == SB_) {                          \
    if (!dry && packed) run_mid4<BM_, BN_, SA_, SB_, true>(X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, ws, p.sk, stream, rsc); \
    else if (!dry) run_mid4<BM_, BN_, SA_, SB_>(X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, ws, p.sk, stream, rsc); \
    done = true;                                                                                   \
  }
    MID4_CASE(128, 128, 4, 6) MID4_CASE(128, 128, 3, 7) MID4_CASE(128, 128, 2, 8)
    MID4_CASE(256, 128, 3, 4) MID4_CASE(256, 128, 2, 6) MID4_CASE(128, 256, 4, 3) MID4_CASE(128, 256, 2, 4)
#undef MID4_CASE
    if (!done) return -2;
  } else if (p.kind == 6) {
    // one-wave-per-SIMD 256x256 tile: every split needs >= 2 K-tiles of 64
    if (N % 128 != 0 || K % 64 != 0 || K / 64 < 2 * p.sk) return -1;
    if (!dry) run_big4(X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, ws, p.sk, stream);

  } else if (p.kind == 5) {
    // mid-M 8-wave staggered GEMM: plan {5, SW (weight ring), SX (activation ring; 0 = SW), 0,
    // BM, BN, sk}
    if (N % p.bn != 0 || K % kBK != 0 || K / kBK < p.sk) return -1;
    if (epi_halves(epi) && p.bn * p.bm / 512 % 32 != 0) return -1;
    const int sx = p.nt > 0 ? p.nt : p.mt;
    bool done = false;
#define MID_CASE(BM_, BN_, SX_, SW_)                                                              \
  if (!done && p.bm == BM_ && p.bn == BN_ && sx == SX_ && p.mt == SW_) {                           \
    if (!dry && packed) run_mid8<BM_, BN_, SX_, SW_, true>(X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, ws, p.sk, stream, rsc); \
    else if (!dry) run_mid8<BM_, BN_, SX_, SW_>(X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, ws, p.sk, stream, rsc); \
    done = true;                                                                                   \
  }
    MID_CASE(256, 128, 3, 3) MID_CASE(256, 128, 2, 6) MID_CASE(256, 128, 3, 4)
    MID_CASE(128, 256, 3, 3) MID_CASE(128, 256, 2, 4)
    MID_CASE(128, 128, 4, 4) MID_CASE(128, 128, 3, 3) MID_CASE(128, 128, 3, 6) MID_CASE(128, 128, 2, 8)
    MID_CASE(128, 128, 2, 2)   // 64 KiB: two workgroups per CU
#undef MID_CASE
    if (!done) return -2;
  } else if (p.kind == 3) {
    // decode ring GEMM: plan {3, SW (weight ring depth), waves, waves along M, BM, BN, sk}
    if (N % p.bn != 0 || K % kBK != 0 || K / kBK < p.sk * 2) return -1;
    const int nwn = p.wk > 0 ? p.nt / p.wk : 0;
    if (epi_halves(epi) && (nwn <= 0 || (p.bn / nwn) % 32 != 0)) return -1;
    bool done = false;
#define DEC_CASE(BM_, BN_, NWM_, NWN_, SW_)                                                      \
  if (!done && p.bm == BM_ && p.bn == BN_ && p.wk == NWM_ && p.nt == NWM_ * NWN_ && p.mt == SW_) { \
    if (!dry) run_dec<BM_, BN_, NWM_, NWN_, SW_>(X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, ws, p.sk, stream, rsc); \
    done = true;                                                                                 \
  }
    DEC_CASE(128, 224, 8, 1, 4) DEC_CASE(128, 224, 8, 1, 3) DEC_CASE(128, 256, 8, 1, 3)
    DEC_CASE(128, 256, 4, 2, 3) DEC_CASE(128, 128, 8, 1, 5) DEC_CASE(128, 128, 4, 2, 5)
    DEC_CASE(128, 160, 8, 1, 4) DEC_CASE(128, 80, 8, 1, 6) DEC_CASE(128, 64, 8, 1, 8)
    DEC_CASE(128, 64, 4, 2, 8) DEC_CASE(64, 128, 4, 2, 6) DEC_CASE(64, 256, 4, 2, 4)
    DEC_CASE(64, 224, 4, 1, 4) DEC_CASE(64, 160, 4, 2, 5) DEC_CASE(64, 64, 4, 2, 8)
#undef DEC_CASE
    if (!done) return -2;
  } else if (p.kind == 8) {
    // streamed product of few rows: plan {8, row tiles, column tiles, waves, chunks in flight, fold, 1}
    const int fold = p.bn;
    if ((fold != 1 && fold != 2 && fold != 4) || p.sk != 1) return -2;
    if (K % (64 * fold) != 0 || N % (16 / fold * p.nt) != 0 || M > 16 / fold * p.mt) return -1;
    if (epi == EPI_SILU_GATE || (epi_halves(epi) && N % 32 != 0)) return -1;
    bool done = false;
#define ST_CASE(MT_, NT_, NW_, U_, F_)                                                                         \
  if (!done && p.mt == MT_ && p.nt == NT_ && p.wk == NW_ && p.bm == U_ && fold == F_) {                        \
    if (!dry) run_stream<MT_, NT_, NW_, U_, F_>(X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, stream, packed); \
    done = true;                                                                                               \
  }
    ST_CASE(1, 1, 4, 4, 4) ST_CASE(1, 1, 4, 4, 2) ST_CASE(1, 1, 8, 4, 2) ST_CASE(1, 2, 8, 4, 2)
    ST_CASE(1, 1, 4, 4, 1) ST_CASE(1, 1, 8, 4, 1) ST_CASE(1, 2, 8, 4, 1) ST_CASE(2, 1, 8, 4, 1)
#undef ST_CASE
    if (!done) return -2;
  } else if (p.kind == 0) {
    if (K % 128 != 0 || M > 16 * p.mt) return -1;
    if (N % (16 * p.nt * (4 / p.wk)) != 0) return -1;
    if (epi_halves(epi) && p.nt % 2 != 0) return -1;
    if (p.sk > 1 && N / (16 * p.nt * (4 / p.wk)) > kSplitCounters) return -1;
    bool done = false;
#define SK_CASE(MT_, NT_, WK_)                                                                   \
  if (!done && p.mt == MT_ && p.nt == NT_ && p.wk == WK_) {                                       \
    if (!dry) run_skinny<MT_, NT_, WK_>(X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, ws, p.sk, stream); \
    done = true;                                                                                  \
  }
#define SK_WK(MT_, NT_) SK_CASE(MT_, NT_, 1) SK_CASE(MT_, NT_, 2) SK_CASE(MT_, NT_, 4)
    SK_WK(1, 1) SK_WK(1, 2) SK_WK(1, 4) SK_WK(2, 1) SK_WK(2, 2) SK_WK(2, 4)
    SK_WK(3, 2) SK_WK(4, 1) SK_WK(4, 2) SK_WK(4, 4)
#undef SK_WK
#undef SK_CASE
    if (!done) return -2;
  } else if (p.kind == 1 && p.nt == 1) {
    // tile plan over a K-tile-blocked weight (pack_w256 layout): 16 / 32 / 64-row tiles of 128 /
    // 256 columns (the packed layout only changes the weight stage's addresses, so every decode
    // tile the row-major table picks, down to the B = 1 bucket, has its packed twin)
    if (N % 256 != 0 || K % 64 != 0 || (p.bm != 16 && p.bm != 32 && p.bm != 64) || (p.bn != 128 && p.bn != 256) ||
        K / kBK < p.sk)
      return -1;
    if (p.sk > 1 && (long)((M + p.bm - 1) / p.bm) * (N / p.bn) > kSplitCounters) return -1;
    bool done = false;
    const int st = p.mt > 0 ? p.mt : 2;
#define TLP_CASE(BM_, BN_, WMW_, ST_)                                                                 \
  if (!done && p.bm == BM_ && p.bn == BN_ && p.wk == WMW_ && st == ST_) {                             \
    if (!dry) run_tile<BM_, BN_, WMW_, ST_, true>(X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, ws, p.sk, stream, rsc); \
    done = true;                                                                                      \
  }
#define TLP_ST(BM_, BN_, WMW_) TLP_CASE(BM_, BN_, WMW_, 2) TLP_CASE(BM_, BN_, WMW_, 3) TLP_CASE(BM_, BN_, WMW_, 4)
    TLP_ST(16, 128, 1) TLP_ST(16, 256, 1) TLP_ST(32, 128, 1) TLP_ST(32, 256, 1)
    TLP_ST(64, 128, 1) TLP_ST(64, 128, 2) TLP_ST(64, 256, 1) TLP_ST(64, 256, 2)
#undef TLP_ST
#undef TLP_CASE
    if (!done) return -2;
  } else {
    if (N % p.bn != 0 || K % kBK != 0) return -1;
    if (p.sk > 1 && (long)((M + p.bm - 1) / p.bm) * (N / p.bn) > kSplitCounters) return -1;
    bool done = false;
    const int st = p.mt > 0 ? p.mt : 2;   // tile plans reuse `mt` as the pipeline depth
#define TL_CASE(BM_, BN_, WMW_, ST_)                                                            \
  if (!done && p.bm == BM_ && p.bn == BN_ && p.wk == WMW_ && st == ST_) {                       \
    if (!dry) run_tile<BM_, BN_, WMW_, ST_>(X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, ws, p.sk, stream, rsc); \
    done = true;                                                                                \
  }
#define TL_ST(BM_, BN_, WMW_) TL_CASE(BM_, BN_, WMW_, 2) TL_CASE(BM_, BN_, WMW_, 3) TL_CASE(BM_, BN_, WMW_, 4)
    TL_ST(16, 128, 1) TL_ST(16, 256, 1) TL_ST(32, 128, 1) TL_ST(32, 256, 1)
    TL_ST(64, 128, 1) TL_ST(64, 128, 2) TL_ST(64, 256, 1) TL_ST(64, 256, 2)
    TL_ST(128, 128, 2) TL_ST(128, 256, 2)
    // CU-balanced decode tiles: N/224 or N/160 tiles x split-K land on exactly 256 workgroups
    // for the Llama-3-70B projections (gate/up 57344 = 256 x 224, QKV 10240 = 64 x 160)
    TL_ST(64, 224, 4) TL_ST(64, 160, 4)
#undef TL_ST
#undef TL_CASE
    if (!done) return -2;
  }
  if (p.sk > 1 && !dry && !defer) {
    const int nout = epi_halves(epi) ? N / 2 : N;
    long total = (long)M * nout;
    int grid = (int)((total + 255) / 256);
    if (grid > 4096) grid = 4096;
    gemm_splitk_reduce_kernel<<<grid, 256, 0, stream>>>(splitk_part(ws), p.sk, M, N, epi, bias,
                                                         out, ldo);
  }
  return 0;
}

// Whether a plan's kernel finds rows ldx and ldw apart. Those that load through buffer descriptors (kinds 4 to 7) have a row's place in a
// tile as 32-bit byte offset below 2^31, and what lies behind rows * ld bytes reads as zeros: rows that overlap, or are one and the same
// (an expanded vector), as much as rows far apart. The others address each row in 64 bits.
static bool plan_reaches(const GemmPlan& p, int K, long ldx, long ldw) {
  if (p.kind < 4 || p.kind > 7) return true;
  const bool mid = p.kind == 5 || p.kind == 7;
  const long reach = 0x7fffffffL / 2, bm = mid ? p.bm : 256, bn = mid ? p.bn : 256;
  return ldx >= K && ldw >= K && ldx <= reach / bm && ldw <= reach / bn;
}

int launch_gemm_plan(const GemmPlan& p, const bf16* X, long ldx, const bf16* W, long ldw, int M,
                     int N, int K, int epi, const bf16* bias, bf16* out, long ldo, float* ws,
                     size_t ws_bytes, hipStream_t stream) {
  if (M <= 0) return 0;
  if (p.sk > 1 && (ws == nullptr || ws_bytes < kCounterBytes + (size_t)p.sk * M * N * sizeof(float)))
    return -3;
  if (!plan_reaches(p, K, ldx, ldw)) return -6;
  return run_plan(p, X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, ws, stream);
}

// Whether a product of few rows streams (gemm_stream_kernel) in place of plan `base`, and how: of the tiles that take M rows the one
// whose busiest compute unit has the least to take in, its weight rows and, at 0.6 of their cost (from the L2), the rows of X past the first
// once per workgroup (1 to 3 % off the best tile on average over 135 N x K by six row counts).
// Up to four rows always, but where a split tile's sums cost nothing extra because their reader takes them as they are: it reads as
// fast then (4096 x 14336 20.0 and 21.2 us, 6144 x 4096 by four rows 10.7 and 12.2) except for one row up to 8192 channels (10240 x
// 8192 28.5 and 26.9). Up to eight rows where X does not weigh in: 4096 channels and 10240 columns (5120 x 2048 11.4 -> 8.3 us, 4096 x
// 4096 9.9 -> 9.0; 14336 x 4096 31.7 and 30.7, but 22.7 on tiles over
// packed weights, which streams would go ahead of), in place of split sums 4096 x 4096 or 2048 channels (2048 x 2048 7.3 -> 4.6, read as
// they are 5.1). Up to 16 rows to 1024 channels (1024 x 1024 5.9 -> 4.3), and to 2048 in place of split sums of a product that widens
// its rows, to two rounds of its tiles (3072 x 2048 9.6 -> 7.0, 8320 x 2048 15.8 and 11.7; those of one that does not are read as they are:
// 2048 x 2048 5.4 and 6.6). Up to 32 rows to 1024 channels
// and 4096 columns (2688 x 1024 7.4 -> 5.4).
static bool stream_plan(int M, int N, int K, int epi, const GemmPlan& base, GemmPlan& p) {
  if (M > 32 || K % 128 != 0 || epi == EPI_SILU_GATE || !plan_overrides().empty()) return false;
  const bool split = base.sk > 1;
  if (M <= 4) {
    if (split && base.kind == 1 && (M > 1 || K > 8192)) return false;
  } else if (M <= 8) {
    if (K > 4096 || N > 10240 || (split && K > 2048 && N > 4096)) return false;
  } else if (M <= 16) {
    if (!(!split && K <= 1024 && N <= 8192) && !(split && K <= 2048 && N > K && N <= 8192)) return false;
  } else if (split || K > 1024 || N > 4096) {
    return false;
  }
  double best = 0;
  const auto tile = [&](int rows, GemmPlan q) {
    const double cost = (N / rows + 255) / 256 * (rows + 0.6 * (M - 1));
    if (best != 0 && cost >= best) return;
    best = cost;
    p = q;
  };
  if (M > 16) {
    p = GemmPlan{8, 2, 1, 8, 4, 1, 1};
  } else if (M > 8) {
    tile(16, GemmPlan{8, 1, 1, K <= 1024 ? 4 : 8, 4, 1, 1});
    tile(32, GemmPlan{8, 1, 2, 8, 4, 1, 1});
  } else {
    if (M <= 4 && K % 256 == 0) tile(4, GemmPlan{8, 1, 1, 4, 4, 4, 1});
    tile(8, GemmPlan{8, 1, 1, K < 2048 ? 4 : 8, 4, 2, 1});
    if (K >= 2048) tile(16, GemmPlan{8, 1, 2, 8, 4, 2, 1});
  }
  return true;
}

// The plan for this call: the tuned/heuristic plan, or the heuristic one when a table entry
// measured for another epilogue cannot run this one (e.g. odd skinny NT with SiLU), or the tile plan for a row scale;
// for few rows the streamed product.
static GemmPlan select_plan(int M, int N, int K, int epi, bool row_scale = false) {
  GemmPlan p = plan_gemm(M, N, K), q;
  if (run_plan(p, nullptr, 0, nullptr, 0, M, N, K, epi, nullptr, nullptr, 0, nullptr, nullptr, true) != 0)
    p = plan_gemm_heuristic(M, N, K);
  if (row_scale) return rowscale_on_tile(p, N) ? plan_tile(M, N, K) : p;
  return stream_plan(M, N, K, epi, p, q) ? q : p;
}

// The plan for operands with these row pitches: where its kernel does not reach the rows, 128-row tiles, K split as far as the workspace holds
static GemmPlan call_plan(int M, int N, int K, int epi, bool row_scale, long ldx, long ldw, size_t ws_bytes) {
  const auto parts = [&](int sk) { return kCounterBytes + (size_t)sk * M * N * sizeof(float); };
  GemmPlan p = select_plan(M, N, K, epi, row_scale);
  if (!plan_reaches(p, K, ldx, ldw)) {
    p = plan_tile(M, N, K);
    while (p.sk > 1 && ws_bytes < parts(p.sk)) --p.sk;
  }
  if (p.sk > 1 && ws_bytes < parts(p.sk)) p.sk = 1;
  return p;
}

GemmPlan gemm_call_plan(int M, int N, int K, int epi, long ldx, long ldw) {
  return call_plan(M, N, K, epi, false, ldx, ldw, ~(size_t)0);
}

bool gemm_streams(int M, int N, int K, int epi) { return M > 0 && select_plan(M, N, K, epi).kind == 8; }

// Two to four rows over packed weights of many columns run as five do: their tiles read them faster than streams take the rows of X in. us by 2
// rows, streams and tiles: 28672 x 4096 44.7 and 37.4, 57344 x 8192 149 and 145, 8192 x 8192 27.1 and 23.9; 4096 x 4096 9.1 and 10.4,
// 128256 x 4096 155 and 160.
bool gemm_packed_first(int M, int N, int K) { return M >= 2 && M <= 4 && N >= 8192 && N <= 65536 && N % 256 == 0 && K >= 4096; }

int gemm_rowscale_check(int M, int N, int K, int epi) {
  if (M <= 0) return 0;
  const RowScale probe{nullptr, 0, 0.f, 0.f};
  if (gemm_streams(M, N, K, epi)) return -4;      // streamed without one
  // (whole column tiles of many rows: behind a norm in one launch, whichever tile runs)
  GemmPlan t;
  if (M > 256 && N % 256 == 0 && !tuned_plan(M, N, K, t)) return -4;
  return run_plan(select_plan(M, N, K, epi, true), nullptr, 0, nullptr, 0, M, N, K, epi, nullptr, nullptr, 0,
                  nullptr, nullptr, true, false, &probe);
}

// Grouped expert GEMM (MoE): BM x 128 tile (BM = 64 or 128 rows per expert tile, chosen by
// the caller from the expected rows per expert), 3-stage pipeline; grid = (max tiles, sk,
// N / 128) with the device tile list deciding which workgroups run. sk > 1 splits K and
// writes f32 slabs part[sk][slots][N] (consumed by moe_combine_slabs: the split-K reduce is
// fused into the weighted combine) — decode-sized expert batches otherwise leave most CUs
// idle on the down projection (N = hidden: 32 column tiles per expert tile).
template <int BM>
static int launch_grouped_bm(const bf16* X, long ldx, const bf16* W, long ldw, long w_estride, int N,
                             int K, int epi, const int* rows, const int4* tiles, const int* count,
                             int max_tiles, int slots, int sk, float* part, bf16* out, long ldo,
                             hipStream_t stream) {
  constexpr int BN = 128, WMW = 2, ST = 3;
  const size_t lds = (size_t)ST * (BM + BN) * kBK * 2;
  static bool attr_set = false;
  if (!attr_set && lds > 65536) {
    hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_tile_kernel<BM, BN, WMW, ST, true>),
                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    attr_set = true;
  }
  dim3 grid(max_tiles, sk, N / BN);
  gemm_tile_kernel<BM, BN, WMW, ST, true><<<grid, kTileThreads, lds, stream>>>(
      X, ldx, W, ldw, slots, N, K, epi, nullptr, out, ldo, sk > 1 ? part : nullptr, rows,
      tiles, count, w_estride);
  return 0;
}

// 256-row expert tiles: the one-wave-per-SIMD tile, but for weights whose rows are a multiple of 32 KB apart: the 256 rows of a K
// step then lie in one memory channel, and the tile, with less in flight, waits for it. 8 experts' down projection of 4096 x 14336,
// rows 8 x 28 KB apart (7 x 32 KB) and 128 bytes more (4 KB: 235 at 300 tokens, 580 at 2870), us: big4 at 300, 976, 2870, 5000 tokens
// 361, 433, 727, 1201 and 220, 315, 559, 956; big8 293, 347, 667, 1033 and 284, 327, 653, 1014. Its rows are offsets of 32 bits from
// X (gathered) or from a tile's first row, those of the other one addresses.
bool grouped_on_big4(long x_rows, long ldx, long ldw, bool silu, bool gathered) {
  const long reach = (gathered ? x_rows : std::min(x_rows, 256L)) * ldx * 2;
  return reach < 0x7fffffffL && (silu || ldw * 2 % 32768 != 0);
}

int launch_gemm_grouped(const bf16* X, long x_rows, long ldx, const bf16* W, long ldw, long w_estride, int N,
                        int K, int epi, const int* rows, const int4* tiles, const int* count,
                        int max_tiles, bf16* out, long ldo, hipStream_t stream, int bm, int slots,
                        int sk, float* part) {
  if (N % 128 != 0 || K % kBK != 0 || max_tiles <= 0) return -1;
  if (epi != EPI_NONE && epi != EPI_SILU) return -1;
  if (sk < 1 || sk > K / kBK || (sk > 1 && (part == nullptr || epi != EPI_NONE || slots <= 0))) return -2;
  if (bm == 256) {
    // prefill-scale expert batches: a 256x256 tile over the tile list, no split
    if (N % 256 != 0 || K / 64 < 2 || sk != 1) return -2;
    static bool attr = false;
    if (!attr) {
      hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_big8_kernel<true>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, kB8LdsBytes);
      for (const void* k : {reinterpret_cast<const void*>(&gemm_big4_kernel<1, EPI_NONE>),
                            reinterpret_cast<const void*>(&gemm_big4_kernel<1, EPI_SILU>)})
        hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kB4LdsBytes);
      attr = true;
    }
    dim3 grid(max_tiles * (N / 256), 1);
    if (grouped_on_big4(x_rows, ldx, ldw, epi == EPI_SILU, rows != nullptr))
      (epi == EPI_SILU ? &gemm_big4_kernel<1, EPI_SILU> : &gemm_big4_kernel<1, EPI_NONE>)
          <<<dim3(big4_grid((long)max_tiles * (N / 256) + 128)), kB4Threads, kB4LdsBytes, stream>>>(
              X, ldx, W, ldw, 0, N, K, nullptr, out, ldo, nullptr, 0, rows, tiles, count, w_estride, ExpertArgs());
    else
      gemm_big8_kernel<true><<<grid, kB8Threads, kB8LdsBytes, stream>>>(
          X, ldx, W, ldw, max_tiles * 256, N, K, epi, nullptr, out, ldo, nullptr, rows, tiles, count, w_estride);
    return 0;
  }
  if (bm == 128)
    return launch_grouped_bm<128>(X, ldx, W, ldw, w_estride, N, K, epi, rows, tiles, count, max_tiles,
                                  slots, sk, part, out, ldo, stream);
  if (bm == 64)
    return launch_grouped_bm<64>(X, ldx, W, ldw, w_estride, N, K, epi, rows, tiles, count, max_tiles,
                                 slots, sk, part, out, ldo, stream);
  return -3;
}

// 256-row groups of the score-routed experts on gemm_big4_kernel (bfly_mixers.h)
void launch_moe_big(bool down, const bf16* X, long ldx, const bf16* W, int N, int K, int max_tiles, const int* ntiles,
                    bf16* out, long ldo, const ExpertArgs& ex, hipStream_t stream) {
  static bool attr = false;
  if (!attr) {
    for (const void* k : {reinterpret_cast<const void*>(&gemm_big4_kernel<2, EPI_GLU>),
                          reinterpret_cast<const void*>(&gemm_big4_kernel<2, EPI_RELU2>),
                          reinterpret_cast<const void*>(&gemm_big4_kernel<3, EPI_NONE>)})
      hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kB4LdsBytes);
    attr = true;
  }
  const dim3 grid(big4_grid((long)max_tiles * (N / 256) + 128), 1);      // (the kernel counts the tiles and halves up to 128 of them)
  if (down)
    gemm_big4_kernel<3, EPI_NONE><<<grid, kB4Threads, kB4LdsBytes, stream>>>(X, ldx, W, K, 0, N, K, nullptr, out, ldo, nullptr, 0,
                                                                   nullptr, nullptr, ntiles, (long)N * K, ex);
  else
    (ex.plain ? &gemm_big4_kernel<2, EPI_RELU2> : &gemm_big4_kernel<2, EPI_GLU>)<<<grid, kB4Threads, kB4LdsBytes, stream>>>(
        X, ldx, W, K, 0, N, K, nullptr, out, ldo, nullptr, 0, nullptr, nullptr, ntiles, (long)N * K, ex);
}

int gemm_check(int M, int N, int K, int epi) {
  if (M <= 0) return 0;
  return run_plan(select_plan(M, N, K, epi), nullptr, 0, nullptr, 0, M, N, K, epi, nullptr, nullptr,
                  0, nullptr, nullptr, true);
}

int launch_gemm_deferred(const bf16* X, long ldx, const bf16* W, long ldw, int M, int N, int K,
                         bf16* out, long ldo, float* ws, size_t ws_bytes, hipStream_t stream,
                         const RowScale* rs) {
  if (M <= 0) return 1;
  const GemmPlan p = call_plan(M, N, K, EPI_NONE, rs != nullptr, ldx, ldw, ws ? ws_bytes : 0);
  const bool defer = p.sk > 1;
  const int rc = run_plan(p, X, ldx, W, ldw, M, N, K, EPI_NONE, nullptr, out, ldo, ws, stream,
                          false, defer, rs);
  if (rc != 0) return rc;
  return defer ? p.sk : 1;
}

size_t gemm_slab_offset_floats() { return kCounterBytes / sizeof(float); }

void launch_splitk_reduce(const float* part, int sk, int M, int N, bf16* out, long ldo,
                          hipStream_t stream) {
  long total = (long)M * N;
  int grid = (int)((total + 255) / 256);
  if (grid > 4096) grid = 4096;
  gemm_splitk_reduce_kernel<<<grid, 256, 0, stream>>>(part, sk, M, N, EPI_NONE, nullptr, out, ldo);
}

int launch_gemm(const bf16* X, long ldx, const bf16* W, long ldw, int M, int N, int K, int epi,
                const bf16* bias, bf16* out, long ldo, float* ws, size_t ws_bytes,
                hipStream_t stream, const RowScale* rs) {
  if (M <= 0) return 0;
  const GemmPlan p = call_plan(M, N, K, epi, rs != nullptr, ldx, ldw, ws ? ws_bytes : 0);
  return run_plan(p, X, ldx, W, ldw, M, N, K, epi, bias, out, ldo, ws, stream, false, false, rs);
}

// Decode GEMM over a K-tile-blocked copy of the weight (layout [N/256][K/64][256][64], made
// once by the engine when HBM allows, models/transformer.pack_decode_weights): the plan the
// row-major weight would run (streams of few rows, 16 / 32 / 64-row tiles and the mid-M kernels of kinds 5 / 7, with
// their split-K; EPI_SILU_GATE: the gate plan) on the packed copy. Each 128-row weight stage is then one 16 KiB run of memory instead of 128
// runs of 128 B a row pitch apart: the Llama-3-70B gate/up GEMM at M = 64 in 145 against
// 158 us, bitwise the same result (tools/packed_probe.py). Returns < 0 (nothing launched)
// when the plan for this shape is not such a tile plan: the caller then uses the row-major
// weight. `dry`: only report whether it applies.
// Packed-weight plans that differ from the row-major table's (tools/packed_probe.py --sweep,
// isolated, weights rotating through HBM; profiles/r6_packed/sweep_m64.jsonl): kind -1 = keep
// this shape on the row-major weight (its row-major plan is faster than any packed one).
struct PackedTuned { int N, K, M; GemmPlan p; };
static const PackedTuned kPackedTuned[] = {
    {8192, 8192, 64, {1, 3, 1, 2, 64, 128, 4}},   // 70B O: 29.3 us vs 32.7 (row-major table plan, split-K 8)
    {4096, 4096, 1, {-1, 0, 0, 0, 0, 0, 0}},      // 8B O: row-major 13.7 us vs 14.2 packed at M = 64;
    {4096, 4096, 16, {-1, 0, 0, 0, 0, 0, 0}},     // packing O / down measured 1-2 % slower per step
    {4096, 4096, 32, {-1, 0, 0, 0, 0, 0, 0}},     // at B = 1 (kinds_b1_ab.log)
    {4096, 4096, 64, {-1, 0, 0, 0, 0, 0, 0}},
};

int launch_gemm_packed(const bf16* X, long ldx, const bf16* Wp, int M, int N, int K, int epi, bf16* out,
                       long ldo, hipStream_t stream, const RowScale* rs, bool dry, float* ws, size_t ws_bytes,
                       bool defer) {
  if (M <= 0) return dry ? 0 : 1;
  if (N % 256 != 0 || K % 64 != 0) return -1;
  const int rows = gemm_packed_first(M, N, K) ? 5 : M;      // the plan's
  if (rs == nullptr && rows == M) {
    const GemmPlan q = select_plan(M, N, K, epi);
    if (q.kind == 8) {
      const int rc = run_plan(q, X, ldx, Wp, K, M, N, K, epi, nullptr, out, ldo, ws, stream, dry, false, nullptr, true);
      return rc != 0 || dry ? rc : 1;
    }
  }
  GemmPlan p = plan_gemm(rows, N, K);
  if (packed_tile(p, rows, N, K)) p = plan_tile(rows, N, K, true);
  if (tuned_enabled() && plan_overrides().empty() && epi != EPI_SILU_GATE) {
    static const int kB[] = {1, 16, 32, 64, 128, 256, 512};
    int bucket = 0;
    for (int b : kB)
      if (b >= rows) { bucket = b; break; }
    for (const PackedTuned& t : kPackedTuned)
      if (t.N == N && t.K == K && t.M == bucket) {
        if (t.p.kind < 0) return -2;
        if (run_plan(t.p, nullptr, 0, nullptr, 0, M, N, K, epi, nullptr, nullptr, 0, nullptr, nullptr, true) == 0)
          p = t.p;
        break;
      }
  }
  if (epi != EPI_SILU_GATE &&
      run_plan(p, nullptr, 0, nullptr, 0, M, N, K, epi, nullptr, nullptr, 0, nullptr, nullptr, true) != 0)
    p = plan_gemm_heuristic(rows, N, K);
  if (epi == EPI_SILU_GATE &&
      run_plan(p, nullptr, 0, nullptr, 0, M, N, K, epi, nullptr, nullptr, 0, nullptr, nullptr, true) != 0) {
    const int bm = M <= 16 ? 16 : M <= 32 ? 32 : M <= 64 ? 64 : 128;
    p = GemmPlan{1, 3, 0, bm <= 32 ? 1 : 2, bm, 128, 1};
  }
  // 160 to 256 tiles of 128 columns: one a compute unit, K unsplit, four stages in flight. Split by what row-major weights need (neighbouring
  // tiles' rows then meet in few memory channels, packed ones do not) they pay for sums. us, before -> here: 20480 x 4096 by 16 rows 37.8 ->
  // 30.0, by 32 39.9 -> 33.0, 24576 x 4096 by 6, 32 and 64 38.9 -> 33.1, 46.7 -> 34.6, 50.9 -> 39.0, 28672 x 4096 by 32 (64-row tiles unsplit before) 40.3 -> 39.3, 43.8
  // -> 35.8 and 39.4 -> 36.4 on three cards, 28672 x 8192 by 16 88 -> 76; outside: 16384 x 4096 by 16 and 32 26.7 and 27.6, 30.0 and 35.0, 36864 x 4096 by 32 62.6 and 64.8.
  const int ctiles = N / 128;
  if (p.kind == 1 && M <= 64 && ctiles >= 160 && ctiles <= 256 && K >= 256 && epi != EPI_SILU_GATE && plan_overrides().empty())
    p = GemmPlan{1, 4, 1, M <= 32 ? 1 : 2, M <= 16 ? 16 : M <= 32 ? 32 : 64, 128, 1};
  // mid-M kernels (kinds 5 / 7): their weight DMA takes the packed layout as a template flag
  const bool mid = (p.kind == 5 || p.kind == 7) && (p.bn == 128 || p.bn == 256);
  if (mid && !dry && !plan_reaches(p, K, ldx, K)) return -2;
  if (!mid && (p.kind != 1 || (p.bm != 16 && p.bm != 32 && p.bm != 64) || (p.bn != 128 && p.bn != 256))) return -2;
  if (!dry && p.sk > 1 && (ws == nullptr || ws_bytes < kCounterBytes + (size_t)p.sk * M * N * sizeof(float)))
    return -3;
  if (!mid) p.nt = 1;
  if (dry)
    return run_plan(p, nullptr, 0, nullptr, 0, M, N, K, epi, nullptr, nullptr, 0, nullptr, nullptr, true, false,
                    nullptr, mid);
  const bool d = defer && p.sk > 1;
  const int rc = run_plan(p, X, ldx, Wp, K, M, N, K, epi, nullptr, out, ldo, ws, stream, false, d, rs, mid);
  if (rc != 0) return rc;
  return d ? p.sk : 1;     // split count of slabs left in the workspace (deferred), else 1
}

// The dense MoE decode path's gate/up GEMM with the routing weight in its epilogue: one launch
// and one pass over the [M, E * ffn] activation fewer per MoE layer (Mixtral 8x7B B = 64:
// moe_gate_scale was 6.5 us per layer, profiles/r5_moe/mixtral_prefill_decode_trace.md). The
// expert GEMM is a weight stream over >= 1792 column tiles, so the tile plan never splits K.
int launch_gemm_silu_gate(const bf16* X, long ldx, const bf16* W, long ldw, int M, int N, int K,
                          bf16* out, long ldo, const float* gates, int gld, int ge0, int gF,
                          hipStream_t stream) {
  if (M <= 0) return 0;
  if (gates == nullptr || gF <= 0 || gF % 16 != 0 || (N / 2) % gF != 0) return -5;
  GemmPlan p = plan_gemm(M, N, K);
  if (run_plan(p, nullptr, 0, nullptr, 0, M, N, K, EPI_SILU_GATE, nullptr, nullptr, 0, nullptr, nullptr, true) != 0) {
    const int bm = M <= 16 ? 16 : M <= 32 ? 32 : M <= 64 ? 64 : 128;
    p = GemmPlan{1, 3, 0, bm <= 32 ? 1 : 2, bm, 128, 1};
  }
  RowScale rs{nullptr, 0, 0.f, 0.f};
  rs.gate = gates;
  rs.gld = gld;
  rs.ge0 = ge0;
  rs.gF = gF;
  return run_plan(p, X, ldx, W, ldw, M, N, K, EPI_SILU_GATE, nullptr, out, ldo, nullptr, stream, false, false, &rs);
}

}  // namespace bfly
