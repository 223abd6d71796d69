// Sequence mixers for heterogeneous layer stacks, generic in head count, head sizes and element
// type (bf16 or f32 activations / caches; scores, softmax, angles, decays and state are f32):
//   rope_partial_kv_kernel    interleaved-pair rotary on the first 2 * nrot dims of q / k heads,
//                             fused with the paged append of k and v
//                             (K [blocks, G, BS, D] rows, V [blocks, G, Dv, BS] transposed: a
//                             page's keys are contiguous for the P V operand)
//   attn_window_paged_kernel  attention of packed rows over the paged cache: causal sliding
//                             window plus the always-visible first `keep_first` positions, and a
//                             per-head sink logit that only enters the softmax denominator
//   gla_scan_kernel           gated linear attention S <- diag(a) S + k v^T, o = S^T q with the
//                             state pooled in per-sequence slots
// Rows of a step are packed: sequence s owns rows row_cu[s] .. row_cu[s+1] (one row for a
// decoded token, several for a prompt chunk), positions[] gives each row's position.
#include <algorithm>

#include "bfly_common.h"
#include "bfly_mixers.h"

namespace bfly {

#include "attn_window.inc"

namespace {

// RB rows per workgroup. A row's sines and cosines (of the f32 angle, in f64) are found once for all its heads; the values of a page
// lie beside those of the rows before and after them, so that rows which follow one another leave as one store, or at least meet in
// the same L2. 8192 rows of 16 + 4 heads of 128, half of each rotated, in bf16: with a row a workgroup, an angle per pair and accesses of two
// bytes 40 us, with this 22.
template <typename T, int RB>
__global__ __launch_bounds__(256) void rope_partial_kv_kernel(T* __restrict__ q, long q_ld, T* __restrict__ k, long k_ld,
                                                              const T* __restrict__ v, long v_ld,
                                                              const int* __restrict__ positions,
                                                              const float* __restrict__ inv_freq, int nrot,
                                                              const int* __restrict__ slots, T* __restrict__ k_cache,
                                                              T* __restrict__ v_cache, int H, int G, int D, int Dv,
                                                              int bs, int T_) {
  constexpr int kTab = RB == 1 ? 512 : 128, E = 16 / sizeof(T);
  typedef T unit __attribute__((ext_vector_type(E)));
  typedef T run __attribute__((ext_vector_type(RB)));
  __shared__ float2 cs[RB][kTab];
  const long t0 = (long)blockIdx.x * RB;
  const int rows = (int)min((long)RB, T_ - t0), tab = min(nrot, kTab);
  auto turn = [&](int j, int r) {
    const float a = (float)positions[t0 + j] * inv_freq[r];
    double sd, cd;
    sincos((double)a, &sd, &cd);
    return make_float2((float)cd, (float)sd);
  };
  for (int i = threadIdx.x; i < rows * tab; i += 256) cs[i / tab][i % tab] = turn(i / tab, i % tab);
  __syncthreads();
  // rotated pairs of the q heads, then of the k heads: in units of 16 bytes, several of them asked for together, where rows allow it
  if (2 * nrot % E == 0 && nrot <= kTab && D % E == 0 && q_ld % E == 0 && (!k || k_ld % E == 0) &&
      (reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k)) % 16 == 0) {
    constexpr int U = RB == 1 ? 1 : 5;
    const int un = 2 * nrot / E, per = (H + (k ? G : 0)) * un, total = rows * per;
    for (int i0 = threadIdx.x; i0 < total; i0 += 256 * U) {
      unit x[U];
      T* p[U];
      const float2* a[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = min(i0 + 256 * u, total - 1), j = i / per, jj = i - j * per, h = jj / un, r = jj - h * un;
        p[u] = (h < H ? q + (t0 + j) * q_ld + (long)h * D : k + (t0 + j) * k_ld + (long)(h - H) * D) + r * E;
        a[u] = &cs[j][r * (E / 2)];
        x[u] = *reinterpret_cast<const unit*>(p[u]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (i0 + 256 * u >= total) break;
#pragma unroll
        for (int e = 0; e < E; e += 2) {
          const float2 c = a[u][e / 2];
          const float f = (float)x[u][e], w = (float)x[u][e + 1];
          x[u][e] = (T)fmaf(f, c.x, -(w * c.y));      // (as everywhere else: left to the compiler, the forms round differently)
          x[u][e + 1] = (T)fmaf(w, c.x, f * c.y);
        }
        *reinterpret_cast<unit*>(p[u]) = x[u];
      }
    }
  } else {
    const int nq = H * nrot, nk = k ? G * nrot : 0;
    for (int j = 0; j < rows; ++j) {
      const long t = t0 + j;
      for (int i = threadIdx.x; i < nq + nk; i += 256) {
        const bool isq = i < nq;
        const int jj = isq ? i : i - nq, h = jj / nrot, r = jj % nrot;
        T* ptr = (isq ? q + t * q_ld : k + t * k_ld) + (long)h * D + 2 * r;
        const float2 a = r < kTab ? cs[j][r] : turn(j, r);
        const float u = (float)ptr[0], w = (float)ptr[1];
        ptr[0] = (T)fmaf(u, a.x, -(w * a.y));
        ptr[1] = (T)fmaf(w, a.x, u * a.y);
      }
    }
  }
  if (!slots || !k) return;
  __syncthreads();      // the rotated k is read back below
  const bool wide = D % E == 0 && k_ld % E == 0 && (reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(k_cache)) % 16 == 0;
  int slot[RB];
  bool follow = rows == RB && bs % RB == 0 && reinterpret_cast<uintptr_t>(v_cache) % 16 == 0;
#pragma unroll
  for (int j = 0; j < RB; ++j) {
    slot[j] = j < rows ? slots[t0 + j] : -1;
    follow = follow && slot[j] == slot[0] + j;
  }
  follow = follow && slot[0] >= 0 && slot[0] % RB == 0;
  for (int j = 0; j < rows; ++j) {
    const int sl = slots[t0 + j];
    if (sl < 0) continue;
    const long blk = sl / bs, off = sl % bs;
    T* to = k_cache + (blk * G * bs + off) * D;
    const T* from = k + (t0 + j) * k_ld;
    if (wide)
      for (int i = threadIdx.x * E; i < G * D; i += 256 * E)
        *reinterpret_cast<unit*>(to + (long)(i / D) * bs * D + i % D) = *reinterpret_cast<const unit*>(from + i);
    else
      for (int i = threadIdx.x; i < G * D; i += 256) to[(long)(i / D) * bs * D + i % D] = from[i];
  }
  for (int i = threadIdx.x; i < G * Dv; i += 256) {
    run x;
#pragma unroll
    for (int j = 0; j < RB; ++j) x[j] = v[(t0 + min(j, rows - 1)) * v_ld + i];
    if (follow) {
      *reinterpret_cast<run*>(v_cache + ((long)(slot[0] / bs) * G * Dv + i) * bs + slot[0] % bs) = x;
    } else {
#pragma unroll
      for (int j = 0; j < RB; ++j)
        if (slot[j] >= 0) v_cache[((long)(slot[j] / bs) * G * Dv + i) * bs + slot[j] % bs] = x[j];
    }
  }
}

// row -> sequence map of a packed step (rows outside every sequence: -1)
__global__ void row_seq_kernel(const int* __restrict__ row_cu, int nseq, int* __restrict__ row_seq, int T) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= T) return;
  int s = -1;
  for (int i = 0; i < nseq; ++i)
    if (t >= row_cu[i] && t < row_cu[i + 1]) { s = i; break; }
  row_seq[t] = s;
}

// Workgroup = (sequence, head, 64-column slice of Dv), 8 waves; wave w owns 8 columns. A lane is
// (column c = lane & 7, row group gg = lane >> 3) and keeps the NR rows d = gg * NR .. + NR - 1 of
// its column's state in registers, so a token costs NR fused updates per lane and three shuffles to
// sum the eight row groups: no barrier inside the token loop. Tokens are staged 16 at a time:
// their decays (a = exp(log sigmoid(z) / tau), f32), keys, scaled queries and values go to LDS in
// one pass (rows past D are zero, so the row loop needs no bound), the outputs of the 16 tokens
// leave through LDS in another.
template <typename T, int NR>
__global__ __launch_bounds__(512) void gla_scan_kernel(const T* __restrict__ q, long q_ld, const T* __restrict__ k,
                                                       long k_ld, const T* __restrict__ v, long v_ld,
                                                       const T* __restrict__ z, long z_ld, float* __restrict__ state,
                                                       const int* __restrict__ state_slots,
                                                       const int* __restrict__ row_cu,
                                                       const int* __restrict__ positions, float inv_tau,
                                                       float q_scale, float* __restrict__ o, int H, int D, int Dv,
                                                       int cost) {
  constexpr int TB = 16, DP = 8 * NR, NT = 512;
  __shared__ __attribute__((aligned(16))) float sa[TB * DP], sk[TB * DP], sq[TB * DP];
  __shared__ float sv[TB][64], so[TB][64];
  const int s = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * 64;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int cl = 8 * w + (lane & 7), gg = lane >> 3;
  const int col = c0 + cl;
  const bool live = col < Dv;
  const int r0 = row_cu[s], r1 = row_cu[s + 1];
  const int slot = state_slots[s];
  if (r1 <= r0 || (cost && scan_in_chunks(r1 - r0, cost))) return;      // (the chunk form's)
  if (slot < 0) {      // padding sequence of a fixed-shape step: defined output, no state
    for (int i = threadIdx.x; i < (r1 - r0) * 64; i += NT)
      if (c0 + (i & 63) < Dv) o[((long)(r0 + (i >> 6)) * H + h) * Dv + c0 + (i & 63)] = 0.f;
    return;
  }
  float* S = state + ((long)slot * H + h) * D * Dv;
  float st[NR];
  const bool fresh = positions[r0] == 0;
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int d = gg * NR + i;
    st[i] = (!fresh && live && d < D) ? S[(long)d * Dv + col] : 0.f;
  }
  for (int t0 = r0; t0 < r1; t0 += TB) {
    const int nb = min(TB, r1 - t0);
    for (int i = threadIdx.x; i < nb * DP; i += NT) {
      const int tt = i / DP, d = i - tt * DP;
      float a = 0.f, kk = 0.f, qq = 0.f;
      if (d < D) {
        const long t = t0 + tt;
        const float zz = (float)z[t * z_ld + (long)h * D + d];
        // log sigmoid(z) = -softplus(-z), stable on both sides
        float ls;
        if constexpr (sizeof(T) == 2) {   // bf16 inputs: hardware exp / log (f32, ~1 ulp)
          ls = zz < 0.f ? zz - __logf(1.f + __expf(zz)) : -__logf(1.f + __expf(-zz));
          a = __expf(ls * inv_tau);
        } else {
          ls = zz < 0.f ? zz - log1pf(expf(zz)) : -log1pf(expf(-zz));
          a = expf(ls * inv_tau);
        }
        kk = (float)k[t * k_ld + (long)h * D + d];
        qq = (float)q[t * q_ld + (long)h * D + d] * q_scale;
      }
      sa[i] = a;
      sk[i] = kk;
      sq[i] = qq;
    }
    for (int i = threadIdx.x; i < nb * 64; i += NT) {
      const int tt = i >> 6, c = i & 63;
      sv[tt][c] = (c0 + c < Dv) ? (float)v[(long)(t0 + tt) * v_ld + (long)h * Dv + c0 + c] : 0.f;
    }
    __syncthreads();
    for (int tt = 0; tt < nb; ++tt) {
      const float vv = sv[tt][cl];
      const f32x4* pa = reinterpret_cast<const f32x4*>(sa + tt * DP + gg * NR);
      const f32x4* pk = reinterpret_cast<const f32x4*>(sk + tt * DP + gg * NR);
      const f32x4* pq = reinterpret_cast<const f32x4*>(sq + tt * DP + gg * NR);
      float po = 0.f;
#pragma unroll
      for (int i4 = 0; i4 < NR / 4; ++i4) {
        const f32x4 a4 = pa[i4], k4 = pk[i4], q4 = pq[i4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          st[4 * i4 + j] = fmaf(a4[j], st[4 * i4 + j], k4[j] * vv);
          po = fmaf(q4[j], st[4 * i4 + j], po);
        }
      }
      po += __shfl_xor(po, 8, 64);
      po += __shfl_xor(po, 16, 64);
      po += __shfl_xor(po, 32, 64);
      if (gg == 0) so[tt][cl] = po;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nb * 64; i += NT) {
      const int tt = i >> 6, c = i & 63;
      if (c0 + c < Dv) o[((long)(t0 + tt) * H + h) * Dv + c0 + c] = so[tt][c];
    }
    // (the next block's staging overwrites sa / sk / sq / sv, which every wave finished reading
    // at the barrier above; so is rewritten only after the next block's first barrier)
  }
  if (live) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int d = gg * NR + i;
      if (d < D) S[(long)d * Dv + col] = st[i];
    }
  }
}

// The same attention for prompts in true f32 (32-token pages, D = 16 DT, Dv = 16 DVT) on the f32 matrix cores: a workgroup
// owns 64 (token, query head of key / value head blockIdx.y) rows, 16 per wave, and stages each visible page
// once for all of them (double buffered in LDS, one barrier per page). S^T = K Q^T and O^T += V^T P as
// 16x16x4 tiles: the scores come out with a row per lane and four keys per lane group, which is the order in which the
// second product takes them, so nothing is rearranged or rounded between the two. Modifiers, window, kept prefix and
// sink as in attn_window_paged_kernel, with its precise functions. The one-wave-per-row form reads every key row once
// per query head, a row per lane: 5 prompts of 370 tokens, 8 heads on 2 of 128, 846 us; this form: see the launch rule.
template <int DT, int DVT>
__global__ __launch_bounds__(256) void attn_window_f32_kernel(const float* __restrict__ q, long q_ld,
                                                              const float* __restrict__ k_cache,
                                                              const float* __restrict__ v_cache,
                                                              const int* __restrict__ tables, int max_blocks,
                                                              const int* __restrict__ row_cu, int nseq,
                                                              const int* __restrict__ positions, float scale, int window,
                                                              int keep_first, const float* __restrict__ sink,
                                                              const float* __restrict__ out_scale,
                                                              float* __restrict__ out, int T, int H, int G, AttnMod md) {
  constexpr int D = 16 * DT, Dv = 16 * DVT, BS = 32, KP = D + 4, VP = BS + 4;
  constexpr int NKS = BS * D / 4 / 256, NVS = Dv * BS / 4 / 256;      // 16-byte segments per thread
  static_assert(BS * D % 1024 == 0 && Dv * BS % 1024 == 0, "whole segments");
  extern __shared__ __attribute__((aligned(16))) float f32_smem[];
  float* Ks = f32_smem;                  // [2][BS][KP]
  float* Vs = Ks + 2 * BS * KP;          // [2][Dv][VP]
  __shared__ int s_range[4][2], s_odd[2];      // s_odd[b]: 1 + the last page in buffer b with a value that is no number
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, qr = lane & 15, gg = lane >> 4;
  int tile = (int)(gridDim.x - 1 - blockIdx.x);
  const int g = blockIdx.y, R = H / G;
  int s = 0, row0 = 0, rend = 0;
  for (; s < nseq; ++s) {
    const int a = row_cu[s] * R, b = row_cu[s + 1] * R;
    const int nt = (b - a + 63) >> 6;
    if (tile < nt) { row0 = a + 64 * tile; rend = b; break; }
    tile -= nt;
  }
  if (s >= nseq) {                       // (the whole workgroup; at least one has no tile: it clears rows of no sequence)
    const int dvo = md.ext() ? md.dv_out : Dv, first = row_cu[0], last = row_cu[nseq];
    const long pad = tile == 0 ? (long)(first + T - last) * R * dvo : 0;
    for (long i = tid; i < pad; i += 256) {
      const int d = (int)(i % dvo), hd = g * R + (int)(i / dvo % R);
      const long r = i / dvo / R, t = r < first ? r : last + (r - first);
      if (md.ext()) attn_store_ext<false, float>(0.f, t, hd, d, dvo, out, md);
      else out[(t * H + hd) * Dv + d] = 0.f;
    }
    return;
  }
  const int fr = row0 + 16 * wave + qr;
  const bool rv = fr < rend;
  const long frow = rv ? fr : row0, row = frow / R;
  const int h = g * R + (int)(frow % R);
  const int p = rv ? positions[row] : -1;
  const int plo = rv ? attn_row_lo(p, window, md.chunk) : 0;
  const float rscale = attn_row_scale(max(p, 0), scale, md);
  const float da = md.dist_a ? md.dist_a[h] : 0.f, db = md.dist_b ? md.dist_b[h] : 0.f;
  int pmin = rv ? p : 0x7fffffff, pmax = p;
#pragma unroll
  for (int x = 1; x < 16; x <<= 1) {
    pmin = min(pmin, __shfl_xor(pmin, x, 64));
    pmax = max(pmax, __shfl_xor(pmax, x, 64));
  }
  if (lane == 0) { s_range[wave][0] = pmin; s_range[wave][1] = pmax; }
  if (tid < 2) s_odd[tid] = 0;
  f32x4 qf[DT];
#pragma unroll
  for (int c = 0; c < DT; ++c) {
    const float* qp = q + row * q_ld + (long)h * D + 16 * c + 4 * gg;
    qf[c] = f32x4{qp[0], qp[1], qp[2], qp[3]};
  }
  __syncthreads();
  int tmin = s_range[0][0], tmax = s_range[0][1];
#pragma unroll
  for (int w = 1; w < 4; ++w) { tmin = min(tmin, s_range[w][0]); tmax = max(tmax, s_range[w][1]); }
  const int wlo = pmax < 0 ? 0 : attn_row_lo(pmin, window, md.chunk);
  const int* tab = tables + (long)s * max_blocks;
  const int kp = (min(keep_first, tmax + 1) + BS - 1) / BS;          // pages of the kept prefix
  const int wp0 = max(attn_row_lo(max(tmin, 0), window, md.chunk) / BS, kp);
  const int npages = kp + max(0, tmax / BS - wp0 + 1);
  auto page_of = [&](int i) { return i < kp ? i : wp0 + (i - kp); };
  const bool seeded = sink != nullptr;
  float m = seeded ? sink[h] : -1e30f, l = seeded && gg == 0 ? 1.f : 0.f;      // (per-lane partial sums)
  f32x4 o[DVT];
#pragma unroll
  for (int t = 0; t < DVT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 kreg[NKS], vreg[NVS];
  auto gload = [&](int i0) {
    const long blk = (long)tab[page_of(i0)] * G + g;
    const float *Kp = k_cache + blk * BS * D, *Vp = v_cache + blk * Dv * BS;
#pragma unroll
    for (int i = 0; i < NKS; ++i) kreg[i] = *reinterpret_cast<const f32x4*>(Kp + 4 * (tid + 256 * i));
#pragma unroll
    for (int i = 0; i < NVS; ++i) vreg[i] = *reinterpret_cast<const f32x4*>(Vp + 4 * (tid + 256 * i));
  };
  if (npages > 0) gload(0);
  for (int pi = 0; pi < npages; ++pi) {
    float* Kb = Ks + (long)(pi & 1) * BS * KP;
    float* Vb = Vs + (long)(pi & 1) * Dv * VP;
#pragma unroll
    for (int i = 0; i < NKS; ++i) {
      const int idx = tid + 256 * i;
      *reinterpret_cast<f32x4*>(Kb + idx / (D / 4) * KP + 4 * (idx % (D / 4))) = kreg[i];
    }
#pragma unroll
    for (int i = 0; i < NVS; ++i) {
      const int idx = tid + 256 * i;
      *reinterpret_cast<f32x4*>(Vb + idx / 8 * VP + 4 * (idx & 7)) = vreg[i];
    }
    float zero = 0.f;      // (x * 0 of an infinity or NaN is NaN)
#pragma unroll
    for (int i = 0; i < NVS; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) zero = fmaf(vreg[i][e], 0.f, zero);
    if (zero != 0.f) s_odd[pi & 1] = pi + 1;
    __syncthreads();      // the page is in LDS; every wave has left the buffer written next
    const bool odd = s_odd[pi & 1] == pi + 1;
    if (pi + 1 < npages) gload(pi + 1);
    const int j0 = page_of(pi) * BS;
    if (j0 > pmax || (j0 + BS <= wlo && j0 >= keep_first)) continue;      // no row of this wave sees the page
    f32x4 st[2];
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      st[kh] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < DT; ++c) {
        const f32x4 kf = *reinterpret_cast<const f32x4*>(Kb + (16 * kh + qr) * KP + 16 * c + 4 * gg);
#pragma unroll
        for (int e = 0; e < 4; ++e) st[kh] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[e], qf[c][e], st[kh], 0, 0, 0);
      }
    }
    const unsigned span = (unsigned)(p - plo + 1);      // visible: p - j in [0, span) or j < kept
    const int kept = min(keep_first, p + 1);
    float sc[8], mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int j = j0 + 16 * (e >> 2) + 4 * gg + (e & 3);
      const int ok = (int)((unsigned)(p - j) < span) | (int)(j < kept);
      const float x = attn_score<false>(st[e >> 2][e & 3], rscale, p - j, da, db, md);
      sc[e] = ok ? x : -INFINITY;
      mx = fmaxf(mx, sc[e]);
    }
    const float mn = fmaxf(m, row4_max(mx));
    const float corr = expf(m - mn);
    m = mn;
    l *= corr;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      sc[e] = expf(sc[e] - mn);      // exp(-inf) = 0 for masked keys
      l += sc[e];
    }
    if (odd) {
#pragma unroll
      for (int t = 0; t < DVT; ++t) o[t] *= corr;
#pragma unroll 1
      for (int j = 0; j < BS; ++j) {
        float pe = sc[0];      // the weight of key j: element 4 (j >> 4) + (j & 3) of lane group (j >> 2) & 3
#pragma unroll
        for (int e = 1; e < 8; ++e) pe = e == (j >> 4) * 4 + (j & 3) ? sc[e] : pe;
        pe = __shfl(pe, qr + 16 * ((j >> 2) & 3), 64);
        const int ok = (int)((unsigned)(p - j0 - j) < span) | (int)(j0 + j < kept);
#pragma unroll
        for (int t = 0; t < DVT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float x = fmaf(pe, Vb[(16 * t + 4 * gg + i) * VP + j], o[t][i]);
            o[t][i] = ok ? x : o[t][i];
          }
      }
      continue;
    }
#pragma unroll
    for (int t = 0; t < DVT; ++t) {
      o[t] *= corr;
#pragma unroll
      for (int kh = 0; kh < 2; ++kh) {
        const f32x4 vf = *reinterpret_cast<const f32x4*>(Vb + (16 * t + qr) * VP + 16 * kh + 4 * gg);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i], sc[4 * kh + i], o[t], 0, 0, 0);
      }
    }
  }
  l = row4_sum(l);
  if (!rv) return;
  const float inv = (out_scale ? out_scale[row * H + h] : 1.f) / l;
#pragma unroll
  for (int t = 0; t < DVT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 16 * t + 4 * gg + i;
      if (!md.ext()) out[(row * H + h) * Dv + d] = o[t][i] * inv;
      else if (d < md.dv_out) attn_store_ext<false, float>(o[t][i] * inv, row, h, d, md.dv_out, out, md);
    }
}

template <int DT, int DVT>
bool attn_window_f32_launch(const float* q, long q_ld, const float* kc, const float* vc, const int* tables, int max_blocks,
                            const int* row_cu, int nseq, const int* positions, float scale, int window, int keep_first,
                            const float* sink, const float* out_scale, float* out, int T, int H, int G, hipStream_t s,
                            const AttnMod& md) {
  constexpr size_t lds = 2 * (32 * (16 * DT + 4) + 16 * DVT * 36) * sizeof(float);
  static bool once = false;
  if (!once) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_window_f32_kernel<DT, DVT>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    once = true;
  }
  const dim3 grid((unsigned)(((long)T * (H / G) + 63) / 64 + nseq), G);
  attn_window_f32_kernel<DT, DVT><<<grid, 256, lds, s>>>(q, q_ld, kc, vc, tables, max_blocks, row_cu, nseq, positions, scale,
                                                         window, keep_first, sink, out_scale, out, T, H, G, md);
  return true;
}

}  // namespace

bool launch_attn_window_f32(const float* q, long q_ld, const float* kc, const float* vc, const int* tables, int max_blocks,
                            const int* row_cu, int nseq, const int* positions, float scale, int window, int keep_first,
                            const float* sink, const float* out_scale, float* out, int T, int H, int G, int D, int Dv,
                            int block_size, hipStream_t s, const AttnMod& md) {
  // prompts: from 32 (row, head) pairs per sequence and key / value head on, at head sizes of whole segments; decoded rows
  // and other shapes keep the one-wave-per-row form, and so do a few prompt rows, whose waves all run at once (one prompt of
  // 16 rows: 8 heads on 2 of 128 12.2 and 10.1 us, 8 on 1 of 256 / 192 17 and 13; of 40 rows level with 16 heads)
  if ((reinterpret_cast<uintptr_t>(kc) | reinterpret_cast<uintptr_t>(vc)) & 15) return false;
  if (block_size != 32 || md.maps != 1 || md.pool > 0 || md.sigmoid || T <= 0 || (long)T * (H / G) < 32L * nseq ||
      (T != nseq && T < 64 && T * H < 1024))
    return false;
#define BFLY_AF(DT, DVT)                                                                                                \
  return attn_window_f32_launch<DT, DVT>(q, q_ld, kc, vc, tables, max_blocks, row_cu, nseq, positions, scale, window,   \
                                         keep_first, sink, out_scale, out, T, H, G, s, md)
  if (D == 32 && Dv == 32) BFLY_AF(2, 2);
  if (D == 64 && Dv == 64) BFLY_AF(4, 4);
  if (D == 96 && Dv == 96) BFLY_AF(6, 6);
  if (D == 128 && Dv == 128) BFLY_AF(8, 8);
  if (D == 128 && Dv == 256) BFLY_AF(8, 16);
  if (D == 192 && Dv == 192) BFLY_AF(12, 12);
  if (D == 256 && Dv == 192) BFLY_AF(16, 12);
  if (D == 256 && Dv == 256) BFLY_AF(16, 16);
#undef BFLY_AF
  return false;
}

void launch_rope_partial_kv(void* q, long q_ld, void* k, long k_ld, const void* v, long v_ld, const int* positions,
                            const float* inv_freq, int nrot, const int* slots, void* k_cache, void* v_cache,
                            int T, int H, int G, int D, int Dv, int block_size, bool f32, hipStream_t s) {
  if (T <= 0) return;
  // Workgroups enough for the chip first; rows of few elements make up for the start of theirs later. bf16, us with a workgroup per row, four
  // rows, eight rows: 16 + 4 heads of 128 / 128, half rotated, 600 rows 7.0 7.4 8.5, 1024 8.7 8.2 9.0, 2000 12.6 10.7 9.9, 4000 19.6 16.2
  // 13.5, 8192 31.5 25.9 19.8; 8 + 2 of 64 1024 5.6 6.5 7.8, 1500 7.0 7.8 7.9, 2000 8.4 8.1 8.1, 4000 13.1 11.0 10.9; 16 + 1 of 256 / 192
  // 1500 7.9 8.4 8.5, 2000 9.6 8.9 8.8; f32, 16 + 1 4000 17.6 12.5 13.9, 8192 29.1 22.2 20.5.
  const int row = 2 * (H + G) * nrot + G * (D + Dv);
  const int rb = nrot > 128 || T < (row < 2048 ? 1792 : 1024) ? 1 : T < 4096 ? 4 : 8;
#define BFLY_RP(TT, RB)                                                                                                       \
  rope_partial_kv_kernel<TT, RB><<<(T + RB - 1) / RB, 256, 0, s>>>((TT*)q, q_ld, (TT*)k, k_ld, (const TT*)v, v_ld, positions, \
                                                                   inv_freq, nrot, slots, (TT*)k_cache, (TT*)v_cache, H, G,   \
                                                                   D, Dv, block_size, T)
#define BFLY_RPN(TT)                   \
  {                                    \
    if (rb == 1) BFLY_RP(TT, 1);       \
    else if (rb == 4) BFLY_RP(TT, 4);  \
    else BFLY_RP(TT, 8);               \
  }
  if (f32) BFLY_RPN(float) else BFLY_RPN(bf16)
#undef BFLY_RPN
#undef BFLY_RP
}

void launch_row_seq(const int* row_cu, int nseq, int* row_seq, int T, hipStream_t s) {
  if (T <= 0) return;
  row_seq_kernel<<<(T + 255) / 256, 256, 0, s>>>(row_cu, nseq, row_seq, T);
}

// launch_attn_window_mfma with AttnMod's extensions (attn_ext.hip)
bool launch_attn_window_mfma_ext(const void* q, long q_ld, const void* k_cache, const void* v_cache, const int* tables,
                                 int max_blocks, const int* row_cu, int nseq, const int* positions, float scale,
                                 int window, int keep_first, const float* sink, const float* out_scale, void* out, int T,
                                 int H, int G, int D, int Dv, int block_size, float* part, long part_floats,
                                 hipStream_t s, const AttnMod& md);

bool launch_attn_window_mfma(const void* q, long q_ld, const void* k_cache, const void* v_cache, const int* tables,
                             int max_blocks, const int* row_cu, int nseq, const int* positions, float scale, int window,
                             int keep_first, const float* sink, const float* out_scale, void* out, int T, int H, int G,
                             int D, int Dv, int block_size, bool fold, float* part, long part_floats, hipStream_t s,
                             const AttnMod& md) {
  if (md.ext())
    return launch_attn_window_mfma_ext(q, q_ld, k_cache, v_cache, tables, max_blocks, row_cu, nseq, positions, scale, window,
                                       keep_first, sink, out_scale, out, T, H, G, D, Dv, block_size, part, part_floats, s,
                                       md);
  if (!fold && md.maps == 1 && G > 0 && H % G == 0) {
    // any grouped attention: the query heads of a key / value head share its tiles where attn_grouped or attn_tile_plan say so; the
    // per-head tiles of MODE 0 read a page once per query head, and are the ones for several maps per value head
    const long pages = attn_pages(window, keep_first, md.chunk, max_blocks);
    const long fit = part ? part_floats / ((long)T * H * (Dv + 2)) : 1;
    if (T > 0 && (attn_grouped(T, H, G, nseq, D, pages) ||
                  attn_tile_plan(T, H, G, nseq, D, Dv, pages, fit, true, false).tiled)) {
      AttnMod mx = md;
      mx.dv_out = Dv;
      mx.out_ld = (long)H * Dv;
      mx.out_vec = !md.out_f32 && (Dv & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0;
      mx.heads = true;
      return launch_attn_window_mfma_ext(q, q_ld, k_cache, v_cache, tables, max_blocks, row_cu, nseq, positions, scale, window,
                                         keep_first, sink, out_scale, out, T, H, G, D, Dv, block_size, part, part_floats, s,
                                         mx);
    }
  }
  return attn_mfma_launch<0>(q, q_ld, k_cache, v_cache, tables, max_blocks, row_cu, nseq, positions, scale, window,
                             keep_first, sink, out_scale, out, T, H, G, D, Dv, block_size, fold, part, part_floats, s, md);
}

void launch_attn_window_paged(const void* q, long q_ld, const void* k_cache, const void* v_cache, const int* tables,
                              int max_blocks, const int* row_seq, int nseq, const int* positions, float scale,
                              int window, int keep_first, const float* sink, const float* out_scale, void* out, int T,
                              int H, int G, int D, int Dv, int block_size, bool f32, hipStream_t s, const AttnMod& md) {
  if (T <= 0) return;
  (void)nseq;
  dim3 grid(T, H);
  const size_t sm = (size_t)(D + 64 + 2) * sizeof(float) + 64 * sizeof(long);
  if (f32)
    attn_window_paged_kernel<float><<<grid, 64, sm, s>>>((const float*)q, q_ld, (const float*)k_cache,
                                                         (const float*)v_cache, tables, max_blocks, row_seq, positions,
                                                         scale, window, keep_first, sink, out_scale, out, H, G,
                                                         D, Dv, block_size, md);
  else
    attn_window_paged_kernel<bf16><<<grid, 64, sm, s>>>((const bf16*)q, q_ld, (const bf16*)k_cache,
                                                        (const bf16*)v_cache, tables, max_blocks, row_seq, positions,
                                                        scale, window, keep_first, sink, out_scale, out, H, G, D,
                                                        Dv, block_size, md);
}

template <typename T>
static int gla_scan_t(const T* q, long q_ld, const T* k, long k_ld, const T* v, long v_ld, const T* z, long z_ld,
                      float* state, const int* state_slots, const int* row_cu, int nseq, const int* positions,
                      float tau, float q_scale, float* o, int H, int D, int Dv, hipStream_t s, int cost) {
  dim3 grid(nseq, H, (Dv + 63) / 64);
  const float it = 1.f / tau;
#define BFLY_GLA(NR)                                                                                              \
  gla_scan_kernel<T, NR><<<grid, 512, 0, s>>>(q, q_ld, k, k_ld, v, v_ld, z, z_ld, state, state_slots, row_cu, positions, \
                                              it, q_scale, o, H, D, Dv, cost)
  if (D <= 32) BFLY_GLA(4);
  else if (D <= 64) BFLY_GLA(8);
  else if (D <= 128) BFLY_GLA(16);
  else if (D <= 256) BFLY_GLA(32);
  else return -1;
#undef BFLY_GLA
  return 0;
}

void launch_gla_chunks(const void* q, long q_ld, const void* k, long k_ld, const void* v, long v_ld, const void* z, long z_ld,
                       float* state, const int* state_slots, const int* row_cu, int nseq, const int* positions, float tau,
                       float q_scale, float* o, float* rec, int T, int H, int D, int Dv, bool f32, hipStream_t s,
                       int cost);      // forget.hip
long chunk_record_floats(long T, long nseq, int H, int D);

bool chunks_in_one_launch(long T, long nseq, int H, int D, int Dv, bool f32, long max_rows, long max_ld, long v_ld);
bool gate_rows_near(int H, int Dv, long v_ld);

struct GlaForms {
  ScanForms form;
  int cost;      // the chunks' (scan_in_chunks)
  bool one;      // in one launch
};
static GlaForms gla_forms(long T, long nseq, int H, int D, int Dv, bool f32, int max_rows, long max_ld, long v_ld) {
  const long wgs = (long)H * ((Dv + 63) / 64);
  const bool queue = nseq * wgs >= 1024;
  GlaForms f{{true, false}, 0, T > 0 && nseq > 0 && chunks_in_one_launch(T, nseq, H, D, Dv, f32, max_rows, max_ld, v_ld)};
  if (f.one) {
    // One launch takes the time of 12 rows of 128 channels a chunk, in true f32 (whose decays are precise functions) of 14, and
    // somewhat more where the workgroups queue. 16 heads of 128, time of chunks over loop for one sequence of 8, 12, 16, 20, 32
    // rows: 1.09, 0.93, 0.79, 0.93, 0.69 (f32 1.43, 1.18, 0.93, 1.18, 0.83), for 200 of them 1.53, 1.26, 1.02, 1.04, 0.74;
    // channels of 64 0.88 and 0.99 (1.03 and 1.30; queueing 1.06) at 16 rows, of 32 0.97 and 1.24 (1.14 and 1.58), of 192 0.53
    // (0.56), of 256 0.87 at 8.
    if (f32) f.cost = chunk_cost(0, D > 128 ? 11 : D > 64 ? (queue ? 15 : 14) : D > 32 && !queue ? 15 : 18);
    else f.cost = chunk_cost(0, D > 128 ? 7 : D > 64 ? (queue ? 13 : 12) : D > 32 && !queue ? 14 : queue ? 18 : 15);
    // More than a chunk only for a longest sequence that is worth it, and (wide channels) with many workgroups. One and two
    // launches, us: 16 heads of 128, one sequence of 32 rows 13.9 12.9, eight 15.8 17.1 (f32 24.7 19.5); 8 heads of 256, one 20.7
    // 19.6, eight 23.2 24.1, of 64 rows 37 32
    const long longest = max_rows > 0 ? max_rows : T - nseq + 1;
    f.one = longest <= 16 || (!f32 && scan_in_chunks(longest, f.cost) && (D <= 32 || (nseq * wgs >= 256 && (D <= 64 || longest <= 32))));
    f.form = scan_forms(T, nseq, f.cost, wgs, max_rows);
    // (beside a launch of the loop two launches are as good, and their line lies later: 16 single rows and four of 32 in 32 heads of
    // 32 14.9 and 12.5 us, in 16 of 128 31.2 and 27.6)
    if ((f32 && nseq * wgs >= 256) || (f.form.rows && f.form.chunks)) f.one = false;
  }
  if (!f.one) {
    // The chunks' two launches take some 11 us and 1.3 us a chunk of 128 channels, the loop 2.5 us and 0.6 us a row (f32 0.75),
    // until the workgroups queue: then it is their work that counts. Chunks and loop in us, 16 heads of 128, one sequence of 20,
    // 32, 64 rows: 13.5 14.8, 13.0 20, 15.9 37; eight of them 16.1 16.5, 16.9 21.6, 22.6 36.9; 200 of 16, 20, 32, 64 149 185, 193
    // 222, 200 347, 333 700; 200 of 12 rows 129 and 149; heads of 64, 200 sequences of 32 rows 72 91, of 32 channels 64 rows 77
    // 119, of 192 12 rows 355 747.
    if (D > 128) f.cost = queue ? chunk_cost(4, 3) : chunk_cost(8, 2);
    else if (D > 64) f.cost = queue ? chunk_cost(6, 6) : f32 ? chunk_cost(14, 3) : chunk_cost(14, 2);
    else if (D > 32) f.cost = queue ? chunk_cost(14, 8) : chunk_cost(24, 3);
    else f.cost = queue ? chunk_cost(36, 5) : chunk_cost(38, 2);
  }
  if (!f.one) f.form = {true, false};
  if (D <= 256 && !f.one && gate_rows_near(H, Dv, v_ld)) f.form = scan_forms(T, nseq, f.cost, wgs, max_rows);
  return f;
}

GlaSteps gla_scan_steps(int T, int nseq, int H, int D, int Dv, bool f32, int max_rows) {
  const GlaForms f = gla_forms(T, nseq, H, D, Dv, f32, max_rows, (long)H * D, (long)H * Dv);
  if (!f.form.chunks) return {1, 0, -1};
  int least = f.form.rows;
  while (f.form.rows && !scan_in_chunks(least, f.cost)) ++least;
  return {f.form.rows, f.one ? 1 : 2, least};
}

long gla_scan_scratch(int T, int nseq, int H, int D, int Dv, bool f32, int max_rows, long max_ld, long v_ld) {
  if (T <= 0 || nseq <= 0) return 0;
  const GlaForms f = gla_forms(T, nseq, H, D, Dv, f32, max_rows, max_ld, v_ld);
  return f.form.chunks && !f.one ? chunk_record_floats(T, nseq, H, D) : 0;
}
int launch_gla_scan(const void* q, long q_ld, const void* k, long k_ld, const void* v, long v_ld, const void* z,
                    long z_ld, float* state, const int* state_slots, const int* row_cu, int nseq,
                    const int* positions, float tau, float q_scale, float* o, float* rec, int T, int H, int D, int Dv, bool f32,
                    hipStream_t s, int max_rows) {
  if (T <= 0 || nseq <= 0) return 0;
  const GlaForms f = gla_forms(T, nseq, H, D, Dv, f32, max_rows, std::max({q_ld, k_ld, z_ld}), v_ld);
  const ScanForms form = f.form;
  int cost = f.cost;
  if (form.chunks)
    launch_gla_chunks(q, q_ld, k, k_ld, v, v_ld, z, z_ld, state, state_slots, row_cu, nseq, positions, tau, q_scale, o, rec, T, H,
                      D, Dv, f32, s, form.rows ? cost : 0);
  if (!form.rows) return 0;
  if (!form.chunks) cost = 0;
  if (f32)
    return gla_scan_t<float>((const float*)q, q_ld, (const float*)k, k_ld, (const float*)v, v_ld, (const float*)z, z_ld,
                             state, state_slots, row_cu, nseq, positions, tau, q_scale, o, H, D, Dv, s, cost);
  return gla_scan_t<bf16>((const bf16*)q, q_ld, (const bf16*)k, k_ld, (const bf16*)v, v_ld, (const bf16*)z, z_ld, state,
                          state_slots, row_cu, nseq, positions, tau, q_scale, o, H, D, Dv, s, cost);
}

void launch_head_norm_gate(const float* o, const float* w, float eps, const void* gate, long g_ld, int act, float mul,
                           void* out, long out_ld, int T, int H, int Dv, bool f32, hipStream_t s);      // forget.hip

// (a wave per head one value at a time took 54 us for 8192 rows of 16 heads of 128; four values per access and several heads
// per wave: 36 us, 16 rows 4.6 us as before)
void launch_gla_out(const float* o, const void* g, long g_ld, const float* norm_w, float eps, void* out, int T, int H,
                    int Dv, bool f32, hipStream_t s) {
  if (T <= 0) return;
  launch_head_norm_gate(o, norm_w, eps, g, g_ld, 1, 1.f, out, (long)H * Dv, T, H, Dv, f32, s);
}

}  // namespace bfly
