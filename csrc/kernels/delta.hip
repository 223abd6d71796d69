// Sandwich-norm residual stacks with a gated delta rule, generic in every size and in the activation
// type (bf16 or f32; the residual, norms, decays, unit norms and the recurrent state are f32 in both):
//   post_norm_add_norm_kernel,
//   post_norm_rows_kernel            x <- x + mult * layer_norm(y) (+ extra), then the next sublayer's
//                                    input layer_norm(x) with its own weight and bias
//   add_norm_kernel                  x <- x + y, then the next sublayer's input rms_norm(x) (pre-norm stacks)
//   short_conv_act_kernel            y_t = act(sum_j w[:, j] z_(t - taps + 1 + j)) per channel over the
//                                    rows of a sequence (plus an optional bias); rows before the step come from the per-sequence
//                                    history pool, zeros before position 0
//   short_conv_state_update_kernel   the pool takes the last taps - 1 rows of every sequence
//   delta_scan_kernel                S <- g S; u = beta (v - S^T k); S <- S + k u^T; o = S^T q per
//                                    (sequence, head), the state pooled per sequence; row by row
//   delta_chunk_kernel               the same in chunks of 16 rows on the f32 matrix cores
//   delta_record_kernel,
//   delta_chain_kernel               the chunks in two launches, for longer sequences
// Rows of a step are packed: sequence s owns rows row_cu[s] .. row_cu[s+1].
#include <algorithm>
#include <cmath>

#include "bfly_common.h"
#include "bfly_delta.h"
#include "bfly_row_parts_dev.h"
#include "bfly_recur_dev.h"

namespace bfly {

namespace {

// the sequence whose row range holds row t (row_cu is non-decreasing; -1: none)
__device__ __forceinline__ int seq_of_row(const int* __restrict__ row_cu, int nseq, int t) {
  int lo = 0, hi = nseq;            // the last s with row_cu[s] <= t
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (row_cu[mid] <= t) lo = mid; else hi = mid;
  }
  return (nseq > 0 && row_cu[lo] <= t && t < row_cu[lo + 1]) ? lo : -1;
}

// mean and 1 / sqrt(var + eps) of the row staged in LDS (f32, two passes); RMS: 0 and 1 / sqrt(mean x^2 + eps)
template <bool RMS>
__device__ __forceinline__ void row_stats(const float* __restrict__ sy, int W, float eps, float* red, float& mean,
                                          float& rstd) {
  mean = 0.f;
  if (!RMS) {
    float a = 0.f;
    for (int c = threadIdx.x; c < W; c += blockDim.x) a += sy[c];
    mean = block_sum(a, red) / (float)W;
  }
  float q = 0.f;
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    const float d = sy[c] - mean;
    q = fmaf(d, d, q);
  }
  rstd = 1.f / sqrtf(block_sum(q, red) / (float)W + eps);
}

// One workgroup per row; the row of y, then the updated row of x, staged in LDS. V = 4 (W % 4 == 0):
// 16-byte accesses (8-byte for bf16); the statistics are the same two-pass sums either way.
// RMS: RMS norms (no biases) in place of the layer norms.
template <typename T, int V, bool RMS>
__global__ __launch_bounds__(1024) void post_norm_add_norm_kernel(float* __restrict__ x, const T* __restrict__ y,
                                                                 const float* __restrict__ nw,
                                                                 const float* __restrict__ nb, float eps, float mult,
                                                                 const float* __restrict__ extra,
                                                                 const float* __restrict__ nw2,
                                                                 const float* __restrict__ nb2, T* __restrict__ h,
                                                                 int W) {
  typedef float fv __attribute__((ext_vector_type(V)));
  typedef T tv __attribute__((ext_vector_type(V)));
  extern __shared__ __attribute__((aligned(16))) float sy[];
  __shared__ float red[16];
  const long t = blockIdx.x;
  for (int c = V * threadIdx.x; c < W; c += V * blockDim.x) {
    const tv yv = *reinterpret_cast<const tv*>(y + t * W + c);
    fv f;
#pragma unroll
    for (int e = 0; e < V; ++e) f[e] = (float)yv[e];
    *reinterpret_cast<fv*>(sy + c) = f;
  }
  __syncthreads();
  float mean, rstd;
  row_stats<RMS>(sy, W, eps, red, mean, rstd);
  for (int c = V * threadIdx.x; c < W; c += V * blockDim.x) {
    const fv yv = *reinterpret_cast<const fv*>(sy + c), wv = *reinterpret_cast<const fv*>(nw + c),
             bv = RMS ? fv(0.f) : *reinterpret_cast<const fv*>(nb + c);
    fv v = *reinterpret_cast<const fv*>(x + t * W + c);
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = v[e] + mult * ((yv[e] - mean) * rstd * wv[e] + bv[e]);
    if (extra) {
      const fv ev = *reinterpret_cast<const fv*>(extra + t * W + c);
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] += ev[e];
    }
    *reinterpret_cast<fv*>(x + t * W + c) = v;
    *reinterpret_cast<fv*>(sy + c) = v;      // (a thread rewrites only what it alone read after the barrier)
  }
  if (!h) return;
  __syncthreads();
  row_stats<RMS>(sy, W, eps, red, mean, rstd);
  for (int c = V * threadIdx.x; c < W; c += V * blockDim.x) {
    const fv xv = *reinterpret_cast<const fv*>(sy + c), wv = *reinterpret_cast<const fv*>(nw2 + c),
             bv = RMS ? fv(0.f) : *reinterpret_cast<const fv*>(nb2 + c);
    tv o;
#pragma unroll
    for (int e = 0; e < V; ++e) o[e] = (T)((xv[e] - mean) * rstd * wv[e] + bv[e]);
    *reinterpret_cast<tv*>(h + t * W + c) = o;
  }
}

// The same with the row in registers (W % 4 == 0, W <= 1024 NV): every input of a row is asked for before the first sum, and
// nothing but four partial sums per reduction goes through LDS. Staged in LDS a row waits for memory twice and for eight
// barriers: 6184 rows of 2048 in bf16 48 -> 27 us (5.5 TB/s), 4000 of 4096 68 -> 34, one row 5.1 -> 3.7.
template <typename T, bool RMS, int NV, int G>
__global__ __launch_bounds__(256) void post_norm_rows_kernel(float* __restrict__ x, const T* __restrict__ y,
                                                             const float* __restrict__ nw, const float* __restrict__ nb,
                                                             float eps, float mult, const float* __restrict__ extra,
                                                             const float* __restrict__ nw2, const float* __restrict__ nb2,
                                                             T* __restrict__ h, int W, RowParts ex) {
  typedef T tv __attribute__((ext_vector_type(4)));
  __shared__ float red[4][4];
  const long t = blockIdx.x;
  const int tid = threadIdx.x, wave = tid >> 6;
  auto at = [&](int i) { return 4 * tid + 1024 * i; };
  tv yv[NV];
  f32x4 v[NV], xv[NV], wv[NV], bv[NV], ev[NV], zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = at(i);
    xv[i] = wv[i] = bv[i] = ev[i] = zero;
    if (c >= W) continue;
    if (!G) yv[i] = *reinterpret_cast<const tv*>(y + t * W + c);
    xv[i] = *reinterpret_cast<const f32x4*>(x + t * W + c);
    if (extra) ev[i] = *reinterpret_cast<const f32x4*>(extra + t * W + c);
    wv[i] = *reinterpret_cast<const f32x4*>(nw + c);
    if (!RMS) bv[i] = *reinterpret_cast<const f32x4*>(nb + c);
  }
  if constexpr (G > 0) {
    row_of_parts<G>(ex, t, W, v);
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) yv[i][e] = (T)v[i][e];      // (rounded as a row in memory)
  }
  auto block4 = [&](float a, int slot) {
    a = wave_sum(a);
    if ((tid & 63) == 0) red[slot][wave] = a;
    __syncthreads();
    return (red[slot][0] + red[slot][1]) + (red[slot][2] + red[slot][3]);
  };
  // mean and 1 / sqrt(var + eps) of the row in v, two passes (RMS: 0 and 1 / sqrt(mean v^2 + eps))
  float mean, rstd;
  auto stats = [&](int slot) {
    mean = 0.f;
    if (!RMS) {
      float a = 0.f;
#pragma unroll
      for (int i = 0; i < NV; ++i)
        if (at(i) < W) a += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
      mean = block4(a, slot) / (float)W;
    }
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (at(i) < W)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float d = v[i][e] - mean;
          q = fmaf(d, d, q);
        }
    rstd = 1.f / sqrtf(block4(q, slot + 1) / (float)W + eps);
  };
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) v[i][e] = at(i) < W ? (float)yv[i][e] : 0.f;
  stats(0);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = at(i);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[i][e] = xv[i][e] + mult * ((v[i][e] - mean) * rstd * wv[i][e] + bv[i][e]);
      if (extra) v[i][e] += ev[i][e];
    }
    if (c >= W) continue;
    *reinterpret_cast<f32x4*>(x + t * W + c) = v[i];
    if (!h) continue;
    wv[i] = *reinterpret_cast<const f32x4*>(nw2 + c);
    if (!RMS) bv[i] = *reinterpret_cast<const f32x4*>(nb2 + c);
  }
  if (!h) return;
  stats(2);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = at(i);
    if (c >= W) continue;
    tv o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (T)((v[i][e] - mean) * rstd * wv[i][e] + bv[i][e]);
    *reinterpret_cast<tv*>(h + t * W + c) = o;
  }
}

// The same step of a pre-norm stack: x <- x + mult y (+ extra), h = rms_norm(x); each row is read once.
template <typename T, int V>
__global__ __launch_bounds__(1024) void add_norm_kernel(float* __restrict__ x, const T* __restrict__ y, float eps, float mult,
                                                        const float* __restrict__ extra, const float* __restrict__ nw2,
                                                        T* __restrict__ h, int W) {
  typedef float fv __attribute__((ext_vector_type(V)));
  typedef T tv __attribute__((ext_vector_type(V)));
  extern __shared__ __attribute__((aligned(16))) float sy[];
  __shared__ float red[16];
  const long t = blockIdx.x;
  float ss = 0.f;
  for (int c = V * threadIdx.x; c < W; c += V * blockDim.x) {
    const tv yv = *reinterpret_cast<const tv*>(y + t * W + c);
    fv v = *reinterpret_cast<const fv*>(x + t * W + c);
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = fmaf(mult, (float)yv[e], v[e]);
    if (extra) v += *reinterpret_cast<const fv*>(extra + t * W + c);
    *reinterpret_cast<fv*>(x + t * W + c) = v;
    *reinterpret_cast<fv*>(sy + c) = v;      // (read back by this thread alone)
#pragma unroll
    for (int e = 0; e < V; ++e) ss = fmaf(v[e], v[e], ss);
  }
  if (!h) return;
  const float r = 1.f / sqrtf(block_sum(ss, red) / (float)W + eps);
  for (int c = V * threadIdx.x; c < W; c += V * blockDim.x) {
    const fv v = *reinterpret_cast<const fv*>(sy + c), wv = *reinterpret_cast<const fv*>(nw2 + c);
    tv o;
#pragma unroll
    for (int e = 0; e < V; ++e) o[e] = (T)(v[e] * r * wv[e]);
    *reinterpret_cast<tv*>(h + t * W + c) = o;
  }
}

// one thread per (row, channel); the bias (nullable), then the taps oldest first
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void short_conv_act_kernel(const TI* __restrict__ z, long z_ld,
                                                             const float* __restrict__ w,
                                                             const float* __restrict__ bias,
                                                             const float* __restrict__ state,
                                                             const int* __restrict__ state_slots,
                                                             const int* __restrict__ row_cu, int nseq,
                                                             const int* __restrict__ positions, TO* __restrict__ out,
                                                             int C, int taps, int act) {
  const int t = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int s = seq_of_row(row_cu, nseq, t);
  float acc = bias ? bias[c] : 0.f;
  if (s >= 0) {
    const int a = row_cu[s], p = positions[t];
    const int slot = state_slots ? state_slots[s] : -1;
    const int n = taps - 1;
    for (int j = 0; j < taps; ++j) {
      const int d = n - j;           // the input d steps back
      float v = 0.f;
      if (t - d >= a) v = (float)z[(long)(t - d) * z_ld + c];
      else if (p - d >= 0 && slot >= 0) v = state[((long)slot * n + (n - (d - (t - a)))) * C + c];
      acc = fmaf(w[(long)c * taps + j], v, acc);
    }
  }
  if (act == 1) acc = acc / (1.f + expf(-acc));
  out[(long)t * C + c] = (TO)acc;
}

// The same for up to 8 taps and C % 4 == 0 with RB consecutive rows per workgroup: a thread owns 4
// channels, keeps their last taps - 1 inputs in registers and slides over the rows, so a row costs one
// load of z; the history is fetched anew (earlier rows, the pool, or zeros) at the block's first row and
// wherever a new sequence begins. Taps are summed in the same order as above.
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void short_conv_act_rows_kernel(const TI* __restrict__ z, long z_ld,
                                                                  const float* __restrict__ w,
                                                                  const float* __restrict__ bias,
                                                                  const float* __restrict__ state,
                                                                  const int* __restrict__ state_slots,
                                                                  const int* __restrict__ row_cu, int nseq,
                                                                  const int* __restrict__ positions,
                                                                  TO* __restrict__ out, int C, int taps, int act, int T,
                                                                  int RB) {
  constexpr int MAXN = 7;
  typedef TI tiv __attribute__((ext_vector_type(4)));
  typedef TO tov __attribute__((ext_vector_type(4)));
  const int t0 = blockIdx.x * RB, t1 = min(T, t0 + RB);
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  if (c >= C) return;
  const int n = taps - 1;
  f32x4 wv[MAXN + 1], hist[MAXN];
#pragma unroll
  for (int j = 0; j <= MAXN; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) wv[j][e] = j < taps ? w[(long)(c + e) * taps + j] : 0.f;
  const f32x4 bv = bias ? *reinterpret_cast<const f32x4*>(bias + c) : f32x4{0.f, 0.f, 0.f, 0.f};
  auto ld = [&](long row) {
    const tiv v = *reinterpret_cast<const tiv*>(z + row * z_ld + c);
    return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
  };
  int s = -1, send = t0;
  bool fetch = true;
  for (int t = t0; t < t1; ++t) {
    if (t >= send) {
      s = seq_of_row(row_cu, nseq, t);
      send = s >= 0 ? row_cu[s + 1] : t + 1;
      fetch = true;
    }
    f32x4 acc = bv;
    if (s >= 0) {
      const f32x4 zc = ld(t);
      if (fetch) {
        const int a = row_cu[s], p = positions[t];
        const int slot = state_slots ? state_slots[s] : -1;
#pragma unroll
        for (int k = 0; k < MAXN; ++k) {
          if (k >= n) break;
          const int d = n - k;
          f32x4 v = {0.f, 0.f, 0.f, 0.f};
          if (t - d >= a) v = ld(t - d);
          else if (p - d >= 0 && slot >= 0)
            v = *reinterpret_cast<const f32x4*>(state + ((long)slot * n + (n - (d - (t - a)))) * C + c);
          hist[k] = v;
        }
        fetch = false;
      }
#pragma unroll
      for (int k = 0; k < MAXN; ++k) {
        if (k >= n) break;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(wv[k][e], hist[k][e], acc[e]);
      }
#pragma unroll
      for (int k = 0; k <= MAXN; ++k)
        if (k == n) {
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[e] = fmaf(wv[k][e], zc[e], acc[e]);
        }
#pragma unroll
      for (int k = 0; k < MAXN; ++k) {
        if (k + 1 < n) hist[k] = hist[k + 1];
        else if (k + 1 == n) hist[k] = zc;
      }
    }
    tov o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (TO)(act == 1 ? acc[e] / (1.f + expf(-acc[e])) : acc[e]);
    *reinterpret_cast<tov*>(out + (long)t * C + c) = o;
  }
}

// Decoding: every sequence has one row (row s), so the convolution and its history update share a launch
// and a thread. Same order of summation as above.
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void short_conv_step_kernel(const TI* __restrict__ z, long z_ld,
                                                              const float* __restrict__ w,
                                                              const float* __restrict__ bias, float* __restrict__ state,
                                                              const int* __restrict__ state_slots,
                                                              const int* __restrict__ positions, TO* __restrict__ out,
                                                              int C, int taps, int act) {
  const long s = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int p = positions[s], slot = state_slots ? state_slots[s] : -1, n = taps - 1;
  const float zc = (float)z[s * z_ld + c];
  float* S = state + (long)slot * n * C + c;
  float acc = bias ? bias[c] : 0.f;
  for (int j = 0; j < n; ++j) {
    const float v = (slot >= 0 && p - (n - j) >= 0) ? S[(long)j * C] : 0.f;
    acc = fmaf(w[(long)c * taps + j], v, acc);
    if (slot >= 0 && j > 0) S[(long)(j - 1) * C] = v;       // (entry j - 1 was read one iteration ago)
  }
  acc = fmaf(w[(long)c * taps + n], zc, acc);
  if (slot >= 0 && n > 0) S[(long)(n - 1) * C] = zc;
  if (act == 1) acc = acc / (1.f + expf(-acc));
  out[s * C + c] = (TO)acc;
}

// one thread per (sequence, channel): entry i of the new history is old entry i + len while that
// exists (read before any entry at or above it is written), then the step's own rows
template <typename TI>
__global__ __launch_bounds__(256) void short_conv_state_update_kernel(const TI* __restrict__ z, long z_ld,
                                                                      float* __restrict__ state,
                                                                      const int* __restrict__ state_slots,
                                                                      const int* __restrict__ row_cu,
                                                                      const int* __restrict__ positions, int C, int n) {
  const int s = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  const int a = row_cu[s], b = row_cu[s + 1], slot = state_slots[s];
  if (c >= C || b <= a || slot < 0) return;
  const int len = b - a, p0 = positions[a];
  float* S = state + (long)slot * n * C + c;
  for (int i = 0; i < n; ++i) {
    const int r = b - (n - i);       // the row that becomes entry i
    float v;
    if (r >= a) v = (float)z[(long)r * z_ld + c];
    else v = (p0 - (a - r) >= 0) ? S[(long)(i + len) * C] : 0.f;
    S[(long)i * C] = v;
  }
}

// sum over the 8 lanes that share lane >> 3, in every lane, by three cross-lane moves inside a row of 16
// (neighbour, next pair, mirrored half row): no LDS traffic, so the token loop's LDS reads stay in flight
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float sum8(float v) {
  v += dpp_move<0xB1>(v);      // quad_perm [1, 0, 3, 2]
  v += dpp_move<0x4E>(v);      // quad_perm [2, 3, 0, 1]
  v += dpp_move<0x141>(v);     // row_half_mirror: lane i of 8 <- lane 7 - i (the other quad's sum)
  return v;
}

// Workgroup = (sequence, head, 64-column slice of Dv), 8 waves; wave w owns 8 columns. A lane is
// (row group gg = lane & 7, column c = lane >> 3) and keeps the NR rows d = gg * NR .. + NR - 1 of its
// column's state in registers. The pool holds a head's state column by column ([Dv, D]: the rows a lane
// owns are contiguous, the eight lanes of a column cover it with 16-byte accesses). Tokens are staged
// 16 at a time: raw keys and queries go to LDS (rows past D are zero, so the row loop needs no bound),
// and per token the scalars of the update: decay g, write strength beta, 1 / |k|, q_scale / |q| (the
// unit norms are folded into scalars: S^T k = kn S^T k_raw and so on, so no element is normalised on
// its own). The next block's inputs travel to registers while the current block is computed. A token
// then costs a dot product of the lane's rows with k (four partial sums), three cross-lane moves to sum
// the eight row groups, one fused pass that updates the rows and accumulates the read-out, and three
// more moves: no barrier inside the token loop. The outputs of the 16 tokens leave through LDS.
template <typename T, int NR>
__global__ __launch_bounds__(512) void delta_scan_kernel(const float* __restrict__ q, long q_ld,
                                                         const float* __restrict__ k, long k_ld,
                                                         const float* __restrict__ v, long v_ld,
                                                         const T* __restrict__ bl, long b_ld, const T* __restrict__ al,
                                                         long a_ld, const float* __restrict__ a_log,
                                                         const float* __restrict__ dt_bias, float* __restrict__ state,
                                                         const int* __restrict__ state_slots,
                                                         const int* __restrict__ row_cu,
                                                         const int* __restrict__ positions, float q_scale,
                                                         float unit_eps, float* __restrict__ o, int H, int G, int D,
                                                         int Dv, int cost) {
  constexpr int TB = 16, DP = 8 * NR, NT = 512, KQ = TB * DP / NT, VN = TB * 64 / NT;
  __shared__ __attribute__((aligned(16))) float sk[TB * DP], sq[TB * DP];
  __shared__ float sv[TB][64], so[TB][64];
  __shared__ float sg[TB], sb[TB], skn[TB], sqn[TB];
  const int s = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * 64;
  const int hk = h / (H / G);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int cl = 8 * w + (lane >> 3), gg = lane & 7;
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
  float* S = state + (((long)slot * H + h) * Dv + col) * D;      // this lane's column
  const bool vec = (D & 3) == 0;
  float st[NR];
  const bool fresh = positions[r0] == 0;
#pragma unroll
  for (int i4 = 0; i4 < NR / 4; ++i4) {
    const int d = gg * NR + 4 * i4;
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
    if (!fresh && live) {
      if (vec && d + 3 < D) x = *reinterpret_cast<const f32x4*>(S + d);
      else
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = d + j < D ? S[d + j] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) st[4 * i4 + j] = x[j];
  }
  const float rate = expf(a_log[h]), dtb = dt_bias[h];
  // the inputs of a block of TB tokens, one slice per thread
  float rk[KQ], rq[KQ], rv[VN], ra = 0.f, rb = 0.f;
  auto fetch = [&](int t0) {
    const int nb = min(TB, r1 - t0);
#pragma unroll
    for (int j = 0; j < KQ; ++j) {
      const int i = threadIdx.x + j * NT, tt = i / DP, d = i - tt * DP;
      const bool ok = tt < nb && d < D;
      const long t = t0 + tt;
      rk[j] = ok ? k[t * k_ld + (long)hk * D + d] : 0.f;
      rq[j] = ok ? q[t * q_ld + (long)hk * D + d] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < VN; ++j) {
      const int i = threadIdx.x + j * NT, tt = i >> 6, c = i & 63;
      rv[j] = (tt < nb && c0 + c < Dv) ? v[(long)(t0 + tt) * v_ld + (long)h * Dv + c0 + c] : 0.f;
    }
    if (threadIdx.x < nb) {
      ra = (float)al[(long)(t0 + threadIdx.x) * a_ld + h];
      rb = (float)bl[(long)(t0 + threadIdx.x) * b_ld + h];
    }
  };
  fetch(r0);
  for (int t0 = r0; t0 < r1; t0 += TB) {
    const int nb = min(TB, r1 - t0);
#pragma unroll
    for (int j = 0; j < KQ; ++j) {
      sk[threadIdx.x + j * NT] = rk[j];
      sq[threadIdx.x + j * NT] = rq[j];
    }
#pragma unroll
    for (int j = 0; j < VN; ++j) sv[(threadIdx.x + j * NT) >> 6][threadIdx.x & 63] = rv[j];
    if (threadIdx.x < nb) {
      const float av = ra + dtb;
      const float sp = av > 20.f ? av : log1pf(expf(av));            // softplus
      sg[threadIdx.x] = expf(-rate * sp);
      sb[threadIdx.x] = 1.f / (1.f + expf(-rb));
    }
    __syncthreads();
    // unit norms: wave w sums the squares of tokens w and w + 8
    for (int tt = w; tt < nb; tt += 8) {
      float a = 0.f, b = 0.f;
      for (int d = lane; d < DP; d += 64) {
        a = fmaf(sk[tt * DP + d], sk[tt * DP + d], a);
        b = fmaf(sq[tt * DP + d], sq[tt * DP + d], b);
      }
      a = wave_sum(a);
      b = wave_sum(b);
      if (lane == 0) {
        skn[tt] = 1.f / sqrtf(a + unit_eps);
        sqn[tt] = q_scale / sqrtf(b + unit_eps);
      }
    }
    __syncthreads();
    if (t0 + TB < r1) fetch(t0 + TB);        // in flight during the token loop
    for (int tt = 0; tt < nb; ++tt) {
      const float vv = sv[tt][cl], g = sg[tt], bt = sb[tt], kn = skn[tt], qn = sqn[tt];
      const f32x4* pk = reinterpret_cast<const f32x4*>(sk + tt * DP + gg * NR);
      const f32x4* pq = reinterpret_cast<const f32x4*>(sq + tt * DP + gg * NR);
      f32x4 kr[NR / 4];
      f32x4 dp = {0.f, 0.f, 0.f, 0.f};      // four partial sums: short dependent chains
#pragma unroll
      for (int i4 = 0; i4 < NR / 4; ++i4) {
        kr[i4] = pk[i4];
#pragma unroll
        for (int j = 0; j < 4; ++j) dp[j] = fmaf(st[4 * i4 + j], kr[i4][j], dp[j]);
      }
      const float dot = sum8((dp[0] + dp[1]) + (dp[2] + dp[3]));
      // the decayed state's read at k is g kn dot; the write is k_unit u^T = k_raw (kn u)
      const float u = bt * (vv - g * (kn * dot));
      const float uk = kn * u;
      f32x4 pp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i4 = 0; i4 < NR / 4; ++i4) {
        const f32x4 q4 = pq[i4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          st[4 * i4 + j] = fmaf(g, st[4 * i4 + j], kr[i4][j] * uk);
          pp[j] = fmaf(q4[j], st[4 * i4 + j], pp[j]);
        }
      }
      const float po = sum8((pp[0] + pp[1]) + (pp[2] + pp[3]));
      if (gg == 0) so[tt][cl] = po * qn;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nb * 64; i += NT) {
      const int tt = i >> 6, c = i & 63;
      if (c0 + c < Dv) o[((long)(t0 + tt) * H + h) * Dv + c0 + c] = so[tt][c];
    }
    // (the next block's staging overwrites sk / sq / sv and the scalars, which every wave finished
    // reading at the barrier above; so is rewritten only after the next block's barriers)
  }
  if (live) {
#pragma unroll
    for (int i4 = 0; i4 < NR / 4; ++i4) {
      const int d = gg * NR + 4 * i4;
      if (vec && d + 3 < D) {
        *reinterpret_cast<f32x4*>(S + d) = f32x4{st[4 * i4], st[4 * i4 + 1], st[4 * i4 + 2], st[4 * i4 + 3]};
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (d + j < D) S[d + j] = st[4 * i4 + j];
      }
    }
  }
}

// orders one wave's LDS accesses: what its lanes wrote before is what they read after
__device__ __forceinline__ void lds_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Steps with more rows than sequences (prompts): chunks of 16 rows on the f32 matrix cores, in the published chunkwise form of the
// delta rule (the inverse of a unit triangular matrix per chunk, the UT transform). Row by row every token is
// two dot products and an update in one dependent chain (0.78 us a token at D = 128); a chunk needs one chain. With
// k, q the unit rows, G_t = g_0 .. g_t and D_tj = g_(j+1) .. g_t (products of decays over the chunk's rows, never
// quotients) and S the state before the chunk,
//   U = (I + L)^-1 diag(beta) (V - diag(G) K S),   L_tj = beta_t D_tj k_t . k_j  (j < t)
//   o_t = G_t q_t S + sum_(j <= t) D_tj (q_t . k_j) u_j,   S <- G_15 S + sum_j D_15,j k_j u_j^T
// Workgroup = (sequence, head, 64 columns of Dv), eight waves in a pipeline of three chunks with one barrier per step:
//   waves 4 .. 7 load chunk p (a quarter of the channels each, in the operand layout of the 16x16x4 tiles), put its raw
//   rows into LDS and form their parts of K K^T, Q K^T and the squared norms; wave 6 also the products of its decays,
//   which wave 7 has computed a step before;
//   wave 4 turns those of chunk p - 1 into (I + L)^-1 diag(beta): forward substitution in the two 8 x 8 blocks on the
//   diagonal (lane m: column m), the block below them as -T22 L21 T11; wave 5 the weights of the second sum;
//   waves 0 .. 3 run chunk p - 2 with 16 columns of the state each. A state tile's accumulator layout (element e of lane
//   group gg: row 16 i + 4 gg + e) is the B operand of K S and Q S, and the accumulators of V - ..., U are the B
//   operands of the products that follow, so nothing of the chain goes through LDS.
// The unit norms are factors of rows and columns. Rows past the sequence: k = q = 0, g = 1, beta = 0. D <= 16 NT.
// A chunk is one matrix product, in which a weight of zero does not hide a NaN: elements of k, v and the logits that are no
// numbers go in as zeros (g = 1, beta = 0), and from the first row that had one on (k or logits: every column; v: its
// column) outputs and the state are NaN, as a row-by-row scan leaves them; rows before it are untouched. (1 to 4 % of the time.)
// Rounding: a chunk's scalars (decay products, norms, factors of L) are formed in 64 bits and rounded once, products over
// channels are summed in pieces of 32 or 64, and the unit diagonal of (I + L)^-1 is applied without a product; with that
// outputs and states are as far from a 64-bit recurrence as the row-by-row kernel's (rms 1.3e-7 and 1.0e-7 relative).
// Eight sequences of 1024 rows, 16 heads, D = Dv = 128: 534 -> 222 us; bound by the two waves of a SIMD in turn, one
// with products (2.2 us a chunk by itself), one with the scalars' chain (1.9 us).
template <typename T, int NT>
__global__ __launch_bounds__(512, NT <= 4 ? 4 : 2) void delta_chunk_kernel(
    const float* __restrict__ q, long q_ld, const float* __restrict__ k, long k_ld, const float* __restrict__ v, long v_ld,
    const T* __restrict__ bl, long b_ld, const T* __restrict__ al, long a_ld, const float* __restrict__ a_log,
    const float* __restrict__ dt_bias, float* __restrict__ state, const int* __restrict__ state_slots,
    const int* __restrict__ row_cu, const int* __restrict__ positions, float q_scale, float unit_eps, int vec,
    float* __restrict__ o, int H, int G, int D, int Dv, int cost) {
  constexpr int C = 16, NQ = NT / 4, NG = NT / 4, NS = NT <= 8 ? 2 : 4, KP = 16 * NT + 4, PP = C + 4;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float* sk = smem;                       // [3][C][KP] raw k
  float* sq = sk + 3 * C * KP;            // [3][C][KP] raw q
  float* skk = sq + 3 * C * KP;           // [2][4][64][4] the waves' parts of K K^T
  float* sqk = skk + 2 * 4 * 256;         // [2][4][64][4] and of Q K^T
  float* snk = sqk + 2 * 4 * 256;         // [2][4][C] of the squared norms
  float* snq = snk + 2 * 4 * C;           // [2][4][C]
  float* sd = snq + 2 * 4 * C;            // [2][64][4] D
  float* sg = sd + 2 * 256;               // [2][4][C]: G, D_15, beta, G_15
  float* sT = sg + 2 * 4 * C;             // [2][C][PP] (I + L)^-1 diag(beta)
  float* sA = sT + 2 * C * PP;            // [2][C][PP] weights D_tj (q_t . k_j) / |k_j|
  float* sc = sA + 2 * C * PP;            // [2][6][C]: G / |k|, D_15 / |k|, G, q_scale / |q|, G_15, beta
  float* sl = sc + 2 * 6 * C;             // [2][2][C] decay and write strength of each row
  int* sj = reinterpret_cast<int*>(sl + 2 * 2 * C);      // [4] first row of a chunk whose k or logits are no numbers, or C
  const int s = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * 64;
  const int hk = h / (H / G);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, m = lane & 15, gg = lane >> 4;
  const int r0 = __builtin_amdgcn_readfirstlane(row_cu[s]), r1 = __builtin_amdgcn_readfirstlane(row_cu[s + 1]);
  const int slot = state_slots[s];
  if (r1 <= r0 || (cost && !scan_in_chunks(r1 - r0, cost))) return;      // (the row-by-row form's)
  if (slot < 0) {      // padding sequence of a fixed-shape step: defined output, no state
    for (int i = tid; i < (r1 - r0) * 64; i += 512)
      if (c0 + (i & 63) < Dv) o[((long)(r0 + (i >> 6)) * H + h) * Dv + c0 + (i & 63)] = 0.f;
    return;
  }
  const int nch = (r1 - r0 + C - 1) / C;
  if (wave < 4) {
    const int col = c0 + 16 * wave + m;
    const bool live = col < Dv;
    float* S = state + (((long)slot * H + h) * Dv + min(col, Dv - 1)) * D;      // this lane's column
    const bool fresh = positions[r0] == 0;
    f32x4 st[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int d = 16 * i + 4 * gg;
      st[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (!fresh) {
        if ((vec & 2) && d < D) st[i] = *reinterpret_cast<const f32x4*>(S + d);
        else
#pragma unroll
          for (int e = 0; e < 4; ++e) st[i][e] = d + e < D ? S[d + e] : 0.f;
      }
    }
    const float* vc = v + (long)h * Dv + min(col, Dv - 1);
    float rv[4];
    auto fetch = [&](int t0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) rv[e] = vc[(long)min(t0 + 4 * gg + e, r1 - 1) * v_ld];
    };
    fetch(r0);
    for (int i = 0; i < 3; ++i) __syncthreads();
    for (int c = 0; c < nch; ++c) {
      const int t0 = r0 + c * C;
      const float* kb = sk + (c % 3) * C * KP;
      const float* qb = sq + (c % 3) * C * KP;
      const float* f = sc + (c & 1) * 6 * C;
      // Operands come from LDS a group of four tiles ahead of their use. Partial sums by element and per NS tiles: short
      // dependent chains, and no longer sums than a row's own dot product takes.
      f32x4 ka[2][4], qa[2][4], pk = {0.f, 0.f, 0.f, 0.f}, pq = pk, u = pk, y = pk;
      float ku[2][4][4];
      auto rows = [&](int g) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          ka[g & 1][i] = *reinterpret_cast<const f32x4*>(kb + m * KP + 16 * (4 * g + i) + 4 * gg);
          qa[g & 1][i] = *reinterpret_cast<const f32x4*>(qb + m * KP + 16 * (4 * g + i) + 4 * gg);
        }
      };
      auto cols = [&](int g) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) ku[g & 1][i][e] = kb[(4 * gg + e) * KP + 16 * (4 * g + i) + m];
      };
      f32x4 ux[4], yx[4];
      rows(0);
      const f32x4 gk = *reinterpret_cast<const f32x4*>(f + 4 * gg), dk = *reinterpret_cast<const f32x4*>(f + C + 4 * gg);
      const f32x4 ti = *reinterpret_cast<const f32x4*>(sT + ((c & 1) * C + m) * PP + 4 * gg);
      const f32x4 bt = *reinterpret_cast<const f32x4*>(f + 5 * C + 4 * gg);
      const float gn = f[4 * C];
      // what the chunk's end needs: early, or (NT <= 4, whose two workgroups per compute unit leave 128 registers) late
      f32x4 gt, qn, wq;
      auto weights = [&] { wq = *reinterpret_cast<const f32x4*>(sA + ((c & 1) * C + m) * PP + 4 * gg); };
      auto last = [&] {
        gt = *reinterpret_cast<const f32x4*>(f + 2 * C + 4 * gg);
        qn = *reinterpret_cast<const f32x4*>(f + 3 * C + 4 * gg);
      };
      if (NT > 4) {
        weights();
        last();
      }
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        if (g + 1 < NG) rows(g + 1);
        else cols(0);
#pragma unroll
        for (int j = 0; j < 4; j += NS) {
          f32x4 xk[4], xq[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) xk[e] = xq[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int i = j; i < j + NS; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              xk[e] = mfma_f32(ka[g & 1][i][e], st[4 * g + i][e], xk[e]);
              xq[e] = mfma_f32(qa[g & 1][i][e], st[4 * g + i][e], xq[e]);
            }
          pk += (xk[0] + xk[1]) + (xk[2] + xk[3]);
          pq += (xq[0] + xq[1]) + (xq[2] + xq[3]);
        }
      }
      // no[e]: 0, or NaN from the first row of this lane's column on that is no number (x * 0 of such an x is NaN); the sums over
      // rows by lane groups. Without a branch, which would split the chunk's one schedule.
      f32x4 no;
      float vv[4], sum = 0.f;
      const int odd = sj[c & 3];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = t0 + 4 * gg + e < r1 ? rv[e] : 0.f, z = fmaf(x, 0.f, 0.f);
        vv[e] = z == 0.f ? x : 0.f;
        sum += z;
        no[e] = sum + (4 * gg + e >= odd ? NAN : 0.f);
      }
      // lane groups 1 and 3 take the sum of 0 and 2, then 2 and 3 that of 0 and 1 (the swaps of row4_sum)
      const auto up = __builtin_amdgcn_permlane16_swap(__float_as_uint(sum), __float_as_uint(sum), false, false);
      const unsigned pair = __float_as_uint(__uint_as_float(up[0]) + __uint_as_float(up[1]));
      const auto far = __builtin_amdgcn_permlane32_swap(pair, pair, false, false);
      no += (gg & 1 ? __uint_as_float(up[0]) : 0.f) + (gg & 2 ? __uint_as_float(far[0]) : 0.f);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float ve = fmaf(-gk[e], pk[e], vv[e]);
        ux[e] = mfma_f32(ti[e], ve, f32x4{0.f, 0.f, 0.f, 0.f});
        u[e] = bt[e] * ve;
      }
      u += (ux[0] + ux[1]) + (ux[2] + ux[3]);
      if (c + 1 < nch) fetch(t0 + C);      // in flight until the next chunk
      if (NT <= 4) weights();
      const f32x4 ud = (u + no) * dk;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        if (g + 1 < NG) cols(g + 1);
        f32x4 x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int i = 0; i < 4; ++i) x[i] = mfma_f32(ku[g & 1][i][e], ud[e], x[i]);
          if (g == 0) yx[e] = mfma_f32(wq[e], u[e], e == 0 ? no : f32x4{0.f, 0.f, 0.f, 0.f});
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) st[4 * g + i][e] = fmaf(st[4 * g + i][e], gn, x[i][e]);
      }
      if (NT <= 4) last();
      y = (yx[0] + yx[1]) + (yx[2] + yx[3]);
      if (live) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int t = t0 + 4 * gg + e;
          if (t < r1) o[((long)t * H + h) * Dv + col] = fmaf(pq[e], gt[e], y[e]) * qn[e];
        }
      }
      __syncthreads();
    }
    if (live) {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int d = 16 * i + 4 * gg;
        if ((vec & 2) && d < D) *reinterpret_cast<f32x4*>(S + d) = st[i];
        else
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (d + e < D) S[d + e] = st[i][e];
      }
    }
    return;
  }
  // ---- waves 4 .. 7: chunk p's rows and their products, then the 16 x 16 matrices of chunk p - 1 ----
  __builtin_amdgcn_s_setprio(2);      // (a chunk's chain of scalars is as long as the products it waits for)
  const int w = wave - 4;
  const float rate = expf(a_log[h]), dtb = dt_bias[h];
  f32x4 rk[NQ], rq[NQ];
  T an = (T)0.f, bn = (T)0.f;      // wave 7: the logits of row m, as stored (a conversion here would wait for the loads)
  auto gates = [&](int t0) {
    const long t = min(t0 + m, r1 - 1);
    an = al[t * a_ld + h];
    bn = bl[t * b_ld + h];
  };
  // wave 7, chunk c: decay and write strength of row m (and a fresh mark of the chunk: its readers are two steps behind)
  auto write_gates = [&](int c) {
    const float av = (float)an + dtb;
    const float sp = av > 20.f ? av : log1pf(expf(av));            // softplus
    const float g = expf(-rate * sp), b = 1.f / (1.f + expf(-(float)bn));
    const bool nan = !(g == g && b == b), in = r0 + c * C + m < r1 && !nan;
    sl[(c & 1) * 2 * C + m] = in ? g : 1.f;
    sl[((c & 1) * 2 + 1) * C + m] = in ? b : 0.f;
    if (lane == 0) sj[c & 3] = C;
    if (__any(nan && r0 + c * C + m < r1)) {
      lds_wave_sync();
      if (nan && r0 + c * C + m < r1) atomicMin(&sj[c & 3], m);
    }
  };
  const float* k0 = k + (long)(r0 + m) * k_ld + (long)hk * D;
  const float* q0 = q + (long)(r0 + m) * q_ld + (long)hk * D;
  auto fetch = [&](int t0) {
    long past = t0 - r0;
    if (t0 + C > r1) past -= max(0, t0 + m - (r1 - 1));      // (rows past the sequence: its last row again)
    const float* kr = k0 + past * k_ld;
    const float* qr = q0 + past * q_ld;
    if (vec & 1) {
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        const int d = min(16 * (NQ * w + i) + 4 * gg, D - 4);
        rk[i] = *reinterpret_cast<const f32x4*>(kr + d);
        rq[i] = *reinterpret_cast<const f32x4*>(qr + d);
      }
    } else {
#pragma unroll
      for (int i = 0; i < NQ; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int d = min(16 * (NQ * w + i) + 4 * gg + e, D - 1);
          rk[i][e] = kr[d];
          rq[i][e] = qr[d];
        }
    }
  };
  if (w == 3) {
    gates(r0);
    write_gates(0);
    if (nch > 1) gates(r0 + C);
  }
  fetch(r0);
  __syncthreads();
  for (int p = 0; p < nch + 2; ++p) {
    if (p < nch) {
      const int t0 = r0 + p * C;
      float* kb = sk + (p % 3) * C * KP + m * KP;
      float* qb = sq + (p % 3) * C * KP + m * KP;
      f32x4 nk = {0.f, 0.f, 0.f, 0.f}, nq = nk, kx[4], qx[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) kx[e] = qx[e] = nk;
      const int in = t0 + m < r1, Dm = in ? D : 0;
      float zero = 0.f;
#pragma unroll
      for (int i = 0; i < NQ; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) zero = fmaf(rk[i][e], 0.f, zero);
      if (__any(zero != 0.f)) {      // (channels past D are copies of the row's own)
        if (zero != 0.f && in) atomicMin(&sj[p & 3], m);
#pragma unroll
        for (int i = 0; i < NQ; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) rk[i][e] = rk[i][e] * 0.f == 0.f ? rk[i][e] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        const int d = 16 * (NQ * w + i) + 4 * gg;
        f32x4 a, b;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool ok = d + e < Dm;
          a[e] = ok ? rk[i][e] : 0.f;
          b[e] = ok ? rq[i][e] : 0.f;
        }
        *reinterpret_cast<f32x4*>(kb + d) = a;
        *reinterpret_cast<f32x4*>(qb + d) = b;
        nk += a * a;
        nq += b * b;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          kx[e] = mfma_f32(a[e], a[e], kx[e]);
          qx[e] = mfma_f32(b[e], a[e], qx[e]);
        }
      }
      if (p + 1 < nch) fetch(t0 + C);
      const float xk = row4_sum((nk[0] + nk[1]) + (nk[2] + nk[3])), xq = row4_sum((nq[0] + nq[1]) + (nq[2] + nq[3]));
      const int at = (p & 1) * 4 + w;
      const f32x4 kk = (kx[0] + kx[1]) + (kx[2] + kx[3]), qk = (qx[0] + qx[1]) + (qx[2] + qx[3]);
      *reinterpret_cast<f32x4*>(skk + (at * 64 + lane) * 4) = kk;
      *reinterpret_cast<f32x4*>(sqk + (at * 64 + lane) * 4) = qk;
      snk[at * C + m] = xk;
      snq[at * C + m] = xq;
      if (w == 2) {
        const float g = sl[(p & 1) * 2 * C + m];
        // column m of D (rows 4 gg + e kept), G_m, D_15,m and G_15
        int mm = m, gm = gg;
        asm volatile("" : "+v"(mm), "+v"(gm));      // (compared anew per chunk: kept masks would fill the scalar registers)
        double x = 1., y = 1.;
        float Gm = 1.f;
        f32x4 dm;
#pragma unroll
        for (int t = 0; t < C; ++t) {
          const double gt = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, g), t));
          y *= gt;
          x = t > mm ? x * gt : 1.;
          Gm = t == mm ? (float)y : Gm;
          if (t < 4) dm[t] = (float)x;
          else dm[t & 3] = gm == t >> 2 ? (float)x : dm[t & 3];
        }
        *reinterpret_cast<f32x4*>(sd + ((p & 1) * 64 + lane) * 4) = dm;
        float* f = sg + (p & 1) * 4 * C + m;
        f[0] = Gm;
        f[C] = (float)x;
        f[2 * C] = sl[((p & 1) * 2 + 1) * C + m];
        f[3 * C] = (float)y;
      } else if (w == 3 && p + 1 < nch) {
        write_gates(p + 1);
        if (p + 2 < nch) gates(t0 + 2 * C);
      }
    }
    if (p > 0 && p <= nch && w < 2) {
      const int b2 = (p - 1) & 1;
      const f32x4 dm = *reinterpret_cast<const f32x4*>(sd + (b2 * 64 + lane) * 4);
      const float* part = w ? sqk : skk;
      float nk = 0.f, nq = 0.f;
      f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        nk += snk[(b2 * 4 + i) * C + m];
        nq += snq[(b2 * 4 + i) * C + m];
        z += *reinterpret_cast<const f32x4*>(part + ((b2 * 4 + i) * 64 + lane) * 4);
      }
      const float* fg = sg + b2 * 4 * C + m;
      // (rows past the sequence: no key, also where unit_eps is 0)
      const double kn = r0 + (p - 1) * C + m < r1 ? 1. / sqrt((double)nk + (double)unit_eps) : 0.;
      float* f = sc + b2 * 6 * C + m;
      float* tb = sT + b2 * C * PP;
      double zd[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) zd[e] = (double)z[e] * ((double)dm[e] * kn);
      if (w) {
#pragma unroll
        for (int e = 0; e < 4; ++e) sA[(b2 * C + 4 * gg + e) * PP + m] = 4 * gg + e >= m ? (float)zd[e] : 0.f;
        f[0] = (float)(fg[0] * kn);
        f[C] = (float)(fg[C] * kn);
        f[2 * C] = fg[0];
        f[3 * C] = (float)((double)q_scale / sqrt((double)nq + (double)unit_eps));
        f[4 * C] = fg[3 * C];
        f[5 * C] = fg[2 * C];
      } else {
        const float beta = fg[2 * C];
        const double rw = beta * kn;
        const int b8 = m & 8, cc = m & 7;
#pragma unroll
        for (int e = 0; e < 4; ++e) tb[(4 * gg + e) * PP + m] = (float)(zd[e] * __shfl(rw, 4 * gg + e, 64));
        lds_wave_sync();
        f32x4 l[8][2];      // rows of this lane's diagonal block
#pragma unroll
        for (int t = 1; t < 8; ++t) {
          l[t][0] = *reinterpret_cast<const f32x4*>(tb + (b8 + t) * PP + b8);
          if (t > 4) l[t][1] = *reinterpret_cast<const f32x4*>(tb + (b8 + t) * PP + b8 + 4);
        }
        f32x4 l21 = {0.f, 0.f, 0.f, 0.f};
        if (m >= 8 && gg < 2) l21 = *reinterpret_cast<const f32x4*>(tb + m * PP + 4 * gg);
        lds_wave_sync();
        float x[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          x[t] = t == cc ? 1.f : 0.f;
#pragma unroll
          for (int j = 0; j < t; ++j) x[t] = fmaf(-l[t][j >> 2][j & 3], x[j], x[t]);
          tb[(b8 + t) * PP + m] = x[t];
          tb[((b8 ^ 8) + t) * PP + m] = 0.f;
        }
        lds_wave_sync();
        const f32x4 ta = *reinterpret_cast<const f32x4*>(tb + m * PP + 4 * gg);
        float tc[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) tc[e] = tb[(4 * gg + e) * PP + m];
        f32x4 y = {0.f, 0.f, 0.f, 0.f}, y2 = y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y = mfma_f32(l21[e], tc[e], y);
#pragma unroll
        for (int e = 0; e < 4; ++e) y2 = mfma_f32(ta[e], y[e], y2);
        lds_wave_sync();
#pragma unroll
        for (int e = 0; e < 4; ++e) tb[(4 * gg + e) * PP + m] = 4 * gg + e > m ? (tc[e] - y2[e]) * beta : 0.f;
      }
    }
    __syncthreads();
  }
}

// The same chunks in two launches, for longer sequences: all of a chunk but its products with the state is independent of the
// chunks before it. delta_record_kernel leaves k and q ([16][KP] rows each, what is no number as zero) of every chunk and key head
// and (I + L)^-1 diag(beta), the weights (both in the operand layout of the 16x16x4 tiles) and the factors of every chunk and head
// in records; delta_chain_kernel runs down a sequence's records with nothing but matrix products and the copies of the next ones.
// A chunk's records are at its sequence's first row / 16 + the sequence's number + its own number there: no two chunks of a step
// share one, and (rows / 16 + sequences) are enough. Sums and their order are those of delta_chunk_kernel.
constexpr int kDeltaSlots = 3, kDeltaHead = 768;      // (floats of a head's record: [64][4], [64][4], six factors of 16 rows, the mark)
constexpr int delta_rows(int NT) { return (32 * (16 * NT + 4) + 255) / 256 * 256; }
__device__ __forceinline__ __amdgpu_buffer_rsrc_t delta_buffer(const void* base, long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)min(bytes, 0x7fffffffL), 0x00020000);
}
template <int N>
__device__ __forceinline__ void delta_vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Workgroup = (key head, chunk): four waves share the channels of the chunk's products, then take the key head's heads in turn.
template <typename T, int NT>
__global__ __launch_bounds__(256) void delta_record_kernel(
    const float* __restrict__ q, long q_ld, const float* __restrict__ k, long k_ld, const T* __restrict__ bl, long b_ld,
    const T* __restrict__ al, long a_ld, const float* __restrict__ a_log, const float* __restrict__ dt_bias,
    const int* __restrict__ state_slots, const int* __restrict__ row_cu, int nseq, float q_scale, float unit_eps, int vec,
    float* __restrict__ rec, int H, int G, int D, int cost, int first) {
  constexpr int C = 16, NQ = NT / 4, KP = 16 * NT + 4, PP = C + 4;
  __shared__ __attribute__((aligned(16))) float skk[4][64][4], sqk[4][64][4], snk[4][C], snq[4][C], stb[4][C * PP];
  __shared__ int s_mark;
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, m = lane & 15, gg = lane >> 4;
  const int hk = blockIdx.x, b = first + blockIdx.y;
  int s = -1;      // the last sequence whose records begin at or before b
  for (int i0 = 0; i0 < nseq; i0 += 64) {
    const int i = i0 + lane;
    const unsigned long long le = __ballot(i < nseq && (row_cu[min(i, nseq)] >> 4) + i <= b);
    s += __popcll(le);
    if (~le) break;
  }
  if (s < 0) return;
  const int r0 = __builtin_amdgcn_readfirstlane(row_cu[s]), r1 = __builtin_amdgcn_readfirstlane(row_cu[s + 1]);
  const int t0 = r0 + C * (b - (r0 >> 4) - s);
  if (t0 >= r1 || (cost && !scan_in_chunks(r1 - r0, cost)) || state_slots[s] < 0) return;
  const int t = min(t0 + m, r1 - 1);            // (rows past the sequence: its last row again)
  const bool in = t0 + m < r1;
  if (tid == 0) s_mark = C;
  __syncthreads();
  {
    const float* kr = k + (long)t * k_ld + (long)hk * D;
    const float* qr = q + (long)t * q_ld + (long)hk * D;
    f32x4 rk[NQ], rq[NQ];
    if (vec & 1) {
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        const int d = min(16 * (NQ * w + i) + 4 * gg, D - 4);
        rk[i] = *reinterpret_cast<const f32x4*>(kr + d);
        rq[i] = *reinterpret_cast<const f32x4*>(qr + d);
      }
    } else {
#pragma unroll
      for (int i = 0; i < NQ; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int d = min(16 * (NQ * w + i) + 4 * gg + e, D - 1);
          rk[i][e] = kr[d];
          rq[i][e] = qr[d];
        }
    }
    float* kb = rec + ((long)blockIdx.y * G + hk) * delta_rows(NT) + m * KP;
    f32x4 nk = {0.f, 0.f, 0.f, 0.f}, nq = nk, kx[4], qx[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) kx[e] = qx[e] = nk;
    const int Dm = in ? D : 0;
    float zero = 0.f;
#pragma unroll
    for (int i = 0; i < NQ; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) zero = fmaf(rk[i][e], 0.f, zero);
    if (__any(zero != 0.f)) {      // (channels past D are copies of the row's own)
      if (zero != 0.f && in) atomicMin(&s_mark, m);
#pragma unroll
      for (int i = 0; i < NQ; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) rk[i][e] = rk[i][e] * 0.f == 0.f ? rk[i][e] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int d = 16 * (NQ * w + i) + 4 * gg;
      f32x4 x, y;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool ok = d + e < Dm;
        x[e] = ok ? rk[i][e] : 0.f;
        y[e] = ok ? rq[i][e] : 0.f;
      }
      *reinterpret_cast<f32x4*>(kb + d) = x;
      *reinterpret_cast<f32x4*>(kb + C * KP + d) = y;
      nk += x * x;
      nq += y * y;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        kx[e] = mfma_f32(x[e], x[e], kx[e]);
        qx[e] = mfma_f32(y[e], x[e], qx[e]);
      }
    }
    const float xk = row4_sum((nk[0] + nk[1]) + (nk[2] + nk[3])), xq = row4_sum((nq[0] + nq[1]) + (nq[2] + nq[3]));
    *reinterpret_cast<f32x4*>(skk[w][lane]) = (kx[0] + kx[1]) + (kx[2] + kx[3]);
    *reinterpret_cast<f32x4*>(sqk[w][lane]) = (qx[0] + qx[1]) + (qx[2] + qx[3]);
    snk[w][m] = xk;
    snq[w][m] = xq;
  }
  __syncthreads();
  rec += (long)gridDim.y * G * delta_rows(NT);
  const int HH = H / G, km = s_mark;
  float nk = 0.f, nq = 0.f;
  f32x4 zk = {0.f, 0.f, 0.f, 0.f}, zq = zk;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    nk += snk[i][m];
    nq += snq[i][m];
    zk += *reinterpret_cast<const f32x4*>(skk[i][lane]);
    zq += *reinterpret_cast<const f32x4*>(sqk[i][lane]);
  }
  // (rows past the sequence: no key, also where unit_eps is 0)
  const double kn = in ? 1. / sqrt((double)nk + (double)unit_eps) : 0.;
  const float qn = (float)((double)q_scale / sqrt((double)nq + (double)unit_eps));
  float* tb = stb[w];
  for (int h = hk * HH + w; h < (hk + 1) * HH; h += 4) {
    float* to = rec + ((long)blockIdx.y * H + h) * kDeltaHead;
    const float av = (float)al[(long)t * a_ld + h] + dt_bias[h], bv = (float)bl[(long)t * b_ld + h];
    const float sp = av > 20.f ? av : log1pf(expf(av));            // softplus
    float g = expf(-expf(a_log[h]) * sp), beta = 1.f / (1.f + expf(-bv));
    const bool nan = !(g == g && beta == beta);
    const unsigned odd = (unsigned)__ballot(nan && in) & 0xffffu;
    g = in && !nan ? g : 1.f;
    beta = in && !nan ? beta : 0.f;
    // column m of D (rows 4 gg + e kept), G_m, D_15,m and G_15
    double x = 1., y = 1.;
    float Gm = 1.f;
    f32x4 dm = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const double gi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, g), i));
      y *= gi;
      x = i > m ? x * gi : 1.;
      Gm = i == m ? (float)y : Gm;
      dm[i & 3] = gg == i >> 2 ? (float)x : dm[i & 3];
    }
    double zd[4];
    // the second sum's weights D_tj (q_t . k_j) / |k_j|
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      zd[e] = (double)zq[e] * ((double)dm[e] * kn);
      tb[(4 * gg + e) * PP + m] = 4 * gg + e >= m ? (float)zd[e] : 0.f;
    }
    lds_wave_sync();
    *reinterpret_cast<f32x4*>(to + 256 + 4 * lane) = *reinterpret_cast<const f32x4*>(tb + m * PP + 4 * gg);
    if (gg == 0) {
      float* f = to + 512 + m;
      f[0] = (float)(Gm * kn);
      f[C] = (float)((float)x * kn);
      f[2 * C] = Gm;
      f[3 * C] = qn;
      f[4 * C] = (float)y;
      f[5 * C] = beta;
      if (m == 0) *reinterpret_cast<int*>(to + 512 + 6 * C) = min(km, odd ? __builtin_ctz(odd) : C);
    }
    lds_wave_sync();
    // (I + L)^-1 diag(beta) as in delta_chunk_kernel
#pragma unroll
    for (int e = 0; e < 4; ++e) zd[e] = (double)zk[e] * ((double)dm[e] * kn);
    const double rw = beta * kn;
    const int b8 = m & 8, cc = m & 7;
#pragma unroll
    for (int e = 0; e < 4; ++e) tb[(4 * gg + e) * PP + m] = (float)(zd[e] * __shfl(rw, 4 * gg + e, 64));
    lds_wave_sync();
    f32x4 l[8][2];      // rows of this lane's diagonal block
#pragma unroll
    for (int i = 1; i < 8; ++i) {
      l[i][0] = *reinterpret_cast<const f32x4*>(tb + (b8 + i) * PP + b8);
      if (i > 4) l[i][1] = *reinterpret_cast<const f32x4*>(tb + (b8 + i) * PP + b8 + 4);
    }
    f32x4 l21 = {0.f, 0.f, 0.f, 0.f};
    if (m >= 8 && gg < 2) l21 = *reinterpret_cast<const f32x4*>(tb + m * PP + 4 * gg);
    lds_wave_sync();
    float xs[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      xs[i] = i == cc ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) xs[i] = fmaf(-l[i][j >> 2][j & 3], xs[j], xs[i]);
      tb[(b8 + i) * PP + m] = xs[i];
      tb[((b8 ^ 8) + i) * PP + m] = 0.f;
    }
    lds_wave_sync();
    const f32x4 ta = *reinterpret_cast<const f32x4*>(tb + m * PP + 4 * gg);
    float tc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) tc[e] = tb[(4 * gg + e) * PP + m];
    f32x4 y1 = {0.f, 0.f, 0.f, 0.f}, y2 = y1;
#pragma unroll
    for (int e = 0; e < 4; ++e) y1 = mfma_f32(l21[e], tc[e], y1);
#pragma unroll
    for (int e = 0; e < 4; ++e) y2 = mfma_f32(ta[e], y1[e], y2);
    lds_wave_sync();
#pragma unroll
    for (int e = 0; e < 4; ++e) tb[(4 * gg + e) * PP + m] = 4 * gg + e > m ? (tc[e] - y2[e]) * beta : 0.f;
    lds_wave_sync();
    *reinterpret_cast<f32x4*>(to + 4 * lane) = *reinterpret_cast<const f32x4*>(tb + m * PP + 4 * gg);
    lds_wave_sync();
  }
}

// Workgroup = (sequence, head, 64 columns of Dv), four waves of 16 columns with the whole height of the state each, in the accumulator
// layout (see delta_chunk_kernel). Bound by the vector units, which f32 products occupy for 32 clocks each and share with everything
// else: 104 products and 250 vector instructions, 2.3 us a chunk at 128 x 128. (As products of three-part bf16 operands, which run
// beside vector instructions, 2.0: splitting the state takes as long as the products did.) All workgroups of a sequence's key head read the same rows: they follow eight apart, in one XCD.
// Records arrive by LDS-DMA, kDeltaSlots chunks ahead. The records [first, first + count) of the step; a sequence that goes on in the
// next ones leaves its state in its slot.
template <int NT>
__global__ __launch_bounds__(256, NT <= 8 ? 2 : 1) void delta_chain_kernel(
    const float* __restrict__ rec, const float* __restrict__ v, long v_ld, float* __restrict__ state,
    const int* __restrict__ state_slots, const int* __restrict__ row_cu, const int* __restrict__ positions, int vec,
    float* __restrict__ o, int nseq, int H, int G, int D, int Dv, int cost, int first, int count) {
  constexpr int C = 16, SL = kDeltaSlots, KP = 16 * NT + 4, RR = delta_rows(NT), U1 = RR / 256, U = U1 + kDeltaHead / 256,
                PER = (U + 3) / 4, REC = U * 256, NS = NT <= 8 ? 2 : 4;
  extern __shared__ __attribute__((aligned(16))) float smem[];      // [SL][REC], then values: [SL][4 waves][4][64]
  const int nz = (Dv + 63) / 64, HH = H / G, per = HH * nz, u = blockIdx.x >> 3, grp = u / per * 8 + (blockIdx.x & 7);
  if (grp / G >= nseq) return;
  const int s = NT <= 8 ? by_length(row_cu, nseq, grp / G, 256 / (H * nz)) : grp / G;
  const int hk = grp % G, h = hk * HH + u % per / nz, c0 = u % nz * 64;
  const int r0 = __builtin_amdgcn_readfirstlane(row_cu[s]), r1 = __builtin_amdgcn_readfirstlane(row_cu[s + 1]);
  if (r1 <= r0 || (cost && !scan_in_chunks(r1 - r0, cost))) return;      // (the row-by-row form's)
  const int at = (r0 >> 4) + s, cb = max(0, first - at), ce = min((r1 - r0 + C - 1) / C, first + count - at);
  if (cb >= ce) return;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, m = lane & 15, gg = lane >> 4;
  const int slot = state_slots[s];
  if (slot < 0) {      // padding sequence of a fixed-shape step: defined output, no state
    const int ta = r0 + cb * C, n = min(r1, r0 + ce * C) - ta;
    for (int i = tid; i < n * 64; i += 256)
      if (c0 + (i & 63) < Dv) o[((long)(ta + (i >> 6)) * H + h) * Dv + c0 + (i & 63)] = 0.f;
    return;
  }
  const int col = c0 + 16 * wave + m;
  const bool live = col < Dv;
  // Addresses are a scalar base and offset per chunk and a constant per lane. Rows past the sequence, rows of the state past D and
  // columns past the head lie past the buffer's end: they read zeros and are not stored, and no lane takes a branch of its own.
  const int dead = live ? 0 : -1;
  float* S = state + ((long)slot * H + h) * Dv * D;
  auto place = [&](int d) { return (col * D + d) * 4 | dead | (d < D ? 0 : -1); };
  f32x4 st[NT];
  {
    const bool fresh = cb == 0 && positions[r0] == 0;
    const auto ss = __builtin_amdgcn_make_buffer_rsrc(S, (short)0, fresh ? 0 : Dv * D * 4, 0x00020000);
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int d = 16 * i + 4 * gg;
      if (vec & 2) st[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ss, place(d), 0, 0));
      else
#pragma unroll
        for (int e = 0; e < 4; ++e) st[i][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ss, place(d + e), 0, 0));
    }
  }
  const auto rs = delta_buffer(rec, 0x7fffffff);
  const int lastn = min(C, r1 - r0 - (ce - 1) * C);      // rows of the last chunk here
  const long vl = (long)(lastn - 1) * v_ld + Dv, ve1 = (long)(C - 1) * v_ld + Dv, ol = ((long)(lastn - 1) * H + 1) * Dv;
  const int vbytes = (int)min(ve1 * 4, 0x7fffffffL), vlast = (int)min(vl * 4, 0x7fffffffL), olast = (int)min(ol * 4, 0x7fffffffL);
  int va[4], oo[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    va[e] = (int)((4 * gg + e) * v_ld + col) * 4 | dead;
    oo[e] = ((4 * gg + e) * H * Dv + col) * 4 | dead;
  }
  const float* vp = v + (long)(r0 + cb * C) * v_ld + (long)h * Dv;
  float* op = o + ((long)(r0 + cb * C) * H + h) * Dv;
  const int rel = at + cb - first, rbase = (rel * G + hk) * RR * 4, hbase = (count * G * RR + (rel * H + h) * kDeltaHead) * 4;
  // operation j of PER + 4 of chunk c's copy: a part of its records, then the lanes' own four values. Past the last chunk: that one
  // again, into a slot nobody reads.
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  auto dma = [&](int c, int sl, int j) {
    c = min(c, ce - 1) - cb;
    if (j < PER) {
      const int x = min(wave + 4 * j, U - 1);
      const int off = x < U1 ? rbase + c * G * RR * 4 + 1024 * x : hbase + c * H * kDeltaHead * 4 + 1024 * (x - U1);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(smem + sl * REC + 256 * x), 16, 16 * lane, off, 0, 0);
    } else {
      const auto vs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(vp + (long)(c * C) * v_ld), (short)0,
                                                        c == ce - 1 - cb ? vlast : vbytes, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(vs, (lds_ptr_t)(smem + SL * REC + ((sl * 4 + wave) * 4 + j - PER) * 64), 4,
                                               va[j - PER], 0, 0, 0);
    }
  };
#pragma unroll
  for (int i = 0; i < SL; ++i)
#pragma unroll
    for (int j = 0; j < PER + 4; ++j) dma(cb + i, i, j);
  f32x4 ka[NT], qa[NT];
  float ku[NT][4], raw[4];
  auto krow = [&](int sl, int i) { ka[i] = *reinterpret_cast<const f32x4*>(smem + sl * REC + m * KP + 16 * i + 4 * gg); };
  auto values = [&](int sl) {
#pragma unroll
    for (int e = 0; e < 4; ++e) raw[e] = smem[SL * REC + ((sl * 4 + wave) * 4 + e) * 64 + lane];
  };
  delta_vm_wait<(SL - 1) * (PER + 4)>();
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < NT; ++i) krow(0, i);
  values(0);
  int sl = 0;
  const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
  // K S first; Q S runs while its sums, (I + L)^-1 and the factors turn them into U, so the matrix cores do not wait. Fragments are
  // read a product ahead: q during K S, the columns of k during Q S, the next chunk's k during the state's update. The one barrier
  // of a chunk lies before the update: behind it the chunk's slot is free.
  for (int c = cb; c < ce; ++c) {
    const float* x0 = smem + sl * REC;
    const float* f = x0 + RR + 512;
    const f32x4 ti = *reinterpret_cast<const f32x4*>(x0 + RR + 4 * lane), wq = *reinterpret_cast<const f32x4*>(x0 + RR + 256 + 4 * lane);
    const f32x4 gk = *reinterpret_cast<const f32x4*>(f + 4 * gg), dk = *reinterpret_cast<const f32x4*>(f + C + 4 * gg);
    const f32x4 gt = *reinterpret_cast<const f32x4*>(f + 2 * C + 4 * gg), qn = *reinterpret_cast<const f32x4*>(f + 3 * C + 4 * gg);
    const f32x4 bt = *reinterpret_cast<const f32x4*>(f + 5 * C + 4 * gg);
    const float gn = f[4 * C];
    const int odd = __builtin_amdgcn_readfirstlane(reinterpret_cast<const int*>(f)[6 * C]);
    f32x4 pk = z4, pq = z4;
#pragma unroll
    for (int i = 0; i < NT; i += NS) {
      f32x4 xk[4] = {z4, z4, z4, z4};
#pragma unroll
      for (int j = i; j < i + NS; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          xk[e] = mfma_f32(ka[j][e], st[j][e], xk[e]);
          if (e == 1) qa[j] = *reinterpret_cast<const f32x4*>(x0 + C * KP + m * KP + 16 * j + 4 * gg);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      pk += (xk[0] + xk[1]) + (xk[2] + xk[3]);
    }
    // no[e]: 0, or NaN from the first row of this lane's column on that is no number (as in delta_chunk_kernel)
    f32x4 no, ux[4], u = z4;
    float ve[4];
#pragma unroll
    for (int i = 0; i < NT; i += NS) {
      f32x4 xq[4] = {z4, z4, z4, z4};
#pragma unroll
      for (int j = i; j < i + NS; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          xq[e] = mfma_f32(qa[j][e], st[j][e], xq[e]);
          ku[j][e] = x0[(4 * gg + e) * KP + 16 * j + m];
        }
        if (j == 0) {
          float vv[4], sum = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float z = fmaf(raw[e], 0.f, 0.f);
            vv[e] = z == 0.f ? raw[e] : 0.f;
            sum += z;
            no[e] = sum + (4 * gg + e >= odd ? NAN : 0.f);
          }
          // lane groups 1 and 3 take the sum of 0 and 2, then 2 and 3 that of 0 and 1 (the swaps of row4_sum)
          const auto up = __builtin_amdgcn_permlane16_swap(__float_as_uint(sum), __float_as_uint(sum), false, false);
          const unsigned pair = __float_as_uint(__uint_as_float(up[0]) + __uint_as_float(up[1]));
          const auto far = __builtin_amdgcn_permlane32_swap(pair, pair, false, false);
          no += (gg & 1 ? __uint_as_float(up[0]) : 0.f) + (gg & 2 ? __uint_as_float(far[0]) : 0.f);
#pragma unroll
          for (int e = 0; e < 4; ++e) ve[e] = fmaf(-gk[e], pk[e], vv[e]);
        }
        if (j == NT / 2 - 1) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            ux[e] = mfma_f32(ti[e], ve[e], z4);
            u[e] = bt[e] * ve[e];
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      pq += (xq[0] + xq[1]) + (xq[2] + xq[3]);
    }
    u += (ux[0] + ux[1]) + (ux[2] + ux[3]);
    const f32x4 ud = (u + no) * dk;
    // A turn of the loop issues PER + 8 memory operations (records, values, outputs), the start has no outputs: with as many of the
    // newest in flight, the next chunk's records have landed (own part).
    if (c - cb < SL - 1) delta_vm_wait<(SL - 2) * (PER + 4)>();
    else delta_vm_wait<(SL - 2) * (PER + 8)>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    const int nx = sl + 1 == SL ? 0 : sl + 1;
    constexpr int OPS = PER + 4, QS = NT / 2;
    f32x4 yx[4];
#pragma unroll
    for (int i = 0; i < NT; i += 4) {
      f32x4 x[4] = {z4, z4, z4, z4};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = mfma_f32(ku[i + j][e], ud[e], x[j]);
        if (i == 0) yx[e] = mfma_f32(wq[e], u[e], e == 0 ? no : z4);
        krow(nx, i + e);
        const int n = i + e - QS;      // the copies, spread over the second half
        if (n >= 0) {
#pragma unroll
          for (int j = n * OPS / QS; j < (n + 1) * OPS / QS; ++j) dma(c + SL, sl, j);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (i == 0) values(nx);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) st[i + j][e] = fmaf(st[i + j][e], gn, x[j][e]);
    }
    sl = nx;
    const f32x4 y = (yx[0] + yx[1]) + (yx[2] + yx[3]);
    const auto out = __builtin_amdgcn_make_buffer_rsrc(op, (short)0, c == ce - 1 ? olast : 0x7fffffff, 0x00020000);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(fmaf(pq[e], gt[e], y[e]) * qn[e]), out, oo[e], 0, 0);
    op += (long)C * H * Dv;
  }
  delta_vm_wait<0>();      // no LDS-DMA may outlive the workgroup
  const auto ss = __builtin_amdgcn_make_buffer_rsrc(S, (short)0, Dv * D * 4, 0x00020000);
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int d = 16 * i + 4 * gg;
    if (vec & 2) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, st[i]), ss, place(d), 0, 0);
    else
#pragma unroll
      for (int e = 0; e < 4; ++e) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(st[i][e]), ss, place(d + e), 0, 0);
  }
}

// threads of a one-row workgroup: about four elements per thread, whole waves, at most 1024
int row_threads(int W) { return std::min(1024, std::max(64, (W / 4 + 63) / 64 * 64)); }

}  // namespace

bool post_norm_in_registers(int W) { return W % 4 == 0 && W > 256 && W <= 4096; }

void launch_post_norm_add_norm(float* x, const void* y, const float* nw, const float* nb, float eps, float mult,
                               const float* extra, const float* nw2, const float* nb2, void* h, int T, int W, bool rms,
                               bool f32, hipStream_t s, const RowParts& ex) {
  if (T <= 0) return;
  const size_t sm = (size_t)W * sizeof(float);
  if (!nw) {      // y as it is, one RMS norm
#define BFLY_AN(TT, V) add_norm_kernel<TT, V><<<T, row_threads(W), sm, s>>>(x, (const TT*)y, eps, mult, extra, nw2, (TT*)h, W)
    if (W % 4 == 0) { if (f32) BFLY_AN(float, 4); else BFLY_AN(bf16, 4); }
    else { if (f32) BFLY_AN(float, 1); else BFLY_AN(bf16, 1); }
#undef BFLY_AN
    return;
  }
  // (wider rows would not fit a workgroup's registers; of narrow ones most of a workgroup would be idle: 4000 rows of 256 9.2 us,
  // staged in LDS by one wave 7.0, of 320 level)
  if (post_norm_in_registers(W)) {
#define BFLY_PNRG(TT, R, NV, G) \
  post_norm_rows_kernel<TT, R, NV, G><<<T, 256, 0, s>>>(x, (const TT*)y, nw, nb, eps, mult, extra, nw2, nb2, (TT*)h, W, ex)
#define BFLY_PNR(TT, R, NV)                           \
  {                                                   \
    if (!ex.y) BFLY_PNRG(TT, R, NV, 0);               \
    else if (ex.K <= 2) BFLY_PNRG(TT, R, NV, 2);      \
    else BFLY_PNRG(TT, R, NV, 4);                     \
  }
#define BFLY_PNR2(TT, R)                                                                             \
  {                                                                                                  \
    if (W <= 1024) BFLY_PNR(TT, R, 1) else if (W <= 2048) BFLY_PNR(TT, R, 2) else BFLY_PNR(TT, R, 4) \
  }
    if (f32) { if (rms) BFLY_PNR2(float, true) else BFLY_PNR2(float, false) }
    else { if (rms) BFLY_PNR2(bf16, true) else BFLY_PNR2(bf16, false) }
#undef BFLY_PNR2
#undef BFLY_PNR
#undef BFLY_PNRG
    return;
  }
#define BFLY_PNAN(TT, V, R)                                                                                          \
  post_norm_add_norm_kernel<TT, V, R><<<T, row_threads(W), sm, s>>>(x, (const TT*)y, nw, nb, eps, mult, extra, nw2, nb2, \
                                                                    (TT*)h, W)
#define BFLY_PNAN2(TT, V)        \
  {                              \
    if (rms) BFLY_PNAN(TT, V, true); else BFLY_PNAN(TT, V, false); \
  }
  if (W % 4 == 0) { if (f32) BFLY_PNAN2(float, 4) else BFLY_PNAN2(bf16, 4) }
  else { if (f32) BFLY_PNAN2(float, 1) else BFLY_PNAN2(bf16, 1) }
#undef BFLY_PNAN2
#undef BFLY_PNAN
}

void launch_short_conv_step(const void* z, long z_ld, const float* w, const float* bias, float* state,
                            const int* state_slots, const int* positions, void* out, int T, int C, int taps, int act,
                            bool f32, bool out_f32, hipStream_t s) {
  if (T <= 0 || C <= 0) return;
  dim3 grid(T, (C + 255) / 256);
#define BFLY_SCS(TI, TO)                                                                                              \
  short_conv_step_kernel<TI, TO><<<grid, 256, 0, s>>>((const TI*)z, z_ld, w, bias, state, state_slots, positions, (TO*)out, \
                                                      C, taps, act)
  if (f32) BFLY_SCS(float, float);
  else if (out_f32) BFLY_SCS(bf16, float);
  else BFLY_SCS(bf16, bf16);
#undef BFLY_SCS
}

void launch_short_conv_act(const void* z, long z_ld, const float* w, const float* bias, const float* state, const int* state_slots,
                           const int* row_cu, int nseq, const int* positions, void* out, int T, int C, int taps, int act,
                           bool f32, bool out_f32, hipStream_t s) {
  if (T <= 0 || C <= 0) return;
  const size_t esz = f32 ? 4 : 2;
  if (taps <= 8 && C % 4 == 0 && z_ld % 4 == 0 && reinterpret_cast<uintptr_t>(z) % (4 * esz) == 0 && T >= 64) {
    // rows per workgroup: enough workgroups to fill the chip first
    const int RB = std::min(16, std::max(1, T / 512));
    dim3 g2((T + RB - 1) / RB, (C / 4 + 255) / 256);
#define BFLY_SCR(TI, TO)                                                                                             \
  short_conv_act_rows_kernel<TI, TO><<<g2, 256, 0, s>>>((const TI*)z, z_ld, w, bias, state, state_slots, row_cu, nseq,     \
                                                        positions, (TO*)out, C, taps, act, T, RB)
    if (f32) BFLY_SCR(float, float);
    else if (out_f32) BFLY_SCR(bf16, float);
    else BFLY_SCR(bf16, bf16);
#undef BFLY_SCR
    return;
  }
  dim3 grid(T, (C + 255) / 256);
#define BFLY_SC(TI, TO)                                                                                              \
  short_conv_act_kernel<TI, TO><<<grid, 256, 0, s>>>((const TI*)z, z_ld, w, bias, state, state_slots, row_cu, nseq, positions, \
                                                     (TO*)out, C, taps, act)
  if (f32) BFLY_SC(float, float);
  else if (out_f32) BFLY_SC(bf16, float);
  else BFLY_SC(bf16, bf16);
#undef BFLY_SC
}

void launch_short_conv_state_update(const void* z, long z_ld, float* state, const int* state_slots, const int* row_cu,
                                    int nseq, const int* positions, int C, int n, bool f32, hipStream_t s) {
  if (nseq <= 0 || n <= 0 || C <= 0) return;
  dim3 grid(nseq, (C + 255) / 256);
  if (f32)
    short_conv_state_update_kernel<float><<<grid, 256, 0, s>>>((const float*)z, z_ld, state, state_slots, row_cu,
                                                               positions, C, n);
  else
    short_conv_state_update_kernel<bf16><<<grid, 256, 0, s>>>((const bf16*)z, z_ld, state, state_slots, row_cu,
                                                              positions, C, n);
}

template <typename T, int NT>
static void delta_chunk_launch(const float* q, long q_ld, const float* k, long k_ld, const float* v, long v_ld, const T* b,
                               long b_ld, const T* a, long a_ld, const float* a_log, const float* dt_bias, float* state,
                               const int* state_slots, const int* row_cu, int nseq, const int* positions, float q_scale,
                               float unit_eps, float* o, int H, int G, int D, int Dv, hipStream_t s, int cost) {
  constexpr int C = 16;
  constexpr size_t lds = (size_t)(6 * C * (16 * NT + 4) + 18 * 256 + 24 * C + 4 * C * (C + 4) + 16 * C + 4) * sizeof(float);
  static bool once = false;
  if (!once) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&delta_chunk_kernel<T, NT>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    once = true;
  }
  // 1: rows of q and k, 2: columns of the state in four-element accesses
  int vec = 0;
  if (D % 4 == 0 && rows_aligned(q, q_ld, 4) && rows_aligned(k, k_ld, 4)) vec |= 1;
  if (D % 4 == 0) vec |= 2;
  dim3 grid(nseq, H, (Dv + 63) / 64);
  delta_chunk_kernel<T, NT><<<grid, 512, lds, s>>>(q, q_ld, k, k_ld, v, v_ld, b, b_ld, a, a_ld, a_log, dt_bias, state, state_slots,
                                                   row_cu, positions, q_scale, unit_eps, vec, o, H, G, D, Dv, cost);
}

// 16-channel tiles of the chunk kernels
static int delta_tiles(int D) { return D <= 64 ? 4 : D <= 128 ? 8 : D <= 192 ? 12 : 16; }
// floats of the records of one chunk, and the chunks of a launch: those of the step, at most 256 MB of records
static long delta_chunk_floats(int H, int G, int D) { return (long)G * delta_rows(delta_tiles(D)) + (long)H * kDeltaHead; }
static long delta_chunks_at_once(long T, long nseq, int H, int G, int D) {
  return std::min((T >> 4) + nseq, std::max(1L, (64L << 20) / delta_chunk_floats(H, G, D)));
}

// Two launches where the times of both forms say so (us, measured): a chunk of one workgroup after the other takes `one` in one launch
// and `two` in the chains, times the rounds of workgroups or, where two share a compute unit, the share; the records come on top.
// 16 heads of 128 on 4, us of one launch -> two: one sequence of 64 rows 20.1 and 20.3, of 128 32.5 -> 29.6, of 2000 397 -> 292,
// 11 of 200 to 800 245 -> 179, 32 of 32 52 -> 40, 64 of 320 560 -> 389; 32 heads of 64 on 8, 64 of 320 312 -> 291; heads of 256, 32 of
// 320 872 -> 781. Of 824 steps that were timed none is slower than in one launch by more than 4 %.
static bool delta_two_launches(long T, long nseq, int H, int G, int D, int Dv, long wgs, int max_rows) {
  const long longest = std::max(1L, max_rows > 0 ? max_rows : T - nseq + 1), like = std::min(nseq, (T + longest - 1) / longest);
  const float one[] = {2.15f, 3.2f, 4.2f, 5.3f}, two[] = {1.4f, 2.35f, 3.8f, 5.1f};
  const float n = (float)((longest + 15) >> 4), w = (float)(like * wgs), share = std::max(1.f, w / 280), rounds = std::ceil(w / 256);
  const int d = (D - 1) / 64;
  const float records = 3.5f + (float)((T >> 4) + nseq) * G * (3 + 2 * (H / G)) * 1e-3f;
  return records + two[d] * n * (D <= 128 ? share : rounds) < one[d] * n * (D <= 64 ? share : rounds);
}

struct DeltaPlan {
  ScanForms form;
  int cost;
  bool records;      // chunks in two launches
};
static DeltaPlan delta_plan(long T, long nseq, int H, int G, int D, int Dv, long v_ld, int max_rows) {
  // A chunk takes the time of 10 rows of 128 channels while the workgroups all run at once, and of 14 where they queue (the
  // loop's have half the LDS): 16 heads of 128, time of chunks over loop for one sequence of 8, 12, 16, 20, 32 rows 1.07, 0.88,
  // 0.80, 0.85, 0.66, for 64 of them 1.24, 1.06, 1.05, 1.23, 0.91; channels of 64 0.82 and 0.94 at 16 rows, of 32 0.91 and 1.14,
  // of 192 0.51 and 0.49. With each sequence in its own form: 32 single rows beside 128 114 and 63 us, now 58; 200 beside 300
  // 249 and 291, now 173.
  const long wgs = (long)H * ((Dv + 63) / 64);
  const bool queue = nseq * wgs >= 1024;
  DeltaPlan p;
  p.cost = D > 128 ? 8 : D > 64 ? (queue ? 14 : 10) : D > 32 ? (queue ? 12 : 10) : queue ? 15 : 12;
  p.form = D > 256 ? ScanForms{true, false} : scan_forms(T, nseq, p.cost, wgs, max_rows);
  p.records = p.form.chunks && std::max({v_ld, (long)H * Dv, (long)D * Dv}) * 64 < (1L << 31) &&      // (32-bit byte offsets)
              delta_two_launches(T, nseq, H, G, D, Dv, wgs, max_rows);
  return p;
}

long delta_record_floats(long T, long nseq, int H, int G, int D, int Dv, long v_ld, int max_rows) {
  if (T <= 0 || nseq <= 0 || !delta_plan(T, nseq, H, G, D, Dv, v_ld, max_rows).records) return 0;
  return delta_chunks_at_once(T, nseq, H, G, D) * delta_chunk_floats(H, G, D);
}

template <typename T, int NT>
static void delta_records_launch(const float* q, long q_ld, const float* k, long k_ld, const float* v, long v_ld, const T* b,
                                 long b_ld, const T* a, long a_ld, const float* a_log, const float* dt_bias, float* state,
                                 const int* state_slots, const int* row_cu, int nseq, const int* positions, float q_scale,
                                 float unit_eps, float* o, float* rec, int T_, int H, int G, int D, int Dv, hipStream_t s, int cost) {
  constexpr size_t lds = (size_t)kDeltaSlots * (delta_rows(NT) + kDeltaHead + 1024) * sizeof(float);
  static bool once = false;
  if (!once) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&delta_chain_kernel<NT>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds);
    once = true;
  }
  // 1: rows of q and k, 2: columns of the state in four-element accesses
  int vec = 0;
  if (D % 4 == 0 && rows_aligned(q, q_ld, 4) && rows_aligned(k, k_ld, 4)) vec |= 1;
  if (D % 4 == 0) vec |= 2;
  const long all = (T_ >> 4) + nseq, most = delta_chunks_at_once(T_, nseq, H, G, D);
  for (long first = 0; first < all; first += most) {
    const int count = (int)std::min(most, all - first);
    delta_record_kernel<T, NT><<<dim3(G, count), 256, 0, s>>>(q, q_ld, k, k_ld, b, b_ld, a, a_ld, a_log, dt_bias, state_slots, row_cu,
                                                             nseq, q_scale, unit_eps, vec, rec, H, G, D, cost, (int)first);
    delta_chain_kernel<NT><<<(nseq * G + 7) / 8 * 8 * (H / G) * ((Dv + 63) / 64), 256, lds, s>>>(
        rec, v, v_ld, state, state_slots, row_cu, positions, vec, o, nseq, H, G, D, Dv, cost, (int)first, count);
  }
}

template <typename T>
static int delta_scan_t(const float* q, long q_ld, const float* k, long k_ld, const float* v, long v_ld, const T* b,
                        long b_ld, const T* a, long a_ld, const float* a_log, const float* dt_bias, float* state,
                        const int* state_slots, const int* row_cu, int nseq, const int* positions, float q_scale,
                        float unit_eps, float* o, float* rec, int T_, int H, int G, int D, int Dv, hipStream_t s, int max_rows) {
  const DeltaPlan plan = delta_plan(T_, nseq, H, G, D, Dv, v_ld, max_rows);
  const int cost = plan.form.rows ? plan.cost : 0;
  if (plan.form.chunks) {
    if (plan.records && !rec) return -2;
#define BFLY_DCH(NT)                                                                                                      \
  (plan.records ? delta_records_launch<T, NT>(q, q_ld, k, k_ld, v, v_ld, b, b_ld, a, a_ld, a_log, dt_bias, state,         \
                                              state_slots, row_cu, nseq, positions, q_scale, unit_eps, o, rec, T_, H, G, D, \
                                              Dv, s, cost)                                                                \
                : delta_chunk_launch<T, NT>(q, q_ld, k, k_ld, v, v_ld, b, b_ld, a, a_ld, a_log, dt_bias, state,           \
                                            state_slots, row_cu, nseq, positions, q_scale, unit_eps, o, H, G, D, Dv, s, cost))
    switch (delta_tiles(D)) {
      case 4: BFLY_DCH(4); break;
      case 8: BFLY_DCH(8); break;
      case 12: BFLY_DCH(12); break;
      default: BFLY_DCH(16);
    }
#undef BFLY_DCH
    if (!plan.form.rows) return 0;
  }
  dim3 grid(nseq, H, (Dv + 63) / 64);
#define BFLY_DELTA(NR)                                                                                             \
  delta_scan_kernel<T, NR><<<grid, 512, 0, s>>>(q, q_ld, k, k_ld, v, v_ld, b, b_ld, a, a_ld, a_log, dt_bias, state, \
                                                state_slots, row_cu, positions, q_scale, unit_eps, o, H, G, D, Dv, \
                                                plan.form.chunks ? plan.cost : 0)
  if (D <= 32) BFLY_DELTA(4);
  else if (D <= 64) BFLY_DELTA(8);
  else if (D <= 128) BFLY_DELTA(16);
  else if (D <= 256) BFLY_DELTA(32);
  else return -1;
#undef BFLY_DELTA
  return 0;
}

int launch_delta_scan(const float* q, long q_ld, const float* k, long k_ld, const float* v, long v_ld, const void* b,
                      long b_ld, const void* a, long a_ld, const float* a_log, const float* dt_bias, float* state,
                      const int* state_slots, const int* row_cu, int nseq, const int* positions, float q_scale,
                      float unit_eps, float* o, float* rec, int T, int H, int G, int D, int Dv, bool f32, hipStream_t s,
                      int max_rows) {
  if (T <= 0 || nseq <= 0) return 0;
  if (f32)
    return delta_scan_t<float>(q, q_ld, k, k_ld, v, v_ld, (const float*)b, b_ld, (const float*)a, a_ld, a_log, dt_bias,
                               state, state_slots, row_cu, nseq, positions, q_scale, unit_eps, o, rec, T, H, G, D, Dv,
                               s, max_rows);
  return delta_scan_t<bf16>(q, q_ld, k, k_ld, v, v_ld, (const bf16*)b, b_ld, (const bf16*)a, a_ld, a_log, dt_bias, state,
                            state_slots, row_cu, nseq, positions, q_scale, unit_eps, o, rec, T, H, G, D, Dv, s, max_rows);
}

}  // namespace bfly
