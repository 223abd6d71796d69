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
// Rows of a step are packed: sequence s owns rows row_cu[s] .. row_cu[s+1].
#include <algorithm>

#include "bfly_common.h"
#include "bfly_delta.h"
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
template <typename T, bool RMS, int NV>
__global__ __launch_bounds__(256) void post_norm_rows_kernel(float* __restrict__ x, const T* __restrict__ y,
                                                             const float* __restrict__ nw, const float* __restrict__ nb,
                                                             float eps, float mult, const float* __restrict__ extra,
                                                             const float* __restrict__ nw2, const float* __restrict__ nb2,
                                                             T* __restrict__ h, int W) {
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
    yv[i] = *reinterpret_cast<const tv*>(y + t * W + c);
    xv[i] = *reinterpret_cast<const f32x4*>(x + t * W + c);
    if (extra) ev[i] = *reinterpret_cast<const f32x4*>(extra + t * W + c);
    wv[i] = *reinterpret_cast<const f32x4*>(nw + c);
    if (!RMS) bv[i] = *reinterpret_cast<const f32x4*>(nb + c);
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

// threads of a one-row workgroup: about four elements per thread, whole waves, at most 1024
int row_threads(int W) { return std::min(1024, std::max(64, (W / 4 + 63) / 64 * 64)); }

}  // namespace

void launch_post_norm_add_norm(float* x, const void* y, const float* nw, const float* nb, float eps, float mult,
                               const float* extra, const float* nw2, const float* nb2, void* h, int T, int W, bool rms,
                               bool f32, hipStream_t s) {
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
  if (W % 4 == 0 && W > 256 && W <= 4096) {
#define BFLY_PNR(TT, R, NV) \
  post_norm_rows_kernel<TT, R, NV><<<T, 256, 0, s>>>(x, (const TT*)y, nw, nb, eps, mult, extra, nw2, nb2, (TT*)h, W)
#define BFLY_PNR2(TT, R)                                                                             \
  {                                                                                                  \
    if (W <= 1024) BFLY_PNR(TT, R, 1); else if (W <= 2048) BFLY_PNR(TT, R, 2); else BFLY_PNR(TT, R, 4); \
  }
    if (f32) { if (rms) BFLY_PNR2(float, true) else BFLY_PNR2(float, false) }
    else { if (rms) BFLY_PNR2(bf16, true) else BFLY_PNR2(bf16, false) }
#undef BFLY_PNR2
#undef BFLY_PNR
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

template <typename T>
static int delta_scan_t(const float* q, long q_ld, const float* k, long k_ld, const float* v, long v_ld, const T* b,
                        long b_ld, const T* a, long a_ld, const float* a_log, const float* dt_bias, float* state,
                        const int* state_slots, const int* row_cu, int nseq, const int* positions, float q_scale,
                        float unit_eps, float* o, int T_, int H, int G, int D, int Dv, hipStream_t s, int max_rows) {
  // A chunk takes the time of 10 rows of 128 channels while the workgroups all run at once, and of 14 where they queue (the
  // loop's have half the LDS): 16 heads of 128, time of chunks over loop for one sequence of 8, 12, 16, 20, 32 rows 1.07, 0.88,
  // 0.80, 0.85, 0.66, for 64 of them 1.24, 1.06, 1.05, 1.23, 0.91; channels of 64 0.82 and 0.94 at 16 rows, of 32 0.91 and 1.14,
  // of 192 0.51 and 0.49. With each sequence in its own form: 32 single rows beside 128 114 and 63 us, now 58; 200 beside 300
  // 249 and 291, now 173.
  const long wgs = (long)H * ((Dv + 63) / 64);
  const bool queue = nseq * wgs >= 1024;
  const int cost = D > 128 ? 8 : D > 64 ? (queue ? 14 : 10) : D > 32 ? (queue ? 12 : 10) : queue ? 15 : 12;
  ScanForms form = scan_forms(T_, nseq, cost, wgs, max_rows);
  if (D > 256) form = {true, false};
  if (form.chunks) {
#define BFLY_DCH(NT)                                                                                                    \
  delta_chunk_launch<T, NT>(q, q_ld, k, k_ld, v, v_ld, b, b_ld, a, a_ld, a_log, dt_bias, state, state_slots, row_cu, nseq, \
                            positions, q_scale, unit_eps, o, H, G, D, Dv, s, form.rows ? cost : 0)
    if (D <= 64) BFLY_DCH(4);
    else if (D <= 128) BFLY_DCH(8);
    else if (D <= 192) BFLY_DCH(12);
    else BFLY_DCH(16);
#undef BFLY_DCH
    if (!form.rows) return 0;
  }
  dim3 grid(nseq, H, (Dv + 63) / 64);
#define BFLY_DELTA(NR)                                                                                             \
  delta_scan_kernel<T, NR><<<grid, 512, 0, s>>>(q, q_ld, k, k_ld, v, v_ld, b, b_ld, a, a_ld, a_log, dt_bias, state, \
                                                state_slots, row_cu, positions, q_scale, unit_eps, o, H, G, D, Dv, form.chunks ? cost : 0)
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
                      float unit_eps, float* o, int T, int H, int G, int D, int Dv, bool f32, hipStream_t s, int max_rows) {
  if (T <= 0 || nseq <= 0) return 0;
  if (f32)
    return delta_scan_t<float>(q, q_ld, k, k_ld, v, v_ld, (const float*)b, b_ld, (const float*)a, a_ld, a_log, dt_bias,
                               state, state_slots, row_cu, nseq, positions, q_scale, unit_eps, o, T, H, G, D, Dv, s,
                               max_rows);
  return delta_scan_t<bf16>(q, q_ld, k, k_ld, v, v_ld, (const bf16*)b, b_ld, (const bf16*)a, a_ld, a_log, dt_bias, state,
                            state_slots, row_cu, nseq, positions, q_scale, unit_eps, o, T, H, G, D, Dv, s, max_rows);
}

}  // namespace bfly
