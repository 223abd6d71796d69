// Parallel residual streams (hyper-connections) with offset-weight RMS norms. The residual is
// S f32 streams per token, xs [T, S, W]. A sublayer reads one mixed-in row
// u = sum_s w_in[s] xs[s], normalised as u / sqrt(mean(u^2) + eps) * (w + offset) (offset 1: the
// weight is stored around zero), and its output y updates every stream from the old ones:
// xs[r] <- sum_s mix[s, r] xs[s] + w_out[r] y. One workgroup per token row; sums, norms and the
// streams are f32 whatever the activation type.
#include "bfly_common.h"
#include "bfly_mixers.h"

namespace bfly {

namespace {

constexpr int kMaxStreams = 16;

// The four passes over a token's streams below (update, mixed-in norm, both, output norm) for up to four streams and rows
// of whole 16-byte segments: a thread holds its columns of every stream in registers from the one read to the one
// write, four columns per access, and the norm takes the mixed row from registers. Bound by memory for large steps
// (S = 2, W = 2048 in bf16: 335 MB per 8192 rows) and by one load - reduce - store chain for decoded rows. The
// column-at-a-time forms further down (other shapes) read the streams twice, each time behind dependent loads: 8192
// rows 123 us, 16 rows 14 us; see launch_hc_rows.
template <typename T, int S, int NV, bool POST, bool PRE>
__global__ __launch_bounds__(256) void hc_rows_kernel(float* __restrict__ xs, const T* __restrict__ y,
                                                      const float* __restrict__ mix, const float* __restrict__ w_out,
                                                      const float* __restrict__ w_in, const float* __restrict__ norm_w,
                                                      float eps, float offset, const long* __restrict__ idx,
                                                      T* __restrict__ out, int W) {
  typedef T tv __attribute__((ext_vector_type(4)));
  __shared__ float red[16];
  const long i = blockIdx.x, t = idx ? idx[i] : i;
  float* x = xs + t * S * W;
  f32x4 v[NV][S], yv[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int c = 4 * ((int)threadIdx.x + 256 * n);
    if (c >= W) continue;
#pragma unroll
    for (int s = 0; s < S; ++s) v[n][s] = *reinterpret_cast<const f32x4*>(x + (long)s * W + c);
    if (POST) {
      const tv a = *reinterpret_cast<const tv*>(y + t * W + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) yv[n][e] = (float)a[e];
    }
  }
  f32x4 nw[NV];
  if (PRE) {      // (in flight beside the streams)
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int c = 4 * ((int)threadIdx.x + 256 * n);
      if (c < W) nw[n] = *reinterpret_cast<const f32x4*>(norm_w + c);
    }
  }
  if (POST) {
    float mx[S][S], wo[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      wo[s] = w_out[s];
#pragma unroll
      for (int r = 0; r < S; ++r) mx[s][r] = mix[s * S + r];
    }
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int c = 4 * ((int)threadIdx.x + 256 * n);
      if (c >= W) continue;
      f32x4 u[S];
#pragma unroll
      for (int r = 0; r < S; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float a = 0.f;
#pragma unroll
          for (int s = 0; s < S; ++s) a = fmaf(mx[s][r], v[n][s][e], a);
          u[r][e] = fmaf(wo[r], yv[n][e], a);
        }
#pragma unroll
      for (int r = 0; r < S; ++r) {
        v[n][r] = u[r];
        *reinterpret_cast<f32x4*>(x + (long)r * W + c) = u[r];
      }
    }
  }
  if (PRE) {
    float wi[S];
#pragma unroll
    for (int s = 0; s < S; ++s) wi[s] = w_in ? w_in[s] : 1.f;
    float ss = 0.f;
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      if (4 * ((int)threadIdx.x + 256 * n) >= W) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float a = 0.f;
#pragma unroll
        for (int s = 0; s < S; ++s) a = fmaf(wi[s], v[n][s][e], a);
        yv[n][e] = a;
        ss = fmaf(a, a, ss);
      }
    }
    ss = block_sum(ss, red);
    const float r = 1.f / sqrtf(ss / (float)W + eps);
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int c = 4 * ((int)threadIdx.x + 256 * n);
      if (c >= W) continue;
      tv o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (T)(yv[n][e] * r * (nw[n][e] + offset));
      *reinterpret_cast<tv*>(out + i * W + c) = o;
    }
  }
}

// four columns per access, the row in registers: W <= 1024 NV
template <typename T, int NV>
__global__ __launch_bounds__(256) void embed_norm_rows_kernel(const int* __restrict__ ids, const T* __restrict__ table,
                                                              const float* __restrict__ norm_w, float eps, float offset,
                                                              float* __restrict__ xs, int S, int W, int vocab) {
  typedef T tv __attribute__((ext_vector_type(4)));
  __shared__ float red[16];
  const int t = blockIdx.x;
  int id = ids[t];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
  const T* row = table + (long)id * W;
  f32x4 v[NV];
  float ss = 0.f;
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int c = 4 * ((int)threadIdx.x + 256 * n);
    if (c >= W) continue;
    const tv a = *reinterpret_cast<const tv*>(row + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[n][e] = (float)a[e];
      ss = fmaf(v[n][e], v[n][e], ss);
    }
  }
  ss = block_sum(ss, red);
  const float r = 1.f / sqrtf(ss / (float)W + eps);
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int c = 4 * ((int)threadIdx.x + 256 * n);
    if (c >= W) continue;
    const f32x4 nw = *reinterpret_cast<const f32x4*>(norm_w + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[n][e] = v[n][e] * r * (nw[e] + offset);
    for (int s = 0; s < S; ++s) *reinterpret_cast<f32x4*>(xs + ((long)t * S + s) * W + c) = v[n];
  }
}

template <typename T>
__global__ __launch_bounds__(256) void embed_norm_streams_kernel(const int* __restrict__ ids, const T* __restrict__ table,
                                                                 const float* __restrict__ norm_w, float eps,
                                                                 float offset, float* __restrict__ xs, int S, int W,
                                                                 int vocab) {
  __shared__ float red[16];
  const int t = blockIdx.x;
  int id = ids[t];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
  const T* row = table + (long)id * W;
  float ss = 0.f;
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    const float v = (float)row[c];
    ss = fmaf(v, v, ss);
  }
  ss = block_sum(ss, red);
  const float r = 1.f / sqrtf(ss / (float)W + eps);
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    const float v = (float)row[c] * r * (norm_w[c] + offset);
    for (int s = 0; s < S; ++s) xs[((long)t * S + s) * W + c] = v;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void hc_pre_kernel(const float* __restrict__ xs, const float* __restrict__ w_in,
                                                     const float* __restrict__ norm_w, float eps, float offset,
                                                     T* __restrict__ out, int S, int W) {
  __shared__ float red[16];
  const long t = blockIdx.x;
  const float* x = xs + t * S * W;
  float ss = 0.f;
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    float u = 0.f;
    for (int s = 0; s < S; ++s) u = fmaf(w_in[s], x[(long)s * W + c], u);
    ss = fmaf(u, u, ss);
  }
  ss = block_sum(ss, red);
  const float r = 1.f / sqrtf(ss / (float)W + eps);
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    float u = 0.f;
    for (int s = 0; s < S; ++s) u = fmaf(w_in[s], x[(long)s * W + c], u);
    out[t * W + c] = (T)(u * r * (norm_w[c] + offset));
  }
}

template <typename T>
__global__ __launch_bounds__(256) void hc_post_kernel(float* __restrict__ xs, const T* __restrict__ y,
                                                      const float* __restrict__ mix, const float* __restrict__ w_out,
                                                      int S, int W) {
  const long t = blockIdx.x;
  float* x = xs + t * S * W;
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    float old[kMaxStreams];
    for (int s = 0; s < S; ++s) old[s] = x[(long)s * W + c];
    const float yv = (float)y[t * W + c];
    for (int r = 0; r < S; ++r) {
      float v = 0.f;
      for (int s = 0; s < S; ++s) v = fmaf(mix[s * S + r], old[s], v);
      x[(long)r * W + c] = fmaf(w_out[r], yv, v);
    }
  }
}

// hc_post followed by the next sublayer's hc_pre on the updated streams, one pass over the row's
// streams for both (the same thread owns a column in both halves, so it rereads what it wrote).
template <typename T>
__global__ __launch_bounds__(256) void hc_post_pre_kernel(float* __restrict__ xs, const T* __restrict__ y,
                                                          const float* __restrict__ mix,
                                                          const float* __restrict__ w_out,
                                                          const float* __restrict__ w_in2,
                                                          const float* __restrict__ norm_w2, float eps, float offset,
                                                          T* __restrict__ out, int S, int W) {
  __shared__ float red[16];
  const long t = blockIdx.x;
  float* x = xs + t * S * W;
  float ss = 0.f;
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    float old[kMaxStreams];
    for (int s = 0; s < S; ++s) old[s] = x[(long)s * W + c];
    const float yv = (float)y[t * W + c];
    float u = 0.f;
    for (int r = 0; r < S; ++r) {
      float v = 0.f;
      for (int s = 0; s < S; ++s) v = fmaf(mix[s * S + r], old[s], v);
      v = fmaf(w_out[r], yv, v);
      x[(long)r * W + c] = v;
      u = fmaf(w_in2[r], v, u);
    }
    ss = fmaf(u, u, ss);
  }
  ss = block_sum(ss, red);
  const float r = 1.f / sqrtf(ss / (float)W + eps);
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    float u = 0.f;
    for (int s = 0; s < S; ++s) u = fmaf(w_in2[s], x[(long)s * W + c], u);
    out[t * W + c] = (T)(u * r * (norm_w2[c] + offset));
  }
}

template <typename T>
__global__ __launch_bounds__(256) void hc_final_kernel(const float* __restrict__ xs, const float* __restrict__ norm_w,
                                                       float eps, float offset, const long* __restrict__ idx,
                                                       T* __restrict__ out, int S, int W) {
  __shared__ float red[16];
  const long i = blockIdx.x;
  const long t = idx ? idx[i] : i;
  const float* x = xs + t * S * W;
  float ss = 0.f;
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    float u = 0.f;
    for (int s = 0; s < S; ++s) u += x[(long)s * W + c];
    ss = fmaf(u, u, ss);
  }
  ss = block_sum(ss, red);
  const float r = 1.f / sqrtf(ss / (float)W + eps);
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    float u = 0.f;
    for (int s = 0; s < S; ++s) u += x[(long)s * W + c];
    out[i * W + c] = (T)(u * r * (norm_w[c] + offset));
  }
}

inline bool al(const void* p, size_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

// hc_rows_kernel where it applies (S <= 4, W % 4 == 0, W <= 8192, aligned rows): 8192 rows of 2 x 2048 in bf16 123 -> 52 us
// with the update and the norm (6.4 TB/s), 16 rows 14 -> 4.6 us
template <typename T, bool POST, bool PRE>
bool launch_hc_rows(float* xs, const T* y, const float* mix, const float* w_out, const float* w_in, const float* norm_w,
                    float eps, float offset, const long* idx, T* out, int R, int S, int W, hipStream_t s) {
  if (S < 1 || S > 4 || W % 4 || W > 8192 || !al(xs, 16) || (POST && !al(y, 4 * sizeof(T))) ||
      (PRE && (!al(norm_w, 16) || !al(out, 4 * sizeof(T)))))
    return false;
#define BFLY_HR(S_, NV) \
  hc_rows_kernel<T, S_, NV, POST, PRE><<<R, 256, 0, s>>>(xs, y, mix, w_out, w_in, norm_w, eps, offset, idx, out, W)
#define BFLY_HRS(NV)                                              \
  {                                                               \
    if (S == 1) BFLY_HR(1, NV);                                   \
    else if (S == 2) BFLY_HR(2, NV);                              \
    else if (S == 3) BFLY_HR(3, NV);                              \
    else BFLY_HR(4, NV);                                          \
  }
  if (W <= 1024) BFLY_HRS(1)
  else if (W <= 2048) BFLY_HRS(2)
  else if (W <= 4096) BFLY_HRS(4)
  else BFLY_HRS(8)
#undef BFLY_HRS
#undef BFLY_HR
  return true;
}

template <typename T>
bool launch_embed_rows(const int* ids, const T* table, const float* norm_w, float eps, float offset, float* xs, int T_, int S,
                       int W, int vocab, hipStream_t s) {
  if (W % 4 || W > 8192 || !al(table, 4 * sizeof(T)) || !al(norm_w, 16) || !al(xs, 16)) return false;
#define BFLY_ER(NV) embed_norm_rows_kernel<T, NV><<<T_, 256, 0, s>>>(ids, table, norm_w, eps, offset, xs, S, W, vocab)
  if (W <= 1024) BFLY_ER(1);
  else if (W <= 2048) BFLY_ER(2);
  else if (W <= 4096) BFLY_ER(4);
  else BFLY_ER(8);
#undef BFLY_ER
  return true;
}

}  // namespace

void launch_embed_norm_streams(const int* ids, const void* table, const float* norm_w, float eps, float offset,
                               float* xs, int T, int S, int W, int vocab, bool f32, hipStream_t s) {
  if (T <= 0) return;
  if (f32 ? launch_embed_rows<float>(ids, (const float*)table, norm_w, eps, offset, xs, T, S, W, vocab, s)
          : launch_embed_rows<bf16>(ids, (const bf16*)table, norm_w, eps, offset, xs, T, S, W, vocab, s))
    return;
  if (f32) embed_norm_streams_kernel<float><<<T, 256, 0, s>>>(ids, (const float*)table, norm_w, eps, offset, xs, S, W, vocab);
  else embed_norm_streams_kernel<bf16><<<T, 256, 0, s>>>(ids, (const bf16*)table, norm_w, eps, offset, xs, S, W, vocab);
}

void launch_hc_pre(const float* xs, const float* w_in, const float* norm_w, float eps, float offset, void* out,
                   int T, int S, int W, bool f32, hipStream_t s) {
  if (T <= 0) return;
  float* xm = const_cast<float*>(xs);      // (only read without the update)
  if (f32 ? launch_hc_rows<float, false, true>(xm, nullptr, nullptr, nullptr, w_in, norm_w, eps, offset, nullptr, (float*)out, T, S, W, s)
          : launch_hc_rows<bf16, false, true>(xm, nullptr, nullptr, nullptr, w_in, norm_w, eps, offset, nullptr, (bf16*)out, T, S, W, s))
    return;
  if (f32) hc_pre_kernel<float><<<T, 256, 0, s>>>(xs, w_in, norm_w, eps, offset, (float*)out, S, W);
  else hc_pre_kernel<bf16><<<T, 256, 0, s>>>(xs, w_in, norm_w, eps, offset, (bf16*)out, S, W);
}

void launch_hc_post(float* xs, const void* y, const float* mix, const float* w_out, int T, int S, int W, bool f32,
                    hipStream_t s) {
  if (T <= 0) return;
  if (f32 ? launch_hc_rows<float, true, false>(xs, (const float*)y, mix, w_out, nullptr, nullptr, 0.f, 0.f, nullptr, nullptr, T, S, W, s)
          : launch_hc_rows<bf16, true, false>(xs, (const bf16*)y, mix, w_out, nullptr, nullptr, 0.f, 0.f, nullptr, nullptr, T, S, W, s))
    return;
  if (f32) hc_post_kernel<float><<<T, 256, 0, s>>>(xs, (const float*)y, mix, w_out, S, W);
  else hc_post_kernel<bf16><<<T, 256, 0, s>>>(xs, (const bf16*)y, mix, w_out, S, W);
}

void launch_hc_post_pre(float* xs, const void* y, const float* mix, const float* w_out, const float* w_in2,
                        const float* norm_w2, float eps, float offset, void* out, int T, int S, int W, bool f32,
                        hipStream_t s) {
  if (T <= 0) return;
  if (f32 ? launch_hc_rows<float, true, true>(xs, (const float*)y, mix, w_out, w_in2, norm_w2, eps, offset, nullptr, (float*)out, T, S, W, s)
          : launch_hc_rows<bf16, true, true>(xs, (const bf16*)y, mix, w_out, w_in2, norm_w2, eps, offset, nullptr, (bf16*)out, T, S, W, s))
    return;
  if (f32)
    hc_post_pre_kernel<float><<<T, 256, 0, s>>>(xs, (const float*)y, mix, w_out, w_in2, norm_w2, eps, offset, (float*)out, S, W);
  else
    hc_post_pre_kernel<bf16><<<T, 256, 0, s>>>(xs, (const bf16*)y, mix, w_out, w_in2, norm_w2, eps, offset, (bf16*)out, S, W);
}

void launch_hc_final(const float* xs, const float* norm_w, float eps, float offset, const long* idx, void* out,
                     int R, int S, int W, bool f32, hipStream_t s) {
  if (R <= 0) return;
  float* xm = const_cast<float*>(xs);
  if (f32 ? launch_hc_rows<float, false, true>(xm, nullptr, nullptr, nullptr, nullptr, norm_w, eps, offset, idx, (float*)out, R, S, W, s)
          : launch_hc_rows<bf16, false, true>(xm, nullptr, nullptr, nullptr, nullptr, norm_w, eps, offset, idx, (bf16*)out, R, S, W, s))
    return;
  if (f32) hc_final_kernel<float><<<R, 256, 0, s>>>(xs, norm_w, eps, offset, idx, (float*)out, S, W);
  else hc_final_kernel<bf16><<<R, 256, 0, s>>>(xs, norm_w, eps, offset, idx, (bf16*)out, S, W);
}

}  // namespace bfly
