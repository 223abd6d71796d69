// Linear attention with a gate per head and channel as decay and its complement as key, and the norm per head that
// follows a linear attention; generic in every size and in the activation type (bf16 or f32; gates, decays, states
// and the recurrence are f32 in both):
//   gate_chunk_kernel, gate_chain_kernel      f = l + (1 - l) sigmoid(z + b), S <- diag(f) S + (1 - f) v^T, o = S^T q,
//                                             in chunks on the f32 matrix cores; also gated linear attention, whose key
//                                             is an input (GLA)
//   gate_scan_kernel                          the same in one launch, for short sequences
//   forget_step_kernel                        the same row by row
//   head_norm_gate_kernel                     RMS norm per head, times an optional weight, a gate and a factor
// Rows of a step are packed: sequence s owns rows row_cu[s] .. row_cu[s+1]; a sequence whose first row is at
// position 0 starts from a zero state whatever its slot holds.
#include <algorithm>
#include <type_traits>

#include "bfly_recur.h"
#include "bfly_recur_dev.h"

namespace bfly {

namespace {

// sigmoid(x) and its complement, each with its own relative accuracy
template <bool FAST>
__device__ __forceinline__ void sigmoid2(float x, float& s, float& c) {
  const float e = FAST ? __expf(-fabsf(x)) : expf(-fabsf(x));
  const float r = FAST ? __builtin_amdgcn_rcpf(1.f + e) : 1.f / (1.f + e);
  s = x < 0.f ? e * r : r;
  c = x < 0.f ? r : e * r;
}

// sigmoid(z)^(1 / tau): exp of the log sigmoid, stable on both sides
template <bool FAST>
__device__ __forceinline__ float gla_decay(float z, float inv_tau) {
  const float e = FAST ? __expf(-fabsf(z)) : expf(-fabsf(z));
  const float ls = fminf(z, 0.f) - (FAST ? __logf(1.f + e) : log1pf(e));
  return FAST ? __expf(ls * inv_tau) : expf(ls * inv_tau);
}

// One element at a byte offset below 2^31 from a uniform base. (Rows of one chunk; callers clamp row and channel to the
// tensor.)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, 0x7fffffff, 0x00027000);
}
template <typename T>
__device__ __forceinline__ T row_load(__amdgpu_buffer_rsrc_t r, int off) {
  if constexpr (sizeof(T) == 2) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0));
  else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

// sum over the 32 lanes of a half wave, in its upper sixteen lanes
__device__ __forceinline__ float half_sum(float v) {
  v = row16_sum(v);
  return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x142, 0xA, 0xF, false));
}

// Chunks of 16 rows. With F_t = f_0 .. f_t and B_j = f_(j+1) .. f_(n-1) (products per channel over the chunk's rows) and S the
// state before it,
//   o_t = (q_t F_t) S + sum_(j <= t) P_tj v_j,  P_tj = sum_d q_td k_jd f_(j+1)d .. f_td,    S <- diag(F_(n-1)) S + sum_j (k_j B_j) v_j^T
// with k = 1 - f. Only products of decays occur, never quotients, so gates of any size are safe. All of a chunk but its
// products with the state is independent of the chunks before it, so it comes in two launches: gate_chunk_kernel leaves q F,
// k B, F_(n-1) and P of every chunk and head in a record, in the operand layout of the 16x16x4 f32 tiles, and
// gate_chain_kernel runs down the records of a sequence with nothing but matrix products and the loads of the next record.
// 8 sequences of 1024 rows, 16 heads of 128 x 128: 72 us for the records (1.1 KB a row and head, written and read once: 3.6
// TB/s) and 102 us for the chains (1.5 us a chunk, a wave's 68 matrix instructions alone 0.9); one kernel for both, whose waves formed
// the gates between two barriers of every chunk, 334 us. One sequence of 2000 rows 624 -> 186 us, in f32 769 -> 193.
// A chunk's record is at its sequence's first row / 16 + the sequence's number + its own number there: no two chunks of a
// step share one, and (rows / 16 + sequences) records are enough.
// Floats of a record: q F, k B [NT][64][4], F [16 NT], P [64][4]; whole KBs, which a wave copies at once
constexpr int chunk_record(int NT) { return (16 * NT * 33 + 256 + 255) / 256 * 256; }
constexpr int kChainSlots = 3;
typedef __attribute__((address_space(3))) void* lds_ptr_t;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void* base, long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)min(bytes, 0x7fffffffL), 0x00020000);
}
template <int N>
__device__ __forceinline__ void vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Workgroup = (head, chunk), two lanes per channel with eight rows each, which form the running products on the way into LDS.
// Of the 16 x 16 weights P the block t >= 8 > j is a matrix product, with the decays split at row 8 (both factors are the
// lanes' own running products); the two 8 x 8 blocks on the diagonal are formed on the vector units: 32 lanes per row t share
// its channels, and q_t times the decays so far is carried down j. Rows past the sequence have f = 1, k = q = 0, channels past
// D k = q = 0. D <= 16 NT, NT even. GLA: f = sigmoid(z)^(1 / tau) and k is an input.
template <typename T, int NT, bool GLA>
__global__ __launch_bounds__(32 * NT) void gate_chunk_kernel(const T* __restrict__ q, long q_ld, const T* __restrict__ key,
                                                             long k_ld, float inv_tau, float q_scale, const T* __restrict__ z,
                                                             long z_ld, const float* __restrict__ f_bias,
                                                             const float* __restrict__ lower,
                                                             const int* __restrict__ state_slots,
                                                             const int* __restrict__ row_cu, int nseq, int act,
                                                             float* __restrict__ rec, int H, int D, int cost, int first) {
  constexpr int C = 16, DP = 16 * NT, NU = (DP + 127) / 128, KP = DP + 4, PP = C + 4, HC = C / 2, W = NT / 2;
  constexpr bool FAST = sizeof(T) == 2;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float* sq = smem;                     // [C][KP] q
  float* sk = sq + C * KP;              // [C][KP] k
  float* sf = sk + C * KP;              // [C + 1][KP] f; row C holds ones
  float* sqf = sf + (C + 1) * KP;       // [C][KP] q F
  float* sqh = sqf + C * KP;            // [HC][KP] q times the decays from row 8 on, of rows 8 .. 15
  float* skh = sqh + HC * KP;           // [HC][KP] k times the decays up to row 7, of rows 0 .. 7
  float* sp = skh + HC * KP;            // [C][PP] weights; those of rows 8 .. 15 on columns 0 .. 7 come as the sum of
  float* sph = sp + C * PP;             // [W][HC][HC] the waves' parts
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, m = lane & 15, gg = lane >> 4;
  const int h = blockIdx.x, b = first + blockIdx.y;
  int s = -1;      // the last sequence whose records begin at or before b
  for (int i0 = 0; i0 < nseq; i0 += 64) {
    const int i = i0 + lane;
    const unsigned long long le = __ballot(i < nseq && (row_cu[min(i, nseq)] >> 4) + i <= b);
    s += __popcll(le);
    if (~le) break;
  }
  if (s < 0) return;
  const int r0 = __builtin_amdgcn_readfirstlane(row_cu[s]), r1 = __builtin_amdgcn_readfirstlane(row_cu[s + 1]);
  const int t0 = r0 + C * (b - (r0 >> 4) - s), n = min(C, r1 - t0);
  if (n <= 0 || (cost && !scan_in_chunks(r1 - r0, cost)) || state_slots[s] < 0) return;
  rec += ((long)blockIdx.y * H + h) * chunk_record(NT);
  // this thread's channel and rows ra .. ra + 7
  const int d = 32 * wave + (lane & 31), hf = lane >> 5, ra = HC * hf, dc = min(d, D - 1), last = n - 1;
  T rq[HC], rk[HC], rz[HC];
  {
    const T* qp = q + (long)t0 * q_ld + (long)h * D + dc;
    const T* zp = z + (long)t0 * z_ld + (long)h * D + dc;
    const T* kp = GLA ? key + (long)t0 * k_ld + (long)h * D + dc : qp;
#pragma unroll
    for (int i = 0; i < HC; ++i) rz[i] = zp[min(ra + i, last) * z_ld];
#pragma unroll
    for (int i = 0; i < HC; ++i) rq[i] = qp[min(ra + i, last) * q_ld];
    if constexpr (GLA)
#pragma unroll
      for (int i = 0; i < HC; ++i) rk[i] = kp[min(ra + i, last) * k_ld];
  }
  const float fb = GLA ? 0.f : f_bias[(long)h * D + dc], lo = GLA ? 0.f : lower[(long)h * D + dc];
  for (int i = tid; i < KP; i += 32 * NT) sf[C * KP + i] = 1.f;
  if (tid < HC * HC) sp[(tid / HC) * PP + HC + tid % HC] = 0.f;      // (above the diagonal blocks)
  float f[HC], kv[HC], w[HC], F = 1.f;
#pragma unroll
  for (int i = 0; i < HC; ++i) {
    float qv;
    if constexpr (GLA) {
      f[i] = gla_decay<FAST>((float)rz[i], inv_tau);
      kv[i] = (float)rk[i];
      qv = (float)rq[i] * q_scale;
    } else {
      float sg, cg;
      sigmoid2<FAST>((float)rz[i] + fb, sg, cg);
      f[i] = fmaf(1.f - lo, sg, lo);
      kv[i] = (1.f - lo) * cg;
      qv = act_in<FAST>((float)rq[i], act);
    }
    const bool in = ra + i < n;
    f[i] = in ? f[i] : 1.f;
    kv[i] = in && d < D ? kv[i] : 0.f;
    qv = in && d < D ? qv : 0.f;
    F *= f[i];
    w[i] = qv * F;
    sq[(ra + i) * KP + d] = qv;
    sk[(ra + i) * KP + d] = kv[i];
    sf[(ra + i) * KP + d] = f[i];
  }
  const float Fo = __shfl_xor(F, 32, 64), qby = hf ? Fo : 1.f, kby = hf ? 1.f : Fo;
  float B = 1.f;
  f32x4 kb[2];
#pragma unroll
  for (int i = HC - 1; i >= 0; --i) {
    const float x = kv[i] * B;
    kb[i >> 2][i & 3] = x * kby;
    if (!hf) skh[i * KP + d] = x;
    B *= f[i];
  }
#pragma unroll
  for (int i = 0; i < HC; ++i) {
    sqf[(ra + i) * KP + d] = w[i] * qby;
    if (hf) sqh[i * KP + d] = w[i];
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
    *reinterpret_cast<f32x4*>(rec + 16 * DP + (((d >> 4) * 64 + (2 * hf + i) * 16 + (d & 15)) << 2)) = kb[i];
  if (!hf) rec[32 * DP + d] = F * Fo;
  __syncthreads();
  // q F; this wave's channels of the weights of rows 8 .. 15 on columns 0 .. 7
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = wave; i < NT; i += W) {
    *reinterpret_cast<f32x4*>(rec + ((i * 64 + lane) << 2)) = *reinterpret_cast<const f32x4*>(sqf + m * KP + 16 * i + 4 * gg);
    const int at = (m & 7) * KP + 16 * i + 4 * gg;
    const f32x4 a = *reinterpret_cast<const f32x4*>(sqh + at), c = *reinterpret_cast<const f32x4*>(skh + at);
#pragma unroll
    for (int e = 0; e < 4; ++e) x = mfma_f32(a[e], c[e], x);
  }
  if (m < HC && gg < 2) {
#pragma unroll
    for (int e = 0; e < 4; ++e) sph[(wave * HC + 4 * gg + e) * HC + m] = x[e];
  }
  // the diagonal blocks: rows tb and 8 + tb, 32 lanes each share the row's channels, lane 16 + j keeps column j
#pragma unroll 1
  for (int i = wave; i < HC; i += W) {
    const int tb = W == 4 && i >= W ? 11 - i : i;      // (four waves get rows of equal work)
    int at[NU];      // (a lane past the channels: the last ones again, with q = 0)
    f32x4 qd[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      at[u] = min(128 * u + 4 * (lane & 31), DP - 4);
      qd[u] = *reinterpret_cast<const f32x4*>(sq + (ra + tb) * KP + at[u]);
      if (128 * u + 4 * (lane & 31) >= DP) qd[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    float keep = 0.f;
#pragma unroll
    for (int j = HC - 1; j >= 0; --j) {
      if (j > tb) continue;
      const float* fr = sf + (j < tb ? ra + j + 1 : C) * KP;      // (its own column: not decayed yet)
      const float* kr = sk + (ra + j) * KP;
      float y = 0.f;
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        qd[u] *= *reinterpret_cast<const f32x4*>(fr + at[u]);
        const f32x4 kk = *reinterpret_cast<const f32x4*>(kr + at[u]);
#pragma unroll
        for (int e = 0; e < 4; ++e) y = fmaf(qd[u][e], kk[e], y);
      }
      y = half_sum(y);
      keep = m == j ? y : keep;
    }
    if ((lane & 16) && m < HC) sp[(ra + tb) * PP + ra + m] = keep;
  }
  __syncthreads();
  if (wave) return;
  f32x4 p = *reinterpret_cast<const f32x4*>(sp + m * PP + 4 * gg);
  if (m >= HC && gg < 2) {
    p = *reinterpret_cast<const f32x4*>(sph + (m - HC) * HC + 4 * gg);
#pragma unroll
    for (int i = 1; i < W; ++i) p += *reinterpret_cast<const f32x4*>(sph + (i * HC + m - HC) * HC + 4 * gg);
  }
  *reinterpret_cast<f32x4*>(rec + 33 * DP + (lane << 2)) = p;
}

// Workgroup = (sequence, head, 64 value columns), four waves of 16 columns with the whole height of the state each. The columns of a
// head read the same records: they follow eight workgroups apart, in one XCD, and heads and sequences over all of them, also the few
// whose records a launch of a long step holds (64 heads of 128, 32 sequences of 512 rows in five launches: 590 us each with the
// sequences first, now 141). The state stays in the accumulator layout (tile i, element e: row d = 16 i + 4 gg + e of lane group gg),
// which is also the B operand of (q F) S. Records arrive by LDS-DMA, SL chunks ahead (a chunk's products take 0.9 us, a record from
// memory two). The records [first, first + count) of the step; a sequence that goes on in the next ones leaves its state in its slot.
// A weight of zero does not hide a NaN: values v that are no numbers go in as zeros, and the outputs of their column are NaN
// from their row on, as a row-by-row scan leaves them. (All other factors meet rows after theirs only.)
template <typename T, int NT>
__global__ __launch_bounds__(256, NT <= 8 ? 2 : 1) void gate_chain_kernel(
    const float* __restrict__ rec, const T* __restrict__ v, long v_ld, float* __restrict__ state,
    const int* __restrict__ state_slots, const int* __restrict__ row_cu, const int* __restrict__ positions,
    float* __restrict__ o, int nseq, int H, int D, int Dv, int cost, int first, int count) {
  constexpr int C = 16, DP = 16 * NT, SL = kChainSlots, REC = chunk_record(NT), U = REC / 256, PER = (U + 3) / 4;
  extern __shared__ __attribute__((aligned(16))) float smem[];      // [SL][REC], then values: [SL][4 waves][4][64]
  const int nz = (Dv + 63) / 64, u = blockIdx.x >> 3, pair = u / nz * 8 + (blockIdx.x & 7);
  if (pair / H >= nseq) return;
  const int s = NT <= 8 ? by_length(row_cu, nseq, pair / H, 256 / (H * nz)) : pair / H, h = pair % H, c0 = u % nz * 64;
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
  float* S = state + ((long)slot * H + h) * D * Dv + col;
  const bool fresh = cb == 0 && positions[r0] == 0;
  f32x4 st[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int d = 16 * i + 4 * gg + e;
      st[i][e] = (!fresh && live && d < D) ? S[(long)d * Dv] : 0.f;
    }
  // All addresses are a scalar base and offset per chunk and a constant per lane: the vector units have the products' operands
  // to scale. Rows past the sequence and columns past the head lie past the buffer's end: they read zeros and are not stored.
  const auto rs = buffer(rec + ((long)(at + cb - first) * H + h) * REC, 0x7fffffff);
  const int lastn = min(C, r1 - r0 - (ce - 1) * C);      // rows of the last chunk here
  const long ve = (long)(C - 1) * v_ld + Dv, vl = (long)(lastn - 1) * v_ld + Dv, ol = ((long)(lastn - 1) * H + 1) * Dv;
  const int vbytes = (int)min(ve * (long)sizeof(T), 0x7fffffffL), vlast = (int)min(vl * (long)sizeof(T), 0x7fffffffL);
  const int olast = (int)min(ol * 4, 0x7fffffffL);
  int va[4], oo[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    va[e] = live ? (int)((4 * gg + e) * v_ld + col) * (int)sizeof(T) : -1;
    oo[e] = live ? ((4 * gg + e) * H * Dv + col) * 4 : -1;
  }
  const T* vp = v + (long)(r0 + cb * C) * v_ld + (long)h * Dv;
  float* op = o + ((long)(r0 + cb * C) * H + h) * Dv;
  // operation j of PER + 4 of chunk c's copy: a part of its record, then the lanes' own four values (one to a word; loads into
  // registers would be waited for with everything in flight). Past the last chunk: that one again, into a slot nobody reads.
  auto dma = [&](int c, int sl, int j) {
    c = min(c, ce - 1);
    if (j < PER) {
      const int u = min(wave + 4 * j, U - 1);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(smem + sl * REC + 256 * u), 16, 16 * lane,
                                               (c - cb) * H * REC * 4 + 1024 * u, 0, 0);
    } else {
      const auto vs = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(vp + (long)((c - cb) * C) * v_ld), (short)0,
                                                        c == ce - 1 ? vlast : vbytes, 0x00020000);
      const lds_ptr_t to = (lds_ptr_t)(smem + SL * REC + ((sl * 4 + wave) * 4 + j - PER) * 64);
      if constexpr (sizeof(T) == 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(vs, to, 2, va[j - PER], 0, 0, 0);
      else __builtin_amdgcn_raw_ptr_buffer_load_lds(vs, to, 4, va[j - PER], 0, 0, 0);
    }
  };
#pragma unroll
  for (int i = 0; i < SL; ++i)
#pragma unroll
    for (int j = 0; j < PER + 4; ++j) dma(cb + i, i, j);
  f32x4 qf[NT], kf[NT], ff[NT];
  float raw[4];
  auto rows = [&](int sl, int i) { qf[i] = *reinterpret_cast<const f32x4*>(smem + sl * REC + ((i * 64 + lane) << 2)); };
  auto values = [&](int sl) {
#pragma unroll
    for (int e = 0; e < 4; ++e) raw[e] = smem[SL * REC + ((sl * 4 + wave) * 4 + e) * 64 + lane];
  };
  vm_wait<(SL - 1) * (PER + 4)>();
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < NT; ++i) rows(0, i);
  values(0);
  int sl = 0;
  // The fragments of a product are read while the one before it runs: k B, F and P during (q F) S, the next chunk's q F during
  // the state's update. The one barrier of a chunk lies between the two: behind it the chunk's slot is free. Everything else,
  // the state's decay and the copies included, stands between products (a lone wave has nothing else to cover it).
  for (int c = cb; c < ce; ++c) {
    const float* x = smem + sl * REC;
    const f32x4 p = *reinterpret_cast<const f32x4*>(x + 33 * DP + (lane << 2));
    f32x4 oa = {0.f, 0.f, 0.f, 0.f}, ob = oa;
    float bv[4], bo[4], zero = 0.f;      // (x * 0 of an infinity or NaN is NaN)
#pragma unroll
    for (int i = 0; i < NT; i += 2) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        oa = mfma_f32(qf[i][e], st[i][e], oa);
        ob = mfma_f32(qf[i + 1][e], st[i + 1][e], ob);
        if (e == 1) {
#pragma unroll
          for (int j = i; j < i + 2; ++j) {
            kf[j] = *reinterpret_cast<const f32x4*>(x + 16 * DP + ((j * 64 + lane) << 2));
            ff[j] = *reinterpret_cast<const f32x4*>(x + 32 * DP + 16 * j + 4 * gg);
          }
        }
        if (i == 0) {
          bv[e] = sizeof(T) == 2 ? __uint_as_float(__float_as_uint(raw[e]) << 16) : raw[e];
          bo[e] = bv[e];
          zero = fmaf(bv[e], 0.f, zero);
        } else if (e > 1) {      // (these tiles have gone into their products)
          st[i - 4 + e] *= ff[i - 4 + e];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    int odd = C;           // first row of this column that is no number
    if (__any(zero != 0.f)) {
#pragma unroll
      for (int e = 3; e >= 0; --e) {
        const bool bad = bv[e] * 0.f != 0.f;
        odd = bad ? 4 * gg + e : odd;
        bo[e] = bad ? 0.f : bv[e];
      }
      odd = min(odd, __shfl_xor(odd, 16, 64));
      odd = min(odd, __shfl_xor(odd, 32, 64));
    }
    // A turn of the loop issues PER + 8 memory operations (a record, values, outputs), the start has no outputs: with as many
    // of the newest in flight, the next chunk's record has landed (own part).
    if (c - cb < SL - 1) vm_wait<(SL - 2) * (PER + 4)>();
    else vm_wait<(SL - 2) * (PER + 8)>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    const int nx = sl + 1 == SL ? 0 : sl + 1;
    constexpr int OPS = PER + 4, QS = 4 * NT / 2;      // (half the slots of a tile's product each)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        if (e == 0 && i >= NT - 2) st[i] *= ff[i];
        st[i] = mfma_f32(kf[i][e], bv[e], st[i]);
        if (i == NT - 1) ob = mfma_f32(p[e], bo[e], ob);
        const int n = e * NT + i;
        if (n < NT) rows(nx, n);
        if (n == NT) values(nx);
        // the copies, spread over the second half
        if (n >= QS) {
#pragma unroll
          for (int j = (n - QS) * OPS / QS; j < (n - QS + 1) * OPS / QS; ++j) dma(c + SL, sl, j);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    sl = nx;
    oa += ob;
    if (__any(odd < C)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) oa[e] = 4 * gg + e >= odd ? NAN : oa[e];
    }
    const auto out = __builtin_amdgcn_make_buffer_rsrc(op, (short)0, c == ce - 1 ? olast : 0x7fffffff, 0x00020000);
#pragma unroll
    for (int e = 0; e < 4; ++e) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(oa[e]), out, oo[e], 0, 0);
    op += (long)C * H * Dv;
  }
  vm_wait<0>();      // no LDS-DMA may outlive the workgroup
  if (live) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int d = 16 * i + 4 * gg + e;
        if (d < D) S[(long)d * Dv] = st[i][e];
      }
  }
}

// Both parts of a chunk in one launch, for steps whose longest sequence has one or a few chunks (one_launch_rows): the second
// launch and the records' way through memory would be most of the time. Workgroup = (sequence, head, 64 value columns), eight
// waves: wave & 3 names 16 columns, wave >> 2 a half of the state's rows. The first DP of 2 DP roles stage q, f and q F, the others
// k and k B; the diagonal blocks of P are formed on the vector units while the matrix cores are busy. Row strides below 2^21
// elements (24-bit byte offsets). Values that are no numbers as in gate_chain_kernel.
template <typename T, int NT, bool GLA>
__global__ __launch_bounds__(512, NT <= 8 ? 4 : 2) void gate_scan_kernel(const T* __restrict__ q, long q_ld,
                                                           const T* __restrict__ key, long k_ld, float inv_tau, float q_scale,
                                                           const T* __restrict__ z, long z_ld, const T* __restrict__ v, long v_ld,
                                                           const float* __restrict__ f_bias,
                                                           const float* __restrict__ lower, float* __restrict__ state,
                                                           const int* __restrict__ state_slots,
                                                           const int* __restrict__ row_cu,
                                                           const int* __restrict__ positions, int act, int vec,
                                                           float* __restrict__ o, int H, int D, int Dv, int cost) {
  constexpr int C = 16, DP = 16 * NT, NH = NT / 2, NU = (DP + 127) / 128, KP = 128 * NU + 4, VP = 68, PP = C + 4;
  constexpr int NI = (2 * DP + 255) / 256, HC = C / 2, NP = NT < 8 ? NT : 8;
  constexpr bool FAST = sizeof(T) == 2, WHOLE = NI * 256 == 2 * DP;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float* sq = smem;                     // [C][KP] q
  float* sk = sq + C * KP;              // [C][KP] k
  float* sf = sk + C * KP;              // [C + 1][KP] f; row C holds ones
  float* sqf = sf + (C + 1) * KP;       // [C][KP] q F
  float* skb = sqf + C * KP;            // [C][KP] k B
  float* sqh = skb + C * KP;            // [HC][KP] q times the decays from row 8 on, of rows 8 .. 15
  float* skh = sqh + HC * KP;           // [HC][KP] k times the decays up to row 7, of rows 0 .. 7
  float* sv = skh + HC * KP;            // [C][VP]
  float* so = sv + C * VP;              // [C][VP] (q F) S over the second half of the state's rows
  float* sp = so + C * VP;              // [C][PP] weights; those of rows 8 .. 15 on columns 0 .. 7 come as the sum of
  float* sph = sp + C * PP;             // [NP][HC][HC] the waves' parts
  float* sl = sph + NP * HC * HC;       // [DP] F of the last row
  const int s = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * 64;
  const int r0 = __builtin_amdgcn_readfirstlane(row_cu[s]), r1 = __builtin_amdgcn_readfirstlane(row_cu[s + 1]);
  if (r1 <= r0 || (cost && !scan_in_chunks(r1 - r0, cost))) return;      // (the row-by-row form's)
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, m = lane & 15, gg = lane >> 4;
  const int slot = state_slots[s];
  if (slot < 0) {      // padding sequence of a fixed-shape step: defined output, no state
    for (int i = tid; i < (r1 - r0) * 64; i += 512)
      if (c0 + (i & 63) < Dv) o[((long)(r0 + (i >> 6)) * H + h) * Dv + c0 + (i & 63)] = 0.f;
    return;
  }
  const int cl = 16 * (wave & 3) + m, col = c0 + cl, d0 = (wave >> 2) * 16 * NH;
  const bool live = col < Dv;
  float* S = state + ((long)slot * H + h) * D * Dv + col;
  const bool fresh = positions[r0] == 0;
  f32x4 st[NH];
#pragma unroll
  for (int i = 0; i < NH; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int d = d0 + 16 * i + 4 * gg + e;
      st[i][e] = (!fresh && live && d < D) ? S[(long)d * Dv] : 0.f;
    }
  for (int i = tid; i < KP; i += 512) sf[C * KP + i] = 1.f;
  if (tid < HC * HC) sp[(tid / HC) * PP + HC + tid % HC] = 0.f;      // (above the diagonal blocks, never written again)
  if (DP < 128 * NU) {      // columns that no role stages
    constexpr int R = 128 * NU - DP > 0 ? 128 * NU - DP : 1;
    for (int i = tid; i < C * R; i += 512) {
      const int at = (i / R) * KP + DP + i % R;
      sq[at] = sk[at] = 0.f;
      sf[at] = 1.f;
    }
  }
  // this thread's roles: channel, rows ra .. ra + 7, bias and lower bound
  const int role = 32 * wave + (lane & 31), hf = lane >> 5, ra = HC * hf;
  float rb[NI], rl[NI];
#pragma unroll
  for (int u = 0; u < NI; ++u) {
    const int idx = role + 256 * u, d = min(idx < DP ? idx : idx - DP, D - 1);
    rb[u] = GLA ? 0.f : f_bias[(long)h * D + d];
    rl[u] = GLA ? 0.f : lower[(long)h * D + d];
  }
  // the next chunk's inputs as they are stored (rows past the sequence: its last row again)
  typedef T t4 __attribute__((ext_vector_type(4)));
  T rq[NI][HC], rz[NI][HC];
  t4 rv;
  auto fetch = [&](int t0) {
    const __amdgpu_buffer_rsrc_t qb = rows_rsrc(q + (long)t0 * q_ld + (long)h * D);
    const __amdgpu_buffer_rsrc_t zb = rows_rsrc(z + (long)t0 * z_ld + (long)h * D);
    const __amdgpu_buffer_rsrc_t kb = rows_rsrc(GLA ? key + (long)t0 * k_ld + (long)h * D : q);
    const int qs = (int)q_ld * (int)sizeof(T), zs = (int)z_ld * (int)sizeof(T), ks = (int)k_ld * (int)sizeof(T);
    const int last = r1 - 1 - t0;
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      const int idx = role + 256 * u;
      const int d = min(idx < DP ? idx : idx - DP, D - 1) * (int)sizeof(T);
      if (idx < DP) {
#pragma unroll
        for (int i = 0; i < HC; ++i) rq[u][i] = row_load<T>(qb, __umul24(min(ra + i, last), qs) + d);
      } else if (GLA && (WHOLE || idx < 2 * DP)) {
#pragma unroll
        for (int i = 0; i < HC; ++i) rq[u][i] = row_load<T>(kb, __umul24(min(ra + i, last), ks) + d);
      }
      if (WHOLE || idx < 2 * DP) {
#pragma unroll
        for (int i = 0; i < HC; ++i) rz[u][i] = row_load<T>(zb, __umul24(min(ra + i, last), zs) + d);
      }
    }
    if (tid >= 256) return;
    const T* vr = v + (long)min(t0 + (tid >> 4), r1 - 1) * v_ld + (long)h * Dv;
    const int c = c0 + 4 * (tid & 15);
    if (vec & 2) {
      rv = *reinterpret_cast<const t4*>(vr + min(c, Dv - 4));
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) rv[e] = vr[min(c + e, Dv - 1)];
    }
  };
  // Gates of this thread's channels into LDS. No branch on rows or channels: a row past the sequence is set to f = 1, k =
  // q = 0 by factors (`tail`: the last chunk has such rows), a channel past D has q = 0 (its state row is never read or
  // stored). The running products cross from one half of the rows to the other between lanes l and l + 32.
  auto stage = [&](int n, auto tail) {
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      const int idx = role + 256 * u;
      const float one = 1.f - rl[u];
      if (idx < DP) {
        const float qm = idx < D ? 1.f : 0.f;
        float F = 1.f, w[HC];
#pragma unroll
        for (int i = 0; i < HC; ++i) {
          float f, qv;
          if constexpr (GLA) {
            f = gla_decay<FAST>((float)rz[u][i], inv_tau);
            qv = (float)rq[u][i] * q_scale * qm;
          } else {
            float sg, cg;
            sigmoid2<FAST>((float)rz[u][i] + rb[u], sg, cg);
            f = fmaf(one, sg, rl[u]);
            qv = act_in<FAST>((float)rq[u][i], act) * qm;
          }
          if (decltype(tail)::value) {
            const float in = ra + i < n ? 1.f : 0.f;
            f = fmaf(in, f, 1.f - in);
            qv *= in;
          }
          F *= f;
          sq[(ra + i) * KP + idx] = qv;
          sf[(ra + i) * KP + idx] = f;
          w[i] = qv * F;
        }
        const float Fo = __shfl_xor(F, 32, 64), by = hf ? Fo : 1.f;
#pragma unroll
        for (int i = 0; i < HC; ++i) {
          sqf[(ra + i) * KP + idx] = w[i] * by;
          if (hf) sqh[i * KP + idx] = w[i];
        }
        if (hf == 0) sl[idx] = F * Fo;
      } else if (WHOLE || idx < 2 * DP) {
        const int d = idx - DP;
        float B = 1.f, w[HC];
#pragma unroll
        for (int i = HC - 1; i >= 0; --i) {
          float f, k;
          if constexpr (GLA) {
            f = gla_decay<FAST>((float)rz[u][i], inv_tau);
            k = (float)rq[u][i];
          } else {
            float sg, cg;
            sigmoid2<FAST>((float)rz[u][i] + rb[u], sg, cg);
            f = fmaf(one, sg, rl[u]);
            k = one * cg;
          }
          if (decltype(tail)::value) {
            const float in = ra + i < n ? 1.f : 0.f;
            f = fmaf(in, f, 1.f - in);
            k *= in;
          }
          sk[(ra + i) * KP + d] = k;
          w[i] = k * B;
          B *= f;
        }
        const float Bo = __shfl_xor(B, 32, 64), by = hf ? 1.f : Bo;
#pragma unroll
        for (int i = 0; i < HC; ++i) {
          skb[(ra + i) * KP + d] = w[i] * by;
          if (!hf) skh[i * KP + d] = w[i];
        }
      }
    }
    if (tid < 256) {
      const int t = tid >> 4, c = 4 * (tid & 15);
      f32x4 a;
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = (t < n && c0 + c + e < Dv) ? (float)rv[e] : 0.f;
      *reinterpret_cast<f32x4*>(sv + t * VP + c) = a;
    }
  };
  fetch(r0);
  for (int t0 = r0; t0 < r1; t0 += C) {
    const int n = min(C, r1 - t0);
    if (n == C) stage(n, std::false_type{});
    else stage(n, std::true_type{});
    if (t0 + C < r1) fetch(t0 + C);      // in flight during the products below
    __syncthreads();
    // (q F) S, then the new state
    f32x4 oc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NH; ++i) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(sqf + m * KP + d0 + 16 * i + 4 * gg);
#pragma unroll
      for (int e = 0; e < 4; ++e) oc = mfma_f32(a[e], st[i][e], oc);
    }
    float bv[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) bv[e] = sv[(4 * gg + e) * VP + cl];
#pragma unroll
    for (int i = 0; i < NH; ++i) {
      st[i] *= *reinterpret_cast<const f32x4*>(sl + d0 + 16 * i + 4 * gg);
#pragma unroll
      for (int e = 0; e < 4; ++e) st[i] = mfma_f32(skb[(4 * gg + e) * KP + d0 + 16 * i + m], bv[e], st[i]);
    }
    // weights of rows 8 .. 15 on columns 0 .. 7: this wave's channels
    if (wave < NP) {
      f32x4 w = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < (NT + 7) / 8; ++i) {
        const int at = (m & 7) * KP + 16 * (wave + 8 * i) + 4 * gg;
        if (NT % 8 && wave + 8 * i >= NT) break;
        const f32x4 a = *reinterpret_cast<const f32x4*>(sqh + at), b = *reinterpret_cast<const f32x4*>(skh + at);
#pragma unroll
        for (int e = 0; e < 4; ++e) w = mfma_f32(a[e], b[e], w);
      }
      if (m < HC && gg < 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) sph[(wave * HC + 4 * gg + e) * HC + m] = w[e];
      }
    }
    // the diagonal blocks: rows tb and 8 + tb, 32 lanes each share the row's channels, lane 16 + j keeps column j
    {
      const int tb = wave < 4 ? wave : 11 - wave, l4 = 4 * (lane & 31);      // (SIMDs get rows of equal work)
      f32x4 qd[NU];
#pragma unroll
      for (int u = 0; u < NU; ++u) qd[u] = *reinterpret_cast<const f32x4*>(sq + (ra + tb) * KP + 128 * u + l4);
      float keep = 0.f;
#pragma unroll
      for (int j = HC - 1; j >= 0; --j) {
        if (j > tb) continue;
        const float* fr = sf + (j < tb ? ra + j + 1 : C) * KP + l4;      // (its own column: not decayed yet)
        const float* kr = sk + (ra + j) * KP + l4;
        float w = 0.f;
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          qd[u] *= *reinterpret_cast<const f32x4*>(fr + 128 * u);
          const f32x4 kk = *reinterpret_cast<const f32x4*>(kr + 128 * u);
#pragma unroll
          for (int e = 0; e < 4; ++e) w = fmaf(qd[u][e], kk[e], w);
        }
        w = half_sum(w);
        keep = m == j ? w : keep;
      }
      if ((lane & 16) && m < HC) sp[(ra + tb) * PP + ra + m] = keep;
    }
    if (wave >= 4) {
#pragma unroll
      for (int e = 0; e < 4; ++e) so[(4 * gg + e) * VP + cl] = oc[e];
    }
    __syncthreads();
    if (wave < 4) {
      f32x4 a = *reinterpret_cast<const f32x4*>(sp + m * PP + 4 * gg);
      if (m >= HC && gg < 2) {
        a = *reinterpret_cast<const f32x4*>(sph + (m - HC) * HC + 4 * gg);
#pragma unroll
        for (int i = 1; i < NP; ++i) a += *reinterpret_cast<const f32x4*>(sph + (i * HC + m - HC) * HC + 4 * gg);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) oc[e] += so[(4 * gg + e) * VP + cl];
      float zero = 0.f;      // (x * 0 of an infinity or NaN is NaN)
#pragma unroll
      for (int e = 0; e < 4; ++e) zero = fmaf(bv[e], 0.f, zero);
      int odd = C;           // first row of this column that is no number
      if (__any(zero != 0.f)) {
#pragma unroll
        for (int e = 3; e >= 0; --e) {
          const bool bad = bv[e] * 0.f != 0.f;
          odd = bad ? 4 * gg + e : odd;
          bv[e] = bad ? 0.f : bv[e];
        }
        odd = min(odd, __shfl_xor(odd, 16, 64));
        odd = min(odd, __shfl_xor(odd, 32, 64));
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) oc = mfma_f32(a[e], bv[e], oc);
      if (__any(odd < C)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) oc[e] = 4 * gg + e >= odd ? NAN : oc[e];
      }
      if (live) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int t = 4 * gg + e;
          if (t < n) o[((long)(t0 + t) * H + h) * Dv + col] = oc[e];
        }
      }
    }
    // (the next chunk's staging writes nothing that is read after the barrier above; sp, sph and so are rewritten only
    // after its own first barrier)
  }
  int De = D;
  asm volatile("" : "+s"(De));      // (the bounds are compared anew: kept masks would fill the scalar registers)
  if (live) {
#pragma unroll
    for (int i = 0; i < NH; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int d = d0 + 16 * i + 4 * gg + e;
        if (d < De) S[(long)d * Dv] = st[i][e];
      }
  }
}

// The same recurrence row by row, for steps of one row per sequence (decoding) and for any D. Workgroup =
// (sequence, head, 64 value columns): 16 lanes of four columns by 16 groups of state rows; the state is read and
// written in place, the row groups' partial read-outs are summed in LDS.
template <typename T>
__global__ __launch_bounds__(256) void forget_step_kernel(const T* __restrict__ q, long q_ld, const T* __restrict__ z,
                                                          long z_ld, const T* __restrict__ v, long v_ld,
                                                          const float* __restrict__ f_bias,
                                                          const float* __restrict__ lower, float* __restrict__ state,
                                                          const int* __restrict__ state_slots,
                                                          const int* __restrict__ row_cu,
                                                          const int* __restrict__ positions, int act, int vec,
                                                          float* __restrict__ o, int H, int D, int Dv) {
  constexpr bool FAST = sizeof(T) == 2;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float* sq = smem;            // [D]
  float* sk = smem + D;        // [D]
  float* sf = smem + 2 * D;    // [D]
  __shared__ f32x4 red[16][16];
  const int s = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * 64;
  const int r0 = row_cu ? row_cu[s] : s, r1 = row_cu ? row_cu[s + 1] : s + 1;
  const int tid = threadIdx.x, cg = tid & 15, dg = tid >> 4;
  const int slot = state_slots[s], c = c0 + 4 * cg;
  if (slot < 0) {
    for (int i = tid; i < (r1 - r0) * 64; i += 256)
      if (c0 + (i & 63) < Dv) o[((long)(r0 + (i >> 6)) * H + h) * Dv + c0 + (i & 63)] = 0.f;
    return;
  }
  float* S = state + ((long)slot * H + h) * D * Dv;
  const bool sv4 = (vec & 4) && c + 3 < Dv;      // 16-byte state rows
  for (int t = r0; t < r1; ++t) {
    for (int d = tid; d < D; d += 256) {
      const float lo = lower[(long)h * D + d];
      float sg, cg2;
      sigmoid2<FAST>((float)z[(long)t * z_ld + (long)h * D + d] + f_bias[(long)h * D + d], sg, cg2);
      sq[d] = act_in<FAST>((float)q[(long)t * q_ld + (long)h * D + d], act);
      sk[d] = (1.f - lo) * cg2;
      sf[d] = lo + (1.f - lo) * sg;
    }
    const f32x4 vv = load4(v + (long)t * v_ld + (long)h * Dv, c, Dv, vec & 2);
    __syncthreads();
    const bool fresh = positions[t] == 0;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (c < Dv)
#pragma unroll 8
      for (int d = dg; d < D; d += 16) {
        float* Sr = S + (long)d * Dv + c;
        f32x4 x = {0.f, 0.f, 0.f, 0.f};
        if (!fresh) {
          if (sv4) x = *reinterpret_cast<const f32x4*>(Sr);
          else
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = c + e < Dv ? Sr[e] : 0.f;
        }
        const float kd = sk[d], qd = sq[d], fd = sf[d];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[e] = fmaf(fd, x[e], kd * vv[e]);
          acc[e] = fmaf(qd, x[e], acc[e]);
        }
        if (sv4) *reinterpret_cast<f32x4*>(Sr) = x;
        else
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (c + e < Dv) Sr[e] = x[e];
      }
    red[dg][cg] = acc;
    __syncthreads();
    if (tid < 64 && c0 + tid < Dv) {
      float a = 0.f;
#pragma unroll
      for (int g = 0; g < 16; ++g) a += red[g][tid >> 2][tid & 3];
      o[((long)t * H + h) * Dv + c0 + tid] = a;
    }
    __syncthreads();
  }
}

// L lanes per (row, head), V values per access
template <typename T, int V, int L>
__global__ __launch_bounds__(256) void head_norm_gate_kernel(const float* __restrict__ o, const float* __restrict__ w,
                                                             float eps, const T* __restrict__ gate, long g_ld, int act,
                                                             float mul, T* __restrict__ out, long out_ld, long n, int H,
                                                             int Dv) {
  typedef float fv __attribute__((ext_vector_type(V)));
  typedef T tv __attribute__((ext_vector_type(V)));
  const long item = blockIdx.x * (long)(256 / L) + threadIdx.x / L;      // t * H + h
  const int l = threadIdx.x % L;
  if (item >= n) return;      // (whole groups of L lanes leave; a group never spans waves)
  const long t = item / H;
  const int h = (int)(item - t * H);
  const float* row = o + item * Dv;
  fv x0 = fv(0.f);
  float ss = 0.f;
  for (int c = V * l; c < Dv; c += V * L) {
    const fv x = *reinterpret_cast<const fv*>(row + c);
    if (c < V * L) x0 = x;
#pragma unroll
    for (int e = 0; e < V; ++e) ss = fmaf(x[e], x[e], ss);
  }
#pragma unroll
  for (int d = L / 2; d > 0; d >>= 1) ss += __shfl_xor(ss, d, 64);
  const float r = mul / sqrtf(ss / (float)Dv + eps);
  for (int c = V * l; c < Dv; c += V * L) {
    const fv x = c < V * L ? x0 : *reinterpret_cast<const fv*>(row + c);
    fv f;
#pragma unroll
    for (int e = 0; e < V; ++e) f[e] = x[e] * r;
    if (w) f *= *reinterpret_cast<const fv*>(w + c);
    if (gate) {
      const tv gv = *reinterpret_cast<const tv*>(gate + t * g_ld + (long)h * Dv + c);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float g = (float)gv[e], sg = 1.f / (1.f + expf(-g));
        f[e] *= act == 1 ? g * sg : sg;
      }
    }
    tv y;
#pragma unroll
    for (int e = 0; e < V; ++e) y[e] = (T)f[e];
    *reinterpret_cast<tv*>(out + t * out_ld + (long)h * Dv + c) = y;
  }
}

// (D <= 256) 16-channel tiles of a record, and the records of a launch: those of the step, at most 256 MB of them
int record_tiles(int D) { return D <= 32 ? 2 : D <= 64 ? 4 : D <= 96 ? 6 : D <= 128 ? 8 : D <= 192 ? 12 : 16; }
long records_at_once(long T, long nseq, int H, int D) {
  const long cap = (256L << 20) / ((long)H * chunk_record(record_tiles(D)) * (long)sizeof(float));
  return std::min((T >> 4) + nseq, std::max(1L, cap));
}

template <typename T, int NT, bool GLA>
void one_launch(const T* q, long q_ld, const T* key, long k_ld, float inv_tau, float q_scale, const T* z, long z_ld, const T* v,
                long v_ld, const float* f_bias, const float* lower, float* state, const int* state_slots, const int* row_cu,
                int nseq, const int* positions, int act, float* o, int H, int D, int Dv, hipStream_t s, int cost) {
  constexpr int DP = 16 * NT, KP = (DP + 127) / 128 * 128 + 4;
  constexpr size_t lds = (size_t)(97 * KP + 2 * 16 * 68 + 16 * 20 + 64 * (NT < 8 ? NT : 8) + DP) * sizeof(float);
  static bool once = false;
  if (!once) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gate_scan_kernel<T, NT, GLA>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    once = true;
  }
  const int vec = (Dv % 4 == 0 && rows_aligned(v, v_ld, sizeof(T))) ? 2 : 0;
  gate_scan_kernel<T, NT, GLA><<<dim3(nseq, H, (Dv + 63) / 64), 512, lds, s>>>(
      q, q_ld, key, k_ld, inv_tau, q_scale, z, z_ld, v, v_ld, f_bias, lower, state, state_slots, row_cu, positions, act, vec, o, H,
      D, Dv, cost);
}

// (rec null: in one launch)
template <typename T, int NT, bool GLA>
void chunk_launch(const T* q, long q_ld, const T* key, long k_ld, float inv_tau, float q_scale, const T* z, long z_ld, const T* v,
                  long v_ld, const float* f_bias, const float* lower, float* state, const int* state_slots, const int* row_cu,
                  int nseq, const int* positions, int act, float* o, float* rec, int T_, int H, int D, int Dv, hipStream_t s,
                  int cost) {
  if (!rec)
    return one_launch<T, NT, GLA>(q, q_ld, key, k_ld, inv_tau, q_scale, z, z_ld, v, v_ld, f_bias, lower, state, state_slots,
                                  row_cu, nseq, positions, act, o, H, D, Dv, s, cost);
  constexpr int KP = 16 * NT + 4;
  constexpr size_t lds = (size_t)(81 * KP + 16 * 20 + 32 * NT) * sizeof(float);
  constexpr size_t chain_lds = (size_t)kChainSlots * (chunk_record(NT) + 1024) * sizeof(float);
  static bool once = false;
  if (!once) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gate_chunk_kernel<T, NT, GLA>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gate_chain_kernel<T, NT>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)chain_lds);
    once = true;
  }
  const long all = (T_ >> 4) + nseq, most = records_at_once(T_, nseq, H, D);
  for (long first = 0; first < all; first += most) {
    const int count = (int)std::min(most, all - first);
    gate_chunk_kernel<T, NT, GLA><<<dim3(H, count), 32 * NT, lds, s>>>(q, q_ld, key, k_ld, inv_tau, q_scale, z, z_ld, f_bias, lower,
                                                                      state_slots, row_cu, nseq, act, rec, H, D, cost,
                                                                      (int)first);
    gate_chain_kernel<T, NT><<<(nseq * H + 7) / 8 * 8 * ((Dv + 63) / 64), 256, chain_lds, s>>>(
        rec, v, v_ld, state, state_slots, row_cu, positions, o, nseq, H, D, Dv, cost, (int)first, count);
  }
}

template <typename T>
void forget_scan_t(const T* q, long q_ld, const T* z, long z_ld, const T* v, long v_ld, const float* f_bias,
                   const float* lower, float* state, const int* state_slots, const int* row_cu, int nseq,
                   const int* positions, int act, float* o, float* rec, int T_, int H, int D, int Dv, bool one_row,
                   hipStream_t s) {
  int vec = 0;      // 2: v rows, 4: state rows in four-element accesses
  if (Dv % 4 == 0 && rows_aligned(v, v_ld, sizeof(T))) vec |= 2;
  if (Dv % 4 == 0) vec |= 4;
  if (one_row || D > 256) {
    dim3 grid(nseq, H, (Dv + 63) / 64);
    forget_step_kernel<T><<<grid, 256, 3 * (size_t)D * sizeof(float), s>>>(
        q, q_ld, z, z_ld, v, v_ld, f_bias, lower, state, state_slots, one_row ? nullptr : row_cu, positions, act, vec, o, H, D,
        Dv);
    return;
  }
#define BFLY_FCH(NT)                                                                                                     \
  chunk_launch<T, NT, false>(q, q_ld, nullptr, 0, 1.f, 1.f, z, z_ld, v, v_ld, f_bias, lower, state, state_slots, row_cu, \
                             nseq, positions, act, o, rec, T_, H, D, Dv, s, 0)
  if (D <= 32) BFLY_FCH(2);
  else if (D <= 64) BFLY_FCH(4);
  else if (D <= 96) BFLY_FCH(6);
  else if (D <= 128) BFLY_FCH(8);
  else if (D <= 192) BFLY_FCH(12);
  else BFLY_FCH(16);
#undef BFLY_FCH
}

template <typename T>
void gla_chunks_t(const T* q, long q_ld, const T* k, long k_ld, const T* v, long v_ld, const T* z, long z_ld, float* state,
                  const int* state_slots, const int* row_cu, int nseq, const int* positions, float tau, float q_scale, float* o,
                  float* rec, int T_, int H, int D, int Dv, hipStream_t s, int cost) {
#define BFLY_GCH(NT)                                                                                                      \
  chunk_launch<T, NT, true>(q, q_ld, k, k_ld, 1.f / tau, q_scale, z, z_ld, v, v_ld, nullptr, nullptr, state, state_slots, \
                            row_cu, nseq, positions, 0, o, rec, T_, H, D, Dv, s, cost)
  if (D <= 32) BFLY_GCH(2);
  else if (D <= 64) BFLY_GCH(4);
  else if (D <= 96) BFLY_GCH(6);
  else if (D <= 128) BFLY_GCH(8);
  else if (D <= 192) BFLY_GCH(12);
  else BFLY_GCH(16);
#undef BFLY_GCH
}

template <typename T, int V>
void head_norm_gate_t(const float* o, const float* w, float eps, const T* gate, long g_ld, int act, float mul, T* out,
                      long out_ld, int T_, int H, int Dv, hipStream_t s) {
  const long n = (long)T_ * H;
#define BFLY_HNG(L)                                                                                                  \
  head_norm_gate_kernel<T, V, L><<<(int)((n + 256 / L - 1) / (256 / L)), 256, 0, s>>>(o, w, eps, gate, g_ld, act, mul, out, \
                                                                                      out_ld, n, H, Dv)
  if (Dv <= 8 * V) BFLY_HNG(8);
  else if (Dv <= 16 * V) BFLY_HNG(16);
  else if (Dv <= 32 * V) BFLY_HNG(32);
  else BFLY_HNG(64);
#undef BFLY_HNG
}

}  // namespace

// Rows of a step's longest sequence up to which one launch takes its chunks: beyond, a chunk's 3 to 6 us there outweigh the second
// launch, the records that go through memory, and 1.1 to 3 us a chunk. `wgs` workgroups of one launch; where they queue, it is their
// work that counts. One launch and two, us, sequences of 16, 32, 64 rows (forget gates, bf16): one of 16 heads of 128 9.4 11.5, 13.0
// 12.8, 20.7 15.6, eight 11.3 13.7, 15.2 16.7, 22.5 22.7, 64 57 55, 79 67, 119 99; one of 8 heads of 64 6.6 10.2, 9.7 11.0, 15.8 12.7, 64
// 9.9 15.3, 14.5 20.4, 24 32, 200 28 39, 43 46, 72 68; 8 of 32 heads of 32 6.3 12.2, 9.2 13.4, 15 16.5, 64 24 25, 40 35, 72 53; one of 8
// heads of 256 11.8 16.8, 17.6 19.3, 29 25, 64 102 115, 150 148, 244 214; in f32 one of 16 heads of 128 10.0 12.2, 14.4 13.6, 23 16.
static int one_launch_rows(long wgs, int D, bool f32) {
  if (f32) return wgs < 256 ? 16 : wgs < 512 ? (D > 64 ? 32 : 16) : 0;
  if (D <= 32) return wgs < 64 ? 32 : wgs < 256 ? 48 : wgs < 512 ? 64 : wgs <= 768 ? 96 : wgs <= 1024 ? 48 : wgs <= 2048 ? 16 : 0;
  if (D <= 64) return wgs < 128 ? 32 : wgs < 256 ? 48 : wgs <= 512 ? 96 : 64;
  if (D <= 128) return wgs < 256 ? 16 : wgs <= (D <= 96 ? 512 : 256) ? 32 : wgs <= 1024 ? 16 : 0;
  if (D <= 192) return wgs <= 1024 ? 16 : 0;
  return wgs < 256 ? 32 : wgs < 512 ? 64 : wgs <= 1024 ? 32 : 16;
}

// The workgroups that count are those of sequences as long as the longest (max_rows 0: it may have every row but one of each other);
// in f32 all of them (16 single rows beside 4 times 8, 16 heads of 128: 26.5 and 23.8 us, in bf16 23.0 and 22.9).
// Its row strides of q, k, z are of 24 bits (max_ld), those of v of any size; two launches have it the other way round (gate_rows_near).
bool gate_rows_near(int H, int Dv, long v_ld) { return std::max(v_ld, (long)H * Dv) * 64 < (1L << 31); }
bool chunks_in_one_launch(long T, long nseq, int H, int D, int Dv, bool f32, long max_rows, long max_ld, long v_ld) {
  if (!gate_rows_near(H, Dv, v_ld)) return D <= 256 && max_ld < (1L << 21);
  const long longest = std::max(1L, max_rows > 0 ? max_rows : T - nseq + 1), like = f32 ? nseq : std::min(nseq, (T + longest - 1) / longest);
  return D <= 256 && max_ld < (1L << 21) && longest <= one_launch_rows(like * H * ((Dv + 63) / 64), D, f32);
}

long chunk_record_floats(long T, long nseq, int H, int D) {
  return D > 256 ? 0 : records_at_once(T, nseq, H, D) * H * chunk_record(record_tiles(D));
}

void launch_forget_scan(const void* q, long q_ld, const void* z, long z_ld, const void* v, long v_ld, const float* f_bias,
                        const float* lower, float* state, const int* state_slots, const int* row_cu, int nseq,
                        const int* positions, int act, float* o, float* rec, int T, int H, int D, int Dv, bool one_row,
                        bool f32, hipStream_t s) {
  if (T <= 0 || nseq <= 0) return;
  if (f32)
    forget_scan_t<float>((const float*)q, q_ld, (const float*)z, z_ld, (const float*)v, v_ld, f_bias, lower, state,
                         state_slots, row_cu, nseq, positions, act, o, rec, T, H, D, Dv, one_row, s);
  else
    forget_scan_t<bf16>((const bf16*)q, q_ld, (const bf16*)z, z_ld, (const bf16*)v, v_ld, f_bias, lower, state, state_slots,
                        row_cu, nseq, positions, act, o, rec, T, H, D, Dv, one_row, s);
}

void launch_gla_chunks(const void* q, long q_ld, const void* k, long k_ld, const void* v, long v_ld, const void* z, long z_ld,
                       float* state, const int* state_slots, const int* row_cu, int nseq, const int* positions, float tau,
                       float q_scale, float* o, float* rec, int T, int H, int D, int Dv, bool f32, hipStream_t s, int cost) {
  if (f32)
    gla_chunks_t<float>((const float*)q, q_ld, (const float*)k, k_ld, (const float*)v, v_ld, (const float*)z, z_ld, state,
                        state_slots, row_cu, nseq, positions, tau, q_scale, o, rec, T, H, D, Dv, s, cost);
  else
    gla_chunks_t<bf16>((const bf16*)q, q_ld, (const bf16*)k, k_ld, (const bf16*)v, v_ld, (const bf16*)z, z_ld, state,
                       state_slots, row_cu, nseq, positions, tau, q_scale, o, rec, T, H, D, Dv, s, cost);
}

void launch_head_norm_gate(const float* o, const float* w, float eps, const void* gate, long g_ld, int act, float mul,
                           void* out, long out_ld, int T, int H, int Dv, bool f32, hipStream_t s) {
  if (T <= 0 || H <= 0) return;
  const size_t esz = f32 ? 4 : 2;
  const bool vec = Dv % 4 == 0 && rows_aligned(out, out_ld, esz) && (!gate || rows_aligned(gate, g_ld, esz)) &&
                   (!w || rows_aligned(w, 0, 4));
#define BFLY_HN(TT, V) head_norm_gate_t<TT, V>(o, w, eps, (const TT*)gate, g_ld, act, mul, (TT*)out, out_ld, T, H, Dv, s)
  if (f32) { if (vec) BFLY_HN(float, 4); else BFLY_HN(float, 1); }
  else { if (vec) BFLY_HN(bf16, 4); else BFLY_HN(bf16, 1); }
#undef BFLY_HN
}

}  // namespace bfly
