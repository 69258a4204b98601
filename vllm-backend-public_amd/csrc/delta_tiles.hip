// The gated delta rule for chunks of many tokens, by tiles of 16 rows of one chunk.
//
// With G_t the log decay summed from the tile's first row to row t (per head, or per key channel), the
// recurrence S <- a S; u = b (v - S^T k); S <- S + k u^T; o = S^T q unrolls over a tile into
//     (I + A) U = b V - b (e^G k) S_0          A_tj = b_t sum_c k_t k_j e^(G_t - G_j)      (j < t)
//     O = (e^G q) S_0 + P U                    P_tj = sum_c q_t k_j e^(G_t - G_j)          (j <= t)
//     S_end = e^G_end S_0 + (e^(G_end - G) k)^T U
// so that only products with S_0 are left to the walk from tile to tile:
//   delta_tiles_prep   every tile and head by itself: unit keys and queries, decays, A and P, and the forward
//                      substitution of (I + A) on the columns of b e^G k (-> W) and b V (-> U0, kept in `o`)
//   delta_tiles_walk   per (chunk, head, 16 value channels): U = U0 - W S, O = (e^G q) S + P U, S update
// All of it is fp32 (the 16x16x4 matrix instruction); G is summed and subtracted in double and every exponent is
// <= 0, so a strong decay neither overflows nor costs a later weak one its digits.
//
// What bounds it: the walk, one tile after the other; 25 matrix instructions a wave and tile at 32 cycles
// each, one barrier, and the tile's 33 KB through the vector caches (80 of 125 us with neither loads nor stores; more sets of them in
// flight, or each set asked for right behind its last use: the same).  Measured, 4 x 2048 rows of 128 x 128 heads in bf16, 8 heads with a
// decay per channel: prep 93, walk 125 us; with the rows of all heads side by side in the workspace (every head's
// 4 KB apart) and 43 KB of LDS, three workgroups a CU, 128 and 144.  A state column's d rows are dealt to the 4 waves of a workgroup; the
// accumulator layout (row 4 (lane / 16) + r, column lane % 16) serves as the right operand as it stands if step r of a product takes
// rows {4 g + r}, so the state never leaves its registers.
#include "common.h"
#include "delta_tiles.h"

#include <type_traits>

namespace mi355 {

namespace {

constexpr int C = 16;                     // rows of a tile

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// padded key channels: a multiple of the 4 waves' 16-row blocks
__host__ __device__ __forceinline__ int padded(int d) { return (d + 63) & ~63; }

// workspace: W [H][rows][dp] | P [H][rows][16] | q | k | e, of `plane` floats each (W, P and a channel's q within a tile of n rows
// as the walk's lanes hold them: vectors of four channels or rows by (wave, vector, lane / 16, row), see `lane_order`):
//   a decay per channel   [H][rows + 16][dp] e^G q | e^(G_end - G) k | e^G_end (a tile's, at its first row)
//   a decay per head      [H][rows + 16] factors of the raw query and key, e^G / (|q| sqrt(d)) and e^(G_end - G) / |k|,
//                         and e^G_end (a tile's, at its first row)
struct Layout {
  float *w, *p, *q, *k, *e;
};
__host__ __device__ __forceinline__ int64_t plane(bool per_channel, int64_t rows, int H, int dp) {
  return (rows + C) * H * (per_channel ? dp : 1);
}
template <bool PC>
__device__ __forceinline__ Layout layout(float* ws, int64_t rows, int H, int dp) {
  const int64_t n = rows * H;
  Layout l;
  l.w = ws;
  l.p = l.w + n * dp;
  l.q = l.p + n * C;
  l.k = l.q + plane(PC, rows, H, dp);
  l.e = l.k + plane(PC, rows, H, dp);
  return l;
}

// log(1 + e^z) for z <= 20: max(z, 0) + log(1 + w), w = e^-|z| as two numbers (2^n and a series in the rest), log(1 + w) = 2 artanh(s) with
// s = w / (2 + w) <= 1/3, its rounding carried along.  Largest and mean square error against 64 bits over [-80, 20]: 9.4e-8 and
// 3.0e-8 of it, where log1pf(expf(z)) has 1.35e-7 and 3.6e-8; sixteen of them a thread, so that they were 27 of 102 us of the preparation
// (8 heads, 4 x 2048 rows) and are 18.
__device__ __forceinline__ float softplus(float z) {
  float m = -fabsf(z);                                    // (a NaN stays one)
  m = m < -120.f ? -120.f : m;
  const float n = rintf(m * 1.44269504088896340736f);
  const float h = fmaf(n, -0.693145751953125f, m), g = fmaf(n, -1.428606820309417e-6f, h), gl = fmaf(n, -1.428606820309417e-6f, h - g);
  float t = 1.0f / 5040.0f;
  t = fmaf(t, g, 1.0f / 720.0f), t = fmaf(t, g, 1.0f / 120.0f), t = fmaf(t, g, 1.0f / 24.0f), t = fmaf(t, g, 1.0f / 6.0f);
  t = fmaf(fmaf(t, g, 0.5f), g * g, gl);
  const int ni = static_cast<int>(n);
  const float a = 1.0f + g, al = (g - (a - 1.0f)) + t;
  float w = a + al, wl = al - (w - a);
  w = ldexpf(w, ni), wl = ldexpf(wl, ni);
  const float q = 2.0f + w, ql = (w - (q - 2.0f)) + wl, r = __builtin_amdgcn_rcpf(q), s = w * r;
  const float sl = (fmaf(-s, q, w) + fmaf(-s, ql, wl)) * r, x = s * s;
  float y = 1.0f / 15.0f;
  y = fmaf(y, x, 1.0f / 13.0f), y = fmaf(y, x, 1.0f / 11.0f), y = fmaf(y, x, 1.0f / 9.0f), y = fmaf(y, x, 1.0f / 7.0f);
  y = fmaf(y, x, 0.2f), y = fmaf(y, x, 1.0f / 3.0f);
  const float low = fmaf(s * x, y, sl);
  return z > 0.f ? z + fmaf(2.0f, low, 2.0f * s) : fmaf(2.0f, low, 2.0f * s);
}
// Where channels 4 c .. 4 c + 3 of a row lie within a tile of n rows, in float4: the walk's wave has 16 DT channels, its lane 4 DT of one
// row.  (By rows each of a wave's loads touches 16 lines, another with every lane: the walk of 4 x 2048 rows of 16 heads took 255 us where
// this takes 205; of 8 heads 125 either way.)
template <int DT>
__device__ __forceinline__ int lane_order(int c, int row, int n) {
  const int wave = c / (4 * DT), kg = c % (4 * DT) / DT, j = c % DT;
  return ((wave * DT + j) * 4 + kg) * n + row;
}
// lanes l, l + 16, l + 32, l + 48 hold four numbers each: lane l + 16 m gets the m-th of the four lanes'
__device__ __forceinline__ void transpose4(float (&y)[4]) {
  auto swap = [](float& a, float& b, auto f) {
    const auto r = f(__float_as_uint(a), __float_as_uint(b));
    a = __uint_as_float(r[0]), b = __uint_as_float(r[1]);
  };
  auto p32 = [](uint32_t a, uint32_t b) { return __builtin_amdgcn_permlane32_swap(a, b, false, false); };
  auto p16 = [](uint32_t a, uint32_t b) { return __builtin_amdgcn_permlane16_swap(a, b, false, false); };
  swap(y[0], y[2], p32), swap(y[1], y[3], p32);
  swap(y[0], y[1], p16), swap(y[2], y[3], p16);
}

template <typename T, bool PC, int DT>
__global__ __launch_bounds__(256, DT <= 2 ? 4 : 1) void delta_tiles_prep_kernel(DeltaTiles a, int vec, int dvec) {
  typedef typename Elem<T>::S E;
  constexpr int dp = 64 * DT, ld = dp + 4, lg = dp + 2, NV = (DT + 1) / 2;
  __shared__ __attribute__((aligned(16))) float Ks[C * ld], Qs[C * ld];        // unit keys, unit queries / sqrt(d)
  __shared__ __attribute__((aligned(16))) float As[C * C], part[4][2][3][64];
  __shared__ __attribute__((aligned(16))) double Gs[PC ? C * lg : C];          // log2 decays, then their sums
  __shared__ __attribute__((aligned(16))) float bs[C], rk[C], rq[C];           // beta, 1 / |key|, 1 / (|query| sqrt(d))
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = blockIdx.y, g = h / (a.H / a.G), d = a.d;
  // tile slots: chunk s owns cu[s] / 16 + s onwards, one for each of its tiles (the ranges never overlap)
  const int slot = static_cast<int>(blockIdx.x);
  int s = -1, cs = 0, ce = 0;
  for (int base = 0; base < a.S; base += 64) {
    const int i = base + lane, j = i < a.S ? i : a.S - 1;
    const int c0 = MI355_LD(int32_t, a.cu_seqlens, a.cu_seqlens + j), c1 = MI355_LD(int32_t, a.cu_seqlens, a.cu_seqlens + j + 1);
    const int n_le = __popcll(__ballot(i < a.S && (c0 >> 4) + i <= slot));
    if (n_le > 0) s = base + n_le - 1, cs = __builtin_amdgcn_readlane(c0, n_le - 1), ce = __builtin_amdgcn_readlane(c1, n_le - 1);
    if (n_le < 64) break;
  }
  if (s < 0) return;
  const int r0 = (slot - (cs >> 4) - s) * C;
  if (r0 >= ce - cs) return;
  const int64_t row0 = cs + r0;
  const int n = ce - cs - r0 < C ? ce - cs - r0 : C;
  const E* qkv = static_cast<const E*>(a.qkv);
  // ---- every load of the workgroup goes out before the first is used (one trip to memory instead of five); rows
  // past the end repeat the last one
  const int t = tid >> 4, x = tid & 15;                   // 16 threads a row, 8 channels each
  const int64_t row = row0 + (t < n ? t : n - 1);
  const E *kr = qkv + row * a.stride + a.k_off + g * d, *qr = qkv + row * a.stride + a.q_off + g * d;
  const E* dr = static_cast<const E*>(a.decay) + row * a.decay_stride + (PC ? h * d : h);
  const float* br = a.dt_bias + (PC ? h * d : h);
  float kv[NV][8], qv[NV][8], zv[PC ? NV : 1][8], bias[PC ? NV : 1][8];
  uint4 kraw[NV], qraw[NV], zraw[NV];
  const float beta = MI355_LDF(T, a.beta, static_cast<const E*>(a.beta) + row * a.beta_stride + h);
  const float alog = MI355_LD(float, a.a_log, a.a_log + h);
  const bool v16 = sizeof(E) == 2 && vec, z16 = sizeof(E) == 2 && dvec;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int c = x * 8 + 128 * j;
    if (v16) {
      kraw[j] = MI355_LD(uint4, a.qkv, kr + (c < d ? c : 0));
      qraw[j] = MI355_LD(uint4, a.qkv, qr + (c < d ? c : 0));
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int ci = c + i < d ? c + i : 0;
        kv[j][i] = MI355_LDF(T, a.qkv, kr + ci), qv[j][i] = MI355_LDF(T, a.qkv, qr + ci);
      }
    }
    if constexpr (PC) {
      if (z16) zraw[j] = MI355_LD(uint4, a.decay, dr + (c < d ? c : 0));
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int ci = c + i < d ? c + i : 0;
        bias[j][i] = MI355_LD(float, a.dt_bias, br + ci);
        if (!z16) zv[j][i] = MI355_LDF(T, a.decay, dr + ci);
      }
    } else if (j == 0) {
      zv[0][0] = MI355_LDF(T, a.decay, dr), bias[0][0] = MI355_LD(float, a.dt_bias, br);
    }
  }
  E vraw[C];                                              // this thread's next column of V, if it has one
  auto load_v = [&](int col) {
    if (col >= dp && col < dp + a.dv) {
      const E* v = qkv + row0 * a.stride + a.v_off + static_cast<int64_t>(h) * a.dv;
#pragma unroll
      for (int i = 0; i < C; ++i) vraw[i] = MI355_LD(E, a.qkv, v + (i < n ? i : n - 1) * a.stride + static_cast<uint32_t>(col - dp));
    }
  };
  load_v(tid);
  if constexpr (sizeof(E) == 2) {
    if (v16)
#pragma unroll
      for (int j = 0; j < NV; ++j) unpack8<T>(kraw[j], kv[j]), unpack8<T>(qraw[j], qv[j]);
    if constexpr (PC) {
      if (z16)
#pragma unroll
        for (int j = 0; j < NV; ++j) unpack8<T>(zraw[j], zv[j]);
    }
  }
  {
    float kk = 0.f, qq = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (x * 8 + 128 * j + i >= d) kv[j][i] = 0.f, qv[j][i] = 0.f;
        kk += kv[j][i] * kv[j][i], qq += qv[j][i] * qv[j][i];
      }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) kk += __shfl_xor(kk, o, 64), qq += __shfl_xor(qq, o, 64);
    kk = 1.0f / sqrtf(kk + 1e-6f);
    qq = (1.0f / sqrtf(static_cast<float>(d))) / sqrtf(qq + 1e-6f);
    if (x == 0) {
      rk[t] = kk, rq[t] = qq;
      bs[t] = t < n ? 1.0f / (1.0f + expf(-beta)) : 0.f;
    }
    // log2 of a decay; below 2^-200 a float is zero all the same
    const float na = -expf(alog) * 1.44269504088896340736f;
    auto log_decay = [&](float z) {
      const float l = na * (z > 20.0f ? z : softplus(z));
      return t < n ? static_cast<double>(l < -200.0f ? -200.0f : l) : 0.0;
    };
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int c = x * 8 + 128 * j;
      if (c >= dp) break;
      float4* ko = reinterpret_cast<float4*>(Ks + t * ld + c);
      float4* qo = reinterpret_cast<float4*>(Qs + t * ld + c);
      ko[0] = make_float4(kv[j][0] * kk, kv[j][1] * kk, kv[j][2] * kk, kv[j][3] * kk);
      ko[1] = make_float4(kv[j][4] * kk, kv[j][5] * kk, kv[j][6] * kk, kv[j][7] * kk);
      qo[0] = make_float4(qv[j][0] * qq, qv[j][1] * qq, qv[j][2] * qq, qv[j][3] * qq);
      qo[1] = make_float4(qv[j][4] * qq, qv[j][5] * qq, qv[j][6] * qq, qv[j][7] * qq);
      if constexpr (PC) {
#pragma unroll
        for (int i = 0; i < 8; ++i) Gs[t * lg + c + i] = c + i < d ? log_decay(zv[j][i] + bias[j][i]) : 0.0;
      }
    }
    if (!PC && x == 0) Gs[t] = log_decay(zv[0][0] + bias[0][0]);
  }
  __syncthreads();
  if (PC) {
    if (tid < dp) {
      double sum = 0.0;
#pragma unroll
      for (int i = 0; i < C; ++i) sum += Gs[i * lg + tid], Gs[i * lg + tid] = sum;
    }
    __syncthreads();
  } else if (tid < C) {
    double sum = 0.0;
    for (int i = 0; i <= tid; ++i) sum += Gs[i];
    __builtin_amdgcn_wave_barrier();                      // (the 16 lanes of one wave: all have read)
    Gs[tid] = sum;
  }
  // Per key channel the factor e^(G_t - G_j) is split at a row R between the two, e^(G_t - G_R) e^(G_R - G_j), so
  // that rows scale their own keys and both parts stay <= 1: blocks of b = 8, 4, 2, 1 rows, t in an odd block, j in
  // the even block ahead of it, R the latter's last row.  Every pair j < t belongs to one b, the highest bit in
  // which t and j differ.  (Direct differences, an exponential per pair and channel: 140 us a launch where this takes 124 to 130.)
  const int li = lane & 15, kg = lane >> 4;
  constexpr int LV = PC ? 4 : 1;
  f32x4 aa[LV], pp[LV], diag = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int v = 0; v < LV; ++v) aa[v] = pp[v] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int c0 = wave * 16; c0 < dp; c0 += 64) {
    const int c = c0 + 4 * kg;
    const float4 kf = *reinterpret_cast<const float4*>(Ks + li * ld + c), qf = *reinterpret_cast<const float4*>(Qs + li * ld + c);
    const float k4[4] = {kf.x, kf.y, kf.z, kf.w}, q4[4] = {qf.x, qf.y, qf.z, qf.w};
    if constexpr (PC) {
      double G[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) G[x] = Gs[li * lg + c + x];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const bool late = (li >> v) & 1;                  // in an odd block of 2^v rows
        const int R = late ? ((li >> v) << v) - 1 : li | ((1 << v) - 1);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const double diff = G[x] - Gs[R * lg + c + x];
          const float e = __builtin_amdgcn_exp2f(static_cast<float>(late ? diff : -diff));
          const float ke = k4[x] * e, kl = late ? ke : 0.f, kr = late ? 0.f : ke;
          aa[v] = mfma4(kl, kr, aa[v]);
          pp[v] = mfma4(late ? q4[x] * e : 0.f, kr, pp[v]);
        }
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) diag = mfma4(q4[x], k4[x], diag);
    } else {
#pragma unroll
      for (int x = 0; x < 4; ++x) aa[0] = mfma4(k4[x], k4[x], aa[0]), pp[0] = mfma4(q4[x], k4[x], pp[0]);
    }
  }
  // wave w sums rows 4 g + w of the waves' parts, its own from its registers (so that four workgroups of 128 channels fit a CU's LDS)
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  float u = 0.f, y = 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float ur = aa[0][r], yr = pp[0][r];
    if constexpr (PC) {
      const int diff = (4 * kg + r) ^ li;
      ur = diff & 8 ? aa[3][r] : diff & 4 ? aa[2][r] : diff & 2 ? aa[1][r] : aa[0][r];
      yr = diff & 8 ? pp[3][r] : diff & 4 ? pp[2][r] : diff & 2 ? pp[1][r] : diff ? pp[0][r] : diag[r];
    }
    if (r == wv) u = ur, y = yr;
    else part[wv][0][r < wv ? r : r - 1][lane] = ur, part[wv][1][r < wv ? r : r - 1][lane] = yr;
  }
  __syncthreads();
  const Layout l = layout<PC>(a.ws, a.rows, a.H, dp);
  const int64_t at0 = row0 * a.H + h;                     // (row, head) of the tile's first row; a row further: + H
  const int64_t hw = h * a.rows + row0, hq = h * (a.rows + C) + row0;
  {
    const int t = 4 * kg + wv, x = li;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w == wv) continue;
      u += part[w][0][wv < w ? wv : wv - 1][lane], y += part[w][1][wv < w ? wv : wv - 1][lane];
    }
    if (!PC) {
      const float e = __builtin_amdgcn_exp2f(fminf(static_cast<float>(Gs[t] - Gs[x]), 0.f));
      u *= e, y *= e;
    }
    As[t * C + x] = x < t ? bs[t] * u : 0.f;
    if (t < n) MI355_ST(float, a.ws, l.p + hw * C + ((x & 3) * 4 + (x >> 2)) * n + t, x <= t ? y : 0.f);
    if (!PC && x == 0 && t < n) {
      const double end = Gs[C - 1];                       // (rows past the last add 0)
      const int64_t at = static_cast<int64_t>(h) * (a.rows + C) + row0 + t;
      MI355_ST(float, a.ws, l.q + at, rq[t] * __builtin_amdgcn_exp2f(static_cast<float>(Gs[t])));
      MI355_ST(float, a.ws, l.k + at, rk[t] * __builtin_amdgcn_exp2f(static_cast<float>(end - Gs[t])));
      if (t == 0) MI355_ST(float, a.ws, l.e + at, __builtin_amdgcn_exp2f(static_cast<float>(end)));
    }
  }
  __syncthreads();
  // ---- forward substitution, a column a thread: first the dp columns of b e^G k, then the dv of b V
  for (int at = tid; at < dp + a.dv; at += 256) {
    float y[C];
    const bool value = at >= dp;
    // (keys: four adjacent columns in lanes 16 apart, to be transposed below)
    const int col = value ? at : (at & ~63) + 4 * (lane & 15) + (lane >> 4);
    auto put = [&](float* to, float (&v)[4], int i) {    // rows i .. i + 3 of the keys' columns
      transpose4(v);
      const int r = i + (lane >> 4);
      if (r < n)
        MI355_ST(float4, a.ws, reinterpret_cast<float4*>(to) + lane_order<DT>((at & ~63) / 4 + (lane & 15), r, n),
                 make_float4(v[0], v[1], v[2], v[3]));
    };
    if (!value) {
      const double end = PC ? Gs[(C - 1) * lg + col] : 0.0;
#pragma unroll
      for (int i0 = 0; i0 < C; i0 += 4) {
        float q[4];
#pragma unroll
        for (int i = i0; i < i0 + 4; ++i) {
          const double G = PC ? Gs[i * lg + col] : Gs[i];
          const float e = __builtin_amdgcn_exp2f(static_cast<float>(G)), k = Ks[i * ld + col];
          y[i] = bs[i] * (k * e);
          if constexpr (PC) {
            q[i - i0] = Qs[i * ld + col] * e;
            if (i < n) MI355_ST(float, a.ws, l.k + (hq + i) * dp + col, k * __builtin_amdgcn_exp2f(static_cast<float>(end - G)));
          }
          if (i & 1) asm volatile("" ::: "memory");
        }
        if constexpr (PC) put(l.q + hq * dp, q, i0);
      }
      if (PC) MI355_ST(float, a.ws, l.e + hq * dp + col, __builtin_amdgcn_exp2f(static_cast<float>(end)));
    } else {
#pragma unroll
      for (int i = 0; i < C; ++i) y[i] = bs[i] * elem_to_f<T>(vraw[i]);
    }
#pragma unroll
    for (int i = 1; i < C; ++i) {
      asm volatile("" ::: "memory");                      // (row by row: A's 120 numbers at once would take as many registers)
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) sum += As[i * C + j] * y[j];
      y[i] -= sum;
    }
    if (value) {
      float* to = a.o + at0 * a.dv + (col - dp);
      const int64_t step = static_cast<int64_t>(a.H) * a.dv;
#pragma unroll
      for (int i = 0; i < C; ++i) {
        if (i < n) MI355_ST(float, a.o, to, y[i]);
        to += step;
      }
    } else {
#pragma unroll
      for (int i = 0; i < C; i += 4) {
        float v[4] = {y[i], y[i + 1], y[i + 2], y[i + 3]};
        put(l.w + hw * dp, v, i);
      }
    }
    load_v(at + 256);
  }
}

// N adjacent elements, read by as few loads as their alignment A allows
template <typename V, int N, int A>
struct alignas(A) Run {
  V v[N];
};
__host__ __device__ constexpr int run_align(int bytes) { return bytes % 16 == 0 ? 16 : bytes % 8 == 0 ? 8 : bytes % 4 == 0 ? 4 : 2; }

// Workgroup (chunk, head, 16 value channels).  The workgroups of one (chunk, head) read the same rows: they
// are dealt so that they fall on one XCD (every eighth block), whose L2 then serves all but the first.
// Wave w keeps key channels [w 16 DT, (w + 1) 16 DT) of the state; position p of its accumulator x is channel DT p + x,
// so that a lane's operands are runs of 4 DT (W, q) and DT (k) channels.
template <typename T, bool PC, bool VEC, int DT>
__global__ __launch_bounds__(256, 2) void delta_tiles_walk_kernel(DeltaTiles a, int groups) {
  typedef typename Elem<T>::S E;
  typedef typename std::conditional<PC, float, E>::type K;          // queries and keys: scaled fp32, or as projected
  constexpr int dp = 64 * DT, NS = 2, ES = static_cast<int>(sizeof(K));
  typedef Run<float, 4 * DT, 16> RunW;
  typedef Run<K, 4 * DT, VEC ? run_align(4 * DT * ES) : ES> RunQ;
  typedef Run<K, DT, VEC ? run_align(DT * ES) : ES> RunK;
  __shared__ float4 xp[2][4][64], yp[2][4][64];           // partial W S - U0 and O of the 4 waves, by turns
  const int unit = (blockIdx.x & 7) + 8 * (blockIdx.x / (8 * groups)), cg = (blockIdx.x >> 3) % groups;
  if (unit >= a.S * a.H) return;
  const int s = unit / a.H, h = unit % a.H, g = h / (a.H / a.G), d = a.d, dv = a.dv;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, kg = lane >> 4;
  const int64_t cs = MI355_LD(int32_t, a.cu_seqlens, a.cu_seqlens + s);
  const int len = static_cast<int>(MI355_LD(int32_t, a.cu_seqlens, a.cu_seqlens + s + 1) - cs);
  if (len <= 0) return;
  const int col = cg * 16 + li, c0 = wave * 16 * DT, cw = c0 + 4 * DT * kg, ck = c0 + DT * li;
  const bool live = col < dv;
  const Layout l = layout<PC>(a.ws, a.rows, a.H, dp);
  [[maybe_unused]] const void* kv_base = PC ? static_cast<const void*>(a.ws) : a.qkv;
  float* sp = a.state + ((static_cast<int64_t>(MI355_LD(int32_t, a.state_slots, a.state_slots + s)) * a.H + h) * d) * dv + col;
  const bool fresh = MI355_LD(int64_t, a.positions, a.positions + cs) == 0;
  f32x4 S[DT];
#pragma unroll
  for (int x = 0; x < DT; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int c = cw + DT * r + x;
      S[x][r] = live && !fresh && c < d ? MI355_LD(float, a.state, sp + static_cast<int64_t>(c) * dv) : 0.f;
    }
  // What a tile brings, as it lies in memory (converted where it is used: a conversion here would wait for the load).
  // No load is guarded: rows past the tile's end repeat its last row (their U is set to 0, their O not stored),
  // channels past d repeat channel 0 (their key is set to 0, so that the padded state stays 0), columns
  // past dv the last column.  Every load is a uniform base (the tile's) plus a 32-bit offset of the lane that stays
  // from tile to tile; only a last tile of fewer rows has its own.
  struct Rows {
    RunW w, e;
    RunQ q;
    RunK k[4];
    Run<float, 4, 4> qf, kf;
    float u, p, end;
  };
  Rows ring[NS];
  const int cl = live ? col : dv - 1;
  const uint32_t row_w = dp * 4u, row_k = PC ? row_w : static_cast<uint32_t>(a.stride * ES);
  uint32_t vp, vw[DT], vq, vu, vk[4];
  auto offsets = [&](int n) {
    const uint32_t rq = li < n ? li : n - 1, ru = 4 * kg + wave < n ? 4 * kg + wave : n - 1;
    vp = ((4 * wave + kg) * n + rq) * 4u;
#pragma unroll
    for (int j = 0; j < DT; ++j) vw[j] = ((4 * (DT * wave + j) + kg) * n + rq) * 16u;
    vq = rq * row_k + (PC || cw < d ? cw : 0) * static_cast<uint32_t>(ES);
    vu = (ru * a.H * dv + cl) * 4u;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t rk = 4 * kg + r < n ? 4 * kg + r : n - 1;
      vk[r] = rk * row_k + (PC || ck < d ? ck : 0) * static_cast<uint32_t>(ES);
    }
  };
#define AT(base, off) (reinterpret_cast<const char*>(base) + (off))
  // What a tile adds to the bases of its first (worked out anew from the rows, the addresses of a tile were some 130 scalar instructions
  // that the one wave of a SIMD has nothing to hide behind).
  const int64_t hr = cs * a.H + h, hw = h * a.rows + cs, hq = h * (a.rows + C) + cs;
  const float *w0 = l.w + hw * dp, *p0 = l.p + hw * C, *e0 = l.e + hq * (PC ? dp : 1), *u0 = a.o + hr * dv;
  const float *q0 = l.q + hq * (PC ? dp : 1), *k0 = l.k + hq * (PC ? dp : 1);
  const E* rows = static_cast<const E*>(a.qkv) + cs * a.stride + g * d;
  const int64_t rows_step = C * a.stride, u_step = static_cast<int64_t>(C) * a.H * dv;
  auto vectors = [&](float (&to)[4 * DT], const float* from) {
#pragma unroll
    for (int j = 0; j < DT; ++j) {
      const float4 u = MI355_LD(float4, a.ws, AT(from, vw[j]));
      to[4 * j] = u.x, to[4 * j + 1] = u.y, to[4 * j + 2] = u.z, to[4 * j + 3] = u.w;
    }
  };
  // NS register sets: a tile's loads travel while the tile ahead of it is worked on
  auto fetch = [&](Rows& f, int64_t i) {
    if (len - i * C < C) offsets(static_cast<int>(len - i * C));
    const int64_t at = i * (C * dp);
    const E* row = rows + i * rows_step;
    [[maybe_unused]] const K* kr;
    if constexpr (PC) kr = k0 + at;
    else kr = row + a.k_off;
    if constexpr (PC) f.e = MI355_LD(RunW, a.ws, AT(e0 + at, cw * 4u));
    vectors(f.w.v, w0 + at);
    if constexpr (PC) {
      vectors(f.q.v, q0 + at);
    } else if constexpr (VEC) {
      f.q = MI355_LD(RunQ, kv_base, AT(row + a.q_off, vq));
    } else {
#pragma unroll
      for (int x = 0; x < 4 * DT; ++x) f.q.v[x] = MI355_LD(K, kv_base, AT(row + a.q_off + (cw + x < d ? x : 0), vq));
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (VEC) {
        f.k[r] = MI355_LD(RunK, kv_base, AT(kr, vk[r]));
      } else {
#pragma unroll
        for (int x = 0; x < DT; ++x) f.k[r].v[x] = MI355_LD(K, kv_base, AT(kr + (ck + x < d ? x : 0), vk[r]));
      }
    }
    f.u = MI355_LD(float, a.o, AT(u0 + i * u_step, vu));
    f.p = MI355_LD(float, a.ws, AT(p0 + i * (C * C), vp));
    if constexpr (!PC) {                                  // (the rows of these are padded by a tile)
      f.qf = MI355_LD(decltype(f.qf), a.ws, AT(q0 + i * C, 16u * kg));
      f.kf = MI355_LD(decltype(f.kf), a.ws, AT(k0 + i * C, 16u * kg));
      f.end = MI355_LD(float, a.ws, AT(e0 + i * C, 0u * kg));
    }
  };
#undef AT
  auto number = [&](K v) -> float {
    if constexpr (PC) return v;
    else return elem_to_f<T>(v);
  };
  const uint32_t vs = (static_cast<uint32_t>(4 * kg + wave) * a.H * dv + col) * 4u;
  auto store = [&](int i) {                               // O of tile i: wave w adds up and stores rows 4 g + w
    float y = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) y += (&yp[i & 1][w][lane].x)[wave];
    if (i * C + 4 * kg + wave < len && live)
      MI355_ST(float, a.o, reinterpret_cast<char*>(a.o + hr * dv + i * u_step) + vs, y);
  };
  const int num = (len + C - 1) / C;
  auto work = [&](Rows& f, int i) {
    f32x4 X = f32x4{0.f, 0.f, 0.f, 0.f}, Y = X;
#pragma unroll
    for (int x = 0; x < DT; ++x)
#pragma unroll
      for (int r = 0; r < 4; ++r) X = mfma4(f.w.v[DT * r + x], S[x][r], X);
    const float u0 = f.u;
    xp[i & 1][wave][lane] = make_float4(X[0] - (wave == 0 ? u0 : 0.f), X[1] - (wave == 1 ? u0 : 0.f), X[2] - (wave == 2 ? u0 : 0.f),
                                        X[3] - (wave == 3 ? u0 : 0.f));
    __syncthreads();
    float4 xs[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) xs[w] = xp[i & 1][w][lane];
    __builtin_amdgcn_sched_barrier(0);                    // the products below run while these come
#pragma unroll
    for (int x = 0; x < DT; ++x)
#pragma unroll
      for (int r = 0; r < 4; ++r) Y = mfma4(number(f.q.v[DT * r + x]), S[x][r], Y);
    const int left = len - i * C - 4 * kg;            // rows of the tile from this lane's first on
    float u[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float x = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) x -= (&xs[w].x)[r];
      u[r] = r < left ? x : 0.f;
    }
    if constexpr (!PC) {
#pragma unroll
      for (int r = 0; r < 4; ++r) Y[r] *= f.qf.v[r];
    }
    const float uw = wave == 0 ? u[0] : wave == 1 ? u[1] : wave == 2 ? u[2] : u[3];
    Y = mfma4(f.p, uw, Y);                                // this wave's quarter of P U
    if constexpr (!PC) {                                  // (rows past the end: their factor may be anything)
#pragma unroll
      for (int r = 0; r < 4; ++r) u[r] = r < left ? u[r] * f.kf.v[r] : 0.f;
    }
#pragma unroll
    for (int x = 0; x < DT; ++x)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[x][r] *= PC ? f.e.v[DT * r + x] : f.end;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int x = 0; x < DT; ++x) {
        const float k = number(f.k[r].v[x]);
        S[x] = mfma4(PC || ck + x < d ? k : 0.f, u[r], S[x]);
      }
    if (i > 0) store(i - 1);                              // (written by all waves ahead of this tile's barrier)
    yp[i & 1][wave][lane] = make_float4(Y[0], Y[1], Y[2], Y[3]);
    fetch(f, i + NS < num ? i + NS : num - 1);            // (past the end: loaded and not used)
  };
  offsets(C);
#pragma unroll
  for (int j = 0; j < NS; ++j) fetch(ring[j], j < num ? j : num - 1);
  int i0 = 0;
  for (; i0 + NS <= num; i0 += NS)
#pragma unroll
    for (int j = 0; j < NS; ++j) work(ring[j], i0 + j);
#pragma unroll
  for (int j = 0; j < NS - 1; ++j)
    if (i0 + j < num) work(ring[j], i0 + j);
  __syncthreads();
  store(num - 1);
  if (live) {
#pragma unroll
    for (int x = 0; x < DT; ++x)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = cw + DT * r + x;
        if (c < d) MI355_ST(float, a.state, sp + static_cast<int64_t>(c) * dv, S[x][r]);
      }
  }
}

template <typename T, bool PC>
void launch(const DeltaTiles& a, hipStream_t stream) {
  const int dp = padded(a.d);
  const bool off8 = a.d % 8 == 0 && a.q_off % 8 == 0 && a.k_off % 8 == 0 && a.stride % 8 == 0;
  const int vec = off8 && aligned16(a.qkv) ? 1 : 0;
  const int dvec = PC && a.d % 8 == 0 && a.decay_stride % 8 == 0 && aligned16(a.decay) ? 1 : 0;
  const dim3 pgrid(static_cast<unsigned>(a.rows / C + a.S), static_cast<unsigned>(a.H));
  const int groups = (a.dv + 15) / 16;
  const unsigned units = static_cast<unsigned>(a.S) * static_cast<unsigned>(a.H);
  const dim3 wgrid((units + 7) / 8 * 8 * static_cast<unsigned>(groups));
#define MI355_WALK(DT)                                                                                                       \
  do {                                                                                                                      \
    hipLaunchKernelGGL((delta_tiles_prep_kernel<T, PC, DT>), pgrid, dim3(256), 0, stream, a, vec, dvec);                    \
    if (PC || (vec && a.d % (4 * DT) == 0))                                                                                 \
      hipLaunchKernelGGL((delta_tiles_walk_kernel<T, PC, true, DT>), wgrid, dim3(256), 0, stream, a, groups);               \
    else hipLaunchKernelGGL((delta_tiles_walk_kernel<T, PC, PC, DT>), wgrid, dim3(256), 0, stream, a, groups);               \
  } while (0)
  if (dp == 64) MI355_WALK(1);
  else if (dp == 128) MI355_WALK(2);
  else if (dp == 192) MI355_WALK(3);
  else MI355_WALK(4);
#undef MI355_WALK
}

}  // namespace

int64_t delta_tiles_workspace(int64_t rows, int H, int d, bool per_channel) {
  return rows * H * (padded(d) + C) + 3 * plane(per_channel, rows, H, padded(d));
}

void launch_delta_tiles(const DeltaTiles& a, int dtype, hipStream_t stream) {
  MI355_DISPATCH_DTYPE3(dtype, {
    if (a.per_channel) launch<TT, true>(a, stream);
    else launch<TT, false>(a, stream);
  });
}

}  // namespace mi355
