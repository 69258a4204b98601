// Rows of queries and keys rotated (and normed over the whole row) by vectors, for the entry points that write K / V pages.
#pragma once
#include "common.h"

namespace mi355 {

// V rows [tokens][kv_heads * v_dim] to V pages [blocks, kv_heads, v_dim, 16], a page's tile turned over in LDS
// (rope_kv_write.hip): v_dim a multiple of 8 up to 256, rows and pages 16-byte aligned.
void launch_v_pages(const uint16_t* v, int64_t v_stride, const int64_t* slot_mapping, uint16_t* v_cache, int num_blocks,
                    int64_t num_tokens, int num_kv_heads, int v_dim, hipStream_t s);

struct KvRows {
  uint16_t* q;
  const uint16_t *k, *v;         // k null: queries only
  int64_t q_stride, k_stride, v_stride;
  const float *wq, *wk;          // NORM: weights over the whole rows
  const float* cos_sin;          // [max_pos][rot]: cos | sin
  int64_t max_pos;
  const int64_t *positions, *slot_mapping;
  uint16_t *k_cache, *v_cache;
  int64_t num_tokens;
  int H, G, d, dv, rot;
  float eps, temp_coef;          // NORM; temp_every > 0: queries times 1 + temp_coef log(floor((p + 1) / temp_every) + 1)
  double temp_every;
};

// Whether the vector form covers these rows: 16-byte pieces throughout.
static inline bool kv_rows_ok(const KvRows& a) {
  return a.d % 8 == 0 && a.rot % 16 == 0 && a.q_stride % 8 == 0 && aligned16(a.q) && (a.rot == 0 || aligned16(a.cos_sin)) &&
         (a.wq == nullptr || (aligned16(a.wq) && aligned16(a.wk))) &&
         (a.k == nullptr || (a.dv % 8 == 0 && a.dv <= 256 && a.k_stride % 8 == 0 && a.v_stride % 8 == 0 && aligned16(a.k) &&
                             aligned16(a.v) && aligned16(a.k_cache) && aligned16(a.v_cache))) &&
         static_cast<int64_t>(a.H + (a.k ? a.G : 0)) * (a.d - a.rot / 2) <= 8 * 4 * 512;
}

// One workgroup per packed row; a thread has N units of 8 rotation pairs (two 16-byte pieces) or of 8 coordinates past
// them.  Bound by memory for prompts: rows through the cache once, in 16-byte pieces, where an element a thread made three
// passes (norm, rotation, V pages by 2 bytes).  8192 rows of 16 + 4 + 4 heads of 128: with the norm 80 us, here 23 to 31 and 6
// to 10 for V; the rotation alone 41, here 23 + 7; 32 decoded rows with the norm 12.0, here 5.7.
template <typename T, bool NORM, bool ROT, int N>
__global__ __launch_bounds__(512) void kv_rows_vec_kernel(KvRows a, int inline_v) {
  __shared__ float scratch[32];
  constexpr int BS = MI355_BLOCK_SIZE;
  const int64_t t = blockIdx.x;
  int64_t p = MI355_LD(int64_t, a.positions, a.positions + t);
  float temp = 1.0f;
  if (NORM && a.temp_every > 0.0) temp += a.temp_coef * logf(static_cast<float>(floor(static_cast<double>(p + 1) / a.temp_every)) + 1.0f);
  p = p < 0 ? 0 : (p >= a.max_pos ? a.max_pos - 1 : p);
  const int64_t slot = MI355_LD(int64_t, a.slot_mapping, a.slot_mapping + t);
  const int half = a.rot >> 1, pairs = half >> 3, units = (a.d - half) >> 3;
  const int heads = a.k != nullptr && slot >= 0 ? a.H + a.G : a.H, total = heads * units;
  const float* cs = a.cos_sin + p * a.rot;
  uint16_t* qr = a.q + t * a.q_stride;
  const uint16_t* kr = a.k + (a.k != nullptr ? t * a.k_stride : 0);
  uint4 x[N], y[N];
  int at[N];                                             // first coordinate of the unit's row piece
  bool is_q[N], pair[N];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const int i = min(static_cast<int>(threadIdx.x + n * blockDim.x), total - 1);
    const int hh = i / units, u = i - hh * units;
    is_q[n] = hh < a.H;
    pair[n] = ROT && u < pairs;
    at[n] = (is_q[n] ? hh : hh - a.H) * a.d + 8 * u + (u < pairs ? 0 : half);
    const uint16_t* src = (is_q[n] ? static_cast<const uint16_t*>(qr) : kr) + at[n];
    [[maybe_unused]] const void* base = is_q[n] ? static_cast<const void*>(a.q) : static_cast<const void*>(a.k);
    x[n] = MI355_LD(uint4, base, src);
    if (ROT) y[n] = MI355_LD(uint4, base, src + (pair[n] ? half : 0));
  }
  float rq = 1.0f, rk = 1.0f;
  if (NORM) {
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int n = 0; n < N; ++n) {
      if (static_cast<int>(threadIdx.x + n * blockDim.x) >= total) continue;
      float f[8], ss = 0.f;
      unpack8<T>(x[n], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
      if (pair[n]) {
        unpack8<T>(y[n], f);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
      }
      if (is_q[n]) sq += ss; else sk += ss;
    }
    rq = temp / sqrtf(block_sum32(sq, scratch) / static_cast<float>(a.H * a.d) + a.eps);
    if (heads > a.H) rk = 1.0f / sqrtf(block_sum32(sk, scratch) / static_cast<float>(a.G * a.d) + a.eps);
  }
  const int64_t page = slot / BS, off = slot % BS;
#pragma unroll
  for (int n = 0; n < N; ++n) {
    if (static_cast<int>(threadIdx.x + n * blockDim.x) >= total) continue;
    if (!NORM && is_q[n] && !pair[n]) continue;          // (stays as it is)
    float f[8], b[8], w[8];
    unpack8<T>(x[n], f);
    const float r = is_q[n] ? rq : rk;
    auto weigh = [&](float (&v)[8], int shift) {
      const float* wp = (is_q[n] ? a.wq : a.wk) + at[n] + shift;
      [[maybe_unused]] const void* wbase = is_q[n] ? a.wq : a.wk;
      const float4 w0 = MI355_LD(float4, wbase, wp), w1 = MI355_LD(float4, wbase, wp + 4);
      w[0] = w0.x, w[1] = w0.y, w[2] = w0.z, w[3] = w0.w, w[4] = w1.x, w[5] = w1.y, w[6] = w1.z, w[7] = w1.w;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = v[e] * r * w[e];
    };
    if (NORM) weigh(f, 0);
    if (pair[n]) {
      const int j = at[n] % a.d;
      unpack8<T>(y[n], b);
      if (NORM) weigh(b, half);
      const float4 c0 = MI355_LD(float4, a.cos_sin, cs + j), c1 = MI355_LD(float4, a.cos_sin, cs + j + 4);
      const float4 s0 = MI355_LD(float4, a.cos_sin, cs + half + j), s1 = MI355_LD(float4, a.cos_sin, cs + half + j + 4);
      const float c[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w}, s[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float f0 = f[e];
        f[e] = f0 * c[e] - b[e] * s[e];
        b[e] = b[e] * c[e] + f0 * s[e];
      }
    }
    if (is_q[n]) {
      MI355_ST(uint4, a.q, qr + at[n], pack8<T>(f));
      if (pair[n]) MI355_ST(uint4, a.q, qr + at[n] + half, pack8<T>(b));
    } else {
      uint16_t* o = a.k_cache + ((page * a.G + at[n] / a.d) * BS + off) * a.d + at[n] % a.d;
      MI355_ST(uint4, a.k_cache, o, pack8<T>(f));
      if (pair[n]) MI355_ST(uint4, a.k_cache, o + half, pack8<T>(b));
    }
  }
  if (!inline_v || heads == a.H) return;
  for (int i = threadIdx.x; i < a.G * a.dv / 8; i += blockDim.x) {
    const uint4 v = MI355_LD(uint4, a.v, a.v + t * a.v_stride + 8 * i);
    const int g = 8 * i / a.dv, j = 8 * i % a.dv;
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    uint16_t* o = a.v_cache + ((page * a.G + g) * a.dv + j) * BS + off;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      MI355_ST(uint16_t, a.v_cache, o + e * BS, static_cast<uint16_t>(e & 1 ? w[e >> 1] >> 16 : w[e >> 1] & 0xFFFFu));
  }
}

template <bool NORM>
static void launch_kv_rows(const KvRows& a, int dtype, hipStream_t s) {
  const int units = (a.H + (a.k != nullptr ? a.G : 0)) * ((a.d - a.rot / 2) / 8);
  const int threads = units >= 512 ? 512 : (units + 63) / 64 * 64;
  // V pages in the row's workgroup, 2 bytes a store, or by tiles of 16 rows and a kv head (a launch of its own; 16 rows that
  // store 2 bytes each meet in a sector).  The tiles pay from half a million numbers on, and where rows run on in their pages:
  // decoded rows lie in pages of their own.  Measured with the rotation, us (in the row / tiles; rows of one run, from its middle,
  // each in a page of its own): 64 rows of 4 heads of 128 4.2 / 5.8, 4.0 / 7.1, 3.9 / 10.3; 256 rows of 16 heads 6.5 / 5.6,
  // 6.5 / 7.2, 7.5 / 12.8; 1024 rows of 4 7.9 / 6.9, 8.0 / 8.2, 8.7 / 14.1; 8192 rows of 4 31 / 21, 31 / 23, 40 / 48.
  const int inline_v = a.num_tokens <= 256 || a.num_tokens * a.G * a.dv < (1 << 19) ? 1 : 0;
#define MI355_KVR(TT, ROT, N) \
  hipLaunchKernelGGL((kv_rows_vec_kernel<TT, NORM, ROT, N>), dim3(static_cast<unsigned>(a.num_tokens)), dim3(threads), 0, s, a, inline_v)
#define MI355_KVR_N(TT, ROT)                     \
  do {                                           \
    if (units <= 512) MI355_KVR(TT, ROT, 1);     \
    else if (units <= 1024) MI355_KVR(TT, ROT, 2); \
    else MI355_KVR(TT, ROT, 4);                  \
  } while (0)
  if (dtype == MI355_BF16) {
    if (a.rot > 0) MI355_KVR_N(BF16, true); else MI355_KVR_N(BF16, false);
  } else {
    if (a.rot > 0) MI355_KVR_N(F16, true); else MI355_KVR_N(F16, false);
  }
#undef MI355_KVR_N
#undef MI355_KVR
  if (!inline_v && a.k != nullptr)
    launch_v_pages(a.v, a.v_stride, a.slot_mapping, a.v_cache, 0x7FFFFFFF, a.num_tokens, a.G, a.dv, s);
}

}  // namespace mi355
