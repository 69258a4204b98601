// The gated delta rule of single tokens (a decode step), from the input projection to the rows that the output matrix
// multiplies: convolution with its state, low-rank decay and gate, the recurrence, the norm over each head and its gate.
//
// A workgroup per (row, key head), 512 threads for each of its R value heads: the key head's convolution channels and
// their state then belong to one workgroup, so that the state is shifted where it is read.  What bounds it is the recurrent
// state's trip from memory and back (128 x 128 fp32 a head) and one chain of loads, sums and two barriers; as five to seven
// launches (convolution 4.8 us, decay and gate 4.5 each, recurrence, head norm 4.7) the chain was the launches.
// Measured in a step of 32 rows: 16 heads on 8 with a decay a head 16.2 us (67 MB; in three launches 26), 8 heads on 4 with a
// decay a channel 13.4 (in five 29).
//
// In a head: 32 lanes of four value columns by 16 groups of rows; a thread holds 8 rows of its columns.  S'q =
// (a S)'q + u (k'q), so that one reduction over the rows serves the removal and the result.
#include "common.h"
#include "window_decode.h"

namespace mi355 {

constexpr int kDeltaD = 128, kDeltaTaps = 4;

struct DeltaDecode {
  uint16_t* out;
  int64_t out_stride;
  const uint16_t* proj;                  // a row: the columns below at their offsets
  int64_t stride;
  int qkv_off, beta_off, a_off, g_off;   // a, g: the raw decay and gate, or (a decay a channel) what their matrices multiply
  const uint16_t *conv_w, *a2, *g2;      // [channels][taps], [heads * 128][rank]
  float* conv_state;                     // [slots][taps - 1][channels]
  int taps, rank;
  const float *a_log, *dt_bias, *norm_w;
  int norm_heads, act;
  float eps;
  float* state;                          // [slots][heads][128][128]
  const int64_t* positions;
  const int32_t* state_slots;
  int H, G;
};

// what a workgroup keeps in LDS
template <int R>
struct DeltaLds {
  float ys[(2 + R) * kDeltaD];                                         // q | k | v of the heads, convolved
  float as[R][kDeltaD], gs[R][kDeltaD], sums[R][8][2][kDeltaD];
};

template <typename T, bool PC, int R>
__device__ __forceinline__ void delta_decode(const DeltaDecode& a, int s, int g, DeltaLds<R>& lds) {
  constexpr int D = kDeltaD, N = D / 16, CH = (2 + R) * D;
  auto &ys = lds.ys;
  auto &as = lds.as, &gs = lds.gs;
  auto &sums = lds.sums;
  const int tid = threadIdx.x, lane = tid & 63;
  const int hl = R == 1 ? 0 : tid >> 9, t = tid & 511, wave = t >> 6, h = g * R + hl;
  const int cl = t & 31, rg = t >> 5;
  const uint16_t* row = a.proj + s * a.stride;
  const int64_t slot = MI355_LD(int32_t, a.state_slots, a.state_slots + s), p = MI355_LD(int64_t, a.positions, a.positions + s);
  const int C = (2 * a.G + a.H) * D, taps = a.taps;
  // ---- all loads out before the first is used: the convolution's, the decay's, then the state
  const bool conv = tid < CH;
  const int ch = tid < D ? g * D + tid : tid < 2 * D ? (a.G + g - 1) * D + tid : (2 * a.G + g * R - 2) * D + tid;
  float* cst = a.conv_state + slot * (taps - 1) * C + ch;
  float in[kDeltaTaps], wv[kDeltaTaps];
  if (conv) {
#pragma unroll
    for (int j = 0; j < kDeltaTaps; ++j) {
      const int m = j < taps ? j : taps - 1;
      wv[j] = T::to_f(MI355_LD(uint16_t, a.conv_w, a.conv_w + static_cast<int64_t>(ch) * taps + m));
      in[j] = m < taps - 1 ? MI355_LD(float, a.conv_state, cst + static_cast<int64_t>(m) * C)
                           : T::to_f(MI355_LD(uint16_t, a.proj, row + a.qkv_off + ch));
    }
  }
  const float alog = MI355_LD(float, a.a_log, a.a_log + h), beta = T::to_f(MI355_LD(uint16_t, a.proj, row + a.beta_off + h));
  // one output of a [heads * 128][rank] matrix for four lanes, a quarter of its inputs each
  const int oc = t >> 2, part = a.rank >> 2;
  auto low_rank = [&](const uint16_t* w, int off) {
    const uint16_t* wr = w + (static_cast<int64_t>(h) * D + oc) * a.rank + (t & 3) * part;
    const uint16_t* xr = row + off + (t & 3) * part;
    float sum = 0.f;
#pragma unroll 4
    for (int i = 0; i < part; i += 8) {
      float x[8], y[8];
      unpack8<T>(MI355_LD(uint4, w, wr + i), x), unpack8<T>(MI355_LD(uint4, a.proj, xr + i), y);
#pragma unroll
      for (int e = 0; e < 8; ++e) sum += x[e] * y[e];
    }
    sum += __shfl_xor(sum, 1, 64);
    return round_f<T>(sum + __shfl_xor(sum, 2, 64));
  };
  const float z = PC ? low_rank(a.a2, a.a_off) + MI355_LD(float, a.dt_bias, a.dt_bias + h * D + oc)
                     : T::to_f(MI355_LD(uint16_t, a.proj, row + a.a_off + h)) + MI355_LD(float, a.dt_bias, a.dt_bias + h);
  const int col = 4 * cl;
  float* sp = a.state + (slot * a.H + h) * (D * D) + col;
  float4 S[N];
#pragma unroll
  for (int j = 0; j < N; ++j) S[j] = MI355_LD(float4, a.state, sp + (j * 16 + rg) * D);
  __builtin_amdgcn_sched_barrier(0);
  if (conv) {
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < kDeltaTaps; ++j)
      if (j < taps && p - (taps - 1 - j) >= 0) acc += wv[j] * in[j];  // (zeros before the start of the sequence)
    ys[tid] = round_f<T>(silu_any(acc));          // (the same bits as the convolution of prompts)
#pragma unroll
    for (int j = 0; j < kDeltaTaps - 1; ++j)
      if (j < taps - 1) MI355_ST(float, a.conv_state, cst + static_cast<int64_t>(j) * C, in[j + 1]);
  }
  const float decay = expf(-expf(alog) * (z > 20.0f ? z : log1pf(expf(z)))), b = 1.0f / (1.0f + expf(-beta));
  if (PC) {
    const float gate = low_rank(a.g2, a.g_off);
    if ((t & 3) == 0) as[hl][oc] = decay, gs[hl][oc] = gate;
  }
  __syncthreads();
  // ---- unit key, unit query / sqrt(d), and their product
  const float k0 = ys[D + lane], k1 = ys[D + 64 + lane], q0 = ys[lane], q1 = ys[64 + lane];
  const float kk = 1.0f / sqrtf(wave_sum(k0 * k0 + k1 * k1) + 1e-6f);
  const float qq = (1.0f / sqrtf(static_cast<float>(D))) / sqrtf(wave_sum(q0 * q0 + q1 * q1) + 1e-6f);
  const float kq = wave_sum(k0 * q0 + k1 * q1) * kk * qq;
  float4 dk = make_float4(0.f, 0.f, 0.f, 0.f), dq = dk;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int i = j * 16 + rg;
    if (p == 0) S[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    const float x = PC ? as[hl][i] : decay, k = ys[D + i] * kk, q = ys[i] * qq;
    S[j].x *= x, S[j].y *= x, S[j].z *= x, S[j].w *= x;
    dk.x += S[j].x * k, dk.y += S[j].y * k, dk.z += S[j].z * k, dk.w += S[j].w * k;
    dq.x += S[j].x * q, dq.y += S[j].y * q, dq.z += S[j].z * q, dq.w += S[j].w * q;
  }
  auto over_rows = [](float v) { return v + __shfl_xor(v, 32, 64); };
  dk = make_float4(over_rows(dk.x), over_rows(dk.y), over_rows(dk.z), over_rows(dk.w));
  dq = make_float4(over_rows(dq.x), over_rows(dq.y), over_rows(dq.z), over_rows(dq.w));
  if (lane < 32) {
    *reinterpret_cast<float4*>(&sums[hl][wave][0][col]) = dk;
    *reinterpret_cast<float4*>(&sums[hl][wave][1][col]) = dq;
  }
  __syncthreads();
  dk = dq = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    const float4 x = *reinterpret_cast<const float4*>(&sums[hl][w][0][col]), y = *reinterpret_cast<const float4*>(&sums[hl][w][1][col]);
    dk.x += x.x, dk.y += x.y, dk.z += x.z, dk.w += x.w;
    dq.x += y.x, dq.y += y.y, dq.z += y.z, dq.w += y.w;
  }
  const float* v = &ys[(2 + hl) * D + col];
  const float u[4] = {b * (v[0] - dk.x), b * (v[1] - dk.y), b * (v[2] - dk.z), b * (v[3] - dk.w)};
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const float k = ys[D + j * 16 + rg] * kk;
    S[j].x += k * u[0], S[j].y += k * u[1], S[j].z += k * u[2], S[j].w += k * u[3];
    MI355_ST(float4, a.state, sp + (j * 16 + rg) * D, S[j]);
  }
  if (rg != 0) return;
  // ---- the head's norm and gate: 32 lanes hold its 128 numbers
  float o[4] = {dq.x + u[0] * kq, dq.y + u[1] * kq, dq.z + u[2] * kq, dq.w + u[3] * kq};
  float ss = o[0] * o[0] + o[1] * o[1] + o[2] * o[2] + o[3] * o[3];
#pragma unroll
  for (int off = 1; off < 32; off <<= 1) ss += __shfl_xor(ss, off, 64);
  const float r = 1.0f / sqrtf(ss / static_cast<float>(D) + a.eps);
  const float4 nw = MI355_LD(float4, a.norm_w, a.norm_w + (a.norm_heads > 1 ? h * D : 0) + col);
  float gt[4];
  if (PC) {
#pragma unroll
    for (int e = 0; e < 4; ++e) gt[e] = gs[hl][col + e];
  } else {
    const uint2 raw = MI355_LD(uint2, a.proj, row + a.g_off + h * D + col);
    gt[0] = T::to_f(raw.x & 0xFFFFu), gt[1] = T::to_f(raw.x >> 16), gt[2] = T::to_f(raw.y & 0xFFFFu), gt[3] = T::to_f(raw.y >> 16);
  }
  const float n4[4] = {nw.x, nw.y, nw.z, nw.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float sg = 1.0f / (1.0f + expf(-gt[e]));
    o[e] = o[e] * r * n4[e] * (a.act == 0 ? gt[e] * sg : sg);
  }
  MI355_ST(uint2, a.out, a.out + s * a.out_stride + h * D + col, make_uint2(T::pack2(o[0], o[1]), T::pack2(o[2], o[3])));
}

template <typename T, bool PC, int R>
__global__ __launch_bounds__(512 * R) void delta_decode_kernel(DeltaDecode a) {
  __shared__ __attribute__((aligned(16))) DeltaLds<R> lds;
  delta_decode<T, PC, R>(a, blockIdx.x, blockIdx.y, lds);
}

// The same beside a sliding-window attention of the same rows (a layer that mixes both): neither needs the other, and
// either leaves half of the chip idle at a few dozen rows.  Workgroups of 16 waves for both: first the attention's, one per
// (row, kv head), then the recurrence's.  Measured in a step of 32 rows, 16 heads on 4 kv heads behind 1024 keys and 8 heads on 4:
// 24.4 us, one after the other 21.9 and 13.4.
// FRESH: the attention's rows as they are projected (WindowFresh), for which a launch of 5 us went ahead: 32 rows 27.3 us with it, 24.2
// here (the table's and the rows' loads travel with the pages').
template <typename T, bool PC, bool FRESH>
__global__ __launch_bounds__(1024) void window_delta_decode_kernel(WindowDecode w, DeltaDecode a, int rows, WindowFresh f) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int b = blockIdx.x, attention = rows * w.G;
  if (b < attention)
    sigmoid_window_decode<T, 128, 128, 16, 1, FRESH>(w, b % rows, b / rows, 0, 1, smem, f,
                                                     reinterpret_cast<uint16_t*>(smem + 16 * (w.H / w.G) * (128 + 4)));
  else delta_decode<T, PC, 2>(a, (b - attention) % rows, (b - attention) / rows, *reinterpret_cast<DeltaLds<2>*>(smem));
}

static int32_t check_delta_decode(const char* name, const DeltaDecode& a, int64_t num_rows, int head_dim, int v_dim, int dtype) {
  MI355_REQUIRE(a.out && a.proj && a.conv_w && a.conv_state && a.a_log && a.dt_bias && a.norm_w && a.state && a.positions && a.state_slots &&
                    (a.a2 == nullptr) == (a.g2 == nullptr),
                MI355_ERR_INVALID, "%s: null pointer", name);
  MI355_REQUIRE(num_rows >= 0 && a.H > 0 && a.G > 0 && a.H % a.G == 0 && a.qkv_off >= 0 && a.beta_off >= 0 && a.a_off >= 0 && a.g_off >= 0 &&
                    (a.norm_heads == 1 || a.norm_heads == a.H) && (a.a2 == nullptr || a.rank > 0),
                MI355_ERR_INVALID, "%s: sizes", name);
  MI355_REQUIRE((dtype == MI355_BF16 || dtype == MI355_F16) && head_dim == kDeltaD && v_dim == kDeltaD && a.H / a.G <= 2 && a.taps >= 2 &&
                    a.taps <= kDeltaTaps && a.G <= 65535,
                MI355_ERR_UNSUPPORTED, "%s: 16-bit storage, heads of 128 x 128, one or two to a key head, 2 to 4 taps", name);
  MI355_REQUIRE(aligned16(a.state) && aligned16(a.norm_w) && (reinterpret_cast<uintptr_t>(a.out) & 7u) == 0 && a.out_stride % 4 == 0 &&
                    (a.a2 == nullptr ? (reinterpret_cast<uintptr_t>(a.proj) & 7u) == 0 && a.stride % 4 == 0 && a.g_off % 4 == 0
                                     : a.rank % 32 == 0 && aligned16(a.a2) && aligned16(a.g2) && aligned16(a.proj) && a.stride % 8 == 0 &&
                                           a.a_off % 8 == 0 && a.g_off % 8 == 0),
                MI355_ERR_UNSUPPORTED, "%s: columns on whole pieces, a rank that is a multiple of 32", name);
  return MI355_OK;
}

}  // namespace mi355

extern "C" int32_t mi355_delta_decode(void* out, int64_t out_stride, const void* proj, int64_t proj_stride, int32_t qkv_off,
                                      int32_t beta_off, int32_t a_off, int32_t g_off, const void* conv_w, float* conv_state,
                                      int32_t taps, const void* a2, const void* g2, int32_t rank, const float* a_log,
                                      const float* dt_bias, const float* norm_w, int32_t norm_heads, int32_t act, float eps,
                                      float* state, const int64_t* positions, const int32_t* state_slots, int32_t num_rows,
                                      int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t v_dim, int32_t dtype,
                                      void* stream) {
  using namespace mi355;
  const DeltaDecode a = {static_cast<uint16_t*>(out), out_stride, static_cast<const uint16_t*>(proj), proj_stride, qkv_off, beta_off, a_off,
                         g_off, static_cast<const uint16_t*>(conv_w), static_cast<const uint16_t*>(a2), static_cast<const uint16_t*>(g2),
                         conv_state, taps, rank, a_log, dt_bias, norm_w, norm_heads, act, eps, state, positions, state_slots, num_heads,
                         num_kv_heads};
  const int32_t rc = check_delta_decode("delta_decode", a, num_rows, head_dim, v_dim, dtype);
  if (rc != MI355_OK || num_rows == 0) return rc;
  const int per = num_heads / num_kv_heads;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid(static_cast<unsigned>(num_rows), static_cast<unsigned>(num_kv_heads));
#define MI355_DD(TT, PC, R) hipLaunchKernelGGL((delta_decode_kernel<TT, PC, R>), grid, dim3(512 * R), 0, s, a)
#define MI355_DD_R(TT)                                     \
  do {                                                     \
    if (a2 != nullptr && per == 2) MI355_DD(TT, true, 2);  \
    else if (a2 != nullptr) MI355_DD(TT, true, 1);         \
    else if (per == 2) MI355_DD(TT, false, 2);             \
    else MI355_DD(TT, false, 1);                           \
  } while (0)
  if (dtype == MI355_BF16) MI355_DD_R(BF16); else MI355_DD_R(F16);
#undef MI355_DD_R
#undef MI355_DD
  return check_launch("delta_decode");
}

static int32_t window_delta_decode(const char* name, const mi355::WindowFresh* fresh, void* attn_out, const void* q, int64_t q_stride,
                                   const void* k_cache, const void* v_cache, const int32_t* block_tables, int32_t max_blocks,
                                   const int32_t* tok_seq, const float* temp, const float* bias, const void* gate, int64_t gate_stride,
                                   int32_t attn_heads, int32_t attn_kv_heads, int32_t window, float scale, void* out, int64_t out_stride,
                                   const void* proj, int64_t proj_stride, int32_t qkv_off, int32_t beta_off, int32_t a_off, int32_t g_off,
                                   const void* conv_w, float* conv_state, int32_t taps, const void* a2, const void* g2, int32_t rank,
                                   const float* a_log, const float* dt_bias, const float* norm_w, int32_t norm_heads, int32_t act, float eps,
                                   float* state, const int64_t* positions, const int32_t* state_slots, int32_t num_rows, int32_t num_heads,
                                   int32_t num_kv_heads, int32_t head_dim, int32_t v_dim, int32_t dtype, void* stream) {
  using namespace mi355;
  const DeltaDecode a = {static_cast<uint16_t*>(out), out_stride, static_cast<const uint16_t*>(proj), proj_stride, qkv_off, beta_off, a_off,
                         g_off, static_cast<const uint16_t*>(conv_w), static_cast<const uint16_t*>(a2), static_cast<const uint16_t*>(g2),
                         conv_state, taps, rank, a_log, dt_bias, norm_w, norm_heads, act, eps, state, positions, state_slots, num_heads,
                         num_kv_heads};
  const int32_t rc = check_delta_decode(name, a, num_rows, head_dim, v_dim, dtype);
  if (rc != MI355_OK) return rc;
  MI355_REQUIRE(attn_out && q && k_cache && v_cache && block_tables && tok_seq && temp && bias, MI355_ERR_INVALID, "%s: null pointer", name);
  MI355_REQUIRE(attn_heads > 0 && attn_kv_heads > 0 && attn_heads % attn_kv_heads == 0 && max_blocks > 0 && window > 0, MI355_ERR_INVALID,
                "%s: sizes", name);
  const size_t sums = sizeof(float) * 16 * (attn_heads / attn_kv_heads) * (128 + 4);
  MI355_REQUIRE(sums <= 65536 && num_heads == 2 * num_kv_heads && q_stride % 8 == 0 && aligned16(q) && aligned16(k_cache) &&
                    aligned16(v_cache) && aligned16(attn_out),
                MI355_ERR_UNSUPPORTED, "%s: at most 7 query heads a kv head, two heads a key head, 16-byte aligned rows", name);
  if (fresh != nullptr) {
    MI355_REQUIRE(fresh->k && fresh->v && fresh->cos_sin && fresh->slot_mapping && fresh->max_pos > 0 && fresh->rot >= 0 && fresh->rot <= 128 &&
                      fresh->k_stride >= attn_kv_heads * 128 && fresh->v_stride >= attn_kv_heads * 128,
                  MI355_ERR_INVALID, "%s: keys, values, table and slots", name);
    MI355_REQUIRE(fresh->rot % 16 == 0 && fresh->k_stride % 8 == 0 && fresh->v_stride % 8 == 0 && aligned16(fresh->k) && aligned16(fresh->v) &&
                      aligned16(fresh->cos_sin),
                  MI355_ERR_UNSUPPORTED, "%s: rotated coordinates a multiple of 16, 16-byte aligned rows", name);
  }
  if (num_rows == 0) return MI355_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const WindowDecode w = {static_cast<uint16_t*>(attn_out), static_cast<const uint16_t*>(q), q_stride, static_cast<const uint16_t*>(k_cache),
                          static_cast<const uint16_t*>(v_cache), block_tables, max_blocks, tok_seq, positions, temp, bias,
                          static_cast<const uint16_t*>(gate), gate_stride, attn_heads, attn_kv_heads, window, scale, nullptr, 0};
  const size_t mine = sums + (fresh != nullptr ? sizeof(uint16_t) * window_fresh_lds(attn_heads / attn_kv_heads, 128, 128) : 0);
  const size_t lds = mine > sizeof(DeltaLds<2>) ? mine : sizeof(DeltaLds<2>);
  const dim3 grid(static_cast<unsigned>(num_rows) * static_cast<unsigned>(attn_kv_heads + num_kv_heads));
#define MI355_WDD(TT, PC)                                                                                                               \
  do {                                                                                                                                  \
    if (fresh != nullptr)                                                                                                               \
      hipLaunchKernelGGL((window_delta_decode_kernel<TT, PC, true>), grid, dim3(1024), lds, s, w, a, num_rows, *fresh);                 \
    else hipLaunchKernelGGL((window_delta_decode_kernel<TT, PC, false>), grid, dim3(1024), lds, s, w, a, num_rows, WindowFresh{});      \
  } while (0)
  if (dtype == MI355_BF16 && a2 != nullptr) MI355_WDD(BF16, true);
  else if (dtype == MI355_BF16) MI355_WDD(BF16, false);
  else if (a2 != nullptr) MI355_WDD(F16, true);
  else MI355_WDD(F16, false);
#undef MI355_WDD
  return check_launch(name);
}

extern "C" int32_t mi355_window_delta_decode(void* attn_out, const void* q, int64_t q_stride, const void* k_cache, const void* v_cache,
                                             const int32_t* block_tables, int32_t max_blocks, const int32_t* tok_seq, const float* temp,
                                             const float* bias, const void* gate, int64_t gate_stride, int32_t attn_heads,
                                             int32_t attn_kv_heads, int32_t window, float scale, void* out, int64_t out_stride,
                                             const void* proj, int64_t proj_stride, int32_t qkv_off, int32_t beta_off, int32_t a_off,
                                             int32_t g_off, const void* conv_w, float* conv_state, int32_t taps, const void* a2,
                                             const void* g2, int32_t rank, const float* a_log, const float* dt_bias, const float* norm_w,
                                             int32_t norm_heads, int32_t act, float eps, float* state, const int64_t* positions,
                                             const int32_t* state_slots, int32_t num_rows, int32_t num_heads, int32_t num_kv_heads,
                                             int32_t head_dim, int32_t v_dim, int32_t dtype, void* stream) {
  return window_delta_decode("window_delta_decode", nullptr, attn_out, q, q_stride, k_cache, v_cache, block_tables, max_blocks, tok_seq, temp,
                             bias, gate, gate_stride, attn_heads, attn_kv_heads, window, scale, out, out_stride, proj, proj_stride, qkv_off,
                             beta_off, a_off, g_off, conv_w, conv_state, taps, a2, g2, rank, a_log, dt_bias, norm_w, norm_heads, act, eps,
                             state, positions, state_slots, num_rows, num_heads, num_kv_heads, head_dim, v_dim, dtype, stream);
}

extern "C" int32_t mi355_window_delta_decode_rows(void* attn_out, const void* q, int64_t q_stride, const void* k, int64_t k_stride,
                                                  const void* v, int64_t v_stride, const float* cos_sin, int32_t max_pos, int32_t rot_dims,
                                                  const int64_t* slot_mapping, void* k_cache, void* v_cache, const int32_t* block_tables,
                                                  int32_t max_blocks, const int32_t* tok_seq, const float* temp, const float* bias,
                                                  const void* gate, int64_t gate_stride, int32_t attn_heads, int32_t attn_kv_heads,
                                                  int32_t window, float scale, void* out, int64_t out_stride, const void* proj,
                                                  int64_t proj_stride, int32_t qkv_off, int32_t beta_off, int32_t a_off, int32_t g_off,
                                                  const void* conv_w, float* conv_state, int32_t taps, const void* a2, const void* g2,
                                                  int32_t rank, const float* a_log, const float* dt_bias, const float* norm_w,
                                                  int32_t norm_heads, int32_t act, float eps, float* state, const int64_t* positions,
                                                  const int32_t* state_slots, int32_t num_rows, int32_t num_heads, int32_t num_kv_heads,
                                                  int32_t head_dim, int32_t v_dim, int32_t dtype, void* stream) {
  const mi355::WindowFresh fresh = {static_cast<const uint16_t*>(k), static_cast<const uint16_t*>(v), k_stride, v_stride, cos_sin, max_pos,
                                    slot_mapping, static_cast<uint16_t*>(k_cache), static_cast<uint16_t*>(v_cache), rot_dims};
  return window_delta_decode("window_delta_decode_rows", &fresh, attn_out, q, q_stride, k_cache, v_cache, block_tables, max_blocks, tok_seq,
                             temp, bias, gate, gate_stride, attn_heads, attn_kv_heads, window, scale, out, out_stride, proj, proj_stride,
                             qkv_off, beta_off, a_off, g_off, conv_w, conv_state, taps, a2, g2, rank, a_log, dt_bias, norm_w, norm_heads, act,
                             eps, state, positions, state_slots, num_rows, num_heads, num_kv_heads, head_dim, v_dim, dtype, stream);
}
