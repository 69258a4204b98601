// Sliding-window attention with sigmoid weights for rows that are a sequence's newest token each: the workgroup's work, for
// launches of it alone and beside other work.
#pragma once

#include "common.h"

namespace mi355 {

constexpr int kWindowPage = MI355_BLOCK_SIZE;

struct WindowDecode {
  uint16_t* out;
  const uint16_t* q;
  int64_t q_stride;
  const uint16_t *k_cache, *v_cache;
  const int32_t* block_tables;
  int max_blocks;
  const int32_t* tok_seq;
  const int64_t* positions;
  const float *temp, *bias;
  const uint16_t* gate;
  int64_t gate_stride;
  int H, G, window;
  float scale;
  float* partial;
  int64_t partial_stride;
};

// Rows that are each the only one of their tile (decoded tokens): one workgroup per (row, kv head g, key range z of nz).  The
// query heads of the kv head lie on the 16 output columns, the waves take steps of 32 keys in turn, K and V go from
// memory to registers as MFMA operands (paged_attn_decode.hip's layout) and STG steps of a wave are in flight.  The
// weights are not normalised: the waves' sums, and the key ranges', simply add up.  partial given: fp32 sums without
// the gate to its slab z.  Bound by what
// one CU draws from memory: 32 rows, 16 heads of 128 on 4 kv heads, 1024 keys each, 17.6 us without ranges (21.9 in a decode
// step), 13 with two and the sum's launch behind it (the tile form, 15 of a tile's 16 rows empty and V by 8 bytes: 34 and 6
// for the sum).  Eight waves a workgroup in place of four: 18.0.
// wsum: NW * rep * (DV + 4) floats of LDS.
template <typename T, int D, int DV, int NW, int STG>
__device__ __forceinline__ void sigmoid_window_decode(const WindowDecode& a, int64_t row, int g, int z, int nz, float* wsum) {
  constexpr int KS = D / 32, NT = DV / 16, DP = DV + 4;
  uint16_t* const out = a.out;
  const uint16_t *const q = a.q, *const k_cache = a.k_cache, *const v_cache = a.v_cache, *const gate = a.gate;
  const int32_t *const block_tables = a.block_tables, *const tok_seq = a.tok_seq;
  const int64_t* const positions = a.positions;
  const float *const temp = a.temp, *const bias = a.bias;
  float* const partial = a.partial;
  const int64_t q_stride = a.q_stride, gate_stride = a.gate_stride, partial_stride = a.partial_stride;
  const int max_blocks = a.max_blocks, H = a.H, G = a.G, window = a.window;
  const float scale = a.scale;
  const int rep = H / G;
  const int lane = threadIdx.x & 63, c = lane & 15, h = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t p = MI355_LD(int64_t, positions, positions + row);
  const int32_t* bt = block_tables + static_cast<int64_t>(MI355_LD(int32_t, tok_seq, tok_seq + row)) * max_blocks;
  const int pos = static_cast<int>(p < 0 ? -1 : p);                  // (below 16 * max_blocks: an int)
  const int lo = pos - window + 1 > 0 ? pos - window + 1 : 0;
  const int last_blk = pos > 0 ? pos / kWindowPage : 0;
  const int stride = 32 * NW * nz;
  int tb = (lo & ~31) + 32 * (z * NW + wave);
  const int koff = ((c >> 2) & 1) * 8 + (c & 3);                     // token row inside the page for K tile a (b: + 4)

  uint4 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)                                    // columns past the group repeat its last head, unused
    qf[ks] = MI355_LD(uint4, q, q + row * q_stride + static_cast<int64_t>(g * rep + (c < rep ? c : rep - 1)) * D + 32 * ks + 8 * h);
  const int head = g * rep + (c < rep ? c : rep - 1);
  const float mul = -1.4426950408889634f * scale * MI355_LD(float, temp, temp + head);
  const float add = -1.4426950408889634f * MI355_LD(float, bias, bias + head);

  uint4 ka[STG][KS], kb[STG][KS], vf[STG][NT];
  // always issued: a step beyond the range asks for one address of a page that the row sees, and is not used
  auto issue = [&](uint4 (&ka_)[KS], uint4 (&b)[KS], uint4 (&v)[NT], int t0) {
    const int live = t0 <= pos ? 1 : 0;
    const int bi = min(t0 / kWindowPage, last_blk);
    const int64_t p0 = MI355_LD(int32_t, block_tables, bt + bi), p1 = MI355_LD(int32_t, block_tables, bt + min(bi + 1, last_blk));
    const uint16_t* kp = k_cache + (((c & 8) ? p1 : p0) * G + g) * (kWindowPage * D) + live * (koff * D + 8 * h);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      ka_[ks] = MI355_LD(uint4, k_cache, kp + 32 * ks);
      b[ks] = MI355_LD(uint4, k_cache, kp + 4 * D + 32 * ks);
    }
    const uint16_t* vp = v_cache + (((h & 2) ? p1 : p0) * G + g) * (kWindowPage * DV) + live * (c * kWindowPage + 8 * (h & 1));
#pragma unroll
    for (int n = 0; n < NT; ++n) v[n] = MI355_LD(uint4, v_cache, vp + n * 16 * kWindowPage);
  };
#pragma unroll
  for (int j = 0; j < STG; ++j) issue(ka[j], kb[j], vf[j], tb + j * stride);
  f32x4 o[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](uint4 (&ka_)[KS], uint4 (&b)[KS], uint4 (&v)[NT], int t0) {
    f32x4 sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      sa = T::mfma(ka_[ks], qf[ks], sa);
      sb = T::mfma(b[ks], qf[ks], sb);
    }
    const int tok0 = t0 + 8 * h;                                     // this lane's keys are tok0 .. tok0 + 7
    float w[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float x = j < 4 ? sa[j & 3] : sb[j & 3];
      w[j] = tok0 + j >= lo && tok0 + j <= pos ? __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * mul + add)) : 0.f;
    }
    const uint4 pf = pack8<T>(w);
    if (t0 + 31 > pos) {                                             // slots past the newest key may hold anything (0 * NaN)
      uint32_t keep[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) keep[e] = (tok0 + 2 * e <= pos ? 0x0000FFFFu : 0u) | (tok0 + 2 * e + 1 <= pos ? 0xFFFF0000u : 0u);
#pragma unroll
      for (int n = 0; n < NT; ++n) v[n].x &= keep[0], v[n].y &= keep[1], v[n].z &= keep[2], v[n].w &= keep[3];
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) o[n] = T::mfma(v[n], pf, o[n]);
  };
  while (tb <= pos) {
#pragma unroll
    for (int j = 0; j < STG; ++j) {
      if (tb <= pos) step(ka[j], kb[j], vf[j], tb);
      issue(ka[j], kb[j], vf[j], tb + STG * stride);
      tb += stride;
    }
  }
  if (c < rep) {
#pragma unroll
    for (int n = 0; n < NT; ++n) *reinterpret_cast<f32x4*>(&wsum[(wave * rep + c) * DP + 16 * n + 4 * h]) = o[n];
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < rep * (DV / 2); idx += 64 * NW) {
    const int hh = idx / (DV / 2), e = 2 * (idx % (DV / 2));
    float2 v = *reinterpret_cast<const float2*>(&wsum[hh * DP + e]);
#pragma unroll
    for (int w = 1; w < NW; ++w) {
      const float2 u = *reinterpret_cast<const float2*>(&wsum[(w * rep + hh) * DP + e]);
      v.x += u.x, v.y += u.y;
    }
    const int64_t at = (row * H + g * rep + hh) * DV + e;
    if (partial != nullptr) {
      MI355_ST(float2, partial, partial + z * partial_stride + at, v);
      continue;
    }
    float gt = 1.0f;
    if (gate != nullptr) gt = 1.0f / (1.0f + expf(-T::to_f(MI355_LD(uint16_t, gate, gate + row * gate_stride + g * rep + hh))));
    MI355_ST(uint32_t, out, out + at, T::pack2(v.x * gt, v.y * gt));
  }
}

}  // namespace mi355
