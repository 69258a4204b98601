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

// FRESH: the rows as they are projected.  The workgroup of a (row, kv head) rotates its queries and the new key by the float32 table
// cos_sin [max_pos][rot] (cos | sin), as rope_partial_kv_write does, takes the new key and value from LDS where its keys
// reach the row's position, and writes both to the slot's page (slot < 0: neither; the page counts as it is).
struct WindowFresh {
  const uint16_t *k, *v;
  int64_t k_stride, v_stride;
  const float* cos_sin;
  int64_t max_pos;
  const int64_t* slot_mapping;
  uint16_t *k_cache, *v_cache;
  int rot;
};
// uint16 of LDS that FRESH needs: rep queries and a key, rows padded to fall on all banks, and a value
__host__ __device__ constexpr int window_fresh_lds(int rep, int d, int dv) { return (rep + 1) * (d + 8) + dv; }

// Rows that are each the only one of their tile (decoded tokens): one workgroup per (row, kv head g, key range z of nz).  The
// query heads of the kv head lie on the 16 output columns, the waves take steps of 32 keys in turn, K and V go from
// memory to registers as MFMA operands (paged_attn_decode.hip's layout) and STG steps of a wave are in flight.  The
// weights are not normalised: the waves' sums, and the key ranges', simply add up.  partial given: fp32 sums without
// the gate to its slab z.  Bound by what
// one CU draws from memory: 32 rows, 16 heads of 128 on 4 kv heads, 1024 keys each, 17.6 us without ranges (21.9 in a decode
// step), 13 with two and the sum's launch behind it (the tile form, 15 of a tile's 16 rows empty and V by 8 bytes: 34 and 6
// for the sum).  Eight waves a workgroup in place of four: 18.0.
// wsum: NW * rep * (DV + 4) floats of LDS.
template <typename T, int D, int DV, int NW, int STG, bool FRESH = false>
__device__ __forceinline__ void sigmoid_window_decode(const WindowDecode& a, int64_t row, int g, int z, int nz, float* wsum,
                                                      const WindowFresh& f = WindowFresh{}, uint16_t* fresh = nullptr) {
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
  int pos = static_cast<int>(p < 0 ? -1 : p);                        // (below 16 * max_blocks: an int)
  if (FRESH) pos = __builtin_amdgcn_readfirstlane(pos);              // (a scalar: FRESH uses up the registers of 16 waves)
  const int lo = pos - window + 1 > 0 ? pos - window + 1 : 0;
  const int last_blk = pos > 0 ? pos / kWindowPage : 0;
  const int stride = 32 * NW * nz;
  int tb = (lo & ~31) + 32 * (z * NW + wave);
  const int koff = ((c >> 2) & 1) * 8 + (c & 3);                     // token row inside the page for K tile a (b: + 4)

  // FRESH: a thread has 4 rotation pairs (two pieces) or 4 coordinates past them of a query or the key, or 4 of the value
  constexpr int LR = D + 8;
  [[maybe_unused]] const int half = FRESH ? f.rot >> 1 : 0, units = (D - half) >> 2, turned = (rep + 1) * units;
  [[maybe_unused]] const int hh = static_cast<int>(threadIdx.x) / units, un = static_cast<int>(threadIdx.x) % units;
  [[maybe_unused]] const bool pair = FRESH && 4 * un < half;
  [[maybe_unused]] const int at = 4 * un + (pair ? 0 : half);
  [[maybe_unused]] int64_t slot = -1;
  [[maybe_unused]] int written = 0;
  [[maybe_unused]] uint2 fx = make_uint2(0u, 0u), fy = fx;
  [[maybe_unused]] float4 co, si;
  if constexpr (FRESH) {
    static_assert(64 * NW >= 8 * D / 4 + DV / 4, "a piece a thread, for up to 7 query heads");
    slot = MI355_LD(int64_t, f.slot_mapping, f.slot_mapping + row);
    if (static_cast<int>(threadIdx.x) < turned) {
      const uint16_t* src = hh < rep ? q + row * q_stride + static_cast<int64_t>(g * rep + hh) * D + at : f.k + row * f.k_stride + g * D + at;
      [[maybe_unused]] const void* base = hh < rep ? static_cast<const void*>(q) : static_cast<const void*>(f.k);
      fx = MI355_LD(uint2, base, src);
      if (pair) {
        const int64_t pc = p < 0 ? 0 : (p >= f.max_pos ? f.max_pos - 1 : p);
        const float* table = f.cos_sin + pc * f.rot + at;
        fy = MI355_LD(uint2, base, src + half);
        co = MI355_LD(float4, f.cos_sin, table), si = MI355_LD(float4, f.cos_sin, table + half);
      }
    } else if (static_cast<int>(threadIdx.x) < turned + DV / 4) {
      fx = MI355_LD(uint2, f.v, f.v + row * f.v_stride + g * DV + 4 * (static_cast<int>(threadIdx.x) - turned));
    }
  }
  uint4 qf[KS];
  if (!FRESH)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)                                  // columns past the group repeat its last head, unused
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
  if constexpr (FRESH) {
    uint16_t* kn = fresh + rep * LR;
    if (static_cast<int>(threadIdx.x) < turned) {
      uint2 rx = fx, ry = fy;
      if (pair) {
        auto turn = [&](uint32_t& u, uint32_t& v, float c0, float c1, float s0, float s1) {      // two pairs
          const float u0 = T::to_f(static_cast<uint16_t>(u & 0xFFFFu)), u1 = T::to_f(static_cast<uint16_t>(u >> 16));
          const float v0 = T::to_f(static_cast<uint16_t>(v & 0xFFFFu)), v1 = T::to_f(static_cast<uint16_t>(v >> 16));
          u = T::pack2(u0 * c0 - v0 * s0, u1 * c1 - v1 * s1);
          v = T::pack2(v0 * c0 + u0 * s0, v1 * c1 + u1 * s1);
        };
        turn(rx.x, ry.x, co.x, co.y, si.x, si.y), turn(rx.y, ry.y, co.z, co.w, si.z, si.w);
        *reinterpret_cast<uint2*>(fresh + hh * LR + at + half) = ry;
      }
      *reinterpret_cast<uint2*>(fresh + hh * LR + at) = rx;
      if (hh == rep && slot >= 0) {
        uint16_t* o = f.k_cache + ((slot / kWindowPage * G + g) * kWindowPage + slot % kWindowPage) * D + at;
        MI355_ST(uint2, f.k_cache, o, rx);
        if (pair) MI355_ST(uint2, f.k_cache, o + half, ry);
      }
    } else if (static_cast<int>(threadIdx.x) < turned + DV / 4) {
      const int ch = 4 * (static_cast<int>(threadIdx.x) - turned);
      *reinterpret_cast<uint2*>(kn + LR + ch) = fx;
      if (slot >= 0) {
        uint16_t* o = f.v_cache + ((slot / kWindowPage * G + g) * DV + ch) * kWindowPage + slot % kWindowPage;
        MI355_ST(uint16_t, f.v_cache, o, static_cast<uint16_t>(fx.x & 0xFFFFu));
        MI355_ST(uint16_t, f.v_cache, o + kWindowPage, static_cast<uint16_t>(fx.x >> 16));
        MI355_ST(uint16_t, f.v_cache, o + 2 * kWindowPage, static_cast<uint16_t>(fx.y & 0xFFFFu));
        MI355_ST(uint16_t, f.v_cache, o + 3 * kWindowPage, static_cast<uint16_t>(fx.y >> 16));
      }
    }
    written = __builtin_amdgcn_readfirstlane(slot >= 0 ? 1 : 0);
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const uint4*>(fresh + (c < rep ? c : rep - 1) * LR + 32 * ks + 8 * h);
  }
  f32x4 o[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](uint4 (&ka_)[KS], uint4 (&b)[KS], uint4 (&v)[NT], int t0) {
    if (FRESH && written && pos - t0 < 32) {                       // the step with the row's own key (wave-uniform)
      const uint16_t* kn = fresh + rep * LR;
      int r = __builtin_amdgcn_readfirstlane(pos - t0), lane = threadIdx.x & 63;
      asm volatile("" : "+s"(r), "+v"(lane));                        // (worked out here: ahead of the loop a register would be missing)
      const int c = lane & 15, h = lane >> 4, mine = 16 * (c >> 3) + ((c >> 2) & 1) * 8 + (c & 3);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const uint4 key = *reinterpret_cast<const uint4*>(kn + 32 * ks + 8 * h);
        if (mine == r) ka_[ks] = key;
        if (mine + 4 == r) b[ks] = key;
      }
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const uint32_t value = kn[LR + 16 * n + c], put = r & 1 ? value << 16 : value, keep = r & 1 ? 0x0000FFFFu : 0xFFFF0000u;
        const int word = r >> 3 == h ? (r & 7) >> 1 : -1;
        v[n].x = word == 0 ? (v[n].x & keep) | put : v[n].x, v[n].y = word == 1 ? (v[n].y & keep) | put : v[n].y;
        v[n].z = word == 2 ? (v[n].z & keep) | put : v[n].z, v[n].w = word == 3 ? (v[n].w & keep) | put : v[n].w;
      }
    }
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
