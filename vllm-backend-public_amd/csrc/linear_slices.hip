// Decode-time linear layer on fp8 fragment-tiled weights (the layout of mi355_tile_weights_fp8), K split over the waves of a workgroup:
// y[M, N] = x[M, K] . W[N, K]^T, up to 32 rows (of a row block).
//
// A workgroup of four waves, one a SIMD, owns TP adjacent 16-row tiles; wave w multiplies the w-th part of K (of the workgroup's K group) with
// all of them.  A wave's fragments of x are then its own and serve TP tiles each: they come from L2 straight to registers, once a
// workgroup, and the loop has neither LDS nor a barrier.  Every weight register is loaded again as soon as it has been used, so that a wave
// has 2 TP KB on their way all the time.  The four partial sums of a tile meet in LDS at the end and are added by one wave in the order of
// K (the two tiles of a SwiGLU pair by the same one).
//
// What bounds it: the weight stream, and x for every workgroup out of L2.  Measured, us, before (x staged in LDS by linear_tiled.hip) / now:
//   3584 -> 37888 (136 MB)   1 row 25.4 / 23.7, 16 rows 26.5 / 23.7, 17 rows 33.7 / 24.8, 32 rows 34.2 / 25.9 (5.2 TB/s)
//   18944 -> 3584 (68 MB)    14.2 / 12.8, 15.1 / 13.8, 16.0 / 14.1, 17.4 / 15.9
//   3584 -> 4608 (17 MB)     6.1 / 5.3, 6.4 / 6.0, 6.9 / 6.2, 7.5 / 7.1; 64 rows in two blocks 10.2 / 9.3
//   3584 -> 3584 (13 MB)     4.6 / 4.8, 5.3 / 5.2, 5.7 / 5.5, 6.4 / 6.2; 64 rows 8.5 / 7.9
// The forms that stage x have 24 to 48 KB of weights on their way a CU, read a fragment of x from LDS for every tile or two, and wait at a
// barrier a slice.  Not for 64 rows in one block: 32.5 where staging takes 30.4 (3584 -> 37888), and with eight waves that share slices of x in
// LDS 30.6; and not for 16-bit weights, twice the bytes for the same products: 4096 -> 28672 39.3 against 37.9 at 32 rows.
#include "linear_slices.h"

namespace mi355 {
namespace {

enum { SL_STORE = 0, SL_SILU_MUL = 1, SL_PARTIAL = 2 };

template <typename T, int MT, int TP, int EPI>
__global__ __launch_bounds__(256, 1) void linear_slices_kernel(LinearSlices a) {
  constexpr int P = EPI == SL_SILU_MUL ? 2 : 1;             // tiles that one wave finishes together
  static_assert(TP % P == 0, "gate and up tiles of a column block share a workgroup");
  __shared__ __attribute__((aligned(16))) f32x4 red[TP][3][MT][64];
  typedef unsigned int vec __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, h = lane >> 4;
  const int tile0 = blockIdx.x * TP, m0 = blockIdx.z * a.block_rows, M = min(a.M - m0, a.block_rows);
  // units of 128 columns of this workgroup's K group, then of this wave: dealt as evenly as they go, one at least
  int u0, u1;
  {
    const int units = a.K >> 7, gy = gridDim.y, ub = units / gy, ur = units % gy, g = blockIdx.y;
    const int p0 = g * ub + min(g, ur), n = ub + (g < ur ? 1 : 0), each = n >> 2, rest = n & 3;
    u0 = p0 + wave * each + min(wave, rest);
    u1 = u0 + each + (wave < rest ? 1 : 0);
  }
  const int steps = (u1 - u0) * 2;                          // of 64 columns: a 1 KB block of every tile
  // weight blocks are ordered [unit][tile][2]
  const char* wb = static_cast<const char*>(a.w) + (static_cast<int64_t>(u0) * a.tiles + tile0) * 2048;
  const int64_t unit_bytes = static_cast<int64_t>(a.tiles) * 2048;
  const int last = a.tiles - 1 - tile0;                     // tiles past the matrix: the last one again, never stored
  const char* xb = reinterpret_cast<const char*>(a.x + static_cast<int64_t>(m0) * a.x_stride) + static_cast<int64_t>(u0) * 256;
  uint32_t xo[MT];                                          // (the rows of a block lie within 4 GB: linear_tiled_launch)
#pragma unroll
  for (int m = 0; m < MT; ++m) xo[m] = static_cast<uint32_t>(min(16 * m + c, M - 1)) * static_cast<uint32_t>(a.x_stride) * 2u + 16u * h;
  vec w[2][TP], xf[2][2 * MT];
  f32x4 acc[TP][MT];
#pragma unroll
  for (int t = 0; t < TP; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Step s of the weights and of x; past the last step, which nobody uses, 16 bytes of the last one for every lane: no branch around a
  // load, it would make the compiler wait for all that are out.
  auto w_at = [&](int s) {
    const int l = min(s, steps - 1);
    return wb + (l >> 1) * unit_bytes + (l & 1) * 1024 + (s < steps ? lane * 16 : 0);
  };
  auto load_x = [&](vec (&to)[2 * MT], int s) {
    const char* p = xb + static_cast<int64_t>(min(s, steps - 1)) * 128;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int m = 0; m < MT; ++m) to[k * MT + m] = MI355_LD(vec, a.x, p + k * 64 + (s < steps ? xo[m] : 0u));
  };
  load_x(xf[0], 0);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const char* p = w_at(j);
#pragma unroll
    for (int t = 0; t < TP; ++t) w[j][t] = MI355_LDNT(vec, a.w, p + min(t, last) * 2048);
  }
  __builtin_amdgcn_sched_barrier(0);
  for (int s0 = 0; s0 < steps; s0 += 2) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      load_x(xf[j ^ 1], s0 + j + 1);
      const char* p = w_at(s0 + j + 2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < TP; ++t) {
        const vec v = w[j][t];
        const uint4 f[2] = {make_uint4(T::fp8x2(v.x, false), T::fp8x2(v.x, true), T::fp8x2(v.y, false), T::fp8x2(v.y, true)),
                            make_uint4(T::fp8x2(v.z, false), T::fp8x2(v.z, true), T::fp8x2(v.w, false), T::fp8x2(v.w, true))};
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const vec b = xf[j][k * MT + m];
            acc[t][m] = T::mfma(f[k], make_uint4(b.x, b.y, b.z, b.w), acc[t][m]);
          }
        w[j][t] = MI355_LDNT(vec, a.w, p + min(t, last) * 2048);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  // ---- the parts of a tile: its wave has its own in registers, the others' come through LDS
#pragma unroll
  for (int t = 0; t < TP; ++t) {
    const int owner = (t / P) & 3;
    if (wave != owner)
#pragma unroll
      for (int m = 0; m < MT; ++m) red[t][(wave - owner - 1) & 3][m][lane] = acc[t][m];
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < TP; t += P) {
    if (wave != ((t / P) & 3) || t > last) continue;         // (a pair lies inside the matrix or outside: N % 32 == 0)
#pragma unroll
    for (int e = t; e < t + P; ++e) {
      const float4 sc = MI355_LD(float4, a.w_scale, a.w_scale + (tile0 + e) * 16 + 4 * h);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int owner = (t / P) & 3;                       // (added in the order of K, whichever wave it is)
        f32x4 v = owner == 0 ? acc[e][m] : red[e][(0 - owner - 1) & 3][m][lane];
#pragma unroll
        for (int k = 1; k < 4; ++k) v += k == owner ? acc[e][m] : red[e][(k - owner - 1) & 3][m][lane];
        acc[e][m] = v;
        acc[e][m][0] = pin_f32(acc[e][m][0] * sc.x), acc[e][m][1] = pin_f32(acc[e][m][1] * sc.y);
        acc[e][m][2] = pin_f32(acc[e][m][2] * sc.z), acc[e][m][3] = pin_f32(acc[e][m][3] * sc.w);
      }
    }
    const int n0 = (tile0 + t) * 16 + 4 * h;
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (EPI == SL_STORE && a.bias != nullptr) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n0 + r < a.N) bias[r] = T::to_f(MI355_LD(uint16_t, a.bias, a.bias + (n0 + r)));
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int mm = 16 * m + c;
      if (mm >= M) continue;
      const f32x4 v = acc[t][m];
      if constexpr (EPI == SL_SILU_MUL) {
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = silu_mul<T>(round_f<T>(v[r]), round_f<T>(acc[t + P - 1][m][r]));
        MI355_ST(uint2, a.y, a.y + static_cast<int64_t>(m0 + mm) * a.y_stride + ((tile0 + t) >> 1) * 16 + 4 * h,
                 make_uint2(T::pack2(o[0], o[1]), T::pack2(o[2], o[3])));
      } else if constexpr (EPI == SL_PARTIAL) {
        float* to = a.partial + (static_cast<int64_t>(blockIdx.y) * a.M + m0 + mm) * a.N + n0;
        if (n0 + 3 < a.N && (a.N & 3) == 0) {
          MI355_ST(float4, a.partial, to, make_float4(v[0], v[1], v[2], v[3]));
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n0 + r < a.N) MI355_ST(float, a.partial, to + r, v[r]);
        }
      } else {
        uint16_t* to = a.y + static_cast<int64_t>(m0 + mm) * a.y_stride + n0;
        if (n0 + 3 < a.N && (a.y_stride & 3) == 0 && (reinterpret_cast<uintptr_t>(a.y) & 7) == 0) {
          MI355_ST(uint2, a.y, to, make_uint2(T::pack2(v[0] + bias[0], v[1] + bias[1]), T::pack2(v[2] + bias[2], v[3] + bias[3])));
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n0 + r < a.N) MI355_ST(uint16_t, a.y, to + r, T::from_f(v[r] + bias[r]));
        }
      }
    }
  }
}

template <typename T, int MT, int TP>
bool launch_tp(int epi, dim3 grid, hipStream_t s, const LinearSlices& a) {
  if (epi == SL_STORE) { hipLaunchKernelGGL((linear_slices_kernel<T, MT, TP, SL_STORE>), grid, dim3(256), 0, s, a); return true; }
  if (epi == SL_PARTIAL) { hipLaunchKernelGGL((linear_slices_kernel<T, MT, TP, SL_PARTIAL>), grid, dim3(256), 0, s, a); return true; }
  if constexpr (TP % 2 == 0) {
    if (epi == SL_SILU_MUL) { hipLaunchKernelGGL((linear_slices_kernel<T, MT, TP, SL_SILU_MUL>), grid, dim3(256), 0, s, a); return true; }
  }
  return false;
}

template <typename T, int MT>
bool launch_mt(int tp, int epi, dim3 grid, hipStream_t s, const LinearSlices& a) {
  switch (tp) {
    case 4: return launch_tp<T, MT, 4>(epi, grid, s, a);
    case 6: return launch_tp<T, MT, 6>(epi, grid, s, a);
    case 7: return launch_tp<T, MT, 7>(epi, grid, s, a);
    case 8: return launch_tp<T, MT, 8>(epi, grid, s, a);
    case 9: return launch_tp<T, MT, 9>(epi, grid, s, a);
    case 10: return launch_tp<T, MT, 10>(epi, grid, s, a);
    default: return false;
  }
}

template <typename T>
bool launch_t(int tp, int epi, dim3 grid, hipStream_t s, const LinearSlices& a, int rows) {
  return rows <= 16 ? launch_mt<T, 1>(tp, epi, grid, s, a) : launch_mt<T, 2>(tp, epi, grid, s, a);
}

}  // namespace

bool launch_linear_slices(const LinearSlices& a, int tp, int k_groups, int epilogue, bool bf16, hipStream_t s) {
  const int rows = a.M < a.block_rows ? a.M : a.block_rows;
  const dim3 grid((a.tiles + tp - 1) / tp, k_groups, (a.M + a.block_rows - 1) / a.block_rows);
  return bf16 ? launch_t<BF16>(tp, epilogue, grid, s, a, rows) : launch_t<F16>(tp, epilogue, grid, s, a, rows);
}

}  // namespace mi355
