// Greedy sampling: per-row argmax over the vocabulary.
//
// One 1024-thread workgroup per row streams the row with 16-byte loads and
// keeps, per thread, a single 64-bit key
//     (order-preserving image of the logit) << 32  |  (0xFFFFFFFF - index)
// whose maximum is the largest logit and, among equal logits, the LOWEST index.
// NaN maps to the top key (torch.argmax treats NaN as the maximum) and -0.0 is
// folded onto +0.0.  Keys are max-reduced with wave64 shuffles and one LDS
// exchange.  HBM-bound single pass: vocab * sizeof(logit) bytes per row.
#include "common.h"

#include <type_traits>

namespace mi355 {

constexpr int kArgmaxThreads = 1024;

__device__ __forceinline__ unsigned long long argmax_key(float v, uint32_t idx) {
  uint32_t u = __float_as_uint(v);
  uint32_t k;
  if (v != v) {
    k = 0xFFFFFFFFu;
  } else {
    if (v == 0.0f) u = 0u;
    k = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  }
  return (static_cast<unsigned long long>(k) << 32) | static_cast<unsigned long long>(0xFFFFFFFFu - idx);
}

__device__ __forceinline__ unsigned long long umax64(unsigned long long a, unsigned long long b) {
  return a > b ? a : b;
}

// Inclusive scan of 64-bit values over the wave's lanes, 0 the neutral element, by data-parallel moves: shifts inside
// the rows of 16 lanes, then a row's last lane to the next row, then lane 31 to the upper half.  (Six moves of two
// registers; the same through the LDS crossbar took ten times as long, and a radix pick is little else.)
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned long long dpp64(unsigned long long v) {
  const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(v & 0xFFFFFFFFull), CTRL, ROWS, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(v >> 32), CTRL, ROWS, 0xF, false);
  return (static_cast<unsigned long long>(static_cast<uint32_t>(hi)) << 32) | static_cast<uint32_t>(lo);
}
template <typename F>
__device__ __forceinline__ unsigned long long wave_scan64(unsigned long long v, F&& op) {
  v = op(v, dpp64<0x111, 0xF>(v));              // row_shr 1, 2, 4, 8 (lanes shifted in from outside a row: 0)
  v = op(v, dpp64<0x112, 0xF>(v));
  v = op(v, dpp64<0x114, 0xF>(v));
  v = op(v, dpp64<0x118, 0xF>(v));
  v = op(v, dpp64<0x142, 0xA>(v));              // row_bcast 15 into rows 1 and 3
  v = op(v, dpp64<0x143, 0xC>(v));              // row_bcast 31 into rows 2 and 3
  return v;
}
__device__ __forceinline__ unsigned long long lane64(unsigned long long v, int lane) {      // a lane's value, for all (lane uniform)
  const uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(v & 0xFFFFFFFFull), lane);
  const uint32_t hi = __builtin_amdgcn_readlane(static_cast<int>(v >> 32), lane);
  return (static_cast<unsigned long long>(hi) << 32) | lo;
}
__device__ __forceinline__ unsigned long long wave_max64(unsigned long long v) {
  return lane64(wave_scan64(v, [](unsigned long long a, unsigned long long b) { return umax64(a, b); }), 63);
}
__device__ __forceinline__ float wave_maxf(float v) {                  // of numbers, no NaN among them
  auto step = [&](float o) { v = fmaxf(v, o); };
#define MI355_DPP_MAX(CTRL, ROWS) step(__int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, ROWS, 0xF, false)))
  MI355_DPP_MAX(0x111, 0xF), MI355_DPP_MAX(0x112, 0xF), MI355_DPP_MAX(0x114, 0xF), MI355_DPP_MAX(0x118, 0xF);
  MI355_DPP_MAX(0x142, 0xA), MI355_DPP_MAX(0x143, 0xC);
#undef MI355_DPP_MAX
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
__device__ __forceinline__ unsigned long long wave_sum64(unsigned long long v) {
  return lane64(wave_scan64(v, [](unsigned long long a, unsigned long long b) { return a + b; }), 63);
}

// KEYED: out[row] is the row's best key itself, with the index moved by index_offset (the
// position of this slice of the vocabulary in the whole one) and the top bit flipped so that
// SIGNED 64-bit max over the slices' keys orders them as the unsigned keys do.
template <int LDT, bool KEYED>
__global__ __launch_bounds__(kArgmaxThreads) void argmax_kernel(int64_t* __restrict__ out,
                                                                const void* __restrict__ logits,
                                                                int64_t stride, int vocab, uint32_t index_offset) {
  const int row = blockIdx.x;
  unsigned long long best = 0ull;
  if (LDT == MI355_F32) {
    const float* p = static_cast<const float*>(logits) + row * stride;
    const int nvec = vocab >> 2;
    for (int v = threadIdx.x; v < nvec; v += kArgmaxThreads) {
      const float4 f = MI355_LD(float4, logits, p + 4 * v);
      best = umax64(best, argmax_key(f.x, 4 * v));
      best = umax64(best, argmax_key(f.y, 4 * v + 1));
      best = umax64(best, argmax_key(f.z, 4 * v + 2));
      best = umax64(best, argmax_key(f.w, 4 * v + 3));
    }
    for (int i = (nvec << 2) + threadIdx.x; i < vocab; i += kArgmaxThreads)
      best = umax64(best, argmax_key(MI355_LD(float, logits, p + i), i));
  } else {
    const uint16_t* p = static_cast<const uint16_t*>(logits) + row * stride;
    const int nvec = vocab >> 3;
    for (int v = threadIdx.x; v < nvec; v += kArgmaxThreads) {
      float f[8];
      const uint4 raw = MI355_LD(uint4, logits, p + 8 * v);
      if (LDT == MI355_BF16) unpack8<BF16>(raw, f); else unpack8<F16>(raw, f);
#pragma unroll
      for (int j = 0; j < 8; ++j) best = umax64(best, argmax_key(f[j], 8 * v + j));
    }
    for (int i = (nvec << 3) + threadIdx.x; i < vocab; i += kArgmaxThreads) {
      const float f = (LDT == MI355_BF16) ? BF16::to_f(MI355_LD(uint16_t, logits, p + i)) : F16::to_f(MI355_LD(uint16_t, logits, p + i));
      best = umax64(best, argmax_key(f, i));
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) best = umax64(best, __shfl_xor(best, off, 64));
  __shared__ unsigned long long part[kArgmaxThreads / 64];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long b = part[0];
#pragma unroll
    for (int i = 1; i < kArgmaxThreads / 64; ++i) b = umax64(b, part[i]);
    const uint32_t idx = 0xFFFFFFFFu - static_cast<uint32_t>(b & 0xFFFFFFFFull);
    if (KEYED) {
      const unsigned long long moved = (b & 0xFFFFFFFF00000000ull) |
                                       static_cast<unsigned long long>(0xFFFFFFFFu - (idx + index_offset));
      MI355_ST(int64_t, out, out + row, static_cast<int64_t>(moved ^ 0x8000000000000000ull));
    } else {
      MI355_ST(int64_t, out, out + row, static_cast<int64_t>(idx));
    }
  }
}

// Chunked form for few rows: one 1024-thread workgroup per row draws its 8 MB alone (14 us for
// 32 x 128256); here a row is cut into `chunks` column ranges, every (row, chunk) workgroup
// max-reduces its range to one key and merges it into keys[row] with a 64-bit atomic max (order
// does not matter for a max: same result on every launch), and a second, tiny kernel turns the
// keys into token ids and clears them for the next launch.
template <int LDT>
__global__ __launch_bounds__(256) void argmax_chunk_kernel(unsigned long long* __restrict__ keys,
                                                            const void* __restrict__ logits, int64_t stride,
                                                            int vocab, int chunk_vecs) {
  constexpr int PER = LDT == MI355_F32 ? 4 : 8;     // elements per 16-byte vector
  const int row = blockIdx.x;
  const int nvec = vocab / PER;
  const int v0 = blockIdx.y * chunk_vecs, v1 = min(nvec, v0 + chunk_vecs);
  unsigned long long best = 0ull;
  if (LDT == MI355_F32) {
    const float* p = static_cast<const float*>(logits) + row * stride;
    for (int v = v0 + threadIdx.x; v < v1; v += 256) {
      const float4 f = MI355_LD(float4, logits, p + 4 * v);
      best = umax64(best, argmax_key(f.x, 4 * v));
      best = umax64(best, argmax_key(f.y, 4 * v + 1));
      best = umax64(best, argmax_key(f.z, 4 * v + 2));
      best = umax64(best, argmax_key(f.w, 4 * v + 3));
    }
    if (blockIdx.y == gridDim.y - 1)
      for (int i = nvec * PER + threadIdx.x; i < vocab; i += 256) best = umax64(best, argmax_key(MI355_LD(float, logits, p + i), i));
  } else {
    const uint16_t* p = static_cast<const uint16_t*>(logits) + row * stride;
    for (int v = v0 + threadIdx.x; v < v1; v += 256) {
      float f[8];
      const uint4 raw = MI355_LD(uint4, logits, p + 8 * v);
      if (LDT == MI355_BF16) unpack8<BF16>(raw, f); else unpack8<F16>(raw, f);
#pragma unroll
      for (int j = 0; j < 8; ++j) best = umax64(best, argmax_key(f[j], 8 * v + j));
    }
    if (blockIdx.y == gridDim.y - 1)
      for (int i = nvec * PER + threadIdx.x; i < vocab; i += 256) {
        const float f = (LDT == MI355_BF16) ? BF16::to_f(MI355_LD(uint16_t, logits, p + i)) : F16::to_f(MI355_LD(uint16_t, logits, p + i));
        best = umax64(best, argmax_key(f, i));
      }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) best = umax64(best, __shfl_xor(best, off, 64));
  __shared__ unsigned long long part[4];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    best = umax64(umax64(part[0], part[1]), umax64(part[2], part[3]));
    if (best != 0ull && MI355_OK_AT(keys, keys + row, 8)) atomicMax(&keys[row], best);   // 0 = an empty column range (every real key is > 0)
  }
}

__global__ void argmax_finish_kernel(int64_t* __restrict__ out, int64_t* __restrict__ out2,
                                     unsigned long long* __restrict__ keys, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const unsigned long long b = MI355_LD(unsigned long long, keys, keys + i);
  MI355_ST(unsigned long long, keys, keys + i, 0ull);                                   // re-armed for the next launch
  const int64_t idx = static_cast<int64_t>(0xFFFFFFFFu - static_cast<uint32_t>(b & 0xFFFFFFFFull));
  MI355_ST(int64_t, out, out + i, idx);
  if (out2 != nullptr) MI355_ST(int64_t, out2, out2 + i, idx);
}

__global__ void argmax_key_to_index_kernel(int64_t* __restrict__ out, const int64_t* __restrict__ keys, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    MI355_ST(int64_t, out, out + i, static_cast<int64_t>(0xFFFFFFFFu - static_cast<uint32_t>(static_cast<unsigned long long>(MI355_LD(int64_t, keys, keys + i)) & 0xFFFFFFFFull)));
}


// ---------------------------------------------------------------------------
// Random sampling: temperature, top-k (any k), top-p (over the whole vocabulary), one
// 1024-thread workgroup per row.  Every arithmetic step is plain fp32 in a fixed order
// (contraction off, polynomial exp and ln) or exact 64-bit integer arithmetic (the
// probability masses), so the result is a pure function of (logits, parameters, seed,
// step) and equals the CPU restatement bit for bit.  Three kinds of row:
//   temperature <= 0      the greedy token (one pass, the argmax key)
//   no cut (top_k <= 0 or >= vocab, and top_p >= 1)
//                         Gumbel-max over the whole row (one pass)
//   a cut                 the kept set as the published samplers define it (see sample_mass
//                         below), then Gumbel-max over the kept set.  Two ways to the set:
//     list  1. one pass keeps every thread's two largest logits (registers); two 8-bit radix
//              passes over those 2048 keys (LDS histogram) give the upper 16 bits of their
//              R-th largest (R = top_k, or 1024 without one): a threshold that at least R
//              logits reach and, for logits without a pathological layout, only a few more do
//           2. a second pass appends every logit >= it to an LDS list (<= 4096 entries) and,
//              for a row without top-k, adds up the mass of the whole row; a bitonic sort
//              orders the list (logit desc, index asc); running sums of the masses; the
//              prefix that reaches the top-p threshold is the kept set
//     exact    when top_k exceeds 1024, the list overflows (huge ties, adversarial layouts)
//              or the nucleus reaches past the list (flat distributions): radix selection
//              straight from the row, by count for top-k and by mass for top-p (sample_exact)
//   Both ways find the same set (integer masses: no rounding), so which one ran cannot be
//   told from the result.
// The streaming passes read the row (vocab * 2 or 4 bytes, L2-resident after the
// first) with 16-byte loads and touch LDS only for the few survivors.
// ---------------------------------------------------------------------------
constexpr int kSampleThreads = 1024;
constexpr int kSampleGuessRank = 1024;   // the LDS list is built around the row's 1024 largest logits (or its top_k, if smaller)
constexpr int kSampleCap = 4096;         // candidates at or above the threshold guess that LDS holds (4 a thread)

// The top-k that cuts, 0: none (off, or of the whole vocabulary).
__device__ __forceinline__ int active_top_k(int top_k, int vocab) { return top_k > 0 && top_k < vocab ? top_k : 0; }

// NaN sorts on top, as in argmax_key: a row that holds a NaN yields the index of its first NaN
// from greedy and from random sampling alike
__device__ __forceinline__ uint32_t sample_key(float v) {
  if (v != v) return 0xFFFFFFFFu;
  uint32_t u = (v == 0.0f) ? 0u : __float_as_uint(v);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float key_to_logit(uint32_t k) {
  if (k == 0u) return -INFINITY;
  const uint32_t u = (k & 0x80000000u) ? (k ^ 0x80000000u) : ~k;
  return __uint_as_float(u);
}

template <int LDT>
__device__ __forceinline__ float load_logit(const void* row, int i) {
  if (LDT == MI355_F32) return MI355_LD(float, row, static_cast<const float*>(row) + i);
  const uint16_t raw = MI355_LD(uint16_t, row, static_cast<const uint16_t*>(row) + i);
  return LDT == MI355_BF16 ? BF16::to_f(raw) : F16::to_f(raw);
}

__device__ __forceinline__ uint32_t mix32(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7FEB352Du;
  x ^= x >> 15;
  x *= 0x846CA68Bu;
  x ^= x >> 16;
  return x;
}

__device__ __forceinline__ uint32_t sample_hash(uint64_t seed, uint64_t step) {
  uint32_t h = mix32(static_cast<uint32_t>(seed) ^ 0x9E3779B9u);
  h = mix32(h ^ static_cast<uint32_t>(seed >> 32));
  h = mix32(h ^ static_cast<uint32_t>(step));
  return mix32(h ^ static_cast<uint32_t>(step >> 32) ^ 0x85EBCA6Bu);
}

__device__ __forceinline__ float sample_uniform(uint64_t seed, uint64_t step) {
  return (static_cast<float>(sample_hash(seed, step) >> 8) + 0.5f) * (1.0f / 16777216.0f);
}

// One uniform per (seed, step, token index), strictly inside (0, 1): 23 hash bits, centred, so
// that both 2^-24 and 1 - 2^-24 are exact fp32 values and log(u), log(-log(u)) stay finite.
__device__ __forceinline__ float sample_uniform_at(uint32_t row_hash, uint32_t index) {
  const uint32_t h = mix32(row_hash ^ mix32(index + 0x632BE5ABu));
  return (static_cast<float>(h >> 9) + 0.5f) * (1.0f / 8388608.0f);
}

// ln(x) for a positive normal x: x = 2^e * m with m in [sqrt(1/2), sqrt(2)), ln(m) = 2 atanh(s),
// s = (m - 1) / (m + 1), |s| < 0.172, odd series to s^9 (next term < 1e-9).  Every operation is one
// IEEE fp32 operation in the order written.
__device__ __forceinline__ float ln_det(float x) {
#pragma clang fp contract(off)
  const uint32_t bits = __float_as_uint(x);
  int e = static_cast<int>(bits >> 23) - 127;
  float m = __uint_as_float((bits & 0x007FFFFFu) | 0x3F800000u);
  if (m > 1.41421354f) {
    m = m * 0.5f;
    e += 1;
  }
  const float s = (m - 1.0f) / (m + 1.0f);
  const float s2 = s * s;
  float p = 0.11111111f;
  p = p * s2;
  p = p + 0.14285715f;
  p = p * s2;
  p = p + 0.2f;
  p = p * s2;
  p = p + 0.33333334f;
  p = p * s2;
  p = p + 1.0f;
  float r = s * p;
  r = r + r;
  const float base = static_cast<float>(e) * 0.69314718f;
  return base + r;
}

// exp(z), z <= 0: 2^n * poly(f) with y = z*log2(e), n = floor(y), f = y - n.
__device__ __forceinline__ float exp_det(float z) {
#pragma clang fp contract(off)
  const float y = z * 1.4426950408889634f;
  const float n = floorf(y);
  if (!(n >= -126.0f)) return 0.0f;
  const float f = y - n;
  const float c[8] = {1.0f, 0.6931471805599453f, 0.2402265069591007f, 0.05550410866482158f,
                      0.009618129107628477f, 0.0013333558146428443f, 0.00015403530393381608f,
                      1.5252733804059840e-05f};
  float r = c[7];
#pragma unroll
  for (int i = 6; i >= 0; --i) {
    r = r * f;
    r = r + c[i];
  }
  const int ni = static_cast<int>(n);
  const float scale = __uint_as_float(static_cast<uint32_t>(ni + 127) << 23);
  return r * scale;
}

// fn(logit, index) for every logit of the row, 16 bytes per lane per load.
template <int LDT, int UNROLL, typename F>
__device__ __forceinline__ void for_each_logit_in(const void* base, int vocab, int v0, int v1, bool tail, F&& fn);

template <int LDT, int UNROLL = 2, typename F>
__device__ __forceinline__ void for_each_logit(const void* base, int vocab, F&& fn) {
  for_each_logit_in<LDT, UNROLL>(base, vocab, 0, vocab, true, fn);
}

// The same over the 16-byte vectors [v0, v1) of the row, plus, if `tail`, the elements after the
// last whole vector.
template <int LDT, int UNROLL, typename F>
__device__ __forceinline__ void for_each_logit_in(const void* base, int vocab, int v0, int v1, bool tail, F&& fn) {
  constexpr int PER = LDT == MI355_F32 ? 4 : 8;
  const int nvec = min(v1, vocab / PER);
#pragma unroll UNROLL
  for (int v = v0 + threadIdx.x; v < nvec; v += static_cast<int>(blockDim.x)) {
    float f[8];
    if (LDT == MI355_F32) {
      const float4 q = MI355_LD(float4, base, static_cast<const float*>(base) + 4 * v);
      f[0] = q.x, f[1] = q.y, f[2] = q.z, f[3] = q.w;
    } else {
      const uint4 raw = MI355_LD(uint4, base, static_cast<const uint16_t*>(base) + 8 * v);
      if (LDT == MI355_BF16) unpack8<BF16>(raw, f); else unpack8<F16>(raw, f);
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) fn(f[j], v * PER + j);
  }
  if (tail)
    for (int i = vocab / PER * PER + threadIdx.x; i < vocab; i += static_cast<int>(blockDim.x)) fn(load_logit<LDT>(base, i), i);
}

// fn(f, n, i0) for every 16-byte vector of the row (n = 4 or 8 logits f[0, n) starting at index
// i0) and, one by one (n = 1), for the elements after the last whole vector.
template <int LDT, int UNROLL, typename F>
__device__ __forceinline__ void for_each_vector_in(const void* base, int vocab, int v0, int v1, bool tail, F&& fn);

template <int LDT, int UNROLL, typename F>
__device__ __forceinline__ void for_each_vector(const void* base, int vocab, F&& fn) {
  for_each_vector_in<LDT, UNROLL>(base, vocab, 0, vocab, true, fn);
}

// The same over the 16-byte vectors [v0, v1) of the row, plus, if `tail`, the elements after the last whole vector.
template <int LDT, int UNROLL, typename F>
__device__ __forceinline__ void for_each_vector_in(const void* base, int vocab, int v0, int v1, bool tail, F&& fn) {
  constexpr int PER = LDT == MI355_F32 ? 4 : 8;
  const int nvec = min(v1, vocab / PER);
#pragma unroll UNROLL
  for (int v = v0 + threadIdx.x; v < nvec; v += static_cast<int>(blockDim.x)) {
    float f[8];
    if (LDT == MI355_F32) {
      const float4 q = MI355_LD(float4, base, static_cast<const float*>(base) + 4 * v);
      f[0] = q.x, f[1] = q.y, f[2] = q.z, f[3] = q.w;
      f[4] = f[5] = f[6] = f[7] = 0.f;
    } else {
      const uint4 raw = MI355_LD(uint4, base, static_cast<const uint16_t*>(base) + 8 * v);
      if (LDT == MI355_BF16) unpack8<BF16>(raw, f); else unpack8<F16>(raw, f);
    }
    fn(f, PER, v * PER);
  }
  if (tail)
    for (int i = vocab / PER * PER + threadIdx.x; i < vocab; i += static_cast<int>(blockDim.x)) {
      float f[8] = {load_logit<LDT>(base, i), 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      fn(f, 1, i);
    }
}

// Workgroup-wide max of the 64-bit keys; thread 0 gets the result.
__device__ __forceinline__ unsigned long long sample_reduce_max(unsigned long long best, unsigned long long* part) {
  best = wave_max64(best);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0)
    for (unsigned i = 1; i < blockDim.x >> 6; ++i) best = umax64(best, part[i]);
  return best;
}

// In-place descending bitonic sort of a[0, P), P a power of two, by the whole workgroup.  The
// caller has made a[] visible (a barrier) before the call; a[] is visible to all after it.
// The array is cut into chunks of C >= 128 elements, one per wave: a compare-exchange step whose
// partner distance j is below C stays inside the chunks and needs no workgroup barrier (a wave's
// LDS operations execute in order), so of the 66 steps of a 2048-element sort only 10 end in one.
template <typename T>
__device__ __forceinline__ void bitonic_desc(T* a, int P) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int C = P >= 128 * (kSampleThreads / 64) ? P / (kSampleThreads / 64) : min(P, 128);
  const bool mine = wave * C < P;
  T* chunk = a + wave * C;
  bool local_dirty = false;
  for (int size = 2; size <= P; size <<= 1) {
    for (int j = size >> 1; j > 0; j >>= 1) {
      if (j < C) {
        if (mine) {
          for (int q = lane; q < (C >> 1); q += 64) {
            const int il = ((q & ~(j - 1)) << 1) | (q & (j - 1));
            const T x = chunk[il], y = chunk[il | j];
            const bool desc = ((wave * C + il) & size) == 0;
            if (desc ? (x < y) : (x > y)) {
              chunk[il] = y;
              chunk[il | j] = x;
            }
          }
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        local_dirty = true;
      } else {
        if (local_dirty) __syncthreads();
        local_dirty = false;
        for (int idx = threadIdx.x; idx < (P >> 1); idx += kSampleThreads) {
          const int i = ((idx & ~(j - 1)) << 1) | (idx & (j - 1));
          const int p = i | j;
          const T x = a[i], y = a[p];
          const bool desc = (i & size) == 0;
          if (desc ? (x < y) : (x > y)) {
            a[i] = y;
            a[p] = x;
          }
        }
        __syncthreads();
      }
    }
  }
  __syncthreads();
}

// By wave 0: the largest digit d of a 256-bin histogram with at least `need` entries in bins
// >= d, and how many of them bin d itself has to supply.  Lane l owns bins 4l .. 4l+3.
__device__ __forceinline__ void radix_pick(const int* hist, int need, int* digit, int* rem) {
  const int lane = threadIdx.x & 63;
  int h4[4], s = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    h4[j] = hist[4 * lane + j];
    s += h4[j];
  }
  int suf = s;                                   // entries in the bins of lanes >= this one
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int t = __shfl_down(suf, off, 64);
    if (lane + off < 64) suf += t;
  }
  int run = suf - s, best = -1, left = 0;
#pragma unroll
  for (int j = 3; j >= 0; --j) {
    if (best < 0 && run + h4[j] >= need) {
      best = 4 * lane + j;
      left = need - run;
    }
    run += h4[j];
  }
  unsigned long long packed = best >= 0 ? (static_cast<unsigned long long>(best + 1) << 32) | static_cast<uint32_t>(left) : 0ull;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) packed = umax64(packed, __shfl_xor(packed, off, 64));
  if (lane == 0) {
    *digit = packed != 0ull ? static_cast<int>(packed >> 32) - 1 : 0;
    *rem = packed != 0ull ? static_cast<int>(packed & 0xFFFFFFFFull) : need;
  }
}

// Whole-vocabulary draw for a row with neither top-k nor top-p: the Gumbel-max form of sampling
// from softmax(logits / t),
//     token = argmax_i ( logit_i / t  -  ln(-ln(u_i)) ),   u_i = sample_uniform_at(hash(seed, step), i),
// one pass over the row, no candidate set.  Scores are compared through the same order-preserving
// keys as everywhere else (a NaN logit wins, ties go to the lowest index).
template <int LDT>
__device__ __forceinline__ unsigned long long sample_full_vocab(const void* __restrict__ base, int vocab, int v0, int v1,
                                                                bool tail, float temp, uint64_t seed, uint64_t step) {
#pragma clang fp contract(off)
  const uint32_t row_hash = sample_hash(seed, step);
  unsigned long long best = 0ull;
  for_each_logit_in<LDT, 2>(base, vocab, v0, v1, tail, [&](float l, int i) {
    const float u = sample_uniform_at(row_hash, static_cast<uint32_t>(i));
    const float a = -ln_det(u);
    const float g = ln_det(a);
    const float scaled = l / temp;
    const float score = scaled - g;
    best = umax64(best, argmax_key(l != l ? l : score, static_cast<uint32_t>(i)));
  });
  return best;
}

// ---- the kept set of a row with a cut, as the published samplers define it (top-k, then top-p
// over what top-k kept, both on logits / temperature):
//   top-k (0 < k < vocab)  keeps every token whose logit reaches the k-th largest logit (ties at
//                          that value all stay)
//   top-p (p < 1)          orders the survivors by (logit descending, index ascending) and keeps
//                          the shortest prefix whose probability mass reaches p of theirs (the
//                          token that crosses p included; never fewer than one)
// Probability masses are exact integers: F_i = floor(exp_det((l_i - l_max) / t) * 2^40), sums in 64
// bits -- no rounding, so no dependence on the order of additions, and the two ways below of
// finding the prefix agree to the token.  The threshold is P = max(1, ceil(double(p) * double(Z))),
// Z the mass of the top-k survivors; the prefix ends at the first token whose running sum
// reaches P.  The token is then drawn from the kept set in the Gumbel-max form (see
// sample_full_vocab): argmax over the kept i of l_i / t - ln(-ln(u_i)), one uniform per (seed, step,
// token index) -- the same draw whichever way the set was found.
__device__ __forceinline__ unsigned long long sample_mass(float l, float l0, float temp) {
#pragma clang fp contract(off)
  float z = (l - l0) / temp;
  if (l == l0) z = 0.0f;                     // also the row maximum itself when it is +inf
  if (z != z) z = -INFINITY;
  const float w = exp_det(z);
  return static_cast<unsigned long long>(w * 1099511627776.0f);   // 2^40: exact scaling, then truncation
}

__device__ __forceinline__ unsigned long long mass_threshold(float top_p, unsigned long long total) {
  const double pz = static_cast<double>(top_p) * static_cast<double>(total);
  const unsigned long long P = static_cast<unsigned long long>(ceil(pz));
  return P < 1ull ? 1ull : P;
}

__device__ __forceinline__ unsigned long long gumbel_key(float l, uint32_t index, float temp, uint32_t row_hash) {
#pragma clang fp contract(off)
  const float u = sample_uniform_at(row_hash, index);
  const float a = -ln_det(u);
  const float g = ln_det(a);
  const float scaled = l / temp;
  const float score = scaled - g;
  return argmax_key(score, index);
}

// By wave 0: the largest digit d of a 256-bin histogram of 64-bit weights (counts or masses) whose
// bins >= d hold at least `need`, and how much of `need` bin d itself has to supply.  Lane l owns
// bins 4l .. 4l+3.  total_out (may be null): the sum of all bins.
__device__ __forceinline__ void radix_pick64(const unsigned long long* hist, unsigned long long need, int* digit,
                                             unsigned long long* rem, unsigned long long* bin_mass) {
  const int lane = threadIdx.x & 63;
  unsigned long long h4[4], s = 0ull;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    h4[j] = hist[4 * lane + j];
    s += h4[j];
  }
  unsigned long long suf = s;                   // weight in the bins of lanes >= this one
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const unsigned long long t = __shfl_down(suf, off, 64);
    if (lane + off < 64) suf += t;
  }
  unsigned long long run = suf - s;
  int best = -1;
  unsigned long long left = 0ull, mass = 0ull;
#pragma unroll
  for (int j = 3; j >= 0; --j) {
    if (best < 0 && run + h4[j] >= need) {
      best = 4 * lane + j;
      left = need - run;
      mass = h4[j];
    }
    run += h4[j];
  }
  // the highest lane with a hit wins
  const unsigned long long any = __ballot(best >= 0);
  const int win = any != 0ull ? 63 - __builtin_clzll(any) : -1;
  if (lane == (win < 0 ? 0 : win)) {
    *digit = win < 0 ? 0 : best;
    *rem = win < 0 ? need : left;
    *bin_mass = win < 0 ? 0ull : mass;
  }
}

// for_each_vector that stops early: `go()` is asked before every vector of a thread (the tail elements are
// visited only if it still says yes).
template <int LDT, typename G, typename F>
__device__ __forceinline__ void for_each_vector_while(const void* base, int vocab, G&& go, F&& fn) {
  constexpr int PER = LDT == MI355_F32 ? 4 : 8;
  const int nvec = vocab / PER;
  for (int v = threadIdx.x; v < nvec && go(); v += kSampleThreads) {
    float f[8];
    if (LDT == MI355_F32) {
      const float4 q = MI355_LD(float4, base, static_cast<const float*>(base) + 4 * v);
      f[0] = q.x, f[1] = q.y, f[2] = q.z, f[3] = q.w;
      f[4] = f[5] = f[6] = f[7] = 0.f;
    } else {
      const uint4 raw = MI355_LD(uint4, base, static_cast<const uint16_t*>(base) + 8 * v);
      if (LDT == MI355_BF16) unpack8<BF16>(raw, f); else unpack8<F16>(raw, f);
    }
    fn(f, PER, v * PER);
  }
  if (go())
    for (int i = nvec * PER + threadIdx.x; i < vocab; i += kSampleThreads) {
      float f[8] = {load_logit<LDT>(base, i), 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      fn(f, 1, i);
    }
}

// One 16-byte vector of the row as fp32 (4 logits of an fp32 row, 8 of a 16-bit one).
template <int LDT>
__device__ __forceinline__ void load_vector(const void* base, int v, float (&f)[8]) {
  if (LDT == MI355_F32) {
    const float4 q = MI355_LD(float4, base, static_cast<const float*>(base) + 4 * v);
    f[0] = q.x, f[1] = q.y, f[2] = q.z, f[3] = q.w;
    f[4] = f[5] = f[6] = f[7] = 0.f;
  } else {
    const uint4 raw = MI355_LD(uint4, base, static_cast<const uint16_t*>(base) + 8 * v);
    if (LDT == MI355_BF16) unpack8<BF16>(raw, f); else unpack8<F16>(raw, f);
  }
}

// fn(logit, index) for every kept token among the vectors [v_begin, v_end) of the row (and, if `tail`, the
// elements after the row's last whole vector): kept = key > Tp, or key == Tp and fewer than `take` tokens with
// that key precede it in index order (take == ~0: all of them stay).  ties_before: such tokens before v_begin.
// Waves own contiguous runs of vectors and a lane one vector of 64 consecutive ones at a time, so a token's rank
// among the ties is the count in the waves before + a scan over the lanes + its place inside the vector.
// eq_base: kSampleThreads / 64 + 1 ints of LDS.  All threads of the workgroup call it.
template <int LDT, typename F>
__device__ __forceinline__ void ordered_kept_pass(const void* base, int vocab, int v_begin, int v_end, bool tail,
                                                  uint32_t Tp, unsigned long long take,
                                                  unsigned long long ties_before, int* eq_base, F&& fn) {
  constexpr int PER = LDT == MI355_F32 ? 4 : 8;
  const int kWaves = blockDim.x >> 6;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  v_end = min(v_end, vocab / PER);
  v_begin = min(v_begin, v_end);
  const int VW = (((v_end - v_begin) + kWaves - 1) / kWaves + 63) / 64 * 64;
  const int w0 = min(v_end, v_begin + wave * VW), w1 = min(v_end, w0 + VW);
  const bool ranked = take != ~0ull;                 // the same in every thread
  unsigned long long eq_run = ties_before;
  if (ranked) {
    int c = 0;
    for (int vb = w0; vb < w1; vb += 64) {
      const int v = vb + lane;
      if (v < w1) {
        float f[8];
        load_vector<LDT>(base, v, f);
#pragma unroll
        for (int j = 0; j < PER; ++j) c += sample_key(f[j]) == Tp ? 1 : 0;
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
    if (lane == 0) eq_base[wave + 1] = c;
    __syncthreads();
    if (tid == 0) {
      eq_base[0] = 0;
      for (int w = 0; w < kWaves; ++w) eq_base[w + 1] += eq_base[w];
    }
    __syncthreads();
    eq_run += static_cast<unsigned long long>(eq_base[wave]);
  }
  for (int vb = w0; vb < w1; vb += 64) {
    const int v = vb + lane;
    const bool valid = v < w1;
    float f[8];
    if (valid) load_vector<LDT>(base, v, f);
    int excl = 0, total = 0;
    if (ranked) {
      int c = 0;
      if (valid) {
#pragma unroll
        for (int j = 0; j < PER; ++j) c += sample_key(f[j]) == Tp ? 1 : 0;
      }
      int incl = c;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int t = __shfl_up(incl, off, 64);
        if (lane >= off) incl += t;
      }
      excl = incl - c;
      total = __shfl(incl, 63, 64);
    }
    if (valid) {
      unsigned long long rank = eq_run + static_cast<unsigned long long>(excl);
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const uint32_t key = sample_key(f[j]);
        bool kept = key > Tp;
        if (key == Tp) {
          kept = !ranked || rank < take;
          ++rank;
        }
        if (kept) fn(f[j], v * PER + j);
      }
    }
    eq_run += static_cast<unsigned long long>(total);
  }
  if (tail && tid == 0) {                              // fewer than PER elements, after every vector of the row
    unsigned long long rank = ties_before + (ranked ? static_cast<unsigned long long>(eq_base[kWaves]) : 0ull);
    for (int i = vocab / PER * PER; i < vocab; ++i) {
      const float f = load_logit<LDT>(base, i);
      const uint32_t key = sample_key(f);
      bool kept = key > Tp;
      if (key == Tp) {
        kept = !ranked || rank < take;
        ++rank;
      }
      if (kept) fn(f, i);
    }
  }
}

// The exact kept set straight from the row, for rows whose candidates do not fit the LDS list
// (top_k beyond the list, a nucleus that reaches past it, huge ties): radix selection over the
// 32-bit order-preserving keys, 8 bits a pass -- by COUNT for the k-th largest key Tk, then by
// MASS among the keys >= Tk for the key Tp at which the running mass reaches the threshold -- and
// the number m of tokens with key == Tp that the prefix still takes (lowest indices first).  Then
// one ordered pass draws by Gumbel-max from {key > Tp} and the first m of {key == Tp}.
// Returns the winning 64-bit key in thread 0.
template <int LDT>
__device__ __forceinline__ unsigned long long sample_exact(const void* base, int vocab, int K1, float tp, float temp,
                                                           float l0, uint32_t row_hash, unsigned long long* hist,
                                                           unsigned long long* part, int* eq_base, int* shi,
                                                           unsigned long long* shl) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // A 16-bit logit widened to fp32 has zero low bits (bf16: 16, fp16: 13), so the low bits of its key
  // follow from the sign -- zeros for a key with the top bit set, ones otherwise: the last passes of
  // a selection over such a row have nothing to decide and are skipped (bf16: two of four, fp16: one).
  constexpr int kLastShift = LDT == MI355_BF16 ? 16 : LDT == MI355_F16 ? 8 : 0;
  auto low_bits = [](uint32_t prefix) -> uint32_t {
    return (prefix & 0x80000000u) ? 0u : ((1u << kLastShift) - 1u);
  };
  // One histogram add per run of equal digits inside a 16-byte vector (a row's neighbours mostly share
  // their leading key bits): the LDS serialises adds to one bin, and at the first level that is most of a pass.
  auto add_runs = [&](const uint32_t (&dig)[8], const unsigned long long (&val)[8], int nf) {
    unsigned long long acc = 0ull;
    uint32_t cur = 0xFFFFFFFFu;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j < nf && dig[j] != 0xFFFFFFFFu) {
        if (dig[j] != cur) {
          if (cur != 0xFFFFFFFFu && acc != 0ull) atomicAdd(&hist[cur], acc);
          cur = dig[j];
          acc = 0ull;
        }
        acc += val[j];
      }
    }
    if (cur != 0xFFFFFFFFu && acc != 0ull) atomicAdd(&hist[cur], acc);
  };
  uint32_t Tk = 0u;
  if (K1 > 0) {
    uint32_t prefix = 0u, mask = 0u;
    unsigned long long need = static_cast<unsigned long long>(K1);
    for (int shift = 24; shift >= kLastShift; shift -= 8) {
      if (tid < 256) hist[tid] = 0ull;
      __syncthreads();
      for_each_vector<LDT, 2>(base, vocab, [&](const float (&f)[8], int nf, int) {
        uint32_t dig[8];
        unsigned long long val[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t key = sample_key(f[j]);
          dig[j] = (key & mask) == prefix ? (key >> shift) & 255u : 0xFFFFFFFFu;
          val[j] = 1ull;
        }
        add_runs(dig, val, nf);
      });
      __syncthreads();
      if (wave == 0) radix_pick64(hist, need, &shi[0], &shl[0], &shl[1]);
      __syncthreads();
      prefix |= static_cast<uint32_t>(shi[0]) << shift;
      mask |= 255u << shift;
      need = shl[0];
      __syncthreads();
    }
    Tk = prefix | (kLastShift ? low_bits(prefix) : 0u);
  }
  uint32_t Tp = Tk;
  unsigned long long take = ~0ull;             // tokens with key == Tp that stay (all of them unless top-p cuts inside the tie)
  if (tp < 1.0f) {
    uint32_t prefix = 0u, mask = 0u;
    unsigned long long need = 0ull;
    for (int shift = 24; shift >= kLastShift; shift -= 8) {
      if (tid < 256) hist[tid] = 0ull;
      __syncthreads();
      for_each_vector<LDT, 2>(base, vocab, [&](const float (&f)[8], int nf, int) {
        uint32_t dig[8];
        unsigned long long val[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t key = sample_key(f[j]);
          const bool in = key >= Tk && (key & mask) == prefix;
          dig[j] = in ? (key >> shift) & 255u : 0xFFFFFFFFu;
          val[j] = in && j < nf ? sample_mass(f[j], l0, temp) : 0ull;
        }
        add_runs(dig, val, nf);
      });
      __syncthreads();
      if (shift == 24) {                         // the first level's histogram holds the whole mass Z of the top-k survivors
        if (wave == 0) {
          unsigned long long t = hist[4 * lane] + hist[4 * lane + 1] + hist[4 * lane + 2] + hist[4 * lane + 3];
          t = wave_sum64(t);
          if (lane == 0) shl[2] = mass_threshold(tp, t);
        }
        __syncthreads();
        need = shl[2];
      }
      if (wave == 0) radix_pick64(hist, need, &shi[0], &shl[0], &shl[1]);
      __syncthreads();
      prefix |= static_cast<uint32_t>(shi[0]) << shift;
      mask |= 255u << shift;
      need = shl[0];
      __syncthreads();
    }
    Tp = prefix | (kLastShift ? low_bits(prefix) : 0u);
    const unsigned long long Fp = sample_mass(key_to_logit(Tp), l0, temp);
    take = Fp > 0ull ? (need + Fp - 1ull) / Fp : ~0ull;     // need >= 1; every token with key == Tp weighs Fp
  }
  unsigned long long best = 0ull;
  ordered_kept_pass<LDT>(base, vocab, 0, vocab, true, Tp, take, 0ull, eq_base, [&](float f, int i) {
    best = umax64(best, gumbel_key(f, static_cast<uint32_t>(i), temp, row_hash));
  });
  __syncthreads();
  return sample_reduce_max(best, part);
}

// ---- the exact path spread over many workgroups.  One workgroup computes exp / ln for a whole row
// at the pace of ONE CU (a pass over 128256 logits with a mass per logit: ~35 us; a flat row needs
// five of them); the launch has up to 256.  A row of the cut launch that needs the exact path
// (and has a slot in the scratch below: the first kExactRows rows) therefore only raises its flag
// there, and a fixed sequence of follow-up launches does the radix selection with the row cut into
// column ranges, one workgroup each:
//   exact_hist_kernel(stage)   stage s < NL: counts per digit of key level s (top-k);
//                              s >= NL: masses per digit of level s - NL (top-p).  Every
//                              workgroup first replays the picks of the earlier stages from their
//                              finished histograms (a few hundred instructions, the same result
//                              in every workgroup), then adds its range's histogram to the row's
//                              with 64-bit integer atomics -- exact, so order-free
//   exact_final_kernel         Gumbel-max over {key > Tp} and the first `take` tokens with
//                              key == Tp (rank = such tokens in the ranges before, counted from
//                              the row, + ordered rank inside the range), merged into out[row]
//                              by a 64-bit atomic max
// NL = key levels that can differ for the logits' type (sample_exact: 2 / 3 / 4).  The launches
// always run (a fixed sequence replays from a HIP graph) and return at once for rows whose flag is
// down.  The scratch is one set per process and GPU: two sampling calls in flight on one GPU at
// the same time (different streams) would share it -- the engine samples on one stream.
constexpr int kExactRows = 256;
constexpr int kExactStages = 8;
static __device__ unsigned long long g_exact_hist[kExactRows][kExactStages][256];
static __device__ unsigned int g_exact_flag[kExactRows];
static __device__ float g_exact_l0[kExactRows];

template <int LDT>
struct ExactLevels {
  static constexpr int kLastShift = LDT == MI355_BF16 ? 16 : LDT == MI355_F16 ? 8 : 0;
  static constexpr int NL = (24 - kLastShift) / 8 + 1;
  __device__ static uint32_t low_bits(uint32_t prefix) { return (prefix & 0x80000000u) ? 0u : ((1u << kLastShift) - 1u); }
};

struct ExactState {
  uint32_t Tk, Tp;               // keys >= Tk survive top-k; Tp: the key at which the top-p prefix ends
  unsigned long long take;       // tokens with key == Tp that stay (~0: all)
  uint32_t prefix, mask;         // of the selection in progress (stage replay)
  unsigned long long need;
};

// radix_pick64 on bins already in registers, result in every lane.  Lane l holds bins 255 - 4l .. 252 - 4l in this order
// (the scan then runs from the highest bin down).
__device__ __forceinline__ void radix_pick_regs(const unsigned long long (&h4)[4], unsigned long long need, int& digit,
                                                unsigned long long& rem) {
  const int lane = threadIdx.x & 63;
  const unsigned long long s = h4[0] + h4[1] + h4[2] + h4[3];
  unsigned long long run = wave_scan64(s, [](unsigned long long a, unsigned long long b) { return a + b; }) - s, left = 0ull;
  int best = -1;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (best < 0 && run + h4[j] >= need) {
      best = 255 - 4 * lane - j;
      left = need - run;
    }
    run += h4[j];
  }
  const unsigned long long any = __ballot(best >= 0);
  const int win = any != 0ull ? __builtin_ctzll(any) : 0;          // the lowest lane with a hit holds the highest bin
  digit = any != 0ull ? __builtin_amdgcn_readlane(best, win) : 0;
  rem = any != 0ull ? lane64(left, win) : need;
}

// Where a row's histograms and its best key lie.  In a caller's workspace (all 64-bit; all but `last` zeroed ahead of
// the launches):
//   [rows] x 32 words: best at 0, the draw's key at 16 | histograms [rows][2 NL][256] | last [rows][chunks][256]
// (each on a line of its own: a line's atomics are served one after the other, and 60 workgroups of every row meet here)
// last: the masses of the last stage, for every column range by itself (how many tokens of the key at which the
// top-p prefix ends lie in the ranges ahead follows from them: such tokens weigh the same).
// best: the order-preserving key of the row's largest logit and its inverted index (a NaN on top); without a
// workspace, in the library's own scratch, for the rows whose flag is up (accessed plainly: it is in no bounds list).
#ifdef MI355_BOUNDS
#define MI355_SCRATCH_LD(ws, p) ((ws) != nullptr ? MI355_LD(unsigned long long, (ws), (p)) : *(p))
#else
#define MI355_SCRATCH_LD(ws, p) (*(p))
#endif
constexpr int kSampleWsHead = 32;
__host__ __device__ __forceinline__ int64_t sample_ws_words(int64_t rows, int stages) { return rows * (kSampleWsHead + stages * 256); }
constexpr int kSampleWsThreads = 256;                       // of a workgroup of this way
constexpr int kSampleWsGroups = 2048;                       // rows x chunks is below this plus the rows

struct ExactRow {
  unsigned long long* hists;     // null: the row takes no part
  float l0;                      // its largest logit
};
template <int LDT>
__device__ __forceinline__ ExactRow exact_row(unsigned long long* ws, int rows, int row, float temp, int K1, float tp);

// Replays the picks of stages [0, upto) of a row from its finished histograms [stage][256].  Wave 0 does it alone: it asks
// for every histogram it will need at once (one memory round trip instead of one per level, each followed by two
// workgroup barriers -- a third of the follow-up launches' time), picks level after level with shuffles only and
// hands the state to the workgroup through LDS (shl scratch).  upto = 2 * NL: the full state.
template <int LDT>
__device__ __forceinline__ ExactState exact_replay(const unsigned long long* ws, const unsigned long long* hists, int upto, int K1,
                                                   float tp, float temp, float l0, unsigned long long* shl) {
  using L = ExactLevels<LDT>;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  ExactState st;
  st.Tk = 0u, st.Tp = 0u, st.take = ~0ull, st.prefix = 0u, st.mask = 0u, st.need = 0ull;
  if (wave == 0) {
    unsigned long long h[2 * L::NL][4];
#pragma unroll
    for (int s_ = 0; s_ < 2 * L::NL; ++s_) {
      const bool on = s_ < upto && (s_ < L::NL ? K1 > 0 : tp < 1.0f);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        h[s_][j] = on ? MI355_SCRATCH_LD(ws, hists + s_ * 256 + 255 - 4 * lane - j) : 0ull;
      }
    }
    // top-k: stages 0 .. NL-1
    if (K1 > 0) {
      st.need = static_cast<unsigned long long>(K1);
#pragma unroll
      for (int lvl = 0; lvl < L::NL; ++lvl) {
        if (lvl < upto) {
          const int shift = 24 - 8 * lvl;
          int digit;
          radix_pick_regs(h[lvl], st.need, digit, st.need);
          st.prefix |= static_cast<uint32_t>(digit) << shift;
          st.mask |= 255u << shift;
        }
      }
      if (upto >= L::NL) st.Tk = st.prefix | (L::kLastShift ? L::low_bits(st.prefix) : 0u);
    }
    st.Tp = st.Tk;
    if (upto >= L::NL) {
      // top-p: stages NL .. 2 NL - 1, a fresh selection among the keys >= Tk
      st.prefix = 0u, st.mask = 0u, st.need = 0ull;
      if (tp < 1.0f) {
#pragma unroll
        for (int lvl = 0; lvl < L::NL; ++lvl) {
          if (L::NL + lvl < upto) {
            const int shift = 24 - 8 * lvl;
            if (lvl == 0)                          // the first level's histogram holds the whole mass Z of the top-k survivors
              st.need = mass_threshold(tp, wave_sum64(h[L::NL][0] + h[L::NL][1] + h[L::NL][2] + h[L::NL][3]));
            int digit;
            radix_pick_regs(h[L::NL + lvl], st.need, digit, st.need);
            st.prefix |= static_cast<uint32_t>(digit) << shift;
            st.mask |= 255u << shift;
          }
        }
        if (upto >= 2 * L::NL) {
          st.Tp = st.prefix | (L::kLastShift ? L::low_bits(st.prefix) : 0u);
          const unsigned long long Fp = sample_mass(key_to_logit(st.Tp), l0, temp);
          st.take = Fp > 0ull ? (st.need + Fp - 1ull) / Fp : ~0ull;
        }
      }
    }
    if (lane == 0) {
      shl[0] = st.take;
      shl[1] = st.need;
      shl[2] = (static_cast<unsigned long long>(st.Tk) << 32) | st.Tp;
      shl[3] = (static_cast<unsigned long long>(st.prefix) << 32) | st.mask;
    }
  }
  __syncthreads();
  st.take = shl[0];
  st.need = shl[1];
  st.Tk = static_cast<uint32_t>(shl[2] >> 32), st.Tp = static_cast<uint32_t>(shl[2] & 0xFFFFFFFFull);
  st.prefix = static_cast<uint32_t>(shl[3] >> 32), st.mask = static_cast<uint32_t>(shl[3] & 0xFFFFFFFFull);
  __syncthreads();
  return st;
}

// Rows that need one key only: greedy ones and draws with neither an active top-k (active_top_k) nor a top-p.
__device__ __forceinline__ bool sample_one_key(float temp, int K1, float top_p) {
  return !(temp > 0.0f) || (K1 == 0 && !(top_p < 1.0f));
}

template <int LDT>
__device__ __forceinline__ ExactRow exact_row(unsigned long long* ws, int rows, int row, float temp, int K1, float tp) {
  if (ws == nullptr) return ExactRow{row < kExactRows && g_exact_flag[row] != 0u ? &g_exact_hist[row][0][0] : nullptr,
                                     row < kExactRows ? g_exact_l0[row] : 0.f};
  const uint32_t key = static_cast<uint32_t>(MI355_LD(unsigned long long, ws, ws + static_cast<int64_t>(row) * kSampleWsHead) >> 32);
  if (sample_one_key(temp, K1, tp) || key == 0xFFFFFFFFu) return ExactRow{nullptr, 0.f};      // (a NaN: its index is known)
  return ExactRow{ws + static_cast<int64_t>(rows) * kSampleWsHead + static_cast<int64_t>(row) * 2 * ExactLevels<LDT>::NL * 256, key_to_logit(key)};
}

// Adds val(logit) of the logits [f, f + nf) with key >= from and the masked bits at prefix to their digits' bins: one
// LDS add per run of equal digits inside the vector (a row's neighbours mostly share their leading bits).
template <typename V>
__device__ __forceinline__ void hist_add(unsigned long long* hist, const float (&f)[8], int nf, uint32_t from, uint32_t mask,
                                         uint32_t prefix, int shift, V&& val) {
  unsigned long long acc = 0ull;
  uint32_t cur = 0xFFFFFFFFu;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if (j < nf) {
      const uint32_t key = sample_key(f[j]);
      if (key >= from && (key & mask) == prefix) {
        const uint32_t d = (key >> shift) & 255u;
        if (d != cur) {
          if (cur != 0xFFFFFFFFu && acc != 0ull) atomicAdd(&hist[cur], acc);
          cur = d;
          acc = 0ull;
        }
        acc += val(f[j]);
      }
    }
  }
  if (cur != 0xFFFFFFFFu && acc != 0ull) atomicAdd(&hist[cur], acc);
}

template <int LDT>
__global__ __launch_bounds__(kSampleThreads) void exact_hist_kernel(
    unsigned long long* __restrict__ ws, const void* __restrict__ logits, int64_t stride, int vocab,
    const float* __restrict__ temperature, const int32_t* __restrict__ top_k, const float* __restrict__ top_p, int chunk_vecs,
    int stage) {
  using L = ExactLevels<LDT>;
  const int row = ws != nullptr ? blockIdx.y : blockIdx.x, range = ws != nullptr ? blockIdx.x : blockIdx.y;
  const int rows = ws != nullptr ? gridDim.y : gridDim.x, ranges = ws != nullptr ? gridDim.x : gridDim.y;
  const int K1 = active_top_k(MI355_LD(int32_t, top_k, top_k + row), vocab);
  const float tp = MI355_LD(float, top_p, top_p + row), temp = MI355_LD(float, temperature, temperature + row);
  const ExactRow er = exact_row<LDT>(ws, rows, row, temp, K1, tp);
  if (er.hists == nullptr) return;
  const bool counting = stage < L::NL;
  if (counting ? K1 == 0 : !(tp < 1.0f)) return;       // this selection is off for the row
  const float l0 = er.l0;
  constexpr int kListed = 2048;
  __shared__ unsigned long long hist[256];
  __shared__ unsigned long long shl[4];
  __shared__ float list[kListed];
  __shared__ int listed;
  const int tid = threadIdx.x;
  const ExactState st = exact_replay<LDT>(ws, er.hists, stage, K1, tp, temp, l0, shl);
  const int shift = 24 - 8 * (counting ? stage : stage - L::NL);
  if (tid < 256) hist[tid] = 0ull;
  __syncthreads();
  const void* base = LDT == MI355_F32 ? static_cast<const void*>(static_cast<const float*>(logits) + row * stride)
                                      : static_cast<const void*>(static_cast<const uint16_t*>(logits) + row * stride);
  const int v0 = range * chunk_vecs, v1 = v0 + chunk_vecs;
  const bool tail = range == ranges - 1;
  if (counting || (st.Tk == 0u && st.mask == 0u)) {
    for_each_vector_in<LDT, 2>(base, vocab, v0, v1, tail, [&](const float (&f)[8], int nf, int) {
      hist_add(hist, f, nf, st.Tk, st.mask, st.prefix, shift,
               [&](float l) -> unsigned long long { return counting ? 1ull : sample_mass(l, l0, temp); });
    });
  } else {
    // few logits weigh here, but some of nearly every wave: collected first, so that full waves compute the masses
    if (tid == 0) listed = 0;
    __syncthreads();
    for_each_vector_in<LDT, 2>(base, vocab, v0, v1, tail, [&](const float (&f)[8], int nf, int) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (j < nf) {
          const uint32_t key = sample_key(f[j]);
          if (key >= st.Tk && (key & st.mask) == st.prefix) {
            const int at = atomicAdd(&listed, 1);
            if (at < kListed) list[at] = f[j];
            else atomicAdd(&hist[(key >> shift) & 255u], sample_mass(f[j], l0, temp));
          }
        }
      }
    });
    __syncthreads();
    const int n = min(listed, kListed);
    for (int i = tid; i < n; i += static_cast<int>(blockDim.x)) atomicAdd(&hist[(sample_key(list[i]) >> shift) & 255u], sample_mass(list[i], l0, temp));
  }
  __syncthreads();
  if (tid < 256) {
    unsigned long long* bin = er.hists + stage * 256 + tid;
    if (hist[tid] != 0ull && (ws == nullptr || MI355_OK_AT(ws, bin, 8))) atomicAdd(bin, hist[tid]);
    if (ws != nullptr && stage == 2 * L::NL - 1)
      MI355_ST(unsigned long long, ws,
               ws + sample_ws_words(rows, 2 * L::NL) + (static_cast<int64_t>(row) * ranges + range) * 256 + tid, hist[tid]);
  }
}

template <int LDT>
__global__ __launch_bounds__(kSampleThreads) void exact_final_kernel(
    int64_t* __restrict__ out, unsigned long long* __restrict__ ws, const void* __restrict__ logits, int64_t stride, int vocab,
    const float* __restrict__ temperature, const int32_t* __restrict__ top_k, const float* __restrict__ top_p,
    const int64_t* __restrict__ seeds, const int64_t* __restrict__ steps, int chunk_vecs) {
  using L = ExactLevels<LDT>;
  const int row = ws != nullptr ? blockIdx.y : blockIdx.x, range = ws != nullptr ? blockIdx.x : blockIdx.y;
  const int rows = ws != nullptr ? gridDim.y : gridDim.x, ranges = ws != nullptr ? gridDim.x : gridDim.y, tid = threadIdx.x;
  const int K1 = active_top_k(MI355_LD(int32_t, top_k, top_k + row), vocab);
  const float tp = MI355_LD(float, top_p, top_p + row), temp = MI355_LD(float, temperature, temperature + row);
  const ExactRow er = exact_row<LDT>(ws, rows, row, temp, K1, tp);
  if (er.hists == nullptr) return;
  const float l0 = er.l0;
  __shared__ unsigned long long shl[4];
  __shared__ int eq_base[kSampleThreads / 64 + 1];
  __shared__ unsigned long long part[kSampleThreads / 64];
  const ExactState st = exact_replay<LDT>(ws, er.hists, 2 * L::NL, K1, tp, temp, l0, shl);
  const void* base = LDT == MI355_F32 ? static_cast<const void*>(static_cast<const float*>(logits) + row * stride)
                                      : static_cast<const void*>(static_cast<const uint16_t*>(logits) + row * stride);
  // tokens at the cut key in the column ranges before this one (only when top-p cuts inside that tie): counted
  // here, from the row itself -- a compare per logit, cheaper than a launch of its own that would leave the counts
  unsigned long long before = 0ull;
  if (st.take != ~0ull && range != 0 && ws != nullptr) {
    const unsigned long long* last = ws + sample_ws_words(rows, 2 * L::NL) + static_cast<int64_t>(row) * ranges * 256 +
                                     ((st.Tp >> L::kLastShift) & 255u);
    unsigned long long m = tid < range ? MI355_LD(unsigned long long, ws, last + tid * 256) : 0ull;
    m = wave_sum64(m);                                   // (at most 64 ranges: the first wave has them all)
    if (tid == 0) part[0] = m / sample_mass(key_to_logit(st.Tp), l0, temp);
    __syncthreads();
    before = part[0];
    __syncthreads();
  } else if (st.take != ~0ull && range != 0) {
    unsigned int mine = 0u;
    for_each_vector_in<LDT, 2>(base, vocab, 0, range * chunk_vecs, false,
                               [&](const float (&f)[8], int nf, int) {
#pragma unroll
                                 for (int j = 0; j < 8; ++j) mine += (j < nf && sample_key(f[j]) == st.Tp) ? 1u : 0u;
                               });
    unsigned long long w = wave_sum64(static_cast<unsigned long long>(mine));
    if ((tid & 63) == 0) part[tid >> 6] = w;
    __syncthreads();
    for (unsigned q = 0; q < blockDim.x >> 6; ++q) before += part[q];
    __syncthreads();
  }
  const uint32_t row_hash = sample_hash(static_cast<uint64_t>(MI355_LD(int64_t, seeds, seeds + row)),
                                        static_cast<uint64_t>(MI355_LD(int64_t, steps, steps + row)));
  unsigned long long best = 0ull;
  ordered_kept_pass<LDT>(base, vocab, range * chunk_vecs, (range + 1) * chunk_vecs,
                         range == ranges - 1, st.Tp, st.take, before, eq_base, [&](float f, int i) {
                           best = umax64(best, gumbel_key(f, static_cast<uint32_t>(i), temp, row_hash));
                         });
  __syncthreads();
  best = sample_reduce_max(best, part);
  unsigned long long* key = ws != nullptr ? ws + static_cast<int64_t>(row) * kSampleWsHead + 16 : reinterpret_cast<unsigned long long*>(out) + row;
  if (tid == 0 && best != 0ull && MI355_OK_AT((ws != nullptr ? static_cast<const void*>(ws) : out), key, 8)) atomicMax(key, best);
}

// ---- the k most likely tokens of a row (the `logprobs` / `top_logprobs` lists of the completion routes): an
// exact selection, in (logit descending, index ascending) order, NaN on top as in the greedy pick.  One workgroup
// per row: radix selection by count over the order-preserving keys for the k-th largest key (the passes a 16-bit
// logit cannot differ in are skipped), then the ordered pass of the samplers' exact search, which keeps every key
// above it and the lowest-indexed of the tokens tied with it, then the k entries rank themselves.
constexpr int kTopkMax = 64;

template <int LDT>
__global__ __launch_bounds__(kSampleThreads) void topk_logits_kernel(
    int64_t* __restrict__ out_ids, float* __restrict__ out_vals, const void* __restrict__ logits, int64_t stride,
    int vocab, int k, const float* __restrict__ lse) {
  using L = ExactLevels<LDT>;
  const int row = blockIdx.x;
  const int tid = threadIdx.x, wave = tid >> 6;
  const void* base = LDT == MI355_F32 ? static_cast<const void*>(static_cast<const float*>(logits) + row * stride)
                                      : static_cast<const void*>(static_cast<const uint16_t*>(logits) + row * stride);
  __shared__ unsigned long long hist[256];
  __shared__ int shi[2];
  __shared__ unsigned long long shl[4];
  __shared__ int eq_base[kSampleThreads / 64 + 1];
  __shared__ unsigned long long found[kTopkMax];
  __shared__ int nfound;
  const int K = min(k, vocab);
  uint32_t prefix = 0u, mask = 0u;
  unsigned long long need = static_cast<unsigned long long>(K);
  for (int shift = 24; shift >= L::kLastShift; shift -= 8) {
    if (tid < 256) hist[tid] = 0ull;
    if (tid == 0) nfound = 0;
    __syncthreads();
    for_each_vector<LDT, 2>(base, vocab, [&](const float (&f)[8], int nf, int) {
      unsigned long long acc = 0ull;             // one LDS add per run of equal digits inside a vector
      uint32_t cur = 0xFFFFFFFFu;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (j < nf) {
          const uint32_t key = sample_key(f[j]);
          if ((key & mask) == prefix) {
            const uint32_t d = (key >> shift) & 255u;
            if (d != cur) {
              if (cur != 0xFFFFFFFFu) atomicAdd(&hist[cur], acc);
              cur = d;
              acc = 0ull;
            }
            acc += 1ull;
          }
        }
      }
      if (cur != 0xFFFFFFFFu) atomicAdd(&hist[cur], acc);
    });
    __syncthreads();
    if (wave == 0) radix_pick64(hist, need, &shi[0], &shl[0], &shl[1]);
    __syncthreads();
    prefix |= static_cast<uint32_t>(shi[0]) << shift;
    mask |= 255u << shift;
    need = shl[0];
    __syncthreads();
  }
  const uint32_t Tk = prefix | (L::kLastShift ? L::low_bits(prefix) : 0u);
  // every key above Tk and the first `need` tokens (by index) with key == Tk: K tokens in all
  ordered_kept_pass<LDT>(base, vocab, 0, vocab, true, Tk, need, 0ull, eq_base, [&](float f, int i) {
    const int at = atomicAdd(&nfound, 1);
    if (at < kTopkMax)
      found[at] = (static_cast<unsigned long long>(sample_key(f)) << 32) |
                  static_cast<unsigned long long>(0xFFFFFFFFu - static_cast<uint32_t>(i));
  });
  __syncthreads();
  const int n = min(nfound, K);
  const float sub = lse != nullptr ? MI355_LD(float, lse, lse + row) : 0.f;
  if (tid < k) {
    int64_t id = -1;
    float val = -INFINITY;
    int rank = tid;
    if (tid < n) {
      const unsigned long long mine = found[tid];
      rank = 0;
      for (int j = 0; j < n; ++j) rank += found[j] > mine ? 1 : 0;       // entries are distinct (their indices are)
      id = static_cast<int64_t>(0xFFFFFFFFu - static_cast<uint32_t>(mine & 0xFFFFFFFFull));
      val = load_logit<LDT>(base, static_cast<int>(id)) - sub;
    }
    MI355_ST(int64_t, out_ids, out_ids + (static_cast<int64_t>(row) * k + rank), id);
    MI355_ST(float, out_vals, out_vals + (static_cast<int64_t>(row) * k + rank), val);
  }
}

__global__ void sample_finish_kernel(int64_t* __restrict__ out, const float* __restrict__ temperature,
                                     const int32_t* __restrict__ top_k, const float* __restrict__ top_p, int n, int vocab) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const bool spread = i < kExactRows && g_exact_flag[i] != 0u;      // its token came from the follow-up launches, as a key
  if (spread) g_exact_flag[i] = 0u;
  if (!spread && !sample_one_key(MI355_LD(float, temperature, temperature + i), active_top_k(MI355_LD(int32_t, top_k, top_k + i), vocab),
                                 MI355_LD(float, top_p, top_p + i)))
    return;
  const unsigned long long b = static_cast<unsigned long long>(MI355_LD(int64_t, out, out + i));
  MI355_ST(int64_t, out, out + i, static_cast<int64_t>(0xFFFFFFFFu - static_cast<uint32_t>(b & 0xFFFFFFFFull)));
}

// One pass, one key: the row is cut into column ranges, every workgroup merges the best key of its
// range into *key (of `buffer`, cleared ahead) with a 64-bit atomic max -- order-free, so the same on every launch -- and a
// later launch turns it into the index.
template <int LDT>
__device__ __forceinline__ unsigned long long sample_one_key_best(const void* base, int vocab, bool greedy, float temp, uint64_t seed,
                                                                  uint64_t step, int range, int ranges, int chunk_vecs,
                                                                  unsigned long long* part) {
  const int v0 = range * chunk_vecs, v1 = v0 + chunk_vecs;
  const bool tail = range == ranges - 1;
  unsigned long long best = 0ull;
  if (greedy)
    for_each_logit_in<LDT, 2>(base, vocab, v0, v1, tail,
                              [&](float f, int i) { best = umax64(best, argmax_key(f, static_cast<uint32_t>(i))); });
  else
    best = sample_full_vocab<LDT>(base, vocab, v0, v1, tail, temp, seed, step);
  return sample_reduce_max(best, part);                   // (thread 0)
}
template <int LDT>
__device__ __forceinline__ void sample_one_key_pass(unsigned long long* key, const void* base, int vocab, bool greedy, float temp,
                                                    uint64_t seed, uint64_t step, int range, int ranges, int chunk_vecs,
                                                    unsigned long long* part, const void* buffer) {
  const unsigned long long best = sample_one_key_best<LDT>(base, vocab, greedy, temp, seed, step, range, ranges, chunk_vecs, part);
  if (threadIdx.x == 0 && best != 0ull && MI355_OK_AT(buffer, key, 8)) atomicMax(key, best);
}

// ---- sampling with a caller's workspace: every row spread over all of its workgroups.  The list way above keeps a row
// with a cut in one workgroup, at the pace of one CU (32 rows of 128256 bf16 logits: 83 us, most of it the masses);
// here the exact search, whose passes split over the launch, serves all of them, and nothing is shared between calls:
//   sample_clear    keys and histograms <- 0
//   sample_first    one-key rows: their pass.  Rows with a cut: the largest logit, and with top-k the first counts
//   exact_hist      the other stages; exact_final: the draw; sample_ws_finish: the keys turned into indices
// 32 rows of 128256 bf16 logits with a mix of cuts: 94 us a call, here 40 (the draws of uncut rows and the launches' gaps).
__global__ __launch_bounds__(256) void sample_clear_kernel(unsigned long long* __restrict__ ws, int64_t words) {
  const int64_t i = 2 * (blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x);
  if (i + 1 < words) MI355_ST(uint4, ws, ws + i, make_uint4(0u, 0u, 0u, 0u));
}

__global__ void sample_ws_finish_kernel(int64_t* __restrict__ out, const unsigned long long* __restrict__ ws,
                                        const float* __restrict__ temperature, const int32_t* __restrict__ top_k,
                                        const float* __restrict__ top_p, int n, int vocab) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const unsigned long long* head = ws + static_cast<int64_t>(i) * kSampleWsHead;
  unsigned long long b = MI355_LD(unsigned long long, ws, head + 16);
  const unsigned long long top = MI355_LD(unsigned long long, ws, head);
  if (!sample_one_key(MI355_LD(float, temperature, temperature + i), active_top_k(MI355_LD(int32_t, top_k, top_k + i), vocab),
                      MI355_LD(float, top_p, top_p + i)) &&
      static_cast<uint32_t>(top >> 32) == 0xFFFFFFFFu)
    b = top;                                               // a NaN: its first index
  MI355_ST(int64_t, out, out + i, static_cast<int64_t>(0xFFFFFFFFu - static_cast<uint32_t>(b & 0xFFFFFFFFull)));
}

template <int LDT>
__global__ __launch_bounds__(kSampleThreads) void sample_first_kernel(
    unsigned long long* __restrict__ ws, const void* __restrict__ logits, int64_t stride, int vocab,
    const float* __restrict__ temperature, const int32_t* __restrict__ top_k, const float* __restrict__ top_p,
    const int64_t* __restrict__ seeds, const int64_t* __restrict__ steps, int chunk_vecs) {
  const int row = blockIdx.y, tid = threadIdx.x;          // (a row's ranges one after the other: they land on different CUs)
  const void* base = LDT == MI355_F32 ? static_cast<const void*>(static_cast<const float*>(logits) + row * stride)
                                      : static_cast<const void*>(static_cast<const uint16_t*>(logits) + row * stride);
  __shared__ unsigned long long part[kSampleThreads / 64];
  __shared__ unsigned long long hist[256];
  const float temp = MI355_LD(float, temperature, temperature + row), tp = MI355_LD(float, top_p, top_p + row);
  const int K1 = active_top_k(MI355_LD(int32_t, top_k, top_k + row), vocab);
  if (sample_one_key(temp, K1, tp)) {
    sample_one_key_pass<LDT>(ws + static_cast<int64_t>(row) * kSampleWsHead + 16, base, vocab, !(temp > 0.0f), temp, static_cast<uint64_t>(MI355_LD(int64_t, seeds, seeds + row)),
                             static_cast<uint64_t>(MI355_LD(int64_t, steps, steps + row)), blockIdx.x,
                             gridDim.x, chunk_vecs, part, ws);
    return;
  }
  const bool counts = K1 > 0;
  if (counts) {
    if (tid < 256) hist[tid] = 0ull;
    __syncthreads();
  }
  const int v0 = blockIdx.x * chunk_vecs, v1 = v0 + chunk_vecs;
  unsigned long long best = 0ull;
  for_each_vector_in<LDT, 2>(base, vocab, v0, v1, blockIdx.x == gridDim.x - 1, [&](const float (&f)[8], int nf, int i0) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < nf) best = umax64(best, argmax_key(f[j], static_cast<uint32_t>(i0 + j)));
    if (counts) hist_add(hist, f, nf, 0u, 0u, 0u, 24, [](float) -> unsigned long long { return 1ull; });
  });
  best = sample_reduce_max(best, part);                  // (its barrier also ends the counting)
  unsigned long long* top = ws + static_cast<int64_t>(row) * kSampleWsHead;
  if (tid == 0 && best != 0ull && MI355_OK_AT(ws, top, 8)) atomicMax(top, best);
  if (counts && tid < 256 && hist[tid] != 0ull) {
    unsigned long long* bin = ws + static_cast<int64_t>(gridDim.y) * kSampleWsHead + static_cast<int64_t>(row) * 2 * ExactLevels<LDT>::NL * 256 + tid;
    if (MI355_OK_AT(ws, bin, 8)) atomicAdd(bin, hist[tid]);
  }
}

// ---- bf16 logits with a caller's workspace: two launches.  A 16-bit logit has 65536 values, so a row is its counts of
// them, and everything a cut needs -- the k-th largest key, the mass of what is left (a value's mass times its count), the
// key at which the nucleus ends -- follows from the counts without another look at the row:
//   sample_count   a workgroup per (row, part of its columns) counts its logits by key in LDS (65536 counters of 16 bits)
//                  and writes the lines of 32 counters that hold any, with a byte a line that says so
//   sample_draw    a workgroup per (row, range of its columns) adds up the counts of all parts (a few hundred lines: a trained
//                  model's logits have some thousand values), selects by prefix sums, and draws over its range; the row's last one to
//                  end turns the best key into the token.  A row's workgroups repeat the selection side by side instead of waiting
//                  for a launch that makes it once
// What bounds it: two chains of look-ups, scans and atomics.  32 rows of 128256 logits with a mix of cuts, us a call: 27.1 as three
// launches with two logarithms for every token that stays (count 6.5, pick 10, draw 12), here 19.5 (count 6.2, draw 13.3; 20.8 with eight
// keys a thread in the selection, of whose masses two threads in five had all); top-p alone 25.4 / 20.2, top-k of 50 alone 19.4 / 17.2, no
// cut 21.4 / 16.4; 64 rows 35.3 / 24.9, 4 rows 21.4 / 20.0 (by then the host's two launches).  Rows of three values (the cut's key holds a third of them) in such a mix: 48 rows 68 / 55.  The launch
// per eight key bits (exact_hist_kernel), seven for bf16, takes 40.
// fp16 keeps the passes: its rows have some ten thousand values, and the selection then takes them in several batches (16 rows
// with a top-p 38 us by passes, 48 by counts).
constexpr int kCountRows = 64;                              // rows up to which a row has four parts and more
constexpr int kCountParts = 16;                             // most parts of a row
constexpr int kSampleListed = 256;                          // tokens at the cut's key that a workgroup of the draw ranks from a list
constexpr int kSampleKept = 1024;                           // tokens that stay for sure that it lists ahead of their draw
constexpr int kCountLines = 2048;                           // lines of 32 counters, 64 bytes each
// parts of a row: 256 workgroups (a CU holds one: 128 KB of counters)
__host__ __device__ __forceinline__ int count_parts(int rows) { return rows >= 64 ? 4 : rows <= 16 ? kCountParts : 256 / rows; }
// workspace, in 64-bit words: [rows] x 32 (the draw's key at 0, workgroups done at 16) | flags [rows][parts][2048 bytes] |
// counters [rows][parts][65536] of 16 bits
__host__ __device__ __forceinline__ int64_t count_ws_words(int64_t rows) {
  return rows * (kSampleWsHead + count_parts(static_cast<int>(rows)) * static_cast<int64_t>(kCountLines / 8 + 16384));
}

// the order-preserving key of a bf16 logit (a NaN on top, -0 as +0), and back to the logit
__device__ __forceinline__ uint32_t key16(uint32_t raw) {
  if ((raw & 0x7FFFu) > 0x7F80u) return 0xFFFFu;
  if (raw == 0x8000u) raw = 0u;
  return raw & 0x8000u ? ~raw & 0xFFFFu : raw | 0x8000u;
}
__device__ __forceinline__ float key16_logit(uint32_t key) {
  return BF16::to_f(static_cast<uint16_t>(key & 0x8000u ? key ^ 0x8000u : ~key));
}

// The workgroups of a row on one XCD (every eighth block) or, where the rows do not come out even, on two: XCD x takes the x-th contiguous part
// of all (row, piece).  An L2 then holds the row and its counts (us in the grid's order / so: 32 rows with a mix of cuts 23.0 / 21.7, rows
// of nearly all values with a top-k of 50 25.7 / 18.8; 17 such rows 25.3 / 19.9, 27 of 32000 with a top-p 28.5 / 22.7).
__device__ __forceinline__ int2 row_and_piece(int rows, int pieces) {
  const int total = rows * pieces, xcd = blockIdx.x & 7;
  const int work = xcd * (total >> 3) + min(xcd, total & 7) + (static_cast<int>(blockIdx.x) >> 3);
  return make_int2(work / pieces, work % pieces);
}

__global__ __launch_bounds__(kSampleThreads) void sample_count_kernel(
    unsigned long long* __restrict__ ws, const uint16_t* __restrict__ logits, int64_t stride, int vocab,
    const float* __restrict__ temperature, const int32_t* __restrict__ top_k, const float* __restrict__ top_p, int rows, int parts, int part_vecs) {
  __shared__ __attribute__((aligned(16))) uint32_t counts[32768];      // two keys a word
  const int2 at = row_and_piece(rows, parts);
  const int row = at.x, part = at.y, tid = threadIdx.x, lane = tid & 63;
  if (part == 0 && tid == 0) {
    unsigned long long* head = ws + static_cast<int64_t>(row) * kSampleWsHead;
    MI355_ST(unsigned long long, ws, head, 0ull);
    MI355_ST(unsigned long long, ws, head + 16, 0ull);
  }
  if (sample_one_key(MI355_LD(float, temperature, temperature + row), active_top_k(MI355_LD(int32_t, top_k, top_k + row), vocab),
                     MI355_LD(float, top_p, top_p + row)))
    return;
  const uint16_t* base = logits + row * stride;
  const int v0 = part * part_vecs, v1 = min(v0 + part_vecs, vocab >> 3);
  auto add = [&](uint32_t k, uint32_t n) { atomicAdd(&counts[k >> 1], n << ((k & 1u) * 16u)); };      // (a part has fewer than 65536 logits)
  for (int i = tid; i < 8192; i += kSampleThreads) reinterpret_cast<uint4*>(counts)[i] = make_uint4(0u, 0u, 0u, 0u);
  __syncthreads();
  for (int v = v0 + tid; v < v1; v += kSampleThreads) {
    const uint4 raw = MI355_LD(uint4, logits, base + 8 * v);
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
    // Eight logits of one value (a masked row) go to their counter together with those of the lanes that have the same eight: at one
    // counter a wave's lanes take their turns (64 rows of 128256 with all but 50 logits masked, us a call: 56, here 32)
    if (w[0] == w[1] && w[0] == w[2] && w[0] == w[3] && w[0] >> 16 == (w[0] & 0xFFFFu)) {
      const uint32_t k = key16(w[0] & 0xFFFFu), first = __builtin_amdgcn_readfirstlane(k);
      const unsigned long long same = __ballot(k == first);
      if (k != first) add(k, 8u);
      else if (lane == __ffsll(same) - 1) add(k, 8u * static_cast<uint32_t>(__popcll(same)));
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) add(key16(w[j] & 0xFFFFu), 1u), add(key16(w[j] >> 16), 1u);
    }
  }
  if (part == parts - 1)
    for (int i = (vocab & ~7) + tid; i < vocab; i += kSampleThreads) add(key16(MI355_LD(uint16_t, logits, base + i)), 1u);
  __syncthreads();
  uint8_t* flags = reinterpret_cast<uint8_t*>(ws + static_cast<int64_t>(rows) * kSampleWsHead) +
                   (static_cast<int64_t>(row) * parts + part) * kCountLines;
  unsigned long long* lines = ws + static_cast<int64_t>(rows) * (kSampleWsHead + parts * (kCountLines / 8)) +
                              (static_cast<int64_t>(row) * parts + part) * 16384;
#pragma unroll
  for (int j = 0; j < 8; ++j) {                                        // four lanes a line
    const int piece = tid + kSampleThreads * j;
    const uint4 c = reinterpret_cast<const uint4*>(counts)[piece];
    const unsigned long long any = __ballot((c.x | c.y | c.z | c.w) != 0u);
    const bool used = ((any >> (lane & ~3)) & 15ull) != 0ull;
    if (used) MI355_ST(uint4, ws, lines + 2 * piece, c);
    if ((lane & 3) == 0) MI355_ST(uint8_t, ws, flags + (piece >> 2), static_cast<uint8_t>(used));
  }
}

// Inclusive prefix sum over the workgroup (16 waves), and the whole sum.  scratch: 16 words; all threads call it.
__device__ __forceinline__ unsigned long long block_scan64(unsigned long long v, unsigned long long* scratch, unsigned long long& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = wave_scan64(v, [](unsigned long long a, unsigned long long b) { return a + b; });
  __syncthreads();                                                     // scratch may still be read from a previous call
  if (lane == 63) scratch[wave] = v;
  __syncthreads();
  unsigned long long before = 0ull;
  total = 0ull;
#pragma unroll
  for (int w = 0; w < kSampleThreads / 64; ++w) {
    const unsigned long long s = scratch[w];
    if (w < wave) before += s;
    total += s;
  }
  return v + before;
}

// What the counts of a row with a cut say: its largest key, the key at which the cut falls, and how many tokens with that key stay
// (~0: all of them).  All 1024 threads call it, the result is the same in all.
struct CountedCut {
  uint32_t top, key;
  unsigned long long take;
};
struct CountedScratch {
  unsigned long long scratch[kSampleThreads / 64], found[2];
  uint16_t used[kCountLines];                                          // the row's lines that hold any, from the highest keys down
};
// The smallest number of tokens of mass F > 0 that hold `need` > 0, fewer than 2^22 (a row by counts has at most 2^20): the hardware's reciprocal is
// within 2^-23 of itself, so that the quotient less one is never above the answer, which is counted up to from there.  (The 64-bit
// division is some 150 instructions one after the other.)
__device__ __forceinline__ unsigned long long tokens_for(unsigned long long need, unsigned long long F) {
  unsigned long long t = static_cast<uint32_t>(static_cast<double>(need) * __builtin_amdgcn_rcp(static_cast<double>(F)));
  t = t > 0ull ? t - 1ull : 0ull;
  while (t * F < need) ++t;
  return t;
}

// ... from the lines in use on, an item being W of a line's keys to a thread
template <int W>
__device__ __forceinline__ CountedCut counted_cut_of(const unsigned long long* ws, const uint8_t* flags, const uint16_t* counters, int parts, int K1,
                                                     float temp, float tp, int lines, CountedScratch& sh) {
  static_assert(W == 4 || W == 8, "8 or 16 bytes of counters");
  constexpr int IL = 32 / W;                                           // items of a line
  typedef typename std::conditional<W == 8, uint4, uint2>::type Counts;
  unsigned long long(&scratch)[kSampleThreads / 64] = sh.scratch;
  unsigned long long(&found)[2] = sh.found;
  uint16_t(&used)[kCountLines] = sh.used;
  const int tid = threadIdx.x;
  const int items = lines * IL;
  // The counts of an item by key, highest first; its highest key.  No branch around a load: all of eight parts' are on
  // their way together (a line that a part has not written holds anything: its flag clears it).
  auto load_item = [&](int item, uint32_t (&n)[W]) -> uint32_t {
#pragma unroll
    for (int e = 0; e < W; ++e) n[e] = 0u;
    if (item >= items) return 0u;
    const int line = used[item / IL], piece = line * IL + IL - 1 - item % IL;
    for (int c0 = 0; c0 < parts; c0 += 8) {
      Counts q[8];
      uint32_t on[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int c = c0 + j < parts ? c0 + j : parts - 1;
        on[j] = MI355_LD(uint8_t, ws, flags + c * kCountLines + line);
        q[j] = MI355_LD(Counts, ws, counters + c * 65536 + piece * W);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t keep = on[j] != 0u && c0 + j < parts ? 0xFFFFFFFFu : 0u;
        uint32_t w[W / 2];
        if constexpr (W == 8) w[0] = q[j].w, w[1] = q[j].z, w[2] = q[j].y, w[3] = q[j].x;
        else w[0] = q[j].y, w[1] = q[j].x;
#pragma unroll
        for (int e = 0; e < W / 2; ++e) n[2 * e] += (w[e] & keep) >> 16, n[2 * e + 1] += w[e] & keep & 0xFFFFu;
      }
    }
    return static_cast<uint32_t>(piece * W + W - 1);
  };
  uint32_t n[W];
  uint32_t top = load_item(tid, n);
  auto sum_n = [&]() {
    uint32_t v = 0u;
#pragma unroll
    for (int e = 0; e < W; ++e) v += n[e];
    return static_cast<unsigned long long>(v);
  };
  // batches of 1024 items (one, unless the row has more than 8192 values' worth of lines)
  int here = 0;
  auto batch = [&](int b) {
    if (b != here) top = load_item(b * kSampleThreads + tid, n);
    here = b;
  };
  const int batches = (items + kSampleThreads - 1) / kSampleThreads;
  if (tid < 64) {                                                      // the row's largest key: of its first line's items
    uint32_t k = 0u;
#pragma unroll
    for (int e = W - 1; e >= 0; --e) k = n[e] != 0u ? top - e : k;
    const unsigned long long most = wave_max64(k);
    if (tid == 0) found[0] = most;
  }
  __syncthreads();
  const uint32_t best_key = static_cast<uint32_t>(found[0]);
  const float l0 = key16_logit(best_key);
  uint32_t Tk = 0u;                                                    // keys of 16 bits
  if (K1 > 0) {
    const unsigned long long need = static_cast<unsigned long long>(K1);
    unsigned long long carry = 0ull;
    for (int b = 0; b < batches; ++b) {
      batch(b);
      unsigned long long total, end = block_scan64(sum_n(), scratch, total) + carry, run = end - sum_n();
      if (run < need && need <= end) {
#pragma unroll
        for (int e = 0; e < W; ++e) {
          if (run < need && run + n[e] >= need) found[1] = top - e;
          run += n[e];
        }
      }
      carry += total;
      if (carry >= need) break;
    }
    __syncthreads();
    Tk = static_cast<uint32_t>(found[1]);
    __syncthreads();
  }
  uint32_t Tp = Tk;
  unsigned long long take = ~0ull;
  if (tp < 1.0f) {
    unsigned long long m[W], sum, Z = 0ull, end = 0ull;
    auto masses = [&]() {
      sum = 0ull;
#pragma unroll
      for (int e = 0; e < W; ++e) {
        m[e] = n[e] != 0u && top - e >= Tk ? n[e] * sample_mass(key16_logit(top - e), l0, temp) : 0ull;
        sum += m[e];
      }
    };
    int seen = 0;                                                      // batches that have any mass
    while (seen < batches) {
      batch(seen);
      masses();
      unsigned long long total;
      end = block_scan64(sum, scratch, total);
      Z += total;
      ++seen;
      // keys below a batch whose lowest has not half of the smallest mass have none
      if (seen < batches) {
        const uint32_t low = static_cast<uint32_t>(used[seen * (kSampleThreads / IL) - 1]) * 32u;
        if (low < Tk || exp_det((key16_logit(low) - l0) / temp) * 2199023255552.0f < 1.0f) break;      // 2^41
      }
    }
    const unsigned long long P = mass_threshold(tp, Z);
    unsigned long long carry = 0ull;
    for (int b = 0; b < seen; ++b) {
      unsigned long long total = Z;
      if (seen > 1) {
        batch(b);
        masses();
        end = block_scan64(sum, scratch, total);
      }
      unsigned long long run = carry + end - sum;
      if (run < P && P <= carry + end) {
#pragma unroll
        for (int e = 0; e < W; ++e) {
          if (run < P && run + m[e] >= P) found[0] = P - run, found[1] = top - e;
          run += m[e];
        }
      }
      carry += total;
      if (carry >= P) break;
    }
    __syncthreads();
    Tp = static_cast<uint32_t>(found[1]);
    const unsigned long long need = found[0], Fp = sample_mass(key16_logit(Tp), l0, temp);
    take = Fp > 0ull ? tokens_for(need, Fp) : ~0ull;
  }
  return {best_key, Tp, take};
}

__device__ __forceinline__ CountedCut counted_cut(const unsigned long long* ws, const uint8_t* flags, const uint16_t* counters, int parts, int K1,
                                                  float temp, float tp, CountedScratch& sh) {
  unsigned long long(&scratch)[kSampleThreads / 64] = sh.scratch;
  uint16_t(&used)[kCountLines] = sh.used;
  const int tid = threadIdx.x;
  // lines in use, highest first: thread t looks at lines 2047 - 2t and 2046 - 2t
  const int hi = kCountLines - 1 - 2 * tid;
  uint32_t mine = 0u;
#pragma unroll
  for (int c = 0; c < kCountParts; ++c) mine |= MI355_LD(uint16_t, ws, flags + (c < parts ? c : 0) * kCountLines + hi - 1);
  unsigned long long lines, at = block_scan64((mine >> 8 & 1u) + (mine & 1u), scratch, lines);
  if (mine & 1u) used[--at] = static_cast<uint16_t>(hi - 1);
  if (mine >> 8 & 1u) used[--at] = static_cast<uint16_t>(hi);
  __syncthreads();
  // (rows of up to 4096 keys' worth of lines, a model's some 3000: every thread has a part of them then, not two in five)
  const int n_lines = static_cast<int>(lines);
  return n_lines <= kSampleThreads / 8 ? counted_cut_of<4>(ws, flags, counters, parts, K1, temp, tp, n_lines, sh)
                                       : counted_cut_of<8>(ws, flags, counters, parts, K1, temp, tp, n_lines, sh);
}

// Gumbel-max over many tokens without two logarithms (of some forty operations) for each: as -ln u >= 1 - u, a score is at most
// l / t - ln(1 - u), which the hardware's logarithm gives to a margin, and as -ln u <= (1 - u) / u it is at least that plus ln u.  The
// scores themselves, bit for bit as everywhere, are formed only for tokens whose bound reaches the best lower bound that the wave
// has seen, one or two of a row.  (64 rows of 128256 logits without a cut, us a call: all scores 32.6, here 19.6.)
__device__ __forceinline__ uint32_t raw16_at(const uint4& raw, int j) {
  const uint32_t x = raw.x, y = raw.y, z = raw.z, w = raw.w, lo = j & 2 ? y + 0u : x + 0u, hi = j & 2 ? w + 0u : z + 0u;      // (values: a choice between members would need an address)
  return (j & 4 ? hi + 0u : lo + 0u) >> (j & 1 ? 16 : 0) & 0xFFFFu;
}
__device__ __forceinline__ unsigned long long gumbel_or_nan(float l, uint32_t i, float temp, uint32_t row_hash) {
  return l != l ? argmax_key(l, i) : gumbel_key(l, i, temp, row_hash);
}
// the best of the tokens `keep` (a bit each) of eight adjacent logits; inv: 1 / temp, low: the wave's lower bound so far.  All lanes of
// the wave call it.
__device__ __forceinline__ unsigned long long bounded_gumbel(const uint4 raw, int i0, uint32_t keep, float temp, float inv, uint32_t row_hash, float& low) {
  const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
  float top[8], most = -__builtin_inff(), far = 1.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float rest = 1.0f - sample_uniform_at(row_hash, static_cast<uint32_t>(i0 + j));        // (exact)
    const float l = BF16::to_f(static_cast<uint16_t>(j & 1 ? w[j >> 1] >> 16 : w[j >> 1] & 0xFFFFu));
    const float b = l * inv - 0.69314718f * __builtin_amdgcn_logf(rest);
    top[j] = keep >> j & 1u ? b : -__builtin_inff();
    if (top[j] > most) most = top[j], far = rest;
  }
  float at_least = most + 0.69314718f * __builtin_amdgcn_logf(1.0f - far) - (fabsf(most) * 2e-6f + 1e-3f);
  at_least = at_least != at_least ? -__builtin_inff() : at_least;      // (an infinity less its margin)
  low = fmaxf(low, wave_maxf(at_least));
  uint32_t near = 0u;
#pragma unroll
  for (int j = 0; j < 8; ++j) near |= top[j] + (fminf(fabsf(top[j]), 1e30f) * 2e-6f + 1e-3f) < low ? 0u : 1u << j;      // (a NaN stays)
  near &= keep;
  unsigned long long best = 0ull;
  if (low == -__builtin_inff()) {                                      // (uniform) logits of -inf have that score whatever their draw
    uint32_t none = 0u;
#pragma unroll
    for (int j = 0; j < 8; ++j) none |= (j & 1 ? w[j >> 1] >> 16 : w[j >> 1] & 0xFFFFu) == 0xFF80u ? 1u << j : 0u;
    none &= near;
    if (none != 0u) best = argmax_key(-__builtin_inff(), static_cast<uint32_t>(i0 + __ffs(none) - 1));
    near &= ~none;
  }
  while (near != 0u) {
    const int j = __ffs(near) - 1;
    near &= near - 1u;
    best = umax64(best, gumbel_or_nan(BF16::to_f(static_cast<uint16_t>(raw16_at(raw, j))), static_cast<uint32_t>(i0 + j), temp, row_hash));
  }
  return best;
}

// The best of the tokens at the cut's key in vectors [v0, v1) of a row (tail: and behind its last), of which those stay whose place among
// the row's, `before` of them ahead of v0, is below `take`: each wave counts its part, then draws by bounds what of it stays.  (A score
// for each: 48 rows of one value with a mix of cuts 56.7 us, here 42.0; with every one of them listed ahead 61.3.)
__device__ __forceinline__ unsigned long long ordered_ties(const uint16_t* logits, int vocab, int v0, int v1, bool tail, uint32_t Tp,
                                                           unsigned long long take, unsigned long long before, int* eq_base, float temp,
                                                           float inv, uint32_t row_hash, float low) {
  constexpr int W = kSampleThreads / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  v1 = max(v0, v1);
  const int VW = ((v1 - v0 + W - 1) / W + 63) / 64 * 64, w0 = min(v1, v0 + wave * VW), w1 = min(v1, w0 + VW);
  auto equal = [&](const uint4& raw, int v) {
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
    uint32_t m = 0u;
#pragma unroll
    for (int j = 0; j < 8; ++j) m |= key16(j & 1 ? w[j >> 1] >> 16 : w[j >> 1] & 0xFFFFu) == Tp ? 1u << j : 0u;
    return v < w1 ? m : 0u;
  };
  auto vector = [&](int v) { return MI355_LD(uint4, logits, logits + 8 * (v < w1 ? v : w1 - 1)); };
  unsigned long long mine = 0ull;
#pragma unroll 4
  for (int v = w0 + lane; v < w1; v += 64) mine += __popc(equal(vector(v), v));
  mine = wave_sum64(mine);
  if (lane == 0) eq_base[wave] = static_cast<int>(mine);
  __syncthreads();
  unsigned long long at = before, best = 0ull;
  for (int i = 0; i < wave; ++i) at += static_cast<unsigned long long>(eq_base[i]);
#pragma unroll 2
  for (int vb = w0; vb < w1 && at < take; vb += 64) {                  // (uniform)
    const int v = vb + lane;
    const uint4 raw = vector(v);
    uint32_t keep = equal(raw, v);
    const unsigned long long upto = at + wave_scan64(static_cast<unsigned long long>(__popc(keep)), [](unsigned long long a, unsigned long long b) { return a + b; });
    at = lane64(upto, 63);
    for (unsigned long long over = upto > take ? upto - take : 0ull; over != 0ull && keep != 0u; --over) keep &= ~(0x80000000u >> __clz(keep));
    best = umax64(best, bounded_gumbel(raw, 8 * v, keep, temp, inv, row_hash, low));
  }
  if (tail && tid == 0) {
    unsigned long long place = before;
    for (int i = 0; i < W; ++i) place += static_cast<unsigned long long>(eq_base[i]);
    for (int i = vocab & ~7; i < vocab; ++i) {
      const uint32_t x = MI355_LD(uint16_t, logits, logits + i);
      if (key16(x) == Tp && place++ < take) best = umax64(best, gumbel_key(BF16::to_f(static_cast<uint16_t>(x)), static_cast<uint32_t>(i), temp, row_hash));
    }
  }
  return best;
}

// Every workgroup of a row works the cut out for itself (they share the lines in the caches), draws over its range of the columns and
// merges its best key; the row's last one turns the key into the token.
__global__ __launch_bounds__(kSampleThreads) void sample_draw_kernel(
    int64_t* __restrict__ out, unsigned long long* __restrict__ ws, const uint16_t* __restrict__ logits, int64_t stride, int vocab,
    const float* __restrict__ temperature, const int32_t* __restrict__ top_k, const float* __restrict__ top_p,
    const int64_t* __restrict__ seeds, const int64_t* __restrict__ steps, int rows, int parts, int part_vecs, int ranges, int chunk_vecs) {
  __shared__ CountedScratch sh;
  __shared__ unsigned long long part_best[kSampleThreads / 64];
  __shared__ int eq_base[kSampleThreads / 64 + 1], ties[3], listed[kSampleListed];
  __shared__ uint2 kept[kSampleKept];                                  // index, logit
  const int2 place_of = row_and_piece(rows, ranges);
  const int row = place_of.x, range = place_of.y, tid = threadIdx.x, lane = tid & 63;
  const float temp = MI355_LD(float, temperature, temperature + row), tp = MI355_LD(float, top_p, top_p + row);
  const uint64_t seed = static_cast<uint64_t>(MI355_LD(int64_t, seeds, seeds + row)), step = static_cast<uint64_t>(MI355_LD(int64_t, steps, steps + row));
  const int K1 = active_top_k(MI355_LD(int32_t, top_k, top_k + row), vocab);
  const uint16_t* base = logits + row * stride;
  unsigned long long* head = ws + static_cast<int64_t>(row) * kSampleWsHead;
  const bool one = sample_one_key(temp, K1, tp);
  const int nvec = vocab >> 3, v0 = range * chunk_vecs, v1 = min(v0 + chunk_vecs, nvec);
  // this thread's first vector travels while the cut is worked out
  uint4 first = make_uint4(0u, 0u, 0u, 0u);
  if (nvec > 0) first = MI355_LD(uint4, logits, base + 8 * min(v0 + tid, nvec - 1));
  CountedCut cut = {0u, 0u, ~0ull};                                    // (a row without a cut: every key is above it)
  const uint8_t* flags = reinterpret_cast<const uint8_t*>(ws + static_cast<int64_t>(rows) * kSampleWsHead) + static_cast<int64_t>(row) * parts * kCountLines;
  const uint16_t* counters = reinterpret_cast<const uint16_t*>(ws + static_cast<int64_t>(rows) * (kSampleWsHead + parts * (kCountLines / 8))) +
                             static_cast<int64_t>(row) * parts * 65536;
  if (tid < 3) ties[tid] = 0;
  if (!one) cut = counted_cut(ws, flags, counters, parts, K1, temp, tp, sh);
  unsigned long long best = 0ull;
  if (!(temp > 0.0f) || cut.top == 0xFFFFu) {                          // greedy (and a NaN in a row with a cut: its first index)
    best = sample_one_key_best<MI355_BF16>(base, vocab, true, temp, seed, step, range, ranges, chunk_vecs, part_best);
  } else {
    const uint32_t Tp = cut.key;
    const unsigned long long take = cut.take;
    const uint32_t row_hash = sample_hash(seed, step);
    const float inv = 1.0f / temp;
    float low = -__builtin_inff();
    __syncthreads();
    // What stays for sure is listed and drawn behind the look, a token a lane, or, where most lanes have some, drawn as it lies; the cut
    // key's tokens are listed.  Most vectors hold neither: their largest logits say so (as 16-bit numbers; a cut below zero: the
    // smallest unsigned ones).
    auto place = [&](int& count, unsigned long long lanes) {           // of a lane in a list to which these lanes add
      const int leader = __ffsll(lanes) - 1;
      int at = 0;
      if (lane == leader) at = atomicAdd(&count, __popcll(lanes));
      return __builtin_amdgcn_readlane(at, leader) + __popcll(lanes & ((1ull << lane) - 1ull));
    };
    bool full = false;                                                 // the list has no room left: that it has not is all that counts then
    auto tie = [&](bool equal, int i) {
      const unsigned long long same = __ballot(equal);
      if (same == 0ull || full) return;
      const int at = place(ties[0], same);
      if (equal && at < kSampleListed) listed[at] = i;
      full = __builtin_amdgcn_readlane(at, 63 - __clzll(same)) >= kSampleListed;
    };
    typedef short s16x2 __attribute__((ext_vector_type(2)));
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    const bool above_zero = Tp > 0x8000u;
    const uint32_t Traw = above_zero ? Tp & 0x7FFFu : Tp == 0x8000u ? Tp : ~Tp & 0xFFFFu;
    auto reaches = [&](const uint4& q) {
      if (above_zero) {
        const s16x2 m = __builtin_elementwise_max(
            __builtin_elementwise_max(__builtin_bit_cast(s16x2, q.x), __builtin_bit_cast(s16x2, q.y)),
            __builtin_elementwise_max(__builtin_bit_cast(s16x2, q.z), __builtin_bit_cast(s16x2, q.w)));
        return max(static_cast<int>(m.x), static_cast<int>(m.y)) >= static_cast<int>(Traw);
      }
      const u16x2 m = __builtin_elementwise_min(
          __builtin_elementwise_min(__builtin_bit_cast(u16x2, q.x), __builtin_bit_cast(u16x2, q.y)),
          __builtin_elementwise_min(__builtin_bit_cast(u16x2, q.z), __builtin_bit_cast(u16x2, q.w)));
      return min(static_cast<uint32_t>(m.x), static_cast<uint32_t>(m.y)) <= Traw;
    };
    constexpr uint32_t kNone = 0xFF80FF80u;                            // -inf twice
    const bool none_stay = !one && Tp == (~kNone & 0xFFFFu) && inv > 0.0f;
    for (int vb = v0; vb < v1; vb += kSampleThreads) {
      const int v = vb + tid;
      const uint4 raw = vb == v0 ? first : MI355_LD(uint4, logits, base + 8 * min(v, nvec - 1));
      uint32_t stay = v < v1 ? 0xFFu : 0u;
      if (!one) {
        if (__ballot(stay != 0u && reaches(raw)) == 0ull) continue;
        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
        uint32_t equal = 0u, above = 0u;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t k = key16(j & 1 ? w[j >> 1] >> 16 : w[j >> 1] & 0xFFFFu);
          equal |= k == Tp ? 1u << j : 0u, above |= k > Tp ? 1u << j : 0u;
        }
        equal &= stay;
        if (take == ~0ull) above |= equal, equal = 0u;
        stay &= above;
        while (!full && __ballot(equal != 0u) != 0ull) {
          tie(equal != 0u, 8 * v + __ffs(equal) - 1);
          equal &= equal - 1u;
        }
        if (__popcll(__ballot(stay != 0u)) < 32) {
          for (unsigned long long some; (some = __ballot(stay != 0u)) != 0ull;) {
            const int at = place(ties[2], some), j = __ffs(stay) - 1;
            if (stay != 0u) {
              const uint32_t x = raw16_at(raw, j);
              if (at < kSampleKept) kept[at] = make_uint2(8 * v + j, x);
              else best = umax64(best, gumbel_key(BF16::to_f(static_cast<uint16_t>(x)), 8 * v + j, temp, row_hash));
              stay &= stay - 1u;
            }
          }
          continue;
        }
      }
      if (__ballot(stay != 0u) == 0ull) continue;
      // (a cut that falls on -inf: of masked vectors alone their first token, without a draw)
      if (none_stay && __ballot(stay != 0u && ((raw.x ^ kNone) | (raw.y ^ kNone) | (raw.z ^ kNone) | (raw.w ^ kNone)) != 0u) == 0ull) {
        if (stay != 0u) best = umax64(best, argmax_key(-__builtin_inff(), static_cast<uint32_t>(8 * v + __ffs(stay) - 1)));
        continue;
      }
      best = umax64(best, bounded_gumbel(raw, 8 * v, stay, temp, inv, row_hash, low));
    }
    if (range == ranges - 1)
      for (int ib = vocab & ~7; ib < vocab; ib += kSampleThreads) {  // (fewer than eight)
        const int i = ib + tid;
        const uint32_t raw = i < vocab ? MI355_LD(uint16_t, logits, base + i) : 0u, k = key16(raw);
        const bool equal = !one && i < vocab && k == Tp;
        if (i < vocab && (one || k > Tp || (equal && take == ~0ull)))
          best = umax64(best, gumbel_or_nan(BF16::to_f(static_cast<uint16_t>(raw)), static_cast<uint32_t>(i), temp, row_hash));
        tie(equal && take != ~0ull, i);
      }
    __syncthreads();
    for (int i = tid; i < min(ties[2], kSampleKept); i += kSampleThreads)
      best = umax64(best, gumbel_key(BF16::to_f(static_cast<uint16_t>(kept[i].y)), kept[i].x, temp, row_hash));
    const int num = ties[0];
    if (num > 0) {                                                     // ranked: behind those of the part ahead of this range
      // (the vectors past the row's last whole one belong to the last part, wherever this range begins)
      const int part = min(v0 / part_vecs, parts - 1);
      int c = 0;
      if (tid < part && MI355_LD(uint8_t, ws, flags + tid * kCountLines + (Tp >> 5)) != 0) c = MI355_LD(uint16_t, ws, counters + tid * 65536 + Tp);
#pragma unroll 4
      for (int v = part * part_vecs + tid; v < min(v0, nvec); v += kSampleThreads) {
        const uint4 raw = MI355_LD(uint4, logits, base + 8 * v);
        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) c += (key16(w[j] & 0xFFFFu) == Tp) + (key16(w[j] >> 16) == Tp);
      }
      if (c != 0) atomicAdd(&ties[1], c);
      __syncthreads();
      const unsigned long long before = static_cast<unsigned long long>(ties[1]);
      const float l = key16_logit(Tp);
      if (num <= kSampleListed) {
        if (tid < num) {
          const int i = listed[tid];
          unsigned long long rank = before;
          for (int j = 0; j < num; ++j) rank += listed[j] < i ? 1 : 0;
          if (rank < take) best = umax64(best, gumbel_key(l, static_cast<uint32_t>(i), temp, row_hash));
        }
      } else if (before < take) {
        best = umax64(best, ordered_ties(base, vocab, v0, v1, range == ranges - 1, Tp, take, before, eq_base, temp, inv, row_hash, low));
      }
      __syncthreads();
    }
    best = sample_reduce_max(best, part_best);
  }
  if (tid == 0 && MI355_OK_AT(ws, head, 8) && MI355_OK_AT(ws, head + 16, 8)) {
    // The key is in memory when its atomic's answer is here, so that the count that follows needs no fence (a fence of
    // the device writes a whole L2 back: 38 us for the 2000 workgroups of 32 rows, here 12).
    const unsigned long long was = atomicMax(head, best);
    asm volatile("s_waitcnt vmcnt(0)" ::"v"(was) : "memory");
    if (atomicAdd(head + 16, 1ull) == static_cast<unsigned long long>(ranges) - 1ull) {
      const unsigned long long b = atomicMax(head, 0ull);
      MI355_ST(int64_t, out, out + row, static_cast<int64_t>(0xFFFFFFFFu - static_cast<uint32_t>(b & 0xFFFFFFFFull)));
    }
  }
}

static int32_t launch_counted(const char* name, int64_t* out, unsigned long long* ws, const void* logits, int64_t stride, int rows, int vocab,
                              const float* temperature, const int32_t* top_k, const float* top_p, const int64_t* seeds, const int64_t* steps,
                              hipStream_t s) {
  const int nvec = vocab >> 3, parts = count_parts(rows), part_vecs = (nvec + parts - 1) / parts + (vocab < 8);
  // ranges of the draw: a workgroup a CU, but whole turns of 256 vectors each
  int ranges = 256 / rows < 64 ? 256 / rows : 64;
  const int chunk_vecs = ((nvec + ranges * 256 - 1) / (ranges * 256) + (nvec == 0)) * 256;
  ranges = nvec > chunk_vecs ? (nvec + chunk_vecs - 1) / chunk_vecs : 1;
  const uint16_t* p = static_cast<const uint16_t*>(logits);
  hipLaunchKernelGGL(sample_count_kernel, dim3(parts * rows), dim3(kSampleThreads), 0, s, ws, p, stride, vocab, temperature, top_k, top_p,
                     rows, parts, part_vecs);
  hipLaunchKernelGGL(sample_draw_kernel, dim3(ranges * rows), dim3(kSampleThreads), 0, s, out, ws, p, stride, vocab, temperature, top_k,
                     top_p, seeds, steps, rows, parts, part_vecs, ranges, chunk_vecs);
  return check_launch(name);
}

template <int LDT>
__global__ __launch_bounds__(kSampleThreads) void sample_kernel(
    int64_t* __restrict__ out, const void* __restrict__ logits, int64_t stride, int vocab,
    const float* __restrict__ temperature, const int32_t* __restrict__ top_k, const float* __restrict__ top_p,
    const int64_t* __restrict__ seeds, const int64_t* __restrict__ steps, int chunk_vecs, int spread_exact) {
#pragma clang fp contract(off)
  const int row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // a flag an aborted call may have left up must not reach this call's follow-up launches (the same thread
  // raises it again further down if this row needs them)
  if (blockIdx.y == 0 && tid == 0 && row < kExactRows) g_exact_flag[row] = 0u;
  const void* base = LDT == MI355_F32
                         ? static_cast<const void*>(static_cast<const float*>(logits) + row * stride)
                         : static_cast<const void*>(static_cast<const uint16_t*>(logits) + row * stride);
  __shared__ unsigned long long comp[kSampleCap];        // candidates: (key << 32) | inverted index
  __shared__ unsigned long long pre[kSampleCap];         // running sums of their masses
  __shared__ unsigned long long hist64[256];
  __shared__ unsigned long long part[kSampleThreads / 64];
  __shared__ unsigned long long shl[6];
  __shared__ int hist[256];
  __shared__ int eq_base[kSampleThreads / 64 + 1];
  __shared__ int sh[4];

  const float temp = MI355_LD(float, temperature, temperature + row);
  const int K1 = active_top_k(MI355_LD(int32_t, top_k, top_k + row), vocab);
  const float tp = MI355_LD(float, top_p, top_p + row);
  const uint64_t seed = static_cast<uint64_t>(MI355_LD(int64_t, seeds, seeds + row));
  const uint64_t step = static_cast<uint64_t>(MI355_LD(int64_t, steps, steps + row));
  const bool greedy = !(temp > 0.0f);
  if (sample_one_key(temp, K1, tp)) {
    sample_one_key_pass<LDT>(reinterpret_cast<unsigned long long*>(out) + row, base, vocab, greedy, temp, seed, step, blockIdx.y,
                             gridDim.y, chunk_vecs, part, out);
    return;
  }
  if (blockIdx.y != 0) return;
  const uint32_t row_hash = sample_hash(seed, step);

  // ---- 1. one pass: every thread's two largest logits (for the threshold guess), the row maximum,
  // and the first NaN (a row that holds a NaN yields its index, like the greedy pick)
  float f1 = -INFINITY, f2 = -INFINITY;
  uint32_t nan_at = 0xFFFFFFFFu;
  for_each_logit<LDT>(base, vocab, [&](float f, int i) {
    if (f != f) nan_at = min(nan_at, static_cast<uint32_t>(i));
    const float g = f != f ? -INFINITY : f;
    f2 = fmaxf(f2, fminf(f1, g));
    f1 = fmaxf(f1, g);
  });
  {
    // (max logit, inverted min NaN index) in one 64-bit max-reduction
    unsigned long long both = (static_cast<unsigned long long>(sample_key(f1)) << 32) |
                              static_cast<unsigned long long>(0xFFFFFFFFu - nan_at);
    unsigned long long hi = both & 0xFFFFFFFF00000000ull, lo = both & 0xFFFFFFFFull;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      hi = umax64(hi, __shfl_xor(hi, off, 64));
      lo = umax64(lo, __shfl_xor(lo, off, 64));
    }
    if (lane == 0) part[wave] = hi | lo;
    __syncthreads();
    if (tid == 0) {
      for (int w = 1; w < kSampleThreads / 64; ++w) {
        hi = umax64(hi, part[w] & 0xFFFFFFFF00000000ull);
        lo = umax64(lo, part[w] & 0xFFFFFFFFull);
      }
      shl[3] = hi | lo;
      sh[3] = 0;                                   // list length
      sh[2] = 0;                                   // ties beyond the k-th entry
      shl[4] = 0ull;                               // mass of the whole row
    }
    __syncthreads();
  }
  const uint32_t first_nan = 0xFFFFFFFFu - static_cast<uint32_t>(shl[3] & 0xFFFFFFFFull);
  if (first_nan != 0xFFFFFFFFu) {
    if (tid == 0) MI355_ST(int64_t, out, out + row, static_cast<int64_t>(first_nan));
    return;
  }
  const float l0 = key_to_logit(static_cast<uint32_t>(shl[3] >> 32));
  unsigned long long best = 0ull;
  bool exact = K1 > kSampleGuessRank;                   // the list is built around the 1024 largest: a deeper top-k goes straight to the exact path
  if (!exact) {
    // the R-th largest of the 2048 per-thread keys, to its upper 16 bits (two 8-bit radix passes in
    // LDS), lower bits clear: at least R logits of the row reach it (the 2048 keys are keys of distinct
    // logits; stand-ins of threads with fewer than two logits are -inf and can only lower the guess)
    const int Rk = min(K1 > 0 ? K1 : kSampleGuessRank, vocab);
    const uint32_t m1 = sample_key(f1), m2 = sample_key(f2);
    uint32_t guess = 0u;
    {
      int need = Rk;
      for (int shift = 24; shift >= 16; shift -= 8) {
        if (tid < 256) hist[tid] = 0;
        __syncthreads();
        const uint32_t above = shift == 24 ? 0u : 0xFF000000u;
        if ((m1 & above) == (guess & above)) atomicAdd(&hist[(m1 >> shift) & 255u], 1);
        if ((m2 & above) == (guess & above)) atomicAdd(&hist[(m2 >> shift) & 255u], 1);
        __syncthreads();
        if (wave == 0) radix_pick(hist, need, &sh[0], &sh[1]);
        __syncthreads();
        guess |= static_cast<uint32_t>(sh[0]) << shift;
        need = sh[1];
      }
    }
    // ---- 2. second pass: every logit at or above the guess goes to the LDS list (one counter bump per
    // lane and vector that has any); a row without top-k also adds up the mass of the WHOLE row, which
    // is what its top-p threshold is a share of
    const float guess_f = key_to_logit(guess);
    unsigned long long zsum = 0ull;
    // (a flat row overflows the list within its first tenth: the pass stops there, the row goes to the exact search)
    auto list_fits = [&]() { return *reinterpret_cast<volatile int*>(&sh[3]) <= kSampleCap; };
    for_each_vector_while<LDT>(base, vocab, list_fits, [&](const float (&f)[8], int nf, int i0) {
      int hits = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) hits += (j < nf && !(f[j] < guess_f)) ? 1 : 0;
      if (K1 == 0) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (j < nf) zsum += sample_mass(f[j], l0, temp);
      }
      if (hits != 0) {
        int pos = atomicAdd(&sh[3], hits);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (j < nf && !(f[j] < guess_f)) {
            if (pos < kSampleCap)
              comp[pos] = (static_cast<unsigned long long>(sample_key(f[j])) << 32) |
                          static_cast<unsigned long long>(0xFFFFFFFFu - static_cast<uint32_t>(i0 + j));
            ++pos;
          }
      }
    });
    if (K1 == 0) {
      zsum = wave_sum64(zsum);
      if (lane == 0) atomicAdd(&shl[4], zsum);
    }
    __syncthreads();
    const int n = sh[3];
    exact = n < Rk || n > kSampleCap;                   // (n < Rk cannot happen; kept as a guard)
    if (!exact) {
      int P2 = 64;
      while (P2 < n) P2 <<= 1;
      for (int i = n + tid; i < P2; i += kSampleThreads) comp[i] = 0ull;
      __syncthreads();
      bitonic_desc(comp, P2);
      // the top-k survivors: the first K1 entries and every later one tied with the K1-th
      int kk = n;
      if (K1 > 0) {
        const uint32_t key_k = static_cast<uint32_t>(comp[K1 - 1] >> 32);
        int extra = 0;
        for (int j = K1 + tid; j < n; j += kSampleThreads) extra += static_cast<uint32_t>(comp[j] >> 32) == key_k ? 1 : 0;
        if (extra != 0) atomicAdd(&sh[2], extra);
        __syncthreads();
        kk = K1 + sh[2];
      }
      // masses and their running sums (exact 64-bit integers): thread t owns entries 4t .. 4t+3
      unsigned long long m4[4], run = 0ull;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = 4 * tid + q;
        m4[q] = j < kk ? sample_mass(key_to_logit(static_cast<uint32_t>(comp[j] >> 32)), l0, temp) : 0ull;
        run += m4[q];
        m4[q] = run;
      }
      unsigned long long incl = run;                     // inclusive scan of the threads' totals inside the wave
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const unsigned long long t = __shfl_up(incl, off, 64);
        if (lane >= off) incl += t;
      }
      if (lane == 63) part[wave] = incl;
      __syncthreads();
      unsigned long long before = incl - run;
      for (int w = 0; w < wave; ++w) before += part[w];
#pragma unroll
      for (int q = 0; q < 4; ++q) pre[4 * tid + q] = before + m4[q];
      if (tid == 0) sh[0] = 0x7FFFFFFF;
      __syncthreads();
      int keep = kk;
      if (tp < 1.0f) {
        const unsigned long long Z = K1 > 0 ? pre[kk - 1] : shl[4];
        const unsigned long long P = mass_threshold(tp, Z);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int j = 4 * tid + q;
          if (j < kk && pre[j] >= P && (j == 0 || pre[j - 1] < P)) atomicMin(&sh[0], j + 1);
        }
        __syncthreads();
        keep = sh[0];
        exact = keep == 0x7FFFFFFF;                     // the nucleus reaches past the list: the exact path
      }
      if (!exact) {
        for (int j = tid; j < keep; j += kSampleThreads) {
          const uint32_t idx = 0xFFFFFFFFu - static_cast<uint32_t>(comp[j] & 0xFFFFFFFFull);
          best = umax64(best, gumbel_key(key_to_logit(static_cast<uint32_t>(comp[j] >> 32)), idx, temp, row_hash));
        }
        __syncthreads();
        best = sample_reduce_max(best, part);
      }
    }
  }
  if (exact && row < kExactRows && spread_exact) {
    // hand the row to the follow-up launches: clear its histograms, leave the row maximum, raise the flag
    __syncthreads();
    unsigned long long* h = &g_exact_hist[row][0][0];
    for (int j = tid; j < kExactStages * 256; j += kSampleThreads) h[j] = 0ull;
    if (tid == 0) {
      g_exact_l0[row] = l0;
      g_exact_flag[row] = 1u;
    }
    return;                                             // out[row] stays 0 (cleared by the launcher): the final launch max-merges into it
  }
  if (exact) {
    __syncthreads();
    best = sample_exact<LDT>(base, vocab, K1, tp, temp, l0, row_hash, hist64, part, eq_base, sh, shl);
  }
  if (tid == 0)
    MI355_ST(int64_t, out, out + row, static_cast<int64_t>(0xFFFFFFFFu - static_cast<uint32_t>(best & 0xFFFFFFFFull)));
}

}  // namespace mi355

namespace mi355 {
static int32_t check_logits(const char* name, const int64_t* out, const void* logits, int64_t logits_stride,
                            int32_t num_rows, int32_t vocab, int32_t logits_dtype, int64_t index_offset) {
  MI355_REQUIRE(out && logits, MI355_ERR_INVALID, "%s: null pointer", name);
  MI355_REQUIRE(num_rows >= 0 && vocab > 0, MI355_ERR_INVALID, "%s: num_rows/vocab out of range", name);
  MI355_REQUIRE(index_offset >= 0 && index_offset + vocab <= 0xFFFFFFFFll, MI355_ERR_INVALID,
                "%s: index_offset + vocab must fit 32 bits", name);
  MI355_REQUIRE(logits_dtype == MI355_BF16 || logits_dtype == MI355_F16 || logits_dtype == MI355_F32,
                MI355_ERR_UNSUPPORTED, "%s: logits dtype %d not supported", name, logits_dtype);
  const int per16 = logits_dtype == MI355_F32 ? 4 : 8;
  MI355_REQUIRE(logits_stride >= vocab && logits_stride % per16 == 0 && aligned16(logits),
                MI355_ERR_INVALID, "%s: logits rows must be 16-byte aligned (stride %lld)", name,
                (long long)logits_stride);
  return MI355_OK;
}

static int32_t argmax_entry(const char* name, int64_t* out, const void* logits, int64_t logits_stride,
                            int32_t num_rows, int32_t vocab, int32_t logits_dtype, bool keyed, int64_t index_offset,
                            void* stream) {
  const int32_t ok = check_logits(name, out, logits, logits_stride, num_rows, vocab, logits_dtype, index_offset);
  if (ok != MI355_OK || num_rows == 0) return ok;
  hipStream_t s = static_cast<hipStream_t>(stream);
  dim3 grid(num_rows), block(kArgmaxThreads);
  const uint32_t off = static_cast<uint32_t>(index_offset);
#define MI355_ARGMAX(LDT)                                                                                         \
  do {                                                                                                            \
    if (keyed)                                                                                                    \
      hipLaunchKernelGGL((argmax_kernel<LDT, true>), grid, block, 0, s, out, logits, logits_stride, vocab, off);  \
    else                                                                                                          \
      hipLaunchKernelGGL((argmax_kernel<LDT, false>), grid, block, 0, s, out, logits, logits_stride, vocab, off); \
  } while (0)
  if (logits_dtype == MI355_F32) MI355_ARGMAX(MI355_F32);
  else if (logits_dtype == MI355_BF16) MI355_ARGMAX(MI355_BF16);
  else MI355_ARGMAX(MI355_F16);
#undef MI355_ARGMAX
  return check_launch(name);
}
}  // namespace mi355

extern "C" int32_t mi355_argmax(int64_t* out_ids, const void* logits, int64_t logits_stride,
                                int32_t num_rows, int32_t vocab, int32_t logits_dtype, void* stream) {
  return mi355::argmax_entry("mi355_argmax", out_ids, logits, logits_stride, num_rows, vocab, logits_dtype, false, 0,
                             stream);
}

extern "C" int32_t mi355_argmax_chunked(int64_t* out_ids, int64_t* out_ids2, int64_t* keys, const void* logits,
                                        int64_t logits_stride, int32_t num_rows, int32_t vocab,
                                        int32_t logits_dtype, void* stream) {
  using namespace mi355;
  const char* name = "mi355_argmax_chunked";
  MI355_REQUIRE(out_ids && keys && logits, MI355_ERR_INVALID, "%s: null pointer", name);
  MI355_REQUIRE(num_rows >= 0 && vocab > 0, MI355_ERR_INVALID, "%s: num_rows/vocab out of range", name);
  MI355_REQUIRE(logits_dtype == MI355_BF16 || logits_dtype == MI355_F16 || logits_dtype == MI355_F32,
                MI355_ERR_UNSUPPORTED, "%s: logits dtype %d not supported", name, logits_dtype);
  const int per16 = logits_dtype == MI355_F32 ? 4 : 8;
  MI355_REQUIRE(logits_stride >= vocab && logits_stride % per16 == 0 && aligned16(logits) &&
                    (reinterpret_cast<uintptr_t>(keys) & 7u) == 0,
                MI355_ERR_INVALID, "%s: logits rows must be 16-byte aligned (stride %lld), keys 8-byte aligned", name,
                (long long)logits_stride);
  if (num_rows == 0) return MI355_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // enough workgroups to draw from every HBM channel (>= ~512), each with at least 2 vectors per thread
  const int nvec = vocab / per16;
  int chunks = (512 + num_rows - 1) / num_rows;
  chunks = chunks < 1 ? 1 : chunks > 64 ? 64 : chunks;
  while (chunks > 1 && (nvec + chunks - 1) / chunks < 512) --chunks;
  const int chunk_vecs = (nvec + chunks - 1) / chunks;
  dim3 grid(num_rows, chunks), block(256);
  auto* kp = reinterpret_cast<unsigned long long*>(keys);
  if (logits_dtype == MI355_F32)
    hipLaunchKernelGGL((argmax_chunk_kernel<MI355_F32>), grid, block, 0, s, kp, logits, logits_stride, vocab, chunk_vecs);
  else if (logits_dtype == MI355_BF16)
    hipLaunchKernelGGL((argmax_chunk_kernel<MI355_BF16>), grid, block, 0, s, kp, logits, logits_stride, vocab, chunk_vecs);
  else
    hipLaunchKernelGGL((argmax_chunk_kernel<MI355_F16>), grid, block, 0, s, kp, logits, logits_stride, vocab, chunk_vecs);
  int32_t rc = check_launch(name);
  if (rc != MI355_OK) return rc;
  hipLaunchKernelGGL(argmax_finish_kernel, dim3((num_rows + 255) / 256), dim3(256), 0, s, out_ids, out_ids2, kp, num_rows);
  return check_launch(name);
}

extern "C" int32_t mi355_argmax_shard_key(int64_t* out_keys, const void* logits, int64_t logits_stride,
                                          int32_t num_rows, int32_t vocab, int32_t logits_dtype,
                                          int64_t index_offset, void* stream) {
  return mi355::argmax_entry("mi355_argmax_shard_key", out_keys, logits, logits_stride, num_rows, vocab, logits_dtype,
                             true, index_offset, stream);
}

extern "C" int32_t mi355_argmax_key_to_index(int64_t* out_ids, const int64_t* keys, int32_t num_rows, void* stream) {
  using namespace mi355;
  const char* name = "mi355_argmax_key_to_index";
  MI355_REQUIRE(out_ids && keys, MI355_ERR_INVALID, "%s: null pointer", name);
  MI355_REQUIRE(num_rows >= 0, MI355_ERR_INVALID, "%s: num_rows out of range", name);
  if (num_rows == 0) return MI355_OK;
  hipLaunchKernelGGL(argmax_key_to_index_kernel, dim3((num_rows + 255) / 256), dim3(256), 0,
                     static_cast<hipStream_t>(stream), out_ids, keys, num_rows);
  return check_launch(name);
}

namespace mi355 {
static int32_t sample_entry(const char* name, int64_t* out_ids, const void* logits, int64_t logits_stride,
                            int32_t num_rows, int32_t vocab, int32_t logits_dtype, const float* temperature,
                            const int32_t* top_k, const float* top_p, const int64_t* seeds, const int64_t* steps,
                            int32_t cut_rows, void* stream) {
  MI355_REQUIRE(temperature && top_k && top_p && seeds && steps, MI355_ERR_INVALID, "%s: null pointer", name);
  const int32_t rc = check_logits(name, out_ids, logits, logits_stride, num_rows, vocab, logits_dtype, 0);
  if (rc != MI355_OK || num_rows == 0) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // one-key rows (greedy, no cut) are spread over `chunks` workgroups each so that few rows still
  // occupy every CU: their pass is ALU-bound (two logarithms and two divisions per logit)
  const int nvec = vocab / (logits_dtype == MI355_F32 ? 4 : 8);
  int chunks = (512 + num_rows - 1) / num_rows;
  chunks = chunks < 1 ? 1 : chunks > 64 ? 64 : chunks;
  while (chunks > 1 && (nvec + chunks - 1) / chunks < kSampleThreads) --chunks;
  const int chunk_vecs = (nvec + chunks - 1) / chunks;
  const hipError_t cleared = hipMemsetAsync(out_ids, 0, sizeof(int64_t) * num_rows, s);
  MI355_REQUIRE(cleared == hipSuccess, MI355_ERR_LAUNCH, "%s: clearing the keys failed: %s", name, hipGetErrorString(cleared));
  dim3 grid(num_rows, chunks), block(kSampleThreads);
  // rows that need the exact kept-set search are spread over the launch's column ranges by follow-up launches
  // (a fixed sequence: they return at once when no row raised its flag); MI355_SAMPLE_SPREAD=0 keeps such rows
  // in their one workgroup
  static const int spread = [] {
    const char* e = getenv("MI355_SAMPLE_SPREAD");
    return (e != nullptr && e[0] == '0') ? 0 : 1;
  }();
  const int spread_exact = spread && cut_rows != 0 && chunks > 1 ? 1 : 0;
#define MI355_SAMPLE_LAUNCH(LDT)                                                                                      \
  do {                                                                                                                \
    hipLaunchKernelGGL((sample_kernel<LDT>), grid, block, 0, s, out_ids, logits, logits_stride, vocab, temperature,    \
                       top_k, top_p, seeds, steps, chunk_vecs, spread_exact);                                          \
    if (spread_exact) {                                                                                               \
      dim3 xgrid(num_rows < kExactRows ? num_rows : kExactRows, chunks);                                              \
      for (int stage = 0; stage < 2 * ExactLevels<LDT>::NL; ++stage)                                                   \
        hipLaunchKernelGGL((exact_hist_kernel<LDT>), xgrid, block, 0, s, nullptr, logits, logits_stride, vocab, temperature, \
                           top_k, top_p, chunk_vecs, stage);                                                          \
      hipLaunchKernelGGL((exact_final_kernel<LDT>), xgrid, block, 0, s, out_ids, nullptr, logits, logits_stride, vocab,  \
                         temperature, top_k, top_p, seeds, steps, chunk_vecs);                                         \
    }                                                                                                                 \
  } while (0)
  if (logits_dtype == MI355_F32) MI355_SAMPLE_LAUNCH(MI355_F32);
  else if (logits_dtype == MI355_BF16) MI355_SAMPLE_LAUNCH(MI355_BF16);
  else MI355_SAMPLE_LAUNCH(MI355_F16);
#undef MI355_SAMPLE_LAUNCH
  const int32_t rc2 = check_launch(name);
  if (rc2 != MI355_OK) return rc2;
  hipLaunchKernelGGL(sample_finish_kernel, dim3((num_rows + 255) / 256), dim3(256), 0, s, out_ids, temperature, top_k,
                     top_p, num_rows, vocab);
  return check_launch(name);
}
}  // namespace mi355

extern "C" int32_t mi355_sample_topk_topp(int64_t* out_ids, const void* logits, int64_t logits_stride,
                                          int32_t num_rows, int32_t vocab, int32_t logits_dtype,
                                          const float* temperature, const int32_t* top_k, const float* top_p,
                                          const int64_t* seeds, const int64_t* steps, void* stream) {
  return mi355::sample_entry("mi355_sample_topk_topp", out_ids, logits, logits_stride, num_rows, vocab, logits_dtype,
                             temperature, top_k, top_p, seeds, steps, 1, stream);
}

extern "C" int32_t mi355_sample_topk_topp_hinted(int64_t* out_ids, const void* logits, int64_t logits_stride,
                                                 int32_t num_rows, int32_t vocab, int32_t logits_dtype,
                                                 const float* temperature, const int32_t* top_k, const float* top_p,
                                                 const int64_t* seeds, const int64_t* steps, int32_t cut_rows,
                                                 void* stream) {
  return mi355::sample_entry("mi355_sample_topk_topp_hinted", out_ids, logits, logits_stride, num_rows, vocab,
                             logits_dtype, temperature, top_k, top_p, seeds, steps, cut_rows, stream);
}

static int64_t sample_passes_bytes(int64_t rows, int stages) {
  return 8 * (mi355::sample_ws_words(rows, stages) + (mi355::kSampleWsGroups + rows) * 256);
}

extern "C" int64_t mi355_sample_workspace(int32_t num_rows, int32_t logits_dtype) {
  using namespace mi355;
  const int stages = 2 * (logits_dtype == MI355_F32 ? ExactLevels<MI355_F32>::NL : logits_dtype == MI355_BF16 ? ExactLevels<MI355_BF16>::NL
                                                                                                             : ExactLevels<MI355_F16>::NL);
  if (num_rows <= 0) return 0;
  const int64_t passes = sample_passes_bytes(num_rows, stages);
  return logits_dtype == MI355_BF16 && num_rows <= kCountRows && 8 * count_ws_words(num_rows) > passes ? 8 * count_ws_words(num_rows) : passes;
}

extern "C" int32_t mi355_sample_topk_topp_ws(int64_t* out_ids, const void* logits, int64_t logits_stride, int32_t num_rows,
                                             int32_t vocab, int32_t logits_dtype, const float* temperature,
                                             const int32_t* top_k, const float* top_p, const int64_t* seeds,
                                             const int64_t* steps, void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace mi355;
  const char* name = "mi355_sample_topk_topp_ws";
  MI355_REQUIRE(temperature && top_k && top_p && seeds && steps, MI355_ERR_INVALID, "%s: null pointer", name);
  const int32_t rc = check_logits(name, out_ids, logits, logits_stride, num_rows, vocab, logits_dtype, 0);
  if (rc != MI355_OK || num_rows == 0) return rc;
  const int stages = 2 * (logits_dtype == MI355_F32 ? ExactLevels<MI355_F32>::NL : logits_dtype == MI355_BF16 ? ExactLevels<MI355_BF16>::NL
                                                                                                             : ExactLevels<MI355_F16>::NL);
  const int64_t need = sample_passes_bytes(num_rows, stages);
  MI355_REQUIRE(workspace && workspace_bytes >= need && aligned16(workspace), MI355_ERR_INVALID,
                "%s: workspace of %lld bytes, %lld needed, 16-byte aligned", name, static_cast<long long>(workspace_bytes),
                static_cast<long long>(need));
  hipStream_t s = static_cast<hipStream_t>(stream);
  unsigned long long* ws = static_cast<unsigned long long*>(workspace);
  // whole turns of a workgroup's threads (a vector each), few enough that 2048 workgroups or 64 a row do
  const int nvec = vocab / (logits_dtype == MI355_F32 ? 4 : 8);
  int chunks = (kSampleWsGroups + num_rows - 1) / num_rows;
  chunks = chunks > 64 ? 64 : chunks;
  const int chunk_vecs = ((nvec + chunks * kSampleWsThreads - 1) / (chunks * kSampleWsThreads) + (nvec == 0)) * kSampleWsThreads;
  chunks = nvec > chunk_vecs ? (nvec + chunk_vecs - 1) / chunk_vecs : 1;
  // counts of 16 bits (a part of a row: at most 65535 logits), and room for them
  if (logits_dtype == MI355_BF16 && num_rows <= kCountRows && workspace_bytes >= 8 * count_ws_words(num_rows) &&
      ((vocab >> 3) / count_parts(num_rows) + 2) * 8 <= 65535) {
    return launch_counted(name, out_ids, ws, logits, logits_stride, num_rows, vocab, temperature, top_k, top_p, seeds, steps, s);
  }
  const int64_t words = sample_ws_words(num_rows, 2 * (logits_dtype == MI355_F32 ? 4 : logits_dtype == MI355_BF16 ? 2 : 3));
  const int64_t threads = words / 2;                     // (two words each)
  hipLaunchKernelGGL(sample_clear_kernel, dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0, s, ws, words);
  const dim3 grid(chunks, num_rows), block(kSampleWsThreads);
#define MI355_SAMPLE_LAUNCH(LDT)                                                                                      \
  do {                                                                                                                \
    hipLaunchKernelGGL((sample_first_kernel<LDT>), grid, block, 0, s, ws, logits, logits_stride, vocab,       \
                       temperature, top_k, top_p, seeds, steps, chunk_vecs);                                           \
    for (int stage = 1; stage < 2 * ExactLevels<LDT>::NL; ++stage)                                                     \
      hipLaunchKernelGGL((exact_hist_kernel<LDT>), grid, block, 0, s, ws, logits, logits_stride, vocab, temperature,   \
                         top_k, top_p, chunk_vecs, stage);                                                            \
    hipLaunchKernelGGL((exact_final_kernel<LDT>), grid, block, 0, s, out_ids, ws, logits, logits_stride, vocab,        \
                       temperature, top_k, top_p, seeds, steps, chunk_vecs);                                           \
  } while (0)
  if (logits_dtype == MI355_F32) MI355_SAMPLE_LAUNCH(MI355_F32);
  else if (logits_dtype == MI355_BF16) MI355_SAMPLE_LAUNCH(MI355_BF16);
  else MI355_SAMPLE_LAUNCH(MI355_F16);
#undef MI355_SAMPLE_LAUNCH
  hipLaunchKernelGGL(sample_ws_finish_kernel, dim3((num_rows + 255) / 256), dim3(256), 0, s, out_ids, ws, temperature, top_k, top_p,
                     num_rows, vocab);
  return check_launch(name);
}

extern "C" int32_t mi355_topk_logits(int64_t* out_ids, float* out_vals, const void* logits, int64_t logits_stride,
                                     int32_t num_rows, int32_t vocab, int32_t logits_dtype, int32_t k,
                                     const float* lse, void* stream) {
  using namespace mi355;
  const char* name = "mi355_topk_logits";
  MI355_REQUIRE(out_vals != nullptr, MI355_ERR_INVALID, "%s: null pointer", name);
  MI355_REQUIRE(k >= 1 && k <= kTopkMax, MI355_ERR_UNSUPPORTED, "%s: k %d outside [1, %d]", name, k, kTopkMax);
  const int32_t rc = check_logits(name, out_ids, logits, logits_stride, num_rows, vocab, logits_dtype, 0);
  if (rc != MI355_OK || num_rows == 0) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  dim3 grid(num_rows), block(kSampleThreads);
  if (logits_dtype == MI355_F32)
    hipLaunchKernelGGL((topk_logits_kernel<MI355_F32>), grid, block, 0, s, out_ids, out_vals, logits, logits_stride, vocab, k, lse);
  else if (logits_dtype == MI355_BF16)
    hipLaunchKernelGGL((topk_logits_kernel<MI355_BF16>), grid, block, 0, s, out_ids, out_vals, logits, logits_stride, vocab, k, lse);
  else
    hipLaunchKernelGGL((topk_logits_kernel<MI355_F16>), grid, block, 0, s, out_ids, out_vals, logits, logits_stride, vocab, k, lse);
  return check_launch(name);
}
