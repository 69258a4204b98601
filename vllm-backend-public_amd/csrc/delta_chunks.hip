// The gated delta rule with a decay per head for prompts of bf16 rows, by chunks of 64 rows on the bf16 matrix instruction.
//
// With G_t the log decay summed from the chunk's first row to row t and s_t = e^G_t / |k_t|, over a chunk
//     R = V - s (K S_0)                        K, Q, V: the rows as they are stored
//     (I + A) U = b R                          A_tj = b_t k_t k_j e^(G_t - G_j) / (|k_t| |k_j|)       (j < t)
//     O = e^G / (|q| sqrt(d)) (Q S_0) + P U    P_tj = q_t k_j e^(G_t - G_j) / (|q_t| sqrt(d) |k_j|)   (j <= t)
//     S_end = e^G_end S_0 + K^T (e^(G_end - G) / |k| U)
//   delta_chunk_prep   every chunk and head by itself: A and P from exact products of stored numbers, (I + A)^-1 by blocks of 16
//                      rows, and from it X = e^(G_end - G) / |k| (I + A)^-1 b and Z = P (I + A)^-1 b
//   delta_chunk_walk   per (sequence, head, 16 value channels): X R and Z R give the update and the output, so that a
//                      chunk costs the chain three products: K S, X R, K^T (X R)
// The state and all sums are fp32.  A stored number meets an fp32 one in three bf16 parts (exact products), two fp32 ones meet in
// the six products of parts that are not below 2^-26 of theirs.  Against 64 bits (relative, six seeds, 512 and 300 rows of 128 x 64):
// outputs 1.23e-7 where tiles of 16 rows had 1.57e-7, states 1.01e-7 and 1.23e-7; keys that are all alike but for a tenth 1.6e-7 and
// 2.0e-7, states 2.28e-7 and 2.04e-7.
// G is summed and subtracted in double and every exponent is <= 0.
//
// What bounds it: the walk's chain of products, exchanges through LDS and barriers (64 us of 97 with no loads in it), and its loads,
// 84 KB a chunk and workgroup through the vector caches; the preparation: see there.  Measured, 4 x 2048 rows, 16 heads of 128 x 128
// (8 keys): prep 47, walk 97 us, by tiles of 16 rows in fp32 117 and 204; one prompt of 2048 rows 18 and 61, before 171 together;
// 32 x 64 rows 69, before 102; 64 rows 20, before 20.  Half as many workgroups with two column blocks each 109 us, one
// wave for the chain and one for the outputs 119.
// The state never leaves its registers: an accumulator's rows (row 4 (lane / 16) + r, column lane % 16) of two blocks are a lane's
// eight numbers of a right operand if the left one's are dealt alike, which for stored rows is eight adjacent channels.
#include "common.h"
#include "delta_tiles.h"

namespace mi355 {

namespace {

constexpr int C = 64;                                     // rows of a chunk
constexpr int kTriBytes = 6 * 3 * 64 * 16;                // a lower triangular 64 x 64 in parts, six steps of 16 x 32
constexpr int kRows = 2 * C + 4;                          // factors of a chunk: R's, O's, the state's

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Two numbers -> their three bf16 parts, packed; all 24 bits of a number are in its parts.  The first two parts rounded: what is left
// out of a product of two fp32 numbers is below 2^-26 of it.
__device__ __forceinline__ void parts3(float x, float y, uint32_t& p0, uint32_t& p1, uint32_t& p2) {
  p0 = BF16::pack2(x, y);
  x -= __uint_as_float(p0 << 16), y -= __uint_as_float(p0 & 0xFFFF0000u);
  p1 = BF16::pack2(x, y);
  x -= __uint_as_float(p1 << 16), y -= __uint_as_float(p1 & 0xFFFF0000u);
  p2 = BF16::pack2(x, y);
}
// two blocks of an accumulator -> the three parts of a right operand
__device__ __forceinline__ void parts3(const f32x4& a, const f32x4& b, uint4 (&p)[3]) {
  parts3(a[0], a[1], p[0].x, p[1].x, p[2].x);
  parts3(a[2], a[3], p[0].y, p[1].y, p[2].y);
  parts3(b[0], b[1], p[0].z, p[1].z, p[2].z);
  parts3(b[2], b[3], p[0].w, p[1].w, p[2].w);
}

// Workspace, for every slot of a chunk: of each key head K, Q and K^T, of each head X and Z (in parts) and the factors of its rows, all as
// left operands lie in the lanes (rows of a projection are some power of two apart: read as they are by 16 rows they fall on few
// channels of the L2; the walk then took 119 us instead of 97).
struct Chunk {
  char *k, *x;                // K | Q | K^T of d * 128 bytes each, X | Z
  float* rows;
};
__host__ __device__ __forceinline__ int64_t chunk_bytes(int H, int G, int d) {
  return static_cast<int64_t>(H) * (2 * kTriBytes + kRows * 4) + static_cast<int64_t>(G) * 3 * d * C * 2;
}
__device__ __forceinline__ Chunk chunk_at(float* ws, int64_t slot, int h, int g, int H, int G, int d) {
  Chunk c;
  char* p = reinterpret_cast<char*>(ws) + slot * chunk_bytes(H, G, d);
  c.k = p + static_cast<int64_t>(g) * 3 * d * C * 2;
  p += static_cast<int64_t>(G) * 3 * d * C * 2;
  c.x = p + static_cast<int64_t>(h) * 2 * kTriBytes;
  c.rows = reinterpret_cast<float*>(p + static_cast<int64_t>(H) * 2 * kTriBytes) + h * kRows;
  return c;
}

// KD: key channels / 32.  A workgroup takes a chunk and up to two heads that share their key.  What bounds it: its loads and the writes
// (60 KB a head and chunk), and a chain of some 80 fp32 matrix instructions a head in the wave that has the inverse's first column.
template <int KD>
__global__ __launch_bounds__(256, 3) void delta_chunk_prep_kernel(DeltaTiles a, int per) {
  constexpr int D = 32 * KD, LK = D + 8, LT = C + 4;      // (row strides in LDS: 16 rows of 16 bytes on all banks)
  __shared__ __attribute__((aligned(16))) uint16_t Ks[C * LK];
  __shared__ __attribute__((aligned(16))) float As[C * LT], Ps[C * LT];
  __shared__ double G2[2][C];
  __shared__ float b2[2][C], rk[C], rq[C];
  // the waves' parts are uneven, and wave i of every workgroup shares a SIMD: they change places from workgroup to workgroup
  const uint32_t id = blockIdx.x + gridDim.x * blockIdx.y, turn = id + (id >> 3) + (id >> 5) + (id >> 8);
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(((tid >> 6) + turn) & 3);
  const int rep = a.H / a.G, sets = (rep + per - 1) / per, g = blockIdx.y / sets, set = blockIdx.y % sets;
  const int h0 = g * rep + per * set, heads = rep - per * set < per ? rep - per * set : per;
  // chunk slots: sequence s owns cu[s] / 64 + s onwards, one for each of its chunks (the ranges never overlap)
  const int slot = static_cast<int>(blockIdx.x);
  int s = -1, cs = 0, ce = 0;
  for (int base = 0; base < a.S; base += 64) {
    const int i = base + lane, j = i < a.S ? i : a.S - 1;
    const int c0 = MI355_LD(int32_t, a.cu_seqlens, a.cu_seqlens + j), c1 = MI355_LD(int32_t, a.cu_seqlens, a.cu_seqlens + j + 1);
    const int n_le = __popcll(__ballot(i < a.S && c0 / C + i <= slot));
    if (n_le > 0) s = base + n_le - 1, cs = __builtin_amdgcn_readlane(c0, n_le - 1), ce = __builtin_amdgcn_readlane(c1, n_le - 1);
    if (n_le < 64) break;
  }
  if (s < 0) return;
  const int r0 = (slot - cs / C - s) * C;
  if (r0 >= ce - cs) return;
  const int64_t row0 = cs + r0;
  const int n = ce - cs - r0 < C ? ce - cs - r0 : C;
  const uint16_t* qkv = static_cast<const uint16_t*>(a.qkv) + row0 * a.stride + g * D;
  // ---- keys -> LDS, this wave's 16 queries as a left operand (rows past the end: zeros); decays and rates of a head by a wave
  uint4 kr[KD], qb[KD];
#pragma unroll
  for (int j = 0; j < KD; ++j) {
    const int i = tid + 256 * j, t = i / (4 * KD), c = i % (4 * KD) * 8, tq = 16 * wave + li;
    kr[j] = MI355_LD(uint4, a.qkv, qkv + (t < n ? t : n - 1) * a.stride + a.k_off + c);
    qb[j] = MI355_LD(uint4, a.qkv, qkv + (tq < n ? tq : n - 1) * a.stride + a.q_off + 32 * j + 8 * kg);
  }
  if (wave < heads) {
    const int64_t row = row0 + (lane < n ? lane : n - 1);
    const int h = h0 + wave;
    const float beta = MI355_LDF(BF16, a.beta, static_cast<const uint16_t*>(a.beta) + row * a.beta_stride + h);
    const float z = MI355_LDF(BF16, a.decay, static_cast<const uint16_t*>(a.decay) + row * a.decay_stride + h) +
                    MI355_LD(float, a.dt_bias, a.dt_bias + h);
    // log2 of a decay; below 2^-200 a float is zero all the same
    const float l = -expf(MI355_LD(float, a.a_log, a.a_log + h)) * 1.44269504088896340736f * (z > 20.0f ? z : log1pf(expf(z)));
    double sum = lane < n ? static_cast<double>(l < -200.0f ? -200.0f : l) : 0.0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const double v = __shfl_up(sum, o, 64);
      if (lane >= o) sum += v;
    }
    G2[wave][lane] = sum;
    b2[wave][lane] = lane < n ? 1.0f / (1.0f + expf(-beta)) : 0.f;
  }
  float q8[KD];
#pragma unroll
  for (int j = 0; j < KD; ++j) {
    const int i = tid + 256 * j, t = i / (4 * KD), c = i % (4 * KD) * 8;
    if (t >= n) kr[j] = make_uint4(0u, 0u, 0u, 0u);
    if (16 * wave + li >= n) qb[j] = make_uint4(0u, 0u, 0u, 0u);
    float kf[8], qf[8], kk = 0.f, qq = 0.f;
    unpack8<BF16>(kr[j], kf), unpack8<BF16>(qb[j], qf);
#pragma unroll
    for (int x = 0; x < 8; ++x) kk += kf[x] * kf[x], qq += qf[x] * qf[x];
#pragma unroll
    for (int o = 1; o < 4 * KD; o <<= 1) kk += __shfl_xor(kk, o, 64);
    if (c == 0) rk[t] = 1.0f / sqrtf(kk + 1e-6f);
    q8[j] = qq;
    *reinterpret_cast<uint4*>(Ks + t * LK + c) = kr[j];
  }
  float qq = KD == 2 ? q8[0] + q8[1] : (q8[0] + q8[1]) + (q8[KD - 2] + q8[KD - 1]);
  qq += __shfl_xor(qq, 16, 64), qq += __shfl_xor(qq, 32, 64);
  if (kg == 0) rq[16 * wave + li] = (1.0f / sqrtf(static_cast<float>(D))) / sqrtf(qq + 1e-6f);
  __syncthreads();
  uint4 kb[KD];
#pragma unroll
  for (int x = 0; x < KD; ++x) kb[x] = *reinterpret_cast<const uint4*>(Ks + (16 * wave + li) * LK + 32 * x + 8 * kg);
  for (int hh = 0; hh < heads; ++hh) {
    int li = lane & 15, kg = lane >> 4;
    asm volatile("" : "+v"(li), "+v"(kg));                // (a head's addresses are worked out anew: kept, they would spill)
    const Chunk out = chunk_at(a.ws, slot, h0 + hh, g, a.H, a.G, D);
    const double* Gs = G2[hh];
    const float* bs = b2[hh];
    // ---- A and P, a block of 16 rows a wave
    {
      double Gt[4];
      float ft[4], qt[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * wave + 4 * kg + r;
        Gt[r] = Gs[t], ft[r] = bs[t] * rk[t], qt[r] = rq[t];
      }
      for (int J = 0; J <= wave; ++J) {
        f32x4 aa = f32x4{0.f, 0.f, 0.f, 0.f}, pp = aa;
#pragma unroll
        for (int x = 0; x < KD; ++x) {
          const uint4 f = *reinterpret_cast<const uint4*>(Ks + (16 * J + li) * LK + 32 * x + 8 * kg);
          aa = BF16::mfma(kb[x], f, aa), pp = BF16::mfma(qb[x], f, pp);
        }
        const int j = 16 * J + li;
        const double Gj = Gs[j];
        const float rj = rk[j];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = 16 * wave + 4 * kg + r;
          const float e = __builtin_amdgcn_exp2f(fminf(static_cast<float>(Gt[r] - Gj), 0.f));
          As[t * LT + j] = t > j ? aa[r] * (ft[r] * rj) * e : 0.f;
          Ps[t * LT + j] = t >= j ? pp[r] * (qt[r] * rj) * e : 0.f;
        }
      }
    }
    if (hh == 0 && set == 0) {                           // K, Q and K^T as left operands, once for the heads that share the key
#pragma unroll
      for (int x = 0; x < KD; ++x) {
        MI355_ST(uint4, a.ws, out.k + ((wave * KD + x) * 64 + lane) * 16, kb[x]);
        MI355_ST(uint4, a.ws, out.k + D * C * 2 + ((wave * KD + x) * 64 + lane) * 16, qb[x]);
      }
#pragma unroll
      for (int i = 0; i < KD; ++i) {                      // block m of 16 channels, rows 32 js + ..
        const int m = (wave * KD + i) >> 1, js = (wave * KD + i) & 1, ch = 32 * (m >> 1) + 8 * (li >> 2) + 4 * (m & 1) + (li & 3);
        uint32_t w[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const uint16_t* p = Ks + (32 * js + 16 * (x >> 1) + 4 * kg + 2 * (x & 1)) * LK + ch;
          w[x] = p[0] | static_cast<uint32_t>(p[LK]) << 16;
        }
        MI355_ST(uint4, a.ws, out.k + 2 * D * C * 2 + ((2 * m + js) * 64 + lane) * 16, make_uint4(w[0], w[1], w[2], w[3]));
      }
    }
    if (wave == 3) {
      const float e = __builtin_amdgcn_exp2f(static_cast<float>(Gs[lane]));
      MI355_ST(float, a.ws, out.rows + lane, lane < n ? rk[lane] * e : 0.f);
      MI355_ST(float, a.ws, out.rows + C + lane, rq[lane] * e);
      if (lane == C - 1) MI355_ST(float, a.ws, out.rows + 2 * C, e);      // (rows past the last add 0 to G)
    }
    // ---- inverses of the four diagonal blocks: a wave each (its own block of A), a column a lane (the lane's four copies the same)
    __builtin_amdgcn_wave_barrier();
    float y[16];
    {
      const float* A = As + 16 * wave * LT + 16 * wave;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        asm volatile("" ::: "memory");                    // (row by row: A's 120 numbers at once would take as many registers)
        float sum = i == li ? 1.f : 0.f;
#pragma unroll
        for (int j = 0; j < i; ++j) sum -= A[i * LT + j] * y[j];
        y[i] = sum;
      }
    }
    __builtin_amdgcn_wave_barrier();
    if (kg == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) As[(16 * wave + i) * LT + 16 * wave + li] = y[i];
    }
    __syncthreads();
    // ---- wave J has block column J of the inverse T (blocks J + m) and of Z; an accumulator is a right operand as it stands if step r
    // takes rows 4 g + r.  Every block of T is used up as soon as it is there, so that the products that wait for one another are few.
    f32x4 T[4], Z[4], sum[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) sum[m] = Z[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) T[0][r] = kg == 0 ? y[r] : kg == 1 ? y[4 + r] : kg == 2 ? y[8 + r] : y[12 + r];
    auto block = [&](const float* M, int I, int J) { return *reinterpret_cast<const float4*>(M + (16 * I + li) * LT + 16 * J + 4 * kg); };
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (wave + i > 3) break;
      asm volatile("" ::: "memory");
      if (i > 0) {
        const float4 d = block(As, wave + i, wave + i);
        const float df[4] = {-d.x, -d.y, -d.z, -d.w};
        T[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; ++r) T[i] = mfma4(df[r], sum[i][r], T[i]);
      }
      float4 l[4], q[4];
#pragma unroll
      for (int m = i; m < 4; ++m) {
        const int I = wave + m < 4 ? wave + m : 3;
        l[m] = block(As, I, wave + i), q[m] = block(Ps, I, wave + i);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int m = i; m < 4; ++m) {
          if (wave + m > 3) break;
          if (m > i) sum[m] = mfma4((&l[m].x)[r], T[i][r], sum[m]);
          Z[m] = mfma4((&q[m].x)[r], T[i][r], Z[m]);
        }
    }
    __syncthreads();
    {
      const double end = Gs[C - 1];
      const float b = bs[16 * wave + li];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        if (wave + m > 3) break;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = 16 * (wave + m) + 4 * kg + r;
          As[t * LT + 16 * wave + li] = T[m][r] * (b * rk[t]) * __builtin_amdgcn_exp2f(static_cast<float>(end - Gs[t]));
          Ps[t * LT + 16 * wave + li] = Z[m][r] * b;
        }
      }
    }
    __syncthreads();
    // ---- both in parts, as left operands: steps (0, 0..1), (1, 0..1), (2, 0..1), (3, 0..1), (2, 2..3), (3, 2..3) of blocks, what
    // lies above the diagonal 0
    {
      const float* M = wave & 1 ? Ps : As;
      char* to = out.x + (wave & 1 ? kTriBytes : 0);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int f = 3 * (wave >> 1) + i, I = f < 4 ? f : f - 2, J = f < 4 ? 0 : 2;
        const float4 u = block(M, I, J), v = I > J ? block(M, I, J + 1) : make_float4(0.f, 0.f, 0.f, 0.f);
        uint4 p[3];
        parts3(f32x4{u.x, u.y, u.z, u.w}, f32x4{v.x, v.y, v.z, v.w}, p);
#pragma unroll
        for (int x = 0; x < 3; ++x) MI355_ST(uint4, a.ws, to + ((f * 3 + x) * 64 + lane) * 16, p[x]);
      }
    }
    if (hh + 1 < heads) __syncthreads();
  }
}

// Workgroup (sequence, head, 16 value channels).  Those of one (sequence, head) read the same rows and chunks: they are dealt so
// that they fall on one XCD (every eighth block), whose L2 then serves all but the first.  Wave w keeps key channels [8 KD w,
// 8 KD (w + 1)) of the state and works out rows [16 w, 16 w + 16) of R, of U = X R and of the output.
template <int KD>
__global__ __launch_bounds__(256, 2) void delta_chunk_walk_kernel(DeltaTiles a, int groups) {
  constexpr int D = 32 * KD, SB = KD / 2;                 // blocks of 16 channels of the state a wave
  __shared__ uint4 Sp[KD][3][64], Rp[2][3][64], Up[2][3][64];      // parts of the state, of R and of U, as right operands
  const int unit = (blockIdx.x & 7) + 8 * (blockIdx.x / (8 * groups)), cg = (blockIdx.x >> 3) % groups;
  if (unit >= a.S * a.H) return;
  const int s = unit / a.H, h = unit % a.H, g = h / (a.H / a.G), dv = a.dv;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, kg = lane >> 4;
  const int cs = MI355_LD(int32_t, a.cu_seqlens, a.cu_seqlens + s);
  const int len = MI355_LD(int32_t, a.cu_seqlens, a.cu_seqlens + s + 1) - cs;
  if (len <= 0) return;
  const int col = cg * 16 + li, num = (len + C - 1) / C;
  const bool live = col < dv;
  const int cl = live ? col : dv - 1;
  const uint16_t* qkv = static_cast<const uint16_t*>(a.qkv);
  float* sp = a.state + ((static_cast<int64_t>(MI355_LD(int32_t, a.state_slots, a.state_slots + s)) * a.H + h) * D) * dv + cl;
  const bool fresh = MI355_LD(int64_t, a.positions, a.positions + cs) == 0;
  // block m of the state: row 4 g + r is channel 32 (m / 2) + 8 g + 4 (m % 2) + r
  auto channel = [&](int x, int r) { return 32 * ((wave * SB + x) >> 1) + 8 * kg + 4 * ((wave * SB + x) & 1) + r; };
  f32x4 S[SB];
#pragma unroll
  for (int x = 0; x < SB; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[x][r] = fresh ? 0.f : MI355_LD(float, a.state, sp + static_cast<int64_t>(channel(x, r)) * dv);
  // What a chunk brings.  Every load is a uniform base plus a lane's 32-bit offset that stays; only a last chunk of fewer rows
  // has its own (rows past the end repeat the last: their factors are 0, or their results are not stored).
  uint4 kf[KD], qf[KD], kt[SB][2], xf[2][3], zf[2][3];
  uint16_t v[4];
  float4 fr, fo;
  float end;
  uint32_t lv[4];
  auto offsets = [&](int n) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 16 * wave + 4 * kg + r < n ? 16 * wave + 4 * kg + r : n - 1;
      lv[r] = (static_cast<uint32_t>(t * a.stride) + cl) * 2u;
    }
  };
#define AT(base, off) (reinterpret_cast<const char*>(base) + (off))
  const Chunk at0 = chunk_at(a.ws, cs / C + s, h, g, a.H, a.G, D);
  const int64_t pitch = chunk_bytes(a.H, a.G, D);
  const uint16_t* values = qkv + static_cast<int64_t>(cs) * a.stride + a.v_off + static_cast<int64_t>(h) * dv;
  auto load_k = [&](int i) {
    const char* p = at0.k + i * pitch + wave * KD * 1024;
#pragma unroll
    for (int x = 0; x < KD; ++x) kf[x] = MI355_LD(uint4, a.ws, AT(p + x * 1024, 16u * lane));
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = MI355_LD(uint16_t, a.qkv, AT(values + static_cast<int64_t>(i) * C * a.stride, lv[r]));
    fr = MI355_LD(float4, a.ws, AT(at0.rows, i * pitch + 64 * wave + 16u * kg));
  };
  auto load_q = [&](int i) {
    const char* p = at0.k + i * pitch + D * C * 2 + wave * KD * 1024;
#pragma unroll
    for (int x = 0; x < KD; ++x) qf[x] = MI355_LD(uint4, a.ws, AT(p + x * 1024, 16u * lane));
    fo = MI355_LD(float4, a.ws, AT(at0.rows, i * pitch + 4 * C + 64 * wave + 16u * kg));
  };
  auto load_tri = [&](uint4 (&f)[2][3], const char* p) {
#pragma unroll
    for (int y = 0; y < 3; ++y) f[0][y] = MI355_LD(uint4, a.ws, AT(p + (wave * 3 + y) * 1024, 16u * lane));
    if (wave >= 2) {
#pragma unroll
      for (int y = 0; y < 3; ++y) f[1][y] = MI355_LD(uint4, a.ws, AT(p + (wave * 3 + 6 + y) * 1024, 16u * lane));
    }
  };
  auto load_kt = [&](int i) {
    const char* p = at0.k + i * pitch + 2 * D * C * 2 + wave * SB * 2048;
#pragma unroll
    for (int x = 0; x < SB; ++x)
#pragma unroll
      for (int js = 0; js < 2; ++js) kt[x][js] = MI355_LD(uint4, a.ws, AT(p + (2 * x + js) * 1024, 16u * lane));
    end = MI355_LD(float, a.ws, AT(at0.rows, i * pitch + 8 * C));
  };
#undef AT
  // onto acc, the parts of R's rows up to this wave's (blocks past the wave's own meet zeros on both sides).  Products of first parts
  // and all others have an accumulator each: every addition to the large one is rounded at its size.
  auto tri_times = [&](const uint4 (&f)[2][3], const uint4 (&R)[2][3], f32x4 acc) {
    f32x4 low = f32x4{0.f, 0.f, 0.f, 0.f};
    auto step = [&](int js) {
      low = BF16::mfma(f[js][2], R[js][0], low);
      acc = BF16::mfma(f[js][0], R[js][0], acc);
      low = BF16::mfma(f[js][1], R[js][1], low);
      low = BF16::mfma(f[js][0], R[js][2], low);
      low = BF16::mfma(f[js][1], R[js][0], low);
      low = BF16::mfma(f[js][0], R[js][1], low);
    };
    step(0);
    if (wave >= 2) step(1);
    return acc + low;
  };
  // an accumulator's four numbers -> parts, half of a right operand
  auto put = [&](uint4 (*to)[64], int half, const f32x4& u) {
    uint32_t p[3][2];
    parts3(u[0], u[1], p[0][0], p[1][0], p[2][0]), parts3(u[2], u[3], p[0][1], p[1][1], p[2][1]);
#pragma unroll
    for (int y = 0; y < 3; ++y) reinterpret_cast<uint2*>(&to[y][lane])[half] = make_uint2(p[y][0], p[y][1]);
  };
  offsets(len < C ? len : C);
  load_k(0), load_q(0), load_tri(xf, at0.x), load_tri(zf, at0.x + kTriBytes), load_kt(0);
  for (int i = 0; i < num; ++i) {
    const int next = i + 1 < num ? i + 1 : i, n = len - i * C, left = n - 16 * wave - 4 * kg;
    if (next > i && len - next * C < C) offsets(len - next * C);
#pragma unroll
    for (int x = 0; x < SB; ++x) put(Sp[(wave * SB + x) >> 1], (wave * SB + x) & 1, S[x]);
    __syncthreads();
    f32x4 X = f32x4{0.f, 0.f, 0.f, 0.f}, Y = X, low = X;
    uint4 sf[KD][3];
#pragma unroll
    for (int x = 0; x < KD; ++x)
#pragma unroll
      for (int y = 2; y >= 0; --y) sf[x][y] = Sp[x][y][lane];
#pragma unroll
    for (int x = 0; x < KD; ++x)
#pragma unroll
      for (int y = 2; y >= 0; --y) (y ? low : X) = BF16::mfma(kf[x], sf[x][y], y ? low : X);
    X += low;
    const float f[4] = {fr.x, fr.y, fr.z, fr.w};
#pragma unroll
    for (int r = 0; r < 4; ++r) X[r] = r < left ? BF16::to_f(v[r]) - f[r] * X[r] : 0.f;
    put(Rp[wave >> 1], wave & 1, X);
    __builtin_amdgcn_sched_barrier(0);
    load_k(next);
    __builtin_amdgcn_sched_barrier(0);
    low = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < KD; ++x)
#pragma unroll
      for (int y = 2; y >= 0; --y) (y ? low : Y) = BF16::mfma(qf[x], sf[x][y], y ? low : Y);
    Y += low;
    __syncthreads();
    uint4 R[2][3];
#pragma unroll
    for (int js = 0; js < 2; ++js)
#pragma unroll
      for (int y = 0; y < 3; ++y) {
        R[js][y] = Rp[js][y][lane];
        if (wave == 2 * js) R[js][y].z = R[js][y].w = 0u;
      }
    const f32x4 U = tri_times(xf, R, f32x4{0.f, 0.f, 0.f, 0.f});
    put(Up[wave >> 1], wave & 1, U);
    __builtin_amdgcn_sched_barrier(0);
    Y[0] *= fo.x, Y[1] *= fo.y, Y[2] *= fo.z, Y[3] *= fo.w;
    load_q(next), load_tri(xf, at0.x + next * pitch);
    __builtin_amdgcn_sched_barrier(0);
    Y = tri_times(zf, R, Y);
    __syncthreads();
#pragma unroll
    for (int x = 0; x < SB; ++x) S[x] *= end;
#pragma unroll
    for (int y = 2; y >= 0; --y)
#pragma unroll
      for (int js = 0; js < 2; ++js) {
        const uint4 u = Up[js][y][lane];
#pragma unroll
        for (int x = 0; x < SB; ++x) S[x] = BF16::mfma(kt[x][js], u, S[x]);
      }
    __builtin_amdgcn_sched_barrier(0);
    load_tri(zf, at0.x + next * pitch + kTriBytes), load_kt(next);
    float* o = a.o + ((static_cast<int64_t>(cs) + i * C + 16 * wave) * a.H + h) * dv;
    const uint32_t lo = (static_cast<uint32_t>(4 * kg * a.H * dv) + cl) * 4u;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < left && live) MI355_ST(float, a.o, reinterpret_cast<char*>(o + r * a.H * dv) + lo, Y[r]);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (live) {
#pragma unroll
    for (int x = 0; x < SB; ++x)
#pragma unroll
      for (int r = 0; r < 4; ++r) MI355_ST(float, a.state, sp + static_cast<int64_t>(channel(x, r)) * dv, S[x][r]);
  }
}

}  // namespace

int64_t delta_chunks_workspace(int64_t rows, int S, int H, int G, int d, bool per_channel) {
  if (per_channel || (d != 64 && d != 128) || rows < static_cast<int64_t>(C) * S) return 0;
  return (rows / C + S) * chunk_bytes(H, G, d) / 4;
}

bool delta_chunks_ok(const DeltaTiles& a, int dtype) {
  return dtype == MI355_BF16 && a.q_off % 8 == 0 && a.k_off % 8 == 0 && a.stride % 8 == 0 && aligned16(a.qkv);
}

void launch_delta_chunks(const DeltaTiles& a, hipStream_t stream) {
  // two heads a workgroup where that still leaves three workgroups a CU (us, one head / two: 2112 and 1056 workgroups 56 / 47, 528 and
  // 264 18 / 25)
  const int64_t slots = a.rows / C + a.S, rep = a.H / a.G;
  const int per = rep > 1 && slots * a.G * ((rep + 1) / 2) >= 768 ? 2 : 1;
  const dim3 pgrid(static_cast<unsigned>(slots), static_cast<unsigned>(a.G * ((rep + per - 1) / per)));
  const int groups = (a.dv + 15) / 16;
  const unsigned units = static_cast<unsigned>(a.S) * static_cast<unsigned>(a.H);
  const dim3 wgrid((units + 7) / 8 * 8 * static_cast<unsigned>(groups));
  if (a.d == 64) {
    hipLaunchKernelGGL((delta_chunk_prep_kernel<2>), pgrid, dim3(256), 0, stream, a, per);
    hipLaunchKernelGGL((delta_chunk_walk_kernel<2>), wgrid, dim3(256), 0, stream, a, groups);
  } else {
    hipLaunchKernelGGL((delta_chunk_prep_kernel<4>), pgrid, dim3(256), 0, stream, a, per);
    hipLaunchKernelGGL((delta_chunk_walk_kernel<4>), wgrid, dim3(256), 0, stream, a, groups);
  }
}

}  // namespace mi355
