// Grouped products on the matrix cores (16-bit storage, fp32 accumulation): for every group g
//     y = a(X_g W_g^T),   W_g [n, k],   a: the identity or relu^2
// Two kinds of groups share the kernel:
//   * a mixture's experts: group e's rows are positions offsets[e] .. offsets[e + 1] of the expert order, read
//     through perm (row perm[p] / top of x) or in place, written at their position.  The row tiles of all experts
//     are numbered by tile_start, so one launch covers whatever the loads are; no count comes to the host;
//   * heads: every group has the same rows (optionally through an index: rows of paged memory), x and y are
//     column slices x_group / y_group elements apart.
// Output addressing: y + (m / 16) * y_block + (m % 16) * y_stride + g * y_group + n, which covers plain rows
// (y_block = 16 y_stride) and pages of 16 tokens; TRANS: ... + n * 16 + m % 16 (pages with the tokens innermost).
// copy > 0: columns k .. k + copy of the x row follow the n outputs of every group (a part shared by all heads).
//
// One workgroup (4 waves) per BM x BN tile of (rows, outputs).  64-wide K steps of X and W go through registers
// into LDS: two steps on their way in registers, two images in LDS, one barrier per step.  An LDS row is 128 bytes, eight 16-byte slots; slot s of row r
// sits at s ^ ((r / 2) & 7): the 16 rows of a fragment read then cover 256 bytes without a bank twice.
#include "common.h"

namespace mi355 {

constexpr int kBK = 64;

struct GroupGemmArgs {
  uint16_t* y;
  int64_t y_block, y_stride, y_group;
  const uint16_t* x;
  int64_t x_stride, x_group, x_rows;
  const int32_t* perm;
  int top;
  const uint16_t* w;
  int64_t w_group;
  const int32_t* offsets;
  const int32_t* tile_start;
  int groups;
  int64_t rows;                        // rows of every group (heads) or of all together (experts)
  int n, k, copy, relu2;
  float limit;
};

// MW: waves along the rows (the other 4 / MW lie along the outputs)
template <typename T, int BM, int BN, int MW, bool TRANS>
__global__ __launch_bounds__(256, 2) void group_gemm_kernel(GroupGemmArgs a) {
  constexpr int NW = 4 / MW, TM = BM / MW / 16, TN = BN / NW / 16;      // a wave's 16 x 16 blocks
  constexpr int XP = BM * 8 / 256, WP = BN * 8 / 256;                   // 16-byte pieces per thread and step
  static_assert(BM * 8 % 256 == 0 && BN * 8 % 256 == 0, "whole pieces per thread");
  __shared__ __attribute__((aligned(16))) uint16_t lds[2][(BM + BN) * kBK];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, kk = lane >> 4;
  // workgroups go to the 8 XCDs in turn: XCD i takes the i-th contiguous part of the tiles
  const int ntn = (a.n + BN - 1) / BN;
  // (of the tiles that exist: the grid is sized for the most there can be)
  int total = gridDim.x;
  if (a.offsets != nullptr) total = min(total, MI355_LD(int32_t, a.tile_start, a.tile_start + a.groups) * ntn);
  if (static_cast<int>(blockIdx.x) >= total) return;    // (uniform over the workgroup)
  const int xcd = blockIdx.x & 7;
  const int work = xcd * (total >> 3) + min(xcd, total & 7) + (blockIdx.x >> 3);
  int mt = work / ntn;
  const int n0 = (work % ntn) * BN;
  int g;
  int64_t lo, hi;
  if (a.offsets != nullptr) {                           // the expert whose tiles hold number mt
    int l = 0, h = a.groups;                            // tile_start[l] <= mt < tile_start[h]
    while (h - l > 1) {
      const int mid = (l + h) >> 1;
      if (MI355_LD(int32_t, a.tile_start, a.tile_start + mid) <= mt) l = mid; else h = mid;
    }
    g = l;
    mt -= MI355_LD(int32_t, a.tile_start, a.tile_start + g);
    lo = MI355_LD(int32_t, a.offsets, a.offsets + g);
    hi = MI355_LD(int32_t, a.offsets, a.offsets + g + 1);
  } else {
    const int per = static_cast<int>((a.rows + BM - 1) / BM);
    g = mt / per;
    mt -= g * per;
    lo = 0;
    hi = a.rows;
  }
  const int64_t m0 = lo + static_cast<int64_t>(mt) * BM;
  if (g >= a.groups || m0 >= hi) return;
  const uint16_t* wg = a.w + g * a.w_group;
  const int r8 = tid >> 3, s8 = tid & 7;
  auto x_row = [&](int64_t p) {                          // row of x that position p reads, always a valid one
    int64_t r = p;
    if (a.perm != nullptr) r = MI355_LD(int32_t, a.perm, a.perm + p) / a.top;
    r = r < 0 ? 0 : (r >= a.x_rows ? a.x_rows - 1 : r);
    return a.x + r * a.x_stride + g * a.x_group;
  };
  const uint16_t* xp[XP];
  const uint16_t* wp[WP];
  int dx[XP], dw[WP];
#pragma unroll
  for (int j = 0; j < XP; ++j) {
    const int r = r8 + 32 * j;
    xp[j] = x_row(m0 + r < hi ? m0 + r : hi - 1);
    dx[j] = r * kBK + ((s8 ^ ((r >> 1) & 7)) << 3);
  }
#pragma unroll
  for (int j = 0; j < WP; ++j) {
    const int r = r8 + 32 * j;
    wp[j] = wg + static_cast<int64_t>(n0 + r < a.n ? n0 + r : a.n - 1) * a.k;
    dw[j] = BM * kBK + r * kBK + ((s8 ^ ((r >> 1) & 7)) << 3);
  }
  typedef unsigned int pvec __attribute__((ext_vector_type(4)));
  pvec rx[2][XP], rw[2][WP];
  // No branch around a load or a store: it would make the compiler drain the loads in flight at its join.  Columns past
  // k (the last step's, and steps past the last) read the last ones instead, and X's are cleared on the way into LDS.
  auto load = [&](int set, int t) {
    const int at = min(t * kBK + 8 * s8, a.k - 8);        // (k a multiple of 8)
#pragma unroll
    for (int j = 0; j < XP; ++j) rx[set][j] = MI355_LD(pvec, a.x, xp[j] + at);
#pragma unroll
    for (int j = 0; j < WP; ++j) rw[set][j] = MI355_LD(pvec, a.w, wp[j] + at);
  };
  auto store = [&](int set, int t) {                     // (image = set)
    const bool have = t * kBK + 8 * s8 < a.k;
#pragma unroll
    for (int j = 0; j < XP; ++j) *reinterpret_cast<pvec*>(&lds[set][dx[j]]) = have ? rx[set][j] : pvec{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < WP; ++j) *reinterpret_cast<pvec*>(&lds[set][dw[j]]) = rw[set][j];
  };
  const int wm = (wave % MW) * (BM / MW), wn = (wave / MW) * (BN / NW);
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int sw = (li >> 1) & 7;                          // (16-row blocks: the swizzle depends on the row in the block alone)
  const int steps = (a.k + kBK - 1) / kBK;
  load(0, 0);
  load(1, 1);
  store(0, 0);
  __syncthreads();
  // step t computes image t % 2, sends for step t + 2 and stores step t + 1 into the other image
  auto step = [&](int t, int set) {
    load(set, t + 2);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int slot = ((4 * ks + kk) ^ sw) << 3;
      uint4 xf[TM], wf[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) xf[i] = *reinterpret_cast<const uint4*>(&lds[set][(wm + 16 * i + li) * kBK + slot]);
#pragma unroll
      for (int j = 0; j < TN; ++j) wf[j] = *reinterpret_cast<const uint4*>(&lds[set][BM * kBK + (wn + 16 * j + li) * kBK + slot]);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = TRANS ? T::mfma(xf[i], wf[j], acc[i][j]) : T::mfma(wf[j], xf[i], acc[i][j]);
    }
    __builtin_amdgcn_s_setprio(0);
    store(set ^ 1, t + 1);
    __syncthreads();
  };
  for (int t = 0; t < steps; t += 2) {                   // (an odd last step is followed by one of cleared X)
    step(t, 0);
    step(t + 1, 1);
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = acc[i][j][r];
        if (a.relu2) {                                   // (of the product as a 16-bit buffer would hold it)
          v[r] = fmaxf(round_f<T>(v[r]), 0.f);
          v[r] *= v[r];
        }
      }
      if (TRANS) {                                       // rows m .. m + 3 of output n
        const int64_t m = m0 + wm + 16 * i + 4 * kk;
        const int n = n0 + wn + 16 * j + li;
        if (n >= a.n || m >= hi) continue;
        uint16_t* p = a.y + (m >> 4) * a.y_block + g * a.y_group + static_cast<int64_t>(n) * 16 + (m & 15);
        if (m + 3 < hi) {
          MI355_ST(uint2, a.y, p, make_uint2(T::pack2(v[0], v[1]), T::pack2(v[2], v[3])));
        } else {
          for (int r = 0; r < 4 && m + r < hi; ++r) MI355_ST(uint16_t, a.y, p + r, T::from_f(v[r]));
        }
      } else {                                           // outputs n .. n + 3 of row m (n a multiple of 4)
        const int64_t m = m0 + wm + 16 * i + li;
        const int n = n0 + wn + 16 * j + 4 * kk;
        if (n >= a.n || m >= hi) continue;
        uint16_t* p = a.y + (m >> 4) * a.y_block + (m & 15) * a.y_stride + g * a.y_group + n;
        MI355_ST(uint2, a.y, p, make_uint2(T::pack2(v[0], v[1]), T::pack2(v[2], v[3])));
      }
    }
  }
  if (a.copy > 0 && n0 == 0) {
    const int per = a.copy >> 3;                         // 16-byte pieces per row
    for (int i = tid; i < BM * per; i += 256) {
      const int64_t m = m0 + i / per;
      if (m >= hi) break;
      const int c = (i % per) * 8;
      MI355_ST(uint4, a.y, a.y + (m >> 4) * a.y_block + (m & 15) * a.y_stride + g * a.y_group + a.n + c,
               MI355_LD(uint4, a.x, x_row(m) + a.k + c));
    }
  }
}


// ---- tiles of 256 x 256: a persistent workgroup of 8 waves a CU -------------------------------------------------------
// What bounds the kernel above at many rows is not the matrix cores: a 128 x 128 tile asks L2 for 64 bytes a clock and CU
// at their full rate, as much as comes.  256 x 256 halves that, and the loads go straight to LDS (lds_dma16).
//
// Waves 0-3 and 4-7 are two groups, one wave of each on a SIMD, half a phase apart: while one group reads its fragments
// and sends loads, the other has the matrix cores; a barrier after every phase keeps them so.  A step is 64 columns of K
// in four phases: fragments of the wave's first 64 rows and of its 64 outputs (16 reads), their products, fragments of the
// other 64 rows (8 reads), their products.  Two images of 64 KB in LDS: the loads of step t + 2 overwrite what both groups have
// read of step t -- the first rows and W after the second read phase, the other rows a step later -- and have four
// phases to land.  Loads run on into the next tile, so that a tile's first loads travel under the end of the one ahead;
// the results' stores travel under the next tile's first phases (wait_vm counts them where a whole tile was stored).  Gathered rows
// (perm) are the exception: what a tile's addresses are read from is waited for with all that is out, in its last two steps.
//
// Row tiles of 256 leave more padding than 128 where the groups' rows are few or end unevenly: an expert's last 1 .. 128
// rows, or all rows if that is the shorter plan for the rounds of workgroups (below), go as tiles of 128 x 256, half the
// phases a step, three images of 48 KB.
//
// Measured in bf16: 32844 rows of 32 experts 2048 -> 1536 195 us (1060 TFLOP/s of the products asked for), 1536 -> 2048
// 205 us; by tiles of 128 x 128 351 and 326 us on the same card.  One plain product of 8192^3 runs at 1510 TFLOP/s here (the library's at
// 1590), and one whose activation would be a launch of its own is the faster way with it at the tile's end (mi355_linear_act): 4096 rows
// 4096 -> 28672 with SwiGLU 667 us (the library and the launch 702), 8192 rows 2048 -> 6144 with relu^2 144 (168), 2048 -> 8192 with GELU 213
// (231).  The units of a gated tile take some 7 us of a CU, during which its matrix cores are idle but for half a phase.
constexpr int kWideThreads = 512, kWideMaxGroups = 512;

// Fragments of one read phase.  By instructions of our own, each block with its wait: the compiler cannot tell which loads
// into LDS a read depends on and would wait for all of them.  X rows 16 apart (2048 bytes); W rows of fragment j at
// (j >> 1) * 32 + (j & 1) * 4, so that a lane's outputs of two fragments are 8 adjacent ones.
__device__ __forceinline__ void wide_read_xw(uint32_t x0, uint32_t x1, uint32_t w0, uint32_t w1, uint4 (&x)[2][4], uint4 (&w)[2][4]) {
  asm volatile(
      "ds_read_b128 %0, %16\n ds_read_b128 %1, %16 offset:2048\n ds_read_b128 %2, %16 offset:4096\n ds_read_b128 %3, %16 offset:6144\n"
      "ds_read_b128 %8, %18\n ds_read_b128 %9, %18 offset:512\n ds_read_b128 %10, %18 offset:4096\n ds_read_b128 %11, %18 offset:4608\n"
      "ds_read_b128 %4, %17\n ds_read_b128 %5, %17 offset:2048\n ds_read_b128 %6, %17 offset:4096\n ds_read_b128 %7, %17 offset:6144\n"
      "ds_read_b128 %12, %19\n ds_read_b128 %13, %19 offset:512\n ds_read_b128 %14, %19 offset:4096\n ds_read_b128 %15, %19 offset:4608\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[0][2]), "=&v"(x[0][3]), "=&v"(x[1][0]), "=&v"(x[1][1]), "=&v"(x[1][2]), "=&v"(x[1][3]),
        "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(w[0][2]), "=&v"(w[0][3]), "=&v"(w[1][0]), "=&v"(w[1][1]), "=&v"(w[1][2]), "=&v"(w[1][3])
      : "v"(x0), "v"(x1), "v"(w0), "v"(w1)
      : "memory");
}
__device__ __forceinline__ void wide_read_x(uint32_t x0, uint32_t x1, uint4 (&x)[2][4]) {      // the 64 rows behind those
  asm volatile(
      "ds_read_b128 %0, %8 offset:8192\n ds_read_b128 %1, %8 offset:10240\n ds_read_b128 %2, %8 offset:12288\n"
      "ds_read_b128 %3, %8 offset:14336\n ds_read_b128 %4, %9 offset:8192\n ds_read_b128 %5, %9 offset:10240\n"
      "ds_read_b128 %6, %9 offset:12288\n ds_read_b128 %7, %9 offset:14336\n s_waitcnt lgkmcnt(0)"
      : "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[0][2]), "=&v"(x[0][3]), "=&v"(x[1][0]), "=&v"(x[1][1]), "=&v"(x[1][2]), "=&v"(x[1][3])
      : "v"(x0), "v"(x1)
      : "memory");
}
__device__ __forceinline__ int wide_read_int(const int* p) {
  int v;
  asm volatile("ds_read_b32 %0, %1\n s_waitcnt lgkmcnt(0)"
               : "=&v"(v)
               : "v"(static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) int*)p)))
               : "memory");
  return v;
}

// Eight units of a gated activation.  silu and the limited unit by the lean quotient where the gate is in its range (a NaN passes through
// it), else as they stand: by every gate for itself, so that a unit's bits depend on its own gate and up alone.  A wave whose gates
// are all in range skips the other form.
template <typename T, int ACT>
__device__ __forceinline__ void gated_units(float (&g)[8], const float (&u)[8], float limit, float (&v)[8]) {
  if constexpr (ACT == MI355_ACT_GELU_MUL) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = gelu_tanh_fast(g[e]) * u[e];
    return;
  }
  constexpr float c = ACT == MI355_ACT_SILU_MUL ? 1.0f : 1.702f;
  float top = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    if (ACT == MI355_ACT_LIMITED_MUL) g[e] = fminf(g[e], limit);
    top = fmaxf(top, fabsf(g[e]));
    v[e] = over_one_plus_exp_lean(g[e], c * g[e]);
  }
  if (!__all(top < kSiluLeanRange / c)) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (fabsf(g[e]) >= kSiluLeanRange / c) v[e] = g[e] / (1.0f + expf(-c * g[e]));
  }
#pragma unroll
  for (int e = 0; e < 8; ++e)
    v[e] = ACT == MI355_ACT_SILU_MUL ? round_f<T>(pin_f32(v[e])) * u[e] : v[e] * (fminf(fmaxf(u[e], -limit), limit) + 1.0f);
}

// per: outputs of a group that lie side by side in y (experts: all n; heads: a head's); a.n: outputs of a row tile
// GATED (an MI355_ACT_*_MUL, 0: none): the one matrix holds n / 2 gate rows and as many up rows, y = a(gate) * up of n / 2 columns.  A wave's
// 64 rows of W are 32 gates and their ups then, so that both lie in the same lane.
template <typename T, bool TRANS, int GATED = 0>
__global__ __launch_bounds__(kWideThreads, 2) void group_gemm_wide_kernel(GroupGemmArgs a, int per) {
  constexpr int kFull = 512 * kBK, kHalf = 384 * kBK;                  // an image: X rows | 256 W rows
  __shared__ __attribute__((aligned(16))) uint16_t lds[3 * kHalf];
  __shared__ int first[4][kWideMaxGroups + 1];                         // rows | tiles of 256 | of 128 beside them | of 128 alone
  static_assert(3 * kHalf >= 2 * kFull, "one buffer for both kinds of tiles");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, kk = lane >> 4;
  const int ntn = (a.n + 255) / 256, W = gridDim.x;
  const bool experts = a.offsets != nullptr;
  // without experts: groups of 1024 rows of the one matrix, whose tiles run side by side on an XCD
  const int groups = experts ? a.groups : static_cast<int>((a.rows + 1023) >> 10);
  int full_tiles, rest_tiles, half_tiles;                              // row tiles of 256 | of 128 beside them | of 128 alone
  if (experts) {
    if (wave == 0) {
      int sum[3] = {0, 0, 0};
      for (int base = 0; base < groups; base += 64) {
        const int e = base + lane, c = e < groups ? e : groups - 1;
        const int lo = MI355_LD(int32_t, a.offsets, a.offsets + c), hi = MI355_LD(int32_t, a.offsets, a.offsets + c + 1);
        const int rows = e < groups ? hi - lo : 0, last = rows & 255;
        int v[3] = {(rows >> 8) + (last > 128), last > 0 && last <= 128, (rows + 127) >> 7};
#pragma unroll
        for (int q = 0; q < 3; ++q) {
#pragma unroll
          for (int o = 1; o < 64; o <<= 1) {
            const int up = __shfl_up(v[q], o, 64);
            if (lane >= o) v[q] += up;
          }
          v[q] += sum[q];
          if (e < groups) first[1 + q][e + 1] = v[q];
          sum[q] = __builtin_amdgcn_readlane(v[q], 63);
        }
        if (e < groups) first[0][e] = lo;
        if (e == groups - 1) first[0][groups] = hi;
      }
      if (lane < 3) first[1 + lane][0] = 0;
    }
    __syncthreads();
    full_tiles = __builtin_amdgcn_readfirstlane(first[1][groups]), rest_tiles = __builtin_amdgcn_readfirstlane(first[2][groups]);
    half_tiles = __builtin_amdgcn_readfirstlane(first[3][groups]);
  } else {
    const int rows = static_cast<int>(a.rows), last = rows & 255;
    full_tiles = (rows >> 8) + (last > 128), rest_tiles = last > 0 && last <= 128, half_tiles = (rows + 127) >> 7;
  }
  // The plan of fewer rounds, in tiles of 128 rows, weighed 29 : 25 (32 experts of 1024 rows by small tiles alone take 1.19 to 1.21
  // times as long, 206 / 173 us 2048 -> 1536, 505 / 418 us 4096 -> 2048; their steps alone run at 1269 against 1445 TFLOP/s, 1.14):
  // workgroups that have no tile of a last partial round take two of the small ones meanwhile.
  bool halves;
  {
    const int f = full_tiles * ntn, h = rest_tiles * ntn, part = f % W;
    const int more = part > 0 ? max(h - 2 * (W - part), 0) : h;
    const int mixed = 2 * ((f + W - 1) / W) + (more + W - 1) / W;
    halves = 29 * ((half_tiles * ntn + W - 1) / W) < 25 * mixed;
  }
  // XCD c takes the c-th contiguous part of the tiles, its workgroups in turn
  const int nx = min(W, 8), xcd = blockIdx.x % nx, mine = blockIdx.x / nx, wgs = (W - xcd + nx - 1) / nx;
  struct Tile {
    int m0, hi, n0, g;
  };
  // tile u of kind q (1: 256 rows, 2: 128 rows beside them, 3: 128 rows alone): a group's row tiles in turn, then the next outputs
  auto place = [&](int q, int u) {
    Tile t;
    const int size = q == 1 ? 256 : 128;
    int at, n;                                                         // first row tile of the group, its number of them
    if (experts) {
      t.g = -1;
      at = n = 0;
      for (int base = 0; base < groups; base += 64) {                  // the group whose tiles hold u: the last that starts by it
        const int e = min(base + lane, groups);
        const int lo = wide_read_int(&first[q][e]);
        const int c = __popcll(__ballot(base + lane < groups && lo * ntn <= u));
        if (c > 0) t.g = base + c - 1, at = __builtin_amdgcn_readlane(lo, c - 1);
        if (c < 64) break;
      }
      n = __builtin_amdgcn_readfirstlane(wide_read_int(&first[q][t.g + 1])) - at;
      t.m0 = __builtin_amdgcn_readfirstlane(wide_read_int(&first[0][t.g]));
      t.hi = __builtin_amdgcn_readfirstlane(wide_read_int(&first[0][t.g + 1]));
    } else {
      const int row_tiles = q == 1 ? full_tiles : q == 2 ? rest_tiles : half_tiles, most = 1024 / size;
      const int c = u / (most * ntn);
      at = c * most, n = min(row_tiles - at, most);
      t.g = 0, t.m0 = c << 10, t.hi = static_cast<int>(a.rows);
    }
    const int local = u - at * ntn;
    t.n0 = local / n * 256;
    // (a small tile beside large ones holds the group's last rows)
    if (q == 2) t.m0 = t.m0 + ((t.hi - t.m0 - 1) & ~255);
    else t.m0 += local % n * size;
    return t;
  };
  const int r = tid >> 3;                                              // row of a 64-row piece this thread brings
  const uint32_t sx = ((tid & 7) ^ ((r >> 1) & 7)) * 16, sw = ((tid & 7) ^ (((r >> 1) & 1) | (((r >> 3) & 3) << 1))) * 16;
  const char* xb = reinterpret_cast<const char*>(a.x);
  auto x_at = [&](const Tile& t, int row) {                            // byte offset of a row of the tile (past its end: its last)
    int64_t p = t.m0 + row < t.hi ? t.m0 + row : t.hi - 1;
    if (a.perm != nullptr) p = MI355_LD(int32_t, a.perm, a.perm + p) / a.top;
    p = p < 0 ? 0 : (p >= a.x_rows ? a.x_rows - 1 : p);
    return static_cast<uint32_t>(p * a.x_stride) * 2u + sx;
  };
  auto w_at = [&](const Tile& t, int row) {
    int n = t.n0 + row < a.n ? t.n0 + row : a.n - 1;
    if constexpr (GATED != 0) {
      const int half = a.n >> 1, col = (t.n0 >> 1) + (row >> 6) * 32 + (row & 31);
      n = (col < half ? col : half - 1) + (row & 32 ? half : 0);
    }
    return static_cast<uint32_t>(n) * static_cast<uint32_t>(a.k) * 2u + sw;
  };
  auto w_base = [&](const Tile& t) { return reinterpret_cast<const char*>(a.w + t.g * a.w_group); };
  const int steps = a.k / kBK;                                         // (two at least, no remainder)
  const int rb = ((li >> 2) << 3) | (li & 3);                          // W row of this lane in a fragment
  const int fx = (li >> 1) & 7, fw = ((rb >> 1) & 1) | (((rb >> 3) & 3) << 1), wn = (wave & 3) * 64;
  const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint16_t*)lds));
  f32x4 acc[2][4][4];
  uint4 xf[2][4], wf[2][4];
  auto clear = [&]() {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[h][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto products = [&](f32x4 (&c)[4][4]) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) c[i][j] = TRANS ? T::mfma(xf[ks][i], wf[ks][j], c[i][j]) : T::mfma(wf[ks][j], xf[ks][i], c[i][j]);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // results of the wave's 64 rows from m on; whole: no row or output past the end
  auto emit = [&](const f32x4 (&c)[4][4], int m0, const Tile& t, bool whole) {
    const int nb = t.n0 + wn, in = nb % per;                           // (a wave's 64 outputs lie in one group)
    uint16_t* y = a.y + (t.g + nb / per) * a.y_group;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (GATED != 0) {                                      // columns n .. n + 7 of row m
        const int m = m0 + 16 * i + li, n = (nb >> 1) + kk * 8;
        float g[8], u[8], v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)                                    // (the products as a 16-bit buffer would hold them)
          g[e] = round_f<T>(c[i][e >> 2][e & 3]), u[e] = round_f<T>(c[i][2 + (e >> 2)][e & 3]);
        gated_units<T, GATED>(g, u, a.limit, v);
        uint16_t* p = a.y + static_cast<int64_t>(m) * a.y_stride + n;
        if (whole) store_one(a.y, p, pack8<T>(v));
        else if (m < t.hi && 2 * n < a.n) MI355_ST(uint4, a.y, p, pack8<T>(v));
      } else if (TRANS) {                                                     // rows m .. m + 3 of output n
        const int m = m0 + 16 * i + 4 * kk;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int n = (j >> 1) * 32 + (j & 1) * 4 + rb;
          uint16_t* p = y + static_cast<int64_t>(m >> 4) * a.y_block + static_cast<int64_t>(in + n) * 16 + (m & 15);
          const f32x4 v = c[i][j];
          const uint2 four = make_uint2(T::pack2(v[0], v[1]), T::pack2(v[2], v[3]));
          if (whole) {
            store_one(a.y, p, four);
          } else if (m + 3 < t.hi && nb + n < a.n) {
            MI355_ST(uint2, a.y, p, four);
          } else if (nb + n < a.n) {
            for (int e = 0; e < 4 && m + e < t.hi; ++e) MI355_ST(uint16_t, a.y, p + e, T::from_f(v[e]));
          }
        }
      } else {                                                         // outputs n .. n + 7 of row m
        const int m = m0 + 16 * i + li;
        uint16_t* row = y + static_cast<int64_t>(m >> 4) * a.y_block + (m & 15) * a.y_stride + in;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          float v[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            v[e] = c[i][2 * s + (e >> 2)][e & 3];
            if (a.relu2) {                                             // (of the product as a 16-bit buffer would hold it)
              v[e] = fmaxf(round_f<T>(v[e]), 0.f);
              v[e] *= v[e];
            }
          }
          const int n = s * 32 + kk * 8;
          if (whole) store_one(a.y, row + n, pack8<T>(v));
          else if (m < t.hi && nb + n < a.n) MI355_ST(uint4, a.y, row + n, pack8<T>(v));
        }
      }
    }
  };
  constexpr int S = TRANS ? 16 : GATED ? 4 : 8;                        // stores of 64 whole rows, an instruction each (store_one)
  if (!halves) {
    const int total = full_tiles * ntn, lo = static_cast<int>(static_cast<int64_t>(total) * xcd / nx),
              end = static_cast<int>(static_cast<int64_t>(total) * (xcd + 1) / nx);
    int u = lo + mine;
    if (u < end) {
      const int wm = (wave >> 2) * 128;
      const uint32_t x0 = base + ((wm + li) * kBK + ((kk ^ fx) << 3)) * 2, x1 = base + ((wm + li) * kBK + (((4 + kk) ^ fx) << 3)) * 2;
      const uint32_t w0 = base + ((256 + wn + rb) * kBK + ((kk ^ fw) << 3)) * 2,
                     w1 = base + ((256 + wn + rb) * kBK + (((4 + kk) ^ fw) << 3)) * 2;
      uint32_t o1[6], o2[2];                                           // this thread's pieces: X rows 0 .. 63 of each 128 and W | the other X rows
      const char* wb;
      int at1 = 0, at2 = 0;
      auto aim1 = [&](const Tile& t) {
#pragma unroll
        for (int j = 0; j < 2; ++j) o1[j] = x_at(t, j * 128 + r);
#pragma unroll
        for (int j = 0; j < 4; ++j) o1[2 + j] = w_at(t, j * 64 + r);
        wb = w_base(t);
        at1 = 0;
      };
      auto aim2 = [&](const Tile& t) {
#pragma unroll
        for (int j = 0; j < 2; ++j) o2[j] = x_at(t, 64 + j * 128 + r);
        at2 = 0;
      };
      auto issue1 = [&](int img) {
#pragma unroll
        for (int j = 0; j < 2; ++j) lds_dma16(a.x, xb + at1 + o1[j], &lds[img * kFull + (j * 128 + wave * 8) * kBK]);
#pragma unroll
        for (int j = 0; j < 4; ++j) lds_dma16(a.w, wb + at1 + o1[2 + j], &lds[img * kFull + (256 + j * 64 + wave * 8) * kBK]);
        at1 += 2 * kBK;
      };
      auto issue2 = [&](int img) {
#pragma unroll
        for (int j = 0; j < 2; ++j) lds_dma16(a.x, xb + at2 + o2[j], &lds[img * kFull + (64 + j * 128 + wave * 8) * kBK]);
        at2 += 2 * kBK;
      };
      Tile cur = place(1, u);
      aim1(cur), aim2(cur);
      issue1(0), issue2(0), issue1(1);
      wait_vm<8>();
      __builtin_amdgcn_s_barrier();
      if (wave >= 4) __builtin_amdgcn_s_barrier();                     // the second group: a phase behind
      int img = 0;
      bool stored = false;                                             // 2 S stores went out ahead of the loads waited for
      while (true) {
        const bool more = u + wgs < end;
        const Tile nxt = place(1, more ? u + wgs : u);                 // (none: loads that nobody reads)
        clear();
        for (int t = 0; t < steps; ++t) {
          const uint32_t o = img * (kFull * 2);
          wide_read_xw(x0 + o, x1 + o, w0 + o, w1 + o, xf, wf);
          if (t == steps - 1) aim2(nxt);
          issue2(img ^ 1);
          if (stored) wait_vm<8 + 2 * S>(); else wait_vm<8>();
          __builtin_amdgcn_s_barrier();
          products(acc[0]);
          __builtin_amdgcn_s_barrier();
          wide_read_x(x0 + o, x1 + o, xf);
          if (t == steps - 2) aim1(nxt);
          issue1(img);
          if (stored) wait_vm<8 + 2 * S>(); else wait_vm<8>();
          stored = false;
          __builtin_amdgcn_s_barrier();
          products(acc[1]);
          __builtin_amdgcn_s_barrier();
          img ^= 1;
        }
        stored = cur.m0 + 256 <= cur.hi && cur.n0 + 256 <= a.n;
        if (stored) emit(acc[0], cur.m0 + wm, cur, true), emit(acc[1], cur.m0 + wm + 64, cur, true);
        else emit(acc[0], cur.m0 + wm, cur, false), emit(acc[1], cur.m0 + wm + 64, cur, false);
        if (!more) break;
        u += wgs, cur = nxt;
      }
      if (wave < 4) __builtin_amdgcn_s_barrier();
      wait_vm<0>();                                                    // (the last loads into LDS: it is used again, or given back)
      __builtin_amdgcn_s_barrier();
    }
  }
  // ---- tiles of 128 x 256
  const int kind = halves ? 3 : 2, total = (halves ? half_tiles : rest_tiles) * ntn;
  const int lo = static_cast<int>(static_cast<int64_t>(total) * xcd / nx), end = static_cast<int>(static_cast<int64_t>(total) * (xcd + 1) / nx);
  // Those that had one large tile less take a small one each ahead of all, then everybody in turn, they first: two small tiles pass
  // beside a large one
  int turn = mine, ahead = wgs;
  if (!halves) {
    const int f = full_tiles * ntn;
    const int had = static_cast<int>(static_cast<int64_t>(f) * (xcd + 1) / nx) - static_cast<int>(static_cast<int64_t>(f) * xcd / nx);
    turn = (mine + wgs - had % wgs) % wgs, ahead = wgs - had % wgs;
  }
  int u = lo + turn + (turn < ahead ? 0 : ahead);
  if (u >= end) return;
  const int wm = (wave >> 2) * 64;
  const uint32_t x0 = base + ((wm + li) * kBK + ((kk ^ fx) << 3)) * 2, x1 = base + ((wm + li) * kBK + (((4 + kk) ^ fx) << 3)) * 2;
  const uint32_t w0 = base + ((128 + wn + rb) * kBK + ((kk ^ fw) << 3)) * 2, w1 = base + ((128 + wn + rb) * kBK + (((4 + kk) ^ fw) << 3)) * 2;
  uint32_t o1[6];
  const char* wb;
  int at1 = 0;
  auto aim = [&](const Tile& t) {
#pragma unroll
    for (int j = 0; j < 2; ++j) o1[j] = x_at(t, j * 64 + r);
#pragma unroll
    for (int j = 0; j < 4; ++j) o1[2 + j] = w_at(t, j * 64 + r);
    wb = w_base(t);
    at1 = 0;
  };
  auto issue = [&](int img) {
#pragma unroll
    for (int j = 0; j < 2; ++j) lds_dma16(a.x, xb + at1 + o1[j], &lds[img * kHalf + (j * 64 + wave * 8) * kBK]);
#pragma unroll
    for (int j = 0; j < 4; ++j) lds_dma16(a.w, wb + at1 + o1[2 + j], &lds[img * kHalf + (128 + j * 64 + wave * 8) * kBK]);
    at1 += 2 * kBK;
  };
  Tile cur = place(kind, u);
  aim(cur);
  issue(0), issue(1);
  wait_vm<6>();
  __builtin_amdgcn_s_barrier();
  if (wave >= 4) __builtin_amdgcn_s_barrier();
  int img = 0;
  bool stored = false;
  while (true) {
    const int v = u + (u - lo < ahead ? ahead : wgs);
    const bool more = v < end;
    const Tile nxt = place(kind, more ? v : u);
    clear();
    for (int t = 0; t < steps; ++t) {
      const uint32_t o = img * (kHalf * 2);
      wide_read_xw(x0 + o, x1 + o, w0 + o, w1 + o, xf, wf);
      if (t == steps - 2) aim(nxt);
      issue(img == 0 ? 2 : img - 1);                                   // step t + 2: what both groups have read of step t - 1
      if (stored) wait_vm<6 + S>(); else wait_vm<6>();
      stored = false;
      __builtin_amdgcn_s_barrier();
      products(acc[0]);
      __builtin_amdgcn_s_barrier();
      img = img == 2 ? 0 : img + 1;
    }
    stored = cur.m0 + 128 <= cur.hi && cur.n0 + 256 <= a.n;
    if (stored) emit(acc[0], cur.m0 + wm, cur, true); else emit(acc[0], cur.m0 + wm, cur, false);
    if (!more) break;
    u = v, cur = nxt;
  }
  if (wave < 4) __builtin_amdgcn_s_barrier();
  wait_vm<0>();
}

// The columns that follow every group's outputs, copied from the group's row of x (a.copy a multiple of 8)
template <typename T>
__global__ __launch_bounds__(256) void group_copy_kernel(GroupGemmArgs a) {
  const int per = a.copy >> 3;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x, m = i / per;
  if (m >= a.rows) return;
  int64_t row = a.perm != nullptr ? MI355_LD(int32_t, a.perm, a.perm + m) : m;
  row = row < 0 ? 0 : (row >= a.x_rows ? a.x_rows - 1 : row);
  const int c = static_cast<int>(i % per) * 8;
  const uint4 v = MI355_LD(uint4, a.x, a.x + row * a.x_stride + a.k + c);
  uint16_t* to = a.y + (m >> 4) * a.y_block + (m & 15) * a.y_stride + a.n + c;
  for (int g = blockIdx.y; g < a.groups; g += gridDim.y) MI355_ST(uint4, a.y, to + g * a.y_group, v);
}

// What the wide tiles take: whole steps of K, 16-byte stores, byte offsets of 32 bits
// (one: a single matrix, whose last outputs may end inside a wave's 64)
static bool wide_fits(const GroupGemmArgs& a, bool trans, bool experts, bool one = false) {
  const int64_t w_rows = experts ? a.n : static_cast<int64_t>(a.n) * a.groups;
  if (a.k % kBK != 0 || a.k < 2 * kBK || a.x_rows * a.x_stride * 2 >= (1ll << 32) || w_rows * a.k * 2 >= (1ll << 32) || a.rows >= (1 << 30) ||
      w_rows >= (1 << 30))
    return false;
  if (a.n % 8 != 0 || a.y_stride % 8 != 0 || a.y_block % 8 != 0 || a.y_group % 8 != 0) return false;
  if (experts) return a.groups <= kWideMaxGroups;
  return a.x_group == 0 && (one || a.n % 64 == 0) && a.w_group == static_cast<int64_t>(a.n) * a.k && (!trans || a.copy == 0);
}

// Where the wide tiles are the faster ones (bf16, us, 128 x 128 tiles / wide; 12 and less are the host's).  They need about
// half a round of 128 x 128 tiles on two workgroups a CU: 32 experts 512 -> 512 of 200 rows 13.7 / 15.6, of 384 rows 18.9 / 17.4,
// 8 experts 512 -> 1536 of 200 rows 13.4 / 16.0, of 384 17.6 / 16.7, 2048 -> 4096 of 128 rows 42 / 33.  Experts of few rows stream their
// weights, and a tile's 128 rows then are mostly padding: 32 experts 2048 -> 4096 of 64 rows 123 / 132, of 128 rows 172 / 154; 128
// experts 2048 -> 512 of 128 rows 94 / 110, of 200 rows 104 / 95.  Outputs that fill little of their last 256 lose it again:
// 32 experts 2048 -> 320 of 1030 rows 78 / 80.  Heads (16 of 512 -> 128, with 64 copied columns, which are a launch of their own
// here): 2000 rows 16.0 / 17.8, 3000 20.1 / 19.4, 8224 48.8 / 40.9; of 128 inputs 4000 rows 14.4 / 18.0.
// A second round of small tiles that is mostly empty costs what the wide ones gain: 64 experts 2048 -> 1024 of 96 rows (about 320 small
// tiles) 86.4 / 99.2, 48 of 1024 -> 1536 (360) 46.6 / 51.4, 64 of 2048 -> 1280 (400) 90.8 / 104.7, but 48 of 1024 -> 1280 (300) 43.6 / 36.9 and
// 64 of 1024 -> 1536 (480) 60.5 / 54.0; and of few inputs, where a tile is mostly its start and end, more: 32 experts 256 -> 2304 of 96 rows
// (360) 21.3 / 24.9, of 200 rows (594) 30.4 / 29.3; 256 -> 4096 of 96 rows (640) 34.3 / 30.0.
static bool wide_pays(const GroupGemmArgs& a, bool experts) {
  const int64_t n = experts ? a.n : static_cast<int64_t>(a.n) * a.groups;
  if (4 * ((n + 255) & ~255ll) > 5 * n) return false;
  if (!experts) return a.k >= 256 && a.rows * n >= 384ll * 128 * 128;
  if (a.rows < (a.groups <= 64 ? 96ll : 160ll) * a.groups || (a.rows + 64ll * a.groups) * n < 288ll * 128 * 128) return false;
  const int64_t small_tiles = (a.rows / 128 + a.groups / 2) * ((n + 255) / 256);
  if (a.groups > 32 && a.rows < 112ll * a.groups && small_tiles > 300 && small_tiles <= 420) return false;
  return a.k > 256 || a.rows >= 192ll * a.groups || small_tiles <= 256 || small_tiles > 512;
}

// Workgroups of the wide kernel for up to `most` tiles: as many on every XCD, since each takes an eighth of the tiles.  With just as many
// workgroups as tiles and no multiple of eight an XCD can have a tile more than workgroups, and the launch a second round: 2048 -> 5184
// of 1500 rows (252 small tiles) 51 us, with 256 workgroups 32; 2048 -> 2112 of 3333 rows 50 and 31.
static dim3 wide_grid(int64_t most) { return dim3(static_cast<unsigned>(most < 256 ? (most + 7) / 8 * 8 : 256)); }

template <typename T>
static void launch_group_gemm(const GroupGemmArgs& a, bool trans, int64_t tiles_m, int bm, hipStream_t s) {
  const bool experts = a.offsets != nullptr;
  if (bm == 128 && wide_fits(a, trans, experts) && wide_pays(a, experts)) {
    GroupGemmArgs b = a;
    if (!experts) b.n = a.n * a.groups, b.groups = 1;
    const int64_t most = (a.rows / 128 + b.groups) * ((b.n + 255) / 256);
    const dim3 grid = wide_grid(most);
    if (trans) hipLaunchKernelGGL((group_gemm_wide_kernel<T, true>), grid, dim3(kWideThreads), 0, s, b, a.n);
    else hipLaunchKernelGGL((group_gemm_wide_kernel<T, false>), grid, dim3(kWideThreads), 0, s, b, a.n);
    if (a.copy > 0)
      hipLaunchKernelGGL(group_copy_kernel<T>, dim3(static_cast<unsigned>((a.rows * (a.copy >> 3) + 255) / 256), 2), dim3(256), 0, s, a);
    return;
  }
#define MI355_GG(BM, BN, MW, TR)                                                                                   \
  hipLaunchKernelGGL((group_gemm_kernel<T, BM, BN, MW, TR>), dim3(static_cast<unsigned>(tiles_m * ((a.n + BN - 1) / BN))), \
                     dim3(256), 0, s, a)
  if (trans) MI355_GG(128, 128, 2, true);
  else if (bm == 32) MI355_GG(32, 64, 1, false);
  else MI355_GG(128, 128, 2, false);
#undef MI355_GG
}

}  // namespace mi355

using namespace mi355;

static int32_t check_group_gemm(const char* name, const GroupGemmArgs& a, int32_t dtype) {
  MI355_REQUIRE(a.y && a.x && a.w, MI355_ERR_INVALID, "%s: null pointer", name);
  MI355_REQUIRE(dtype == MI355_BF16 || dtype == MI355_F16, MI355_ERR_UNSUPPORTED, "%s: 16-bit storage only", name);
  MI355_REQUIRE(a.groups > 0 && a.rows >= 0 && a.n > 0 && a.k > 0 && a.top > 0 && a.x_rows > 0, MI355_ERR_INVALID, "%s: sizes", name);
  MI355_REQUIRE(a.k % 8 == 0 && a.n % 4 == 0 && a.copy >= 0 && a.copy % 8 == 0 && a.x_stride % 8 == 0 && a.x_group % 8 == 0 &&
                    a.w_group % 8 == 0 && a.y_stride % 4 == 0 && a.y_block % 4 == 0 && a.y_group % 4 == 0 && aligned16(a.x) &&
                    aligned16(a.w) && aligned16(a.y),
                MI355_ERR_UNSUPPORTED, "%s: %d inputs (a multiple of 8), %d outputs (of 4), 16-byte aligned rows", name, a.k, a.n);
  MI355_REQUIRE(a.copy == 0 || (a.n % 8 == 0 && a.y_stride % 8 == 0 && a.y_block % 8 == 0 && a.y_group % 8 == 0), MI355_ERR_UNSUPPORTED,
                "%s: copied columns need outputs on 16-byte boundaries", name);
  return MI355_OK;
}

extern "C" int32_t mi355_expert_gemm(void* y, const void* x, int64_t x_rows, const void* w, const int32_t* offsets,
                                     const int32_t* tile_start, const int32_t* perm, int32_t top, int64_t num_rows,
                                     int32_t experts, int32_t out_width, int32_t in_width, int32_t relu2, int32_t dtype,
                                     void* stream) {
  MI355_REQUIRE(offsets && tile_start, MI355_ERR_INVALID, "expert_gemm: null pointer");
  GroupGemmArgs a = {static_cast<uint16_t*>(y), 16ll * out_width, out_width, 0, static_cast<const uint16_t*>(x), in_width, 0, x_rows,
                     perm, top, static_cast<const uint16_t*>(w), static_cast<int64_t>(out_width) * in_width, offsets, tile_start,
                     experts, num_rows, out_width, in_width, 0, relu2};
  const int32_t rc = check_group_gemm("expert_gemm", a, dtype);
  if (rc != MI355_OK || num_rows == 0) return rc;
  const int64_t tiles = num_rows / 128 + experts;        // no fewer than the experts' tiles together
  MI355_REQUIRE(tiles * ((out_width + 127) / 128) <= 0x7FFFFFFF, MI355_ERR_UNSUPPORTED, "expert_gemm: too many tiles");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == MI355_BF16) launch_group_gemm<BF16>(a, false, tiles, 128, s); else launch_group_gemm<F16>(a, false, tiles, 128, s);
  return check_launch("expert_gemm");
}

extern "C" int32_t mi355_linear_act(void* y, int64_t y_stride, const void* x, int64_t x_stride, const void* w, int64_t num_rows,
                                    int32_t out_width, int32_t in_width, int32_t activation, float limit, int32_t dtype, void* stream) {
  MI355_REQUIRE(activation >= MI355_ACT_RELU2 && activation <= MI355_ACT_NONE, MI355_ERR_INVALID, "linear_act: unknown activation %d", activation);
  const bool gated = activation != MI355_ACT_RELU2 && activation != MI355_ACT_NONE;
  GroupGemmArgs a = {static_cast<uint16_t*>(y), 16 * y_stride, y_stride, 0, static_cast<const uint16_t*>(x), x_stride, 0, num_rows,
                     nullptr, 1, static_cast<const uint16_t*>(w), static_cast<int64_t>(out_width) * in_width, nullptr, nullptr, 1,
                     num_rows, out_width, in_width, 0, activation == MI355_ACT_RELU2, limit};
  MI355_REQUIRE(y && x && w, MI355_ERR_INVALID, "linear_act: null pointer");
  MI355_REQUIRE(dtype == MI355_BF16 || dtype == MI355_F16, MI355_ERR_UNSUPPORTED, "linear_act: 16-bit storage only");
  MI355_REQUIRE(num_rows >= 0 && out_width > 0 && in_width > 0, MI355_ERR_INVALID, "linear_act: sizes");
  MI355_REQUIRE(x_stride >= in_width && y_stride >= (gated ? out_width / 2 : out_width), MI355_ERR_INVALID, "linear_act: rows overlap");
  if (num_rows == 0) return MI355_OK;
  MI355_REQUIRE(wide_fits(a, false, false, true) && x_stride % 8 == 0 && (!gated || out_width % 64 == 0) && aligned16(x) && aligned16(w) && aligned16(y),
                MI355_ERR_UNSUPPORTED, "linear_act: %d inputs (a multiple of 64, 128 at least), %d outputs (of 8, gated 64), 16-byte aligned rows, "
                "operands below 4 GB", in_width, out_width);
  const int64_t most = (num_rows / 128 + 1) * ((out_width + 255) / 256);
  const dim3 grid = wide_grid(most);
  hipStream_t s = static_cast<hipStream_t>(stream);
#define MI355_LA(A)                                                                                                            \
  case A:                                                                                                                      \
    if (dtype == MI355_BF16)                                                                                                   \
      hipLaunchKernelGGL((group_gemm_wide_kernel<BF16, false, A>), grid, dim3(kWideThreads), 0, s, a, out_width);              \
    else                                                                                                                       \
      hipLaunchKernelGGL((group_gemm_wide_kernel<F16, false, A>), grid, dim3(kWideThreads), 0, s, a, out_width);               \
    break
  switch (activation == MI355_ACT_NONE ? MI355_ACT_RELU2 : activation) {
    MI355_LA(MI355_ACT_RELU2);                          // (0: the ungated kernel, whose arguments say whether)
    MI355_LA(MI355_ACT_GELU_MUL);
    MI355_LA(MI355_ACT_SILU_MUL);
    MI355_LA(MI355_ACT_LIMITED_MUL);
  }
#undef MI355_LA
  return check_launch("linear_act");
}

extern "C" int32_t mi355_head_gemm(void* y, int64_t y_block, int64_t y_stride, int64_t y_group, const void* x, int64_t x_stride,
                                   int64_t x_group, int64_t x_rows, const int32_t* index, const void* w, int64_t num_rows,
                                   int32_t heads, int32_t out_width, int32_t in_width, int32_t copy, int32_t transposed,
                                   int32_t dtype, void* stream) {
  GroupGemmArgs a = {static_cast<uint16_t*>(y), y_block, y_stride, y_group, static_cast<const uint16_t*>(x), x_stride, x_group, x_rows,
                     index, 1, static_cast<const uint16_t*>(w), static_cast<int64_t>(out_width) * in_width, nullptr, nullptr, heads,
                     num_rows, out_width, in_width, copy, 0};
  const int32_t rc = check_group_gemm("head_gemm", a, dtype);
  if (rc != MI355_OK || num_rows == 0) return rc;
  MI355_REQUIRE(index != nullptr || x_rows >= num_rows, MI355_ERR_INVALID, "head_gemm: fewer rows than asked for");
  MI355_REQUIRE(!transposed || copy == 0, MI355_ERR_INVALID, "head_gemm: no copied columns beside transposed outputs");
  const int bm = num_rows <= 64 && !transposed ? 32 : 128;
  const int64_t tiles = ((num_rows + bm - 1) / bm) * heads;
  MI355_REQUIRE(tiles * ((out_width + 63) / 64) <= 0x7FFFFFFF, MI355_ERR_UNSUPPORTED, "head_gemm: too many tiles");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == MI355_BF16) launch_group_gemm<BF16>(a, transposed != 0, tiles, bm, s);
  else launch_group_gemm<F16>(a, transposed != 0, tiles, bm, s);
  return check_launch("head_gemm");
}
