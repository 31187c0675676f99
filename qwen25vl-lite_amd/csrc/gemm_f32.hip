// True float32 matrix product  C[M,N] = A[M,K] * W[N,K]^T (+ bias[N]),  W as a Linear stores it.
// Every output's sum has one order that K alone sets, so a row's result does not depend on M or on the tile it falls
// in: K is cut into at most eight ranges (range_of) and these into runs of 32 values.  A run's products join one
// accumulator that begins at zero, one fused multiply-add after the other, 16 values at a time with k mod 16 in the order 0
// 4 8 12 1 5 9 13 2 6 10 14 3 7 11 15; the runs' sums are added from the range's first to its last, then the ranges'.
//
// v_mfma_f32_16x16x4_f32 takes float32 operands as they are and forms its four products of an output
// in order of the inner index with one rounding each: on random, widely scaled, denormal
// and mixed inputs its results have the bits of a chain of fmaf.  So the tiles below run on the matrix
// cores (157 TFLOP/s of float32, twice what single multiply-adds of the vector units reach) and give
// what the plain kernel at the end gives.  The order within 16 values is that of lanes which each read 16 bytes: lane group g
// holds values 4 g ... 4 g + 3, and the t-th instruction takes the t-th of each.
//
// Why ranges: one chain an output is 32 cycles for four values of K wherever the outputs are few (8 x 2,048 x 11,008: 37 us at
// least, 118 as measured), and cannot be shared out; ranges run in waves and blocks beside each other.  Short
// runs round off less (error against 64 bits at K = 2,048 1.3e-7 of the
// result, one chain 8.1e-7; at 11,008 1.7e-7 and 1.9e-6).  Before and after, weights from memory: 6 x 2,048 x 11,008 118 and 25 us, 6 x 22,016 x
// 2,048 46 and 35 (5.1 TB/s), 6 x 151,936 x 2,048 240 and 202 (6.2 TB/s), 6 x 2,048 x 2,048 25 and 9; 164 x 2,048 x 11,008 193 and 95, 164 x 22,016 x
// 2,048 237 and 201, 700 x 22,016 x 2,048 872 and 588 (107 TFLOP/s).
#include "common.h"

#include <cmath>
#include <type_traits>

typedef float f32x4_t __attribute__((ext_vector_type(4)));

#define TM 64
#define TN 64
#define TK 16
#define MOST_RANGES 8
#define RUN 32
static_assert(RUN == 2 * TK, "the plain kernel joins a run's sums every second step");

// Values of K in a range: an eighth, in steps of 64, 256 at least.
__host__ __device__ __forceinline__ int range_of(int K) {
  const int r = ((K + MOST_RANGES - 1) / MOST_RANGES + 63) / 64 * 64;
  return r < 256 ? 256 : r;
}

// Any strides and any K: 64x64 tile per block, 16x16 threads, 4x4 outputs per thread, K step 16.
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ A, int lda,
                                                       const float* __restrict__ W, int ldw,
                                                       const float* __restrict__ bias, float* __restrict__ C, int ldc,
                                                       int M, int N, int K) {
  __shared__ float sa[TK][TM + 4];
  __shared__ float sw[TK][TN + 4];
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  const int range = range_of(K);
  float run[4][4], acc[4][4], total[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) run[i][j] = acc[i][j] = total[i][j] = 0.f;
  auto join = [](float (&to)[4][4], float (&from)[4][4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        to[i][j] += from[i][j];
        from[i][j] = 0.f;
      }
  };
  // 64 rows x 16 k per operand: 1024 elements, 4 per thread, asked for while the 16 values of k before are multiplied
  const int kk = threadIdx.x % TK, r0 = threadIdx.x / TK;
  const float* pa[4];
  const float* pw[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {       // (rows that do not exist are read from the last one that does; their sums are not stored)
    pa[e] = A + (size_t)min(m0 + r0 + 16 * e, M - 1) * lda;
    pw[e] = W + (size_t)min(n0 + r0 + 16 * e, N - 1) * ldw;
  }
  float va[4], vw[4];
  auto load = [&](int k0) {
    const int gk = min(k0 + kk, K - 1);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      va[e] = pa[e][gk];
      vw[e] = pw[e][gk];
    }
  };
  load(0);
  int next = range;
  for (int k0 = 0; k0 < K; k0 += TK) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sa[kk][r0 + 16 * e] = k0 + kk < K ? va[e] : 0.f;
      sw[kk][r0 + 16 * e] = k0 + kk < K ? vw[e] : 0.f;
    }
    __syncthreads();
    load(k0 + TK);
#pragma unroll
    for (int step = 0; step < TK; ++step) {
      const int kk = 4 * (step & 3) + (step >> 2);
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = sa[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = sw[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) run[i][j] = fmaf(a[i], b[j], run[i][j]);
    }
    __syncthreads();
    if (k0 % RUN != 0) join(acc, run);          // (a run is two steps)
    if (k0 + TK == next) {
      join(total, acc);
      next += range;
    }
  }
  join(acc, run);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int gm = m0 + ty * 4 + i;
    if (gm >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gn = n0 + tx * 4 + j;
      if (gn < N) C[(size_t)gm * ldc + gn] = (total[i][j] + acc[i][j]) + (bias ? bias[gn] : 0.f);
    }
  }
}

// Lane l of the wave puts its 16 bytes at M0 + 16 l of LDS.  KEEP: the lines may stay in the caches (rows
// that other blocks read too); otherwise they are read once.
template <bool KEEP>
__device__ __forceinline__ void fetch16_to_lds(const void* base, uint32_t lane_bytes, uint32_t lds_at) {
  if (KEEP)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_bytes), "s"(base), "s"(lds_at)
                 : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(lane_bytes), "s"(base), "s"(lds_at)
                 : "memory", "m0");
}
// Wait until at most N of this wave's fetches are outstanding (they finish in order).
template <int N>
__device__ __forceinline__ void wait_fetches() {
  static_assert(N < 64, "the counter's range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
}
// The same for a number of steps that is only known at run time, at most MOST, of LOADS fetches each.
template <int MOST, int LOADS>
__device__ __forceinline__ void wait_steps(int ahead) {
  if constexpr (MOST == 0) {
    wait_fetches<0>();
  } else {
    if (ahead >= MOST) wait_fetches<MOST * LOADS>();
    else wait_steps<MOST - 1, LOADS>(ahead);
  }
}

// Up to 16 rows: reading W once is the bound.  A block of eight waves has 8 WF outputs at a time, each wave one of K's
// ranges.  A wave fetches its steps of 32 values ahead through a ring of LDS of its own, across its tiles, W's lines
// whole (8 rows of 128 bytes an instruction) and marked as read once: no barrier stands between a fetch and its use, only
// the sums of the ranges meet once a tile.  XF fetches of 8 rows of A a step.  WF = 1 where that leaves a tile for each compute
// unit at most: one unit fetches some 40 GB/s, so all should (6 x 2,048 x 11,008 with 16 outputs a block, on half of them, 29 us for 25).
#define F32_STREAM_ROWS 16
template <int WF, int XF>
__global__ __launch_bounds__(64 * MOST_RANGES) void gemm_f32_stream_kernel(const float* __restrict__ A, int lda,
                                                                           const float* __restrict__ W, int ldw,
                                                                           const float* __restrict__ bias, float* __restrict__ C,
                                                                           int ldc, int M, int N, int K, int tiles, int groups, int turns,
                                                                           int ranges, int part) {
  constexpr int STEP = 32, ROWS_W = 8 * WF, FETCHES = WF + XF, STAGE = FETCHES * 1024, SUMS = MOST_RANGES * 1024;   // SUMS: bytes of a tile's
  constexpr int STAGES = (163840 - 2 * SUMS) / MOST_RANGES / STAGE;
  __shared__ __attribute__((aligned(16))) char lds[MOST_RANGES * STAGES * STAGE + 2 * SUMS];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
  const int range = range_of(K), group = wave * part >> 16;       // wave / ranges
  const int k_first = (wave - group * ranges) * range, ksteps = group < groups ? (min(K - k_first, range) + STEP - 1) / STEP : 0;
  const int my_tiles = (turns - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x, steps = ksteps * my_tiles;
  char* sums = lds + MOST_RANGES * STAGES * STAGE;
  const char* mine = lds + wave * STAGES * STAGE;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds + wave * STAGES * STAGE;
  // a fetch brings rows 8 j ... 8 j + 7; place s of row rho holds chunk s ^ ((rho / 2) mod 8).  Rows that do not exist are read
  // from ones that do, their sums are not stored; so are chunks beyond K, which the multiplication replaces by zeros.
  const int row8 = lane >> 3;
  auto chunk_at = [&](int j) { return (lane & 7) ^ (((8 * j + row8) >> 1) & 7); };
  uint32_t fa[XF], fw[WF];
#pragma unroll
  for (int j = 0; j < XF; ++j) fa[j] = (uint32_t)min(8 * j + row8, M - 1) * (uint32_t)lda * 4;
  int asked = 0, ask_k = 0, ask_turn = blockIdx.x, ask_stage = 0;
  const float* wbase = W;
  auto ask = [&]() __attribute__((always_inline)) {
    if (asked >= steps) return;
    if (ask_k == 0) {
      const int ask_tile = min(ask_turn * groups + group, tiles - 1);
      wbase = W + (size_t)ask_tile * ROWS_W * ldw;
#pragma unroll
      for (int j = 0; j < WF; ++j) {
        const int n = 8 * j + row8;
        fw[j] = (uint32_t)(ask_tile * ROWS_W + n < N ? n : 0) * (uint32_t)ldw * 4;
      }
    }
    const uint32_t at = lds0 + ask_stage * STAGE;
    const int k0 = k_first + ask_k * STEP;
    auto bytes = [&](int j) {
      const int k = k0 + 4 * chunk_at(j);
      return (uint32_t)(k < K ? k : 0) * 4;
    };
#pragma unroll
    for (int j = 0; j < WF; ++j) fetch16_to_lds<false>(wbase, fw[j] + bytes(j), at + j * 1024);
#pragma unroll
    for (int j = 0; j < XF; ++j) fetch16_to_lds<true>(A, fa[j] + bytes(j), at + (WF + j) * 1024);
    ++asked;
    ask_stage = ask_stage + 1 == STAGES ? 0 : ask_stage + 1;
    if (++ask_k == ksteps) {
      ask_k = 0;
      ask_turn += gridDim.x;
    }
  };
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i) ask();
  f32x4_t acc{0.f, 0.f, 0.f, 0.f};
  const int wr = WF == 1 ? r & 7 : r, xr = XF == 1 ? r & 7 : r;       // (sums of rows twice there are not stored)
  const uint32_t sw = (wr >> 1) & 7, xsw = (xr >> 1) & 7;
  int stage = 0, s = 0;
  for (int i = 0; i < my_tiles; ++i) {
    for (int k = 0; k < ksteps; ++k, ++s) {
      wait_steps<STAGES - 2, FETCHES>(asked - 1 - s);
      __builtin_amdgcn_sched_barrier(0);
      const char* pw = mine + stage * STAGE + wr * 128;
      const char* px = mine + stage * STAGE + WF * 1024 + xr * 128;
      f32x4_t w4[2], x4[2];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        w4[c] = *reinterpret_cast<const f32x4_t*>(pw + (((4 * c + g) ^ sw) << 4));
        x4[c] = *reinterpret_cast<const f32x4_t*>(px + (((4 * c + g) ^ xsw) << 4));
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);       // read: the next fetches go where the step before this one lay
      __builtin_amdgcn_sched_barrier(0);
      ask();
      const int left = K - (k_first + k * STEP);
      if (left < STEP) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
          if (4 * (4 * c + g) >= left) w4[c] = x4[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
      f32x4_t run{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) run = __builtin_amdgcn_mfma_f32_16x16x4f32(w4[c][e], x4[c][e], run, 0, 0, 0);
      acc += run;
      stage = stage + 1 == STAGES ? 0 : stage + 1;
    }
    char* here = sums + (i & 1) * SUMS;
    if (group < groups) {
      *reinterpret_cast<f32x4_t*>(here + wave * 1024 + lane * 16) = acc;
      acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();               // (fetches stay in flight.)  The sums of the tile before the last have been read, too
    __builtin_amdgcn_sched_barrier(0);
    // output n of row m: lane 16 (n / 4) + m holds it as its number n mod 4
    const int m = threadIdx.x >> 4 & 15, n = threadIdx.x & 15;
    for (int at = threadIdx.x >> 8; at < groups; at += 2) {
      const int gn = (((int)blockIdx.x + i * (int)gridDim.x) * groups + at) * ROWS_W + n;
      if (m >= M || n >= ROWS_W || gn >= N) continue;
      const float* q = reinterpret_cast<const float*>(here) + (at * ranges * 64 + (n >> 2) * 16 + m) * 4 + (n & 3);
      float total = 0.f;
      for (int w = 0; w < ranges; ++w) total += q[w * 256];
      C[(size_t)m * ldc + gn] = total + (bias ? bias[gn] : 0.f);
    }
  }
  wait_fetches<0>();
}

// More rows: WN x WM waves, each with TNW x TMW tiles of 16 outputs (rows of W) by 16 rows of A; K in steps of 32 values
// through STAGES stages of LDS, the matrix cores the bound.  Registers and LDS leave room for four blocks a compute unit, which
// hide each other's barriers (1,500 x 2,048 x 11,008: 595 us; tiles of 128 x 128, a block a unit, 757).  A block has all of K's ranges or one (`per`).  slabs: the
// sums of range i go to slab i, so many floats apart; otherwise their sum goes to C.
// ONCE: no other block reads these rows of W.
template <int WN, int WM, int TNW, int TMW, int STAGES, bool ONCE>
__global__ __launch_bounds__(64 * WN * WM, 4) void gemm_f32_tile_kernel(const float* __restrict__ A, int lda,
                                                                     const float* __restrict__ W, int ldw,
                                                                     const float* __restrict__ bias, float* __restrict__ C,
                                                                     int ldc, int M, int N, int K, int per, long long slabs) {
  constexpr int NWAVES = WN * WM, ROWS_W = 16 * WN * TNW, ROWS_A = 16 * WM * TMW, KT = 32;
  constexpr int LOADS = (ROWS_W + ROWS_A) / 8 / NWAVES, STAGE = (ROWS_W + ROWS_A) * KT * 4;
  static_assert(LOADS * 8 * NWAVES == ROWS_W + ROWS_A, "the fetches divide evenly among the waves");
  static_assert((STAGES - 2) * LOADS < 64, "the counter's range");
  __shared__ __attribute__((aligned(16))) char lds[STAGES * STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
  const int wn = wave % WN, wm = wave / WN;
  const int tiles_n = (N + ROWS_W - 1) / ROWS_W, n0 = blockIdx.x % tiles_n * ROWS_W, m0 = blockIdx.x / tiles_n * ROWS_A;
  const float* wbase = W + (size_t)n0 * ldw;
  const float* abase = A + (size_t)m0 * lda;
  const int range = range_of(K), k_first = blockIdx.y * per * range, k_end = min(K, k_first + per * range);

  // this wave's fetches of a step: 8 rows each, W's first.  Place s of row rho holds chunk s ^ ((rho / 2) mod 8).  Rows and
  // chunks that do not exist are read from ones that do.
  uint32_t from[LOADS];
  int chunk[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int rho = (wave * LOADS + j) * 8 + (lane >> 3);
    chunk[j] = (lane & 7) ^ ((rho >> 1) & 7);
    if ((wave * LOADS + j) * 8 < ROWS_W) {
      const int n = n0 + rho < N ? rho : 0;
      from[j] = (uint32_t)((size_t)n * ldw * 4);
    } else {
      const int m = m0 + rho - ROWS_W < M ? rho - ROWS_W : 0;
      from[j] = (uint32_t)((size_t)m * lda * 4);
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  int ask_stage = 0;
  auto issue = [&](int step) __attribute__((always_inline)) {
    const uint32_t at = lds0 + (uint32_t)ask_stage * STAGE + (uint32_t)wave * (LOADS * 1024);
    ask_stage = ask_stage + 1 == STAGES ? 0 : ask_stage + 1;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const int k = k_first + step * KT + 4 * chunk[j];
      const uint32_t bytes = from[j] + (uint32_t)(k < K ? k : 0) * 4;
      if ((wave * LOADS + j) * 8 < ROWS_W) fetch16_to_lds<!ONCE>(wbase, bytes, at + j * 1024);
      else fetch16_to_lds<true>(abase, bytes, at + j * 1024);
    }
  };
  f32x4_t acc[TNW][TMW], total[TNW][TMW];
#pragma unroll
  for (int n = 0; n < TNW; ++n)
#pragma unroll
    for (int m = 0; m < TMW; ++m) acc[n][m] = total[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // a lane holds, of (n, m): row 16 (wm TMW + m) + r of A, outputs 16 (wn TNW + n) + 4 g ...
  auto store = [&](float* to, int ld, const f32x4_t (*v)[TMW], const float* add) __attribute__((always_inline)) {
    const bool fours = ld % 4 == 0 && (uintptr_t)to % 16 == 0;
#pragma unroll
    for (int m = 0; m < TMW; ++m) {
      const int gm = m0 + (wm * TMW + m) * 16 + r;
      if (gm >= M) continue;
#pragma unroll
      for (int n = 0; n < TNW; ++n) {
        const int gn = n0 + (wn * TNW + n) * 16 + 4 * g;
        float* o = to + (size_t)gm * ld + gn;
        f32x4_t x = v[n][m];
        if (add) {
#pragma unroll
          for (int i = 0; i < 4; ++i) x[i] += gn + i < N ? add[gn + i] : 0.f;
        }
        if (fours && gn + 4 <= N) {
          *reinterpret_cast<f32x4_t*>(o) = x;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (gn + i < N) o[i] = x[i];
        }
      }
    }
  };

  const int steps = (k_end - k_first + KT - 1) / KT;
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i)
    if (i < steps) issue(i);
  // Half a step's operands are read from LDS while those of the half before are multiplied: all waves pass a barrier
  // together, so that reading and multiplying would else take turns.
  const uint32_t sw = (r >> 1) & 7;
  f32x4_t w4[2][TNW], x4[2][TMW], run[TNW][TMW];
  int stage = 0, left = min(range, k_end - k_first), slab = blockIdx.y * per;
  auto read = [&](auto half) __attribute__((always_inline)) {
    constexpr int H = decltype(half)::value;
    const char* p = lds + stage * STAGE + r * 128 + (((4 * H + g) ^ sw) << 4);
#pragma unroll
    for (int n = 0; n < TNW; ++n) w4[H][n] = *reinterpret_cast<const f32x4_t*>(p + (wn * TNW + n) * 2048);
#pragma unroll
    for (int m = 0; m < TMW; ++m) x4[H][m] = *reinterpret_cast<const f32x4_t*>(p + (ROWS_W + (wm * TMW + m) * 16) * 128);
  };
  auto multiply = [&](auto half) __attribute__((always_inline)) {
    constexpr int H = decltype(half)::value;
    if (left < KT && 4 * (4 * H + g) >= left) {          // chunks beyond K are no part of the sums
#pragma unroll
      for (int n = 0; n < TNW; ++n) w4[H][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m < TMW; ++m) x4[H][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int n = 0; n < TNW; ++n)
#pragma unroll
        for (int m = 0; m < TMW; ++m)
          run[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w4[H][n][e], x4[H][m][e],
                                                           H == 0 && e == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : run[n][m], 0, 0, 0);
  };
  auto join = [&](f32x4_t (&to)[TNW][TMW], const f32x4_t (&from)[TNW][TMW]) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < TNW; ++n)
#pragma unroll
      for (int m = 0; m < TMW; ++m) to[n][m] += from[n][m];
  };
  constexpr std::integral_constant<int, 0> first{};
  constexpr std::integral_constant<int, 1> second{};
  for (int s = 0; s <= steps; ++s) {
    if (s < steps) {
      const int ahead = steps - 1 - s < STAGES - 2 ? steps - 1 - s : STAGES - 2;
      wait_steps<STAGES - 2, LOADS>(ahead);
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();        // every wave's part of step s is there, and step s - 1 has been read
      __builtin_amdgcn_sched_barrier(0);
      if (s + STAGES - 1 < steps) issue(s + STAGES - 1);
      read(first);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (s > 0) {
      multiply(second);
      join(acc, run);
      left -= KT;
      if (left <= 0) {
        left = min(range, k_end - k_first - s * KT);
        if (slabs) store(C + (slab++) * slabs, N, acc, nullptr);
        join(total, acc);
#pragma unroll
        for (int n = 0; n < TNW; ++n)
#pragma unroll
          for (int m = 0; m < TMW; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
    if (s < steps) {
      __builtin_amdgcn_sched_barrier(0);
      read(second);
      __builtin_amdgcn_sched_barrier(0);
      multiply(first);
      stage = stage + 1 == STAGES ? 0 : stage + 1;
    }
  }
  if (!slabs) store(C, ldc, total, bias);
}

// The ranges' sums, added from the first to the last.
__global__ __launch_bounds__(256) void gemm_f32_add_kernel(const float* __restrict__ sums, int ranges, long long slab,
                                                           const float* __restrict__ bias, float* __restrict__ C, int ldc, int M, int N) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n >= N) return;
  for (int m = blockIdx.y; m < M; m += gridDim.y) {
    const float* p = sums + (size_t)m * N + n;
    float v[MOST_RANGES];
#pragma unroll
    for (int i = 0; i < MOST_RANGES; ++i) v[i] = i < ranges ? p[i * slab] : 0.f;
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < MOST_RANGES; ++i)
      if (i < ranges) total += v[i];
    C[(size_t)m * ldc + n] = total + (bias ? bias[n] : 0.f);
  }
}

// How a product of more than 16 rows is cut: tiles of 64 outputs by 64 rows (by 32 where that is all rows) or of 32 by 32, and a block for all of
// K or one for each range, whose sums a kernel behind then adds.  The estimate is of microseconds: a step of 32 values takes a block `alone`
// where a compute unit has no other and each one `full` where they share its matrix cores; 0.92 more for the first fetches and the stores of each
// round of four blocks a unit; W read and the results written at 8.8 TB/s, which joins that as the root of squares; the adding kernel 1.8 and the slabs
// read at 6.5 TB/s (a cut has to be 4 per cent shorter).  Fitted to 1,326 products of 17 to 1,500 rows, 64 to 80,000 outputs and K of 64 to 11,008, each in all four forms (rms 7 per
// cent): what it chooses takes 0.4 per cent longer than the best on average.  Large tiles alone, cut by their number: 12, most where K or the
// outputs are few (64 x 256 x 256 11 us and 8, 164 x 64 x 11,008 42 and 25).
struct F32Plan {
  int rows_w, rows, per, parts;      // of W and of A in a tile; per: ranges of a block
};
static F32Plan f32_plan(int M, int N, int K, int cus) {
  const int range = range_of(K), ranges = (K + range - 1) / range;
  F32Plan best{};
  double least = 1e300;
  for (int form = 0; form < (ranges > 1 ? 4 : 2); ++form) {
    const bool small = form & 1, cut = form & 2;
    const int rows_w = small ? 32 : 64, rows = small || M <= 32 ? 32 : 64;
    const double full = small ? 0.222 : rows == 32 ? 0.402 : 0.616, alone = small ? 0.406 : rows == 32 ? 0.584 : 0.772;
    const long long tiles = (long long)((N + rows_w - 1) / rows_w) * ((M + rows - 1) / rows);
    const int steps = ((cut ? range : K) + 31) / 32;
    const double blocks = (double)tiles * (cut ? ranges : 1) / cus, sharing = blocks < 8 ? ceil(blocks) : blocks;
    const double results = 4.0 * M * N * (cut ? ranges : 1), memory = (4.0 * N * K + results) / 8.8e6;
    double us = steps * (alone > full * sharing ? alone : full * sharing) + 0.92 * ceil(blocks / 4);
    us = sqrt(us * us + memory * memory);
    if (cut) us = 1.04 * (us + 1.8 + results / 6.45e6);
    if (us < least) {
      least = us;
      best = F32Plan{rows_w, rows, cut ? 1 : ranges, cut ? ranges : 1};
    }
  }
  return best;
}
static bool f32_tiles(int lda, int ldw, int K) {      // 64 rows of W or A from a block's first one lie within 32 bits of bytes
  return K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && lda < (1 << 22) && ldw < (1 << 22);
}

// Floats that qvl_gemm_f32 needs beside its operands (0: none).
extern "C" long long qvl_gemm_f32_scratch(int lda, int ldw, int M, int N, int K, int cus) {
  if (M <= F32_STREAM_ROWS || N <= 0 || K <= 0 || cus <= 0 || !f32_tiles(lda, ldw, K)) return 0;
  const F32Plan p = f32_plan(M, N, K, cus);
  const int range = range_of(K);
  return p.parts > 1 ? (long long)((K + range - 1) / range) * M * N : 0;
}

// scratch: qvl_gemm_f32_scratch floats.
extern "C" int qvl_gemm_f32(const void* A, int lda, const void* W, int ldw, const void* bias, void* C, int ldc, void* scratch, int M,
                            int N, int K, int cus, hipStream_t stream) {
  if (M <= 0 || N <= 0) return QVL_OK;
  if (K <= 0 || lda < K || ldw < K || ldc < N || cus <= 0) return QVL_ERR_SHAPE;
  const float* a = (const float*)A;
  const float* w = (const float*)W;
  const float* b = (const float*)bias;
  if (f32_tiles(lda, ldw, K) && ((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0) {
    if (M <= F32_STREAM_ROWS) {
      const bool narrow = N <= 8 * cus;
      const int tiles = narrow ? (N + 7) / 8 : (N + 15) / 16;
      // Tiles beside each other in a block where there are fewer ranges than waves: as many as make the longest block short, whose unit five
      // waves keep busy (40,000 outputs, 4 rows, K = 256: 32 us with one wave, 14 with five; K = 64 12.8 and 8).
      const int range = range_of(K), ranges = (K + range - 1) / range;
      int groups = 1;
      double least = 1e300;
      for (int n = 1; n * ranges <= MOST_RANGES; ++n) {
        const double cost = (double)(((tiles + n - 1) / n + cus - 1) / cus) * n / (n * ranges < 5 ? n * ranges / 5.0 : 1.0);
        if (cost < least) least = cost, groups = n;
      }
      const int turns = (tiles + groups - 1) / groups, part = 65536 / ranges + 1;
      const dim3 grid(turns < cus ? turns : cus), block(64 * MOST_RANGES);
#define GO(WF, XF) hipLaunchKernelGGL((gemm_f32_stream_kernel<WF, XF>), grid, block, 0, stream, a, lda, w, ldw, b, (float*)C, ldc, M, N, K, tiles, groups, turns, ranges, part)
      if (narrow && M <= 8) GO(1, 1);
      else if (narrow) GO(1, 2);
      else if (M <= 8) GO(2, 1);
      else GO(2, 2);
#undef GO
      return qvl_launch_status();
    }
    const F32Plan p = f32_plan(M, N, K, cus);
    if (p.parts > 1 && !scratch) return QVL_ERR_SHAPE;
    float* to = p.parts > 1 ? (float*)scratch : (float*)C;
    const long long slab = p.parts > 1 ? (long long)M * N : 0;
    const long long tiles_n = (N + p.rows_w - 1) / p.rows_w, tiles_m = (M + p.rows - 1) / p.rows;
    if (tiles_n * tiles_m > 0xffffffffll / 256) return QVL_ERR_LIMIT;      // threads of a grid
    const dim3 grid((unsigned)(tiles_n * tiles_m), p.parts);
#define GO(...) hipLaunchKernelGGL((gemm_f32_tile_kernel<__VA_ARGS__>), grid, dim3(256), 0, stream, a, lda, w, ldw, b, to, ldc, M, N, K, p.per, slab)
    if (p.rows_w == 32) GO(2, 2, 1, 1, 4, false);
    else if (p.rows == 64 && tiles_m == 1) GO(2, 2, 2, 2, 2, true);
    else if (p.rows == 64) GO(2, 2, 2, 2, 2, false);
    else GO(4, 1, 1, 2, 3, true);
#undef GO
    if (p.parts > 1) {
      const int range = range_of(K);
      hipLaunchKernelGGL(gemm_f32_add_kernel, dim3((N + 255) / 256, M < 65535 ? M : 65535), dim3(256), 0, stream, (const float*)scratch, (K + range - 1) / range,
                         slab, b, (float*)C, ldc, M, N);
    }
    return qvl_launch_status();
  }
  const dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM);
  if (grid.y > 65535) return QVL_ERR_LIMIT;
  hipLaunchKernelGGL(gemm_f32_kernel, grid, dim3(256), 0, stream, a, lda, w, ldw, b, (float*)C, ldc, M, N, K);
  return qvl_launch_status();
}
