// True float32 matrix product  C[M,N] = A[M,K] * W[N,K]^T (+ bias[N]),  W as a Linear stores it.
// Every output element sums its K products in index order 0..K-1 in one accumulator, one fused
// multiply-add after the other, so a row's result does not depend on M or on the tile it falls in.
//
// v_mfma_f32_16x16x4_f32 takes float32 operands as they are and forms its four products of an output
// the same way, in order of the inner index with one rounding each: on random, widely scaled, denormal
// and mixed inputs its results have the bits of a chain of fmaf.  So the tiles below run on the matrix
// cores (157 TFLOP/s of float32, twice what single multiply-adds of the vector units reach) and give
// what the plain kernel at the end gives.
//
// What bounds the product: up to 64 rows (a decode step) reading W once; with more rows the matrix
// cores.  With few outputs a block has one chain and little to hide its reads of LDS behind: 8 x 2,048 x 11,008 takes 118 us, of which
// the chain, 32 cycles for four values of K, is 37.
// Both operands come through LDS with loads that put their 16 bytes there directly, several steps of K
// ahead; a row's 16-byte chunks are exchanged by bits of the row's number, so that the 16 rows that one
// operand read touches lie in different banks.  Measured at the 3B decoder's sizes, two layers and the head,
// one step of 164 rows and three of 6 or 7: their products take 3.19 ms instead of the plain kernel's 21.0 ms.
#include "common.h"

#include <type_traits>

typedef float f32x4_t __attribute__((ext_vector_type(4)));

#define TM 64
#define TN 64
#define TK 16

// Any strides and any K: 64x64 tile per block, 16x16 threads, 4x4 outputs per thread, K step 16.
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ A, int lda,
                                                       const float* __restrict__ W, int ldw,
                                                       const float* __restrict__ bias, float* __restrict__ C, int ldc,
                                                       int M, int N, int K) {
  __shared__ float sa[TK][TM + 4];
  __shared__ float sw[TK][TN + 4];
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

  for (int k0 = 0; k0 < K; k0 += TK) {
    // 64 rows x 16 k per operand: 1024 elements, 4 per thread
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int idx = threadIdx.x + 256 * e;
      const int rr = idx / TK, kk = idx % TK;
      const int gm = m0 + rr, gn = n0 + rr, gk = k0 + kk;
      sa[kk][rr] = (gm < M && gk < K) ? A[(size_t)gm * lda + gk] : 0.f;
      sw[kk][rr] = (gn < N && gk < K) ? W[(size_t)gn * ldw + gk] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < TK; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = sa[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = sw[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int gm = m0 + ty * 4 + i;
    if (gm >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gn = n0 + tx * 4 + j;
      if (gn < N) C[(size_t)gm * ldc + gn] = acc[i][j] + (bias ? bias[gn] : 0.f);
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

// WN x WM waves, each with TNW x TMW tiles of 16 outputs (rows of W) by 16 rows of A; K in steps of KT values
// through STAGES stages of LDS.  K a multiple of 4, rows of A and W on 16-byte boundaries.
template <int WN, int WM, int TNW, int TMW, int KT, int STAGES>
__global__ __launch_bounds__(64 * WN * WM) void gemm_f32_mfma_kernel(const float* __restrict__ A, int lda,
                                                                     const float* __restrict__ W, int ldw,
                                                                     const float* __restrict__ bias, float* __restrict__ C,
                                                                     int ldc, int M, int N, int K) {
  constexpr int NWAVES = WN * WM, ROWS_W = 16 * WN * TNW, ROWS_A = 16 * WM * TMW;
  constexpr int CH = KT / 4;                                  // 16-byte chunks of a row of a stage
  constexpr int ROWS_LOAD = 64 / CH;                          // rows one wave's fetch covers (1 KB)
  constexpr int LOADS = (ROWS_W + ROWS_A) / ROWS_LOAD / NWAVES;
  static_assert(LOADS * ROWS_LOAD * NWAVES == ROWS_W + ROWS_A, "the fetches divide evenly among the waves");
  static_assert(ROWS_W % ROWS_LOAD == 0 && ROWS_A % ROWS_LOAD == 0, "a fetch lies in one operand");
  static_assert((STAGES - 2) * LOADS < 64, "the counter's range");
  __shared__ __attribute__((aligned(16))) float stage[STAGES][(ROWS_W + ROWS_A) * KT];
  const int wave = NWAVES == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
  const int wn = wave % WN, wm = wave / WN;
  const int n0 = blockIdx.x * ROWS_W, m0 = blockIdx.y * ROWS_A;
  const float* wbase = W + (size_t)n0 * ldw;
  const float* abase = A + (size_t)m0 * lda;

  // this wave's fetches of a step: rows (wave LOADS + j) ROWS_LOAD ... of the stage, W's rows first.  Place s of row
  // rho holds chunk s ^ (rho mod CH).  A row that does not exist is read from one that does (its sums are not stored).
  uint32_t from[LOADS];
  int chunk[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int rho = (wave * LOADS + j) * ROWS_LOAD + lane / CH;
    chunk[j] = (lane % CH) ^ (rho & (CH - 1));
    if ((wave * LOADS + j) * ROWS_LOAD < ROWS_W) {
      const int n = n0 + rho < N ? rho : 0;
      from[j] = (uint32_t)((size_t)n * ldw * 4);
    } else {
      const int m = m0 + rho - ROWS_W < M ? rho - ROWS_W : 0;
      from[j] = (uint32_t)((size_t)m * lda * 4);
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)&stage[0][0];
  auto issue = [&](int step) {
    const uint32_t at = lds0 + (uint32_t)(step % STAGES) * ((ROWS_W + ROWS_A) * KT * 4) + (uint32_t)wave * (LOADS * 1024);
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      // a chunk beyond K (in the last step) is read from the row's first: it is not multiplied
      const int k = step * KT + 4 * chunk[j];
      const uint32_t bytes = from[j] + (uint32_t)(k < K ? k : 0) * 4;
      if ((wave * LOADS + j) * ROWS_LOAD < ROWS_W) fetch16_to_lds<(WM > 1)>(wbase, bytes, at + j * 1024);
      else fetch16_to_lds<true>(abase, bytes, at + j * 1024);
    }
  };
  f32x4_t acc[TNW][TMW];
#pragma unroll
  for (int n = 0; n < TNW; ++n)
#pragma unroll
    for (int m = 0; m < TMW; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int steps = (K + KT - 1) / KT;
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i)
    if (i < steps) issue(i);
  // With one tile a wave, a step's operands are read from LDS while those of the step before are multiplied: the chain of
  // products of one sum is all there is to hide the reads behind (8 x 2,048 x 11,008: 140 -> 118 us; 64 rows 169 -> 153).  Four waves
  // side by side on many outputs hide it behind each other (22,016 x 2,048: 43.8, so 44.6).
  if constexpr (TNW == 1 && TMW == 1 && WN < 4) {
    float fw[2][CH], fa[2][CH];
    auto read = [&](int s, auto buf) __attribute__((always_inline)) {
      constexpr int B = decltype(buf)::value;
      const float* sw = stage[s % STAGES];
      const float* sa = sw + ROWS_W * KT;
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int row = wn * 16 + r;
        fw[B][c] = sw[row * KT + 4 * (c ^ (row & (CH - 1))) + g];
        const int ra = wm * 16 + r;
        fa[B][c] = sa[ra * KT + 4 * (c ^ ((ROWS_W + ra) & (CH - 1))) + g];
      }
    };
    auto multiply = [&](int s, auto buf) __attribute__((always_inline)) {
      constexpr int B = decltype(buf)::value;
      const int chunks = s + 1 < steps || K % KT == 0 ? CH : (K % KT) / 4;
      if (chunks == CH) {
#pragma unroll
        for (int c = 0; c < CH; ++c) acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[B][c], fa[B][c], acc[0][0], 0, 0, 0);
      } else {
#pragma unroll
        for (int c = 0; c < CH; ++c)       // (unrolled, a branch each: an index at run time would move the operands about)
          if (c < chunks) acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[B][c], fa[B][c], acc[0][0], 0, 0, 0);
      }
    };
    auto step = [&](int s, auto here, auto before) __attribute__((always_inline)) {
      if (s < steps) {
        const int ahead = steps - 1 - s < STAGES - 2 ? steps - 1 - s : STAGES - 2;
        wait_steps<STAGES - 2, LOADS>(ahead);
        __syncthreads();                     // every wave's part of step s is there, and step s - 1 has been read
        if (s + STAGES - 1 < steps) issue(s + STAGES - 1);
        read(s, here);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (s > 0) multiply(s - 1, before);
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    for (int s = 0; s <= steps; s += 2) {
      step(s, even, odd);
      if (s < steps) step(s + 1, odd, even);
    }
  } else {
    for (int s = 0; s < steps; ++s) {
      const int ahead = steps - 1 - s < STAGES - 2 ? steps - 1 - s : STAGES - 2;
      wait_steps<STAGES - 2, LOADS>(ahead);
      __syncthreads();                       // every wave's part of step s is there, and step s - 1 has been multiplied
      if (s + STAGES - 1 < steps) issue(s + STAGES - 1);
      const float* sw = stage[s % STAGES];
      const float* sa = sw + ROWS_W * KT;
      auto multiply = [&](int c) {           // chunk c: four values of K, lane group g has the g-th
        float fw[TNW], fa[TMW];
#pragma unroll
        for (int n = 0; n < TNW; ++n) {
          const int row = (wn * TNW + n) * 16 + r;
          fw[n] = sw[row * KT + 4 * (c ^ (row & (CH - 1))) + g];
        }
#pragma unroll
        for (int m = 0; m < TMW; ++m) {
          const int row = (wm * TMW + m) * 16 + r;
          fa[m] = sa[row * KT + 4 * (c ^ ((ROWS_W + row) & (CH - 1))) + g];
        }
#pragma unroll
        for (int n = 0; n < TNW; ++n)
#pragma unroll
          for (int m = 0; m < TMW; ++m) acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[n], fa[m], acc[n][m], 0, 0, 0);
      };
      if (s + 1 < steps || K % KT == 0) {
#pragma unroll
        for (int c = 0; c < CH; ++c) multiply(c);
      } else {
        for (int c = 0; c < (K % KT) / 4; ++c) multiply(c);
      }
    }
  }
  // a lane holds, of (n, m): row 16 (wm TMW + m) + r of A, outputs 16 (wn TNW + n) + 4 g ...
#pragma unroll
  for (int m = 0; m < TMW; ++m) {
    const int gm = m0 + (wm * TMW + m) * 16 + r;
    if (gm >= M) continue;
#pragma unroll
    for (int n = 0; n < TNW; ++n) {
      const int gn = n0 + (wn * TNW + n) * 16 + 4 * g;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (gn + i < N) C[(size_t)gm * ldc + gn + i] = acc[n][m][i] + (bias ? bias[gn + i] : 0.f);
    }
  }
}

extern "C" int qvl_gemm_f32(const void* A, int lda, const void* W, int ldw, const void* bias, void* C, int ldc, int M,
                            int N, int K, int cus, hipStream_t stream) {
  if (M <= 0 || N <= 0) return QVL_OK;
  if (K <= 0 || lda < K || ldw < K || ldc < N || cus <= 0) return QVL_ERR_SHAPE;
  // 128 rows of W or A from a block's first one lie within 32 bits of bytes
  const bool tiles = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && ((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0 &&
                     lda < (1 << 22) && ldw < (1 << 22);
#define GO(WN, WM, TNW, TMW, KT, STAGES)                                                                             \
  do {                                                                                                               \
    const dim3 grid((N + 16 * WN * TNW - 1) / (16 * WN * TNW), (M + 16 * WM * TMW - 1) / (16 * WM * TMW));             \
    if (grid.y > 65535) return QVL_ERR_LIMIT;                                                                        \
    hipLaunchKernelGGL((gemm_f32_mfma_kernel<WN, WM, TNW, TMW, KT, STAGES>), grid, dim3(64 * WN * WM), 0, stream,    \
                       (const float*)A, lda, (const float*)W, ldw, (const float*)bias, (float*)C, ldc, M, N, K);     \
    return qvl_launch_status();                                                                                      \
  } while (0)
  if (tiles) {
    // Few rows: a block of four waves takes 64 outputs of all rows, so that W is read once, where that fills the
    // device; fewer outputs are spread over blocks of one wave (16 outputs) or, with more than 16 rows, of 32 x 32.
    const bool wide = (long long)N >= 64LL * cus;
    if (M <= 16) {
      if (wide) GO(4, 1, 1, 1, 64, 4);
      GO(1, 1, 1, 1, 64, 9);
    }
    if (M <= 64 && wide) {
      if (M <= 32) GO(4, 1, 1, 2, 64, 3);
      if (M <= 48) GO(4, 1, 1, 3, 64, 4);
      GO(4, 1, 1, 4, 64, 4);
    }
    // The largest tiles of which there are two for every compute unit; the chain of one tile is short only in small ones.
    const long long big = (long long)((N + 127) / 128) * ((M + 127) / 128), mid = (long long)((N + 63) / 64) * ((M + 63) / 64);
    if (big >= 2LL * cus) GO(2, 2, 4, 4, 32, 4);
    if (mid >= 2LL * cus) GO(2, 2, 2, 2, 32, 4);
    GO(2, 2, 1, 1, 32, 4);
  }
#undef GO
  const dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM);
  if (grid.y > 65535) return QVL_ERR_LIMIT;
  hipLaunchKernelGGL(gemm_f32_kernel, grid, dim3(256), 0, stream, (const float*)A, lda, (const float*)W, ldw,
                     (const float*)bias, (float*)C, ldc, M, N, K);
  return qvl_launch_status();
}
