// The inner loop of products with many rows: a block of eight waves multiplies BN rows of W with BM rows of
// X (both bfloat16, K values a row) on the matrix cores, K in steps of 64.
//
// What bounds it is feeding v_mfma_f32_16x16x32_bf16: with every wave waiting at the same barriers the
// matrix cores idle while operands come out of LDS.  So the waves work in two groups of four, one wave of
// each on every SIMD, that are one phase apart: while one group multiplies (a quarter of its step) the other
// reads its next operands out of LDS and asks for fetches.  The waves of a block stand WN x WM; a wave owns NT x MT
// tiles of 16 x 16 as four quarters of NT / 2 x MT / 2.
//
// A step's operands lie in four regions: W's rows of the waves' first and second halves, X's likewise.  A
// region is fetched again, for the step after next, one phase after its last reader has passed, so a fetch
// (straight into LDS) has more than a step's time to arrive with only two buffers (three or four: no faster).  Rows of 128 bytes; the
// 16-byte chunk c of row rho lies at place c ^ ((rho >> 1) & 7), which spreads the 16 rows of an operand read over
// all banks.
//
// Each phase reads one region: W's first half, X's second, W's second, and X's first of the next step, into registers of
// its own.  With both first halves in one phase that phase's reads take longer than the other group's products, and one
// phase has none.  Steps come in pairs, so that a region's place is a constant.  Both, against one step a round and the halves together:
// 4,096 x 37,888 x 3,584 gated 820 us for 853 (the places alone 834), 2,048 x 3,584 x 18,944 in two ranges 204 for 212, 2,048 x 22,016 x
// 2,048 gated in tiles of 128 x 256 195 for 209, 281 x 2,048 x 2,048 of 128 x 128 9.5 for 10.3.
//
// Measured on 4,096 x 37,888 x 3,584 gated with tiles of 256 x 256: 820 us = 1.36 PFLOP/s; the library's product of 8,192 cubed 1.34.
#pragma once
#include "common.h"

#include <type_traits>

typedef __bf16 tp_bf16x8 __attribute__((ext_vector_type(8)));
typedef float tp_f32x4 __attribute__((ext_vector_type(4)));
typedef float tp_f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ void tp_fetch16(const void* base, uint32_t lane_bytes, uint32_t lds_at) {
  // lane l of the wave puts its 16 bytes at M0 + 16 l of LDS
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_bytes), "s"(base), "s"(lds_at)
               : "memory", "m0");
}
// Wait until at most N of this wave's fetches are outstanding (they finish in order).
template <int N>
__device__ __forceinline__ void tp_wait_fetches() {
  static_assert(N < 64, "the counter's range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
}
__device__ __forceinline__ void tp_wait_lds() { __builtin_amdgcn_s_waitcnt(0xc07f); }
__device__ __forceinline__ void tp_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

// Lane l of the wave puts its 16 bytes at M0 + 16 l of LDS; the lines are not kept in the caches.
__device__ __forceinline__ void tp_fetch16_once(const void* base, uint32_t lane_bytes, uint32_t lds_at) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(lane_bytes), "s"(base), "s"(lds_at)
               : "memory", "m0");
}
// All but the `ahead` steps of LOADS fetches asked for last have come (at most MOST are ahead).
template <int MOST, int LOADS>
__device__ __forceinline__ void tp_wait_steps(int ahead) {
  if constexpr (MOST <= 0) {
    tp_wait_fetches<0>();
  } else {
    if (ahead >= MOST) tp_wait_fetches<MOST * LOADS>();
    else tp_wait_steps<MOST - 1, LOADS>(ahead);
  }
}

// An address that is the same for the whole wave, in scalar registers.
__device__ __forceinline__ const void* tp_uniform(const void* p) {
  const unsigned long long a = (unsigned long long)(uintptr_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return (const void*)(uintptr_t)((unsigned long long)hi << 32 | lo);
}

template <int WN_, int WM_, int NT_, int MT_>
struct Tile {
  static constexpr int WN = WN_, WM = WM_, NT = NT_, MT = MT_;
  static constexpr int BN = 16 * WN * NT, BM = 16 * WM * MT;
  // of a wave's tiles the first half (the larger one) and the second
  static constexpr int N0 = (NT + 1) / 2, N1 = NT / 2, M0 = (MT + 1) / 2, M1 = MT / 2, NH = N0, MH = M0;
  static constexpr int rows_w(int h) { return 16 * WN * (h ? N1 : N0); }         // of a region
  static constexpr int rows_x(int h) { return 16 * WM * (h ? M1 : M0); }
  // fetches of 8 rows a wave has in a region; where they do not divide evenly some rows are fetched twice (the same
  // bytes to the same place), so that all waves wait for as many
  static constexpr int LW0 = (rows_w(0) + 63) / 64, LW1 = (rows_w(1) + 63) / 64, LX0 = (rows_x(0) + 63) / 64, LX1 = (rows_x(1) + 63) / 64;
  static constexpr int BUF = (BN + BM) * 128, LDS = 2 * BUF;
  static_assert(WN * WM == 8 && NT >= 2 && MT >= 2 && LDS <= 163840, "eight waves, two halves, what LDS holds");

  int wave, lane, g, r, wn, wm;
  uint32_t fa[2][LW0], fb[2][LX0];   // byte offset of this lane's 16 bytes at K = 0, from W's and from X's base
  tp_f32x4 acc[NT][MT];

  __device__ __forceinline__ Tile() {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lane = threadIdx.x & 63;
    g = lane >> 4;
    r = lane & 15;
    wn = wave % WN;
    wm = wave / WN;
  }
  // group of 8 rows that this wave's fetch j in a region of `rows` rows brings, L fetches a wave
  template <int L>
  __device__ __forceinline__ int group_of(int j, int rows) const {
    const int i = wave * L + j;
    return rows % (64 * L) == 0 || i < rows / 8 ? i : i - rows / 8;
  }
  // chunk of its row that this lane fetches
  __device__ __forceinline__ int chunk_of(int rho) const { return (lane & 7) ^ ((rho >> 1) & 7); }
  // w_at(h, rho), x_at(h, rho): byte offset of row rho of region h (rows of a wave's half one after the other,
  // waves in order): of the tile's row w_row(h, rho), x_row(h, rho)
  __device__ static __forceinline__ int w_row(int h, int rho) {
    const int n = 16 * (h ? N1 : N0);
    return rho / n * (16 * NT) + h * 16 * N0 + rho % n;
  }
  __device__ static __forceinline__ int x_row(int h, int rho) {
    const int m = 16 * (h ? M1 : M0);
    return rho / m * (16 * MT) + h * 16 * M0 + rho % m;
  }
  template <typename WAt, typename XAt>
  __device__ __forceinline__ void set_rows(WAt w_at, XAt x_at) {
    auto region = [&](auto half) __attribute__((always_inline)) {
      constexpr int h = decltype(half)::value, LW = h ? LW1 : LW0, LX = h ? LX1 : LX0;
#pragma unroll
      for (int j = 0; j < LW; ++j) {
        const int rho = group_of<LW>(j, rows_w(h)) * 8 + (lane >> 3);
        fa[h][j] = w_at(h, rho) + 16 * chunk_of(rho);
      }
#pragma unroll
      for (int j = 0; j < LX; ++j) {
        const int rho = group_of<LX>(j, rows_x(h)) * 8 + (lane >> 3);
        fb[h][j] = x_at(h, rho) + 16 * chunk_of(rho);
      }
    };
    region(std::integral_constant<int, 0>{});
    region(std::integral_constant<int, 1>{});
  }

  // acc = the tile's products over `steps` steps of 64 values from w and x on.  half_last: the last step has 32
  // values only.  meanwhile(): what is done while the first values are on their way.
  struct Nothing {
    __device__ __forceinline__ void operator()() const {}
  };
  template <typename Meanwhile = Nothing>
  __device__ __forceinline__ void multiply(char* lds, const void* w, const void* x, int steps, bool half_last, Meanwhile meanwhile = Meanwhile()) {
    constexpr std::integral_constant<int, 0> I{};
    constexpr std::integral_constant<int, 1> II{};
    w = tp_uniform(w);
    x = tp_uniform(x);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[n][m] = tp_f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
    // A fetch asked for beyond the last step brings the last step's values again, to a region nobody reads any
    // more: every step has the same fetches, so the waits can count them.
    auto at_step = [&](int s, uint32_t rho) {
      const int t = s < steps ? s : steps - 1;
      uint32_t bytes = (uint32_t)t * 128;
      if (half_last && t == steps - 1 && (((uint32_t)lane & 7) ^ ((rho >> 1) & 7)) >= 4) bytes -= 64;
      return bytes;
    };
    auto issue_w = [&](auto half, int s, int buf) __attribute__((always_inline)) {
      constexpr int h = decltype(half)::value, L = h ? LW1 : LW0;
      const uint32_t at = lds0 + buf + h * rows_w(0) * 128;
#pragma unroll
      for (int j = 0; j < L; ++j) {
        const int group = group_of<L>(j, rows_w(h));
        tp_fetch16(w, fa[h][j] + at_step(s, group * 8 + (lane >> 3)), at + group * 1024);
      }
    };
    auto issue_x = [&](auto half, int s, int buf) __attribute__((always_inline)) {
      constexpr int h = decltype(half)::value, L = h ? LX1 : LX0;
      const uint32_t at = lds0 + buf + (BN + h * rows_x(0)) * 128;
#pragma unroll
      for (int j = 0; j < L; ++j) {
        const int group = group_of<L>(j, rows_x(h));
        tp_fetch16(x, fb[h][j] + at_step(s, group * 8 + (lane >> 3)), at + group * 1024);
      }
    };
    const uint32_t sw = (r >> 1) & 7;
    uint32_t chunk[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) chunk[k] = (uint32_t)(r * 128) + (((4 * k + g) ^ sw) << 4);
    tp_bf16x8 a[N0][2], b0[2][M0][2], b1[M1][2];
    auto read_w = [&](auto half, int buf) __attribute__((always_inline)) {
      constexpr int h = decltype(half)::value, N = h ? N1 : N0;
      const char* p = lds + buf + h * rows_w(0) * 128 + wn * (16 * N) * 128;
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int k = 0; k < 2; ++k) a[i][k] = *reinterpret_cast<const tp_bf16x8*>(p + chunk[k] + i * 2048);
    };
    auto read_x = [&](auto half, int buf, auto& b) __attribute__((always_inline)) {
      constexpr int h = decltype(half)::value, M = h ? M1 : M0;
      const char* p = lds + buf + (BN + h * rows_x(0)) * 128 + wm * (16 * M) * 128;
#pragma unroll
      for (int i = 0; i < M; ++i)
#pragma unroll
        for (int k = 0; k < 2; ++k) b[i][k] = *reinterpret_cast<const tp_bf16x8*>(p + chunk[k] + i * 2048);
    };
    auto quarter = [&](auto half_n, auto half_m, int s, auto& b) __attribute__((always_inline)) {
      constexpr int hn = decltype(half_n)::value, hm = decltype(half_m)::value;
      auto part = [&](int k) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < (hn ? N1 : N0); ++n)
#pragma unroll
          for (int m = 0; m < (hm ? M1 : M0); ++m)
            acc[hn * N0 + n][hm * M0 + m] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[n][k], b[m][k], acc[hn * N0 + n][hm * M0 + m], 0, 0, 0);
      };
      part(0);
      if (!half_last || s + 1 < steps) part(1);
    };
    // One step; its first half of X is in b already, the next step's goes to b_next.
    auto step = [&](int s, int here, auto& b, auto& b_next) __attribute__((always_inline)) {
      const int other = BUF - here;
      read_w(I, here);
      issue_w(II, s + 1, other);
      tp_wait_fetches<LW1 + LW0 + LX0 + LX1 + LW1>();   // X's second half of step s (behind it: W1 W0 X0 X1 W1)
      tp_wait_lds();                        // this wave has read: the regions may be filled again
      tp_barrier();
      quarter(I, I, s, b);
      tp_barrier();
      read_x(II, here, b1);
      issue_w(I, s + 2, here);
      tp_wait_fetches<LW0 + LX0 + LX1 + LW1 + LW0>();   // W's second half of step s
      tp_wait_lds();
      tp_barrier();
      quarter(I, II, s, b1);
      tp_barrier();
      read_w(II, here);
      issue_x(I, s + 2, here);
      tp_wait_fetches<LX1 + LW1 + LW0 + LX0>();         // the first halves of step s + 1
      tp_wait_lds();
      tp_barrier();
      quarter(II, II, s, b1);
      tp_barrier();
      read_x(I, other, b_next);             // (behind the last step: what lies there, for nothing)
      issue_x(II, s + 2, here);
      tp_wait_lds();
      tp_barrier();
      quarter(II, I, s, b);
      tp_barrier();
    };
    issue_w(I, 0, 0); issue_x(I, 0, 0); issue_x(II, 0, 0); issue_w(II, 0, 0); issue_w(I, 1, BUF); issue_x(I, 1, BUF); issue_x(II, 1, BUF);
    if constexpr (!std::is_same<Meanwhile, Nothing>::value) {
      __builtin_amdgcn_sched_barrier(0);
      meanwhile();
      __builtin_amdgcn_sched_barrier(0);
    }
    tp_wait_fetches<LX1 + LW1 + LW0 + LX0 + LX1>();     // the first halves of step 0
    tp_barrier();
    if (wave >= 4) tp_barrier();            // the second group, a phase behind
    read_x(I, 0, b0[0]);
    for (int s = 0; s < steps; s += 2) {
      step(s, 0, b0[0], b0[1]);
      if (s + 1 < steps) step(s + 1, BUF, b0[1], b0[0]);
    }
    if (wave < 4) tp_barrier();
    tp_wait_fetches<0>();                   // nothing may land in LDS that is no longer this block's
  }
};
