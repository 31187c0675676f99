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
// (straight into LDS) has more than a step's time to arrive with only two buffers.  Rows of 128 bytes; the
// 16-byte chunk c of row rho lies at place c ^ ((rho >> 1) & 7), which spreads the 16 rows of an operand read over
// all banks.
//
// Measured on 4,096 x 8,192 x 8,192 with tiles of 256 x 256: 1.48 PFLOP/s; the same tiles with all waves in step and
// one step of prefetch 1.29; the library's product of 8,192 cubed 1.34.
#pragma once
#include "common.h"

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

template <int WN_, int WM_, int NT_, int MT_>
struct Tile {
  static constexpr int WN = WN_, WM = WM_, NT = NT_, MT = MT_;
  static constexpr int BN = 16 * WN * NT, BM = 16 * WM * MT, NH = NT / 2, MH = MT / 2;
  static constexpr int LA = BN / 128, LB = BM / 128;         // fetches of 8 rows a wave has in a region of W, of X
  static constexpr int RA = BN * 64, RB = BM * 64;           // bytes of a region
  static constexpr int BUF = 2 * RA + 2 * RB, LDS = 2 * BUF;
  static_assert(WN * WM == 8 && NT % 2 == 0 && MT % 2 == 0 && BN % 128 == 0 && BM % 128 == 0, "eight waves, whole fetches");

  int wave, lane, g, r, wn, wm;
  uint32_t fa[2][LA], fb[2][LB];   // byte offset of this lane's 16 bytes at K = 0, from W's and from X's base
  uint32_t back;                   // bytes a lane steps back in a last step of 32 values (its chunk lies beyond K)
  tp_f32x4 acc[NT][MT];

  __device__ __forceinline__ Tile() {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lane = threadIdx.x & 63;
    g = lane >> 4;
    r = lane & 15;
    wn = wave % WN;
    wm = wave / WN;
  }
  // chunk of its row that this lane fetches, for the fetch whose rows begin at a multiple of 8
  __device__ __forceinline__ int chunk_of(int rho) const { return (lane & 7) ^ ((rho >> 1) & 7); }
  // w_at(h, rho), x_at(h, rho): byte offset of row rho of region h (rows of a wave's half one after the other,
  // waves in order): of the tile's row w_row(h, rho), x_row(h, rho)
  __device__ static __forceinline__ int w_row(int h, int rho) { return rho / (16 * NH) * (16 * NT) + h * 16 * NH + rho % (16 * NH); }
  __device__ static __forceinline__ int x_row(int h, int rho) { return rho / (16 * MH) * (16 * MT) + h * 16 * MH + rho % (16 * MH); }
  template <typename WAt, typename XAt>
  __device__ __forceinline__ void set_rows(WAt w_at, XAt x_at) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int j = 0; j < LA; ++j) {
        const int rho = (wave * LA + j) * 8 + (lane >> 3);
        fa[h][j] = w_at(h, rho) + 16 * chunk_of(rho);
      }
#pragma unroll
      for (int j = 0; j < LB; ++j) {
        const int rho = (wave * LB + j) * 8 + (lane >> 3);
        fb[h][j] = x_at(h, rho) + 16 * chunk_of(rho);
      }
    }
  }

  // acc = the tile's products over `steps` steps of 64 values from w and x on.  half_last: the last step has 32
  // values only.
  __device__ __forceinline__ void multiply(char* lds, const void* w, const void* x, int steps, bool half_last) {
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[n][m] = tp_f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
    // A fetch asked for beyond the last step brings the last step's values again, to a region nobody reads any
    // more: every step has the same fetches, so the waits can count them.
    auto at_step = [&](int s, uint32_t rho8) {
      const int t = s < steps ? s : steps - 1;
      uint32_t bytes = (uint32_t)t * 128;
      if (half_last && t == steps - 1 && (((uint32_t)lane & 7) ^ ((rho8 >> 1) & 7)) >= 4) bytes -= 64;
      return bytes;
    };
    auto issue_w = [&](int h, int s) {
      const uint32_t at = lds0 + (s & 1) * BUF + h * RA + wave * (LA * 1024);
#pragma unroll
      for (int j = 0; j < LA; ++j) tp_fetch16(w, fa[h][j] + at_step(s, (wave * LA + j) * 8 + (lane >> 3)), at + j * 1024);
    };
    auto issue_x = [&](int h, int s) {
      const uint32_t at = lds0 + (s & 1) * BUF + 2 * RA + h * RB + wave * (LB * 1024);
#pragma unroll
      for (int j = 0; j < LB; ++j) tp_fetch16(x, fb[h][j] + at_step(s, (wave * LB + j) * 8 + (lane >> 3)), at + j * 1024);
    };
    const uint32_t sw = (r >> 1) & 7;
    uint32_t ra[2], rb[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      ra[k] = (uint32_t)((wn * 16 * NH + r) * 128) + (((4 * k + g) ^ sw) << 4);
      rb[k] = (uint32_t)((wm * 16 * MH + r) * 128) + (((4 * k + g) ^ sw) << 4);
    }
    tp_bf16x8 a[NH][2], b0[MH][2], b1[MH][2];
    auto read_w = [&](int h, int s) {
      const char* p = lds + (s & 1) * BUF + h * RA;
#pragma unroll
      for (int i = 0; i < NH; ++i)
#pragma unroll
        for (int k = 0; k < 2; ++k) a[i][k] = *reinterpret_cast<const tp_bf16x8*>(p + ra[k] + i * 2048);
    };
    auto read_x = [&](int h, int s, tp_bf16x8 (*b)[2]) {
      const char* p = lds + (s & 1) * BUF + 2 * RA + h * RB;
#pragma unroll
      for (int i = 0; i < MH; ++i)
#pragma unroll
        for (int k = 0; k < 2; ++k) b[i][k] = *reinterpret_cast<const tp_bf16x8*>(p + rb[k] + i * 2048);
    };
    auto part = [&](int hn, int hm, int k, tp_bf16x8 (*b)[2]) {
#pragma unroll
      for (int n = 0; n < NH; ++n)
#pragma unroll
        for (int m = 0; m < MH; ++m)
          acc[hn * NH + n][hm * MH + m] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[n][k], b[m][k], acc[hn * NH + n][hm * MH + m], 0, 0, 0);
    };
    auto quarter = [&](int hn, int hm, int s, tp_bf16x8 (*b)[2]) {
      part(hn, hm, 0, b);
      if (!half_last || s + 1 < steps) part(hn, hm, 1, b);
    };
    issue_w(0, 0); issue_x(0, 0); issue_x(1, 0); issue_w(1, 0); issue_w(0, 1); issue_x(0, 1); issue_x(1, 1);
    tp_wait_fetches<2 * LA + 3 * LB>();     // the first halves of step 0
    tp_barrier();
    if (wave >= 4) tp_barrier();            // the second group, a phase behind
    for (int s = 0; s < steps; ++s) {
      read_w(0, s);
      read_x(0, s, b0);
      issue_w(1, s + 1);
      tp_wait_fetches<3 * LA + 2 * LB>();   // X's second half of step s (behind it: W1 W0 X0 X1 W1)
      tp_wait_lds();                        // this wave has read: the regions may be filled again
      tp_barrier();
      quarter(0, 0, s, b0);
      tp_barrier();
      read_x(1, s, b1);
      issue_w(0, s + 2);
      tp_wait_fetches<3 * LA + 2 * LB>();   // W's second half of step s
      tp_wait_lds();
      tp_barrier();
      quarter(0, 1, s, b1);
      tp_barrier();
      read_w(1, s);
      issue_x(0, s + 2);
      tp_wait_lds();
      tp_barrier();
      quarter(1, 1, s, b1);
      tp_barrier();
      issue_x(1, s + 2);
      tp_wait_fetches<2 * LA + 3 * LB>();   // the first halves of step s + 1
      tp_barrier();
      quarter(1, 0, s, b0);
      tp_barrier();
    }
    if (wave < 4) tp_barrier();
    tp_wait_fetches<0>();                   // nothing may land in LDS that is no longer this block's
  }
};
