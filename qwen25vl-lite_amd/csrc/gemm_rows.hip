// Products with up to 64 rows: out = X[M, K] . W[N, K]^T, bfloat16 operands, float32 sums, stored as they are, as bfloat16, through
// the gated activation of W's rows (groups of 8 gate and 8 up rows, or all gate rows first), or as one slab of sums for each range of K (those, and
// gated ones of 17 to 64 rows with few rows of W a wave, by a second kernel, whose waves share a step's columns by halves).
//
// What bounds it is reading W once.  A wave owns up to 32 rows of W and all rows of X (operands of
// v_mfma_f32_32x32x16_bf16), eight waves are a block and a block has a compute unit to itself; the rows a wave takes at a time
// are chosen so that all waves of the device have the same number of tiles (37,888 gated outputs on 2,048 waves: one
// round of 10 channels).  Both operands come through LDS in steps of 64 values of K, all 160 KB of it being steps on
// their way: W marked as read once, X out of the L2 for every tile again.  The steps of one tile follow those of the tile
// before, so fetches stay in flight from the first tile to the last.  Where X is in the registers of waves that share
// a tile of W (gemm_resident) it must fit them; here its rows and K are free, and eight waves read it at LDS's rate: 32 rows
// of W a wave for 64 of X keep that below half of what LDS can do.
//
// Per call in a decode step: gate|up of the 7B decoder (37,888 x 3,584), 8 rows, 43.0 us = 6.3 TB/s (gemm_resident, with the
// norm inside, 50), 64 rows (in halves, below) 50.0 = 5.4 TB/s (the library's product 61.2 and the activation's kernel 5.0); of the 72B decoder
// (59,136 x 8,192), 19 rows, 149 = 6.5 TB/s (174 and 4.6); heads of 152,064 x 3,584, 8 rows, 164, 64 rows, 194 (212), x 8,192, 19
// rows, 433 (465).  A plain read of as much reaches 7.3 TB/s.  Four waves a
// block and two blocks a compute unit: 57 for 50; operands read and multiplied in turn, tile after tile of 16 rows: 65.
#include "tile_product.h"

#include <type_traits>

#define ROWS_WAVES 8
#define ROWS_LDS 163840
#define CUT_ROWS 32      // rows of W of a group of waves, where a product is cut along K
#define CUT_GROUPS (CUT_ROWS / 8)

enum { ROWS_BF16 = 0, ROWS_F32 = 1, ROWS_GATED = 2, ROWS_HALVES = 3 };

struct RowsArgs {
  const bf16_t* x;
  long long ldx;
  const bf16_t* w;
  long long ldw;
  void* out;
  long long ldo;
  int M, N, K;
  int per;          // rows of W a wave (in halves: a group of waves) takes at a time (gated: channels)
  int tiles;        // of all of W
  int blocks;       // that share the tiles (of one range of K)
  int rounds;       // tiles of a wave
  int range_steps;  // (halves) steps of 64 values in a range of K; range i has the blocks i * blocks .. and the slab i of out
  long long slab;
  int gelu;
  float alpha, limit, shift;
  int pairs;        // neighbouring results may be stored at once: two of bfloat16, four of a slab
};

// g sigmoid(alpha g) (u + shift); limit > 0: g capped at it, u clamped to +-limit.
__device__ __forceinline__ float clamped_gate(const RowsArgs& p, float g, float u) {
  if (p.limit > 0.f) {
    g = fminf(g, p.limit);
    u = fminf(fmaxf(u, -p.limit), p.limit);
  }
  return g / (1.0f + expf(-p.alpha * g)) * (u + p.shift);
}

// MT column tiles of 32 rows of X; F fetches of 8 rows of W a step and wave: tiles of up to 8 F rows (4 F channels).
template <int MT, int F, int OUT>
__global__ __launch_bounds__(64 * ROWS_WAVES) void gemm_rows_kernel(RowsArgs p) {
  constexpr int W_BYTES = ROWS_WAVES * F * 1024, STAGE = W_BYTES + MT * 4096, STAGES = ROWS_LDS / STAGE;
  // MT = 1: X's four fetches of a step are made by two waves each (the same bytes to the same place), so that every wave
  // waits for as many
  constexpr int X_PLACES = 4 * MT;
  constexpr int HALF = 2 * F;                 // gated: gates among a lane's 4 F sums
  // float32 results: a lane holds one row of W (neighbouring lanes store neighbouring results); else neighbouring rows of W, so
  // that gate and up value meet in a lane and two results of two bytes are stored at once
  constexpr bool X_FIRST = OUT == ROWS_F32, GATED = OUT == ROWS_GATED || OUT == ROWS_HALVES;
  __shared__ __attribute__((aligned(16))) char lds[STAGES * STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, hi = lane >> 5, r = lane & 31;
  auto tile_of = [&](int round) { return (int)(blockIdx.x + round * p.blocks) * ROWS_WAVES + wave; };
  const int ksteps = (p.K + 63) / 64, steps = ksteps * p.rounds;
  const int last_chunks = p.K % 64 ? (p.K % 64) / 8 : 8;     // of a last step, 8 values each
  // row of W behind row i of a tile (-1: there is none).  Gated: row i's sums are number 4 (i / 8) + i mod 4 of the lanes
  // whose hi is (i / 4) mod 2, and the first half of a lane's sums are gates, the others their up values.
  auto w_row = [&](int tile, int i) {
    if (tile >= p.tiles) return -1;
    if (GATED) {
      const int s = 4 * (i >> 3) + (i & 3), up = s >= HALF, j = ((i >> 2) & 1) * HALF + s - up * HALF, c = tile * p.per + j;
      if (j >= p.per || 2 * c >= p.N) return -1;
      return OUT == ROWS_HALVES ? c + up * (p.N / 2) : (c >> 3) * 16 + (c & 7) + 8 * up;
    }
    const int n = tile * p.per + i;
    return (i < p.per && n < p.N) ? n : -1;
  };
  // this lane's fetches: rows 8 j + lane / 8 of the wave's tile, the row's chunk (lane mod 8) ^ ((row / 2) mod 8), and of X
  // row 8 x_place + lane / 8.  A row that does not exist is read from one that does; its sums are not stored.
  uint32_t fw[F];
  auto set_tile = [&](int tile) __attribute__((always_inline)) {
    const int exists = max(w_row(tile, 0), 0);
#pragma unroll
    for (int j = 0; j < F; ++j) {
      const int rho = 8 * j + (lane >> 3);
      int n = w_row(tile, rho);
      if (n < 0) n = exists;
      fw[j] = (uint32_t)n * (uint32_t)p.ldw * 2 + 16 * ((lane & 7) ^ ((rho >> 1) & 7));
    }
  };
  const int x_place = wave % X_PLACES, x_row = 8 * x_place + (lane >> 3);
  const uint32_t fx = (uint32_t)(x_row < p.M ? x_row : 0) * (uint32_t)p.ldx * 2 + 16 * ((lane & 7) ^ ((x_row >> 1) & 7));
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)&lds[0];
  // Blocks begin a tile at different places of K and go round: all at the same place would ask the same few memory
  // channels (rows lie a power of two of bytes apart in wide models; 59,136 x 8,192, 19 rows: 162 us for 200).
  const int turn = (int)((blockIdx.x * 29u) % (unsigned)ksteps);
  int asked = 0, ask_k = 0, ask_round = 0, ask_stage = 0, ask_at = turn;
  auto ask = [&]() __attribute__((always_inline)) {          // the next step's fetches, if there is one
    if (asked >= steps) return;
    if (ask_k == 0) set_tile(tile_of(ask_round));
    const uint32_t at = lds0 + ask_stage * STAGE, k = (uint32_t)ask_at * 128;
    if (last_chunks == 8 || ask_at != ksteps - 1) {
#pragma unroll
      for (int j = 0; j < F; ++j) tp_fetch16_once(p.w, fw[j] + k, at + (wave * F + j) * 1024);
      tp_fetch16(p.x, fx + k, at + W_BYTES + x_place * 1024);
    } else {
      // chunks that lie beyond K are read from the step's first: they are not multiplied
      auto back = [&](int row) { const int c = (lane & 7) ^ ((row >> 1) & 7); return c < last_chunks ? 0u : 16u * c; };
#pragma unroll
      for (int j = 0; j < F; ++j) tp_fetch16_once(p.w, fw[j] + k - back(8 * j + (lane >> 3)), at + (wave * F + j) * 1024);
      tp_fetch16(p.x, fx + k - back(x_row), at + W_BYTES + x_place * 1024);
    }
    ++asked;
    ask_stage = ask_stage + 1 == STAGES ? 0 : ask_stage + 1;
    if (++ask_at == ksteps) ask_at = 0;
    if (++ask_k == ksteps) {
      ask_k = 0;
      ++ask_round;
    }
  };
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i) ask();
  const uint32_t sw = (r >> 1) & 7;
  // rows of a tile beyond its 8 F are not fetched: their operand is another row's, their sums are not stored
  const int wr = r < 8 * F ? r : r - 8 * F;
  const uint32_t wsw = (wr >> 1) & 7;
  // A sum is formed of short runs: the products of a step go to CHAINS sums in turn, and these join the rest every eight steps.
  // What an addition rounds off then stays small: 64 rows x 152,064 x 3,584, error against 64 bits 1.0e-7 of the result, in one chain of
  // 224 products 3.7e-7 (the library's product likewise), for 204 and 205 us.  Joined every two or four steps, the waits for the products show:
  // 37,888 x 3,584 gated, 64 rows, 54 us for 52.
  constexpr int CHAINS = MT == 1 ? 4 : 2;
  tp_f32x16 run[CHAINS][MT], acc[MT];
  auto finish = [&](int round) __attribute__((always_inline)) {
    const int tile = tile_of(round);
    if (tile >= p.tiles) return;
    if constexpr (X_FIRST) {
      const int n = tile * p.per + r;
      if (r >= p.per || n >= p.N) return;
      float* out = reinterpret_cast<float*>(p.out) + n + 4 * hi * p.ldo;
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          if (32 * t + 8 * (i >> 2) + 4 * hi + (i & 3) < p.M) *out = acc[t][i];
          out += (i & 3) == 3 ? 5 * p.ldo : p.ldo;
        }
    } else {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int m = 32 * t + r;
        if (m >= p.M) continue;
        bf16_t* out = reinterpret_cast<bf16_t*>(p.out) + (size_t)m * p.ldo;
        // results in pairs: numbers 2 i and 2 i + 1 of the lane's
#pragma unroll
        for (int i = 0; i < (GATED ? HALF / 2 : HALF); ++i) {
          float v0 = acc[t][2 * i], v1 = acc[t][2 * i + 1];
          if (OUT == ROWS_GATED) {
            v0 = gate_act(v0, p.gelu) * acc[t][HALF + 2 * i];
            v1 = gate_act(v1, p.gelu) * acc[t][HALF + 2 * i + 1];
          } else if (OUT == ROWS_HALVES) {
            v0 = clamped_gate(p, v0, acc[t][HALF + 2 * i]);
            v1 = clamped_gate(p, v1, acc[t][HALF + 2 * i + 1]);
          }
          const int j = GATED ? hi * HALF + 2 * i : 8 * (i >> 1) + 4 * hi + 2 * (i & 1);
          const int n = tile * p.per + j, end = GATED ? p.N / 2 : p.N;
          if (j >= p.per || n >= end) continue;
          if (p.pairs && n + 1 < end) {
            *reinterpret_cast<uint32_t*>(out + n) = (uint32_t)f32_to_bf16(v0) | ((uint32_t)f32_to_bf16(v1) << 16);
          } else {
            out[n] = f32_to_bf16(v0);
            if (n + 1 < end) out[n + 1] = f32_to_bf16(v1);
          }
        }
      }
    }
  };
  // The operands of a step are read from LDS while those of the step before are multiplied: all waves pass a barrier
  // together, so that reading and multiplying would else take turns.
  tp_bf16x8 w8[2][4], x8[2][MT][4];
  int stage = 0, mul_k = turn, mul_left = ksteps, mul_round = 0;
  auto read = [&](auto buf) __attribute__((always_inline)) {
    constexpr int B = decltype(buf)::value;
    const char* pw = lds + stage * STAGE + wave * F * 1024 + wr * 128;
    const char* px = lds + stage * STAGE + W_BYTES + r * 128;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      w8[B][k] = *reinterpret_cast<const tp_bf16x8*>(pw + (((2 * k + hi) ^ wsw) << 4));
#pragma unroll
      for (int t = 0; t < MT; ++t) x8[B][t][k] = *reinterpret_cast<const tp_bf16x8*>(px + t * 4096 + (((2 * k + hi) ^ sw) << 4));
    }
    stage = stage + 1 == STAGES ? 0 : stage + 1;
  };
  auto multiply = [&](auto buf) __attribute__((always_inline)) {
    constexpr int B = decltype(buf)::value;
    if (last_chunks < 8 && mul_k == ksteps - 1) {      // chunks beyond K are no part of the sums
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (2 * k + hi >= last_chunks) {
          w8[B][k] = tp_bf16x8{};
#pragma unroll
          for (int t = 0; t < MT; ++t) x8[B][t][k] = tp_bf16x8{};
        }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        tp_f32x16& c = run[k % CHAINS][t];
        c = X_FIRST ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(x8[B][t][k], w8[B][k], c, 0, 0, 0)
                    : __builtin_amdgcn_mfma_f32_32x32x16_bf16(w8[B][k], x8[B][t][k], c, 0, 0, 0);
      }
    if (++mul_k == ksteps) mul_k = 0;
    if ((--mul_left & 7) == 0) {
      __builtin_amdgcn_sched_barrier(0);      // (a branch: the additions wait for the products, and are not for every step)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        acc[t] += CHAINS == 4 ? (run[0][t] + run[1][t]) + (run[CHAINS - 2][t] + run[CHAINS - 1][t]) : run[0][t] + run[1][t];
#pragma unroll
        for (int c = 0; c < CHAINS; ++c) run[c][t] = tp_f32x16{};
      }
      if (mul_left == 0) {
        finish(mul_round++);
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = tp_f32x16{};
        mul_left = ksteps;
      }
    }
  };
  auto step = [&](int s, auto here, auto before) __attribute__((always_inline)) {
    if (s < steps) {
      tp_wait_steps<STAGES - 2, F + 1>(asked - 1 - s);      // all but the steps asked for behind this one have come
      tp_wait_lds();
      tp_barrier();                           // every wave's part of the step is there, and the step before has been read
      ask();
      read(here);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (s > 0) multiply(before);
  };
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    acc[t] = tp_f32x16{};
#pragma unroll
    for (int c = 0; c < CHAINS; ++c) run[c][t] = tp_f32x16{};
  }
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  for (int s = 0; s <= steps; s += 2) {
    step(s, even, odd);
    if (s < steps) step(s + 1, odd, even);
  }
  tp_wait_fetches<0>();
}

// Gated products of 17 to 64 rows and those cut along K: as above, but the block's waves stand four by two, wave w with the rows of W of group w mod 4
// and the half w / 4 of every step's columns.  LDS gives an operand of X once for up to 64 rows of W instead of 32, and what
// is multiplied is tiles of 16 rows, not 32, so that few of them are empty (22,016 gated rows on 256 blocks are 22 for each group).  The halves' sums meet in
// LDS when all of K has been read; a wave has one set of rows.  A compute unit takes in 30 to 35 GB/s by way of LDS, so nothing is fetched twice:
// a step's fetches of W and X are dealt out one by one, some waves having one more.
//
// Per call, 24 and 64 rows (in brackets waves with rows of their own and all of a step's columns): 22,016 x 2,048 gated 17.6 and 22.3 us (21.4, 27.5), 37,888 x
// 3,584 47.1 and 50.0 (47.0, 51.6); cut, 19 and 64 rows, 3,584 x 18,944 24.8 and 27.7 (26.7, 31.3), 2,048 x 11,008 10.4 and 12.3 (12.1, 13.6), 8,192 x
// 29,568 78.8 and 88.7 (81.8, 101.4), 10,240 x 8,192 30.1 and 32.7 (31.9, 38.1), 3,584 x 3,584 7.3 and 9.1 (8.8, 10.3).  Error against 64 bits of the cut
// products' sums: 0.7 to 1.04e-7 at any number of rows (0.7 to 1.02e-7 up to 32 rows, 0.84 to 1.16e-7 beyond).
// RG: groups of 8 rows of W of a wave; MT: column tiles of 16 rows of X.
template <int RG, int MT, int OUT>
__global__ __launch_bounds__(64 * ROWS_WAVES) void gemm_halves_kernel(RowsArgs p) {
  constexpr bool GATED = OUT == ROWS_GATED || OUT == ROWS_HALVES;
  constexpr int NT = (RG + 1) / 2, W_BYTES = 4 * RG * 1024, STAGE = W_BYTES + MT * 2048;
  constexpr int ALL = 4 * RG + 2 * MT, EACH = ALL / 8, FEW = ALL % 8, F = EACH + (FEW > 0);      // fetches of 8 rows a step: the first FEW waves one more
  constexpr int STAGES = 4, MERGE = 4 * NT * MT * 1024;            // (five steps on their way instead of four are no faster, three slower)
  static_assert(STAGES * STAGE <= ROWS_LDS && MERGE <= STAGES * STAGE, "the halves' sums lie where the steps were");
  __shared__ __attribute__((aligned(16))) char lds[STAGES * STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
  const int group = wave & 3, half = wave >> 2, q = lane >> 3;
  const int range = blockIdx.x / p.blocks, block = blockIdx.x - range * p.blocks;
  const int k_first = range * p.range_steps * 64, k_values = min(p.K - k_first, p.range_steps * 64);
  const int steps = (k_values + 63) / 64, last_chunks = k_values % 64 ? (k_values % 64) / 8 : 8;     // of a last step, 8 values each
  // Outputs (gated: channels) of group i of the block: per of them from (4 block + i) per on.  Row rho of a group is row rho mod 16 of tile rho / 16; of a
  // gated tile, rows 4 j, 4 j + 1 are gates of channels 2 j, 2 j + 1 and rows 4 j + 2, 4 j + 3 their up values: a lane's four sums.
  const int items = GATED ? p.N / 2 : p.N;
  auto w_row = [&](int first, int rho) {
    if (GATED) {
      const int c = min(first + 8 * (rho >> 4) + 2 * ((rho >> 2) & 3) + (rho & 1), min(first + p.per, items) - 1), up = (rho >> 1) & 1;
      return OUT == ROWS_HALVES ? c + up * items : (c >> 3) * 16 + (c & 7) + 8 * up;
    }
    return min(first + rho, min(first + p.per, items) - 1);        // rows that do not exist are read from the last that does
  };
  // A step's fetch i brings 8 rows of W, the 8 RG rows of group 0 first, or behind those of X; wave w makes the fetches w, w + 8, ...
  uint32_t from0[F], chunk[F];
#pragma unroll
  for (int j = 0; j < F; ++j) {
    const int i = wave + 8 * j, of = min(i / RG, 3), x_row = 8 * (i - 4 * RG) + q, rho = i < 4 * RG ? 8 * (i - of * RG) + q : x_row;
    chunk[j] = (lane & 7) ^ ((rho >> 1) & 7);
    const uint32_t row = i < 4 * RG ? (uint32_t)w_row(min((4 * block + of) * p.per, items - 1), rho) * (uint32_t)p.ldw
                                    : (uint32_t)(x_row < p.M ? x_row : 0) * (uint32_t)p.ldx;
    from0[j] = row * 2 + 16 * chunk[j] + (uint32_t)k_first * 2;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)&lds[0];
  const int turn = (int)((blockIdx.x * 29u) % (unsigned)steps);    // (as above)
  int asked = 0, ask_stage = 0, ask_at = turn;
  auto ask = [&]() __attribute__((always_inline)) {
    if (asked >= steps) return;
    const uint32_t at = lds0 + ask_stage * STAGE, k = (uint32_t)ask_at * 128;
    const bool cut = last_chunks < 8 && ask_at == steps - 1;       // chunks beyond K are read from the step's first: they are not multiplied
#pragma unroll
    for (int j = 0; j < F; ++j) {
      const int i = wave + 8 * j;
      if (j == EACH && wave >= FEW) break;
      const uint32_t from = from0[j] + k - (cut && chunk[j] >= (uint32_t)last_chunks ? 16u * chunk[j] : 0u);
      if (i < 4 * RG) tp_fetch16_once(p.w, from, at + i * 1024);
      else tp_fetch16(p.x, from, at + i * 1024);
    }
    ++asked;
    ask_stage = ask_stage + 1 == STAGES ? 0 : ask_stage + 1;
    if (++ask_at == steps) ask_at = 0;
  };
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i) ask();
  // A sum is formed of short runs, as above: the steps' products go to two sums in turn, which join the rest every eight steps (where registers hold
  // one only, every four).
  constexpr int CHAINS = NT * MT <= 12 ? 2 : 1;
  tp_f32x4 run[CHAINS][NT][MT], acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int c = 0; c < MT; ++c) run[0][t][c] = run[CHAINS - 1][t][c] = acc[t][c] = tp_f32x4{0.f, 0.f, 0.f, 0.f};
  // of an operand: row r of 16, chunk 4 half + g
  const uint32_t of = r * 128 + (((4 * half + g) ^ (r >> 1)) << 4);
  tp_bf16x8 w8[2][NT], x8[2][MT];
  int stage = 0, mul_k = turn;
  auto read = [&](auto buf) __attribute__((always_inline)) {
    constexpr int B = decltype(buf)::value;
    const char* from = lds + stage * STAGE + of;
#pragma unroll
    for (int t = 0; t < NT; ++t) w8[B][t] = *reinterpret_cast<const tp_bf16x8*>(from + (group * RG + 2 * t) * 1024);
#pragma unroll
    for (int c = 0; c < MT; ++c) x8[B][c] = *reinterpret_cast<const tp_bf16x8*>(from + W_BYTES + c * 2048);
    stage = stage + 1 == STAGES ? 0 : stage + 1;
  };
  auto multiply = [&](auto buf, bool join) __attribute__((always_inline)) {
    constexpr int B = decltype(buf)::value;
    if (last_chunks < 8 && mul_k == steps - 1 && 4 * half + g >= last_chunks) {      // chunks beyond K are no part of the sums
#pragma unroll
      for (int t = 0; t < NT; ++t) w8[B][t] = tp_bf16x8{};
#pragma unroll
      for (int c = 0; c < MT; ++c) x8[B][c] = tp_bf16x8{};
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int c = 0; c < MT; ++c) {
        tp_f32x4& sum = run[B % CHAINS][t][c];
        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w8[B][t], x8[B][c], sum, 0, 0, 0);
      }
    if (++mul_k == steps) mul_k = 0;
    if (join) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int c = 0; c < MT; ++c) {
          acc[t][c] += CHAINS == 2 ? run[0][t][c] + run[CHAINS - 1][t][c] : run[0][t][c];
          run[0][t][c] = run[CHAINS - 1][t][c] = tp_f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
  };
  auto step = [&](int s, auto here, auto before) __attribute__((always_inline)) {
    if (s < steps) {
      if (FEW > 0 && wave < FEW) tp_wait_steps<STAGES - 2, EACH + 1>(asked - 1 - s);
      else tp_wait_steps<STAGES - 2, EACH>(asked - 1 - s);     // all but the steps asked for behind this one have come
      tp_wait_lds();
      tp_barrier();                          // every wave's part of the step is there, and the step before has been read
      ask();
      read(here);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (s > 0) multiply(before, s % (4 * CHAINS) == 0 || s == steps);
  };
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  for (int s = 0; s <= steps; s += 2) {
    step(s, even, odd);
    if (s < steps) step(s + 1, odd, even);
  }
  tp_wait_fetches<0>();
  tp_wait_lds();
  __syncthreads();                           // the stages have been read: their place is the halves'
  float* sums = reinterpret_cast<float*>(lds) + group * NT * MT * 256 + 4 * lane;
  if (half == 1) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int c = 0; c < MT; ++c) *reinterpret_cast<tp_f32x4*>(sums + (t * MT + c) * 256) = acc[t][c];
  }
  __syncthreads();
  if (half == 1) return;
  const int first = (4 * block + group) * p.per, end = min(first + p.per, items);
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int c = 0; c < MT; ++c) {
      const int m = 16 * c + r;
      const tp_f32x4 v = acc[t][c] + *reinterpret_cast<const tp_f32x4*>(sums + (t * MT + c) * 256);
      if (m >= p.M) continue;
      if constexpr (GATED) {
        const int n = first + 8 * t + 2 * g;
        float v0, v1;
        if (OUT == ROWS_GATED) v0 = gate_act(v[0], p.gelu) * v[2], v1 = gate_act(v[1], p.gelu) * v[3];
        else v0 = clamped_gate(p, v[0], v[2]), v1 = clamped_gate(p, v[1], v[3]);
        bf16_t* out = reinterpret_cast<bf16_t*>(p.out) + (size_t)m * p.ldo + n;
        if (p.pairs && n + 1 < end) {
          *reinterpret_cast<uint32_t*>(out) = (uint32_t)f32_to_bf16(v0) | ((uint32_t)f32_to_bf16(v1) << 16);
        } else {
          if (n < end) out[0] = f32_to_bf16(v0);
          if (n + 1 < end) out[1] = f32_to_bf16(v1);
        }
      } else {
        const int n = first + 16 * t + 4 * g;
        float* out = reinterpret_cast<float*>(p.out) + range * p.slab + (size_t)m * p.ldo + n;
        if (p.pairs && n + 3 < end) {
          *reinterpret_cast<tp_f32x4*>(out) = v;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (n + i < end) out[i] = v[i];
        }
      }
    }
}

static int rows_check(const RowsArgs& p, const void* x, const void* w, const void* out, int cus) {
  if (p.M > 64) return QVL_ERR_LIMIT;
  if (p.K <= 0 || p.K % 8 || p.ldx < p.K || p.ldw < p.K || p.ldx % 8 || p.ldw % 8 || !x || !w || !out || cus <= 0 ||
      ((uintptr_t)x % 16) || ((uintptr_t)w % 16))
    return QVL_ERR_SHAPE;
  // offsets from the first row are 32-bit
  if ((unsigned long long)((p.N - 1) * p.ldw + p.K) * 2 >= 0xffffff00ull || (unsigned long long)((p.M - 1) * p.ldx + p.K) * 2 >= 0xffffff00ull)
    return QVL_ERR_LIMIT;
  return QVL_OK;
}
static int rows_launch(RowsArgs& p, int mode, hipStream_t stream) {
  const int rows = mode >= ROWS_GATED ? 2 * p.per : p.per, fetches = rows <= 16 ? 2 : (rows + 7) / 8;
  const dim3 grid((unsigned)p.blocks), block(64 * ROWS_WAVES);
#define GO(MT, F, OUT) hipLaunchKernelGGL((gemm_rows_kernel<MT, F, OUT>), grid, block, 0, stream, p)
#define PLAIN(MT, F)                            \
  if (mode == ROWS_BF16) GO(MT, F, ROWS_BF16);  \
  else if (mode == ROWS_F32) GO(MT, F, ROWS_F32)
#define MODE(MT, F)                                   \
  PLAIN(MT, F);                                       \
  else if (mode == ROWS_GATED) GO(MT, F, ROWS_GATED); \
  else GO(MT, F, ROWS_HALVES)
  if (p.M <= 32) {
    if (fetches == 2) { MODE(1, 2); }
    else if (fetches == 3) { MODE(1, 3); }
    else { MODE(1, 4); }
  } else {
    if (fetches == 2) { PLAIN(2, 2); else return QVL_ERR_LIMIT; }      // (gated ones of so few rows a wave run in halves)
    else if (fetches == 3) { MODE(2, 3); }
    else { MODE(2, 4); }
  }
#undef MODE
#undef PLAIN
#undef GO
  return qvl_launch_status();
}

// p.per: of a group of waves.
static int halves_launch(RowsArgs& p, int ranges, int mode, hipStream_t stream) {
  const int groups = mode >= ROWS_GATED ? (p.per + 3) / 4 : (p.per + 7) / 8;      // of 8 rows
  const dim3 grid((unsigned)(p.blocks * ranges)), block(64 * ROWS_WAVES);
#define GO(RG, MT, OUT) hipLaunchKernelGGL((gemm_halves_kernel<RG, MT, OUT>), grid, block, 0, stream, p)
#define ROWS(RG, OUT)                          \
  do {                                         \
    if (p.M <= 32) GO(RG, 2, OUT);             \
    else if (p.M <= 48) GO(RG, 3, OUT);        \
    else GO(RG, 4, OUT);                       \
  } while (0)
#define GROUPS(RG)                             \
  case RG:                                     \
    if (mode == ROWS_GATED) ROWS(RG, ROWS_GATED); \
    else ROWS(RG, ROWS_HALVES);                \
    break
  if (mode == ROWS_F32) {
    if (p.M <= 16) GO(CUT_GROUPS, 1, ROWS_F32);
    else ROWS(CUT_GROUPS, ROWS_F32);
    return qvl_launch_status();
  }
  switch (groups) {
    GROUPS(1);
    GROUPS(2);
    GROUPS(3);
    GROUPS(4);
    GROUPS(5);
    GROUPS(6);
    default: return QVL_ERR_LIMIT;
  }
#undef GROUPS
#undef ROWS
#undef GO
  return qvl_launch_status();
}

// x: bfloat16 [M, K], rows ldx apart, M at most 64; w: bfloat16 [N, K], rows ldw apart; both on 16-byte boundaries, K a multiple
// of 8.  mode 0: out bfloat16 [M, N]; 1: float32; 2: W's rows in groups of 8 gate + 8 up, out bfloat16 [M, N / 2] = act(gate) up;
// 3: N / 2 gate rows, then the up rows, out = g sigmoid(alpha g) (u + shift), g capped at limit, u clamped to +-limit.
extern "C" int qvl_gemm_rows(const void* x, long long ldx, const void* w, long long ldw, void* out, long long ldo, int M, int N,
                             int K, int mode, int gelu, float alpha, float limit, float shift, int cus, hipStream_t stream) {
  if (M <= 0 || N <= 0) return QVL_OK;
  if (mode < 0 || mode > 3 || (mode == 2 && N % 16) || (mode == 3 && N % 2) || ldo < (mode >= 2 ? N / 2 : N)) return QVL_ERR_SHAPE;
  RowsArgs p;
  p.x = (const bf16_t*)x; p.ldx = ldx; p.w = (const bf16_t*)w; p.ldw = ldw; p.out = out; p.ldo = ldo;
  p.M = M; p.N = N; p.K = K; p.gelu = gelu; p.alpha = alpha; p.limit = limit; p.shift = shift; p.slab = 0; p.range_steps = (K + 63) / 64;
  const int bad = rows_check(p, x, w, out, cus);
  if (bad) return bad;
  // the fewest rounds over a block a compute unit, then the fewest rows a wave that these rounds need
  const long long items = mode >= 2 ? N / 2 : N, most = mode >= 2 ? 16 : 32, waves = (long long)cus * ROWS_WAVES;
  const long long rounds = (items + most * waves - 1) / (most * waves);
  p.per = (int)((items + rounds * waves - 1) / (rounds * waves));
  if (mode != 1) p.per = (p.per + 1) / 2 * 2;
  p.pairs = ldo % 2 == 0 && (uintptr_t)out % 4 == 0;
  p.tiles = (int)((items + p.per - 1) / p.per);
  p.blocks = min(cus, (p.tiles + ROWS_WAVES - 1) / ROWS_WAVES);
  p.rounds = (p.tiles + p.blocks * ROWS_WAVES - 1) / (p.blocks * ROWS_WAVES);
  // Tiles of at most 24 rows: with more of 32 full the waves do as well without halves (17 to 64 rows: 22,016 x 2,048, 12 rows a wave, 17.6 to 22.4 us in
  // halves for 21.4 to 27.6; 37,888 x 3,584, 20, 47.1 to 50.2 for 47.0 to 52.9; 59,136 x 8,192, 30, 157 to 162 for 152 to 156).
  if (mode >= ROWS_GATED && M > 16 && rounds == 1 && 2 * p.per <= 24) {
    p.per = (int)((items + 4ll * cus - 1) / (4ll * cus));
    p.blocks = (int)((items + 4ll * p.per - 1) / (4ll * p.per));
    p.pairs = p.pairs && p.per % 2 == 0;
    return halves_launch(p, 1, mode, stream);
  }
  return rows_launch(p, mode, stream);
}

// Products whose result is added to something anyway, cut into ranges of K so that every compute unit has a block: out float32
// [ranges, M, N], the sums over each range.  32 rows of W a group of waves: fewer make X's part of what is fetched larger, more make more slabs to write
// and add (3,584 x 18,944, 64 rows: 27.9 us, with 24 rows 30.0, with 48 28.7; 8,192 x 8,192 26.9, 29.5, 28.2).  A range has at least four steps.
struct RowsCut {
  int blocks, range_steps, ranges;
};
static RowsCut rows_cut(int N, int K, int cus) {
  RowsCut c;
  c.blocks = (N + 4 * CUT_ROWS - 1) / (4 * CUT_ROWS);
  const int steps = (K + 63) / 64, want = max(1, cus / c.blocks);
  c.range_steps = max(4, (steps + want - 1) / want);
  c.ranges = (steps + c.range_steps - 1) / c.range_steps;
  return c;
}
// How many slabs qvl_gemm_rows_cut writes (0: it does not take these sizes).
extern "C" int qvl_gemm_rows_ranges(int M, int N, int K, int cus) {
  if (M <= 0 || M > 64 || N <= 0 || K <= 0 || K % 8 || cus <= 0) return 0;
  return rows_cut(N, K, cus).ranges;
}
extern "C" int qvl_gemm_rows_cut(const void* x, long long ldx, const void* w, long long ldw, void* out, int M, int N, int K, int cus,
                                 hipStream_t stream) {
  if (M <= 0 || N <= 0) return QVL_OK;
  RowsArgs p;
  p.x = (const bf16_t*)x; p.ldx = ldx; p.w = (const bf16_t*)w; p.ldw = ldw; p.out = out; p.ldo = N;
  p.M = M; p.N = N; p.K = K; p.gelu = 0; p.alpha = 1.f; p.limit = p.shift = 0.f; p.slab = (long long)M * N;
  const int bad = rows_check(p, x, w, out, cus);
  if (bad) return bad;
  const RowsCut c = rows_cut(N, K, cus);
  p.per = CUT_ROWS;
  p.tiles = 0;
  p.blocks = c.blocks;
  p.range_steps = c.range_steps;
  p.rounds = 1;
  p.pairs = N % 4 == 0 && (uintptr_t)out % 16 == 0;
  return halves_launch(p, c.ranges, ROWS_F32, stream);
}

