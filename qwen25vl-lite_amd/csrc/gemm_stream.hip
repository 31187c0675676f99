// Products with up to 16 rows: X[M, K] . W[N, K]^T, bfloat16 operands, float32 sums, of which every block forms its share of the
// outputs over all of K: a wave has an eighth of K and all of the block's rows of W.  The results are added to the float32 residual, or go
// through the gated activation.
//
// What bounds it is reading W once.  Every compute unit has one block with as many rows of W as the others (11,008 gated channels
// on 256 units: 43 each, 3,584 outputs: 14), whose sums a wave keeps in registers, tiles of 16 rows in a row, while it goes
// through its columns 64 at a time.  Operands come through a ring of LDS places of 2 KB (whole lines) that belongs to the
// wave: it waits for its own fetches only and asks for the next as soon as a place has been read, so nothing is waited for from the
// first fetch to the last and the waves meet once, when their sums are added in wave order.  X's columns come through the same ring,
// once for all of the block's rows.  Few places do. Two, three and four a wave where it has one tile of
// outputs: 3,584 x 18,944, 8 rows 26.0 us, 23.9, 24.8, 16 rows 30.9, 28.0, 28.7; 2,048 x 11,008, 8 rows 11.6, 11.1, 11.4, 16 rows 16.9, 13.2, 13.6; 3,584 x
// 3,584, 1 row 7.3, 7.0, 7.0: there it has three. With more tiles three and four are the same within 2 per cent either way (22,016 x 2,048 gated, 1 row 17.6
// and 17.9, 59,136 x 8,192, 16 rows 147.3 and 146.4), and it has four.
//
// The norm between two products of a layer has no kernel of its own.  Where the residual is formed here its new rows are left times the next
// norm's gain, with each block's sums of their squares; the product behind the norm takes these rows and divides its sums by
// the rows' root mean squares (the scale of a row is a factor of all of its products).
//
// Measured in a captured sequence of calls on fresh weights, microseconds (in brackets what stood there before): 3,584 x 18,944 into the residual, 1 row 23.0, 8
// rows 24.1, 16 rows 28.3 (in slabs 25.4, 24.8, 25.5 and the norm that adds them 3.6 to 4.8); 2,048 x 11,008 10.0, 10.9 (10.7, 11.1 and the norm);
// 8,192 x 8,192 24.9, 24.7, 24.6 (28.3, 29.8, 26.2 and the norm); 3,584 x 3,584 6.9, 7.1, 8.0 (gemm_resident 7.7, 8.2, 9.1); 2,048 x 2,048 4.4, 4.6; gated
// 22,016 x 2,048 17.7 to 18.4 (with the norm inside gemm_resident 20.8 to 23.8, gemm_rows behind a norm 22.3 to 23.6); 37,888 x 3,584 43.7 to 45.0
// (47.2 to 48.0); 59,136 x 8,192 148 to 149 (149 to 150).  A plain read takes 8.0 for 45 MB, 15.2 for 90, 22 for 136 and 41 for 272.
// A decode step of 8 layers, 3B sizes, 1 row: 457 us for 511; 7B, 8 rows: 970 for 1,038.
#include "tile_product.h"

#define STREAM_WAVES 8
#define ITEM 2048                                  // bytes of a place of a wave's ring, two fetches
#define STREAM_EXTRA 16384
#define STREAM_PARTS 256                           // places of a row's sums of squares

enum { STREAM_INTO = 0, STREAM_GATED = 1 };

struct StreamArgs {
  const bf16_t* x;        // [M, K], rows ldx apart
  const bf16_t* w;        // [N, K], rows ldw apart
  long long ldx, ldw;
  int M, N, K;
  int items;              // outputs (gated: channels), dealt out evenly to the blocks
  int runs;               // a wave's groups follow each other (else wave w has groups w, w + 8, ...)
  long long t_step, h_step;   // bytes of W between tiles, and between the halves of a tile
  // The rows of X are rows of the sum times a norm's gain, not yet divided by their root mean square: row m's squares add up to those
  // of squares[m * STREAM_PARTS ...], `parts` of them (null: X is as it is)
  const float* squares;
  int parts;
  float eps;
  // STREAM_INTO: h += product; the new rows are then left for the product behind the next norm: times `gain` as bfloat16 in `left`, with
  // every block's sum of squares in left_squares[m * STREAM_PARTS + block] (null: not)
  float* h;
  long long ldh;
  const float* gain;
  bf16_t* left;
  float* left_squares;
  bf16_t* out;            // gated: rows ldo apart
  long long ldo;
  int gelu;
};

// The wave's oldest S items have come; `waiting`: how many it has asked for and not read.
template <int RING, int S>
__device__ __forceinline__ void stream_wait(int waiting) {
  static_assert(RING <= 4 && S <= RING, "the steps below");
  if (waiting == RING) {
    tp_wait_fetches<2 * (RING - S)>();
  } else {                                         // the last round through the ring
    const int younger = waiting - S;
    if (younger >= 2) tp_wait_fetches<4>();
    else if (younger >= 1) tp_wait_fetches<2>();
    else tp_wait_fetches<0>();
  }
  __builtin_amdgcn_sched_barrier(0);
}

// An item is 16 rows of 64 columns (two fetches of 8 rows), or with fewer rows more columns: X's items are 4 rows of 256 columns (XR = 4), 8 of 128
// (8) or 16 of 64 (twice with NARROW); W's are NT tiles of 16 rows (gated: 8 channels), with NARROW one of 8 rows and 128 columns.  A
// group is XU steps of 64 columns: X's items, then W's of one step after the other.
template <int NT, int XR, int OUT, bool NARROW>
__global__ __launch_bounds__(64 * STREAM_WAVES) void gemm_stream_kernel(StreamArgs p) {
  constexpr bool GATED = OUT == STREAM_GATED;
  constexpr int XU = XR == 4 ? 4 : XR == 8 || NARROW ? 2 : 1, XS = NARROW && XR == 16 ? 2 : 1;
  constexpr int WU = NARROW ? 2 : 1;                               // steps of an item of W
  constexpr int GROUP = XS + XU / WU * NT;                         // items of a group
  constexpr int RING = OUT == STREAM_INTO && NT == 1 ? 3 : 4;       // places of a wave's ring
  constexpr int SUMS = STREAM_WAVES * NT * 1024, RINGS = STREAM_WAVES * RING * ITEM, PLACE = SUMS > RINGS ? SUMS : RINGS;
  static_assert(!(NARROW && (GATED || NT > 1)) && PLACE + STREAM_EXTRA <= 163840, "what is built");
  __shared__ __attribute__((aligned(16))) char lds[PLACE + STREAM_EXTRA];
  float* extra = reinterpret_cast<float*>(lds + PLACE);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
  const int first = (int)((long long)p.items * blockIdx.x / gridDim.x), end = (int)((long long)p.items * (blockIdx.x + 1) / gridDim.x);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)&lds[0], ring0 = lds0 + wave * RING * ITEM;

  // ---- what the epilogue reads, asked for first --------------------------------------------------
  // INTO: thread -> (row em of X, row enl of a tile): the old sum and the gain of every second tile
  constexpr int ENDS = OUT == STREAM_INTO ? (NT * 256 + 511) / 512 : 1;
  float old[ENDS], gain[ENDS];
  const int em = (threadIdx.x >> 4) & 15, enl = threadIdx.x & 15;
  if constexpr (OUT == STREAM_INTO) {
#pragma unroll
    for (int i = 0; i < ENDS; ++i) {
      const int n = first + 16 * (2 * i + (threadIdx.x >> 8)) + enl;
      const bool live = em < p.M && n < end;
      old[i] = live ? p.h[em * p.ldh + n] : 0.f;
      gain[i] = live && p.gain ? p.gain[n] : 0.f;
    }
  }
  if (p.squares) {
    for (int m = wave; m < p.M; m += STREAM_WAVES)
      tp_fetch16(p.squares, (uint32_t)m * STREAM_PARTS * 4 + lane * 16, lds0 + PLACE + m * 1024);
  }

  // ---- the stream: groups of 64 XU columns, wave w takes groups w, w + 8, ... ---------------------
  // Blocks begin at different places and go round: all at the same place would ask the same few memory channels.
  const int groups = (p.K + 64 * XU - 1) / (64 * XU);
  const int w_first = (int)((long long)groups * wave / STREAM_WAVES);
  const int mine = p.runs ? (int)((long long)groups * (wave + 1) / STREAM_WAVES) - w_first : (groups - wave + STREAM_WAVES - 1) / STREAM_WAVES;
  const int turn = mine > 0 ? (int)((blockIdx.x * 29u) % (unsigned)mine) : 0;
  auto column_of = [&](int i) { return (p.runs ? w_first + i : wave + STREAM_WAVES * i) * 64 * XU; };      // first of the wave's group i
  // Where rows have 128 bytes, row rho's 16-byte chunk c lies at place c ^ ((rho >> 1) & 7), with 256 bytes at c ^ 4 rho: the rows of an
  // operand read touch all banks.
  const int q = lane >> 3;
  const uint32_t chunk0 = 16 * ((lane & 7) ^ (q >> 1)), chunk1 = NARROW ? chunk0 + 128 : chunk0 ^ 64;      // of an item's fetches
  auto row_of = [&](int c) { return (OUT == STREAM_GATED ? (uint32_t)((c >> 3) * 16 + (c & 7)) : (uint32_t)c) * (uint32_t)p.ldw * 2; };
  // rows that do not exist are read from the last that does
  const uint32_t body = row_of(first + (NT > 1 ? q : 0));
  const uint32_t tail0 = row_of(min(GATED ? first + 8 * (NT - 1) + q : first + 16 * (NT - 1) + q, end - 1));
  const uint32_t tail1 = GATED || NARROW ? tail0 : row_of(min(first + 16 * (NT - 1) + 8 + q, end - 1));
  const uint32_t body0 = body + chunk0, body1 = body + chunk1, last0 = tail0 + chunk0, last1 = tail1 + chunk1;
  const uint32_t x_chunk0 = XR == 4 ? 16 * ((lane & 15) ^ (4 * (lane >> 4))) : chunk0;
  const uint32_t x_chunk1 = XR == 4 ? x_chunk0 + 256 : XR == 8 ? chunk0 + 128 : chunk0 ^ 64;
  auto x_row = [&](int m) { return (uint32_t)(m < p.M ? m : 0) * (uint32_t)p.ldx * 2; };
  const uint32_t x0 = x_row(XR == 4 ? lane >> 4 : q) + x_chunk0, x1 = x_row(XR == 4 ? lane >> 4 : XR == 8 ? q : 8 + q) + x_chunk1;
  int a_left = mine * GROUP, a_pos = 0, a_t = 0, a_turn = turn, a_at = 0, waiting = 0, a_col = column_of(turn);
  const char* a_w = reinterpret_cast<const char*>(p.w + a_col);      // W's columns of the step
  const char* a_tile = a_w;
  // (K ends in a group: chunks beyond it are read from the group's first column, and not multiplied)
  auto inside = [&](uint32_t from, uint32_t chunk, int step) {
    return a_col + 64 * step + (int)(chunk >> 1) < p.K ? from : from - chunk - 128 * step;
  };
  auto ask = [&]() __attribute__((always_inline)) {
    if (a_left == 0) return;
    --a_left;
    ++waiting;
    const uint32_t at = ring0 + a_at;
    a_at = a_at == (RING - 1) * ITEM ? 0 : a_at + ITEM;
    const bool cut = a_col + 64 * XU > p.K;
    if (a_pos < XS) {
      uint32_t f0 = x0, f1 = x1;
      const int step = XS == 2 ? a_pos : 0;          // 16 rows of 64 columns twice
      if (XS == 2) f0 += 128 * step, f1 += 128 * step;
      if (cut) f0 = inside(f0, x_chunk0, step), f1 = inside(f1, x_chunk1, step);
      const void* base = tp_uniform(p.x + a_col);
      tp_fetch16(base, f0, at);
      tp_fetch16(base, f1, at + 1024);
      ++a_pos;
    } else {
      uint32_t f0 = body0, f1 = body1;
      const char *base0 = a_tile, *base1 = NT > 1 ? a_tile + p.h_step : a_tile;
      if (a_t == NT - 1) {
        f0 = last0;
        f1 = last1;
        base0 = a_w;
        base1 = GATED ? a_w + p.h_step : a_w;
      }
      if (cut) {
        // (what is taken off reaches back to the group's first column: the steps before this one's lie in the offset, not in the base)
        const int step = XU / WU > 1 ? (a_pos - XS) / NT * WU : 0, skipped = 128 * step;
        base0 -= skipped;
        base1 -= skipped;
        f0 = inside(f0 + skipped, chunk0, step);
        f1 = inside(f1 + skipped, chunk1, step);
      }
      tp_fetch16_once(tp_uniform(base0), f0, at);
      tp_fetch16_once(tp_uniform(base1), f1, at + 1024);
      a_tile += p.t_step;
      ++a_pos;
      if (++a_t == NT) {
        a_t = 0;
        a_w += 128 * WU;
        a_tile = a_w;
        if (a_pos == GROUP) {
          a_pos = 0;
          a_turn = a_turn + 1 == mine ? 0 : a_turn + 1;
          a_col = column_of(a_turn);
          a_w = a_tile = reinterpret_cast<const char*>(p.w + a_col);
        }
      }
    }
  };
  for (int i = 0; i < RING; ++i) ask();
  if (p.squares) {
    // one over a row's root mean square, where the row's squares are (the first the wave has asked for)
    if (waiting == RING) tp_wait_fetches<2 * RING>();
    else tp_wait_fetches<0>();
    __builtin_amdgcn_sched_barrier(0);
    for (int m = wave; m < p.M; m += STREAM_WAVES) {
      const float4 v = *reinterpret_cast<const float4*>(extra + m * 256 + 4 * lane);
      const int have = p.parts - 4 * lane;
      const float s = wave_sum(((have > 0 ? v.x : 0.f) + (have > 1 ? v.y : 0.f)) + ((have > 2 ? v.z : 0.f) + (have > 3 ? v.w : 0.f)));
      if (lane == 0) extra[m * 256] = 1.0f / sqrtf(s / (float)p.K + p.eps);
    }
  }

  // ---- the sums ------------------------------------------------------------------------------------
  // A sum is formed of runs of 8 products (256 values of K): one chain over all of a wave's K rounds off a third more.
  tp_f32x4 acc[NT], run[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = run[t] = tp_f32x4{0.f, 0.f, 0.f, 0.f};
  int m_turn = turn;
  uint32_t at = 0;                                 // of the item to read next, in the wave's ring
  auto next = [&](uint32_t from) { return from == (RING - 1) * ITEM ? 0u : from + ITEM; };
  const char* ring = lds + wave * RING * ITEM;
  // places of this lane's operand of the first 32 columns of a step: 16 rows of 128 bytes, 8 of 128, 4 of 256; of the second 32 columns: ^ 64
  const uint32_t of16 = r * 128 + ((g ^ (r >> 1)) << 4), of8 = (r & 7) * 128 + ((g ^ ((r >> 1) & 3)) << 4), of4 = (r & 3) * 256 + ((g ^ ((r & 3) << 2)) << 4);
  auto operand = [&](uint32_t place) { return *reinterpret_cast<const tp_bf16x8*>(ring + place); };
  for (int i = 0; i < mine; ++i) {
    const int left = p.K - column_of(m_turn);                  // columns of the group that exist
    m_turn = m_turn + 1 == mine ? 0 : m_turn + 1;
    const bool cut = left < 64 * XU;
    tp_bf16x8 x[XU][2];
    stream_wait<RING, XS>(waiting);
#pragma unroll
    for (int u = 0; u < XU; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if constexpr (XR == 4) x[u][j] = operand(at + (u >> 1) * 1024 + (of4 ^ ((u & 1) * 128) ^ (j * 64)));
        else if constexpr (XR == 8) x[u][j] = operand(at + u * 1024 + (of8 ^ (j * 64)));
        else x[u][j] = operand((u == 0 ? at : next(at)) + (of16 ^ (j * 64)));
      }
    at = next(at);
    if (XS == 2) at = next(at);
    tp_wait_lds();
    __builtin_amdgcn_sched_barrier(0);
    if (cut) {
#pragma unroll
      for (int u = 0; u < XU; ++u)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          if (64 * u + 32 * j + 8 * g >= left) x[u][j] = tp_bf16x8{};
    }
    waiting -= XS;
#pragma unroll
    for (int s = 0; s < XS; ++s) ask();
#pragma unroll
    for (int u = 0; u < XU; u += WU)
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        stream_wait<RING, 1>(waiting);
        tp_bf16x8 a[WU][2];
#pragma unroll
        for (int v = 0; v < WU; ++v)
#pragma unroll
          for (int j = 0; j < 2; ++j) a[v][j] = operand(at + (NARROW ? v * 1024 + (of8 ^ (j * 64)) : of16 ^ (j * 64)));
        at = next(at);
        tp_wait_lds();
        __builtin_amdgcn_sched_barrier(0);
        if (cut) {
#pragma unroll
          for (int v = 0; v < WU; ++v)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              if (64 * (u + v) + 32 * j + 8 * g >= left) a[v][j] = tp_bf16x8{};
        }
        --waiting;
        ask();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < WU; ++v)
#pragma unroll
          for (int j = 0; j < 2; ++j) run[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[v][j], x[u + v][j], run[t], 0, 0, 0);
      }
    if ((i & (4 / XU - 1)) == 4 / XU - 1) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        acc[t] += run[t];
        run[t] = tp_f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
  }
  tp_wait_fetches<0>();
  // ---- the waves' sums, added in wave order ------------------------------------------------------------
  float (*sums)[NT * 256] = reinterpret_cast<float (*)[NT * 256]>(lds);
  __syncthreads();                   // the rings have been read
#pragma unroll
  for (int t = 0; t < NT; ++t)
    if (r < p.M) *reinterpret_cast<tp_f32x4*>(&sums[wave][t * 256 + r * 16 + 4 * g]) = acc[t] + run[t];
  __syncthreads();
  float square = 0.f;
  if constexpr (OUT == STREAM_INTO) {
#pragma unroll
    for (int i = 0; i < ENDS; ++i) {
      const int e = threadIdx.x + 512 * i, n = first + 16 * (e >> 8) + enl;
      if (e >= NT * 256 || em >= p.M || n >= end) continue;
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < STREAM_WAVES; ++w) v += sums[w][e];
      v += old[i];
      p.h[em * p.ldh + n] = v;
      if (p.gain) p.left[(size_t)em * p.N + n] = f32_to_bf16(v * gain[i]);
      square += v * v;
    }
  } else {
    // thread -> (tile, row of X, four channels)
    for (int e = threadIdx.x; e < NT * p.M * 2; e += 512) {
      const int j = 4 * (e & 1), tm = e >> 1, t = tm / p.M, m = tm - t * p.M, c = first + 8 * t + j, at = t * 256 + m * 16 + j;
      float4 a = *reinterpret_cast<const float4*>(&sums[0][at]), b = *reinterpret_cast<const float4*>(&sums[0][at + 8]);
#pragma unroll
      for (int w = 1; w < STREAM_WAVES; ++w) {
        const float4 a1 = *reinterpret_cast<const float4*>(&sums[w][at]), b1 = *reinterpret_cast<const float4*>(&sums[w][at + 8]);
        a.x += a1.x, a.y += a1.y, a.z += a1.z, a.w += a1.w;
        b.x += b1.x, b.y += b1.y, b.z += b1.z, b.w += b1.w;
      }
      const float scale = p.squares ? extra[m * 256] : 1.f;
      const float gate[4] = {a.x, a.y, a.z, a.w}, up[4] = {b.x, b.y, b.z, b.w};
      bf16_t* to = p.out + (size_t)m * p.ldo + c;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (c + k < end) to[k] = f32_to_bf16(gate_act(gate[k] * scale, p.gelu) * (up[k] * scale));
    }
  }
  if constexpr (OUT == STREAM_INTO) {
    if (!p.gain) return;
    // the 16 threads of a row, then the two halves of the block
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) square += __shfl_xor(square, o, QVL_WAVE);
    if (NT > 1) {
      if (threadIdx.x >= 256 && enl == 0) extra[em] = square;
      __syncthreads();
      if (threadIdx.x < 256) square += extra[em];
    }
    if (threadIdx.x < 256 && enl == 0 && em < p.M) p.left_squares[em * STREAM_PARTS + blockIdx.x] = square;
  }
}

static int stream_check(const StreamArgs& p, int cus) {
  if (p.K <= 0 || p.K % 8 || p.ldx < p.K || p.ldw < p.K || p.ldx % 8 || p.ldw % 8 || !p.x || !p.w || cus <= 0 || ((uintptr_t)p.x % 16) ||
      ((uintptr_t)p.w % 16))
    return QVL_ERR_SHAPE;
  // offsets from the first row are 32-bit
  if ((unsigned long long)((p.N - 1) * p.ldw + p.K) * 2 >= 0xffffff00ull || (unsigned long long)((p.M - 1) * p.ldx + p.K) * 2 >= 0xffffff00ull)
    return QVL_ERR_LIMIT;
  return QVL_OK;
}

// The rows of X an item holds (4, 8 or 16) with which the busiest wave has the fewest items: fewer rows, more columns an item, but groups that
// deal out K less evenly.  w_items: of a step of 64 columns (narrow: of two, with the first two kinds).
static int stream_rows(int M, int K, int w_items, bool narrow) {
  int best = 16;
  long long least = 0x7fffffffffffffffll;
  for (int rows = 16, steps = 1; rows >= 4 && rows >= M; rows /= 2, steps *= 2) {
    if (narrow && rows == 16) continue;             // (what fewer rows leave is taken)
    const long long groups = (K + 64 * steps - 1) / (64 * steps);
    const long long items = (groups + STREAM_WAVES - 1) / STREAM_WAVES * (narrow && rows < 16 ? 1 + steps / 2 : 1 + steps * w_items);
    if (items < least) {
      least = items;
      best = rows;
    }
  }
  return best;
}

// Rows 8 KB apart, or a multiple of it, lie in the same few memory channels at the same column, and groups w, w + 8, ... of several rows close
// together: the waves then go through eighths of K instead (8,192 x 8,192, 1 row: 25.7 us for 32.7; 3,584 x 18,944 23.8 for 22.7).
static int stream_runs(long long ldw, int tiles) { return tiles > 1 && ldw % 4096 == 0; }

#define STREAM_MOST_INTO 4        // tiles of a block
#define STREAM_MOST_GATED 16

// h (float32 [M, N], rows ldh apart) += x . w^T for up to 16 rows.  gain (float32 [N] or null): the new rows of h are left for the product
// behind the norm with that gain: left (bfloat16 [M, N]) = h * gain, left_squares (float32 [M, 256]): sums of squares of a row's
// parts, whose number is qvl_gemm_stream_parts(N, cus).
extern "C" int qvl_gemm_stream_parts(int N, int cus) {
  if (N <= 0 || cus <= 0) return 0;
  return min(min(cus, STREAM_PARTS), N);
}
extern "C" int qvl_gemm_stream_takes_into(int M, int N, int K, int cus) {
  const int blocks = qvl_gemm_stream_parts(N, cus);
  return M > 0 && M <= 16 && K > 0 && K % 8 == 0 && blocks > 0 && (N + blocks - 1) / blocks <= 16 * STREAM_MOST_INTO;
}
extern "C" int qvl_gemm_stream_into(const void* x, long long ldx, const void* w, long long ldw, void* h, long long ldh, const void* gain,
                                    void* left, void* left_squares, int M, int N, int K, int cus, hipStream_t stream) {
  if (M <= 0 || N <= 0) return QVL_OK;
  StreamArgs p{};
  p.x = (const bf16_t*)x; p.ldx = ldx; p.w = (const bf16_t*)w; p.ldw = ldw; p.M = M; p.N = N; p.K = K;
  const int bad = stream_check(p, cus);
  if (bad) return bad;
  if (!h || ldh < N || (gain && (!left || !left_squares))) return QVL_ERR_SHAPE;
  if (!qvl_gemm_stream_takes_into(M, N, K, cus)) return QVL_ERR_LIMIT;
  p.h = (float*)h; p.ldh = ldh; p.gain = (const float*)gain; p.left = (bf16_t*)left; p.left_squares = (float*)left_squares;
  p.items = N;
  const int blocks = qvl_gemm_stream_parts(N, cus);
  p.t_step = 32 * ldw;
  p.h_step = 16 * ldw;
  const int rows = (N + blocks - 1) / blocks, tiles = (rows + 15) / 16;
  const bool narrow = rows <= 8;
  const int kind = stream_rows(M, K, tiles, narrow);
  p.runs = stream_runs(ldw, tiles);
  const dim3 grid(blocks), block(64 * STREAM_WAVES);
#define GO(NT, XR, NARROW) hipLaunchKernelGGL((gemm_stream_kernel<NT, XR, STREAM_INTO, NARROW>), grid, block, 0, stream, p)
#define TILES(NT)                  \
  case NT:                         \
    if (kind == 4) GO(NT, 4, false); \
    else if (kind == 8) GO(NT, 8, false); \
    else GO(NT, 16, false);        \
    break
  if (narrow) {
    if (kind == 4) GO(1, 4, true);
    else if (kind == 8) GO(1, 8, true);
    else GO(1, 16, true);
    return qvl_launch_status();
  }
  switch (tiles) {
    TILES(1);
    TILES(2);
    TILES(3);
    TILES(4);
    default: return QVL_ERR_LIMIT;
  }
#undef TILES
#undef GO
  return qvl_launch_status();
}

// out (bfloat16 [M, N / 2], rows ldo apart) = act(gate) up of x . w^T for up to 16 rows; w's rows in groups of 8 gate + 8 up.  squares (float32 [M, 256],
// on a 16-byte boundary), parts, eps: x is rows of a sum times a norm's gain as qvl_gemm_stream_into leaves them; null: x as it is.
extern "C" int qvl_gemm_stream_takes_gated(int M, int N, int K, int cus) {
  if (M <= 0 || M > 16 || N <= 0 || N % 16 || K <= 0 || K % 8 || cus <= 0) return 0;
  const int items = N / 2, blocks = min(cus, items), tiles = ((items + blocks - 1) / blocks + 7) / 8;
  return tiles <= STREAM_MOST_GATED;
}
extern "C" int qvl_gemm_stream_gated(const void* x, long long ldx, const void* w, long long ldw, void* out, long long ldo, const void* squares,
                                     int parts, float eps, int M, int N, int K, int gelu, int cus, hipStream_t stream) {
  if (M <= 0 || N <= 0) return QVL_OK;
  StreamArgs p{};
  p.x = (const bf16_t*)x; p.ldx = ldx; p.w = (const bf16_t*)w; p.ldw = ldw; p.M = M; p.N = N; p.K = K;
  const int bad = stream_check(p, cus);
  if (bad) return bad;
  if (!out || N % 16 || ldo < N / 2 || (squares && (parts <= 0 || parts > STREAM_PARTS || ((uintptr_t)squares % 16))))
    return QVL_ERR_SHAPE;
  if (!qvl_gemm_stream_takes_gated(M, N, K, cus)) return QVL_ERR_LIMIT;
  p.out = (bf16_t*)out; p.ldo = ldo; p.gelu = gelu;
  p.squares = (const float*)squares; p.parts = parts; p.eps = eps;
  p.items = N / 2;
  const int blocks = min(cus, p.items);
  p.t_step = 32 * ldw;
  p.h_step = 16 * ldw;
  const int tiles = ((p.items + blocks - 1) / blocks + 7) / 8, kind = M <= 8 ? stream_rows(M <= 4 ? 5 : M, K, tiles, false) : 16;
  p.runs = stream_runs(ldw, tiles);
  const dim3 grid(blocks), block(64 * STREAM_WAVES);
#define GO(NT, XR) hipLaunchKernelGGL((gemm_stream_kernel<NT, XR, STREAM_GATED, false>), grid, block, 0, stream, p)
#define TILES(NT)            \
  case NT:                   \
    if (kind == 8) GO(NT, 8); \
    else GO(NT, 16);         \
    break
  switch (tiles) {
    TILES(1); TILES(2); TILES(3); TILES(4); TILES(5); TILES(6); TILES(7); TILES(8);
    TILES(9); TILES(10); TILES(11); TILES(12); TILES(13); TILES(14); TILES(15); TILES(16);
    default: return QVL_ERR_LIMIT;
  }
#undef TILES
#undef GO
  return qvl_launch_status();
}
