// Products with more rows than the decode kernels keep: out = X[M, K] . W[N, K]^T, bfloat16 operands, float32 sums, with what
// follows the product done on the sums: a cast, the square of relu, a gated activation (gate and up rows of W in
// groups of 8 + 8, or gate rows first), or float32 slabs over ranges of K for whoever adds them next.
//
// The inner loop is tile_product.h's.  Tiles of 256 x 256 run fastest, others where a device of 256
// compute units would otherwise stand half empty or rows be padded; the choice is by an estimate of the time (shape_for).  Measured, the
// library's product (with the activation's kernel behind it where there is one) in brackets: 2,048 x 37,888 x 3,584
// gated 421 us (624), 2,048 x 3,584 x 18,944 in two ranges 204 (377), 281 x 22,016 x 2,048 gated 37 (55), 281 x 2,048 x 11,008 in ranges 23
// (50), 281 x 2,048 x 2,048 in ranges 10 (20).
//
// Blocks go to the XCDs in turn, each with an L2 of its own: XCD x takes a contiguous run of the tiles, ordered so that
// the 32 blocks it holds at a time share few rows of W and X (eight tiles of X's rows, then the next tile of W's).
#include "tile_product.h"

#include <cmath>

enum { OUT_BF16 = 0, OUT_F32 = 1, OUT_GROUPED = 2, OUT_HALVES = 3, OUT_HEADS = 4, OUT_SCALED = 5 };     // (scaled: grouped, of such rows)

struct TileArgs {
  const bf16_t* x;
  long long ldx;
  const bf16_t* w;
  long long ldw;
  void* out;
  long long ldo;
  int M, N, K;
  int rows;              // OUT_HALVES: rows of W before its up rows (N = 2 rows); else N
  int tiles_m, tiles_n, splits;
  int relu2, gelu;
  float alpha, limit, shift;
  // OUT_SCALED: X's rows are rows of a sum times a norm's gain, not yet divided by their root mean square: row m's squares add up to the first `parts`
  // numbers from squares[TILE_PARTS m] on
  const float* squares;
  int parts;
  float eps;
  // OUT_HEADS: W holds nq query, nkv key and nkv value heads of HEAD rows; out takes the rotated queries [M, nq, HEAD]
  const float* bias;     // [N] or null
  const float4* cs;      // [M, HEAD / 2]: cosine and sine, two frequencies a value
  const int* slot;       // [M]: page * ps + place in it, or -1
  bf16_t* kc;            // [page][nkv][ps][HEAD]
  bf16_t* vc;            // [page][nkv][HEAD][ps]
  int nq, nkv, ps;
};
#define HEAD 128
#define TILE_PARTS 256     // places of a row's sums of squares

__device__ __forceinline__ uint32_t two_bf16(float a, float b) {
  typedef __bf16 pair_t __attribute__((ext_vector_type(2)));
  const pair_t v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}
// four neighbouring results
__device__ __forceinline__ void store4(bf16_t* o, const float* v, int n, bool whole) {
  if (whole) {
    *reinterpret_cast<uint2*>(o) = uint2{two_bf16(v[0], v[1]), two_bf16(v[2], v[3])};
  } else {
    for (int i = 0; i < n && i < 4; ++i) o[i] = f32_to_bf16(v[i]);
  }
}
__device__ __forceinline__ void store4(float* o, const float* v, int n, bool whole) {
  if (whole) {
    *reinterpret_cast<float4*>(o) = float4{v[0], v[1], v[2], v[3]};
  } else {
    for (int i = 0; i < n && i < 4; ++i) o[i] = v[i];
  }
}
__device__ __forceinline__ float clamped_gate(float g, float u, const TileArgs& p) {
  if (p.limit > 0.f) {
    g = fminf(g, p.limit);
    u = fminf(fmaxf(u, -p.limit), p.limit);
  }
  return g / (1.0f + expf(-p.alpha * g)) * (u + p.shift);
}

// OUT_HEADS: channels f and f + 64 of a head are rotated together, so the waves that share a head (one of 8 tiles of W's rows, two of
// 4) have half of their tiles in either half of the head: tile n < NT / 2 and tile n + NT / 2 meet in a lane.
// The row of W behind row rho of region h:
template <typename T>
__device__ __forceinline__ int head_row(int h, int rho) {
  constexpr int SHARE = 8 / T::NT > 0 ? 8 / T::NT : 1, RUN = 16 * (T::NT / 2);
  const int wave = rho / RUN;
  return wave / SHARE * HEAD + h * (HEAD / 2) + wave % SHARE * RUN + rho % RUN;
}

// The sums of a tile of OUT_HEADS: bias, rotation, queries out, keys and values into their pages, each rounded once.  What this saves is
// the float32 product's way to memory and back and a launch: 2,048 rows x 4,608 x 3,584 70 us, the library's product and the rotation's
// kernel 62 + 20 (with one chain of sums for each output both, the same bits), 4,096 rows 135 for 162.
template <typename T>
__device__ __forceinline__ void store_heads(const T& t, const TileArgs& p, int n0, int m0) {
  constexpr int SHARE = 8 / T::NT > 0 ? 8 / T::NT : 1, RUN = 16 * (T::NT / 2);
  const int head = n0 / HEAD + t.wn / SHARE, kind = head < p.nq ? 0 : head < p.nq + p.nkv ? 1 : 2;      // the same for a wave
  if (head * HEAD >= p.N) return;
  const int f0 = t.wn % SHARE * RUN + 4 * t.g;      // and f0 + 16 n, of the lane's sums
  float4 b[T::NT];
#pragma unroll
  for (int n = 0; n < T::NT; ++n)
    b[n] = p.bias ? *reinterpret_cast<const float4*>(p.bias + head * HEAD + f0 + n % (T::NT / 2) * 16 + n / (T::NT / 2) * (HEAD / 2))
                  : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int m = 0; m < T::MT; ++m) {
    const int gm = m0 + (t.wm * T::MT + m) * 16 + t.r;
    if (gm >= p.M) continue;
    bf16_t* to = reinterpret_cast<bf16_t*>(p.out) + ((size_t)gm * p.nq + head) * HEAD;
    int apart = 1;       // from a channel to the next
    if (kind) {
      const int s = p.slot[gm];
      if (s < 0) continue;
      const int page = s / p.ps, place = s - page * p.ps;
      const size_t of = (size_t)page * p.nkv + (head - p.nq - (kind == 2 ? p.nkv : 0));
      to = kind == 1 ? p.kc + (of * p.ps + place) * HEAD : p.vc + of * HEAD * p.ps + place;
      if (kind == 2) apart = p.ps;
    }
#pragma unroll
    for (int n = 0; n < T::NT / 2; ++n) {
      const int f = f0 + 16 * n;
      const tp_f32x4 s1 = t.acc[n][m], s2 = t.acc[n + T::NT / 2][m];
      const float4 b1 = b[n], b2 = b[n + T::NT / 2];
      const float x1[4] = {s1[0] + b1.x, s1[1] + b1.y, s1[2] + b1.z, s1[3] + b1.w};
      const float x2[4] = {s2[0] + b2.x, s2[1] + b2.y, s2[2] + b2.z, s2[3] + b2.w};
      if (kind == 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          to[(size_t)(f + i) * apart] = f32_to_bf16(x1[i]);
          to[(size_t)(f + i + HEAD / 2) * apart] = f32_to_bf16(x2[i]);
        }
        continue;
      }
      const float4 c01 = p.cs[(size_t)gm * (HEAD / 4) + f / 2], c23 = p.cs[(size_t)gm * (HEAD / 4) + f / 2 + 1];     // (c0, s0, c1, s1)
      const float c[4] = {c01.x, c01.z, c23.x, c23.z}, sn[4] = {c01.y, c01.w, c23.y, c23.w};
      float lo[4], hi[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        lo[i] = x1[i] * c[i] - x2[i] * sn[i];
        hi[i] = x2[i] * c[i] + x1[i] * sn[i];
      }
      store4(to + f, lo, 4, true);
      store4(to + f + HEAD / 2, hi, 4, true);
    }
  }
}

// One over the root mean square of each row of X that this lane has results of.  A row's four lanes (g) take four of its numbers at a time; those of
// the first 32 are asked for in front of the first fetches of W and X and added up behind them, on their way (22,016 x 2,048, 420 rows 47.2 us, waited for
// in front of them 49.6, of rows that need no scale 44.8; the norm's kernel that falls away takes 4.0 and 10 us of the host).
template <typename T>
struct RowScales {
  float4 first[T::MT][2];
  float scale[T::MT];

  __device__ __forceinline__ const float* at(const T& t, const TileArgs& p, int m0, int m) const {
    const int gm = m0 + (t.wm * T::MT + m) * 16 + t.r;
    return p.squares + (size_t)(gm < p.M ? gm : 0) * TILE_PARTS;
  }
  __device__ __forceinline__ void ask(const T& t, const TileArgs& p, int m0) {
#pragma unroll
    for (int m = 0; m < T::MT; ++m)
#pragma unroll
      for (int i = 0; i < 2; ++i) first[m][i] = *reinterpret_cast<const float4*>(at(t, p, m0, m) + 16 * i + 4 * t.g);
  }
  __device__ static __forceinline__ float some(const float4& v, int have) {      // the first `have`: those behind the last part hold anything
    return ((have > 0 ? v.x : 0.f) + (have > 1 ? v.y : 0.f)) + ((have > 2 ? v.z : 0.f) + (have > 3 ? v.w : 0.f));
  }
  __device__ __forceinline__ void finish(const T& t, const TileArgs& p, int m0) {
    const int have = p.parts - 4 * t.g;
#pragma unroll
    for (int m = 0; m < T::MT; ++m) scale[m] = some(first[m][0], have) + some(first[m][1], have - 16);
    for (int k = 32; k < p.parts; k += 16) {
#pragma unroll
      for (int m = 0; m < T::MT; ++m) scale[m] += some(*reinterpret_cast<const float4*>(at(t, p, m0, m) + min(k + 4 * t.g, TILE_PARTS - 4)), have - k);
    }
#pragma unroll
    for (int m = 0; m < T::MT; ++m) {
      float s = scale[m];
      s += __shfl_xor(s, 16, QVL_WAVE);
      s += __shfl_xor(s, 32, QVL_WAVE);
      scale[m] = 1.0f / sqrtf(s / (float)p.K + p.eps);
    }
  }
};

template <typename T, int OUT>
__global__ __launch_bounds__(512) void gemm_tile_kernel(TileArgs p) {
  __shared__ __attribute__((aligned(16))) char lds[T::LDS];
  T t;
  const int tiles = p.tiles_m * p.tiles_n, all = tiles * p.splits, per = (all + 7) / 8;
  const int turn = blockIdx.x >> 3, id = (blockIdx.x & 7) * per + turn;
  if (turn >= per || id >= all) return;
  const int split = id / tiles, at = id - split * tiles;
  // eight tiles of X's rows beside each other, then the next tile of W's rows
  const int band = at / (8 * p.tiles_n), in_band = at - band * 8 * p.tiles_n;
  const int wide = min(8, p.tiles_m - 8 * band);
  const int tile_m = 8 * band + in_band % wide, tile_n = in_band / wide;
  constexpr int OUT_N = OUT == OUT_HALVES ? T::BN / 2 : T::BN;       // rows of W (of each half) from n0 on
  const int n0 = tile_n * OUT_N, m0 = tile_m * T::BM;
  // this split's range of K
  const int steps_all = (p.K + 63) / 64;
  const int s0 = (int)((long long)steps_all * split / p.splits), s1 = (int)((long long)steps_all * (split + 1) / p.splits);
  const bf16_t* w = p.w + (size_t)n0 * p.ldw + (size_t)s0 * 64;
  const bf16_t* x = p.x + (size_t)m0 * p.ldx + (size_t)s0 * 64;
  RowScales<T> rows;
  if (OUT == OUT_SCALED) rows.ask(t, p, m0);
  // rows that do not exist are read from one that does; their sums are not stored
  t.set_rows(
      [&](int h, int rho) {
        if (OUT == OUT_HALVES) {     // first half: gate rows, second half: their up rows
          const int n = n0 + rho < p.rows ? rho : 0;
          return (uint32_t)(((size_t)n + (h ? p.rows : 0)) * p.ldw * 2);
        }
        const int n = OUT == OUT_HEADS ? head_row<T>(h, rho) : T::w_row(h, rho);
        return (uint32_t)((size_t)(n0 + n < p.N ? n : 0) * p.ldw * 2);
      },
      [&](int h, int rho) {
        const int m = T::x_row(h, rho);
        return (uint32_t)((size_t)(m0 + m < p.M ? m : 0) * p.ldx * 2);
      });
  t.multiply(lds, w, x, s1 - s0, p.K % 64 != 0 && s1 == steps_all, [&]() __attribute__((always_inline)) {
    if (OUT == OUT_SCALED) rows.finish(t, p, m0);
  });
  // a lane holds, of tile (n, m): X's row 16 m + r, W's rows 16 n + 4 g ... + 3
  if constexpr (OUT == OUT_HEADS) {
    store_heads(t, p, n0, m0);
    return;
  }
#pragma unroll
  for (int m = 0; m < T::MT; ++m) {
    const int gm = m0 + (t.wm * T::MT + m) * 16 + t.r;
    if (OUT == OUT_BF16 || OUT == OUT_F32) {
      if (gm >= p.M) continue;
#pragma unroll
      for (int n = 0; n < T::NT; ++n) {
        const int gn = n0 + (t.wn * T::NT + n) * 16 + 4 * t.g;
        if (gn >= p.N) continue;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[i] = t.acc[n][m][i];
          if (p.relu2) {
            v[i] = fmaxf(v[i], 0.f);
            v[i] *= v[i];
          }
        }
        const bool whole = gn + 4 <= p.N && p.ldo % 4 == 0;
        if (OUT == OUT_BF16) store4(reinterpret_cast<bf16_t*>(p.out) + (size_t)gm * p.ldo + gn, v, p.N - gn, whole);
        else store4(reinterpret_cast<float*>(p.out) + ((size_t)split * p.M + gm) * p.ldo + gn, v, p.N - gn, whole);
      }
    } else if (OUT == OUT_HALVES) {
      if (gm >= p.M) continue;
#pragma unroll
      for (int n = 0; n < T::NH; ++n) {
        const int gn = n0 + (t.wn * T::NH + n) * 16 + 4 * t.g;
        if (gn >= p.rows) continue;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = clamped_gate(t.acc[n][m][i], t.acc[n + T::NH][m][i], p);
        store4(reinterpret_cast<bf16_t*>(p.out) + (size_t)gm * p.ldo + gn, v, p.rows - gn, gn + 4 <= p.rows && p.ldo % 4 == 0);
      }
    } else {
      // rows 0 .. 7 of a tile of 16 are gate rows (lanes of g 0 and 1), rows 8 .. 15 their up rows.  Of two
      // neighbouring tiles the lanes below 32 take the first, the others the second: one exchange of halves
      // gives every lane a gate and its up value.
#pragma unroll
      for (int n = 0; n < T::NT; n += 2) {
        static_assert(T::NT % 2 == 0, "tiles in pairs");
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float one = t.acc[n][m][i], next = t.acc[n + 1][m][i];
          const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(one), __float_as_uint(next), false, false);
          const float scale = OUT == OUT_SCALED ? rows.scale[m] : 1.f;
          v[i] = gate_act(__uint_as_float((uint32_t)both[0]) * scale, p.gelu) * (__uint_as_float((uint32_t)both[1]) * scale);
        }
        const int first = n0 + (t.wn * T::NT + n + (t.g >> 1)) * 16;      // the lane's tile's first row of W
        if (gm < p.M && first < p.N)
          store4(reinterpret_cast<bf16_t*>(p.out) + (size_t)gm * p.ldo + first / 2 + 4 * (t.g & 1), v, 4, p.ldo % 4 == 0);
      }
    }
  }
}

// The tile's shape for a product in `splits` ranges of K.  The estimate is of microseconds: a step of 64 values
// costs a block `alone` where most compute units are idle and `full` where all work (with every matrix core busy the clock and the
// caches give way), a launch 3 us and each of its rounds 2.9 (the first fetches, the stores); results are written at 5.9 TB/s and read once
// more at 4.5; and W comes at 7.5 TB/s at most, which joins the rest as the root of squares.  Where two blocks share a compute unit, a last
// round of up to half the room has a unit for each block, else some blocks have to share.  Fitted to 124 products of 70 to 4,096 rows at
// the 3B, 7B and 72B decoders' sizes, each with all shapes and cuts (rms 6 per cent).
struct TileShape {
  int bn, bm, a_unit;     // blocks a compute unit holds
  double alone, full;
};
#define SHAPES_N 10
static const TileShape SHAPES[SHAPES_N] = {{256, 256, 1, 0.967, 1.361}, {128, 256, 1, 0.629, 0.816}, {256, 128, 1, 0.678, 0.825},
                                           {128, 128, 2, 0.502, 0.884}, {192, 192, 1, 0.727, 0.922}, {128, 192, 2, 0.597, 1.164},
                                           {192, 256, 1, 0.784, 1.089}, {192, 320, 1, 0.992, 1.362}, {128, 320, 1, 0.758, 0.985},
                                           {256, 192, 1, 0.888, 1.129}};

static int shape_for(int M, int N, int K, int splits, int cus, unsigned may = ~0u) {      // may: a bit for each shape
  int best = 0;
  double least = 1e30;
  const int steps = (K + 63) / 64;
  const double memory = 3.0 + (double)N * K * 2.0 / 7.52e6;
  for (int i = 0; i < SHAPES_N; ++i) {
    if (!(may >> i & 1)) continue;
    const TileShape& s = SHAPES[i];
    const long long blocks = (long long)((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn) * splits, room = (long long)cus * s.a_unit;
    const long long whole = blocks / room;
    const double rest = (double)(blocks - whole * room) / room;
    const double depth = (steps + splits - 1) / splits, bytes = (double)M * N * (splits > 1 ? 4.0 * splits : 2.0);
    double us = 3.0 + whole * (depth * s.full + 2.9) + bytes / 5.92e6;
    const double busy = s.a_unit == 1 ? rest : (2.0 * rest > 1.0 ? 1.0 : 0.0);
    if (rest > 0) us += depth * (s.alone + (s.full - s.alone) * busy) + 2.9;
    us = sqrt(us * us + memory * memory) + bytes / 4.5e6;
    if (us < least) least = us, best = i;
  }
  return best;
}

#define MOST_SPLITS 12

// How many ranges K is cut into, and which products are left to the library: by an estimate among the four shapes of powers of two alone,
// whatever shape then runs.
//
// The ranges set the order of an output's sum, and a product that is cut hands its sums on in float32 where one that is not may round them to
// bfloat16: the shapes above change neither.  Ranges by the estimate above, fitted on 256 compute units, gave up float32 sums on parts of a
// device (2,048 x 2,048, 1,031 rows, 128 units: three slabs here, none by it) and gained nothing over sixteen whole passes (fitted and here: 2,048
// rows at 7B sizes 7,239 us and 7,265, portions of 2,048 beside long contexts 28.67 ms and 28.84, a Gogudra pass 12.35 and 12.23).
//
// With far fewer blocks than compute units the library, which cuts K by itself, is faster, and the other shapes' more blocks for the same
// work do not move that line: of 40 products that they alone would take over it the library was the faster in 35 (2,560 x 8,192, 1,991 rows:
// 79 us against 87; 7,168 x 2,368, 605: 29 and 36; 3,584 x 4,736, 2,396: 77 and 75), by 4 per cent on average.
struct Count {
  long long blocks;
  int splits;
};
static Count count_for(int M, int N, int K, int most_splits, int cus) {
  static const TileShape COUNTED[4] = {{256, 256, 1, 1.08, 1.43}, {128, 256, 1, 0.72, 0.96}, {256, 128, 1, 0.79, 0.94}, {128, 128, 2, 0.53, 1.02}};
  const int steps = (K + 63) / 64;
  double least = 1e30;
  Count count{0, 1};
  for (const TileShape& s : COUNTED) {
    const long long tiles = (long long)((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn);
    for (int splits = 1; splits <= most_splits && (splits == 1 || splits * 4 <= steps); ++splits) {
      const long long blocks = tiles * splits, room = (long long)cus * s.a_unit, whole = blocks / room;
      const double rest = (double)(blocks - whole * room) / room, depth = (steps + splits - 1) / splits;
      const double busy = s.a_unit == 1 ? rest : (2.0 * rest > 1.0 ? 1.0 : 0.0);
      double us = 8.0 + whole * (depth * s.full + 4.0);
      if (rest > 0) us += depth * (s.alone + (s.full - s.alone) * busy) + 4.0;
      if (splits > 1) us += splits * (double)M * N * 8.0 / 4.5e6;
      if (us < least) least = us, count = Count{tiles, splits};
    }
  }
  return count;
}

// Ranges of K that tile_slabs (tile.py) takes.
extern "C" int qvl_gemm_tile_splits(int M, int N, int K, int cus) {
  if (M <= 0 || N <= 0 || K <= 0 || cus <= 0) return 0;
  return count_for(M, N, K, MOST_SPLITS, cus).splits;
}
// Blocks of the uncut product, which prefers_tile (tile.py) holds against the compute units.
extern "C" int qvl_gemm_tile_blocks(int M, int N, int K, int cus) {
  if (M <= 0 || N <= 0 || K <= 0 || cus <= 0) return 0;
  const long long blocks = count_for(M, N, K, 1, cus).blocks;
  return (int)(blocks < 0x7fffffff ? blocks : 0x7fffffff);
}

// x: bfloat16 [M, K], rows ldx apart; W: bfloat16 [N, K], rows ldw apart; both on 16-byte boundaries, K a multiple of 32.
// mode 0: out bfloat16 [M, N] (relu2: max(product, 0)^2); 1: out float32 [splits][M][N], the slabs' sum is the product;
// 2: N in groups of 8 gate + 8 up rows, out bfloat16 [M, N / 2] = act(gate) up (gelu: gelu's tanh form, else silu);
// 3: N / 2 gate rows, then the up rows: out = g sigmoid(alpha g) (u + shift), g capped at limit, u clamped to +-limit.
// tile: -1, or the shape to take (0 .. 9).
static int tile_launch(const void* x, long long ldx, const void* w, long long ldw, void* out, long long ldo, int M, int N,
                       int K, int mode, int splits, int relu2, int gelu, float alpha, float limit, float shift, int tile,
                       int cus, const void* squares, int parts, float eps, hipStream_t stream) {
  if (M <= 0 || N <= 0) return QVL_OK;
  if (K <= 0 || K % 32 || ldx < K || ldw < K || ldx % 8 || ldw % 8 || !x || !w || !out || cus <= 0 || splits < 1 ||
      ((uintptr_t)x % 16) || ((uintptr_t)w % 16) || ((uintptr_t)out % 16) || splits > (K + 63) / 64 || (mode != 1 && splits != 1))
    return QVL_ERR_SHAPE;
  if ((mode == 2 && N % 16) || (mode == 3 && N % 2) || ldo < (mode >= 2 ? N / 2 : N)) return QVL_ERR_SHAPE;
  if (mode < 0 || mode > 3 || tile >= SHAPES_N) return QVL_ERR_SHAPE;
  // byte offsets from a tile's first row are 32-bit (in mode 3 the up rows lie N / 2 rows further on)
  const unsigned long long w_span = (mode == 3 ? (unsigned long long)N / 2 + 256 : 256ull) * ldw * 2, x_span = 256ull * ldx * 2;
  if (w_span >= 0xffff0000ull || x_span >= 0xffff0000ull) return QVL_ERR_LIMIT;
  TileArgs p;
  p.x = (const bf16_t*)x; p.ldx = ldx; p.w = (const bf16_t*)w; p.ldw = ldw; p.out = out; p.ldo = ldo;
  p.M = M; p.N = N; p.K = K; p.rows = mode == 3 ? N / 2 : N; p.splits = splits; p.relu2 = relu2; p.gelu = gelu;
  p.alpha = alpha; p.limit = limit; p.shift = shift;
  p.squares = (const float*)squares; p.parts = parts; p.eps = eps;
  int shape = tile >= 0 ? tile : shape_for(M, N, K, splits, cus);
  if ((unsigned long long)SHAPES[shape].bm * ldx * 2 >= 0xffff0000ull) shape = 0;
  const TileShape& s = SHAPES[shape];
  const int out_n = mode == 3 ? s.bn / 2 : s.bn;
  p.tiles_m = (M + s.bm - 1) / s.bm;
  p.tiles_n = (p.rows + out_n - 1) / out_n;
  const long long all = (long long)p.tiles_m * p.tiles_n * splits;
  if (all > 0x7ffffff0ll / 8) return QVL_ERR_LIMIT;
  const dim3 grid((unsigned)((all + 7) / 8 * 8));
#define GO(OUT, WN, WM, NT, MT) hipLaunchKernelGGL((gemm_tile_kernel<Tile<WN, WM, NT, MT>, OUT>), grid, dim3(512), 0, stream, p)
#define SHAPE(OUT)                       \
  do {                                   \
    if (shape == 0) GO(OUT, 2, 4, 8, 4); \
    else if (shape == 1) GO(OUT, 2, 4, 4, 4); \
    else if (shape == 2) GO(OUT, 4, 2, 4, 4); \
    else if (shape == 3) GO(OUT, 2, 4, 4, 2); \
    else if (shape == 4) GO(OUT, 2, 4, 6, 3); \
    else if (shape == 5) GO(OUT, 2, 4, 4, 3); \
    else if (shape == 6) GO(OUT, 2, 4, 6, 4); \
    else if (shape == 7) GO(OUT, 2, 4, 6, 5); \
    else if (shape == 8) GO(OUT, 2, 4, 4, 5); \
    else GO(OUT, 2, 4, 8, 3);            \
  } while (0)
  if (mode == 0) SHAPE(OUT_BF16);
  else if (mode == 1) SHAPE(OUT_F32);
  else if (mode == 2 && squares) SHAPE(OUT_SCALED);
  else if (mode == 2) SHAPE(OUT_GROUPED);
  else SHAPE(OUT_HALVES);
#undef SHAPE
#undef GO
  return qvl_launch_status();
}
extern "C" int qvl_gemm_tile(const void* x, long long ldx, const void* w, long long ldw, void* out, long long ldo, int M, int N,
                             int K, int mode, int splits, int relu2, int gelu, float alpha, float limit, float shift, int tile,
                             int cus, hipStream_t stream) {
  return tile_launch(x, ldx, w, ldw, out, ldo, M, N, K, mode, splits, relu2, gelu, alpha, limit, shift, tile, cus, nullptr, 0, 0.f, stream);
}
// Mode 2 for rows x of a sum times a norm's gain that are still to be divided by their root mean square: row m's squares add up to squares[256 m ...],
// `parts` numbers (float32 [M, 256] on a 16-byte boundary).
extern "C" int qvl_gemm_tile_scaled(const void* x, long long ldx, const void* w, long long ldw, void* out, long long ldo, const void* squares, int parts,
                                    float eps, int M, int N, int K, int gelu, int tile, int cus, hipStream_t stream) {
  if (!squares || parts <= 0 || parts > TILE_PARTS || (uintptr_t)squares % 16) return QVL_ERR_SHAPE;
  return tile_launch(x, ldx, w, ldw, out, ldo, M, N, K, 2, 1, 0, gelu, 1.f, 0.f, 0.f, tile, cus, squares, parts, eps, stream);
}

// Shapes whose waves hold both halves of a head (8 or 4 tiles of W's rows).
#define HEAD_SHAPES ((1u << 0) | (1u << 1) | (1u << 2) | (1u << 3) | (1u << 5) | (1u << 8) | (1u << 9))

// The stacked projection of nq query, nkv key and nkv value heads of 128 channels with what follows it in the kernel: q_out bfloat16
// [M, nq, 128] rotated; rotated keys and values into the page slots of their tokens, kc [page][nkv][ps][128], vc [page][nkv][128][ps]
// (slot[m] = page * ps + place, or -1: not written).  bias: float32 [(nq + 2 nkv) 128] or null; cs: float32 [M, 64, 2].  x, w, tile
// as in qvl_gemm_tile; everything on 16-byte boundaries.
extern "C" int qvl_gemm_tile_heads(const void* x, long long ldx, const void* w, long long ldw, const void* bias, const void* cs,
                                   const void* slot, void* q_out, void* kc, void* vc, int M, int K, int nq, int nkv, int ps, int tile,
                                   int cus, hipStream_t stream) {
  if (M <= 0) return QVL_OK;
  if (nq <= 0 || nkv < 0 || nq > 0xffff || nkv > 0xffff || (nkv && (ps <= 0 || !slot || !kc || !vc))) return QVL_ERR_SHAPE;
  const int N = (nq + 2 * nkv) * HEAD;
  if (K <= 0 || K % 32 || ldx < K || ldw < K || ldx % 8 || ldw % 8 || !x || !w || !cs || !q_out || cus <= 0 ||
      (((uintptr_t)x | (uintptr_t)w | (uintptr_t)bias | (uintptr_t)cs | (uintptr_t)q_out | (uintptr_t)kc | (uintptr_t)vc) % 16))
    return QVL_ERR_SHAPE;
  if (tile >= SHAPES_N || (tile >= 0 && !(HEAD_SHAPES >> tile & 1))) return QVL_ERR_SHAPE;
  // byte offsets from a tile's first row are 32-bit
  if (256ull * ldw * 2 >= 0xffff0000ull || 256ull * ldx * 2 >= 0xffff0000ull) return QVL_ERR_LIMIT;
  TileArgs p;
  p.x = (const bf16_t*)x; p.ldx = ldx; p.w = (const bf16_t*)w; p.ldw = ldw; p.out = q_out; p.ldo = 0;
  p.M = M; p.N = N; p.K = K; p.rows = N; p.splits = 1; p.relu2 = p.gelu = 0; p.alpha = p.limit = p.shift = 0.f;
  p.squares = nullptr; p.parts = 0; p.eps = 0.f;
  p.bias = (const float*)bias; p.cs = (const float4*)cs; p.slot = (const int*)slot; p.kc = (bf16_t*)kc; p.vc = (bf16_t*)vc;
  p.nq = nq; p.nkv = nkv; p.ps = ps;
  int shape = tile >= 0 ? tile : shape_for(M, N, K, 1, cus, HEAD_SHAPES);
  if ((unsigned long long)SHAPES[shape].bm * ldx * 2 >= 0xffff0000ull) shape = 0;
  p.tiles_m = (M + SHAPES[shape].bm - 1) / SHAPES[shape].bm;
  p.tiles_n = (N + SHAPES[shape].bn - 1) / SHAPES[shape].bn;
  const long long all = (long long)p.tiles_m * p.tiles_n;
  if (all > 0x7ffffff0ll / 8) return QVL_ERR_LIMIT;
  const dim3 grid((unsigned)((all + 7) / 8 * 8));
#define GO(WN, WM, NT, MT) hipLaunchKernelGGL((gemm_tile_kernel<Tile<WN, WM, NT, MT>, OUT_HEADS>), grid, dim3(512), 0, stream, p)
  if (shape == 0) GO(2, 4, 8, 4);
  else if (shape == 1) GO(2, 4, 4, 4);
  else if (shape == 2) GO(4, 2, 4, 4);
  else if (shape == 3) GO(2, 4, 4, 2);
  else if (shape == 5) GO(2, 4, 4, 3);
  else if (shape == 8) GO(2, 4, 4, 5);
  else GO(2, 4, 8, 3);
#undef GO
  return qvl_launch_status();
}
