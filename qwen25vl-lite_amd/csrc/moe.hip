// A feed-forward made of many small experts, of which every token uses a few:
//   route    scores of the router's logits, the choice of experts within the best groups, weights
//   sort     the (token, choice) pairs listed by expert
//   products x W_e^T for every expert's pairs: gate|up with the gated activation, then down
//   combine  the weighted sum of a token's experts, plus what a shared expert gave
// float32 and bfloat16 storage; scores, weights and sums are float32.  A pair is p = token * top + choice.
#include "tile_product.h"

#include <cmath>

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float sigmoid_f(float z) { return 1.0f / (1.0f + expf(-z)); }

// ---------------------------------------------------------------------------------------
// Router.  z [N, E] float32 logits.  s = sigmoid(z) (score_fn 0) or softmax(z) over the experts
// (score_fn 1).  Experts e with the same e / (E / groups) are one group, ranked by the sum of its
// top two s (its only one, if it has one member); the choice is the `top` highest s among the members
// of the `keep` highest-ranked groups (ties: the lower index).  Weights: the
// chosen s divided by (their sum + floor) if `normalize`, times `scale`.
// One wave per token; E <= 512, groups <= 64.
// ---------------------------------------------------------------------------------------
#define MOE_MAX_E 512

struct RouteArgs {
  const float* z;
  int* ids;
  float* wts;
  int N, E, top, groups, keep, score_fn, normalize;
  float scale, floor_;
};

// The largest of a wave's values (no NaN among them) in every lane: within rows of 16 lanes by rotations, across them by swaps.
__device__ __forceinline__ float largest(float v) {
  auto turned = [&](auto by) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x120 + decltype(by)::value, 0xf, 0xf, true));
  };
  v = fmaxf(v, turned(std::integral_constant<int, 8>{}));
  v = fmaxf(v, turned(std::integral_constant<int, 4>{}));
  v = fmaxf(v, turned(std::integral_constant<int, 2>{}));
  v = fmaxf(v, turned(std::integral_constant<int, 1>{}));
  const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float((uint32_t)x[0]), __uint_as_float((uint32_t)x[1]));
  const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float((uint32_t)y[0]), __uint_as_float((uint32_t)y[1]));
}

// Token n by one wave; s and gs: this wave's MOE_MAX_E and 64 floats of LDS (read where there are groups).  What bounds it is the chain of
// choices: each takes a maximum over the wave (rotations and swaps of registers; by way of LDS six choices of 32 experts took 4 us
// more) and one lane's answer, the lowest index where several lanes hold the largest score.
__device__ __forceinline__ void route_token(const RouteArgs& p, int n, float* s, float* gs) {
  const int lane = threadIdx.x & 63, E = p.E;
  const float* zr = p.z + (size_t)n * E;
  float score[MOE_MAX_E / 64];      // of this lane's experts, e = lane + 64 i
#pragma unroll
  for (int i = 0; i < MOE_MAX_E / 64; ++i) {
    const int e = lane + 64 * i;
    score[i] = e < E ? zr[e] : -INFINITY;
  }
  if (p.score_fn == 1) {
    float mx = -INFINITY, sum = 0.f;
#pragma unroll
    for (int i = 0; i < MOE_MAX_E / 64; ++i)
      if (64 * i < E) mx = fmaxf(mx, score[i]);
    mx = largest(mx);
#pragma unroll
    for (int i = 0; i < MOE_MAX_E / 64; ++i)
      if (lane + 64 * i < E) {
        score[i] = expf(score[i] - mx);
        sum += score[i];
      }
    sum = wave_sum(sum);
#pragma unroll
    for (int i = 0; i < MOE_MAX_E / 64; ++i) score[i] = score[i] / sum;
  } else {
#pragma unroll
    for (int i = 0; i < MOE_MAX_E / 64; ++i)
      if (64 * i < E) score[i] = sigmoid_f(score[i]);
  }
  unsigned long long allowed = ~0ull;
  const int per = E / p.groups;
  if (p.groups > 1) {
#pragma unroll
    for (int i = 0; i < MOE_MAX_E / 64; ++i)
      if (lane + 64 * i < E) s[lane + 64 * i] = score[i];
    __builtin_amdgcn_wave_barrier();
    if (lane < p.groups) {
      float a = -INFINITY, b = -INFINITY;   // the two largest
      for (int i = 0; i < per; ++i) {
        const float v = s[lane * per + i];
        if (v > a) { b = a; a = v; }
        else if (v > b) b = v;
      }
      gs[lane] = per > 1 ? a + b : a;
    }
    __builtin_amdgcn_wave_barrier();
    bool allowed_group = false;
    if (lane < p.groups) {
      int ahead = 0;
      const float mine = gs[lane];
      for (int g = 0; g < p.groups; ++g) ahead += (gs[g] > mine || (gs[g] == mine && g < lane)) ? 1 : 0;
      allowed_group = ahead < p.keep;
    }
    allowed = __ballot(allowed_group);
  }
  // a score of -1 can never be chosen before an allowed one
#pragma unroll
  for (int i = 0; i < MOE_MAX_E / 64; ++i) {
    const int e = lane + 64 * i;
    score[i] = (e < E && ((allowed >> (p.groups > 1 ? e / per : 0)) & 1ull)) ? score[i] : -1.0f;
  }
  float total = 0.f;
  float my_w = 0.f;   // lane t keeps the weight of choice t (top <= 64)
  int my_id = 0;
  for (int t = 0; t < p.top; ++t) {
    float mine = -2.0f;
    int at = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < MOE_MAX_E / 64; ++i)
      if (64 * i < E && score[i] > mine) { mine = score[i]; at = lane + 64 * i; }
    // the wave's best: larger score first, then the lower index
    const float best = largest(mine);
    const unsigned long long equal = __ballot(mine == best);
    if (__popcll(equal) > 1) {
      if (mine != best) at = 0x7fffffff;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) at = min(at, __shfl_xor(at, o, QVL_WAVE));
    } else {
      at = __builtin_amdgcn_readlane(at, __ffsll(equal) - 1);
    }
#pragma unroll
    for (int i = 0; i < MOE_MAX_E / 64; ++i)
      if (at == lane + 64 * i) score[i] = -3.0f;
    total += best;
    if (lane == t) { my_w = best; my_id = at; }
  }
  if (lane < p.top) {
    const float w = p.normalize ? my_w / (total + p.floor_) : my_w;
    p.ids[(size_t)n * p.top + lane] = my_id;
    p.wts[(size_t)n * p.top + lane] = w * p.scale;
  }
}

__global__ __launch_bounds__(256) void moe_route_kernel(RouteArgs p) {
  __shared__ float s_all[4][MOE_MAX_E];
  __shared__ float g_all[4][64];
  const int wave = threadIdx.x >> 6, n = blockIdx.x * 4 + wave;
  if (n < p.N) route_token(p, n, s_all[wave], g_all[wave]);
}

// ---------------------------------------------------------------------------------------
// Pairs listed by expert: offsets[e] .. offsets[e + 1] of `sorted` hold the pairs that chose expert
// e (in no fixed order: a pair's row of a product does not depend on its neighbours).  One block of 1024 threads.
// ---------------------------------------------------------------------------------------
struct SortSpace {
  int count[MOE_MAX_E], start[MOE_MAX_E + 1];
};
__device__ __forceinline__ void sort_block(SortSpace& sh, const int* ids, int* __restrict__ sorted, int* __restrict__ offsets, int P, int E) {
  for (int e = threadIdx.x; e < E; e += blockDim.x) sh.count[e] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < P; p += blockDim.x) {
    const int e = ids[p];
    if (e >= 0 && e < E) atomicAdd(&sh.count[e], 1);
  }
  __syncthreads();
  if (threadIdx.x < 64) {      // the first wave adds up the counts before each expert
    int before = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + threadIdx.x, mine = e < E ? sh.count[e] : 0;
      int upto = mine;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(upto, o, QVL_WAVE);
        if ((int)threadIdx.x >= o) upto += v;
      }
      if (e < E) {
        sh.start[e] = before + upto - mine;
        sh.count[e] = 0;
      }
      before += __shfl(upto, 63, QVL_WAVE);
    }
    if (threadIdx.x == 0) sh.start[E] = before;
  }
  __syncthreads();
  for (int e = threadIdx.x; e <= E; e += blockDim.x) offsets[e] = sh.start[e];
  for (int p = threadIdx.x; p < P; p += blockDim.x) {
    const int e = ids[p];
    if (e >= 0 && e < E) sorted[sh.start[e] + atomicAdd(&sh.count[e], 1)] = p;
  }
}

__global__ __launch_bounds__(1024) void moe_sort_kernel(const int* __restrict__ ids, int* __restrict__ sorted,
                                                        int* __restrict__ offsets, int P, int E) {
  __shared__ SortSpace sh;
  sort_block(sh, ids, sorted, offsets, P, E);
}

// Both for a few tokens, one block, which saves a launch: 8 tokens of 32 experts, six of them, 5.6 us and 5.8 in two.  Up to eight, two of the block's
// waves a SIMD: more share a SIMD, or come one after another, where routing by itself has a block for every four (16 tokens 6.8 us and 5.8, 64
// 16.9 and 6.0; of 256 experts in 8 groups 8 tokens 10.7 and 10.8, 16 12.5 and 11.0, 64 35.6 and 11.3).
#define ROUTE_SORT_TOKENS 8
__global__ __launch_bounds__(1024) void moe_route_sort_kernel(RouteArgs p, int* __restrict__ sorted, int* __restrict__ offsets) {
  __shared__ float s_all[ROUTE_SORT_TOKENS][MOE_MAX_E];
  __shared__ float g_all[ROUTE_SORT_TOKENS][64];
  __shared__ SortSpace sh;
  const int wave = threadIdx.x >> 6;
  if (wave < ROUTE_SORT_TOKENS && wave < p.N) route_token(p, wave, s_all[wave], g_all[wave]);
  __syncthreads();      // (a block's stores are seen by all of it)
  sort_block(sh, p.ids, sorted, offsets, p.N * p.top, p.E);
}

static int route_check(const RouteArgs& p) {
  if (p.E <= 0 || p.top <= 0 || p.groups <= 0 || p.keep <= 0 || p.keep > p.groups || p.E % p.groups || p.top > p.keep * (p.E / p.groups))
    return QVL_ERR_SHAPE;
  return p.E > MOE_MAX_E || p.groups > 64 || p.top > 64 ? QVL_ERR_LIMIT : QVL_OK;
}

// Tokens that are routed and listed in one launch.
extern "C" int qvl_moe_route_rows() { return ROUTE_SORT_TOKENS; }

// sorted, offsets: null, or also the pairs by expert as qvl_moe_sort gives them.
extern "C" int qvl_moe_route(const void* z, void* ids, void* wts, void* sorted, void* offsets, int N, int E, int top, int groups, int keep,
                             float scale, int score_fn, int normalize, float floor_, hipStream_t stream) {
  if (N <= 0) return QVL_OK;
  const RouteArgs p{(const float*)z, (int*)ids, (float*)wts, N, E, top, groups, keep, score_fn, normalize, scale, floor_};
  const int bad = route_check(p);
  if (bad) return bad;
  if (sorted && offsets && N <= ROUTE_SORT_TOKENS) {
    hipLaunchKernelGGL(moe_route_sort_kernel, dim3(1), dim3(1024), 0, stream, p, (int*)sorted, (int*)offsets);
    return qvl_launch_status();
  }
  hipLaunchKernelGGL(moe_route_kernel, dim3((N + 3) / 4), dim3(256), 0, stream, p);
  if (hipGetLastError() != hipSuccess) return QVL_ERR_LAUNCH;
  if (sorted && offsets)
    hipLaunchKernelGGL(moe_sort_kernel, dim3(1), dim3(1024), 0, stream, (const int*)ids, (int*)sorted, (int*)offsets, N * top, E);
  return qvl_launch_status();
}

extern "C" int qvl_moe_sort(const void* ids, void* sorted, void* offsets, int P, int E, hipStream_t stream) {
  if (P <= 0) return QVL_OK;
  if (E <= 0) return QVL_ERR_SHAPE;
  if (E > MOE_MAX_E) return QVL_ERR_LIMIT;
  hipLaunchKernelGGL(moe_sort_kernel, dim3(1), dim3(1024), 0, stream, (const int*)ids, (int*)sorted, (int*)offsets, P, E);
  return qvl_launch_status();
}

// ---------------------------------------------------------------------------------------
// The experts' products.  For the pair p at place i of `sorted` (expert e by `offsets`):
//   in = x[p / div, :]            (div = top for the first product, whose rows are tokens; 1 for the second)
//   plain:  out[p, c] = in . W[e, c, :]
//   gated:  g = min(in . W[e, c, :], limit), u = clamp(in . W[e, R + c, :], -limit, limit)  (no clamps if limit <= 0)
//           out[p, c] = g * sigmoid(alpha g) * (u + shift)            (W[e] holds R gate rows, then R up rows)
//   plain with act 1:  out[p, c] = max(in . W[e, c, :], 0)^2
// Any sizes and both storage types: one wave per output value, lanes split K (the sum's order is fixed).
// ---------------------------------------------------------------------------------------
struct ExpertArgs {
  const void* x;
  long long ldx;
  const void* w;        // [E, rows_w, K]
  const int* sorted;
  const int* offsets;
  void* out;            // [P, R], rows ldo values apart
  long long ldo;
  int P, E, R, K, div, gated;
  int act;              // on a plain product's values: 0 none, 1 the square of relu
  float alpha, limit, shift;
};

__device__ __forceinline__ float gated_value(float g, float u, float alpha, float limit, float shift) {
  if (limit > 0.f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
  }
  return g * sigmoid_f(alpha * g) * (u + shift);
}

__device__ __forceinline__ float plain_value(float v, int act) {
  if (act == 1) {
    v = fmaxf(v, 0.f);
    v *= v;
  }
  return v;
}

__device__ __forceinline__ int expert_of(const int* offsets, int E, int i) {
  int e = 0;
  while (e + 1 < E && offsets[e + 1] <= i) ++e;
  return e;
}

// Which expert the tile-th tile of `per` pairs belongs to, and the places of `sorted` it covers, first .. last - 1 at
// most (e = E: there is no such tile).  Every lane looks at an expert of its own, so nothing waits for one load
// after the other.
struct ExpertTile {
  int e, first, last;
};
__device__ __forceinline__ ExpertTile expert_tile(const int* __restrict__ offsets, int E, int tile, int per) {
  const int lane = threadIdx.x & 63;
  int before = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane;
    const int f = e < E ? offsets[e] : 0, l = e < E ? offsets[e + 1] : 0;
    const int nt = (l - f + per - 1) / per;
    int upto = nt;                       // tiles of this expert and of those in lower lanes
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(upto, o, QVL_WAVE);
      if (lane >= o) upto += v;
    }
    const int at = before + upto - nt;   // this expert's first tile
    const unsigned long long mine = __ballot(tile >= at && tile < at + nt);
    if (mine) {
      const int src = __ffsll(mine) - 1;
      const int skip = (tile - __shfl(at, src, QVL_WAVE)) * per;
      return ExpertTile{__builtin_amdgcn_readfirstlane(e0 + src), __builtin_amdgcn_readfirstlane(__shfl(f, src, QVL_WAVE) + skip),
                        __builtin_amdgcn_readfirstlane(__shfl(l, src, QVL_WAVE))};
    }
    before += __shfl(upto, 63, QVL_WAVE);
  }
  return ExpertTile{E, 0, 0};
}

template <typename T, typename TO>
__global__ __launch_bounds__(256) void moe_rows_kernel(ExpertArgs a) {
  const int i = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int e = expert_of(a.offsets, a.E, i);
  const int p = a.sorted[i];
  const T* xr = (const T*)a.x + (size_t)(p / a.div) * a.ldx;
  const int rows_w = a.gated ? 2 * a.R : a.R;
  const T* we = (const T*)a.w + (size_t)e * rows_w * a.K;
  for (int c = blockIdx.y * 4 + wave; c < a.R; c += gridDim.y * 4) {
    const T* wg = we + (size_t)c * a.K;
    float g = 0.f, u = 0.f;
    for (int k = lane; k < a.K; k += 64) g += ldf<T>(xr + k) * ldf<T>(wg + k);
    g = wave_sum(g);
    if (a.gated) {
      const T* wu = we + (size_t)(a.R + c) * a.K;
      for (int k = lane; k < a.K; k += 64) u += ldf<T>(xr + k) * ldf<T>(wu + k);
      u = wave_sum(u);
      g = gated_value(g, u, a.alpha, a.limit, a.shift);
    } else {
      g = plain_value(g, a.act);
    }
    if (lane == 0) stf<TO>((TO*)a.out + (size_t)p * a.ldo + c, g);
  }
}

// bfloat16 on the matrix cores, few pairs an expert (a decode step: the experts' weights are read once each and that is
// the time it takes).  An item is 32 pairs of an expert at most and the rows of W of a block of eight waves, `per` rows
// (gated: channels) a wave, operands of v_mfma_f32_32x32x16_bf16.  One block a compute unit works through item after item:
// how many experts have pairs is known on the device only, so `per` is chosen here, as the fewest that
// take no more rounds of items over all blocks than the most would.  W and the gathered rows of x come through LDS in steps
// of 64 values of K, W marked as read once, 144 KB of steps on their way, the steps of an item behind those of the item before.
// 48 pairs over 32 experts, K 3,584, 2 x 2,368 rows: 134 us = 6.3 TB/s; K 2,368, 3,584 rows: 72 us = 5.9 TB/s.  16 rows of W a
// wave straight into registers, half a line a row, 16 pairs a block: 235 and 118 us.
#define FEW_WAVES 8
#define FEW_PAIRS 32
template <bool GATED, typename TO>
__global__ __launch_bounds__(64 * FEW_WAVES) void moe_few_kernel(ExpertArgs a) {
  constexpr int F = 4, W_BYTES = FEW_WAVES * F * 1024, STAGE = W_BYTES + 4096, STAGES = 4, HALF = 2 * F;
  constexpr int MOST = GATED ? 16 : 32;
  __shared__ __attribute__((aligned(16))) char lds[STAGES * STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, hi = lane >> 5, r = lane & 31;
  int tiles = 0;                              // of at most 32 pairs, over all experts
  for (int e0 = 0; e0 < a.E; e0 += 64) {
    const int e = e0 + lane;
    int n = e < a.E ? (a.offsets[e + 1] - a.offsets[e] + FEW_PAIRS - 1) / FEW_PAIRS : 0;
#pragma unroll
    for (int o = 32; o; o >>= 1) n += __shfl_xor(n, o, QVL_WAVE);
    tiles += n;
  }
  tiles = __builtin_amdgcn_readfirstlane(tiles);
  const int blocks = gridDim.x;
  auto groups_of = [&](int per) { return (a.R + FEW_WAVES * per - 1) / (FEW_WAVES * per); };
  const long long most_items = (long long)tiles * groups_of(MOST);
  const long long rounds_all = (most_items + blocks - 1) / blocks;
  const long long shares = max(1ll, rounds_all * blocks * FEW_WAVES);
  int per = (int)max(1ll, min((long long)MOST, ((long long)tiles * a.R + shares - 1) / shares));
  while (per < MOST && (long long)tiles * groups_of(per) > rounds_all * blocks) ++per;
  const int groups = groups_of(per), items = tiles * groups;
  const int first_item = blockIdx.x, rounds = first_item < items ? (items - first_item + blocks - 1) / blocks : 0;
  const int ksteps = (a.K + 63) / 64, steps = ksteps * rounds;
  const int last_chunks = a.K % 64 ? (a.K % 64) / 8 : 8;     // of a last step, 8 values each
  // Row of W behind row i of a wave's tile (-1: there is none).  Row i's sums are number 4 (i / 8) + i mod 4 of the lanes whose
  // hi is (i / 4) mod 2; gated: the first half of a lane's sums are gates, the others their up values.
  auto w_row = [&](int c0, int i) {
    int j = i, up = 0;
    if (GATED) {
      const int s = 4 * (i >> 3) + (i & 3);
      up = s >= HALF;
      j = ((i >> 2) & 1) * HALF + s - up * HALF;
    }
    return (j < per && c0 + j < a.R) ? c0 + j + up * a.R : -1;
  };
  // this lane's fetches: rows 8 j + lane / 8 of the wave's tile, the row's chunk (lane mod 8) ^ ((row / 2) mod 8), and of x
  // row 8 (wave mod 4) + lane / 8 (two waves fetch the same: every wave then waits for as many).  A row that does not exist
  // is read from one that does; its sums are not stored.
  uint32_t fw[F], fx = 0;
  const char* w_base = (const char*)a.w;
  const int x_place = wave & 3, x_row = 8 * x_place + (lane >> 3);
  auto column = [&](int item) { return ((item % groups) * FEW_WAVES + wave) * per; };
  auto set_item = [&](int item) __attribute__((always_inline)) {
    const ExpertTile at = expert_tile(a.offsets, a.E, item / groups, FEW_PAIRS);
    w_base = (const char*)a.w + (size_t)at.e * (GATED ? 2 * a.R : a.R) * a.K * 2;
    const int c0 = column(item), exists = max(w_row(c0, 0), 0);
#pragma unroll
    for (int j = 0; j < F; ++j) {
      const int rho = 8 * j + (lane >> 3);
      int n = w_row(c0, rho);
      if (n < 0) n = exists;
      fw[j] = (uint32_t)n * (uint32_t)a.K * 2 + 16 * ((lane & 7) ^ ((rho >> 1) & 7));
    }
    const int i = at.first + x_row;
    fx = (uint32_t)(a.sorted[i < at.last ? i : at.first] / a.div) * (uint32_t)a.ldx * 2 + 16 * ((lane & 7) ^ ((x_row >> 1) & 7));
  };
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)&lds[0];
  // blocks begin an item at different places of K and go round, so that they do not all ask the same few memory channels
  const int turn = (int)((blockIdx.x * 29u) % (unsigned)ksteps);
  int asked = 0, ask_k = 0, ask_item = first_item, ask_stage = 0, ask_at = turn;
  auto ask = [&]() __attribute__((always_inline)) {          // the next step's fetches, if there is one
    if (asked >= steps) return;
    if (ask_k == 0) set_item(ask_item);
    const uint32_t at = lds0 + ask_stage * STAGE, k = (uint32_t)ask_at * 128;
    // chunks of a last step that lie beyond K are read from its first: they are not multiplied
    const int chunks = ask_at == ksteps - 1 ? last_chunks : 8;
    auto back = [&](int row) { const int c = (lane & 7) ^ ((row >> 1) & 7); return c < chunks ? 0u : 16u * c; };
#pragma unroll
    for (int j = 0; j < F; ++j) tp_fetch16_once(w_base, fw[j] + k - back(8 * j + (lane >> 3)), at + (wave * F + j) * 1024);
    tp_fetch16(a.x, fx + k - back(x_row), at + W_BYTES + x_place * 1024);
    ++asked;
    ask_stage = ask_stage + 1 == STAGES ? 0 : ask_stage + 1;
    if (++ask_at == ksteps) ask_at = 0;
    if (++ask_k == ksteps) {
      ask_k = 0;
      ask_item += blocks;
    }
  };
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i) ask();
  const uint32_t sw = (r >> 1) & 7;
  tp_f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  int stage = 0, at_k = turn, left = ksteps, item = first_item;
  for (int s = 0; s < steps; ++s) {
    tp_wait_steps<STAGES - 2, F + 1>(asked - 1 - s);      // all but the steps asked for behind this one have come
    tp_wait_lds();
    tp_barrier();                           // every wave's part of the step is there, and the step before has been read
    ask();
    const char* pw = lds + stage * STAGE + (wave * F * 8 + r) * 128;
    const char* px = lds + stage * STAGE + W_BYTES + r * 128;
    tp_bf16x8 w8[4], x8[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      w8[k] = *reinterpret_cast<const tp_bf16x8*>(pw + (((2 * k + hi) ^ sw) << 4));
      x8[k] = *reinterpret_cast<const tp_bf16x8*>(px + (((2 * k + hi) ^ sw) << 4));
    }
    if (last_chunks < 8 && at_k == ksteps - 1) {           // chunks beyond K are no part of the sums
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (2 * k + hi >= last_chunks) w8[k] = x8[k] = tp_bf16x8{};
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w8[k], x8[k], acc, 0, 0, 0);
    stage = stage + 1 == STAGES ? 0 : stage + 1;
    if (++at_k == ksteps) at_k = 0;
    if (--left) continue;
    // an item's sums: a lane holds pair r of the tile
    const ExpertTile at = expert_tile(a.offsets, a.E, item / groups, FEW_PAIRS);
    const int c0 = column(item), i = at.first + r;
    if (i < at.last) {
      TO* o = (TO*)a.out + (size_t)a.sorted[i] * a.ldo + c0;
#pragma unroll
      for (int n = 0; n < (GATED ? HALF : 16); ++n) {
        const int j = GATED ? hi * HALF + n : 8 * (n >> 2) + 4 * hi + (n & 3);
        if (j >= per || c0 + j >= a.R) continue;
        stf<TO>(o + j, GATED ? gated_value(acc[n], acc[n + HALF], a.alpha, a.limit, a.shift) : plain_value(acc[n], a.act));
      }
    }
#pragma unroll
    for (int n = 0; n < 16; ++n) acc[n] = 0.f;
    left = ksteps;
    item += blocks;
  }
  tp_wait_fetches<0>();
}

// Many pairs an expert: tiles of TILE_M pairs x TILE_N rows of W (gated: TILE_N / 2 gate rows and the up rows
// of the same outputs), K in steps of TILE_K through LDS.  The 256 threads fetch the next step's values of x
// (gathered rows) and of W into registers while the step in LDS is multiplied, then put them into the other
// of two buffers; the 16-byte chunks of a row are exchanged by bits of the row number, so that the 16 lanes
// that read one chunk of 16 rows hit all 64 banks.  The four waves stand 2 x 2: each owns 64 pairs and
// 16 NW rows of W (gated: 8 NW gate rows and their up rows): 4 NW products of 16 x 16 x 32 a step from
// 4 + NW operand reads.
// Measured on 12,288 pairs over 32 experts, K 3,584, 2 x 2,368 rows (gate|up): TILE_K 64, NW 4: 1,000 us; TILE_K 32:
// 1,030; NW 8 (tiles of 128 x 256: fewer operand reads and fetched bytes a product, but the sums leave
// room for one wave a SIMD): 1,220 (TILE_K 64), 1,420 (TILE_K 32); fetching two steps ahead into a
// second set of registers: 1,230.
#ifndef TILE_K
#define TILE_K 64
#endif
#ifndef NW
#define NW 4                                           // tiles of 16 rows of W a wave multiplies
#endif
#define TILE_M 128
#define TILE_N (32 * NW)
#define ROW_CHUNKS (TILE_K / 8)                        // 16-byte chunks of a row of a tile
#define X_CHUNKS (TILE_M * ROW_CHUNKS / 256)           // chunks of x a thread fetches a step
#define W_CHUNKS (TILE_N * ROW_CHUNKS / 256)           // and of W

__device__ __forceinline__ int lds_slot(int row, int chunk) {
#if TILE_K == 64
  return row * 8 + (chunk ^ ((row >> 1) & 7));
#else
  return row * 4 + (chunk ^ ((row >> 2) & 3));
#endif
}

template <bool GATED, typename TO>
__global__ __launch_bounds__(256) void moe_tile_kernel(ExpertArgs a, int tiles_m, int tiles_n) {
  __shared__ __attribute__((aligned(16))) uint4 s_x[2][TILE_M * ROW_CHUNKS];
  __shared__ __attribute__((aligned(16))) uint4 s_w[2][TILE_N * ROW_CHUNKS];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lg = lane >> 4, r = lane & 15;
  const int wm = wave >> 1, wn = wave & 1;
  // Blocks go to the XCDs in turn (block b to XCD b mod 8, each with an L2 of its own).  The 32 blocks that
  // an XCD's compute units hold at a time are made 4 tiles of pairs x 8 tiles of rows of W: they walk K at
  // about the same pace, so a slice of x is fetched into that L2 once for 8 blocks and a slice of W once for 4.
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  const int super = (idx >> 5) * 8 + xcd, inner = idx & 31;
  const int supers_m = (tiles_m + 3) / 4;
  const int tile_n = (super / supers_m) * 8 + (inner >> 2);
  int tile = (super % supers_m) * 4 + (inner & 3);
  if (tile >= tiles_m || tile_n >= tiles_n) return;
  int e = 0, first = 0, last = 0;
  for (; e < a.E; ++e) {
    first = a.offsets[e];
    last = a.offsets[e + 1];
    const int nt = (last - first + TILE_M - 1) / TILE_M;
    if (tile < nt) break;
    tile -= nt;
  }
  if (e >= a.E) return;
  first += tile * TILE_M;
  constexpr int HALF = TILE_N / 2;
  constexpr int OUT_COLS = GATED ? HALF : TILE_N;           // output columns of a block
  const int c0 = tile_n * OUT_COLS;
  const int rows_w = GATED ? 2 * a.R : a.R;
  const bf16_t* we = (const bf16_t*)a.w + (size_t)e * rows_w * a.K;

  // what this thread fetches each step: chunks of 16 bytes of x and of W.  No load stands inside a branch
  // (the compiler would wait for each before the next): a chunk that does not exist is read from one
  // that does (row 0, column 0 of the step) and replaced by zeros.
  const bf16_t* gx[X_CHUNKS];
  const bf16_t* gw[W_CHUNKS];
  bool x_ok[X_CHUNKS], w_ok[W_CHUNKS];
#pragma unroll
  for (int j = 0; j < X_CHUNKS; ++j) {
    const int id = threadIdx.x + 256 * j, row = id / ROW_CHUNKS, ch = id % ROW_CHUNKS;
    const int i = first + row;
    const int pair = i < last ? a.sorted[i] : -1;
    x_ok[j] = pair >= 0;
    gx[j] = (const bf16_t*)a.x + (size_t)(pair < 0 ? 0 : pair / a.div) * a.ldx + 8 * ch;
  }
#pragma unroll
  for (int j = 0; j < W_CHUNKS; ++j) {
    const int id = threadIdx.x + 256 * j, row = id / ROW_CHUNKS, ch = id % ROW_CHUNKS;
    int wrow;                                               // row of W_e behind row `row` of the tile
    if (GATED) wrow = row < HALF ? c0 + row : a.R + c0 + (row - HALF);
    else wrow = c0 + row;
    w_ok[j] = GATED ? (c0 + (row % HALF) < a.R) : (wrow < a.R);
    gw[j] = we + (size_t)(w_ok[j] ? wrow : 0) * a.K + 8 * ch;
  }
  uint4 rx[X_CHUNKS], rw[W_CHUNKS];
  auto fetch = [&](int k) {
    const int ch = threadIdx.x % ROW_CHUNKS;                // 256 is a multiple of ROW_CHUNKS: the same for every j
    const bool k_ok = k + 8 * ch < a.K;
    const int at = k_ok ? k : k - 8 * ch;
#pragma unroll
    for (int j = 0; j < X_CHUNKS; ++j) {
      const uint4 v = *reinterpret_cast<const uint4*>(gx[j] + at);
      const bool ok = x_ok[j] && k_ok;
      rx[j] = uint4{ok ? v.x : 0u, ok ? v.y : 0u, ok ? v.z : 0u, ok ? v.w : 0u};
    }
#pragma unroll
    for (int j = 0; j < W_CHUNKS; ++j) {
      const uint4 v = *reinterpret_cast<const uint4*>(gw[j] + at);
      const bool ok = w_ok[j] && k_ok;
      rw[j] = uint4{ok ? v.x : 0u, ok ? v.y : 0u, ok ? v.z : 0u, ok ? v.w : 0u};
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int j = 0; j < X_CHUNKS; ++j) {
      const int id = threadIdx.x + 256 * j;
      s_x[buf][lds_slot(id / ROW_CHUNKS, id % ROW_CHUNKS)] = rx[j];
    }
#pragma unroll
    for (int j = 0; j < W_CHUNKS; ++j) {
      const int id = threadIdx.x + 256 * j;
      s_w[buf][lds_slot(id / ROW_CHUNKS, id % ROW_CHUNKS)] = rw[j];
    }
  };
  f32x4_t acc[NW][4];    // [tile of 16 rows of W][tile of 16 pairs]
#pragma unroll
  for (int n = 0; n < NW; ++n)
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // rows of the W tile this wave multiplies: gated, its gate rows and the up rows of the same outputs
  constexpr int PER_WAVE = GATED ? 8 * NW : 16 * NW;        // output columns of a wave
  int wrow0[NW];
#pragma unroll
  for (int n = 0; n < NW; ++n)
    wrow0[n] = GATED ? (n < NW / 2 ? wn * PER_WAVE + n * 16 : HALF + wn * PER_WAVE + (n - NW / 2) * 16) : wn * PER_WAVE + n * 16;

  fetch(0);
  put(0);
  __syncthreads();
  int buf = 0;
  for (int k = 0; k < a.K; k += TILE_K) {
    const bool more = k + TILE_K < a.K;
    if (more) fetch(k + TILE_K);
#pragma unroll
    for (int kk = 0; kk < TILE_K / 32; ++kk) {
      bf16x8_t fx[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) fx[m] = __builtin_bit_cast(bf16x8_t, s_x[buf][lds_slot(wm * 64 + m * 16 + r, 4 * kk + lg)]);
#pragma unroll
      for (int n = 0; n < NW; ++n) {
        const bf16x8_t fw = __builtin_bit_cast(bf16x8_t, s_w[buf][lds_slot(wrow0[n] + r, 4 * kk + lg)]);
#pragma unroll
        for (int m = 0; m < 4; ++m) acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw, fx[m], acc[n][m], 0, 0, 0);
      }
    }
    if (more) put(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
  // a lane holds, of (n, m): pair wm 64 + 16 m + r, W rows wrow0[n] + 4 lg .. + 3
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int i = first + wm * 64 + m * 16 + r;
    if (i >= last) continue;
    const int pair = a.sorted[i];
    TO* o = (TO*)a.out + (size_t)pair * a.ldo;
#pragma unroll
    for (int n = 0; n < (GATED ? NW / 2 : NW); ++n) {
      const int c = c0 + wn * PER_WAVE + n * 16 + 4 * lg;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (c + j >= a.R) break;
        float v = acc[n][m][j];
        if (GATED) v = gated_value(v, acc[n + NW / 2][m][j], a.alpha, a.limit, a.shift);
        else v = plain_value(v, a.act);
        stf<TO>(o + c + j, v);
      }
    }
  }
}

// The same product through the inner loop of tile_product.h: tiles of 128 pairs x 256 rows of W (gated: 128 gate
// rows and the up rows of the same outputs; a wave's gate and up values of an output end in one lane).  K must be a
// multiple of 32 and offsets within x and within an expert's W 32-bit.  Measured on 12,384 pairs over 32 experts, K
// 3,584: 2 x 2,368 rows 574 us (tiles of 128 x 256 with all waves in step: 874); down 291.
// Tiles of 256 pairs give each operand in LDS to twice the products, for half a tile more of padding an expert: from WIDE_PAIRS pairs an
// expert on (on average), where that comes out in fewer or shorter rounds of blocks (qvl_moe_wide_pairs).  Of 128 and of 256, gated | down: 32 experts, 2 x
// 2,368 x 3,584, 387 pairs 604 and 475 us | 304 and 260, 450 604 and 614 | 302 and 357; 8 experts, 2 x 1,376 x 2,048, 387 pairs 72 and 105 |
// 35 and 48, 562 104 and 108 | 58 and 51.
typedef Tile<4, 2, 4, 4> ExpertsTile;
typedef Tile<2, 4, 8, 4> WideTile;
#define WIDE_PAIRS 256

template <typename TO>
__device__ __forceinline__ void store_expert4(TO* o, const float* v, int n, bool whole);
template <>
__device__ __forceinline__ void store_expert4<float>(float* o, const float* v, int n, bool whole) {
  if (whole) {
    *reinterpret_cast<float4*>(o) = float4{v[0], v[1], v[2], v[3]};
  } else {
    for (int i = 0; i < 4; ++i)
      if (i < n) o[i] = v[i];
  }
}
template <>
__device__ __forceinline__ void store_expert4<bf16_t>(bf16_t* o, const float* v, int n, bool whole) {
  if (whole) {
    *reinterpret_cast<uint2*>(o) = uint2{(uint32_t)f32_to_bf16(v[0]) | (uint32_t)f32_to_bf16(v[1]) << 16,
                                         (uint32_t)f32_to_bf16(v[2]) | (uint32_t)f32_to_bf16(v[3]) << 16};
  } else {
    for (int i = 0; i < 4; ++i)
      if (i < n) o[i] = f32_to_bf16(v[i]);
  }
}

template <typename T, bool GATED, typename TO>
__global__ __launch_bounds__(512) void moe_stream_kernel(ExpertArgs a, int tiles_m, int tiles_n, int whole4) {
  __shared__ __attribute__((aligned(16))) char lds[T::LDS];
  // blocks of one XCD at a time: 4 tiles of pairs x 8 tiles of rows of W (see moe_tile_kernel)
  const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  const int super = (idx >> 5) * 8 + xcd, inner = idx & 31;
  const int supers_m = (tiles_m + 3) / 4;
  const int tile_n = (super / supers_m) * 8 + (inner >> 2), tile_m = (super % supers_m) * 4 + (inner & 3);
  if (tile_m >= tiles_m || tile_n >= tiles_n) return;
  const ExpertTile at = expert_tile(a.offsets, a.E, tile_m, T::BM);
  if (at.e >= a.E) return;
  constexpr int OUT_COLS = GATED ? T::BN / 2 : T::BN;
  const int c0 = tile_n * OUT_COLS;
  const int rows_w = GATED ? 2 * a.R : a.R;
  const bf16_t* we = (const bf16_t*)a.w + (size_t)at.e * rows_w * a.K;
  T t;
  // rows that do not exist are read from one that does; their sums are not stored
  t.set_rows(
      [&](int h, int rho) {
        if (GATED) return (uint32_t)(((size_t)(c0 + rho < a.R ? c0 + rho : 0) + (h ? a.R : 0)) * a.K * 2);
        const int n = c0 + T::w_row(h, rho);
        return (uint32_t)((size_t)(n < a.R ? n : 0) * a.K * 2);
      },
      [&](int h, int rho) {
        const int i = at.first + T::x_row(h, rho);
        return (uint32_t)((size_t)(a.sorted[i < at.last ? i : at.first] / a.div) * a.ldx * 2);
      });
  t.multiply(lds, we, a.x, (a.K + 63) / 64, a.K % 64 != 0);
#pragma unroll
  for (int m = 0; m < T::MT; ++m) {
    const int i = at.first + (t.wm * T::MT + m) * 16 + t.r;
    if (i >= at.last) continue;
    TO* o = (TO*)a.out + (size_t)a.sorted[i] * a.ldo;
#pragma unroll
    for (int n = 0; n < (GATED ? T::NH : T::NT); ++n) {
      const int c = c0 + (t.wn * (GATED ? T::NH : T::NT) + n) * 16 + 4 * t.g;
      if (c >= a.R) continue;
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[j] = GATED ? gated_value(t.acc[n][m][j], t.acc[n + (GATED ? T::NH : 0)][m][j], a.alpha, a.limit, a.shift)
                     : plain_value(t.acc[n][m][j], a.act);
      store_expert4<TO>(o + c, v, a.R - c, whole4 && c + 4 <= a.R);
    }
  }
}

// How long tiles of bm pairs take, in microseconds: the rounds of the XCD that gets most blocks (they go there in groups of 4 x 8 tiles),
// each a step of 64 values of K after the other, `alone` where most compute units are idle and `full` where all work, and 2.9 more for its
// first fetches and its stores.  The pairs' shares are not known on the host: an expert is taken to waste
// `waste` of a tile.
static double stream_us(int P, int E, int bm, double waste, int tiles_n, int K, double alone, double full, int cus) {
  const int there = P / bm + (E < P ? E : P), used = (int)((double)P / bm + waste * E + 0.5), real = used < there ? used : there;
  const int supers_m = (there + 3) / 4, supers = supers_m * ((tiles_n + 7) / 8);
  double most = (double)real * tiles_n / 8;
  if (supers <= 1024) {
    long long blocks[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int s = 0; s < supers; ++s) {
      const int m = real - 4 * (s % supers_m), n = tiles_n - 8 * (s / supers_m);
      blocks[s & 7] += (m < 0 ? 0 : m < 4 ? m : 4) * (n < 8 ? n : 8);
    }
    for (long long b : blocks) most = (double)b > most ? (double)b : most;
  }
  const double rounds = most * 8 / cus, whole = floor(rounds), rest = rounds - whole;
  const int steps = (K + 63) / 64;
  return whole * (steps * full + 2.9) + (rest > 0 ? steps * (alone + (full - alone) * rest) + 2.9 : 0.0);
}
// Whether tiles of 256 pairs are the faster ones.  Of 264 products (8, 32 and 64 experts of 768 to 4,096 outputs, 262 to 1,300 pairs each) two are
// over 2 per cent slower than with tiles of 128 (8 and 12), and 1.7 per cent of the time is lost on average; by the number of pairs alone 66 were
// (up to 46), and 4.9 per cent was lost.
extern "C" int qvl_moe_wide_pairs(int P, int E, int R, int K, int gated, int cus) {
  if (P <= 0 || E <= 0 || R <= 0 || K <= 0 || cus <= 0 || P < WIDE_PAIRS * (long long)E) return 0;
  const int cols = gated ? ExpertsTile::BN / 2 : ExpertsTile::BN, tiles_n = (R + cols - 1) / cols;
  // (0.4 is what routers' choices at random wasted; 0.55 as well, so that some pairs more in one expert's tile are not a round more)
  const double narrow = stream_us(P, E, ExpertsTile::BM, 0.4, tiles_n, K, 0.678, 0.825, cus);
  return stream_us(P, E, WideTile::BM, 0.4, tiles_n, K, 0.967, 1.361, cus) < narrow &&
         stream_us(P, E, WideTile::BM, 0.55, tiles_n, K, 0.967, 1.361, cus) < narrow;
}

// x_dtype / out_dtype: 0 float32, 1 bfloat16.  float32 operands write float32; bfloat16 operands
// write either.  The matrix-core kernel runs for bfloat16 with K a multiple of 8 and rows of x on
// 16-byte boundaries; `big_tiles` asks for the kernels with tiles of 128 or 256 pairs through LDS (many pairs an expert).
extern "C" int qvl_moe_experts(const void* x, long long ldx, int x_dtype, const void* w, const void* sorted,
                               const void* offsets, void* out, long long ldo, int out_dtype, int P, int E, int R, int K,
                               int div,
                               int gated, float alpha, float limit, float shift, int act, int big_tiles,
                               int cus, hipStream_t stream) {
  if (P <= 0) return QVL_OK;
  if (E <= 0 || R <= 0 || K <= 0 || div <= 0 || ldx < K || ldo < R || !x || !w || !sorted || !offsets || !out) return QVL_ERR_SHAPE;
  ExpertArgs a;
  a.x = x; a.ldx = ldx; a.w = w; a.sorted = (const int*)sorted; a.offsets = (const int*)offsets; a.out = out; a.ldo = ldo;
  a.P = P; a.E = E; a.R = R; a.K = K; a.div = div; a.gated = gated; a.act = gated ? 0 : act; a.alpha = alpha; a.limit = limit; a.shift = shift;
  if (x_dtype == 1 && K % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0) {
    if (out_dtype != 0 && out_dtype != 1) return QVL_ERR_DTYPE;
    const unsigned long long x_rows = (unsigned long long)((P + div - 1) / div);
    if (big_tiles && K % 32 == 0 && x_rows * (unsigned long long)ldx * 2 < 0xffff0000ull &&
        (unsigned long long)(gated ? 2 * R : R) * K * 2 < 0xffff0000ull) {
      const bool wide = qvl_moe_wide_pairs(P, E, R, K, gated, cus);
      const int bm = wide ? WideTile::BM : ExpertsTile::BM;
      const int cols = gated ? ExpertsTile::BN / 2 : ExpertsTile::BN;
      const int tiles_m = P / bm + (E < P ? E : P), tiles_n = (R + cols - 1) / cols;
      if ((long long)tiles_m * tiles_n > 0x7ffffff0ll) return QVL_ERR_LIMIT;
      const int supers = ((tiles_m + 3) / 4) * ((tiles_n + 7) / 8);
      const dim3 tgrid((unsigned)((supers + 7) / 8) * 8 * 32);
      const int whole4 = ldo % 4 == 0 && ((uintptr_t)out % 16) == 0;    // four neighbouring results as one store
#define STREAM(T, G, TO) hipLaunchKernelGGL((moe_stream_kernel<T, G, TO>), tgrid, dim3(512), 0, stream, a, tiles_m, tiles_n, whole4)
#define SHAPE(G, TO)                     \
  do {                                   \
    if (wide) STREAM(WideTile, G, TO);   \
    else STREAM(ExpertsTile, G, TO);     \
  } while (0)
      if (gated && out_dtype == 1) SHAPE(true, bf16_t);
      else if (gated) SHAPE(true, float);
      else if (out_dtype == 1) SHAPE(false, bf16_t);
      else SHAPE(false, float);
#undef SHAPE
#undef STREAM
      return qvl_launch_status();
    }
    if (big_tiles) {
      const int cols = gated ? TILE_N / 2 : TILE_N;
      const int tiles_m = P / TILE_M + (E < P ? E : P), tiles_n = (R + cols - 1) / cols;
      if ((long long)tiles_m * tiles_n > 0x7ffffff0ll) return QVL_ERR_LIMIT;
      // whole groups of 4 x 8 tiles, 8 groups (one per XCD) at a time
      const int supers = ((tiles_m + 3) / 4) * ((tiles_n + 7) / 8);
      const dim3 tgrid((unsigned)((supers + 7) / 8) * 8 * 32);
      if (gated && out_dtype == 1)
        hipLaunchKernelGGL((moe_tile_kernel<true, bf16_t>), tgrid, dim3(256), 0, stream, a, tiles_m, tiles_n);
      else if (gated) hipLaunchKernelGGL((moe_tile_kernel<true, float>), tgrid, dim3(256), 0, stream, a, tiles_m, tiles_n);
      else if (out_dtype == 1)
        hipLaunchKernelGGL((moe_tile_kernel<false, bf16_t>), tgrid, dim3(256), 0, stream, a, tiles_m, tiles_n);
      else hipLaunchKernelGGL((moe_tile_kernel<false, float>), tgrid, dim3(256), 0, stream, a, tiles_m, tiles_n);
      return qvl_launch_status();
    }
    if (cus <= 0) return QVL_ERR_SHAPE;
    if (x_rows * (unsigned long long)ldx * 2 < 0xffff0000ull && (unsigned long long)(gated ? 2 * R : R) * K * 2 < 0xffff0000ull &&
        (long long)(P / FEW_PAIRS + (E < P ? E : P)) * ((R + FEW_WAVES - 1) / FEW_WAVES) < 0x7ffffff0ll) {
#define FEW(G, TO) hipLaunchKernelGGL((moe_few_kernel<G, TO>), dim3(cus), dim3(64 * FEW_WAVES), 0, stream, a)
      if (gated && out_dtype == 1) FEW(true, bf16_t);
      else if (gated) FEW(true, float);
      else if (out_dtype == 1) FEW(false, bf16_t);
      else FEW(false, float);
#undef FEW
      return qvl_launch_status();
    }
  }
  int by = (R + 3) / 4;
  if (by > 64) by = 64;
  const dim3 grid(P, by);
  if (x_dtype == 0 && out_dtype == 0) hipLaunchKernelGGL((moe_rows_kernel<float, float>), grid, dim3(256), 0, stream, a);
  else if (x_dtype == 1 && out_dtype == 1) hipLaunchKernelGGL((moe_rows_kernel<bf16_t, bf16_t>), grid, dim3(256), 0, stream, a);
  else if (x_dtype == 1 && out_dtype == 0) hipLaunchKernelGGL((moe_rows_kernel<bf16_t, float>), grid, dim3(256), 0, stream, a);
  else return QVL_ERR_DTYPE;
  return qvl_launch_status();
}

// ---------------------------------------------------------------------------------------
// out[n, :] = sum over k of wts[n, k] * y[n top + k, :], in the order of k, plus `extra[n, :]` (what
// a shared expert gave: float32 or bfloat16, or float32 slabs added in order; null: nothing).
// ---------------------------------------------------------------------------------------
// four consecutive values as float32
template <typename T> __device__ __forceinline__ float4 ld4(const T* p);
template <> __device__ __forceinline__ float4 ld4<float>(const float* p) { return *reinterpret_cast<const float4*>(p); }
template <> __device__ __forceinline__ float4 ld4<bf16_t>(const bf16_t* p) {
  const uint2 v = *reinterpret_cast<const uint2*>(p);
  return float4{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                __uint_as_float(v.y & 0xffff0000u)};
}

// VEC 4: a thread owns four neighbouring columns of one token (H a multiple of 4); VEC 1: one column.
// Its loads are all on their way before the first is used.
template <typename TY, typename TX, int VEC>
__global__ __launch_bounds__(256) void moe_combine_kernel(const TY* __restrict__ y, const float* __restrict__ wts,
                                                          const TX* __restrict__ extra, int nslabs, long long slab_stride,
                                                          float* __restrict__ out, int top, int H) {
  const size_t n = blockIdx.x;
  const int c = (blockIdx.y * 256 + threadIdx.x) * VEC;
  if (c >= H) return;
  const float* wr = wts + n * top;
  if (VEC == 4) {
    float4 v = float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int k = 0; k < top; ++k) {
      const float4 t = ld4<TY>(y + (n * top + k) * (size_t)H + c);
      const float w = wr[k];
      v.x += w * t.x; v.y += w * t.y; v.z += w * t.z; v.w += w * t.w;
    }
    if (extra) {
      float4 x = ld4<TX>(extra + n * H + c);
      for (int s = 1; s < nslabs; ++s) {
        const float4 t = ld4<TX>(extra + (size_t)s * slab_stride + n * H + c);
        x.x += t.x; x.y += t.y; x.z += t.z; x.w += t.w;
      }
      v.x += x.x; v.y += x.y; v.z += x.z; v.w += x.w;
    }
    *reinterpret_cast<float4*>(out + n * H + c) = v;
  } else {
    float v = 0.f;
#pragma unroll 8
    for (int k = 0; k < top; ++k) v += wr[k] * ldf<TY>(y + (n * top + k) * (size_t)H + c);
    if (extra) {
      float x = ldf<TX>(extra + n * H + c);
      for (int s = 1; s < nslabs; ++s) x += ldf<TX>(extra + (size_t)s * slab_stride + n * H + c);
      v += x;
    }
    out[n * H + c] = v;
  }
}

extern "C" int qvl_moe_combine(const void* y, int y_dtype, const void* wts, const void* extra, int extra_dtype,
                               int nslabs, long long slab_stride, void* out, int N, int top, int H, hipStream_t stream) {
  if (N <= 0) return QVL_OK;
  if (top <= 0 || H <= 0 || nslabs < 1 || (nslabs > 1 && extra_dtype != 0)) return QVL_ERR_SHAPE;
#define LAUNCH(TY, TX)                                                                                         \
  if (vec4)                                                                                                        \
    hipLaunchKernelGGL((moe_combine_kernel<TY, TX, 4>), dim3(N, (H / 4 + 255) / 256), dim3(256), 0, stream,          \
                       (const TY*)y, (const float*)wts, (const TX*)extra, nslabs, slab_stride, (float*)out, top, H); \
  else                                                                                                             \
    hipLaunchKernelGGL((moe_combine_kernel<TY, TX, 1>), dim3(N, (H + 255) / 256), dim3(256), 0, stream,              \
                       (const TY*)y, (const float*)wts, (const TX*)extra, nslabs, slab_stride, (float*)out, top, H)
  const bool vec4 = H % 4 == 0 && slab_stride % 4 == 0 && ((uintptr_t)y % 16) == 0 && ((uintptr_t)extra % 16) == 0 &&
                    ((uintptr_t)out % 16) == 0;
  if (y_dtype == 0 && extra_dtype == 0) { LAUNCH(float, float); }
  else if (y_dtype == 0 && extra_dtype == 1) { LAUNCH(float, bf16_t); }
  else if (y_dtype == 1 && extra_dtype == 0) { LAUNCH(bf16_t, float); }
  else if (y_dtype == 1 && extra_dtype == 1) { LAUNCH(bf16_t, bf16_t); }
  else return QVL_ERR_DTYPE;
#undef LAUNCH
  return qvl_launch_status();
}
