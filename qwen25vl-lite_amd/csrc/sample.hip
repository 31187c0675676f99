// Sampling one token per logits row on the device (reference src/qwen25vl_lite/sampling.py:44-106):
// penalties over the tokens generated so far, then greedy argmax (temperature <= 0) or
// temperature, top-k, min-p, top-p and a draw from what is left.  A row's token depends on nothing
// else in the batch: every sum is either of whole numbers, which no order changes, or runs in a
// fixed order.
//
// The draw inverts the distribution function with a uniform number u of the row: the token is the
// first index whose running probability mass exceeds u.  u comes with the row's settings, or from
// the row's seed (below).
//
// What bounds it: a row of 152,064 logits is 0.6 MB, and one compute unit reads some tens of GB/s by
// itself, so a row is cut into pieces of 4,096 scores and each pass over it runs in as many blocks.
// A threshold (the k-th largest score; the score at which the mass reaches top-p) is found by its
// bits, 11, 11 and 10 at a time: a pass counts the scores, or adds up their mass, by the next bits
// among those that agree with the bits already fixed, and the next kernel's blocks pick the bin.
// Masses are whole numbers of 2^-40 of the largest score's (of more for rows beyond 2^23 scores, whose sum
// would not fit 64 bits), which is finer than a float32 sum of them and lets the blocks add in any order.  One block a row that searched bit by bit, 32 passes for each
// threshold, took 3.70 ms for 64 rows of 152,064 (greedy, top-p, top-k with top-p and penalties, min-p
// in turn); these passes together 117 in nine kernels.
//
// Most rows need none of these passes: what their cuts leave is a short list.  Each group of 256 scores of a row has a
// largest one; the k-th largest of those is no larger than the k-th largest score, and scores that far below the largest one that
// all of a row's could not make up 1 - top_p never matter.  So one pass gathers what such a bound leaves (and adds up all
// mass, where top-p needs it), and a block a row finds the thresholds among these few and draws, with the same sums.  Rows
// whose list is longer than LIST, or whose list does not reach top-p, go the long way; the others' blocks there end at once.
// The 64 rows above: 45 us in three kernels, all of it reading and finding.  Rows that draw from all of their scores are not tried.
#include "common.h"
#include <cmath>
#include <cstddef>
#include <type_traits>

#define PIECE 4096          // scores a block owns in a pass over a row
#define THREADS 256
#define BINS 2048           // bins of a threshold's search: 11 bits of a score's key at a time
#define CHUNKS 1024         // contiguous ranges of a row whose masses the draw adds one after the other
#define GROUPS 16           // groups of 256 scores of a piece, whose largest are kept
#define LIST 1024           // scores of a short list
#define GUESS 620           // scores that are expected in a list where top-p alone cuts: some below LIST, since their number is guessed
#define STEPS 2048          // steps of 1/64 below a row's largest score that bounds are told apart by; the last one is open

struct RowParams {
  float temperature, top_p, min_p, u;
  float repetition, presence, frequency;
  int top_k;
  int prev_begin, prev_end;  // this row's generated tokens in prev_ids
  uint32_t seed;             // with `seeded`: u is the first draw of a generator with this seed
  int seeded;
};

struct ArgmaxPart {
  float value;
  int index;
};

// What is known of a row's two thresholds between the passes: [0] the k-th largest score's key (a
// count), [1] the key at which the mass reaches top-p.  After the search of level l, `key` has the
// bits of the levels up to l, and `left` says how much of the target the scores with those bits must bring.
struct Threshold {
  uint32_t key[4];
  unsigned long long left[4];
};

// A row's scratch memory.
struct RowScratch {
  Threshold found[2];
  float u;
  unsigned int listed;          // scores asked into the list (more than LIST: it is of no use)
  int todo_row;                 // of the i-th row: the i-th of those that go the long way
  int pad;
  unsigned long long all_mass, pad2;
  float list_score[LIST];
  int list_index[LIST];
  unsigned int count[3][BINS];
  unsigned long long mass[3][BINS];
  float chunk_mass[CHUNKS];
};
static_assert(offsetof(RowScratch, chunk_mass) % 16 == 0 && sizeof(RowScratch) % 16 == 0, "the chunks' masses are read four at a time");

__device__ __forceinline__ uint32_t order_key(float f) {
  uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ bool penalised(const RowParams& p) {
  return p.prev_end > p.prev_begin && (p.repetition != 1.f || p.presence != 0.f || p.frequency != 0.f);
}
__device__ __forceinline__ bool cuts_k(const RowParams& p, int V) { return p.temperature > 0.f && p.top_k > 0 && p.top_k < V; }
__device__ __forceinline__ bool cuts_p(const RowParams& p) { return p.temperature > 0.f && p.top_p < 1.f; }
// A row that draws from all of its scores, too many for a list.
__device__ __forceinline__ bool draws_whole(const RowParams& p, int V) {
  return p.temperature > 0.f && V > LIST && !cuts_k(p, V) && !cuts_p(p) && !(p.min_p > 0.f);
}

// The row's scores: the penalised ones have been written out, already divided by the temperature.
struct Scores {
  const float* at;
  float temperature;   // 1 where nothing is left to divide
  __device__ __forceinline__ float operator()(int i) const { return at[i] / temperature; }
};
__device__ __forceinline__ Scores scores_of(const RowParams& p, const float* logits, const float* scores, int m, int V) {
  const bool out = penalised(p);
  return Scores{(out ? scores : logits) + (size_t)m * V, out || p.temperature <= 0.f ? 1.f : p.temperature};
}

// Thread t's scores of a piece: number j is the piece's score piece_index(j, t), those beyond n the first one again.
__device__ __forceinline__ int piece_index(int j, int tid) { return (j >> 2) * 4 * THREADS + 4 * tid + (j & 3); }
__device__ __forceinline__ void load_piece(const float* at, int n, int V, float (&v)[PIECE / THREADS]) {
  const int tid = threadIdx.x;
  if (V % 4 == 0 && (uintptr_t)at % 16 == 0) {        // then a piece's end is a multiple of four, too
#pragma unroll
    for (int j = 0; j < PIECE / THREADS; j += 4) {
      const int i = piece_index(j, tid);
      const float4 x = *reinterpret_cast<const float4*>(at + (i < n ? i : 0));
      v[j] = x.x; v[j + 1] = x.y; v[j + 2] = x.z; v[j + 3] = x.w;
    }
  } else {
#pragma unroll
    for (int j = 0; j < PIECE / THREADS; ++j) {
      const int i = piece_index(j, tid);
      v[j] = at[i < n ? i : 0];
    }
  }
}

__device__ __forceinline__ void better(float& bv, int& bi, float ov, int oi) {
  if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
}
// The wave's largest value, the lowest index among equals; every lane gets it.
__device__ __forceinline__ void wave_argmax(float& bv, int& bi) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o, QVL_WAVE);
    const int oi = __shfl_xor(bi, o, QVL_WAVE);
    better(bv, bi, ov, oi);
  }
}
// A row's largest score from its pieces' (whole block, result for every thread).
__device__ __forceinline__ ArgmaxPart row_argmax(const ArgmaxPart* parts, int m, int pieces, int V, ArgmaxPart* s_best) {
  if (threadIdx.x < 64) {
    float bv = -INFINITY;
    int bi = V;
    for (int s = threadIdx.x; s < pieces; s += 64) {
      const ArgmaxPart q = parts[(size_t)m * pieces + s];
      better(bv, bi, q.value, q.index);
    }
    wave_argmax(bv, bi);
    if (threadIdx.x == 0) *s_best = ArgmaxPart{bv, bi};
  }
  __syncthreads();
  return *s_best;
}

// The first number of the 32-bit Mersenne Twister (M. Matsumoto and T. Nishimura, 1998, the
// initialisation of 2002) seeded with `seed`, its lower 24 bits as a fraction: what the row's generator
// draws first.  The first output needs words 0, 1 and 397 of the state only.
__device__ float first_uniform(uint32_t seed) {
  uint32_t word = seed, w1 = 0;
  for (uint32_t i = 1; i <= 397; ++i) {
    word = 1812433253u * (word ^ (word >> 30)) + i;
    if (i == 1) w1 = word;
  }
  const uint32_t mixed = (seed & 0x80000000u) | (w1 & 0x7fffffffu);
  uint32_t y = word ^ (mixed >> 1) ^ ((w1 & 1u) ? 0x9908b0dfu : 0u);
  y ^= y >> 11;
  y ^= (y << 7) & 0x9d2c5680u;
  y ^= (y << 15) & 0xefc60000u;
  y ^= y >> 18;
  return (float)(y & 0xffffffu) * (1.0f / 16777216.0f);
}

// The first pass: a piece's largest score (of penalised rows the penalised and scaled scores, which are
// written to `scores`) and, of rows that draw, its groups' largest.  With scratch there is one block more a row,
// which draws the row's uniform number.
__global__ __launch_bounds__(THREADS) void sample_scan_kernel(const float* __restrict__ logits, float* __restrict__ scores,
                                                              const RowParams* __restrict__ params,
                                                              const int* __restrict__ prev_ids,
                                                              RowScratch* __restrict__ scratch,
                                                              ArgmaxPart* __restrict__ parts, float* __restrict__ groups,
                                                              int* __restrict__ todo, int M, int V, int pieces) {
  __shared__ int seen[PIECE];     // how often each of the piece's tokens has been generated
  __shared__ float vals[THREADS / 64];
  __shared__ int idxs[THREADS / 64];
  const int tid = threadIdx.x;
  int at = blockIdx.x;
  if (scratch) {
    // the rows' own blocks come first: a seed's first number is a chain of 397 products
    if (at < M) {
      if (tid == 0) {
        const RowParams p = params[at];
        scratch[at].listed = draws_whole(p, V) ? LIST + 1u : 0u;
        scratch[at].all_mass = 0ull;
        if (at == 0) *todo = 0;
        scratch[at].u = p.temperature > 0.f && p.seeded ? first_uniform(p.seed) : p.u;
      }
      return;
    }
    at -= M;
  }
  const int m = at / pieces, s = at - m * pieces;
  const RowParams p = params[m];
  const bool draws = p.temperature > 0.f;
  const int lo = s * PIECE, n = min(PIECE, V - lo);
  float v[PIECE / THREADS];
  load_piece(logits + (size_t)m * V + lo, n, V, v);
  if (penalised(p)) {
#pragma unroll
    for (int j = 0; j < PIECE / THREADS; ++j) seen[j * THREADS + tid] = 0;
    __syncthreads();
    const int* prev = prev_ids + p.prev_begin;
    const int L = p.prev_end - p.prev_begin;
    for (int i = tid; i < L; i += THREADS) {
      const int t = prev[i];
      if (t >= lo && t < lo + n) atomicAdd(&seen[t - lo], 1);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PIECE / THREADS; ++j) {
      const int count = seen[piece_index(j, tid)];
      if (count == 0) continue;
      float x = v[j];
      if (p.repetition != 1.f) x = x > 0.f ? x / p.repetition : x * p.repetition;
      v[j] = x - p.presence - p.frequency * (float)count;
    }
#pragma unroll
    for (int j = 0; j < PIECE / THREADS; ++j) {
      const int i = piece_index(j, tid);
      if (draws) v[j] = v[j] / p.temperature;
      if (draws && i < n) scores[(size_t)m * V + lo + i] = v[j];
    }
  } else if (draws) {
#pragma unroll
    for (int j = 0; j < PIECE / THREADS; ++j) v[j] = v[j] / p.temperature;
  }
  float bv = -INFINITY;
  int bi = V;
#pragma unroll
  for (int j = 0; j < PIECE / THREADS; ++j) {
    const int i = piece_index(j, tid);
    if (i < n && v[j] > bv) { bv = v[j]; bi = lo + i; }   // indices rise within a thread: the first of equals stays
  }
  if (scratch && draws) {
    float top = fmaxf(bv, __shfl_xor(bv, 1, QVL_WAVE));
#pragma unroll
    for (int o = 2; o < THREADS / GROUPS; o <<= 1) top = fmaxf(top, __shfl_xor(top, o, QVL_WAVE));
    if (tid % (THREADS / GROUPS) == 0) groups[((size_t)m * pieces + s) * GROUPS + tid / (THREADS / GROUPS)] = top;
  }
  wave_argmax(bv, bi);
  if ((tid & 63) == 0) { vals[tid >> 6] = bv; idxs[tid >> 6] = bi; }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < THREADS / 64; ++w) better(bv, bi, vals[w], idxs[w]);
    parts[(size_t)m * pieces + s] = ArgmaxPart{bv, bi};
  }
}

// `one`: the largest score's mass, a power of two
__device__ __forceinline__ unsigned long long mass_of(float e, float one) { return e > 0.f ? (unsigned long long)(e * one) : 0ull; }

// The sum of the threads before this one (whole block; one place for each wave in s_wave).
template <typename T>
__device__ __forceinline__ T sum_before(T own, T* s_wave) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  T sum = own;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const T x = __shfl_up(sum, o, QVL_WAVE);
    if (lane >= o) sum += x;
  }
  if (lane == 63) s_wave[wave] = sum;
  __syncthreads();
  sum -= own;
  for (int w = 0; w < wave; ++w) sum += s_wave[w];
  return sum;
}

// The running sums of x, added one after the other from `acc` on (one thread; n a multiple of 16, both on 16-byte boundaries).  What
// bounds it is a sum's latency, if the values come early enough: 16 are read while those before are added.
__device__ __forceinline__ float chain(const float* x, float* sums, int n, float acc) {
  float4 v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = reinterpret_cast<const float4*>(x)[i];
  for (int t = 0; t < n; t += 16) {
    const int next = t + 16 < n ? t + 16 : t;
    float4 w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[i] = v[i];
      v[i] = reinterpret_cast<const float4*>(x + next)[i];
    }
    __builtin_amdgcn_sched_barrier(0);      // (the reads first)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[i].x = acc += w[i].x;
      w[i].y = acc += w[i].y;
      w[i].z = acc += w[i].z;
      w[i].w = acc += w[i].w;
      reinterpret_cast<float4*>(sums + t)[i] = w[i];
    }
  }
  return acc;
}

// The lowest and the highest number (whole block) of those that a wave has in `first` and `last`, whose bit 0 is number `base`; joined to
// what the wave had.  Minima and maxima in shared memory would take a wave's lanes one by one.
struct Ends {
  int low, high;
  __device__ __forceinline__ void join(unsigned long long first, unsigned long long last, int base) {
    if (first) low = min(low, base + __ffsll(first) - 1);
    if (last) high = max(high, base + 63 - __clzll(last));
  }
  __device__ __forceinline__ void share(int2* s_ends) {
    if ((threadIdx.x & 63) == 0) s_ends[threadIdx.x >> 6] = int2{low, high};
    __syncthreads();
    for (int w = 0; w < THREADS / 64; ++w) {
      low = min(low, s_ends[w].x);
      high = max(high, s_ends[w].y);
    }
  }
};

// How far below the row's largest score a score is, in steps.
__device__ __forceinline__ int step_of(float x, float mx) { return (int)fminf((mx - x) * 64.f, (float)(STEPS - 1)); }

// Gathers the scores that the row's cuts can leave, and all mass where top-p alone cuts.
__global__ __launch_bounds__(THREADS) void sample_list_kernel(const float* __restrict__ logits, const float* __restrict__ scores,
                                                              const RowParams* __restrict__ params,
                                                              RowScratch* __restrict__ scratch,
                                                              const ArgmaxPart* __restrict__ parts,
                                                              const float* __restrict__ groups, int V, int pieces, int guess, float one) {
  __shared__ unsigned int steps[STEPS], sums[THREADS / 64];
  __shared__ unsigned long long mass[THREADS / 64];
  __shared__ ArgmaxPart s_best;
  __shared__ int s_k, s_p;
  __shared__ unsigned int s_count, s_base;
  const int m = blockIdx.y, s = blockIdx.x, tid = threadIdx.x;
  const RowParams p = params[m];
  if (p.temperature <= 0.f || draws_whole(p, V)) return;
  RowScratch& r = scratch[m];
  const Scores score = scores_of(p, logits, scores, m, V);
  const int lo = s * PIECE, n = min(PIECE, V - lo);
  float v[PIECE / THREADS];
  load_piece(score.at + lo, n, V, v);
  const bool k_cut = cuts_k(p, V), p_cut = cuts_p(p);
  const float mx = row_argmax(parts, m, pieces, V, &s_best).value;
  int bound = STEPS - 1;          // scores up to this many steps below the largest go into the list
  if (p.min_p > 0.f) bound = min(bound, (int)fminf(-logf(p.min_p) * 64.f + 2.f, (float)(STEPS - 1)));
  if (k_cut || (p_cut && !(p.min_p > 0.f))) {
    for (int i = tid; i < STEPS; i += THREADS) steps[i] = 0u;
    if (tid == 0) s_k = s_p = STEPS - 1;
    __syncthreads();
    const float* top = groups + (size_t)m * pieces * GROUPS;
    for (int i = tid; i < pieces * GROUPS; i += THREADS) {
      const float x = top[i];
      if (x > -INFINITY) atomicAdd(&steps[step_of(x, mx)], 1u);
    }
    __syncthreads();
    constexpr int PER = STEPS / THREADS;
    unsigned int own[PER], sum = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      own[i] = steps[tid * PER + i];
      sum += own[i];
    }
    const unsigned int k = (unsigned int)p.top_k;
    unsigned int before = sum_before(sum, sums);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (before < k && before + own[i] >= k) s_k = tid * PER + i;
      if (before < (unsigned int)guess && before + own[i] >= (unsigned int)guess) s_p = tid * PER + i;
      before += own[i];
    }
    __syncthreads();
    if (k_cut) bound = min(bound, s_k);
    else bound = min(s_p, (int)fminf(logf((float)V / fmaxf(1.f - p.top_p, 1e-7f)) * 64.f + 2.f, (float)(STEPS - 1)));
  }
  if (bound == STEPS - 1 && V > LIST) {        // every score
    if (s == 0 && tid == 0) atomicAdd(&r.listed, LIST + 1u);
    return;
  }
  if (tid == 0) s_count = 0u;
  __syncthreads();
  // a score that is no number, or none that is: the long way
  bool odd = !(fabsf(mx) < INFINITY);
  const bool sum_all = p_cut && !k_cut && !(p.min_p > 0.f);
  unsigned long long own_mass = 0;
  unsigned int place[PIECE / THREADS];
#pragma unroll
  for (int j = 0; j < PIECE / THREADS; ++j) {
    place[j] = 0xffffffffu;
    if (piece_index(j, tid) >= n) continue;
    v[j] = v[j] / score.temperature;
    odd |= v[j] != v[j];
    if (sum_all) own_mass += mass_of(expf(v[j] - mx), one);
    if (step_of(v[j], mx) <= bound) place[j] = atomicAdd(&s_count, 1u);
  }
  if (odd) atomicAdd(&s_count, LIST + 1u);
  if (sum_all) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) own_mass += __shfl_xor(own_mass, o, QVL_WAVE);
    if ((tid & 63) == 0) mass[tid >> 6] = own_mass;
  }
  __syncthreads();
  if (tid == 0) {
    s_base = s_count ? atomicAdd(&r.listed, s_count < LIST + 1u ? s_count : LIST + 1u) : 0u;
    if (sum_all) {
      unsigned long long sum = 0;
      for (int w = 0; w < THREADS / 64; ++w) sum += mass[w];
      if (sum) atomicAdd(&r.all_mass, sum);
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PIECE / THREADS; ++j) {
    if (place[j] == 0xffffffffu) continue;
    const unsigned int at = s_base + place[j];
    if (at < LIST) {
      r.list_score[at] = v[j];
      r.list_index[at] = lo + piece_index(j, tid);
    }
  }
}

// A row's token from its list, by the rules of the long way: thresholds by the keys' bits, masses of chunks added from their first
// index on, chunks one after the other (chunks without mass add nothing, so those of the list are enough).  A threshold is found
// by steps below the largest score first, then among the scores of its step.  What is left is put in order by chunks: each score's place
// is found among its chunk's alone.  Compared with all others, 900 scores took 42 us (8 rows of 32,000, min-p 0.05), this 16.
__global__ __launch_bounds__(THREADS) void sample_short_kernel(const RowParams* __restrict__ params,
                                                               RowScratch* __restrict__ scratch,
                                                               const ArgmaxPart* __restrict__ parts, int* __restrict__ out,
                                                               int* __restrict__ todo, int V, int pieces, float one) {
  constexpr int PER = LIST / THREADS, OWN = STEPS / THREADS;
  __shared__ unsigned long long steps[STEPS], s_sum[THREADS / 64], s_above;
  __shared__ unsigned long long in_mass[LIST];        // the threshold's step: its scores' masses (or ones) and keys
  __shared__ uint32_t in_key[LIST], s_cut;
  __shared__ int index[LIST], kept_index[LIST], run_at[LIST], s_step, s_in;
  __shared__ int2 s_ends[THREADS / 64];
  __shared__ float weight[LIST];
  __shared__ __attribute__((aligned(16))) float run_mass[LIST], run_sum[LIST];
  __shared__ unsigned int s_counts[THREADS / 64], s_all;
  __shared__ float s_z;
  __shared__ ArgmaxPart s_best;
  const int m = blockIdx.x, tid = threadIdx.x;
  const RowParams p = params[m];
  const ArgmaxPart best = row_argmax(parts, m, pieces, V, &s_best);
  if (p.temperature <= 0.f) {
    if (tid == 0) out[m] = best.index < V ? best.index : 0;
    return;
  }
  RowScratch& r = scratch[m];
  const bool k_cut = cuts_k(p, V), p_cut = cuts_p(p);
  const float mx = best.value;
  const int n = r.listed <= LIST ? (int)r.listed : 0;       // (0: the long way; a list has the largest score at least)
  float w[PER];
  uint32_t key[PER];
  int ix[PER], st[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int at = i * THREADS + tid;
    const float x = at < n ? r.list_score[at] : -INFINITY;
    ix[i] = at < n ? r.list_index[at] : 0;
    key[i] = order_key(x);
    st[i] = at < n ? step_of(x, mx) : -1;
    w[i] = at < n ? expf(x - mx) : 0.f;
    if (p.min_p > 0.f && w[i] < p.min_p) w[i] = 0.f;
  }
  // the key at which the parts of the scores from the largest down reach the target: false if they do not
  auto threshold = [&](auto part, unsigned long long target) -> bool {
    for (int i = tid; i < STEPS; i += THREADS) steps[i] = 0ull;
    if (tid == 0) {
      s_step = -1;
      s_in = 0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const unsigned long long x = part(i);
      if (st[i] >= 0 && x) atomicAdd(&steps[st[i]], x);
    }
    __syncthreads();
    unsigned long long own[OWN], sum = 0;
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
      own[i] = steps[tid * OWN + i];
      sum += own[i];
    }
    unsigned long long before = sum_before(sum, s_sum);
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
      if (before < target && before + own[i] >= target) {
        s_step = tid * OWN + i;
        s_above = before;
      }
      before += own[i];
    }
    __syncthreads();
    if (s_step < 0) return false;
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (st[i] == s_step) {
        const int at = atomicAdd(&s_in, 1);
        in_key[at] = key[i];
        in_mass[at] = part(i);
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (st[i] != s_step) continue;
      unsigned long long above = s_above, reach = s_above;
      for (int j = 0; j < s_in; ++j) {
        above += in_key[j] > key[i] ? in_mass[j] : 0ull;
        reach += in_key[j] >= key[i] ? in_mass[j] : 0ull;
      }
      if (above < target && reach >= target) s_cut = key[i];
    }
    __syncthreads();
    return true;
  };
  if (k_cut && n > 0) {
    // (fewer than k in the list: the others have no mass by min-p)
    if (threshold([&](int i) { return 1ull; }, (unsigned long long)p.top_k)) {
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if (key[i] < s_cut) w[i] = 0.f;
    }
    __syncthreads();
  }
  bool done = n > 0;
  if (p_cut && done) {
    // the mass of what top-k and min-p leave; without them every score has a part
    unsigned long long all = r.all_mass;
    if (k_cut || p.min_p > 0.f) {
      unsigned long long sum = 0;
#pragma unroll
      for (int i = 0; i < PER; ++i) sum += mass_of(w[i], one);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, QVL_WAVE);
      if ((tid & 63) == 0) s_sum[tid >> 6] = sum;
      __syncthreads();
      all = 0;
      for (int i = 0; i < THREADS / 64; ++i) all += s_sum[i];
      __syncthreads();
    }
    done = threshold([&](int i) { return mass_of(w[i], one); }, max(1ull, (unsigned long long)ceil((double)p.top_p * (double)all)));
    if (done) {
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if (key[i] < s_cut) w[i] = 0.f;
    }
  }
  bool left = false;        // (a min-p above 1 leaves nothing)
#pragma unroll
  for (int i = 0; i < PER; ++i) left |= w[i] > 0.f;
  done = __syncthreads_or(done && left);
  if (!done) {
    for (int i = tid; i < 3 * BINS; i += THREADS) {
      (&r.count[0][0])[i] = 0u;
      (&r.mass[0][0])[i] = 0ull;
    }
    if (tid == 0) scratch[atomicAdd(todo, 1)].todo_row = m;
    return;
  }
  // what is left, by the chunks of the draw: a chunk's scores in the order of their indices, the chunks that have any one after the other
  unsigned int* count = reinterpret_cast<unsigned int*>(steps);
  unsigned int* start = count + CHUNKS;
  for (int i = tid; i < CHUNKS; i += THREADS) count[i] = 0u;
  __syncthreads();
  const int C = (V + CHUNKS - 1) / CHUNKS;
  int nth[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i)
    if (w[i] > 0.f) nth[i] = (int)atomicAdd(&count[ix[i] / C], 1u);
  __syncthreads();
  constexpr int MINE = CHUNKS / THREADS;
  unsigned int has[MINE], sum = 0;                  // how many chunks with scores, and 16 bits above, how many scores
#pragma unroll
  for (int i = 0; i < MINE; ++i) {
    has[i] = count[tid * MINE + i];
    sum += (has[i] << 16) + (has[i] ? 1u : 0u);
  }
  const unsigned int before = sum_before(sum, s_counts);
  if (tid == THREADS - 1) s_all = before + sum;
  unsigned int at = before;
#pragma unroll
  for (int i = 0; i < MINE; ++i) {
    start[tid * MINE + i] = at >> 16;
    at += (has[i] << 16) + (has[i] ? 1u : 0u);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PER; ++i)
    if (w[i] > 0.f) kept_index[start[ix[i] / C] + nth[i]] = ix[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (!(w[i] > 0.f)) continue;
    const int c = ix[i] / C, from = (int)start[c], others = (int)count[c];
    int rank = from;
    for (int j = 0; j < others; ++j) rank += kept_index[from + j] < ix[i];
    index[rank] = ix[i];
    weight[rank] = w[i];
  }
  const int kept = (int)(s_all >> 16), runs = (int)(s_all & 0xffffu), padded = (runs + 15) / 16 * 16;
  for (int i = runs + tid; i < padded; i += THREADS) run_mass[i] = 0.f;
  __syncthreads();
  at = before;
#pragma unroll
  for (int i = 0; i < MINE; ++i) {
    if (has[i]) {
      float acc = 0.f;
      for (unsigned int j = 0; j < has[i]; ++j) acc += weight[(at >> 16) + j];
      run_at[at & 0xffffu] = (int)(at >> 16);
      run_mass[at & 0xffffu] = acc;
    }
    at += (has[i] << 16) + (has[i] ? 1u : 0u);
  }
  __syncthreads();
  if (tid == 0) s_z = chain(run_mass, run_sum, padded, 0.f);
  __syncthreads();
  const float aim = r.u * s_z;
  Ends ends{LIST, 0};
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int t = i * THREADS + tid;
    ends.join(__ballot(t < runs && run_sum[t] > aim), 0ull, t & ~63);
  }
  ends.share(s_ends);
  if (tid == 0) {
    const bool found = ends.low < LIST;
    const int t = found ? ends.low : runs - 1, from = run_at[t], to = t + 1 < runs ? run_at[t + 1] : kept;
    const float pick = found ? aim - (t ? run_sum[t - 1] : 0.f) : INFINITY;
    float acc = 0.f;
    int token = index[from];
    for (int j = from; j < to; ++j) {
      token = index[j];
      acc += weight[j];
      if (acc > pick) break;
    }
    out[m] = token;
  }
}

// The highest of the bins at which the sum of the bins from the top down reaches `target` (the lowest
// bin if none does), and what the bins above it bring.  Whole block; T the bins' type.
template <typename T>
__device__ void pick_bin(const T* bins, unsigned long long target, int& bin, unsigned long long& above,
                         unsigned long long* s_sum, int* s_bin, unsigned long long* s_above) {
  constexpr int PER = BINS / THREADS;
  const int tid = threadIdx.x;
  // thread t owns the bins from the top: BINS - 1 - t PER ... downwards
  unsigned long long own[PER], sum = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    own[i] = bins[BINS - 1 - tid * PER - i];
    sum += own[i];
  }
  s_sum[tid] = sum;
  if (tid == 0) { *s_bin = 0; *s_above = 0; }
  __syncthreads();
  for (int o = 1; o < THREADS; o <<= 1) {      // running sums over the threads
    const unsigned long long x = tid >= o ? s_sum[tid - o] : 0ull;
    __syncthreads();
    s_sum[tid] += x;
    __syncthreads();
  }
  unsigned long long before = s_sum[tid] - sum;
  if (before < target && s_sum[tid] >= target) {   // one thread at most
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (before + own[i] >= target) {
        *s_bin = BINS - 1 - tid * PER - i;
        *s_above = before;
        break;
      }
      before += own[i];
    }
  } else if (tid == THREADS - 1 && s_sum[tid] < target) {
    *s_above = s_sum[tid] - own[PER - 1];
  }
  __syncthreads();
  bin = *s_bin;
  above = *s_above;
}

// The key's bits that level l looks at.
__device__ __forceinline__ int level_shift(int level) { return level == 0 ? 21 : (level == 1 ? 10 : 0); }

// What level `level` of a search begins with: the bits fixed so far and the part of the target that is
// left, from the bins of the level before.  The row's first block keeps them for the kernels behind.
template <bool MASS>
__device__ void search_state(RowScratch& r, const RowParams& p, int level, bool keeper, uint32_t& key,
                             unsigned long long& left, unsigned long long* s_sum, int* s_bin, unsigned long long* s_above) {
  key = 0;
  left = 0;
  if (level == 0) return;
  Threshold& t = r.found[MASS ? 1 : 0];
  unsigned long long target;
  if (level == 1) {
    if (MASS) {
      // top_p of the mass of what top-k and min-p have left: the sum of the first level's bins
      constexpr int PER = BINS / THREADS;
      unsigned long long sum = 0;
      for (int i = 0; i < PER; ++i) sum += r.mass[0][threadIdx.x * PER + i];
      s_sum[threadIdx.x] = sum;
      __syncthreads();
      for (int o = THREADS / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) s_sum[threadIdx.x] += s_sum[threadIdx.x + o];
        __syncthreads();
      }
      // (a top_p below float32's range is 0 here: the largest score stays)
      target = max(1ull, (unsigned long long)ceil((double)p.top_p * (double)s_sum[0]));
      __syncthreads();
    } else {
      target = (unsigned long long)p.top_k;
    }
  } else {
    key = t.key[level - 2];
    target = t.left[level - 2];
  }
  int bin;
  unsigned long long above;
  if (MASS) pick_bin(r.mass[level - 1], target, bin, above, s_sum, s_bin, s_above);
  else pick_bin(r.count[level - 1], target, bin, above, s_sum, s_bin, s_above);
  key |= (uint32_t)bin << level_shift(level - 1);
  left = target - above;
  if (keeper && threadIdx.x == 0) {
    t.key[level - 1] = key;
    t.left[level - 1] = left;
  }
}

// The k-th largest score's key.  `last`: the last level's bins have not been searched yet.
__device__ uint32_t kth_key(RowScratch& r, const RowParams& p, bool last, bool keeper, unsigned long long* s_sum, int* s_bin,
                            unsigned long long* s_above) {
  if (!last) return r.found[0].key[2];
  uint32_t key;
  unsigned long long left;
  search_state<false>(r, p, 3, keeper, key, left, s_sum, s_bin, s_above);
  __syncthreads();
  return key;
}

// One level of a search: the pieces' scores into the row's bins.
template <bool MASS>
__global__ __launch_bounds__(THREADS) void sample_bins_kernel(const float* __restrict__ logits, const float* __restrict__ scores,
                                                              const RowParams* __restrict__ params,
                                                              RowScratch* __restrict__ scratch,
                                                              const ArgmaxPart* __restrict__ parts,
                                                              const int* __restrict__ todo, int V, int pieces,
                                                              int level, float one) {
  typedef typename std::conditional<MASS, unsigned long long, unsigned int>::type bin_t;
  __shared__ bin_t bins[BINS];
  __shared__ unsigned long long s_sum[THREADS], s_above;
  __shared__ int s_bin;
  __shared__ ArgmaxPart s_best;
  if ((int)blockIdx.y >= *todo) return;
  const int m = scratch[blockIdx.y].todo_row, s = blockIdx.x, tid = threadIdx.x;
  const RowParams p = params[m];
  if (!(MASS ? cuts_p(p) : cuts_k(p, V))) return;
  RowScratch& r = scratch[m];
  const Scores score = scores_of(p, logits, scores, m, V);
  const int lo = s * PIECE, n = min(PIECE, V - lo);
  float v[PIECE / THREADS];
  load_piece(score.at + lo, n, V, v);
  for (int i = tid; i < BINS; i += THREADS) bins[i] = 0;
  const float mx = MASS ? row_argmax(parts, m, pieces, V, &s_best).value : 0.f;
  uint32_t key;
  unsigned long long left;
  uint32_t kth = 0;
  if (MASS && cuts_k(p, V)) kth = kth_key(r, p, level == 0, s == 0, s_sum, &s_bin, &s_above);
  search_state<MASS>(r, p, level, s == 0, key, left, s_sum, &s_bin, &s_above);
  __syncthreads();
  const int shift = level_shift(level);
  const uint32_t fixed = level == 0 ? 0u : (0xffffffffu << level_shift(level - 1)), low = level == 2 ? 0x3ffu : 0x7ffu;
#pragma unroll
  for (int j = 0; j < PIECE / THREADS; ++j) {
    if (piece_index(j, tid) >= n) continue;
    const float x = v[j] / score.temperature;
    const uint32_t k = order_key(x);
    if ((k & fixed) != key) continue;
    if (MASS) {
      if (k < kth) continue;
      const float e = expf(x - mx);
      if (p.min_p > 0.f && e < p.min_p) continue;
      const unsigned long long w = mass_of(e, one);
      if (w) atomicAdd(&bins[(k >> shift) & low], (bin_t)w);
    } else {
      atomicAdd(&bins[(k >> shift) & low], (bin_t)1);
    }
  }
  __syncthreads();
  bin_t* out = MASS ? (bin_t*)r.mass[level] : (bin_t*)r.count[level];
  for (int i = tid; i < BINS; i += THREADS)
    if (bins[i]) atomicAdd(&out[i], bins[i]);
}

// The masses of the row's chunks for the draw, each added from its first index to its last.
#define CHUNKS_A_BLOCK 32
__global__ __launch_bounds__(THREADS) void sample_chunks_kernel(const float* __restrict__ logits, const float* __restrict__ scores,
                                                                const RowParams* __restrict__ params,
                                                                RowScratch* __restrict__ scratch,
                                                                const ArgmaxPart* __restrict__ parts,
                                                                const int* __restrict__ todo, int V, int pieces) {
  __shared__ float tile[CHUNKS_A_BLOCK][65];
  __shared__ unsigned long long s_sum[THREADS], s_above;
  __shared__ int s_bin;
  __shared__ ArgmaxPart s_best;
  if ((int)blockIdx.y >= *todo) return;
  const int m = scratch[blockIdx.y].todo_row, tid = threadIdx.x;
  const RowParams p = params[m];
  RowScratch& r = scratch[m];
  const Scores score = scores_of(p, logits, scores, m, V);
  const float mx = row_argmax(parts, m, pieces, V, &s_best).value;
  uint32_t cut = 0;
  if (cuts_k(p, V)) cut = kth_key(r, p, !cuts_p(p), blockIdx.x == 0, s_sum, &s_bin, &s_above);
  if (cuts_p(p)) {
    uint32_t key;
    unsigned long long left;
    search_state<true>(r, p, 3, blockIdx.x == 0, key, left, s_sum, &s_bin, &s_above);
    cut = max(cut, key);
  }
  const int C = (V + CHUNKS - 1) / CHUNKS, first = blockIdx.x * CHUNKS_A_BLOCK;
  constexpr int EACH = CHUNKS_A_BLOCK * 64 / THREADS;
  float mine = 0.f, x[EACH];
  // 64 scores of every chunk, a wave one chunk's at a time; asked for while those before are added
  auto index = [&](int at, int j) { return (long long)(first + ((j * THREADS + tid) >> 6)) * C + at + (tid & 63); };
  auto there = [&](int at, int j) { return at + (tid & 63) < C && index(at, j) < V; };
  auto load = [&](int at) {
#pragma unroll
    for (int j = 0; j < EACH; ++j) x[j] = there(at, j) ? score.at[index(at, j)] : 0.f;
  };
  load(0);
  for (int at = 0; at < C; at += 64) {
    float e[EACH];
#pragma unroll
    for (int j = 0; j < EACH; ++j) {
      // (one assignment: of `e[j] = ...; if (...) e[j] = 0` the compiler lost the second for j = 0)
      const float v = x[j] / score.temperature, w = expf(v - mx);
      const bool kept = there(at, j) & (order_key(v) >= cut) & !(p.min_p > 0.f && w < p.min_p);
      e[j] = kept ? w : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < EACH; ++j) tile[(j * THREADS + tid) >> 6][tid & 63] = e[j];
    if (at + 64 < C) load(at + 64);
    __syncthreads();
    if (tid < CHUNKS_A_BLOCK)
#pragma unroll 32
      for (int o = 0; o < 64; ++o) mine += tile[tid][o];
  }
  if (tid < CHUNKS_A_BLOCK) r.chunk_mass[first + tid] = mine;
}

// The token: the largest score's index, or the draw.  What bounds it is the chain of 1,024 sums; 12 us a row where minima and maxima in shared
// memory, which take a wave's lanes one by one, and sums read eight at a time made it 20 to 28.
__global__ __launch_bounds__(THREADS) void sample_pick_kernel(const float* __restrict__ logits, const float* __restrict__ scores,
                                                              const RowParams* __restrict__ params,
                                                              RowScratch* __restrict__ scratch,
                                                              const ArgmaxPart* __restrict__ parts, int* __restrict__ out,
                                                              const int* __restrict__ todo, int V, int pieces) {
  __shared__ __attribute__((aligned(16))) float sums[CHUNKS], prefix[CHUNKS];
  __shared__ ArgmaxPart s_best;
  __shared__ int2 s_ends[THREADS / 64];
  __shared__ float s_z;
  int m = blockIdx.x;
  const int tid = threadIdx.x;
  if (scratch) {
    if ((int)blockIdx.x >= *todo) return;
    m = scratch[blockIdx.x].todo_row;
  }
  const RowParams p = params[m];
  const ArgmaxPart best = row_argmax(parts, m, pieces, V, &s_best);
  if (!scratch) {                      // no row draws
    if (tid == 0) out[m] = best.index < V ? best.index : 0;
    return;
  }
  RowScratch& r = scratch[m];
  const float mx = best.value;
  for (int i = tid; i < CHUNKS / 4; i += THREADS)
    reinterpret_cast<float4*>(sums)[i] = reinterpret_cast<const float4*>(r.chunk_mass)[i];
  __syncthreads();
  if (tid == 0) s_z = chain(sums, prefix, CHUNKS, 0.f);      // prefix[t]: the mass up to chunk t
  __syncthreads();
  const float target = r.u * s_z;
  Ends ends{CHUNKS, 0};
#pragma unroll
  for (int i = 0; i < CHUNKS / THREADS; ++i) {
    const int t = i * THREADS + tid;
    const bool any = sums[t] > 0.f;
    ends.join(__ballot(any && prefix[t] > target), __ballot(any), t & ~63);
  }
  ends.share(s_ends);
  const bool found = ends.low < CHUNKS;
  const int chunk = found ? ends.low : ends.high;
  const float pick = found ? target - (chunk ? prefix[chunk - 1] : 0.f) : INFINITY;
  // within the chunk: the scores' masses from its first index on, until they exceed the rest
  uint32_t cut = cuts_k(p, V) ? r.found[0].key[2] : 0u;
  if (cuts_p(p)) cut = max(cut, r.found[1].key[2]);
  const Scores score = scores_of(p, logits, scores, m, V);
  const int C = (V + CHUNKS - 1) / CHUNKS, lo = chunk * C, hi = min(V, lo + C);
  float acc = 0.f;
  Ends token{V, lo};
  for (int at = lo; at < hi; at += THREADS) {
    float e = 0.f;
    if (at + tid < hi) {
      const float x = score(at + tid), w = expf(x - mx);
      e = w > 0.f && order_key(x) >= cut && !(p.min_p > 0.f && w < p.min_p) ? w : 0.f;
    }
    __syncthreads();                   // sums, prefix and ends have been read
    sums[tid] = e;
    __syncthreads();
    if (tid == 0) acc = chain(sums, prefix, (min(hi - at, THREADS) + 15) / 16 * 16, acc);
    __syncthreads();
    token.join(__ballot(e > 0.f && prefix[tid] > pick), __ballot(e > 0.f), at + (tid & ~63));
    token.share(s_ends);
    if (token.low < V) break;
  }
  if (tid == 0) out[m] = token.low < V ? token.low : token.high;
}

static int pieces_of(int V) { return (V + PIECE - 1) / PIECE; }

// Of the groups of a row's whole pieces, how many have a score above the one with GUESS scores above it, if these lie anywhere: a
// group has none with probability exp(-GUESS / groups).  (384 of the 592 groups of 151,936 scores; all but one of 32,000's 112.  As many
// groups at any size left rows of less than 98,304 scores without a guess: eight of 32,000 at top-p 0.9, peaked, 116 us, with it 63.)
static int guess_of(int V) {
  const double groups = (double)(V / PIECE) * GROUPS;
  return V <= LIST || groups < 1 ? 0x7fffffff : (int)lround(groups * (1.0 - exp(-GUESS / groups)));
}

// Room a row needs: in `parts` always, in `scratch` if any row draws.
extern "C" long long qvl_sample_parts_bytes(int V) { return (long long)pieces_of(V) * (long long)(sizeof(ArgmaxPart) + GROUPS * sizeof(float)); }
extern "C" long long qvl_sample_scratch_bytes() { return (long long)sizeof(RowScratch); }
extern "C" int qvl_sample_params_size() { return (int)sizeof(RowParams); }

// logits: float32 [M, V].  scores: as large, written for rows that draw with penalties (null if there are none).
// scratch: M * qvl_sample_scratch_bytes() bytes on a 16-byte boundary, null if no row draws.  parts: M * qvl_sample_parts_bytes(V).
// out: the rows' tokens, and behind them, if rows draw, how many rows go the long way.
// top_k, top_p: whether any row has that cut (the passes for it are left out otherwise); cuts: whether any row that draws has a
// cut (the lists are left out otherwise).
// ways: 1 the short way, after which out[M] rows have no token yet; 2 the long way for these, with all buffers as the short
// one left them; 3 both.
extern "C" int qvl_sample_rows(const void* logits, void* scores, const void* params, const void* prev_ids, void* scratch,
                               void* parts, void* out, int M, int V, int top_k, int top_p, int cuts, int ways,
                               hipStream_t stream) {
  if (M <= 0) return QVL_OK;
  if (V <= 0 || !logits || !params || !prev_ids || !parts || !out) return QVL_ERR_SHAPE;
  if (((uintptr_t)scratch % 16) != 0 || ways < 1 || ways > 3) return QVL_ERR_SHAPE;
  const int pieces = pieces_of(V);
  if (M > 65535 || (long long)M * (pieces + 1) > 0x7fffffffll) return QVL_ERR_LIMIT;
  const float* lg = (const float*)logits;
  float* sc = (float*)scores;
  const RowParams* rp = (const RowParams*)params;
  RowScratch* rs = (RowScratch*)scratch;
  ArgmaxPart* ap = (ArgmaxPart*)parts;
  float* groups = (float*)(ap + (size_t)M * pieces);
  int* ids = (int*)out;
  int* todo = ids + M;
  float one = 1099511627776.0f;                                   // 2^40
  for (long long v = 1ll << 23; v < V; v <<= 1) one *= 0.5f;      // the sum of a row's masses fits 63 bits
  const dim3 block(THREADS);
  if (ways & 1) {
    hipLaunchKernelGGL(sample_scan_kernel, dim3(M * pieces + (scratch ? M : 0)), block, 0, stream, lg, sc, rp, (const int*)prev_ids, rs, ap,
                       groups, todo, M, V, pieces);
    if (scratch) {
      if (cuts || V <= LIST)
        hipLaunchKernelGGL(sample_list_kernel, dim3(pieces, M), block, 0, stream, lg, sc, rp, rs, ap, groups, V, pieces, guess_of(V), one);
      hipLaunchKernelGGL(sample_short_kernel, dim3(M), block, 0, stream, rp, rs, ap, ids, todo, V, pieces, one);
    } else {
      hipLaunchKernelGGL(sample_pick_kernel, dim3(M), block, 0, stream, lg, sc, rp, rs, ap, ids, todo, V, pieces);
    }
  }
  if ((ways & 2) && scratch) {
    if (top_k)
      for (int level = 0; level < 3; ++level)
        hipLaunchKernelGGL(sample_bins_kernel<false>, dim3(pieces, M), block, 0, stream, lg, sc, rp, rs, ap, todo, V, pieces, level, one);
    if (top_p)
      for (int level = 0; level < 3; ++level)
        hipLaunchKernelGGL(sample_bins_kernel<true>, dim3(pieces, M), block, 0, stream, lg, sc, rp, rs, ap, todo, V, pieces, level, one);
    hipLaunchKernelGGL(sample_chunks_kernel, dim3(CHUNKS / CHUNKS_A_BLOCK, M), block, 0, stream, lg, sc, rp, rs, ap, todo, V, pieces);
    hipLaunchKernelGGL(sample_pick_kernel, dim3(M), block, 0, stream, lg, sc, rp, rs, ap, ids, todo, V, pieces);
  }
  return qvl_launch_status();
}
