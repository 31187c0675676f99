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
// in turn); these passes together take 113 us.
#include "common.h"
#include <type_traits>

#define PIECE 4096          // scores a block owns in a pass over a row
#define THREADS 256
#define BINS 2048           // bins of a threshold's search: 11 bits of a score's key at a time
#define CHUNKS 1024         // contiguous ranges of a row whose masses the draw adds one after the other

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
  int pad[3];
  unsigned int count[3][BINS];
  unsigned long long mass[3][BINS];
  float chunk_mass[CHUNKS];
};

__device__ __forceinline__ uint32_t order_key(float f) {
  uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ bool penalised(const RowParams& p) {
  return p.prev_end > p.prev_begin && (p.repetition != 1.f || p.presence != 0.f || p.frequency != 0.f);
}
__device__ __forceinline__ bool cuts_k(const RowParams& p, int V) { return p.temperature > 0.f && p.top_k > 0 && p.top_k < V; }
__device__ __forceinline__ bool cuts_p(const RowParams& p) { return p.temperature > 0.f && p.top_p < 1.f; }

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
// written to `scores`), and empty bins for the searches.  With scratch there is one block more a row,
// which draws the row's uniform number.
__global__ __launch_bounds__(THREADS) void sample_scan_kernel(const float* __restrict__ logits, float* __restrict__ scores,
                                                              const RowParams* __restrict__ params,
                                                              const int* __restrict__ prev_ids,
                                                              RowScratch* __restrict__ scratch,
                                                              ArgmaxPart* __restrict__ parts, int V, int pieces) {
  __shared__ int seen[PIECE];     // how often each of the piece's tokens has been generated
  __shared__ float vals[THREADS / 64];
  __shared__ int idxs[THREADS / 64];
  const int m = blockIdx.y, s = blockIdx.x, tid = threadIdx.x;
  const RowParams p = params[m];
  const bool draws = p.temperature > 0.f;
  if (scratch && draws) {
    // empty bins: the blocks of the row share them out
    const int step = gridDim.x * THREADS;
    if (cuts_k(p, V))
      for (int i = s * THREADS + tid; i < 3 * BINS; i += step) (&scratch[m].count[0][0])[i] = 0u;
    if (cuts_p(p))
      for (int i = s * THREADS + tid; i < 3 * BINS; i += step) (&scratch[m].mass[0][0])[i] = 0ull;
  }
  if (s == pieces) {
    if (tid == 0) scratch[m].u = p.seeded ? first_uniform(p.seed) : p.u;
    return;
  }
  const float* lg = logits + (size_t)m * V;
  const int lo = s * PIECE, n = min(PIECE, V - lo);
  float v[PIECE / THREADS];
#pragma unroll
  for (int j = 0; j < PIECE / THREADS; ++j) {
    const int i = j * THREADS + tid;
    v[j] = lg[lo + (i < n ? i : 0)];
  }
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
      const int count = seen[j * THREADS + tid];
      if (count == 0) continue;
      float x = v[j];
      if (p.repetition != 1.f) x = x > 0.f ? x / p.repetition : x * p.repetition;
      v[j] = x - p.presence - p.frequency * (float)count;
    }
#pragma unroll
    for (int j = 0; j < PIECE / THREADS; ++j) {
      const int i = j * THREADS + tid;
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
    const int i = j * THREADS + tid;
    if (i < n && v[j] > bv) { bv = v[j]; bi = lo + i; }   // indices rise within a thread: the first of equals stays
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
                                                              const ArgmaxPart* __restrict__ parts, int V, int pieces,
                                                              int level, float one) {
  typedef typename std::conditional<MASS, unsigned long long, unsigned int>::type bin_t;
  __shared__ bin_t bins[BINS];
  __shared__ unsigned long long s_sum[THREADS], s_above;
  __shared__ int s_bin;
  __shared__ ArgmaxPart s_best;
  const int m = blockIdx.y, s = blockIdx.x, tid = threadIdx.x;
  const RowParams p = params[m];
  if (!(MASS ? cuts_p(p) : cuts_k(p, V))) return;
  RowScratch& r = scratch[m];
  const Scores score = scores_of(p, logits, scores, m, V);
  const int lo = s * PIECE, n = min(PIECE, V - lo);
  float v[PIECE / THREADS];
#pragma unroll
  for (int j = 0; j < PIECE / THREADS; ++j) {
    const int i = j * THREADS + tid;
    v[j] = score.at[lo + (i < n ? i : 0)];
  }
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
    if (j * THREADS + tid >= n) break;
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
                                                                const ArgmaxPart* __restrict__ parts, int V, int pieces) {
  __shared__ float tile[CHUNKS_A_BLOCK][65];
  __shared__ unsigned long long s_sum[THREADS], s_above;
  __shared__ int s_bin;
  __shared__ ArgmaxPart s_best;
  const int m = blockIdx.y, tid = threadIdx.x;
  const RowParams p = params[m];
  if (p.temperature <= 0.f) return;
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
  float mine = 0.f;
  for (int at = 0; at < C; at += 64) {
    __syncthreads();
    // 64 scores of every chunk, a wave one chunk's at a time
#pragma unroll
    for (int j = 0; j < CHUNKS_A_BLOCK * 64 / THREADS; ++j) {
      const int c = (j * THREADS + tid) >> 6, o = tid & 63;
      const long long i = (long long)(first + c) * C + at + o;
      float e = 0.f;
      if (at + o < C && i < V) {
        const float x = score((int)i);
        e = expf(x - mx);
        if (order_key(x) < cut || (p.min_p > 0.f && e < p.min_p)) e = 0.f;
      }
      tile[c][o] = e;
    }
    __syncthreads();
    if (tid < CHUNKS_A_BLOCK)
#pragma unroll 16
      for (int o = 0; o < 64; ++o) mine += tile[tid][o];
  }
  if (tid < CHUNKS_A_BLOCK) r.chunk_mass[first + tid] = mine;
}

// The token: the largest score's index, or the draw.
__global__ __launch_bounds__(THREADS) void sample_pick_kernel(const float* __restrict__ logits, const float* __restrict__ scores,
                                                              const RowParams* __restrict__ params,
                                                              RowScratch* __restrict__ scratch,
                                                              const ArgmaxPart* __restrict__ parts, int* __restrict__ out,
                                                              int V, int pieces) {
  __shared__ __attribute__((aligned(16))) float sums[CHUNKS];
  __shared__ float prefix[CHUNKS];
  __shared__ __attribute__((aligned(16))) float tile[THREADS];
  __shared__ ArgmaxPart s_best;
  __shared__ int s_chunk, s_last, s_token;
  __shared__ float s_z;
  const int m = blockIdx.x, tid = threadIdx.x;
  const RowParams p = params[m];
  const ArgmaxPart best = row_argmax(parts, m, pieces, V, &s_best);
  if (p.temperature <= 0.f) {
    if (tid == 0) out[m] = best.index < V ? best.index : 0;
    return;
  }
  RowScratch& r = scratch[m];
  const float mx = best.value;
  for (int i = tid; i < CHUNKS / 4; i += THREADS)
    reinterpret_cast<float4*>(sums)[i] = reinterpret_cast<const float4*>(r.chunk_mass)[i];
  if (tid == 0) { s_chunk = CHUNKS; s_last = 0; s_token = -1; }
  __syncthreads();
  if (tid == 0) {
    // the chunks' masses one after the other: prefix[t] is the mass before chunk t
    float acc = 0.f;
    for (int t = 0; t < CHUNKS; t += 8) {
      const float4 a = reinterpret_cast<const float4*>(sums)[t / 4], b = reinterpret_cast<const float4*>(sums)[t / 4 + 1];
      const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        prefix[t + i] = acc;
        acc += x[i];
      }
    }
    s_z = acc;
  }
  __syncthreads();
  const float target = r.u * s_z;
  for (int t = tid; t < CHUNKS; t += THREADS) {
    if (!(sums[t] > 0.f)) continue;
    if (prefix[t] + sums[t] > target) atomicMin(&s_chunk, t);
    atomicMax(&s_last, t);
  }
  __syncthreads();
  const bool found = s_chunk < CHUNKS;
  const int chunk = found ? s_chunk : s_last;
  const float pick = found ? target - prefix[chunk] : INFINITY;
  // within the chunk: the scores' masses from its first index on, until they exceed the rest
  uint32_t cut = cuts_k(p, V) ? r.found[0].key[2] : 0u;
  if (cuts_p(p)) cut = max(cut, r.found[1].key[2]);
  const Scores score = scores_of(p, logits, scores, m, V);
  const int C = (V + CHUNKS - 1) / CHUNKS, lo = chunk * C, hi = min(V, lo + C);
  float acc = 0.f;
  int last = lo;
  for (int at = lo; at < hi; at += THREADS) {
    float e = 0.f;
    if (at + tid < hi) {
      const float x = score(at + tid);
      e = expf(x - mx);
      if (order_key(x) < cut || (p.min_p > 0.f && e < p.min_p)) e = 0.f;
    }
    tile[tid] = e;
    __syncthreads();
    if (tid == 0) {
      int token = -1;      // places beyond the chunk hold zeros
      for (int i = 0; i < THREADS && at + i < hi && token < 0; i += 8) {
        const float4 a = reinterpret_cast<const float4*>(tile)[i / 4], b = reinterpret_cast<const float4*>(tile)[i / 4 + 1];
        const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (x[j] > 0.f && token < 0) {
            last = at + i + j;
            acc += x[j];
            if (acc > pick) token = last;
          }
        }
      }
      s_token = token;
    }
    __syncthreads();
    if (s_token >= 0) break;
  }
  if (tid == 0) out[m] = s_token >= 0 ? s_token : last;
}

static int pieces_of(int V) { return (V + PIECE - 1) / PIECE; }

// Room a row needs: in `parts` always, in `scratch` if any row draws.
extern "C" long long qvl_sample_parts_bytes(int V) { return (long long)pieces_of(V) * (long long)sizeof(ArgmaxPart); }
extern "C" long long qvl_sample_scratch_bytes() { return (long long)sizeof(RowScratch); }
extern "C" int qvl_sample_params_size() { return (int)sizeof(RowParams); }

// logits: float32 [M, V].  scores: as large, written for rows that draw with penalties (null if there are none).
// scratch: M * qvl_sample_scratch_bytes() bytes on a 16-byte boundary, null if no row draws.  parts: M * qvl_sample_parts_bytes(V).
// top_k, top_p: whether any row has that cut (the passes for it are left out otherwise).
extern "C" int qvl_sample_rows(const void* logits, void* scores, const void* params, const void* prev_ids, void* scratch,
                               void* parts, void* out, int M, int V, int top_k, int top_p, hipStream_t stream) {
  if (M <= 0) return QVL_OK;
  if (V <= 0 || !logits || !params || !prev_ids || !parts || !out) return QVL_ERR_SHAPE;
  if (((uintptr_t)scratch % 16) != 0) return QVL_ERR_SHAPE;
  if (M > 65535) return QVL_ERR_LIMIT;
  const float* lg = (const float*)logits;
  float* sc = (float*)scores;
  const RowParams* rp = (const RowParams*)params;
  RowScratch* rs = (RowScratch*)scratch;
  ArgmaxPart* ap = (ArgmaxPart*)parts;
  const int pieces = pieces_of(V);
  float one = 1099511627776.0f;                                   // 2^40
  for (long long v = 1ll << 23; v < V; v <<= 1) one *= 0.5f;      // the sum of a row's masses fits 63 bits
  hipLaunchKernelGGL(sample_scan_kernel, dim3(pieces + (scratch ? 1 : 0), M), dim3(THREADS), 0, stream, lg, sc, rp,
                     (const int*)prev_ids, rs, ap, V, pieces);
  if (scratch) {
    if (top_k)
      for (int level = 0; level < 3; ++level)
        hipLaunchKernelGGL(sample_bins_kernel<false>, dim3(pieces, M), dim3(THREADS), 0, stream, lg, sc, rp, rs, ap, V, pieces, level, one);
    if (top_p)
      for (int level = 0; level < 3; ++level)
        hipLaunchKernelGGL(sample_bins_kernel<true>, dim3(pieces, M), dim3(THREADS), 0, stream, lg, sc, rp, rs, ap, V, pieces, level, one);
    hipLaunchKernelGGL(sample_chunks_kernel, dim3(CHUNKS / CHUNKS_A_BLOCK, M), dim3(THREADS), 0, stream, lg, sc, rp, rs, ap, V, pieces);
  }
  hipLaunchKernelGGL(sample_pick_kernel, dim3(M), dim3(THREADS), 0, stream, lg, sc, rp, rs, ap, (int*)out, V, pieces);
  return qvl_launch_status();
}
