// Paged attention for any head size, float32 or bfloat16 storage, float32 arithmetic.
// One wave (four where sizes are multiples of four) per (token, query head).  It serves prompt portions and decoded tokens alike: a
// token at sequence index p sees keys lo..p of its request, lo = max(0, p - window + 1) with
// a window, else 0 (reference attention.py:336-402 for the mask, text.py:78 for the scale); with
// a window it also sees the request's first `keep_first` keys, wherever the window stands.  With `chunk` it
// sees the keys from its chunk's first position on (chunks of that many positions from the sequence's start).
// With `turn` [N, vd/2, 2] (cosines and sines of each token's angles) the values in the cache are turned by their
// own positions, and a head's output is turned back by its token's: pair m is channels m and m + vd/2, or
// (`turn_pairs`) 2m and 2m + 1.
// Values may have another width (vd) than keys (hd).  With `sinks` (one float32 per query head) the
// softmax's denominator also holds exp(sink): a place that has no key and no value and is not scaled.
// Keys are walked in blocks of 64 by absolute index, so a token's result does not depend on
// how its request was cut into steps or on what else is in the batch.
#include "common.h"

#define ATTN_MAX_HD 512

template <typename T>
__global__ void attn_generic_kernel(const T* __restrict__ q, const T* __restrict__ kc, const T* __restrict__ vc,
                                    const int* __restrict__ block_table, int table_width,
                                    const int* __restrict__ token_req, const int* __restrict__ token_seqpos,
                                    T* __restrict__ out, int nh, int nkv, int hd, int vd, int ps, int window,
                                    int keep_first, int chunk, float scale, const float* __restrict__ sinks,
                                    const float2* __restrict__ turn, int turn_pairs) {
  __shared__ float sq[ATTN_MAX_HD];
  const int n = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int r = token_req[n], p = token_seqpos[n];
  const int kvh = h / (nh / nkv);
  int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
  if (chunk > 0) lo = max(lo, p - p % chunk);
  const int kept = keep_first < lo ? keep_first : lo;       // keys [0, kept) are seen besides [lo, p]
  const int skip_from = (kept + 63) / 64, skip_to = lo / 64;  // blocks of 64 keys with nothing to see
  const T* qr = q + ((size_t)n * nh + h) * hd;
  for (int d = lane; d < hd; d += 64) sq[d] = ldf<T>(qr + d);
  __syncthreads();
  const int* bt = block_table + (size_t)r * table_width;

  float m = -INFINITY, l = 0.f;
  float acc[ATTN_MAX_HD / 64];
#pragma unroll
  for (int i = 0; i < ATTN_MAX_HD / 64; ++i) acc[i] = 0.f;

  for (int c = 0; c * 64 <= p; ++c) {
    if (c == skip_from && skip_to > skip_from) c = skip_to;
    const int j = c * 64 + lane;
    const bool valid = (j >= lo || j < kept) && j <= p;
    float s = -INFINITY;
    if (valid) {
      const int pk = bt[j / ps];
      const size_t page = (size_t)(pk < 0 ? 0 : pk);   // a table without this page: read page 0, never out of bounds
      const T* kr = kc + ((page * nkv + kvh) * ps + (size_t)(j % ps)) * hd;
      float dot = 0.f;
      for (int d = 0; d < hd; ++d) dot += sq[d] * ldf<T>(kr + d);
      s = dot * scale;
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float base = m_new > -INFINITY ? m_new : 0.f;   // (scores of -inf alone have no weight beside later ones)
    const float pj = valid ? expf(s - base) : 0.f;
    const float alpha = expf(m - base);   // m = -inf at first: alpha = 0
    l = l * alpha + wave_sum(pj);
#pragma unroll
    for (int i = 0; i < ATTN_MAX_HD / 64; ++i) acc[i] *= alpha;
    const int jend = (p - c * 64 < 63) ? p - c * 64 : 63;
    for (int jj = 0; jj <= jend; ++jj) {
      const float pv = __shfl(pj, jj, QVL_WAVE);
      const int ja = c * 64 + jj;
      if (ja < lo && ja >= kept) continue;
      const int pv_page = bt[ja / ps];
      const size_t page = (size_t)(pv_page < 0 ? 0 : pv_page);
      const T* vr = vc + ((page * nkv + kvh) * vd) * ps + (size_t)(ja % ps);
#pragma unroll
      for (int i = 0; i < ATTN_MAX_HD / 64; ++i) {
        const int d = lane + 64 * i;
        if (d < vd) acc[i] += pv * ldf<T>(vr + (size_t)d * ps);
      }
    }
    m = m_new;
  }
  if (sinks) {
    const float sk = sinks[h];
    const float m_all = fmaxf(m, sk);
    const float alpha = expf(m - m_all);
    l = l * alpha + expf(sk - m_all);
#pragma unroll
    for (int i = 0; i < ATTN_MAX_HD / 64; ++i) acc[i] *= alpha;
  }
  T* o = out + ((size_t)n * nh + h) * vd;
  const float inv = 1.0f / l;
  if (turn) {
    __syncthreads();          // the query has been read for the last time: its place takes the output
#pragma unroll
    for (int i = 0; i < ATTN_MAX_HD / 64; ++i) {
      const int d = lane + 64 * i;
      if (d < vd) sq[d] = acc[i] * inv;
    }
    __syncthreads();
    const int half = vd >> 1;
    const float2* tn = turn + (size_t)n * half;
    for (int d = lane; d < vd; d += 64) {
      const bool first = turn_pairs ? !(d & 1) : d < half;
      const float2 t = tn[turn_pairs ? d >> 1 : (first ? d : d - half)];
      const float v = sq[d], w = sq[turn_pairs ? d ^ 1 : (first ? d + half : d - half)];
      stf<T>(o + d, first ? v * t.x + w * t.y : v * t.x - w * t.y);
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < ATTN_MAX_HD / 64; ++i) {
    const int d = lane + 64 * i;
    if (d < vd) stf<T>(o + d, acc[i] * inv);
  }
}

// Four values from memory, as float32.
__device__ __forceinline__ float4 load4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 load4(const bf16_t* p) {
  const uint2 v = *reinterpret_cast<const uint2*>(p);
  return float4{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u)};
}

// The same where head size and page size are multiples of four, in one, two or four waves.  What bounds a token's few keys is the time until a load comes
// back, so loads are wide and many are in flight: four waves take the blocks of 64 keys in turn, each with a
// softmax of its own (joined at the end, in the waves' order); eight lanes read a key's row side by side, and a lane
// reads a channel's values of four keys at once.  CH: channels of a value, in sixteens, at most.
// float32, 16 heads of 128 over 2 of keys: 7 tokens at 25 to 100 keys 51 us with the wave above, 11 with these; 164 tokens of two prompts 57 and 33.
// Values of more than 128 channels are read 128 at a time: with all of a value's reads in one array the compiler kept it in scratch memory (28 heads of
// 512, bfloat16, 64 tokens at 1,000 keys 3,697 us, so 937, with the wave above 1,973; of 256, 64 tokens at 64 keys 224, 88 and 67).
template <typename T, int CH, int ATTN_WAVES>
__global__ __launch_bounds__(64 * ATTN_WAVES) void attn_generic_vec_kernel(
    const T* __restrict__ q, const T* __restrict__ kc, const T* __restrict__ vc, const int* __restrict__ block_table, int table_width,
    const int* __restrict__ token_req, const int* __restrict__ token_seqpos, T* __restrict__ out, int nh, int nkv, int hd, int vd, int ps,
    int window, int keep_first, int chunk, float scale, const float* __restrict__ sinks, const float2* __restrict__ turn, int turn_pairs) {
  __shared__ __attribute__((aligned(16))) float sq[ATTN_MAX_HD];
  __shared__ __attribute__((aligned(16))) float prob[ATTN_WAVES][64];
  __shared__ float part[ATTN_WAVES][CH * 16], part_m[ATTN_WAVES], part_l[ATTN_WAVES];
  const int n = blockIdx.x, h = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = token_req[n], p = token_seqpos[n];
  const int kvh = h / (nh / nkv);
  int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
  if (chunk > 0) lo = max(lo, p - p % chunk);
  const int kept = keep_first < lo ? keep_first : lo;       // keys [0, kept) are seen besides [lo, p]
  const int skip_from = (kept + 63) / 64, skipped = max(lo / 64 - skip_from, 0);  // blocks of 64 keys with nothing to see
  const T* qr = q + ((size_t)n * nh + h) * hd;
  for (int d = threadIdx.x; d < hd; d += 64 * ATTN_WAVES) sq[d] = ldf<T>(qr + d);
  __syncthreads();
  const int* bt = block_table + (size_t)r * table_width;

  float m = -INFINITY, l = 0.f;
  float acc[CH];       // channel 16 i + lane / 4, of the keys whose number / 4 has the rest lane mod 4
#pragma unroll
  for (int i = 0; i < CH; ++i) acc[i] = 0.f;
  const int sub = lane & 7, quad = lane & 3, chan = lane >> 2, blocks = p < 0 ? 0 : p / 64 + 1 - skipped;
  for (int b = wave; b < blocks; b += ATTN_WAVES) {
    const int first = 64 * (b < skip_from ? b : b + skipped);
    // scores: in pass i, eight lanes have key 8 (lane / 8) + i; it is lane number 8 (lane / 8) + i that keeps it
    float s = -INFINITY;
    const int mine = first + lane;
    const bool valid = (mine >= lo || mine < kept) && mine <= p;
    const T* row[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      int j = min(first + (lane & 56) + i, p);
      if constexpr (ATTN_WAVES < 4) j = j < lo && j >= kept ? p : j;       // (a key that is not seen: one that is; its score is left out)
      const int pk = bt[j / ps];
      const size_t page = (size_t)(pk < 0 ? 0 : pk);   // a table without this page: read page 0, never out of bounds
      row[i] = kc + ((page * nkv + kvh) * ps + (size_t)(j % ps)) * hd;
    }
    float dot[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int d = 4 * sub; d < hd; d += 32) {
      const float4 a = *reinterpret_cast<const float4*>(sq + d);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float4 k = load4(row[i] + d);
        dot[i] += a.x * k.x;
        dot[i] += a.y * k.y;
        dot[i] += a.z * k.z;
        dot[i] += a.w * k.w;
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int o = 1; o < 8; o <<= 1) dot[i] += __shfl_xor(dot[i], o, QVL_WAVE);
      if (sub == i && valid) s = dot[i] * scale;
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float base = m_new > -INFINITY ? m_new : 0.f;   // (scores of -inf alone have no weight beside later ones or other waves')
    const float pj = valid ? expf(s - base) : 0.f;
    const float alpha = expf(m - base);   // m = -inf at first: alpha = 0
    l = l * alpha + wave_sum(pj);
    m = m_new;
    prob[wave][lane] = pj;
#pragma unroll
    for (int i = 0; i < CH; ++i) acc[i] *= alpha;
    __builtin_amdgcn_wave_barrier();       // (a wave's own lines: its writes come before its reads)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int j0 = first + 16 * t + 4 * quad;
      if (first + 16 * t > p) break;
      if constexpr (ATTN_WAVES < 4)
        if (first + 16 * t + 15 < lo && first + 16 * t >= kept) continue;      // none of the sixteen is seen
      const int at = min(j0, p & ~3), pk = bt[at / ps];
      const size_t page = (size_t)(pk < 0 ? 0 : pk);
      const T* v = vc + ((page * nkv + kvh) * vd) * ps + (size_t)(at % ps);
      const float4 w = *reinterpret_cast<const float4*>(&prob[wave][16 * t + 4 * quad]);
      // values of keys that are not seen may be anything
      auto seen = [&](int j) { return (j >= lo || j < kept) && j <= p; };
      const bool s0 = seen(j0), s1 = seen(j0 + 1), s2 = seen(j0 + 2), s3 = seen(j0 + 3);
      // (eight at a time: more in flight cost the registers that other waves would have)
#pragma unroll
      for (int c = 0; c < CH; c += 8) {
        if (c && 16 * c >= vd) break;
        float4 x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int d = 16 * (c + i) + chan;
          if (16 * (c + i) < vd) x[i] = load4(v + (size_t)(d < vd ? d : 0) * ps);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if (16 * (c + i) >= vd) break;
          acc[c + i] += s0 ? w.x * x[i].x : 0.f;
          acc[c + i] += s1 ? w.y * x[i].y : 0.f;
          acc[c + i] += s2 ? w.z * x[i].z : 0.f;
          acc[c + i] += s3 ? w.w * x[i].w : 0.f;
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int i = 0; i < CH; ++i) {
#pragma unroll
    for (int o = 1; o < 4; o <<= 1) acc[i] += __shfl_xor(acc[i], o, QVL_WAVE);
    if (quad == 0) part[wave][16 * i + chan] = acc[i];
  }
  if (lane == 0) {
    part_m[wave] = m;
    part_l[wave] = l;
  }
  __syncthreads();
  const float sk = sinks ? sinks[h] : -INFINITY;
  float top = sk;
#pragma unroll
  for (int w = 0; w < ATTN_WAVES; ++w) top = fmaxf(top, part_m[w]);
  float factor[ATTN_WAVES], total = 0.f;
#pragma unroll
  for (int w = 0; w < ATTN_WAVES; ++w) {
    factor[w] = w < blocks ? expf(part_m[w] - top) : 0.f;
    total += part_l[w] * factor[w];
  }
  if (sinks) total += expf(sk - top);
  const float inv = 1.0f / total;
  auto value = [&](int d) {
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < ATTN_WAVES; ++w) v += part[w][d] * factor[w];
    return v * inv;
  };
  T* o = out + ((size_t)n * nh + h) * vd;
  const int half = vd >> 1;
  const float2* tn = turn + (size_t)n * half;
  for (int d = threadIdx.x; d < vd; d += 64 * ATTN_WAVES) {
    const float v = value(d);
    if (turn) {
      const bool one = turn_pairs ? !(d & 1) : d < half;
      const float2 t = tn[turn_pairs ? d >> 1 : (one ? d : d - half)];
      const float w = value(turn_pairs ? d ^ 1 : (one ? d + half : d - half));
      stf<T>(o + d, one ? v * t.x + w * t.y : v * t.x - w * t.y);
    } else {
      stf<T>(o + d, v);
    }
  }
}

extern "C" int qvl_attn_generic(const void* q, const void* kc, const void* vc, const void* block_table,
                                int table_width, const void* token_req, const void* token_seqpos, void* out, int N,
                                int nh, int nkv, int hd, int vd, int ps, int window, int keep_first, int chunk,
                                float scale, const void* sinks, const void* turn, int turn_pairs, int dtype,
                                hipStream_t stream) {
  if (N <= 0) return QVL_OK;
  if (nh <= 0 || nkv <= 0 || nh % nkv || hd <= 0 || vd <= 0 || ps <= 0 || table_width <= 0 || keep_first < 0 ||
      chunk < 0 || (turn && vd % 2))
    return QVL_ERR_SHAPE;
  if (hd > ATTN_MAX_HD || vd > ATTN_MAX_HD || nh > 65535) return QVL_ERR_LIMIT;
  const dim3 grid(N, nh);
  const bool vec = hd % 4 == 0 && ps % 4 == 0 && ((uintptr_t)kc % 16) == 0 && ((uintptr_t)vc % 16) == 0;
#define VEC(T, CH, WAVES)                                                                                                \
  hipLaunchKernelGGL((attn_generic_vec_kernel<T, CH, WAVES>), grid, dim3(64 * WAVES), 0, stream, (const T*)q, (const T*)kc, \
                     (const T*)vc, (const int*)block_table, table_width, (const int*)token_req, (const int*)token_seqpos, \
                     (T*)out, nh, nkv, hd, vd, ps, window, keep_first, chunk, scale, (const float*)sinks,                 \
                     (const float2*)turn, turn_pairs)
#define CHANNELS(T, WAVES)                       \
  do {                                           \
    if (vd <= 128) VEC(T, 8, WAVES);             \
    else if (vd <= 256) VEC(T, 16, WAVES);       \
    else VEC(T, ATTN_MAX_HD / 16, WAVES);        \
  } while (0)
  if (vec && (dtype == 0 || dtype == 1)) {
    // A token that sees few keys, in two blocks of 64 at most, has no work for four waves (16 heads of 64 over 2, bfloat16, 2,000 tokens, windows of 16
    // and 64 keys: the kernel above 100 and 278 us, four waves 305 and 327, one 91 and two 164)
    long long most = window > 0 ? window : 0x7fffffff;
    if (chunk > 0 && chunk < most) most = chunk;
    if (keep_first > 0) most += keep_first;
    if (dtype == 0 && most <= 32) CHANNELS(float, 1);
    else if (dtype == 0 && most <= 64) CHANNELS(float, 2);
    else if (dtype == 0) CHANNELS(float, 4);
    else if (most <= 32) CHANNELS(bf16_t, 1);
    else if (most <= 64) CHANNELS(bf16_t, 2);
    else CHANNELS(bf16_t, 4);
    return qvl_launch_status();
  }
#undef CHANNELS
#undef VEC
  if (dtype == 0)
    hipLaunchKernelGGL(attn_generic_kernel<float>, grid, dim3(64), 0, stream, (const float*)q, (const float*)kc,
                       (const float*)vc, (const int*)block_table, table_width, (const int*)token_req,
                       (const int*)token_seqpos, (float*)out, nh, nkv, hd, vd, ps, window, keep_first, chunk,
                       scale, (const float*)sinks, (const float2*)turn, turn_pairs);
  else if (dtype == 1)
    hipLaunchKernelGGL(attn_generic_kernel<bf16_t>, grid, dim3(64), 0, stream, (const bf16_t*)q, (const bf16_t*)kc,
                       (const bf16_t*)vc, (const int*)block_table, table_width, (const int*)token_req,
                       (const int*)token_seqpos, (bf16_t*)out, nh, nkv, hd, vd, ps, window, keep_first, chunk,
                       scale, (const float*)sinks, (const float2*)turn, turn_pairs);
  else
    return QVL_ERR_DTYPE;
  return qvl_launch_status();
}
