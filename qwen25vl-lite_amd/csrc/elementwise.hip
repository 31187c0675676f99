// Row-wise kernels of the decoder step: embedding gather, residual add + RMSNorm,
// rotation + cache write, SwiGLU.  Each works for float32 and bfloat16 storage and any
// row width; all arithmetic is float32.
#include "common.h"
#include <cstring>

// ---------------------------------------------------------------------------------------
// Embedding gather: out[n, :] = scale * float32(table[ids[n], :])       (reference text.py:213)
// ---------------------------------------------------------------------------------------
// With it the step's tables of cosines and sines (see rope_table_kernel): both need the step's integers alone, and a decode step's launch
// costs more than either (one row each of 3,584: rows 7.4 us with values one by one and their launch 4.7).
#define EMBED_TABLES 4
struct RotationTable {
  const float* inv_freq;
  const int* freq_row;
  float2* out;
  int rot_half;
  float amplitude;
};
struct EmbedArgs {
  const int* ids;
  const void* table;
  float* out;
  int H, V;
  float scale;
  const int* pos;
  int pos_stride;
  RotationTable tables[EMBED_TABLES];
};

__device__ __forceinline__ void rotation_row(const RotationTable& t, const int* __restrict__ pos, int pos_stride, int n) {
  for (int f = threadIdx.x; f < t.rot_half; f += blockDim.x) {
    const int row = t.freq_row[f];
    float c = 1.f, s = 0.f;
    if (row >= 0) {
      sincosf((float)pos[(size_t)row * pos_stride + n] * t.inv_freq[f], &s, &c);
      c *= t.amplitude;
      s *= t.amplitude;
    }
    t.out[(size_t)n * t.rot_half + f] = float2{c, s};
  }
}

template <typename T> struct norm_raw;      // four values as they lie
template <> struct norm_raw<float> { typedef float4 type; };
template <> struct norm_raw<bf16_t> { typedef uint2 type; };

// grid (N, 1 + tables).  E: values of a row that a thread takes at a time.  Eight of bfloat16 wait for memory half as often, four let a wave's
// stores fill whole lines: of 3,584 values 64 rows 2.43 us and 2.52, 512 rows 3.84 and 3.49, 2,048 rows 9.2 and 7.6 (9.0 one by one).
template <typename T, int E>
__global__ __launch_bounds__(256) void embed_kernel(EmbedArgs p) {
  const int n = blockIdx.x;
  if (blockIdx.y > 0) {
    rotation_row(p.tables[blockIdx.y - 1], p.pos, p.pos_stride, n);
    return;
  }
  int id = p.ids[n];
  id = id < 0 ? 0 : (id >= p.V ? p.V - 1 : id);  // ids are validated on the host; never read outside the table
  const T* row = reinterpret_cast<const T*>(p.table) + (size_t)id * p.H;
  float* o = p.out + (size_t)n * p.H;
  if constexpr (E > 1) {
#pragma unroll 4
    for (int i = threadIdx.x * E; i < p.H; i += 256 * E) {
      struct __attribute__((aligned(E * sizeof(T)))) Values { T v[E]; };
      const Values e = *reinterpret_cast<const Values*>(row + i);
#pragma unroll
      for (int k = 0; k < E; k += 4)
        *reinterpret_cast<float4*>(o + i + k) = float4{ldf<T>(e.v + k) * p.scale, ldf<T>(e.v + k + 1) * p.scale, ldf<T>(e.v + k + 2) * p.scale,
                                                       ldf<T>(e.v + k + 3) * p.scale};
    }
  } else {
    for (int i = threadIdx.x; i < p.H; i += 256) o[i] = ldf<T>(row + i) * p.scale;
  }
}
#define EMBED_MANY 256      // rows from which four values at a time are faster

// rotations: `tables` RotationTable records (host memory, of any alignment), at most EMBED_TABLES; pos as in qvl_rope_table.
extern "C" int qvl_embed_gather(const void* ids, const void* table, void* out, int N, int H, int V, int dtype, float scale,
                                const void* pos, int pos_stride, int tables, const void* rotations, hipStream_t stream) {
  if (N <= 0) return QVL_OK;
  if (H <= 0 || V <= 0 || tables < 0 || tables > EMBED_TABLES || (tables && (!pos || pos_stride < N || !rotations))) return QVL_ERR_SHAPE;
  EmbedArgs p;
  p.ids = (const int*)ids; p.table = table; p.out = (float*)out; p.H = H; p.V = V; p.scale = scale; p.pos = (const int*)pos; p.pos_stride = pos_stride;
  static_assert(sizeof(RotationTable) == 32, "three pointers, a count and a factor, as the caller packs them");
  for (int t = 0; t < tables; ++t) {
    memcpy(&p.tables[t], (const char*)rotations + t * sizeof(RotationTable), sizeof(RotationTable));
    if (p.tables[t].rot_half < 0) return QVL_ERR_SHAPE;
  }
  const dim3 grid(N, 1 + tables);
  const bool aligned = (((uintptr_t)table | (uintptr_t)out) & 15) == 0;
#define GO(T, E) hipLaunchKernelGGL((embed_kernel<T, E>), grid, dim3(256), 0, stream, p)
  if (dtype == 0) {
    if (aligned && H % 4 == 0) GO(float, 4);
    else GO(float, 1);
  } else if (dtype == 1) {
    if (aligned && H % 8 == 0 && N < EMBED_MANY) GO(bf16_t, 8);
    else if (aligned && H % 4 == 0) GO(bf16_t, 4);
    else GO(bf16_t, 1);
  } else {
    return QVL_ERR_DTYPE;
  }
#undef GO
  return qvl_launch_status();
}

// ---------------------------------------------------------------------------------------
// A replayed step's integers (15 to 270 KB at batch 8 to 64) from pinned host memory, read where they lie.  The runtime's copy of more than 16 KB runs on
// a copy engine, and the step's graph waits for its signal: 20 to 23 us from the last kernel in front of the copy to the first behind it, with this
// kernel 10.  A pass of 16 steps at batch 8 of 7B sizes 15,530 us to 15,330, of 8 steps at batch 64 10,360 to 10,240; smaller transfers, which the runtime
// makes with a kernel of its own, take as long as they did.  The loads go to the host's memory whatever the caches hold of it.
// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void from_host_kernel(const unsigned long long* __restrict__ from, unsigned long long* __restrict__ to, int n) {
  const int i = blockIdx.x * 512 + threadIdx.x, j = i + 256;
  unsigned long long a = 0, b = 0;
  if (i < n) a = __hip_atomic_load(from + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (j < n) b = __hip_atomic_load(from + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (i < n) to[i] = a;
  if (j < n) to[j] = b;
}

// from: pinned host memory, to: device memory, `pairs` pairs of 4-byte words, both on 8-byte boundaries.
extern "C" int qvl_from_host(const void* from, void* to, long long pairs, hipStream_t stream) {
  if (pairs <= 0) return QVL_OK;
  if (!from || !to || (((uintptr_t)from | (uintptr_t)to) & 7)) return QVL_ERR_SHAPE;
  if (pairs > 0x7ffffc00ll) return QVL_ERR_LIMIT;
  hipLaunchKernelGGL(from_host_kernel, dim3((unsigned)((pairs + 511) / 512)), dim3(256), 0, stream, (const unsigned long long*)from,
                     (unsigned long long*)to, (int)pairs);
  return qvl_launch_status();
}

// ---------------------------------------------------------------------------------------
// Residual add + RMSNorm  (reference layers.py:27-31, text.py:196-205)
//   v = h[row] + delta[row]            (delta optional; the sum is float32; delta may come as
//                                       several slabs [slab][row], partial sums of a product cut
//                                       along its inner size, which are added in slab order)
//   h[row] = v                         (unless `rows` selects rows: then h is left alone)
//   out[m] = v * (1/sqrt(mean(v^2) + eps)) * w
// One block per row; the reduction order depends on H only (and the two kernels for widths that 4 divides have the same),
// so a row's result does not depend on what else is in the batch.
// ---------------------------------------------------------------------------------------
template <typename TD, typename TO>
__global__ void add_rmsnorm_kernel(float* __restrict__ h, const TD* __restrict__ delta, const float* __restrict__ w,
                                   TO* __restrict__ out, const int* __restrict__ rows, int H, float eps, int nslabs,
                                   long long slab_stride) {
  __shared__ float red[17];
  const int m = blockIdx.x;
  const int row = rows ? rows[m] : m;
  float* hr = h + (size_t)row * H;
  const TD* dr = delta ? delta + (size_t)row * H : nullptr;
  auto delta_at = [&](int i) {
    float d = ldf<TD>(dr + i);
    for (int c = 1; c < nslabs; ++c) d += ldf<TD>(dr + (size_t)c * slab_stride + i);
    return d;
  };
  float ss = 0.f;
  for (int i = threadIdx.x; i < H; i += blockDim.x) {
    float v = hr[i];
    if (dr) v += delta_at(i);
    ss += v * v;
    if (dr && !rows) hr[i] = v;
  }
  const float total = block_sum(ss, red);
  const float rs = 1.0f / sqrtf(total / (float)H + eps);
  TO* o = out + (size_t)m * H;
  for (int i = threadIdx.x; i < H; i += blockDim.x) {
    float v = hr[i];
    if (dr && rows) v += delta_at(i);
    stf<TO>(o + i, (v * rs) * w[i]);
  }
}

// The same with every value held in registers between the two passes: rows whose width is a
// multiple of 4 and at most NORM_VEC_MAX * 4 * 256, read and written 4 values at a time.
#define NORM_VEC_MAX 8
#define NORM_ROWS 512      // many rows, for which the kernels below are made differently

__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
template <typename T> __device__ __forceinline__ void st4(T* p, float4 v);
template <> __device__ __forceinline__ void st4<float>(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
template <> __device__ __forceinline__ void st4<bf16_t>(bf16_t* p, float4 v) {
  uint2 o;
  o.x = (uint32_t)f32_to_bf16(v.x) | ((uint32_t)f32_to_bf16(v.y) << 16);
  o.y = (uint32_t)f32_to_bf16(v.z) | ((uint32_t)f32_to_bf16(v.w) << 16);
  *reinterpret_cast<uint2*>(p) = o;
}

// The sum of squares of these kernels and of the one for slabs below has one order, that of 16 waves of 64 lanes with one or two
// pieces each, whatever the number of threads: here a wave stands for up to four.
__device__ __forceinline__ float add_squares(float ss, float4 x) { 
  return ss + fmaf(x.w, x.w, fmaf(x.z, x.z, fmaf(x.y, x.y, x.x * x.x)));
}
template <int N>
__device__ __forceinline__ float norm_total(const float* sums) {
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) t += sums[i];
  return t;
}

// VEC: 4-value pieces of a thread.  Everything it needs is asked for before anything is waited for, converted or stored (a store to h
// would hold up the loads of h behind it, a branch around a load the next load): pieces past the row's end read its last one.  Of an
// addend in slabs (float32), one slab at a time, in order.
// Bytes bound it from about a thousand rows on: 4,096 rows of 3,584 with a bfloat16 addend 28.5 -> 26.9 us, 6.6 TB/s; below, latency: 64
// rows of 8,192 7.4 -> 5.4, when the loads waited for each other's stores and the weights for the sum.
// LATE, for NORM_ROWS rows or more of more than 4,096 values: four pieces at a time and the weights behind the sum.  Asked for at once, eight
// pieces take 145 registers, three waves a SIMD, and the memory idles (with a bfloat16 addend 1,024 x 5,120 13.8 us, 10.4 so; 1,024 x 8,192 19.9
// and 17.7; without one 4,096 x 8,192 40.0 and 33.7).
__device__ __forceinline__ float4 norm_value(float4 v) { return v; }
__device__ __forceinline__ float4 norm_value(uint2 v) {
  return float4{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                __uint_as_float(v.y & 0xffff0000u)};
}

template <typename TD, typename TO, int VEC, bool LATE>
__global__ __launch_bounds__(256) void add_rmsnorm_vec_kernel(float* __restrict__ h, const TD* __restrict__ delta,
                                                              const float* __restrict__ w, TO* __restrict__ out,
                                                              const int* __restrict__ rows, int H, float eps, int nslabs,
                                                              long long slab_stride) {
  constexpr int PART = VEC < 4 ? VEC : 4;
  typedef typename norm_raw<TD>::type Raw;
  __shared__ __attribute__((aligned(16))) float sums[4 * PART];
  const int m = blockIdx.x;
  const int row = rows ? rows[m] : m;
  float* hr = h + (size_t)row * H;
  const int nvec = H >> 2;
  constexpr int STEP = LATE ? 4 : VEC;      // pieces asked for at once
  int at[VEC];
  float4 v[VEC], g[VEC];
#pragma unroll
  for (int j = 0; j < VEC; ++j) at[j] = 4 * min((int)threadIdx.x + 256 * j, nvec - 1);
#pragma unroll
  for (int j0 = 0; j0 < VEC; j0 += STEP) {
    const int j1 = j0 + STEP < VEC ? j0 + STEP : VEC;
#pragma unroll
    for (int j = j0; j < j1; ++j) v[j] = ld4(hr + at[j]);
    if (!delta) continue;
    const TD* dr = delta + (size_t)row * H;
    Raw d[VEC];
#pragma unroll
    for (int j = j0; j < j1; ++j) d[j] = *reinterpret_cast<const Raw*>(dr + at[j]);
    float4 sum[VEC];
    if (!LATE) {
#pragma unroll
      for (int j = j0; j < j1; ++j) g[j] = ld4(w + at[j]);
    }
#pragma unroll
    for (int j = j0; j < j1; ++j) sum[j] = norm_value(d[j]);
    for (int c = 1; c < nslabs; ++c) {
#pragma unroll
      for (int j = j0; j < j1; ++j) d[j] = *reinterpret_cast<const Raw*>(dr + (size_t)c * slab_stride + at[j]);
#pragma unroll
      for (int j = j0; j < j1; ++j) {
        const float4 e = norm_value(d[j]);
        sum[j].x += e.x; sum[j].y += e.y; sum[j].z += e.z; sum[j].w += e.w;
      }
    }
#pragma unroll
    for (int j = j0; j < j1; ++j) {
      v[j].x += sum[j].x; v[j].y += sum[j].y; v[j].z += sum[j].z; v[j].w += sum[j].w;
      if (!rows && (int)threadIdx.x + 256 * j < nvec) st4<float>(hr + at[j], v[j]);
    }
  }
  if (!delta && !LATE) {
#pragma unroll
    for (int j = 0; j < VEC; ++j) g[j] = ld4(w + at[j]);
  }
  float ss[PART] = {};
#pragma unroll
  for (int j = 0; j < VEC; ++j)
    if ((int)threadIdx.x + 256 * j < nvec) ss[j % PART] = add_squares(ss[j % PART], v[j]);
#pragma unroll
  for (int j = 0; j < PART; ++j) {
    ss[j] = wave_sum(ss[j]);
    if ((threadIdx.x & 63) == 0) sums[4 * j + (threadIdx.x >> 6)] = ss[j];
  }
  __syncthreads();
  const float rs = 1.0f / sqrtf(norm_total<4 * PART>(sums) / (float)H + eps);
  TO* o = out + (size_t)m * H;
#pragma unroll
  for (int j0 = 0; j0 < VEC; j0 += STEP) {
    const int j1 = j0 + STEP < VEC ? j0 + STEP : VEC;
    if (LATE) {
#pragma unroll
      for (int j = j0; j < j1; ++j) g[j] = ld4(w + at[j]);
    }
#pragma unroll
    for (int j = j0; j < j1; ++j) {
      if ((int)threadIdx.x + 256 * j < nvec)
        st4<TO>(o + at[j], float4{(v[j].x * rs) * g[j].x, (v[j].y * rs) * g[j].y, (v[j].z * rs) * g[j].z, (v[j].w * rs) * g[j].w});
    }
  }
}

// The addend as slabs of partial sums (float32 [slab][row][H]) for fewer than NORM_ROWS rows: a block of 1024 threads per row, a thread
// per 4 values (rows of up to 4,096) or 8.  The loads of ONCE slabs are asked for at a time, sixteen of one piece, four of two (they do not
// depend on each other, only the sum has an order: slab 0, 1, 2, ...), with the first of them the rows of h and w.  Latency bounds it:
// fewer rows than fill the chip wait for memory once for every ONCE slabs here and once a slab in the kernel above (3,584 values, eight slabs:
// 64 rows 4.1 us and 5.0, 256 rows 5.6 and 7.0).  Threads past a row of up to 4,096 leave as waves: a condition at every load took most of a microsecond (1,024
// values, 64 rows 4.2 us, 3.4 so).  Sixteen loads of two pieces, eight slabs, do not fit the registers (rows of 8,192, four slabs, 64 of them
// 5.8 us and 5.0; of 5,120, eight slabs, 6.5 and 5.4).
// Many rows are bound by bytes: blocks of 1024 threads that are all at the same point leave the memory idle (of two slabs 512 rows 7.4
// and 6.0, 2,048 rows 26.5 and 20.8).
template <typename TO, int VEC>
__global__ __launch_bounds__(1024) void add_rmsnorm_slabs_kernel(float* __restrict__ h, const float* __restrict__ delta,
                                                                 const float* __restrict__ w, TO* __restrict__ out,
                                                                 const int* __restrict__ rows, int H, float eps,
                                                                 int nslabs, long long slab_stride) {
  constexpr int ONCE = VEC == 1 ? 16 : 4;
  __shared__ __attribute__((aligned(16))) float sums[16];
  const int m = blockIdx.x;
  const int row = rows ? rows[m] : m;
  float* hr = h + (size_t)row * H;
  const float* dr = delta + (size_t)row * H;
  int at[VEC];
  float4 v[VEC], g[VEC];
  float ss = 0.f;
  if (VEC > 1 || 4 * (int)threadIdx.x < H) {      // (pieces past the end of a row of more than 4,096 read its last one)
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      at[j] = min(4 * ((int)threadIdx.x + 1024 * j), H - 4);
      v[j] = ld4(hr + at[j]);
      g[j] = ld4(w + at[j]);
    }
    float4 d[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) d[j] = float4{0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < nslabs; c0 += ONCE) {
      float4 e[ONCE][VEC];
#pragma unroll
      for (int c = 0; c < ONCE; ++c)
#pragma unroll
        for (int j = 0; j < VEC; ++j)
          e[c][j] = c0 + c < nslabs ? ld4(dr + (size_t)(c0 + c) * slab_stride + at[j]) : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < ONCE; ++c)
#pragma unroll
        for (int j = 0; j < VEC; ++j)
          if (c0 + c < nslabs) { d[j].x += e[c][j].x; d[j].y += e[c][j].y; d[j].z += e[c][j].z; d[j].w += e[c][j].w; }
    }
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      v[j].x += d[j].x; v[j].y += d[j].y; v[j].z += d[j].z; v[j].w += d[j].w;
      if (4 * ((int)threadIdx.x + 1024 * j) < H) {
        if (!rows) st4<float>(hr + at[j], v[j]);
        ss = add_squares(ss, v[j]);
      }
    }
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float rs = 1.0f / sqrtf(norm_total<16>(sums) / (float)H + eps);
  TO* o = out + (size_t)m * H;
#pragma unroll
  for (int j = 0; j < VEC; ++j) {
    if (4 * ((int)threadIdx.x + 1024 * j) < H)
      st4<TO>(o + at[j], float4{(v[j].x * rs) * g[j].x, (v[j].y * rs) * g[j].y, (v[j].z * rs) * g[j].z, (v[j].w * rs) * g[j].w});
  }
}

// delta: null, or nslabs slabs of [rows of h][H], slab_stride elements apart (nslabs 1: one addend).
extern "C" int qvl_add_rmsnorm(void* h, const void* delta, const void* w, void* out, const void* rows, int M, int H,
                               float eps, int delta_dtype, int out_dtype, int nslabs, long long slab_stride,
                               hipStream_t stream) {
  if (M <= 0) return QVL_OK;
  if (H <= 0 || nslabs < 1 || (nslabs > 1 && slab_stride < H)) return QVL_ERR_SHAPE;
  const int threads = H >= 2048 ? 512 : 256;
  const bool wide = H % 4 == 0 && H <= NORM_VEC_MAX * 4 * 256, slabs = nslabs > 1 && delta;
  const bool vec = wide && (!slabs || (delta_dtype == 0 && slab_stride % 4 == 0));
  if (vec && slabs && M < NORM_ROWS) {
#define QVL_NORM_SLABS(TO, VEC)                                                                                    \
  hipLaunchKernelGGL((add_rmsnorm_slabs_kernel<TO, VEC>), dim3(M), dim3(1024), 0, stream, (float*)h,               \
                     (const float*)delta, (const float*)w, (TO*)out, (const int*)rows, H, eps, nslabs, slab_stride)
    if (out_dtype == 0 && H <= 4096) QVL_NORM_SLABS(float, 1);
    else if (out_dtype == 0) QVL_NORM_SLABS(float, 2);
    else if (out_dtype == 1 && H <= 4096) QVL_NORM_SLABS(bf16_t, 1);
    else if (out_dtype == 1) QVL_NORM_SLABS(bf16_t, 2);
    else return QVL_ERR_DTYPE;
#undef QVL_NORM_SLABS
    return qvl_launch_status();
  }
#define QVL_NORM_VEC(TD, TO, VEC, LATE)                                                                            \
  hipLaunchKernelGGL((add_rmsnorm_vec_kernel<TD, TO, VEC, LATE>), dim3(M), dim3(256), 0, stream, (float*)h,        \
                     (const TD*)delta, (const float*)w, (TO*)out, (const int*)rows, H, eps, nslabs, slab_stride)
#define QVL_NORM_CASE(DD, OD, TD, TO)                                                                              \
  if (delta_dtype == DD && out_dtype == OD) {                                                                      \
    if (vec && H <= 1024) QVL_NORM_VEC(TD, TO, 1, false);                                                          \
    else if (vec && H <= 2048) QVL_NORM_VEC(TD, TO, 2, false);                                                     \
    else if (vec && H <= 4096) QVL_NORM_VEC(TD, TO, 4, false);                                                     \
    else if (vec && M < NORM_ROWS) QVL_NORM_VEC(TD, TO, 8, false);                                                 \
    else if (vec && H <= 5120) QVL_NORM_VEC(TD, TO, 5, true);                                                      \
    else if (vec && H <= 6144) QVL_NORM_VEC(TD, TO, 6, true);                                                      \
    else if (vec && H <= 7168) QVL_NORM_VEC(TD, TO, 7, true);                                                      \
    else if (vec) QVL_NORM_VEC(TD, TO, 8, true);                                                                   \
    else                                                                                                           \
      hipLaunchKernelGGL((add_rmsnorm_kernel<TD, TO>), dim3(M), dim3(threads), 0, stream, (float*)h,               \
                         (const TD*)delta, (const float*)w, (TO*)out, (const int*)rows, H, eps, nslabs,            \
                         slab_stride);                                                                             \
    return qvl_launch_status();                                                                                    \
  }
  QVL_NORM_CASE(0, 0, float, float)
  QVL_NORM_CASE(0, 1, float, bf16_t)
  QVL_NORM_CASE(1, 1, bf16_t, bf16_t)
  QVL_NORM_CASE(1, 0, bf16_t, float)
#undef QVL_NORM_CASE
#undef QVL_NORM_VEC
  return QVL_ERR_DTYPE;
}

// ---------------------------------------------------------------------------------------
// Rotation + cache write  (reference rope.py:48-96, cache.py:440-460)
// x[n] holds nq query heads, then nkv key heads, then nkv value heads, each hd wide.
// For frequency f < rot_half the angle is float32(pos[freq_row[f]][n]) * inv_freq[f]; the pair
// is (f, f + rot_half):  out[f] = x[f] c - x[f+rot_half] s,  out[f+rot_half] = x[f+rot_half] c + x[f] s.
// Channels from 2*rot_half on pass unrotated.  Queries go to q_out; keys (rotated) and values
// go into the page slot of the token: K as [page][kv head][slot][hd], V as [page][kv head][hd][slot].
// ---------------------------------------------------------------------------------------
template <typename TI, typename T>
__global__ void rope_kv_write_kernel(const TI* __restrict__ x, int x_stride, const float* __restrict__ bias,
                                     const int* __restrict__ pos, int pos_stride,
                                     const float* __restrict__ inv_freq, const int* __restrict__ freq_row,
                                     const float2* __restrict__ cs, const int* __restrict__ slot,
                                     T* __restrict__ q_out, T* __restrict__ kc, T* __restrict__ vc, int nq, int nkv,
                                     int hd, int rot_half, int ps) {
  const int n = blockIdx.x;
  const int hh = blockIdx.y;
  const TI* src = x + (size_t)n * x_stride + (size_t)hh * hd;
  const float* b = bias ? bias + (size_t)hh * hd : nullptr;
  if (hh >= nq + nkv) {  // value head: copy
    const int s = slot[n];
    if (s < 0) return;
    const int kvh = hh - nq - nkv;
    const size_t page = (size_t)(s / ps), off = (size_t)(s % ps);
    T* dst = vc + ((page * nkv + kvh) * hd) * ps + off;
    for (int d = threadIdx.x; d < hd; d += blockDim.x) {
      float v = ldf<TI>(src + d) + (b ? b[d] : 0.f);
      stf<T>(dst + (size_t)d * ps, v);
    }
    return;
  }
  T* dst;
  if (hh < nq) {
    dst = q_out + ((size_t)n * nq + hh) * hd;
  } else {
    const int s = slot[n];
    if (s < 0) return;
    const int kvh = hh - nq;
    const size_t page = (size_t)(s / ps), off = (size_t)(s % ps);
    dst = kc + ((page * nkv + kvh) * ps + off) * hd;
  }
  for (int f = threadIdx.x; f < rot_half; f += blockDim.x) {
    float x1 = ldf<TI>(src + f) + (b ? b[f] : 0.f);
    float x2 = ldf<TI>(src + f + rot_half) + (b ? b[f + rot_half] : 0.f);
    float c = 1.f, s = 0.f;
    if (cs) {  // the step's table of cosines and sines: every head and layer reads the same values
      const float2 v = cs[(size_t)n * rot_half + f];
      c = v.x;
      s = v.y;
    } else {
      const int row = freq_row[f];
      if (row >= 0) {
        const float ang = (float)pos[(size_t)row * pos_stride + n] * inv_freq[f];
        sincosf(ang, &s, &c);
      }
    }
    stf<T>(dst + f, x1 * c - x2 * s);
    stf<T>(dst + f + rot_half, x2 * c + x1 * s);
  }
  for (int d = 2 * rot_half + threadIdx.x; d < hd; d += blockDim.x)
    stf<T>(dst + d, ldf<TI>(src + d) + (b ? b[d] : 0.f));
}

// The same for float32 sums, bfloat16 outputs and the table of cosines and sines in hand, with
// all widths multiples of 4: a thread per 4 neighbouring channels (and the 4 they are rotated with), 16-byte loads and 8-byte stores.
// x may come as nslabs slabs, slab_stride elements apart (partial sums of a product cut along its inner
// size): they are added in slab order, then the bias; AT_ONCE slabs are asked for before the first is added.
// The y blocks of a token share its channels: a block each with many tokens, which fill the device and hide the loads of
// one slab behind another's; with few, as many as make one item a thread and eight slabs at once, since one block would then
// work through slab after slab of every item alone while the device idles (64 tokens, 28 + 2 x 4 heads of 128, 7
// slabs: 14.0 us by one block a token and one slab at a time, 6.3; 2,048 tokens, 1 slab: 19.9 and 21.8).
template <int AT_ONCE>
__global__ __launch_bounds__(256) void rope_kv_write_wide_kernel(
    const float* __restrict__ x, int x_stride, const float* __restrict__ bias, const float2* __restrict__ cs,
    const int* __restrict__ slot, bf16_t* __restrict__ q_out, bf16_t* __restrict__ kc, bf16_t* __restrict__ vc, int nq,
    int nkv, int hd, int rot_half, int ps, int nslabs, long long slab_stride) {
  const int n = blockIdx.x;
  const float* src = x + (size_t)n * x_stride;
  auto sums = [&](int at) {
    float4 v = *reinterpret_cast<const float4*>(src + at);
    for (int c0 = 1; c0 < nslabs; c0 += AT_ONCE) {
      float4 e[AT_ONCE];
#pragma unroll
      for (int c = 0; c < AT_ONCE; ++c)
        if (c0 + c < nslabs) e[c] = *reinterpret_cast<const float4*>(src + (size_t)(c0 + c) * slab_stride + at);
#pragma unroll
      for (int c = 0; c < AT_ONCE; ++c)
        if (c0 + c < nslabs) { v.x += e[c].x; v.y += e[c].y; v.z += e[c].z; v.w += e[c].w; }
    }
    if (bias) {
      const float4 b = *reinterpret_cast<const float4*>(bias + at);
      v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w;
    }
    return v;
  };
  const int s = nkv ? slot[n] : -1;
  const size_t page = s >= 0 ? (size_t)(s / ps) : 0, off = s >= 0 ? (size_t)(s % ps) : 0;
  auto pack4 = [](float4 v) {
    uint2 o;
    o.x = (uint32_t)f32_to_bf16(v.x) | ((uint32_t)f32_to_bf16(v.y) << 16);
    o.y = (uint32_t)f32_to_bf16(v.z) | ((uint32_t)f32_to_bf16(v.w) << 16);
    return o;
  };
  // items: (rotated head, 4 frequencies); (rotated head, 4 channels past the rotation); (value head, 4 channels)
  const int per_head = rot_half / 4, rotated = (nq + nkv) * per_head, tail = (hd - 2 * rot_half) / 4;
  const int rest = rotated + (nq + nkv) * tail, items = rest + (s >= 0 ? nkv * (hd / 4) : 0);
  for (int it = blockIdx.y * 256 + threadIdx.x; it < items; it += gridDim.y * 256) {
    if (it >= rest) {  // values: [page][kv head][channel][slot]
      const int i = it - rest, kvh = i / (hd / 4), d = (i - kvh * (hd / 4)) * 4;
      const float4 v = sums((nq + nkv + kvh) * hd + d);
      bf16_t* dst = vc + ((page * nkv + kvh) * hd + d) * ps + off;
      dst[0] = f32_to_bf16(v.x);
      dst[(size_t)ps] = f32_to_bf16(v.y);
      dst[(size_t)2 * ps] = f32_to_bf16(v.z);
      dst[(size_t)3 * ps] = f32_to_bf16(v.w);
      continue;
    }
    const bool turns = it < rotated;
    const int i = turns ? it : it - rotated, each = turns ? per_head : tail, hh = i / each;
    const int f = (i - hh * each) * 4 + (turns ? 0 : 2 * rot_half);
    if (hh >= nq && s < 0) continue;
    bf16_t* dst = hh < nq ? q_out + ((size_t)n * nq + hh) * hd : kc + ((page * nkv + (hh - nq)) * ps + off) * hd;
    const float4 x1 = sums(hh * hd + f);
    if (!turns) {
      *reinterpret_cast<uint2*>(dst + f) = pack4(x1);
      continue;
    }
    const float4 x2 = sums(hh * hd + f + rot_half);
    const float4 c01 = *reinterpret_cast<const float4*>(cs + (size_t)n * rot_half + f);      // (c0, s0, c1, s1)
    const float4 c23 = *reinterpret_cast<const float4*>(cs + (size_t)n * rot_half + f + 2);
    const float4 lo = {x1.x * c01.x - x2.x * c01.y, x1.y * c01.z - x2.y * c01.w, x1.z * c23.x - x2.z * c23.y,
                       x1.w * c23.z - x2.w * c23.w};
    const float4 hi = {x2.x * c01.x + x1.x * c01.y, x2.y * c01.z + x1.y * c01.w, x2.z * c23.x + x1.z * c23.y,
                       x2.w * c23.z + x1.w * c23.w};
    *reinterpret_cast<uint2*>(dst + f) = pack4(lo);
    *reinterpret_cast<uint2*>(dst + f + rot_half) = pack4(hi);
  }
}

// cs: null, or float32 [N, rot_half, 2] from qvl_rope_table (then pos, inv_freq and freq_row are not read).
// nslabs > 1: x is float32 slabs of partial sums, slab_stride elements apart; taken with float32 in,
// bfloat16 out, cs given and all widths multiples of 4 only (else QVL_ERR_SHAPE).
extern "C" int qvl_rope_kv_write(const void* x, int x_stride, const void* bias, const void* pos, int pos_stride,
                                 const void* inv_freq, const void* freq_row, const void* cs, const void* slot,
                                 void* q_out, void* kc,
                                 void* vc, int N, int nq, int nkv, int hd, int rot_half, int ps, int in_dtype,
                                 int dtype, int nslabs, long long slab_stride, hipStream_t stream) {
  if (N <= 0) return QVL_OK;
  if (nslabs < 1 || (nslabs > 1 && (slab_stride < (long long)(nq + 2 * nkv) * hd || slab_stride % 4))) return QVL_ERR_SHAPE;
  if (nq < 0 || nkv < 0 || nq + nkv == 0 || hd <= 0 || rot_half < 0 || 2 * rot_half > hd || ps <= 0)
    return QVL_ERR_SHAPE;
  if (x_stride < (nq + 2 * nkv) * hd) return QVL_ERR_SHAPE;
  if (nq + 2 * nkv > 65535) return QVL_ERR_LIMIT;
  if (in_dtype == 0 && dtype == 1 && cs && hd % 4 == 0 && rot_half % 4 == 0 && x_stride % 4 == 0 &&
      (((uintptr_t)x | (uintptr_t)bias | (uintptr_t)cs) & 15) == 0 && (((uintptr_t)q_out | (uintptr_t)kc) & 7) == 0) {
    const int items = (nq + nkv) * (rot_half / 4 + (hd - 2 * rot_half) / 4) + nkv * (hd / 4);
#define QVL_ROPE_WIDE(AT_ONCE, share)                                                                                      \
  hipLaunchKernelGGL((rope_kv_write_wide_kernel<AT_ONCE>), dim3(N, share), dim3(256), 0, stream, (const float*)x, x_stride,   \
                     (const float*)bias, (const float2*)cs, (const int*)slot, (bf16_t*)q_out, (bf16_t*)kc, (bf16_t*)vc, nq,  \
                     nkv, hd, rot_half, ps, nslabs, slab_stride)
    if (N >= 512) QVL_ROPE_WIDE(1, 1);
    else QVL_ROPE_WIDE(8, min(64, (items + 255) / 256));
#undef QVL_ROPE_WIDE
    return qvl_launch_status();
  }
  if (nslabs > 1) return QVL_ERR_SHAPE;
  const dim3 grid(N, nq + 2 * nkv);
#define QVL_ROPE_CASE(ID, OD, TI, T)                                                                               \
  if (in_dtype == ID && dtype == OD) {                                                                             \
    hipLaunchKernelGGL((rope_kv_write_kernel<TI, T>), grid, dim3(64), 0, stream, (const TI*)x, x_stride,           \
                       (const float*)bias, (const int*)pos, pos_stride, (const float*)inv_freq,                    \
                       (const int*)freq_row, (const float2*)cs, (const int*)slot, (T*)q_out, (T*)kc, (T*)vc, nq,   \
                       nkv, hd, rot_half, ps);                                                                     \
    return qvl_launch_status();                                                                                    \
  }
  QVL_ROPE_CASE(0, 0, float, float)
  QVL_ROPE_CASE(0, 1, float, bf16_t)
  QVL_ROPE_CASE(1, 1, bf16_t, bf16_t)
#undef QVL_ROPE_CASE
  return QVL_ERR_DTYPE;
}

// ---------------------------------------------------------------------------------------
// The rotation's cosines and sines of a step, for kernels that rotate without computing angles:
// out[n, f] = amplitude * (cos, sin) of pos[freq_row[f], n] * inv_freq[f], or (1, 0) where freq_row[f] < 0.
// ---------------------------------------------------------------------------------------
__global__ void rope_table_kernel(const int* __restrict__ pos, int pos_stride, RotationTable table) {
  rotation_row(table, pos, pos_stride, blockIdx.x);
}

extern "C" int qvl_rope_table(const void* pos, int pos_stride, const void* inv_freq, const void* freq_row, void* out,
                              int N, int rot_half, float amplitude, hipStream_t stream) {
  if (N <= 0 || rot_half <= 0) return QVL_OK;
  if (pos_stride < N) return QVL_ERR_SHAPE;
  hipLaunchKernelGGL(rope_table_kernel, dim3(N), dim3(64), 0, stream, (const int*)pos, pos_stride,
                     RotationTable{(const float*)inv_freq, (const int*)freq_row, (float2*)out, rot_half, amplitude});
  return qvl_launch_status();
}

// ---------------------------------------------------------------------------------------
// SwiGLU: out[n, i] = silu(gate[n, i]) * up[n, i],  silu(z) = z / (1 + exp(-z))  (reference text.py:66);
// with `gelu` the activation is the tanh form of gelu.
// x[n] holds gate and up: plain, gate in columns 0..I-1 and up in I..2I-1; grouped, alternating
// groups of 8 gate columns and 8 up columns (feature i: gate at 16 (i/8) + i%8, up 8 further),
// the layout that lets the product before it apply the activation to a 16-row tile by itself.
// ---------------------------------------------------------------------------------------
template <typename T>
__global__ void swiglu_kernel(const T* __restrict__ x, T* __restrict__ out, int I, int grouped, int gelu) {
  const int n = blockIdx.y;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= I) return;
  const T* row = x + (size_t)n * 2 * I;
  const int gc = grouped ? 16 * (i >> 3) + (i & 7) : i;
  const int uc = grouped ? gc + 8 : I + i;
  const float g = ldf<T>(row + gc), u = ldf<T>(row + uc);
  stf<T>(out + (size_t)n * I + i, gate_act(g, gelu) * u);
}

// bfloat16 rows whose width is a multiple of 8: eight values per thread, 16-byte loads and stores.
__global__ __launch_bounds__(256) void swiglu_bf16x8_kernel(const bf16_t* __restrict__ x, bf16_t* __restrict__ out,
                                                            int I, long long total8, int grouped, int gelu) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const int per_row = I >> 3;
  for (long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x; idx < total8;
       idx += (long long)gridDim.x * blockDim.x) {
    const long long n = idx / per_row;
    const int c = (int)(idx - n * per_row) << 3;
    const bf16_t* row = x + (size_t)n * 2 * I;
    const u32x4 gv = *reinterpret_cast<const u32x4*>(row + (grouped ? 2 * c : c));
    const u32x4 uv = *reinterpret_cast<const u32x4*>(row + (grouped ? 2 * c + 8 : I + c));
    u32x4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float g0 = __uint_as_float(gv[k] << 16), g1 = __uint_as_float(gv[k] & 0xffff0000u);
      const float u0 = __uint_as_float(uv[k] << 16), u1 = __uint_as_float(uv[k] & 0xffff0000u);
      const float a0 = gate_act(g0, gelu) * u0, a1 = gate_act(g1, gelu) * u1;
      o[k] = (uint32_t)f32_to_bf16(a0) | ((uint32_t)f32_to_bf16(a1) << 16);
    }
    *reinterpret_cast<u32x4*>(out + (size_t)n * I + c) = o;
  }
}

extern "C" int qvl_swiglu(const void* x, void* out, int N, int I, int dtype, int grouped, int gelu, hipStream_t stream) {
  if (N <= 0) return QVL_OK;
  if (I <= 0 || (grouped && I % 8)) return QVL_ERR_SHAPE;
  if (N > 65535) return QVL_ERR_LIMIT;
  const dim3 grid((I + 255) / 256, N);
  if (dtype == 0)
    hipLaunchKernelGGL(swiglu_kernel<float>, grid, dim3(256), 0, stream, (const float*)x, (float*)out, I, grouped, gelu);
  else if (dtype == 1 && I % 8 == 0 && (((uintptr_t)x | (uintptr_t)out) & 15) == 0) {
    const long long total8 = (long long)N * (I >> 3);
    long long blocks = (total8 + 255) / 256;
    blocks = blocks > 8192 ? 8192 : blocks;
    hipLaunchKernelGGL(swiglu_bf16x8_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, (const bf16_t*)x,
                       (bf16_t*)out, I, total8, grouped, gelu);
  } else if (dtype == 1)
    hipLaunchKernelGGL(swiglu_kernel<bf16_t>, grid, dim3(256), 0, stream, (const bf16_t*)x, (bf16_t*)out, I,
                       grouped, gelu);
  else
    return QVL_ERR_DTYPE;
  return qvl_launch_status();
}

// ---------------------------------------------------------------------------------------
// Page copy (reference cache.py:537-545): page src[i] -> page dst[i] in every layer of a cache
// tensor [layers, pages, page_bytes].  Used when a request is forked: whole pages are shared,
// the page being filled is copied.
// ---------------------------------------------------------------------------------------
__global__ void copy_pages_kernel(char* __restrict__ cache, size_t layer_bytes, int page_bytes,
                                  const int* __restrict__ src, const int* __restrict__ dst) {
  const int i = blockIdx.x, layer = blockIdx.y;
  const uint4* from = reinterpret_cast<const uint4*>(cache + layer * layer_bytes + (size_t)src[i] * page_bytes);
  uint4* to = reinterpret_cast<uint4*>(cache + layer * layer_bytes + (size_t)dst[i] * page_bytes);
  for (int c = threadIdx.x; c < page_bytes / 16; c += blockDim.x) to[c] = from[c];
}

extern "C" int qvl_copy_pages(void* cache, long long layer_bytes, int page_bytes, const void* src, const void* dst,
                              int n, int layers, hipStream_t stream) {
  if (n <= 0 || layers <= 0) return QVL_OK;
  if (page_bytes <= 0 || page_bytes % 16 || layer_bytes < page_bytes || ((uintptr_t)cache & 15)) return QVL_ERR_SHAPE;
  if (layers > 65535) return QVL_ERR_LIMIT;
  hipLaunchKernelGGL(copy_pages_kernel, dim3(n, layers), dim3(256), 0, stream, (char*)cache, (size_t)layer_bytes,
                     page_bytes, (const int*)src, (const int*)dst);
  return qvl_launch_status();
}
