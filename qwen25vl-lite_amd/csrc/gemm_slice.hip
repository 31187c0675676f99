// The stacked q | k | v projection of an attention for the up to 64 rows of a decode step: X[M, K] . W[N, K]^T, bfloat16 operands,
// float32 sums, with bias, rotation and cache write on the sums.
//
// What bounds it is one trip to memory and the start and end of a launch: 18 rows of W a compute unit (4,608 x 3,584 on 256
// units, 129 KB) are 5 us of reading.  So every block has one tile and everything it reads of W is asked for before anything is
// waited for: a block's eight waves take an eighth of K each, a wave's operands of W (v_mfma_f32_16x16x32_bf16) come from memory
// straight into registers, and the waves' sums meet in LDS once.  A load of W covers 16 rows of 64 bytes; neighbouring steps, asked for back to
// back, share a line, and W is not marked as read once, which would fetch the line's second half anew.
//
// X is the same for all blocks and comes from the L2, but every compute unit has to take in all of it (64 rows of 3,584: 458 KB): in
// operand layout at 37 GB/s (64 rows 22.7 us), by way of LDS in loads of whole lines faster (16.5).
//
// The rows of W are dealt out evenly whatever their number: a block has `per` pairs of channels (f, f + hd / 2) of a head, 9 of 4,608
// rows on 256 units, 5 of 2,560, the first of each in one tile of 16, the second in another, so that they meet in a lane; lanes beyond them ask for
// nothing.  Tiles of 16 rows of queries and keys, then what is left of the values (gemm_resident) took two rounds there and 144 units here: 1, 8, 16,
// 32, 64 rows of 4,608 x 3,584 9.1, 9.8, 10.1, 12.5, 16.5 us for 12.6, 13.1, 14.3, 18.2, 21.3; of 2,560 x 2,048 5.5, 5.5, 5.7, 7.1, 9.8 for 8.4, 8.7, 9.8,
// 11.8, 14.5; of 6,144 x 4,096 12.5, 13.0, 13.4, 16.0, 20.3 for 16.9, 17.2, 18.1, 18.9 (slabs and the rotation's kernel), 27.4.
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

struct SliceArgs {
  const bf16_t* x;      // [M, K], rows ldx apart
  const bf16_t* w;      // [N, K], rows ldw apart
  const float* bias;    // [N] or null
  int ldx, ldw;
  int M, N, K;
  int pairs, per;       // of rows of W, in all and of a block, at most 16
  int steps;            // of 32 values of K, of a wave: even
  const float2* cs;     // [M, hd / 2]: cosine and sine
  const int* slot;      // [M]: page * ps + place, or -1
  bf16_t* q_out;        // [M, nq hd]
  bf16_t* kc;           // [page][nkv][ps][hd]
  bf16_t* vc;           // [page][nkv][hd][ps]
  int nq, nkv, hd, ps;
  // The rows of X are rows of the sum times a norm's gain, not yet divided by their root mean square: row m's squares add up to
  // those of squares[256 m ...], `parts` of them (up to 16 rows; null: X is as it is)
  const float* squares;
  int parts;
  float eps;
};

#define PAST_END 0x80000000u      // no buffer reaches it (the host checks): a lane that asks there, or a little beyond, gets zeros without traffic
#define SLICE_WAVES 8
#define HOLD_ORDER() __builtin_amdgcn_sched_barrier(0)

__device__ __forceinline__ bf16x8_t load16(__amdgpu_buffer_rsrc_t r, uint32_t at, int fixed) {
  return __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(r, at, fixed, 0));
}

__device__ __forceinline__ void fetch16_to_lds(const void* base, uint32_t lane_bytes, uint32_t lds_at) {
  // lane l of the wave puts its 16 bytes at M0 + 16 l of LDS
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_bytes), "s"(base), "s"(lds_at)
               : "memory", "m0");
}
// Wait until at most N of this wave's loads are outstanding (they finish in order).
template <int N>
__device__ __forceinline__ void wait_loads() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
}

// All but the `ahead` stages of LOADS loads asked for last have come (at most MOST are ahead).
template <int MOST, int LOADS>
__device__ __forceinline__ void wait_stages(int ahead) {
  if constexpr (MOST <= 0) {
    wait_loads<0>();
  } else {
    if (ahead >= MOST) wait_loads<MOST * LOADS>();
    else wait_stages<MOST - 1, LOADS>(ahead);
  }
}

// S: steps of a wave at most; CT: column tiles of 16 rows of X.
template <int S, int CT>
__global__ __launch_bounds__(64 * SLICE_WAVES) void gemm_slice_kernel(SliceArgs p) {
  constexpr int ENDS = (256 * CT + 64 * SLICE_WAVES - 1) / (64 * SLICE_WAVES);      // pairs of results a thread finishes
  constexpr int STAGE = CT * 16 * 128;                                              // two steps of a wave's rows of X in LDS
  constexpr int DEEP = CT <= 2 ? 8 / CT : 2;                                        // stages of a wave that LDS holds
  static_assert(CT > 1 || DEEP >= S / 2, "fetch_x leaves out loads");
  __shared__ float scale[16];
  constexpr int SUMS = SLICE_WAVES * 2 * CT * 256 * 4, RING = SLICE_WAVES * DEEP * STAGE;
  __shared__ __attribute__((aligned(16))) char lds[SUMS > RING ? SUMS : RING];
  float (*sums)[2][CT * 256] = reinterpret_cast<float (*)[2][CT * 256]>(lds);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
  const int half = p.hd >> 1, first = blockIdx.x * p.per, k_wave = wave * p.steps * 32, k0 = k_wave + 8 * g;
  // how many of this lane's steps begin inside K (K is a multiple of 8) and inside the wave's slice
  const int inside = min(p.steps, (p.K - k0 + 31) >> 5);
  const auto w_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.w), 0, (int)(((uint32_t)(p.N - 1) * p.ldw + p.K) * 2), 0x00020000);
  // X by way of LDS: stage s holds 128 bytes of every row, chunk c (16 bytes) of row m at place c ^ ((m >> 1) & 7): the 16 rows
  // of an operand read touch all banks.  A load brings 8 rows, whole lines.  Rows beyond M are row 0, chunks beyond K the slice's first
  // (their products are left out, or not stored).
  const uint32_t ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)&lds[0] + wave * DEEP * STAGE;
  auto fetch_x = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2 * CT; ++j) {
      if (CT == 1 && 8 * j >= p.M) break;      // (DEEP holds all stages of one column tile: nothing counts these loads)
      const int m = 8 * j + (lane >> 3), k = k_wave + 64 * s + 8 * ((lane & 7) ^ ((m >> 1) & 7));
      const uint32_t at = ((uint32_t)(m < p.M ? m : 0) * p.ldx + (k < p.K ? k : k_wave < p.K ? k_wave : 0)) * 2;
      fetch16_to_lds(p.x, at, ring + s % DEEP * STAGE + j * 1024);
    }
  };
  const int stages = p.steps >> 1;
#pragma unroll
  for (int s = 0; s < DEEP && s < S / 2; ++s)
    if (s < stages) fetch_x(s);
  uint32_t w_at[2];
  {
    const int i = first + r;
    const bool exists = r < p.per && i < p.pairs;
    const int row = i / half * p.hd + i % half;
#pragma unroll
    for (int t = 0; t < 2; ++t) w_at[t] = exists ? ((uint32_t)(row + t * half) * p.ldw + k0) * 2 : PAST_END;
  }
  bf16x8_t w[S][2];
#pragma unroll
  for (int u = 0; u < S; ++u)
#pragma unroll
    for (int t = 0; t < 2; ++t) w[u][t] = load16(w_buf, u < inside ? w_at[t] : PAST_END, u * 64);
  float4 square[2];       // of rows wave and wave + 8
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    square[i] = float4{0.f, 0.f, 0.f, 0.f};
    if (CT == 1 && p.squares && wave + 8 * i < p.M && 4 * lane < p.parts)
      square[i] = *reinterpret_cast<const float4*>(p.squares + (wave + 8 * i) * 256 + 4 * lane);
  }
  // what the results need beside the sums; result e of the block: row e / 16 of X, pair e mod 16
  float b0[ENDS], b1[ENDS];
  float2 turn[ENDS];     // (of queries and keys)
  int slot[ENDS];
#pragma unroll
  for (int i = 0; i < ENDS; ++i) {
    const int e = threadIdx.x + 64 * SLICE_WAVES * i, m = e >> 4, pair = first + (e & 15);
    b0[i] = b1[i] = 0.f;
    turn[i] = float2{1.f, 0.f};
    slot[i] = -1;
    if (m >= p.M || (e & 15) >= p.per || pair >= p.pairs) continue;
    const int head = pair / half, f = pair % half;
    if (p.bias) b0[i] = p.bias[head * p.hd + f], b1[i] = p.bias[head * p.hd + f + half];
    if (head < p.nq + p.nkv) turn[i] = p.cs[m * half + f];
    if (head >= p.nq) slot[i] = p.slot[m];
  }
  HOLD_ORDER();
  // The two halves of a wave's slice are summed apart (one chain rounds off a quarter more).
  f32x4_t acc[2][2][CT];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int c = 0; c < CT; ++c) acc[h][t][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < S / 2; ++s) {
    if (s >= stages) break;
    // The first stages were asked for before W: they are there when W's steps are.  The others were asked for last but for the stages
    // behind them.
    if (s < DEEP) asm volatile("" ::"v"(w[2 * s][0]), "v"(w[2 * s][1]) : "memory");
    else wait_stages<DEEP - 1, 2 * CT>(stages - 1 - s);
    const char* from = lds + (wave * DEEP + s % DEEP) * STAGE + r * 128;
    bf16x8_t x[2][CT];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        x[h][c] = *reinterpret_cast<const bf16x8_t*>(from + c * 2048 + (((4 * h + g) ^ ((r >> 1) & 7)) << 4));
        if (k_wave + p.steps * 32 > p.K && 2 * s + h >= inside) x[h][c] = bf16x8_t{};
      }
    if (s + DEEP < stages) {
      __builtin_amdgcn_s_waitcnt(0xc07f);      // the stage has been read
      HOLD_ORDER();
      fetch_x(s + DEEP);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c)
          acc[2 * s >= S / 2][t][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[2 * s + h][t], x[h][c], acc[2 * s >= S / 2][t][c], 0, 0, 0);
  }
  if (CT == 1 && p.squares) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int m = wave + 8 * i, have = p.parts - 4 * lane;
      if (m >= p.M) break;
      const float s = wave_sum((square[i].x + (have > 1 ? square[i].y : 0.f)) + ((have > 2 ? square[i].z : 0.f) + (have > 3 ? square[i].w : 0.f)));
      if (lane == 0) scale[m] = 1.0f / sqrtf(s / (float)p.K + p.eps);
    }
  }
  __syncthreads();      // the sums' place is the stages'
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int c = 0; c < CT; ++c) *reinterpret_cast<f32x4_t*>(&sums[wave][t][(16 * c + r) * 16 + 4 * g]) = acc[0][t][c] + acc[1][t][c];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ENDS; ++i) {
    const int e = threadIdx.x + 64 * SLICE_WAVES * i, m = e >> 4, pair = first + (e & 15);
    if (m >= p.M || (e & 15) >= p.per || pair >= p.pairs) continue;
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int s = 0; s < SLICE_WAVES; ++s) a += sums[s][0][e], b += sums[s][1][e];
    const int head = pair / half, f = pair % half;
    if (CT == 1 && p.squares) a *= scale[m], b *= scale[m];
    a += b0[i];
    b += b1[i];
    bf16_t* to;
    int apart = half;
    if (head < p.nq) {
      to = p.q_out + ((size_t)m * p.nq + head) * p.hd + f;
    } else {
      if (slot[i] < 0) continue;
      const bool key = head < p.nq + p.nkv;
      const int page = slot[i] / p.ps, place = slot[i] - page * p.ps;
      const size_t of = (size_t)page * p.nkv + (head - p.nq - (key ? 0 : p.nkv));
      to = key ? p.kc + (of * p.ps + place) * p.hd + f : p.vc + (of * p.hd + f) * p.ps + place;
      if (!key) apart = half * p.ps;
    }
    // (values are stored as they are: turned by (1, 0), one that is not finite would take the other along)
    const bool turns = head < p.nq + p.nkv;
    to[0] = f32_to_bf16(turns ? a * turn[i].x - b * turn[i].y : a);
    to[apart] = f32_to_bf16(turns ? b * turn[i].x + a * turn[i].y : b);
  }
}

// K that a block's waves cover in one go.
#define SLICE_K(S) (32 * SLICE_WAVES * (S))

// Whether the kernel takes a projection: up to 64 rows, inner sizes up to 4,096 in steps of 8, at most 16 pairs of rows of W a compute unit.
extern "C" int qvl_gemm_slice_takes(int M, int N, int K, int cus) {
  return M > 0 && M <= 64 && K > 0 && K % 8 == 0 && K <= SLICE_K(16) && N > 0 && N % 2 == 0 && cus > 0 && N <= 32ll * cus;
}

extern "C" int qvl_gemm_slice_most_k() { return SLICE_K(16); }

// The stacked projection of nq query, nkv key and nkv value heads of hd channels (hd even) with bias (float32 or null), rotation and cache write:
// q_out bfloat16 [M, nq hd]; keys and values into their pages, kc [page][nkv][ps][hd], vc [page][nkv][hd][ps] (slot[m] = page * ps
// + place, or -1).  cs: float32 [M, hd / 2, 2].  squares (float32 [M, 256], on a 16-byte boundary), parts, eps: x is rows of a sum times a norm's gain as
// qvl_gemm_stream_into leaves them (up to 16 rows); null: x as it is.
extern "C" int qvl_gemm_slice_rope(const void* x, int ldx, const void* w, int ldw, const void* bias, const void* cs, const void* slot,
                                   void* q_out, void* kc, void* vc, int M, int K, int nq, int nkv, int hd, int ps, int cus,
                                   const void* squares, int parts, float eps, hipStream_t stream) {
  if (M <= 0) return QVL_OK;
  if (nq <= 0 || nkv < 0 || hd <= 0 || hd % 2 || !cs || ((uintptr_t)cs % 8) || !q_out || (nkv && (ps <= 0 || !slot || !kc || !vc)) ||
      (long long)(nq + 2ll * nkv) * hd > 0x7fffffffll)
    return QVL_ERR_SHAPE;
  SliceArgs p;
  p.x = (const bf16_t*)x; p.ldx = ldx; p.w = (const bf16_t*)w; p.ldw = ldw; p.bias = (const float*)bias;
  p.M = M; p.N = (nq + 2 * nkv) * hd; p.K = K; p.pairs = p.N / 2;
  p.cs = (const float2*)cs; p.slot = (const int*)slot; p.q_out = (bf16_t*)q_out; p.kc = (bf16_t*)kc; p.vc = (bf16_t*)vc;
  p.nq = nq; p.nkv = nkv; p.hd = hd; p.ps = ps;
  p.squares = (const float*)squares; p.parts = parts; p.eps = eps;
  if (squares && (M > 16 || parts <= 0 || parts > 256 || ((uintptr_t)squares % 16))) return QVL_ERR_SHAPE;
  if (!qvl_gemm_slice_takes(M, p.N, K, cus)) return QVL_ERR_LIMIT;
  if (ldx < K || ldw < K || ldx % 8 || ldw % 8 || !x || !w || (((uintptr_t)x | (uintptr_t)w) % 16)) return QVL_ERR_SHAPE;
  // byte offsets are 32-bit, and PAST_END lies behind them
  if ((unsigned long long)M * ldx * 2 >= 0x7fffff00ull || (unsigned long long)p.N * ldw * 2 >= 0x7fffff00ull) return QVL_ERR_LIMIT;
  p.per = (p.pairs + cus - 1) / cus;
  p.steps = ((K + 32 * SLICE_WAVES - 1) / (32 * SLICE_WAVES) + 1) / 2 * 2;
  const dim3 grid((p.pairs + p.per - 1) / p.per), block(64 * SLICE_WAVES);
#define GO(S, CT) hipLaunchKernelGGL((gemm_slice_kernel<S, CT>), grid, block, 0, stream, p)
#define COLUMNS(S)                \
  do {                            \
    if (M <= 16) GO(S, 1);        \
    else if (M <= 32) GO(S, 2);   \
    else if (M <= 48) GO(S, 3);   \
    else GO(S, 4);                \
  } while (0)
  if (p.steps <= 8) COLUMNS(8);
  else if (p.steps <= 14) COLUMNS(14);
  else COLUMNS(16);
#undef COLUMNS
#undef GO
  return qvl_launch_status();
}
