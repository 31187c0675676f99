// Products with some hundred rows and inner sizes of a few thousand: X[M, K] . W[N, K]^T, bfloat16 operands, float32 sums, not cut along K: added to
// the float32 residual, or the stacked q | k | v projection with bias, rotation and cache write on the sums.
//
// Tiles of 128 x 128 (gemm_tile.hip) leave most compute units idle there unless K is cut, and then what the product writes (float32 slabs), the flush
// of it and the kernel that reads it again take as long as the product.  Here a block has 64 rows of W and 64 or 80 of X, small tiles for all
// compute units.  What bounds that is both operands' way into LDS (110 GB/s a compute unit out of the L2) and one barrier a step, so steps have 128
// values of K, three of them on their way while one is multiplied; the eight waves stand two by four: 32 rows of W and a quarter of a step's columns each, so that LDS
// delivers an operand of X once for 32 rows of W.  The quarters' sums meet in LDS when all of K has been read.
// Blocks with the same rows of W follow each other on one XCD (workgroups go to the XCDs in turn): W comes from memory once.
//
// Per call, in brackets slabs and the kernel that reads them: 2,048 x 2,048 into the residual and the norm behind it, 280 rows 14.6 us (17.9), 420 15.3 (20.7);
// 16 + 2 x 2 heads of 2,048, 280 rows 13.5 (20.8), 420 16.7 (22.9).  Three, four or five steps on their way, and blocks that begin at one or at
// different places of K, the same within 2 per cent; steps of 64 columns 12.5 us for 11.2 (2,048 x 2,048, 420 rows).  Error of the sums against 64
// bits 0.86e-7 of the result (tiles in slabs 1.2 to 1.5e-7).  420 prompt tokens, 8 layers of 3B sizes: 1,245 us to 1,109.
//
// Where a norm waits behind the sum, whose reader takes rows that are not yet divided by their root mean square, the blocks leave the new rows times the
// norm's gain and their sums of squares (1.2 us), and the norm's kernel (4.0 us, and a launch of a host that is hardly ahead) falls away: the pass above
// 2 per cent, one that mixes prompts and decoding 0.6.
#include "tile_product.h"

#include <type_traits>

#define MID_WAVES 8
#define MID_N 64
#define MID_LDS 163840
#define MID_PARTS 256                            // places of a row's sums of squares

enum { MID_INTO = 0, MID_HEADS = 1 };

struct MidArgs {
  const bf16_t* x;       // [M, K], rows ldx apart
  const bf16_t* w;       // [N, K], rows ldw apart
  long long ldx, ldw;
  int M, N, K;
  int n_blocks, m_blocks;
  float* h;              // MID_INTO: [M, N] += product, rows ldh apart
  long long ldh;
  int wide;              // four results may be read and written at once
  const float* gain;     // [N], of the norm behind the sum, or null: then nothing is left for it
  bf16_t* left;          // [M, N]: the new h times gain
  float* left_squares;   // [M, MID_PARTS]: of a row of the new h the sum of squares of every block's outputs
  // MID_HEADS: W's rows are nq query, nkv key and nkv value heads of 128 channels
  const float* bias;     // [N] or null
  const float2* cs;      // [M, 64]: cosine and sine
  const int* slot;       // [M]: page * ps + place, or -1
  bf16_t* q_out;         // [M, nq 128]
  bf16_t* kc;            // [page][nkv][ps][128]
  bf16_t* vc;            // [page][nkv][128][ps]
  int nq, nkv, ps;
};

// MT column tiles of 16 rows of X.
template <int MT, int OUT>
__global__ __launch_bounds__(64 * MID_WAVES) void gemm_mid_kernel(MidArgs p) {
  constexpr int STAGE = (MID_N + 16 * MT) * 256, STAGES = 4;
  constexpr int ALL = (MID_N + 16 * MT) / 4, EACH = ALL / 8, FEW = ALL % 8, F = EACH + (FEW > 0);      // fetches of 4 rows a step: the first FEW waves one more
  constexpr int SUMS = 4 * 4 * MT * 256;                            // of all quarters
  static_assert(STAGES * STAGE <= MID_LDS && SUMS * 4 <= STAGES * STAGE, "the quarters' sums lie where the steps were");
  __shared__ __attribute__((aligned(16))) char lds[STAGES * STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
  const int group = wave & 1, quarter = wave >> 1;
  const int turn8 = blockIdx.x >> 3, block = (int)(blockIdx.x & 7) + 8 * (turn8 / p.m_blocks), m0 = turn8 % p.m_blocks * 16 * MT;
  if (block >= p.n_blocks) return;
  const int steps = (p.K + 127) / 128, last_chunks = p.K % 128 ? (p.K % 128) / 8 : 16;      // of a last step, 8 values each
  // row of W behind row i of the block.  Heads: 32 channels of a head, then the 32 they are turned with.
  auto w_row = [&](int i) {
    if (OUT == MID_HEADS) return (block >> 1) * 128 + (block & 1) * 32 + (i & 31) + (i >> 5) * 64;
    return min(MID_N * block + i, p.N - 1);                         // rows that do not exist are read from the last that does
  };
  // A step's fetch i brings 4 rows of 256 bytes, W's first, then X's; wave w makes the fetches w, w + 8, ...  Row rho's 16-byte chunk c lies at place
  // c ^ (rho mod 16): the 16 rows of an operand read touch all banks.
  uint32_t from0[F], chunk[F];
#pragma unroll
  for (int j = 0; j < F; ++j) {
    const int i = wave + 8 * j, rho = 4 * (i < 16 ? i : i - 16) + g, m = m0 + rho;
    chunk[j] = r ^ (rho & 15);
    const uint32_t row = i < 16 ? (uint32_t)w_row(rho) * (uint32_t)p.ldw : (uint32_t)(m < p.M ? m : 0) * (uint32_t)p.ldx;
    from0[j] = row * 2 + 16 * chunk[j];
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)&lds[0];
  // Blocks begin at different places of K and go round (those with the same rows of W at the same): all at the same place would ask the same few
  // memory channels.
  const int turn = (int)((block * 29u) % (unsigned)steps);
  int asked = 0, ask_stage = 0, ask_at = turn;
  auto ask = [&]() __attribute__((always_inline)) {
    if (asked >= steps) return;
    const uint32_t at = lds0 + ask_stage * STAGE, k = (uint32_t)ask_at * 256;
    const bool cut = last_chunks < 16 && ask_at == steps - 1;        // chunks beyond K are read from the step's first: they are not multiplied
#pragma unroll
    for (int j = 0; j < F; ++j) {
      const int i = wave + 8 * j;
      if (j == EACH && wave >= FEW) break;
      const uint32_t from = from0[j] + k - (cut && chunk[j] >= (uint32_t)last_chunks ? 16u * chunk[j] : 0u);
      tp_fetch16(i < 16 ? p.w : p.x, from, at + i * 1024);
    }
    ++asked;
    if (++ask_at == steps) ask_at = 0;
    ask_stage = ask_stage + 1 == STAGES ? 0 : ask_stage + 1;
  };
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i) ask();
  // A sum is formed of short runs: the steps' products go to two sums in turn, which join the rest every eight steps.
  tp_f32x4 run[2][2][MT], acc[2][MT];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int c = 0; c < MT; ++c) run[0][t][c] = run[1][t][c] = acc[t][c] = tp_f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t of = r * 256 + (((4 * quarter + g) ^ r) << 4);     // row r of 16, chunk 4 quarter + g
  tp_bf16x8 w8[2][2], x8[2][MT];
  int stage = 0, mul_at = turn;
  auto read = [&](auto buf) __attribute__((always_inline)) {
    constexpr int B = decltype(buf)::value;
    const char* from = lds + stage * STAGE + of;
#pragma unroll
    for (int t = 0; t < 2; ++t) w8[B][t] = *reinterpret_cast<const tp_bf16x8*>(from + (2 * group + t) * 4096);
#pragma unroll
    for (int c = 0; c < MT; ++c) x8[B][c] = *reinterpret_cast<const tp_bf16x8*>(from + MID_N * 256 + c * 4096);
    stage = stage + 1 == STAGES ? 0 : stage + 1;
  };
  auto multiply = [&](auto buf, int s) __attribute__((always_inline)) {      // step s's
    constexpr int B = decltype(buf)::value;
    if (last_chunks < 16 && mul_at == steps - 1 && 4 * quarter + g >= last_chunks) {      // chunks beyond K are no part of the sums
#pragma unroll
      for (int t = 0; t < 2; ++t) w8[B][t] = tp_bf16x8{};
#pragma unroll
      for (int c = 0; c < MT; ++c) x8[B][c] = tp_bf16x8{};
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int c = 0; c < MT; ++c) run[B][t][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w8[B][t], x8[B][c], run[B][t][c], 0, 0, 0);
    if (++mul_at == steps) mul_at = 0;
    if ((s & 7) == 7 || s == steps - 1) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int c = 0; c < MT; ++c) {
          acc[t][c] += run[0][t][c] + run[1][t][c];
          run[0][t][c] = run[1][t][c] = tp_f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
  };
  auto step = [&](int s, auto here, auto before) __attribute__((always_inline)) {
    if (s < steps) {
      if (FEW > 0 && wave < FEW) tp_wait_steps<STAGES - 2, EACH + 1>(asked - 1 - s);
      else tp_wait_steps<STAGES - 2, EACH>(asked - 1 - s);          // all but the steps asked for behind this one have come
      tp_wait_lds();
      tp_barrier();                           // every wave's part of the step is there, and the step before has been read
      ask();
      read(here);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (s > 0) multiply(before, s - 1);
  };
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  for (int s = 0; s <= steps; s += 2) {
    step(s, even, odd);
    if (s < steps) step(s + 1, odd, even);
  }
  // MID_INTO: what the sums are added to, and the gain, are on their way while the quarters meet
  constexpr int ENDS = (16 * 16 * MT + 64 * MID_WAVES - 1) / (64 * MID_WAVES);
  const int mine = MID_N * block + 4 * (threadIdx.x & 15);      // the first of this lane's four outputs
  const bool four = OUT == MID_INTO && p.wide && mine + 3 < p.N;
  tp_f32x4 h4[ENDS], g4 = {0.f, 0.f, 0.f, 0.f};
  if (four) {
    if (p.gain) g4 = *reinterpret_cast<const tp_f32x4*>(p.gain + mine);
#pragma unroll
    for (int t = 0; t < ENDS; ++t) {
      const int m = m0 + ((threadIdx.x + 64 * MID_WAVES * t) >> 4);
      h4[t] = *reinterpret_cast<const tp_f32x4*>(p.h + min(m, p.M - 1) * p.ldh + mine);
    }
  }
  tp_wait_fetches<0>();
  tp_wait_lds();
  __syncthreads();                            // the stages have been read: their place is the quarters'
  // [quarter][tile of 16 rows of W][column tile][row of X][row of W]
  float* sums = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int c = 0; c < MT; ++c)
      *reinterpret_cast<tp_f32x4*>(sums + ((quarter * 4 + 2 * group + t) * MT + c) * 256 + r * 16 + 4 * g) = acc[t][c];
  __syncthreads();
  // four neighbouring rows of W, from row 4 i of the block on, of row m of the block's rows of X
  auto total = [&](int i, int m) {
    const float* at = sums + ((i >> 2) * MT + (m >> 4)) * 256 + (m & 15) * 16 + 4 * (i & 3);
    tp_f32x4 v = *reinterpret_cast<const tp_f32x4*>(at);
#pragma unroll
    for (int k = 1; k < 4; ++k) v += *reinterpret_cast<const tp_f32x4*>(at + k * (4 * MT * 256));
    return v;
  };
  if constexpr (OUT == MID_INTO) {
#pragma unroll
    for (int t = 0; t < ENDS; ++t) {
      const int e = threadIdx.x + 64 * MID_WAVES * t, i = e & 15, m = e >> 4, n = mine;      // (a row's sixteen lanes stay together)
      if (m >= 16 * MT || m0 + m >= p.M) break;
      float* h = p.h + (m0 + m) * p.ldh + n;
      bf16_t* left = p.left + (size_t)(m0 + m) * p.N + n;
      tp_f32x4 v = total(i, m);
      if (four) {
        v += h4[t];
        *reinterpret_cast<tp_f32x4*>(h) = v;
        if (p.gain) {                 // (N is a multiple of 4 there, gain and left lie on 16-byte boundaries)
          const uint32_t a = f32_to_bf16(v[0] * g4[0]), b = f32_to_bf16(v[1] * g4[1]), c = f32_to_bf16(v[2] * g4[2]), d = f32_to_bf16(v[3] * g4[3]);
          *reinterpret_cast<uint2*>(left) = uint2{a | b << 16, c | d << 16};
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (n + j < p.N) {
            h[j] = v[j] = h[j] + v[j];
            if (p.gain) left[j] = f32_to_bf16(v[j] * p.gain[n + j]);
          } else {
            v[j] = 0.f;
          }
        }
      }
      if (p.gain) {
        float square = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) square += __shfl_xor(square, o, QVL_WAVE);
        if (i == 0) p.left_squares[(size_t)(m0 + m) * MID_PARTS + block] = square;
      }
    }
  } else {
    for (int e = threadIdx.x; e < 8 * 16 * MT; e += 64 * MID_WAVES) {
      const int i = e & 7, m = m0 + (e >> 3), head = block >> 1, f = (block & 1) * 32 + 4 * i;
      if (m >= p.M) continue;
      tp_f32x4 a = total(i, e >> 3), b = total(i + 8, e >> 3);
      if (p.bias) {
        a += *reinterpret_cast<const tp_f32x4*>(p.bias + head * 128 + f);
        b += *reinterpret_cast<const tp_f32x4*>(p.bias + head * 128 + f + 64);
      }
      if (head < p.nq + p.nkv) {              // (values are stored as they are)
        const tp_f32x4 t0 = *reinterpret_cast<const tp_f32x4*>(p.cs + (size_t)m * 64 + f), t1 = *reinterpret_cast<const tp_f32x4*>(p.cs + (size_t)m * 64 + f + 2);
        const tp_f32x4 c = {t0[0], t0[2], t1[0], t1[2]}, s = {t0[1], t0[3], t1[1], t1[3]}, a0 = a;
        a = a0 * c - b * s;
        b = b * c + a0 * s;
      }
      bf16_t lo[4], hi[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) lo[j] = f32_to_bf16(a[j]), hi[j] = f32_to_bf16(b[j]);
      const uint2 first = {(uint32_t)lo[0] | (uint32_t)lo[1] << 16, (uint32_t)lo[2] | (uint32_t)lo[3] << 16};
      const uint2 second = {(uint32_t)hi[0] | (uint32_t)hi[1] << 16, (uint32_t)hi[2] | (uint32_t)hi[3] << 16};
      if (head < p.nq) {
        bf16_t* q = p.q_out + ((size_t)m * p.nq + head) * 128 + f;
        *reinterpret_cast<uint2*>(q) = first;
        *reinterpret_cast<uint2*>(q + 64) = second;
        continue;
      }
      const int slot = p.slot[m];
      if (slot < 0) continue;
      const int page = slot / p.ps, place = slot - page * p.ps, kv = head - p.nq;
      if (kv < p.nkv) {
        bf16_t* k = p.kc + (((size_t)page * p.nkv + kv) * p.ps + place) * 128 + f;
        *reinterpret_cast<uint2*>(k) = first;
        *reinterpret_cast<uint2*>(k + 64) = second;
      } else {
        bf16_t* v = p.vc + (((size_t)page * p.nkv + kv - p.nkv) * 128 + f) * p.ps + place;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[(size_t)j * p.ps] = lo[j];
          v[(size_t)(64 + j) * p.ps] = hi[j];
        }
      }
    }
  }
}

// 64 or 80 rows of X a block, whichever leaves fewer rounds of blocks on the compute units, and then fewer rows that do not exist.
static int mid_tiles(int M, int n_blocks, int cus) {
  const long long b4 = (long long)n_blocks * ((M + 63) / 64), b5 = (long long)n_blocks * ((M + 79) / 80);
  const long long t4 = 4 * ((b4 + cus - 1) / cus), t5 = 5 * ((b5 + cus - 1) / cus);
  return t5 < t4 ? 5 : 4;
}
template <int OUT>
static int mid_launch(MidArgs& p, int cus, hipStream_t stream) {
  if (p.K <= 0 || p.K % 8 || p.ldx < p.K || p.ldw < p.K || p.ldx % 8 || p.ldw % 8 || !p.x || !p.w || cus <= 0 || (((uintptr_t)p.x | (uintptr_t)p.w) % 16))
    return QVL_ERR_SHAPE;
  // offsets from the first row are 32-bit
  if ((unsigned long long)((p.N - 1) * p.ldw + p.K) * 2 >= 0xffffff00ull || (unsigned long long)((p.M - 1) * p.ldx + p.K) * 2 >= 0xffffff00ull)
    return QVL_ERR_LIMIT;
  p.n_blocks = (p.N + MID_N - 1) / MID_N;
  const int tiles = mid_tiles(p.M, p.n_blocks, cus);
  p.m_blocks = (p.M + 16 * tiles - 1) / (16 * tiles);
  const dim3 grid((unsigned)((p.n_blocks + 7) / 8 * 8 * p.m_blocks)), block(64 * MID_WAVES);
  if (tiles == 5) hipLaunchKernelGGL((gemm_mid_kernel<5, OUT>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((gemm_mid_kernel<4, OUT>), grid, block, 0, stream, p);
  return qvl_launch_status();
}

// h (float32 [M, N], rows ldh apart) += x . w^T; x: bfloat16 [M, K], rows ldx apart; w: bfloat16 [N, K], rows ldw apart; both on 16-byte boundaries, K a
// multiple of 8.  gain (float32 [N], or null), for the norm behind the sum: left (bfloat16 [M, N]) = the new h times gain, left_squares (float32 [M, 256]): the
// sums of squares of 64 values each of a row of the new h, one after the other.
extern "C" int qvl_gemm_mid_into(const void* x, long long ldx, const void* w, long long ldw, void* h, long long ldh, const void* gain, void* left,
                                 void* left_squares, int M, int N, int K, int cus, hipStream_t stream) {
  if (M <= 0 || N <= 0) return QVL_OK;
  if (!h || ldh < N || (gain && (!left || !left_squares || N > MID_N * MID_PARTS))) return QVL_ERR_SHAPE;
  MidArgs p{};
  p.x = (const bf16_t*)x; p.ldx = ldx; p.w = (const bf16_t*)w; p.ldw = ldw; p.M = M; p.N = N; p.K = K;
  p.gain = (const float*)gain; p.left = (bf16_t*)left; p.left_squares = (float*)left_squares;
  p.h = (float*)h; p.ldh = ldh; p.wide = ldh % 4 == 0 && (uintptr_t)h % 16 == 0 && (!gain || (N % 4 == 0 && ((uintptr_t)gain | (uintptr_t)left) % 16 == 0));
  return mid_launch<MID_INTO>(p, cus, stream);
}

// The stacked projection of nq query, nkv key and nkv value heads of 128 channels with bias (float32 or null), rotation and cache write: q_out bfloat16
// [M, nq 128]; keys and values into their pages, kc [page][nkv][ps][128], vc [page][nkv][128][ps] (slot[m] = page * ps + place, or -1).  cs: float32
// [M, 64, 2].  bias, cs, q_out, kc on 16-byte boundaries.
extern "C" int qvl_gemm_mid_heads(const void* x, long long ldx, const void* w, long long ldw, const void* bias, const void* cs, const void* slot, void* q_out,
                                  void* kc, void* vc, int M, int K, int nq, int nkv, int ps, int cus, hipStream_t stream) {
  if (M <= 0) return QVL_OK;
  if (nq <= 0 || nkv < 0 || !cs || !q_out || (nkv && (ps <= 0 || !slot || !kc || !vc)) ||
      (((uintptr_t)bias | (uintptr_t)cs | (uintptr_t)q_out | (uintptr_t)kc) % 16) || (long long)(nq + 2ll * nkv) * 128 > 0x7fffffffll)
    return QVL_ERR_SHAPE;
  MidArgs p{};
  p.x = (const bf16_t*)x; p.ldx = ldx; p.w = (const bf16_t*)w; p.ldw = ldw; p.M = M; p.N = (nq + 2 * nkv) * 128; p.K = K;
  p.bias = (const float*)bias; p.cs = (const float2*)cs; p.slot = (const int*)slot; p.q_out = (bf16_t*)q_out; p.kc = (bf16_t*)kc; p.vc = (bf16_t*)vc;
  p.nq = nq; p.nkv = nkv; p.ps = ps;
  return mid_launch<MID_HEADS>(p, cus, stream);
}
