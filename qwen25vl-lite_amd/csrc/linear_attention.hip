// Linear attention with a decayed outer-product state, one head at a time:
//   S_t = diag(a_t) S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t
// S is [LA_DIM, vdim] float32 per (request slot, head).  The decay a_t is one constant per head, or
// one value per key channel and token: a_t = sigmoid(z_t)^(1/tau) from float32 z, or a forget gate with a
// floor, a_t = l + (1 - l) sigmoid(z_t + b) with l and b per key channel, whose complement is the key,
// k_t = 1 - a_t (no key is read then), or a double exponential, a_t = exp(-exp(z_t + b)).  With a bonus u per
// key channel the output is formed before the state moves on and the token's own outer product enters it weighted:
// o_t = (S_(t-1) + diag(u) k_t v_t^T)^T q_t.  q, k and v are columns of the projection's rows (float32 or
// bfloat16; the offsets may also lead to other matrices of the same row stride), with an optional silu on each (`act`: bit 0 q, bit 1 k, bit 2 v) and a scale on q applied in
// float32 as they are read.  Compiled per key size (-DLA_DIM=...).
//
// The scan: a block of four waves owns 64 value channels of one head of one request and walks the
// request's tokens of this step in order, starting from the state its slot holds and leaving the
// new state there.  Lane = value channel; each wave keeps LA_DIM / 4 rows of S in registers (a key
// size that four does not divide is shared by two waves, or kept by one).
// Tokens are staged LA_TB at a time: q, k and the decays go to LDS (every lane reads the same
// word), the four partial sums of o meet in LDS.  The order of every sum is fixed by the sizes
// alone, so a token's result does not depend on how its sequence was cut into steps or on what
// else the batch holds.
//
// One prompt alone has only heads x vdim / 64 such blocks.  With G > 1 the key channels are cut
// into G groups, each with blocks of its own (four waves of LA_DIM / (4 G) rows); a group's sums of
// o go to its own slab of the output, [G, N, heads * vdim], and whoever reads the output adds the
// slabs in order (the norm that follows does).
#include "common.h"
#include <atomic>

#ifndef LA_DIM
#define LA_DIM 64
#endif
// waves of a block: four share the rows of S where the key size divides by four, else two or one
#define LA_WAVES (LA_DIM % 4 == 0 ? 4 : (LA_DIM % 2 == 0 ? 2 : 1))
#define LA_THREADS (64 * LA_WAVES)
#define LA_TB (LA_DIM > 256 ? 4 : (LA_DIM > 128 ? 8 : 16))

__device__ __forceinline__ float la_act(float z, int act) { return act ? z / (1.0f + expf(-z)) : z; }

// how the decay is given: a constant per head; sigmoid(z)^(1/tau); a floored forget gate whose complement is the key
#define LA_HEAD 0
#define LA_CHANNEL 1
#define LA_FORGET 2
#define LA_EXP 3        // exp(-exp(z + b))
// the complement of the floored forget gate, (1 - l) (1 - sigmoid(z)) = (1 - l) / (1 + exp(z)): this is the key,
// and the decay is 1 minus it
__device__ __forceinline__ float la_forget_key(float z, float lower) { return (1.0f - lower) / (1.0f + expf(z)); }

// log(sigmoid(z)) = min(z, 0) - log1p(exp(-|z|)); times 1/tau: the decay's logarithm
__device__ __forceinline__ float la_log_decay(float z, float inv_tau) { return (fminf(z, 0.f) - log1pf(expf(-fabsf(z)))) * inv_tau; }

// COLS: value channels of a lane (64 apart).  What bounds a long run is LDS and the vector unit: every value of q, k and the decays
// that a wave reads serves 64 channels with one of a lane, 128 with two, and staging is shared likewise (29 chunks of 64 tokens, 28
// heads: of 64 x 128 with a decay for each channel 117 us and 88, of 128 x 128 with one for each head 159 and 135).  Fewer tokens at a
// time and a bound on registers, for a fourth block a compute unit: 89 and 146.  (When two are taken: qvl_la_chunk_columns.)
// CHUNK: the runs are chunks of a request's (see below): each starts from zero, its state is row `run` of `state`, and
// `last` gets the product of its decays.
template <typename TP, int MODE, int G, bool BONUS, int COLS, bool CHUNK>
__global__ __launch_bounds__(LA_THREADS) void la_scan_kernel(
    const TP* __restrict__ proj, long long proj_stride, long long q_off, long long k_off, long long v_off,
    const float* __restrict__ head_decay, const float* __restrict__ z, long long z_stride, float inv_tau,
    const float* __restrict__ lower, const float* __restrict__ zbias, const float* __restrict__ bonus,
    float* __restrict__ state, const int* __restrict__ cu_q, const int* __restrict__ req_slots,
    float* __restrict__ out, long long out_slab, float* __restrict__ last, int H, int vdim, int act, float q_scale) {
  constexpr int TB = COLS > 1 && LA_DIM > 64 ? 8 : LA_TB;      // tokens staged at a time
  // key channels of this block's group (a G that does not divide the rows among the waves is never launched)
  constexpr int DG = LA_DIM % (LA_WAVES * G) == 0 ? LA_DIM / G : LA_DIM;
  constexpr int LA_ROWS = DG / LA_WAVES;    // rows of S a wave keeps
  __shared__ float qs[TB][DG];
  __shared__ float ks[TB][DG];
  constexpr bool CHANNEL_DECAY = MODE != LA_HEAD;
  __shared__ float as[CHANNEL_DECAY ? TB : 1][DG];
  // The logarithms of a channel's decays are summed by the threads that stage them where these are the same all the way.  (By way of LDS
  // they cost the fourth block of a compute unit: 63 chunks, 16 heads of 128 x 64 with a decay for each channel 271 us, so
  // 187.)
  constexpr bool OWN = LA_THREADS % DG == 0, LISTED = CHUNK && CHANNEL_DECAY && !OWN;
  __shared__ float logs[LISTED ? TB : 1][LISTED ? DG : 1], log_sums[LISTED ? DG : 1];
  __shared__ float po[TB][LA_WAVES][64 * COLS];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int head = blockIdx.y, req = blockIdx.z;
  const int vtile = blockIdx.x / G, group = blockIdx.x % G;
  const int d0 = group * DG;
  const int vcol = vtile * 64 * COLS + lane;      // and 64 further on
  const int begin = cu_q[req], end = cu_q[req + 1];
  if (begin >= end) return;
  out += (size_t)group * out_slab;
  float* srow = state + (((size_t)(CHUNK ? req : req_slots[req]) * H + head) * LA_DIM + d0 + (size_t)wave * LA_ROWS) * vdim + vcol;
  float S[COLS][LA_ROWS];
#pragma unroll
  for (int c = 0; c < COLS; ++c)
#pragma unroll
    for (int i = 0; i < LA_ROWS; ++i) S[c][i] = !CHUNK && vcol + 64 * c < vdim ? srow[(size_t)i * vdim + 64 * c] : 0.f;
  const float fixed = CHANNEL_DECAY ? 1.f : head_decay[head];
  float U[BONUS ? LA_ROWS : 1];
  if (BONUS) {
#pragma unroll
    for (int i = 0; i < LA_ROWS; ++i) U[BONUS ? i : 0] = bonus[head * LA_DIM + d0 + wave * LA_ROWS + i];
  }

  float log_sum = 0.f;
  if (LISTED && vtile == 0)      // (a channel's sum is one thread's all the way)
    for (int d = tid; d < DG; d += LA_THREADS) log_sums[LISTED ? d : 0] = 0.f;
  for (int t0 = begin; t0 < end; t0 += TB) {
    const int nt = end - t0 < TB ? end - t0 : TB;
    for (int idx = tid; idx < nt * DG; idx += LA_THREADS) {
      const int t = idx / DG, d = idx % DG;
      const TP* row = proj + (size_t)(t0 + t) * proj_stride + (size_t)head * LA_DIM + d0 + d;
      qs[t][d] = la_act(ldf<TP>(row + q_off), act & 1) * q_scale;
      if (MODE == LA_FORGET) {
        const int hd = head * LA_DIM + d0 + d;
        const float zz = z[(size_t)(t0 + t) * z_stride + hd] + (zbias ? zbias[hd] : 0.f);
        const float key = la_forget_key(zz, lower[hd]);
        ks[t][d] = key;
        as[t][d] = 1.0f - key;
        if (CHUNK) {
          const float lg = log1pf(-key);
          if (OWN) log_sum += lg;
          else logs[LISTED ? t : 0][LISTED ? d : 0] = lg;
        }
      } else {
        ks[t][d] = la_act(ldf<TP>(row + k_off), act & 2);
        if (MODE == LA_CHANNEL || MODE == LA_EXP) {
          const int hd = head * LA_DIM + d0 + d;
          const float zz = z[(size_t)(t0 + t) * z_stride + hd];
          const float lg = MODE == LA_EXP ? -expf(zz + (zbias ? zbias[hd] : 0.f)) : la_log_decay(zz, inv_tau);
          as[t][d] = expf(lg);
          if (CHUNK && OWN) log_sum += lg;
          if (LISTED) logs[LISTED ? t : 0][LISTED ? d : 0] = lg;
        }
      }
    }
    float vt[TB][COLS];
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
      for (int c = 0; c < COLS; ++c)
        vt[t][c] = (vcol + 64 * c < vdim && t < nt)
                       ? la_act(ldf<TP>(proj + (size_t)(t0 + t) * proj_stride + v_off + (size_t)head * vdim + vcol + 64 * c), act & 4)
                       : 0.f;
    __syncthreads();
    if (LISTED && vtile == 0)
      for (int d = tid; d < DG; d += LA_THREADS) {
        float sum = log_sums[LISTED ? d : 0];
        for (int t = 0; t < nt; ++t) sum += logs[LISTED ? t : 0][LISTED ? d : 0];
        log_sums[LISTED ? d : 0] = sum;
      }
#pragma unroll
    for (int t = 0; t < TB; ++t) {
      if (t < nt) {
        float acc[COLS] = {};
#pragma unroll
        for (int i = 0; i < LA_ROWS; ++i) {
          const int d = wave * LA_ROWS + i;
          const float a = CHANNEL_DECAY ? as[t][d] : fixed, k = ks[t][d], q = qs[t][d];
#pragma unroll
          for (int c = 0; c < COLS; ++c) {
            float& St = S[c][i];
            if (BONUS) {
              const float kv = k * vt[t][c];
              acc[c] += (St + U[BONUS ? i : 0] * kv) * q;
              St = a * St + kv;
            } else {
              St = a * St + k * vt[t][c];
              acc[c] += St * q;
            }
          }
        }
#pragma unroll
        for (int c = 0; c < COLS; ++c) po[t][wave][64 * c + lane] = acc[c];
      }
    }
    __syncthreads();
    for (int idx = tid; idx < nt * 64 * COLS; idx += LA_THREADS) {
      const int t = idx / (64 * COLS), l = idx % (64 * COLS);
      const int c = vtile * 64 * COLS + l;
      if (c < vdim) {
        float sum = po[t][0][l];
#pragma unroll
        for (int w = 1; w < LA_WAVES; ++w) sum += po[t][w][l];
        out[((size_t)(t0 + t) * H + head) * vdim + c] = sum;
      }
    }
    __syncthreads();
  }
  if (CHUNK && vtile == 0) {
    float* parts = &po[0][0][0];      // (read by all behind the last barrier)
    if (CHANNEL_DECAY && OWN) {
      parts[tid] = log_sum;
      __syncthreads();
    }
    for (int d = tid; d < DG; d += LA_THREADS) {
      float sum = CHANNEL_DECAY ? log_sums[LISTED ? d : 0] : logf(fixed) * (float)(end - begin);
      if (CHANNEL_DECAY && OWN) {
        sum = 0.f;
#pragma unroll
        for (int i = 0; i < LA_THREADS / DG; ++i) sum += parts[i * DG + d];
      }
      last[((size_t)req * H + head) * LA_DIM + d0 + d] = expf(sum);
    }
  }
#pragma unroll
  for (int c = 0; c < COLS; ++c)
    if (vcol + 64 * c < vdim) {
#pragma unroll
      for (int i = 0; i < LA_ROWS; ++i) srow[(size_t)i * vdim + 64 * c] = S[c][i];
    }
}

// ---------------------------------------------------------------------------------------
// Long runs, cut into chunks that are scanned side by side.  With P_t = a_c0 * ... * a_t (per key
// channel, from the chunk's first token c0 to t, t included) and S' the state before the chunk:
//   o_t = (scan from a zero state)_t + S'^T (q_t * P_t),      S_end = diag(P_last) S' + U
// where U is the state the scan from zero ends with; with a bonus, whose outputs are formed before the state moves
// on, P_(t-1) stands in the first line (1 for the chunk's first token).  The scan above runs every chunk as if it were a
// request of its own; la_carry_kernel carries the state from chunk to chunk, and la_join_kernel forms q_t * P_t and its product with
// the state before the chunk, on the float32 matrix instruction.
//
// 1,608 tokens of eight requests, 28 heads: of 64 x 128 with a decay for each channel 140 us (scan 88, carry 16, join 36), of 128 x 128
// with one for each head 206 (135, 29, 40).  With a scan from cleared rows, q_t * P_t and the products through memory, and these put
// back into token order by a kernel of their own, they were 208 and 263.
// ---------------------------------------------------------------------------------------

// grid (chunks, H, parts of the value channels), 256 threads: rows begin .. end - 1 of `out` [N, H * vdim] = (q_t * P_t)^T S', S' the chunk's row of `states`.
// A thread sums the logarithms of its channel's decays over a part of the chunk's tokens, learns through LDS what the parts before
// it add up to, and walks its tokens again to leave q_t * P_t in LDS; then a wave takes 32 value channels at a time.  What bounds it is
// latency: eight tokens' loads are asked for at once (44 us one by one, 36 so).  Registers leave three blocks a compute unit up to 128 key
// channels (122 to 128, and 32 of the sums; for a fourth block the compiler spills), beyond it is LDS: two blocks of 256 channels, one of 512.
// (Chunks of more tokens than LDS holds are taken LA_JOIN at a time.)  Where chunks and heads are few, up to 128 value channels go to a block
// of their own each, which forms q_t * P_t anew (4 chunks, 4 heads of 256 x 512, one decay for each head: 70 us of the
// whole scan, by one block 118).
#define LA_JOIN 64
#define LA_SPAN (LA_DIM <= 256 ? LA_DIM : 256)       // channels that threads stand side by side for
#define LA_PARTS (256 / LA_SPAN < 16 ? 256 / LA_SPAN : 16)
#define LA_WIDE ((LA_DIM + 15) / 16 * 16)

typedef float la_f32x4 __attribute__((ext_vector_type(4)));

template <typename TP, int MODE>
__global__ __launch_bounds__(256) void la_join_kernel(const TP* __restrict__ proj, long long proj_stride, long long q_off,
                                                      const float* __restrict__ head_decay, const float* __restrict__ z, long long z_stride,
                                                      float inv_tau, const float* __restrict__ lower, const float* __restrict__ zbias,
                                                      const int* __restrict__ chunk_cu, const float* __restrict__ states,
                                                      float* __restrict__ out, int H, int vdim, int act, float q_scale, int before) {
  __shared__ float part_sum[LA_PARTS][LA_SPAN], upto[LA_DIM];      // upto: logarithms of all decays so far
  // four values of padding: the 16 rows of an operand read lie in different banks
  __shared__ __attribute__((aligned(16))) float qp[LA_JOIN][LA_WIDE + 4];
  const int chunk = blockIdx.x, head = blockIdx.y, part = threadIdx.x / LA_SPAN;
  const bool works = part < LA_PARTS;      // (a few threads are left over where LA_SPAN does not divide 256)
  if (LA_WIDE > LA_DIM)
    for (int i = threadIdx.x; i < LA_JOIN * 16; i += 256)
      if (LA_WIDE - 16 + i % 16 >= LA_DIM) qp[i / 16][LA_WIDE - 16 + i % 16] = 0.f;
  for (int i = threadIdx.x; i < LA_DIM; i += 256) upto[i] = 0.f;
  const int chunk_end = chunk_cu[chunk + 1];
  for (int begin = chunk_cu[chunk]; begin < chunk_end; begin += LA_JOIN) {
    const int end = min(begin + LA_JOIN, chunk_end);
    const int per = (end - begin + LA_PARTS - 1) / LA_PARTS;
    const int lo = works ? min(begin + part * per, end) : end, hi = min(lo + per, end);
    for (int d0 = 0; d0 < LA_DIM; d0 += LA_SPAN) {
      const int d = d0 + (int)threadIdx.x % LA_SPAN;
      const bool exists = d < LA_DIM;
      const float fixed_log = MODE != LA_HEAD ? 0.f : logf(head_decay[head]);
      const float my_lower = MODE == LA_FORGET && exists ? lower[head * LA_DIM + d] : 0.f;
      const float my_bias = ((MODE == LA_FORGET || MODE == LA_EXP) && zbias && exists) ? zbias[head * LA_DIM + d] : 0.f;
      auto log_decay = [&](float zz) {
        if (MODE == LA_HEAD) return fixed_log;
        if (MODE == LA_EXP) return -expf(zz + my_bias);
        if (MODE == LA_FORGET) return log1pf(-la_forget_key(zz + my_bias, my_lower));
        return la_log_decay(zz, inv_tau);
      };
      __syncthreads();      // the part sums and the rows before have been read
      float mine = 0.f;
      if (exists)
        for (int t0 = lo; t0 < hi; t0 += 8) {
          float zz[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) zz[i] = MODE == LA_HEAD ? 0.f : z[(size_t)min(t0 + i, hi - 1) * z_stride + (size_t)head * LA_DIM + d];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            if (t0 + i >= hi) break;
            const float lg = log_decay(zz[i]);
            mine += lg;
            qp[t0 + i - begin][d] = lg;
          }
        }
      if (works) part_sum[part][d - d0] = mine;
      __syncthreads();
      float acc = exists ? upto[d] : 0.f;     // log of the running product, from the chunk's first token on
      if (works && exists) {
        for (int p = 0; p < part; ++p) acc += part_sum[p][d - d0];
        for (int t0 = lo; t0 < hi; t0 += 8) {
          float qq[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) qq[i] = ldf<TP>(proj + (size_t)min(t0 + i, hi - 1) * proj_stride + q_off + (size_t)head * LA_DIM + d);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            if (t0 + i >= hi) break;
            const float earlier = acc;        // the decays before the token
            acc += qp[t0 + i - begin][d];
            qp[t0 + i - begin][d] = la_act(qq[i], act & 1) * q_scale * expf(before ? earlier : acc);
          }
        }
      }
      __syncthreads();
      if (exists && part == LA_PARTS - 1) upto[d] = acc;
    }
    __syncthreads();
    // v_mfma_f32_16x16x4_f32: A 16 tokens x 4 channels, B 4 channels x 16 values.  Lane group g holds channels 4 g .. 4 g + 3 of 16 and
    // gives one of them to each of four instructions.
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15, tiles = (end - begin + 15) / 16;
    const float* S = states + ((size_t)chunk * H + head) * LA_DIM * vdim;
    for (int c0 = (blockIdx.z * 4 + wave) * 32; c0 < vdim; c0 += 128 * gridDim.z) {
      la_f32x4 sum[4][2];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int c = 0; c < 2; ++c) sum[t][c] = la_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
      for (int k = 0; k < LA_WIDE; k += 16) {
        float b[4][2];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const int row = k + 4 * g + j, col = c0 + 16 * c + r;
            b[j][c] = row < LA_DIM && col < vdim ? S[(size_t)row * vdim + col] : 0.f;
          }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if (t >= tiles) break;
          const float4 a = *reinterpret_cast<const float4*>(&qp[16 * t + r][k + 4 * g]);
          const float av[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int c = 0; c < 2; ++c) sum[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[j], b[j][c], sum[t][c], 0, 0, 0);
        }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const int col = c0 + 16 * c + r;
          if (col >= vdim) continue;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int tok = begin + 16 * t + 4 * g + j;
            if (tok < end) out[((size_t)tok * H + head) * vdim + col] = sum[t][c][j];
          }
        }
    }
  }
}

// One thread per element of a head's state: for the request's chunks in order, scratch[c] (the chunk's
// U) is replaced by the state before the chunk, and the request's slot gets the state after its last.
__global__ void la_carry_kernel(float* __restrict__ scratch, const float* __restrict__ last, float* __restrict__ state,
                                const int* __restrict__ req_first, const int* __restrict__ req_slots, int H, int vdim) {
  const int req = blockIdx.y;
  const long long per_slot = (long long)H * LA_DIM * vdim;
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= per_slot) return;
  const long long hd = e / vdim;      // head * LA_DIM + d
  float* mine = state + (size_t)req_slots[req] * per_slot + e;
  float S = *mine;
  for (int c = req_first[req]; c < req_first[req + 1]; ++c) {
    float* u = scratch + (size_t)c * per_slot + e;
    const float before = S;
    S = last[(size_t)c * H * LA_DIM + hd] * S + *u;
    *u = before;
  }
  *mine = S;
}

// The last of the kernels for chunks (see above); before != 0: q_t meets the decays of the tokens before it only (outputs formed before the
// state moves on).
extern "C" int qvl_la_join(const void* proj, long long proj_stride, long long q_off, int proj_dtype, const void* head_decay, const void* z,
                           long long z_stride, float inv_tau, const void* lower, const void* zbias, int exp_decay, int before,
                           const void* chunk_cu, const void* states, void* out, int chunks, int H, int dim, int vdim, int act,
                           float q_scale, int cus, hipStream_t stream) {
  if (chunks <= 0) return QVL_OK;
  if (dim != LA_DIM || H <= 0 || vdim <= 0 || (!head_decay && !z) || (lower && !z) || (exp_decay && (lower || !z)))
    return QVL_ERR_SHAPE;
  if (H > 65535) return QVL_ERR_LIMIT;
  const long long room = 2ll * cus / ((long long)chunks * H), all = (vdim + 127) / 128;
  const int parts = (int)(room < 1 ? 1 : room < all ? room : all);
#define LAUNCH(TP, MODE)                                                                                                     \
  hipLaunchKernelGGL((la_join_kernel<TP, MODE>), dim3(chunks, H, parts), dim3(256), 0, stream, (const TP*)proj, proj_stride, q_off,  \
                     (const float*)head_decay, (const float*)z, z_stride, inv_tau, (const float*)lower, (const float*)zbias,  \
                     (const int*)chunk_cu, (const float*)states, (float*)out, H, vdim, act, q_scale, before)
#define BY_MODE(TP) { if (exp_decay) LAUNCH(TP, LA_EXP); else if (lower) LAUNCH(TP, LA_FORGET); else if (z) LAUNCH(TP, LA_CHANNEL); else LAUNCH(TP, LA_HEAD); }
  if (proj_dtype == 0) BY_MODE(float)
  else if (proj_dtype == 1) BY_MODE(bf16_t)
  else return QVL_ERR_DTYPE;
#undef BY_MODE
#undef LAUNCH
  return qvl_launch_status();
}

extern "C" int qvl_la_carry(void* scratch, const void* last, void* state, const void* req_first, const void* req_slots,
                            int R, int H, int dim, int vdim, hipStream_t stream) {
  if (R <= 0) return QVL_OK;
  if (dim != LA_DIM || H <= 0 || vdim <= 0) return QVL_ERR_SHAPE;
  if (R > 65535) return QVL_ERR_LIMIT;
  const long long per_slot = (long long)H * LA_DIM * vdim;
  hipLaunchKernelGGL(la_carry_kernel, dim3((unsigned)((per_slot + 255) / 256), R), dim3(256), 0, stream, (float*)scratch,
                     (const float*)last, (float*)state, (const int*)req_first, (const int*)req_slots, H, vdim);
  return qvl_launch_status();
}

extern "C" int qvl_la_key_size() { return LA_DIM; }

// Value channels of a lane in the scan of chunks, for `pairs` of (full) chunks and heads.  Two where one would take the blocks in more than one round
// and two in one: what a round takes is a block's way through its 64 tokens, longer with two channels.  16 heads, two and one: of 64 x 128
// with a decay for each channel 512 pairs 114 us and 96, 640 121 and 139, 1,504 239 and 243; of 128 x 128 with one for each head 512 135 and 115, 640
// 147 and 174, 1,504 320 and 304; of 256 x 256, 8 heads, 256 pairs 290 and 366 (one decay for each head 221 and 181), 320 480 and 407.
#define LA_TWO_DIM 256      // beyond, the state of two channels does not fit the registers
#define LA_TWO (LA_DIM <= LA_TWO_DIM ? 2 : 1)
template <typename TP, int MODE, bool BONUS, int COLS>
static int la_blocks_a_unit() {
  static std::atomic<int> known{0};
  int n = known.load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, la_scan_kernel<TP, MODE, 1, BONUS, COLS, true>, LA_THREADS, 0) != hipSuccess || n < 1) {
      (void)hipGetLastError();
      n = 1;
    }
    known.store(n, std::memory_order_relaxed);
  }
  return n;
}

extern "C" int qvl_la_chunk_columns(int proj_dtype, int has_z, int has_lower, int exp_decay, int has_bonus, long long pairs, int vdim, int cus) {
  if (vdim <= 64 || LA_DIM > LA_TWO_DIM || pairs <= 0) return 1;
  const long long one = pairs * ((vdim + 63) / 64), two = pairs * ((vdim + 127) / 128);
#define TWO_PAYS(TP, MODE, BONUS) \
  (one > (long long)cus * la_blocks_a_unit<TP, MODE, BONUS, 1>() && two <= (long long)cus * la_blocks_a_unit<TP, MODE, BONUS, LA_TWO>())
#define BY_MODE(TP)                                          \
  (exp_decay && has_bonus ? TWO_PAYS(TP, LA_EXP, true)       \
   : exp_decay            ? TWO_PAYS(TP, LA_EXP, false)      \
   : has_lower            ? TWO_PAYS(TP, LA_FORGET, false)   \
   : has_z                ? TWO_PAYS(TP, LA_CHANNEL, false)  \
                          : TWO_PAYS(TP, LA_HEAD, false))
  return (proj_dtype == 1 ? BY_MODE(bf16_t) : BY_MODE(float)) ? 2 : 1;
#undef BY_MODE
#undef TWO_PAYS
}

// proj: rows of `proj_stride` values holding q (H * LA_DIM columns from q_off), k (from k_off) and v
// (H * vdim columns from v_off).  head_decay [H] float32, or z float32 rows (H * LA_DIM columns) with
// inv_tau, or z with lower (and zbias, which may be null) float32 [H * LA_DIM]: the floored forget gate, whose
// complement is the key (k_off is not read), or z with exp_decay (and zbias or null): exp(-exp(z + zbias)), with which
// a bonus float32 [H * LA_DIM] may come.  state [slots, H, LA_DIM, vdim] float32; cu_q [R + 1], req_slots [R]; out float32
// [groups, N, H * vdim] (groups 1, 2, 4 or 8 with LA_DIM a multiple of 4 * groups), slabs `out_slab` apart.
extern "C" int qvl_la_scan(const void* proj, long long proj_stride, long long q_off, long long k_off, long long v_off,
                           int proj_dtype, const void* head_decay, const void* z, long long z_stride, float inv_tau,
                           const void* lower, const void* zbias, int exp_decay, const void* bonus, void* state, const void* cu_q, const void* req_slots, void* out, long long out_slab, int groups, int columns, void* last, int R,
                           int H, int dim, int vdim, int act, float q_scale, hipStream_t stream) {
  if (R <= 0) return QVL_OK;
  if (dim != LA_DIM || H <= 0 || vdim <= 0 || (!head_decay && !z) || (lower && !z) ||
      (exp_decay && (lower || !z)))
    return QVL_ERR_SHAPE;
  if (bonus && !exp_decay) return QVL_ERR_SHAPE;
  if (groups != 1 && groups != 2 && groups != 4 && groups != 8) return QVL_ERR_SHAPE;
  if (LA_DIM % (LA_WAVES * groups)) return QVL_ERR_SHAPE;
  if (H > 65535 || R > 65535) return QVL_ERR_LIMIT;
  if (columns != 1 && (columns != 2 || !last || groups != 1 || LA_DIM > LA_TWO_DIM)) return QVL_ERR_SHAPE;
  const dim3 grid((vdim + 64 * columns - 1) / (64 * columns) * groups, H, R);
#define RUN(TP, CH, G, BONUS, COLS, CHUNK)                                                                                    \
  hipLaunchKernelGGL((la_scan_kernel<TP, CH, G, BONUS, COLS, CHUNK>), grid, dim3(LA_THREADS), 0, stream, (const TP*)proj,     \
                     proj_stride, q_off, k_off, v_off, (const float*)head_decay, (const float*)z, z_stride, inv_tau,          \
                     (const float*)lower, (const float*)zbias, (const float*)bonus, (float*)state, (const int*)cu_q,          \
                     (const int*)req_slots, (float*)out, out_slab, (float*)last, H, vdim, act, q_scale)
#define LAUNCH(TP, CH, G, BONUS)                          \
  do {                                                    \
    if (columns == 2) RUN(TP, CH, 1, BONUS, LA_TWO, true); \
    else if (last) RUN(TP, CH, G, BONUS, 1, true);        \
    else RUN(TP, CH, G, BONUS, 1, false);                 \
  } while (0)
// (only numbers of groups that the key size has are compiled: a size that is met for the first time, 24, takes 13 s)
#define GROUPS_2(TP, CH, BONUS)
#define GROUPS_4(TP, CH, BONUS)
#define GROUPS_8(TP, CH, BONUS)
#if LA_DIM % (LA_WAVES * 2) == 0
#undef GROUPS_2
#define GROUPS_2(TP, CH, BONUS) case 2: LAUNCH(TP, CH, 2, BONUS); break;
#endif
#if LA_DIM % (LA_WAVES * 4) == 0
#undef GROUPS_4
#define GROUPS_4(TP, CH, BONUS) case 4: LAUNCH(TP, CH, 4, BONUS); break;
#endif
#if LA_DIM % (LA_WAVES * 8) == 0
#undef GROUPS_8
#define GROUPS_8(TP, CH, BONUS) case 8: LAUNCH(TP, CH, 8, BONUS); break;
#endif
#define BY_GROUPS(TP, CH, BONUS)                  \
  switch (groups) {                               \
    case 1: LAUNCH(TP, CH, 1, BONUS); break;      \
    GROUPS_2(TP, CH, BONUS)                       \
    GROUPS_4(TP, CH, BONUS)                       \
    GROUPS_8(TP, CH, BONUS)                       \
    default: return QVL_ERR_SHAPE;                \
  }
#define BY_MODE(TP)                                                                                                 \
  {                                                                                                                 \
    if (exp_decay && bonus) { BY_GROUPS(TP, LA_EXP, true) }                                                         \
    else if (exp_decay) { BY_GROUPS(TP, LA_EXP, false) }                                                            \
    else if (lower) { BY_GROUPS(TP, LA_FORGET, false) }                                                                         \
    else if (z) { BY_GROUPS(TP, LA_CHANNEL, false) }                                                                       \
    else { BY_GROUPS(TP, LA_HEAD, false) }                                                                                 \
  }
  if (proj_dtype == 0) BY_MODE(float)
  else if (proj_dtype == 1) BY_MODE(bf16_t)
  else return QVL_ERR_DTYPE;
#undef BY_MODE
#undef BY_GROUPS
#undef GROUPS_8
#undef GROUPS_4
#undef GROUPS_2
#undef LAUNCH
#undef RUN
  return qvl_launch_status();
}
