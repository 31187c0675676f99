// Products with at most 64 rows (a decode step's projections): out[M, N] = X[M, K] . W[N, K]^T,
// bfloat16 operands, float32 accumulation.  The step is bound by reading W once from HBM, so W
// is the streamed operand and everything around the product is folded into this kernel, because
// between two products a short kernel of its own costs more than its arithmetic (its code and
// data have just been flushed from the caches by the weights).
//
// A block of 8 waves owns row tiles of W (tile, tile + gridDim.x, ...).  A tile has `rows` <= 16
// rows of W (= outputs); the host picks `rows` so that the tiles divide evenly among the compute
// units (3584 outputs on 256 units: 256 tiles of 14 rather than 224 of 16); the matrix-core tile's
// other rows are read from one that exists and not stored.
// Wave w covers the 32 RK values of K from 32 RK w on (RK = 16: 512; a second build with RK = 8 serves
// inner sizes up to 2,048, where with 512 values a wave half the waves would have none), as the A operand (W rows)
// and B operand (X rows) of v_mfma_f32_16x16x32_bf16; the waves' sums meet in LDS and are added in wave order.
// Up to 16 rows of X are one column tile of the matrix instruction, 17 to 32 rows two (MT = 2): every W fragment is
// multiplied with all of them.  X stays in the waves' registers for all of the block's tiles if K fits one pass
// (K <= 256 RK); a longer K is walked in passes, X read again for each.  More rows are spread over
// teams of blocks (below).
//
// How W comes in decides the speed.  A load into registers in the instruction's own layout covers 16 rows of 64 bytes:
// half a cache line a row, and each line is asked for twice (gate|up of the 7B decoder, 271.6 MB, 8 rows: 51 us = 5.3
// TB/s; marked as read once, 54.7, the line's second half fetched anew).  So a wave brings its own columns of a tile into LDS with loads
// that put their 16 bytes there directly, 256 bytes of 4 rows at a time, whole lines, marked as read once, and reads the
// operands back from there (that product with its norm 49.9 us; without the norm 46, every block reads and norms all rows
// first: with K beyond 2,048 products of so many outputs go to gemm_rows.hip, 43 and a norm kernel of 5).  Per call in a decode step: 7B
// decoder, 8 rows, the down product's ranges 24.8 us = 5.5 TB/s, q|k|v 12.4, o 8.2; 3B decoder, 1 row, gate|up with its norm 20.6 us
// = 4.4 TB/s.  A plain read of much memory reaches 7.3 TB/s.  A wave waits for its own loads only (no
// barrier but the one of the merge), four units of 128 columns go round, each asked for again the moment it has been
// read, so that the next tile is on its way while a tile's sums are merged.
//
// What is folded in:
//   prologue  PRO_NORM      X = rmsnorm(H) * w, from the float32 residual H (statistics in float32,
//                           each wave sums its own columns, the block adds the waves in order)
//   epilogue  EPI_RESIDUAL  out += product, out being the float32 residual
//             EPI_SWIGLU    W's rows come in groups of 8 gate rows, 8 up rows; out[M, N/2] =
//                           act(gate) * up, in bfloat16 (act: silu, or the tanh form of gelu)
//             EPI_ROPE      W is the stacked query | key | value projection.  A tile of a query or
//                           key head takes 8 channels and the 8 channels they are rotated with
//                           (half a head further), so the rotation happens here; queries are
//                           written out, keys and values go straight into their page slots
//   ranges of K             out[c] = the sums over range c of K (qvl_gemm_split below), for products whose result
//                           joins the residual sum: the norm that follows adds the slabs in order
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

typedef __amdgpu_buffer_rsrc_t rsrc_t;
// An offset no buffer reaches: what is loaded there is zero.  Buffers stay below it (the host checks).
#define PAST_END 0xffffff00u
#define BUFFER_LIMIT 0xffffff00ull

__device__ __forceinline__ rsrc_t buffer_of(const void* p, unsigned long long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, p ? (int)(uint32_t)bytes : 0, 0x00020000);
}
// `fixed` is a compile-time part of the offset: it rides in the instruction, the lanes' part in one register.
__device__ __forceinline__ u32x4_t buffer_load16(rsrc_t r, uint32_t byte_offset, int fixed = 0) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, byte_offset, fixed, 0);
}
__device__ __forceinline__ float buffer_load_f32(rsrc_t r, uint32_t byte_offset) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, byte_offset, 0, 0));
}

#define HOLD_ORDER() __builtin_amdgcn_sched_barrier(0)   // nothing is scheduled across this point

#define RW 8    // waves per block
#ifndef RK
#define RK 16   // 32-wide K steps per wave and pass (the host loads a build with 8 for inner sizes up to 2,048: all waves then have columns)
#endif
#define PASS_K (RW * RK * 32)
#define TWO_TILE_K (PASS_K - 256 < 3840 ? PASS_K : 3840)   // the longest K with 17 to 32 rows in one pass (4,096 would fit; the callers' rule is older and no decoder's width lies between)
#define UNIT 4                  // K steps of a unit: 128 columns, 256 bytes a row
#define UNIT_BYTES (16 * 256)
#define UNIT_LOADS 4            // loads of 1 KB: 4 rows each
#define UNITS (RK / UNIT)       // of a wave's columns

enum { PRO_PLAIN = 0, PRO_NORM = 1 };
enum { EPI_STORE = 0, EPI_RESIDUAL = 1, EPI_SWIGLU = 2, EPI_ROPE = 3 };
#define ACT_RELU2 2

struct ResidentArgs {
  const bf16_t* X;       // PRO_PLAIN: [M, K]
  int ldx;
  const float* H;        // PRO_NORM: float32 [M, K]
  int ldh;
  const float* norm_w;   // PRO_NORM: [K]
  float eps;
  const bf16_t* W;       // [N, K]
  int ldw;
  const float* bias;     // [N] or null (EPI_STORE and EPI_RESIDUAL)
  void* out;
  int ldo;
  int M, N, K, ntiles;
  int rows;              // rows of W per tile, 1..16 (16 with EPI_SWIGLU and EPI_ROPE)
  // More rows of X than a block carries: `groups` blocks form a team that walks the same tiles of W,
  // block g of the team with rows g * (16 MT) ... of X.  The blocks of a team run on the same XCD
  // at the same pace, so the tile that the first of them brings in from HBM the others find in
  // that XCD's L2 (or in the memory-side cache): W leaves HBM once.
  int groups;
  // EPI_ROPE: W rows are nq query heads, nkv key heads, nkv value heads of hd channels each
  // (hd a multiple of 16, rotation over the whole head in pairs (f, f + hd/2))
  const float* cs;       // [M, hd/2, 2] cosine and sine of each token's angle at each frequency
  const int* slot;       // [M] flat slot of each token in the cache (page * ps + offset), -1: none
  bf16_t* q_out;         // [M, nq hd]
  bf16_t* kc;            // [pages, nkv, ps, hd]
  bf16_t* vc;            // [pages, nkv, hd, ps]
  int nq, nkv, hd, ps;
  int pair_tiles;        // tiles of query and key heads (16 rows each); value tiles of `rows` rows follow
  // EPI_SWIGLU: the first whole_tiles tiles are whole groups of 8 + 8 rows; each group after them
  // is cut into `parts` tiles of `pairs` gate rows and their up rows, so that the last round of
  // tiles is as even as the rounds before it
  int whole_tiles, parts, pairs;
  int gelu;              // EPI_SWIGLU: 1: the activation is the tanh form of gelu; EPI_STORE: ACT_RELU2: max(product, 0)^2 is stored
  // Several products of the same sizes side by side (EPI_STORE, one block a team): product i has the blocks
  // i * stack_blocks .. and its operands and result lie i strides further on (in elements)
  int stack_blocks;      // 0: one product
  long long stack_x, stack_w, stack_o;
  int all_k;             // ranges of one K: item i has the columns i * stack_x .. of all_k (0: every item has K columns)
};

__device__ __forceinline__ bf16x8_t load8(const bf16_t* p) {
  return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(p));
}
__device__ __forceinline__ bf16x8_t zero8() {
  u32x4_t z = {0u, 0u, 0u, 0u};
  return __builtin_bit_cast(bf16x8_t, z);
}
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  bf16x2_t v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}

// Lane l of the wave puts its 16 bytes at M0 + 16 l of LDS.  `once`: the lines are read by this block alone and need not stay in the caches.
__device__ __forceinline__ void fetch16_to_lds(const void* base, uint32_t lane_bytes, uint32_t lds_at, bool once) {
  if (once)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(lane_bytes), "s"(base), "s"(lds_at)
                 : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_bytes), "s"(base), "s"(lds_at)
                 : "memory", "m0");
}
// Wait until at most N of this wave's loads are outstanding (they finish in order).
template <int N>
__device__ __forceinline__ void wait_loads() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
}
__device__ __forceinline__ void wait_units(int younger) {   // all but the `younger` units asked for last have come
  if (younger >= 3) wait_loads<3 * UNIT_LOADS>();
  else if (younger == 2) wait_loads<2 * UNIT_LOADS>();
  else if (younger == 1) wait_loads<UNIT_LOADS>();
  else wait_loads<0>();
}
// A barrier that leaves loads from memory in flight.
__device__ __forceinline__ void meet() {
  __builtin_amdgcn_s_waitcnt(0xc07f);      // this wave's accesses to LDS are done
  HOLD_ORDER();
  __builtin_amdgcn_s_barrier();
  HOLD_ORDER();
}

template <typename TO, int PRO, int EPI, bool ONE_PASS, int MT>
__global__ __launch_bounds__(64 * RW) void gemm_resident_kernel(ResidentArgs p) {
  constexpr int COLS = 16 * MT;   // rows of X the block carries
  constexpr int RING = 4;
  // MT = 1: two buffers, a tile's sums are read while the next tile's are written; else one, and a second barrier.
  // The norm weights borrow the sums' place before the first tile.
  constexpr int RED = MT == 1 ? 2 : 1;
  static_assert(PRO != PRO_NORM || RK * 32 <= RED * 16 * COLS, "the norm weights fit");
  __shared__ __attribute__((aligned(16))) char ring[RW][RING][UNIT_BYTES];
  __shared__ __attribute__((aligned(16))) float red[RED][RW][16 * COLS];
  __shared__ float rowsq[RW][16];
  float (*gains)[RK * 32] = reinterpret_cast<float (*)[RK * 32]>(&red[0][0][0]);  // norm weights of each wave's columns
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, lg = lane >> 4, r = lane & 15;
  const int k_wave = wave * RK * 32;           // the wave's first column within a pass
  const int k_lane = k_wave + 8 * lg;          // first K index of this lane within a pass
  int block = blockIdx.x, blocks = gridDim.x;
  if (EPI == EPI_STORE && p.stack_blocks > 0) {
    const int item = block / p.stack_blocks;
    block -= item * p.stack_blocks;
    blocks = p.stack_blocks;
    p.X += item * p.stack_x;
    p.W += item * p.stack_w;
    p.out = reinterpret_cast<TO*>(p.out) + item * p.stack_o;
    if (p.all_k) p.K = min(p.K, p.all_k - item * (int)p.stack_x);
  }
  // how many of this lane's 32-wide steps of the pass that starts at k0 begin inside K (K is a
  // multiple of 8, as is every lane's first index: a step lies inside K or outside)
  auto steps_inside = [&](int k0) { return (p.K - k0 - k_lane + 31) >> 5; };
  // the same for the two halves of a lane's values under PRO_NORM, columns 4 lg .. and 16 + 4 lg .. of a step
  const int inside_lo = (p.K - k_wave - 4 * lg + 31) >> 5, inside_hi = (p.K - k_wave - 16 - 4 * lg + 31) >> 5;
  // how many units of the wave's columns of that pass hold any of K
  auto units_inside = [&](int k0) {
    const int n = (p.K - k0 - k_wave + 127) >> 7;
    return n < 0 ? 0 : (n < UNITS ? n : UNITS);
  };
  // what the kernel reads beside W, each behind a descriptor that knows its size (a null pointer: size 0): a lane that has
  // nothing to load asks past the end and gets zeros without traffic, so no load sits inside a branch
  const rsrc_t x_buf = buffer_of(p.X, ((unsigned long long)(p.M - 1) * p.ldx + p.K) * 2);
  const rsrc_t h_buf = buffer_of(p.H, ((unsigned long long)(p.M - 1) * p.ldh + p.K) * 4);
  const rsrc_t gain_buf = buffer_of(p.norm_w, (unsigned long long)p.K * 4);
  const rsrc_t bias_buf = buffer_of(p.bias, (unsigned long long)p.N * 4);
  const rsrc_t old_buf = buffer_of(EPI == EPI_RESIDUAL ? p.out : nullptr, ((unsigned long long)(p.M - 1) * p.ldo + p.N) * 4);
  const rsrc_t cs_buf = buffer_of(p.cs, (unsigned long long)p.M * p.hd * 4);
  const rsrc_t slot_buf = buffer_of(p.slot, (unsigned long long)p.M * 4);
  // Workgroups go to the XCDs in turn, so blocks b, b + 8, b + 16, ... share an XCD: consecutive
  // ones of them form a team.
  int team = block, teams = blocks, m0 = 0;   // m0: this block's first row of X
  if (p.groups > 1) {   // the grid is a multiple of 8 groups
    const int xcd_turn = blockIdx.x >> 3;
    team = (xcd_turn / p.groups) * 8 + (blockIdx.x & 7);
    teams = (int)(gridDim.x >> 3) / p.groups * 8;
    m0 = (xcd_turn % p.groups) * COLS;
  }
  const bool once = p.groups <= 1;            // nobody else reads the block's tiles of W
  // Teams take tiles in turn: with runs of neighbouring tiles instead, blocks would read a multiple of a power of two
  // of bytes apart (151,936 outputs of K 2,048: 114 us for 106).
  // the rows of a tile, and the row of W behind row i of a tile
  auto tile_rows = [&](int tile) { return (EPI == EPI_ROPE && tile < p.pair_tiles) ? 16 : p.rows; };
  auto w_row = [&](int tile, int i) {
    if (EPI == EPI_ROPE) {
      if (tile < p.pair_tiles) {  // 8 channels of a query or key head and the 8 they are rotated with
        const int tph = p.hd >> 4, head = tile / tph, sub = tile - head * tph;
        return head * p.hd + 8 * sub + (i & 7) + (i >> 3) * (p.hd >> 1);
      }
      return (p.nq + p.nkv) * p.hd + (tile - p.pair_tiles) * p.rows + i;   // value rows
    }
    if (EPI == EPI_SWIGLU && tile >= p.whole_tiles) {
      // a part of one of the last groups: `pairs` gate rows and the up rows that belong to them
      const int part = tile - p.whole_tiles, group = p.whole_tiles + part / p.parts, s = part % p.parts;
      return (i & 7) < p.pairs ? group * 16 + (i >> 3) * 8 + s * p.pairs + (i & 7) : -1;
    }
    return tile * p.rows + i;
  };

  // ---- the stream of W ------------------------------------------------------------------------
  // The wave's units in the order they are read: tile after tile, within a tile pass after pass, within a pass
  // its units.  Row rho of a unit lies at 256 rho; place s of it holds the row's 16-byte chunk s ^ rho, so that the 16
  // rows of an operand read touch all banks.  (ft, fp, fu): the unit asked for next.
  const int passes = ONE_PASS ? 1 : (p.K + PASS_K - 1) / PASS_K;
  int ft = team, fp = 0, fu = 0, f_units = units_inside(0), f_slot = 0, waiting = 0;   // waiting: units asked for and not read
  uint32_t from[UNIT_LOADS];
  auto set_from = [&](int tile) {
#pragma unroll
    for (int j = 0; j < UNIT_LOADS; ++j) {
      const int rho = 4 * j + lg;
      int row = w_row(tile, rho);
      if (rho >= tile_rows(tile) || row < 0 || row >= p.N) row = w_row(tile, 0);   // exists; its sums are stored once only
      from[j] = ((uint32_t)row * p.ldw + k_wave + 8 * (r ^ rho)) * 2;
    }
  };
  const uint32_t ring0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)&ring[wave][0][0];
  if (ft < p.ntiles) set_from(ft);
  auto ask = [&]() {       // the next unit, if there is one
    while (fu >= f_units) {
      if (ft >= p.ntiles) return;
      fu = 0;
      if (++fp >= passes) {
        fp = 0;
        ft += teams;
        if (ft < p.ntiles) set_from(ft);
      }
      f_units = units_inside(fp * PASS_K);
      if (ft >= p.ntiles || (passes == 1 && f_units == 0)) {
        ft = p.ntiles;
        f_units = fu = 0;
        return;
      }
    }
    if (ft >= p.ntiles) return;
    const int k = fp * PASS_K + fu * 128;
    // a chunk beyond K is read from the row's first columns of the unit: it is not multiplied
    const int left = p.K - k - k_wave;
#pragma unroll
    for (int j = 0; j < UNIT_LOADS; ++j) {
      const int c = 8 * (r ^ (4 * j + lg));
      const uint32_t at = from[j] + (uint32_t)k * 2 - (c < left ? 0u : (uint32_t)c * 2);
      fetch16_to_lds(p.W, at, ring0 + f_slot * UNIT_BYTES + j * 1024, once);
    }
    f_slot = f_slot + 1 == RING ? 0 : f_slot + 1;
    ++fu;
    ++waiting;
  };

  auto ask_first = [&] {
#pragma unroll
    for (int i = 0; i < RING; ++i) ask();
  };

  // ---- the X operand of one pass ------------------------------------------------------------
  // Column tile t holds rows 16 t .. 16 t + 15 of X.  again: another column tile's norm came before
  // (the norm weights are in LDS already, and the statistics' place may still be read).
  // first: the wave's first units are asked for right behind the rows.
  auto load_x = [&](int t, int k0, bf16x8_t* xb, bool again, bool first) {
    const int row = m0 + 16 * t + r;
    const bool m_ok = row < p.M;
    const int inside = steps_inside(k0);
    if (PRO == PRO_PLAIN) {
      const uint32_t at = m_ok ? ((uint32_t)row * p.ldx + k0 + k_lane) * 2 : PAST_END;
#pragma unroll
      for (int u = 0; u < RK; ++u)
        xb[u] = __builtin_bit_cast(bf16x8_t, buffer_load16(x_buf, u < inside ? at : PAST_END, u * 64));
      HOLD_ORDER();
      if (first) ask_first();
    } else {
      // rmsnorm of the float32 rows: this pass covers all of K (ONE_PASS), so the block's waves
      // hold whole rows between them.  A lane's eight values of a step are columns 4 lg .. and 16 + 4 lg .. (and W's
      // operand is read likewise): a load then covers 64 neighbouring bytes of a row, not four times 16 of 128.  A lane fetches neighbouring norm weights of its wave; they reach the lanes that
      // need them through LDS.
      const uint32_t at = m_ok ? ((uint32_t)row * p.ldh + k_wave + 4 * lg) * 4 : PAST_END;
      float4 v[RK][2];
#pragma unroll
      for (int u = 0; u < RK; ++u) {
        v[u][0] = __builtin_bit_cast(float4, buffer_load16(h_buf, u < inside_lo ? at : PAST_END, u * 128));
        v[u][1] = __builtin_bit_cast(float4, buffer_load16(h_buf, u < inside_hi ? at : PAST_END, u * 128 + 64));
      }
      constexpr int G = RK * 32 / 256;         // norm weights of the wave, 4 a lane, 256 a load
      float4 g4[G];
#pragma unroll
      for (int i = 0; i < G; ++i)
        g4[i] = __builtin_bit_cast(float4, buffer_load16(gain_buf, again ? PAST_END : (uint32_t)(k_wave + 256 * i + 4 * lane) * 4));
      HOLD_ORDER();
      if (first) ask_first();
      float ss = 0.f;
#pragma unroll
      for (int u = 0; u < RK; ++u)
        ss += v[u][0].x * v[u][0].x + v[u][0].y * v[u][0].y + v[u][0].z * v[u][0].z + v[u][0].w * v[u][0].w +
              v[u][1].x * v[u][1].x + v[u][1].y * v[u][1].y + v[u][1].z * v[u][1].z + v[u][1].w * v[u][1].w;
      ss += __shfl_xor(ss, 16, QVL_WAVE);
      ss += __shfl_xor(ss, 32, QVL_WAVE);
      if (again) meet();   // the other column tile's statistics have been read
      if (lg == 0) rowsq[wave][r] = ss;
      if (!again) {
#pragma unroll
        for (int i = 0; i < G; ++i) *reinterpret_cast<float4*>(&gains[wave][256 * i + 4 * lane]) = g4[i];
      }
      meet();
      float total = 0.f;
#pragma unroll
      for (int w = 0; w < RW; ++w) total += rowsq[w][r];
      const float rs = 1.0f / sqrtf(total / (float)p.K + p.eps);
#pragma unroll
      for (int u = 0; u < RK; ++u) {
        if (u < inside_lo) {
          const float4 g0 = *reinterpret_cast<const float4*>(&gains[wave][4 * lg + u * 32]);
          const float4 g1 = *reinterpret_cast<const float4*>(&gains[wave][4 * lg + u * 32 + 16]);
          u32x4_t o = {pack2((v[u][0].x * rs) * g0.x, (v[u][0].y * rs) * g0.y),
                       pack2((v[u][0].z * rs) * g0.z, (v[u][0].w * rs) * g0.w),
                       pack2((v[u][1].x * rs) * g1.x, (v[u][1].y * rs) * g1.y),
                       pack2((v[u][1].z * rs) * g1.z, (v[u][1].w * rs) * g1.w)};
          xb[u] = __builtin_bit_cast(bf16x8_t, o);
        } else {
          xb[u] = zero8();
        }
      }
    }
  };
  // What the epilogue of a tile reads from memory, for the element (m, nl) this thread finishes.
  struct Epi {
    float bias, old;
    float2 cs;
    int slot;
  };
  constexpr int EPT = (16 * COLS + 64 * RW - 1) / (64 * RW);   // elements of a tile a thread finishes
  auto epi_load = [&](int tile, int i) {
    Epi e;
    e.bias = e.old = 0.f;
    e.cs = float2{1.f, 0.f};
    e.slot = -1;
    if (EPI == EPI_SWIGLU || (EPI == EPI_STORE && !p.bias)) return e;
    const int el = threadIdx.x + 64 * RW * i;
    const int m = m0 + (el >> 4), nl = el & 15;
    const int n = tile < p.ntiles ? w_row(tile, nl) : -1;
    const bool live = el < 16 * COLS && m < p.M && nl < tile_rows(tile) && n >= 0 && n < p.N;
    e.bias = buffer_load_f32(bias_buf, live ? (uint32_t)n * 4 : PAST_END);
    if (EPI == EPI_RESIDUAL) e.old = buffer_load_f32(old_buf, live ? ((uint32_t)m * p.ldo + n) * 4 : PAST_END);
    if (EPI == EPI_ROPE) {
      const int head = live ? n / p.hd : 0, d = n - head * p.hd, half = p.hd >> 1;
      const bool turns = live && head < p.nq + p.nkv;
      const uint32_t at = turns ? ((uint32_t)m * half + (d < half ? d : d - half)) * 8 : PAST_END;
      e.cs = float2{buffer_load_f32(cs_buf, at), buffer_load_f32(cs_buf, at + 4)};
      if (!turns) e.cs = float2{1.f, 0.f};
      const int slot = __builtin_bit_cast(int, buffer_load_f32(slot_buf, (live && head >= p.nq) ? (uint32_t)m * 4 : PAST_END));
      e.slot = (live && head >= p.nq) ? slot : -1;
    }
    return e;
  };
  // ---- merge the waves' sums of one tile and write the result -----------------------------------
  // A wave's sums lie as [row of X][row of the tile]: a lane writes its four at once, and the
  // thread that finishes element e = 16 m + nl reads word e of every wave.
  // MT = 1, one barrier per tile: the sums go into the buffer that was read two tiles ago; whoever
  // reads it has passed the barrier of the tile in between since.
  // Else one buffer: a second barrier keeps the next tile's sums out until these are read.
  // The two halves of a wave's columns are summed apart: one chain over all of its columns rounds off a quarter more (8 x 3,584 x 3,584,
  // error against 64 bits 1.35e-7 of the result, so 1.0e-7; a pass of decode steps takes 0.2 to 0.4 per cent longer).
  constexpr int HALVES = UNITS > 1 ? 2 : 1;
  f32x4_t acc[HALVES][MT];
  int parity = 0;
  auto finish = [&](int tile, const Epi* epi) {
    float (*buf)[16 * COLS] = red[MT == 1 ? parity : 0];
    parity ^= 1;
#pragma unroll
    for (int t = 0; t < MT; ++t)
      *reinterpret_cast<f32x4_t*>(&buf[wave][(16 * t + r) * 16 + 4 * lg]) = HALVES > 1 ? acc[0][t] + acc[HALVES - 1][t] : acc[0][t];
    meet();
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int e = threadIdx.x + 64 * RW * i;
      if (e >= 16 * COLS) continue;
      const int m = m0 + (e >> 4), nl = e & 15, n = w_row(tile, nl);
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < RW; ++w) sum += buf[w][e];
      if (EPI == EPI_SWIGLU) {
        const float up = __shfl_down(sum, 8, QVL_WAVE);  // rows 8..15 of the tile are the up rows
        if (nl < 8 && m < p.M && n >= 0 && n < p.N) {
          bf16_t* o = reinterpret_cast<bf16_t*>(p.out);
          o[(size_t)m * p.ldo + (n >> 4) * 8 + (n & 7)] = f32_to_bf16(gate_act(sum, p.gelu) * up);
        }
      } else if (EPI == EPI_ROPE) {
        sum += epi[i].bias;
        const float other = __shfl_xor(sum, 8, QVL_WAVE);   // the channel this one is rotated with
        const int head = n / p.hd, d = n - head * p.hd;
        if (m < p.M && nl < tile_rows(tile) && n < p.N) {
          // values are stored as they are (turned by (1, 0), one that is not finite would take its neighbour along); rows 0..7 of
          // a rotated tile are the first halves
          const float val = head >= p.nq + p.nkv ? sum
                            : nl < 8 ? sum * epi[i].cs.x - other * epi[i].cs.y : sum * epi[i].cs.x + other * epi[i].cs.y;
          if (head < p.nq) {
            p.q_out[((size_t)m * p.nq + head) * p.hd + d] = f32_to_bf16(val);
          } else if (epi[i].slot >= 0) {
            const size_t page = (size_t)(epi[i].slot / p.ps), off = (size_t)(epi[i].slot % p.ps);
            if (head < p.nq + p.nkv)
              p.kc[((page * p.nkv + (head - p.nq)) * p.ps + off) * p.hd + d] = f32_to_bf16(val);
            else
              p.vc[((page * p.nkv + (head - p.nq - p.nkv)) * p.hd + d) * p.ps + off] = f32_to_bf16(val);
          }
        }
      } else if (m < p.M && nl < p.rows && n < p.N) {
        sum += epi[i].bias;
        if (EPI == EPI_STORE && p.gelu == ACT_RELU2) {
          sum = fmaxf(sum, 0.f);
          sum *= sum;
        }
        if (EPI == EPI_RESIDUAL) {
          float* o = reinterpret_cast<float*>(p.out);
          o[(size_t)m * p.ldo + n] = epi[i].old + sum;
        } else {
          stf<TO>(reinterpret_cast<TO*>(p.out) + (size_t)m * p.ldo + n, sum);
        }
      }
    }
    if (MT >= 2) meet();
  };

  bf16x8_t xb[MT][RK];
  auto load_all_x = [&](int k0, bool first) {
#pragma unroll
    for (int t = MT - 1; t >= 0; --t) load_x(t, k0, xb[t], t != MT - 1, first && t == MT - 1);
    // From here on the waits are counted: the compiler, which does not know of the units, would wait for the rows
    // behind units that are asked for later.
    wait_loads<0>();
    if (PRO == PRO_NORM) meet();   // the norm weights lie where the first tile's sums go
  };
  if (ONE_PASS) load_all_x(0, true);
  else ask_first();
  int slot = 0;
  for (int tile = team; tile < p.ntiles; tile += teams) {
    Epi e[EPT];
#pragma unroll
    for (int i = 0; i < EPT; ++i) e[i] = epi_load(tile, i);
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int h = 0; h < HALVES; ++h) acc[h][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int pass = 0; pass < passes; ++pass) {
      const int k0 = pass * PASS_K;
      if (!ONE_PASS) load_all_x(k0, false);
      const int inside = steps_inside(k0), units = units_inside(k0);
#pragma unroll
      for (int u = 0; u < UNITS; ++u) {
        if (u >= units) break;
        HOLD_ORDER();
        wait_units(waiting - 1);
        HOLD_ORDER();
        const char* at = &ring[wave][slot][r * 256];
        bf16x8_t a[UNIT];
#pragma unroll
        for (int i = 0; i < UNIT; ++i) {
          if (PRO == PRO_NORM) {
            const int c = 4 * i + (lg >> 1), half = (lg & 1) * 8;
            const uint2 lo = *reinterpret_cast<const uint2*>(at + ((c ^ r) << 4) + half);
            const uint2 hi = *reinterpret_cast<const uint2*>(at + (((c + 2) ^ r) << 4) + half);
            a[i] = __builtin_bit_cast(bf16x8_t, u32x4_t{lo.x, lo.y, hi.x, hi.y});
          } else {
            a[i] = *reinterpret_cast<const bf16x8_t*>(at + (((4 * i + lg) ^ r) << 4));
          }
        }
        if (p.K - k0 - k_wave < 128 * (u + 1)) {     // the unit in which K ends: what lies beyond is no part of the sum
#pragma unroll
          for (int i = 0; i < UNIT; ++i) {
            if (PRO == PRO_NORM) {
              u32x4_t v = __builtin_bit_cast(u32x4_t, a[i]);
              if (u * UNIT + i >= inside_lo) v.x = v.y = 0u;
              if (u * UNIT + i >= inside_hi) v.z = v.w = 0u;
              a[i] = __builtin_bit_cast(bf16x8_t, v);
            } else if (u * UNIT + i >= inside) {
              a[i] = zero8();
            }
          }
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);          // the unit has been read: its place may be filled again
        HOLD_ORDER();
        slot = slot + 1 == RING ? 0 : slot + 1;
        --waiting;
        ask();
        HOLD_ORDER();
#pragma unroll
        for (int i = 0; i < UNIT; ++i)
#pragma unroll
          for (int t = 0; t < MT; ++t) {
            f32x4_t& sum = acc[u * HALVES / UNITS][t];
            sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], xb[t][u * UNIT + i], sum, 0, 0, 0);
          }
      }
    }
    finish(tile, e);
  }
  wait_loads<0>();       // nothing may land in LDS that is no longer this block's
}

// How M rows are carried: column tiles per block (MT), blocks per team (groups), and whether X stays
// in the block for all its tiles (one pass over K).  Up to 32 rows one block carries them all.
// More rows, or 17 to 32 rows with a norm and a K too long for one pass, are
// spread over the blocks of a team; a device with too few compute units for teams (fewer than 8
// per group) is refused (mt = 0).
struct Plan {
  int mt, groups;
  bool one_pass;
};
static Plan plan_for(int M, int K, bool norm, int blocks) {
  if (M <= 16) return Plan{1, 1, K <= PASS_K};
  const bool two_fit = K <= TWO_TILE_K;
  if (M <= 32 && two_fit) return Plan{2, 1, true};
  if (two_fit && blocks >= 8 * ((M + 31) / 32)) return Plan{2, (M + 31) / 32, true};
  const int singles = (M + 15) / 16;
  if ((M > 32 || norm) && blocks >= 8 * singles) return Plan{1, singles, K <= PASS_K};
  if (M <= 32) return Plan{2, 1, false};
  return Plan{0, 1, false};
}
// the number of teams the plan's grid has: what the tiles are divided among
static int plan_teams(const Plan& pl, int blocks) { return pl.groups == 1 ? blocks : blocks / (8 * pl.groups) * 8; }

template <typename TO, int PRO, int EPI>
static int launch(ResidentArgs p, const Plan& pl, int blocks, hipStream_t stream) {
  const int teams = plan_teams(pl, blocks);
  p.groups = pl.groups;
  const dim3 grid(pl.groups == 1 ? (teams < p.ntiles ? teams : p.ntiles) : teams * pl.groups), block(64 * RW);
#define QVL_GO(ONE, MT) hipLaunchKernelGGL((gemm_resident_kernel<TO, PRO, EPI, ONE, MT>), grid, block, 0, stream, p)
  if (PRO == PRO_NORM && !pl.one_pass) return QVL_ERR_LIMIT;   // a norm is only folded into a single pass
  if (pl.mt == 1) {
    if (pl.one_pass) QVL_GO(true, 1);
    else if constexpr (PRO == PRO_PLAIN) QVL_GO(false, 1);
  } else if (pl.mt == 2) {
    if (pl.one_pass) QVL_GO(true, 2);
    else if constexpr (PRO == PRO_PLAIN) QVL_GO(false, 2);
  } else {
    return QVL_ERR_LIMIT;
  }
#undef QVL_GO
  return qvl_launch_status();
}

// Whether qvl_gemm_resident(_rope) forms the norm of M rows of width K itself on a device with this
// many compute units.
extern "C" int qvl_gemm_resident_folds_norm(int M, int K, int blocks) {
  if (M <= 0 || M > 64 || K <= 0 || K > PASS_K || blocks <= 0) return 0;
  const Plan pl = plan_for(M, K, true, blocks);
  return pl.one_pass && pl.mt <= 2;
}

// Whether every operand lies within what a buffer descriptor and a 32-bit byte offset reach.
static bool fits_descriptors(long long M, long long N, long long K, long long ldw, long long ldx, long long ldh,
                             long long ldo) {
  const unsigned long long w = ((N - 1) * ldw + K) * 2ull, x = ((M - 1) * ldx + K) * 2ull,
                           h = ((M - 1) * ldh + K) * 4ull, o = ((M - 1) * ldo + N) * 4ull;
  return w < BUFFER_LIMIT && x < BUFFER_LIMIT && h < BUFFER_LIMIT && o < BUFFER_LIMIT;
}
// The most bytes a weight matrix may span ((N - 1) ldw + K elements of two bytes).
extern "C" unsigned long long qvl_gemm_resident_max_weight_bytes() { return BUFFER_LIMIT - 1; }

extern "C" int qvl_gemm_resident_pass_k() { return PASS_K; }
// the longest K with which 17 to 32 rows stay resident (and with which their norm is folded in)
extern "C" int qvl_gemm_resident_two_tile_k() { return TWO_TILE_K; }

// x: bfloat16 [M, K] (h null), or h: float32 [M, K] with norm_w [K] and eps (x null): X = rmsnorm(h) * norm_w.
// epilogue 0: out[M, N] in out_dtype (0 float32, 1 bfloat16); 1: out (float32 [M, N]) += product;
// 2: out[M, N/2] bfloat16 = silu(gate) * up for W rows in groups of 8 gate, 8 up; 4: the same with gelu's tanh form;
// 5: out[M, N] in out_dtype = max(product (+ bias), 0)^2.
// max_blocks: blocks to launch at most (the number of compute units).
extern "C" int qvl_gemm_resident(const void* x, int ldx, const void* h, int ldh, const void* norm_w, float eps,
                                 const void* W, int ldw, const void* bias, void* out, int ldo, int M, int N, int K,
                                 int out_dtype, int epilogue, int max_blocks, hipStream_t stream) {
  if (M <= 0 || N <= 0) return QVL_OK;
  const int gelu = epilogue == 4 ? 1 : (epilogue == 5 ? ACT_RELU2 : 0);
  if (epilogue == 4) epilogue = EPI_SWIGLU;
  if (epilogue == 5) epilogue = EPI_STORE;
  if (M > 64) return QVL_ERR_LIMIT;
  if (M > 32 && K > PASS_K) return QVL_ERR_LIMIT;   // teams of more than two keep their rows for a single pass
  if (K <= 0 || K % 8 || ldw % 8 || ldw < K || max_blocks <= 0 || !W || !out) return QVL_ERR_SHAPE;
  if (!fits_descriptors(M, N, K, ldw, ldx, ldh, ldo)) return QVL_ERR_LIMIT;
  const bool norm = h != nullptr;
  const Plan pl = plan_for(M, K, norm, max_blocks);
  const int teams = plan_teams(pl, max_blocks);
  if (norm) {
    if (x || !norm_w || K > PASS_K || ldh % 4 || ldh < K) return QVL_ERR_SHAPE;
    if (!qvl_gemm_resident_folds_norm(M, K, max_blocks)) return QVL_ERR_LIMIT;
  } else if (!x || ldx % 8 || ldx < K) {
    return QVL_ERR_SHAPE;
  }
  if (epilogue == EPI_SWIGLU) {
    if (N % 16 || ldo < N / 2 || bias) return QVL_ERR_SHAPE;
  } else if (ldo < N) {
    return QVL_ERR_SHAPE;
  }
  ResidentArgs p;
  p.X = (const bf16_t*)x; p.ldx = ldx; p.H = (const float*)h; p.ldh = ldh; p.norm_w = (const float*)norm_w;
  p.eps = eps; p.W = (const bf16_t*)W; p.ldw = ldw; p.bias = (const float*)bias; p.out = out; p.ldo = ldo;
  p.M = M; p.N = N; p.K = K; p.gelu = gelu; p.stack_blocks = 0; p.stack_x = p.stack_w = p.stack_o = 0; p.all_k = 0;
  p.cs = nullptr; p.slot = nullptr;
  p.q_out = nullptr; p.kc = nullptr; p.vc = nullptr; p.nq = p.nkv = p.hd = p.ps = 0; p.pair_tiles = 0;
  // as many rounds of tiles as 16-row tiles need, with rows per tile cut down to what fills them evenly
  p.rows = 16;
  if (epilogue != EPI_SWIGLU) {
    const long long per_round = 16LL * teams;
    const long long rounds = (N + per_round - 1) / per_round;   // (more rounds of shorter tiles lose: a load instruction then carries fewer rows)
    p.rows = (int)((N + rounds * teams - 1) / (rounds * teams));
  }
  p.ntiles = (N + p.rows - 1) / p.rows;
  p.whole_tiles = p.ntiles; p.parts = 1; p.pairs = 8;
  if (epilogue == EPI_SWIGLU) {
    const int groups = N / 16, left = groups % teams;
    if (groups > teams && left > 0) {
      while (p.parts < 8 && left * p.parts * 2 <= teams) p.parts *= 2;
      p.pairs = 8 / p.parts;
      p.whole_tiles = groups - left;
      p.ntiles = p.whole_tiles + left * p.parts;
    }
  }
#define QVL_RES(TO, EPI) \
  return norm ? launch<TO, PRO_NORM, EPI>(p, pl, max_blocks, stream) : launch<TO, PRO_PLAIN, EPI>(p, pl, max_blocks, stream)
  if (epilogue == EPI_STORE && out_dtype == 0) QVL_RES(float, EPI_STORE);
  if (epilogue == EPI_STORE && out_dtype == 1) QVL_RES(bf16_t, EPI_STORE);
  if (epilogue == EPI_RESIDUAL) QVL_RES(float, EPI_RESIDUAL);
  if (epilogue == EPI_SWIGLU) QVL_RES(bf16_t, EPI_SWIGLU);
#undef QVL_RES
  return QVL_ERR_DTYPE;
}

// out[i] = x[i] W[i]^T for `count` products of the same sizes, bfloat16 in, out_dtype out: x [M, K] (rows ldx apart) every
// x_stride elements, W [N, K] every w_stride, out [M, N] every o_stride.  M at most 32, K for one pass over the
// weights; every product gets its share of max_blocks (at least one).
extern "C" int qvl_gemm_resident_stack(const void* x, int ldx, long long x_stride, const void* W, int ldw, long long w_stride,
                                       void* out, int ldo, long long o_stride, int count, int M, int N, int K, int out_dtype,
                                       int max_blocks, hipStream_t stream) {
  if (M <= 0 || N <= 0 || count <= 0) return QVL_OK;
  if (K <= 0 || K % 8 || ldw % 8 || ldw < K || ldx % 8 || ldx < K || ldo < N || x_stride % 8 || w_stride % 8 || !x || !W || !out ||
      max_blocks < count)
    return QVL_ERR_SHAPE;
  if (M > 32 || !fits_descriptors(M, N, K, ldw, ldx, 0, ldo)) return QVL_ERR_LIMIT;
  const int share = max_blocks / count;
  const Plan pl = plan_for(M, K, false, share);
  if (pl.groups != 1 || !pl.one_pass || pl.mt < 1) return QVL_ERR_LIMIT;
  ResidentArgs p;
  p.X = (const bf16_t*)x; p.ldx = ldx; p.H = nullptr; p.ldh = 0; p.norm_w = nullptr; p.eps = 0.f; p.W = (const bf16_t*)W;
  p.ldw = ldw; p.bias = nullptr; p.out = out; p.ldo = ldo; p.M = M; p.N = N; p.K = K; p.gelu = 0; p.groups = 1;
  p.cs = nullptr; p.slot = nullptr;
  p.q_out = nullptr; p.kc = nullptr; p.vc = nullptr; p.nq = p.nkv = p.hd = p.ps = 0; p.pair_tiles = 0;
  const long long rounds = (N + 16LL * share - 1) / (16LL * share);
  p.rows = (int)((N + rounds * share - 1) / (rounds * share));
  p.ntiles = (N + p.rows - 1) / p.rows;
  p.whole_tiles = p.ntiles; p.parts = 1; p.pairs = 8;
  p.stack_blocks = share < p.ntiles ? share : p.ntiles;
  p.stack_x = x_stride; p.stack_w = w_stride; p.stack_o = o_stride; p.all_k = 0;
  const dim3 grid(p.stack_blocks * count), block(64 * RW);
#define QVL_STACK(TO)                                                                                                      \
  if (pl.mt == 1) hipLaunchKernelGGL((gemm_resident_kernel<TO, PRO_PLAIN, EPI_STORE, true, 1>), grid, block, 0, stream, p); \
  else hipLaunchKernelGGL((gemm_resident_kernel<TO, PRO_PLAIN, EPI_STORE, true, 2>), grid, block, 0, stream, p)
  if (out_dtype == 0) { QVL_STACK(float); }
  else if (out_dtype == 1) { QVL_STACK(bf16_t); }
  else return QVL_ERR_DTYPE;
#undef QVL_STACK
  return qvl_launch_status();
}

// Ranges of K over blocks: how a product is cut on a device with `cus` compute units.  A block carries all rows for at most
// PASS_K columns; among the numbers of ranges around the least possible the one is taken whose busiest block
// reads the fewest bytes (7B down projection, 3,584 x 18,944: 5 ranges of 51 blocks with up to 5 tiles of 15 rows), each
// range beyond the least costing a slab more for the norm that adds them.
struct Cut {
  int chunks, chunk_k, per_chunk, rows, ntiles;
};
static Cut cut_for(int M, int N, int K, int cus) {
  const int least = (K + PASS_K - 1) / PASS_K;
  Cut best{0, 0, 0, 0, 0};
  double best_cost = 1e30;
  for (int chunks = least; chunks <= least + 6 && chunks <= cus; ++chunks) {
    Cut c;
    c.chunks = chunks;
    c.chunk_k = ((K + chunks - 1) / chunks + 31) / 32 * 32;
    if (c.chunk_k > PASS_K || (long long)c.chunk_k * (chunks - 1) >= K) continue;
    c.per_chunk = cus / chunks;
    const long long per_round = 16LL * c.per_chunk, rounds = (N + per_round - 1) / per_round;
    c.rows = (int)((N + rounds * c.per_chunk - 1) / (rounds * c.per_chunk));
    c.ntiles = (N + c.rows - 1) / c.rows;
    if (c.per_chunk > c.ntiles) c.per_chunk = c.ntiles;
    const long long tiles = (c.ntiles + c.per_chunk - 1) / c.per_chunk;
    const double cost = (double)tiles * c.rows * c.chunk_k * 2 * cus + 16.0 * chunks * M * N;
    if (cost < best_cost) {
      best_cost = cost;
      best = c;
    }
  }
  return best;
}

// Whether qvl_gemm_split takes these sizes, and how many slabs it then writes (0: it does not).
extern "C" int qvl_gemm_split_chunks(int M, int N, int K, int cus) {
  if (M <= 0 || M > 16 || N <= 0 || K <= 0 || K % 8 || cus <= 0) return 0;
  return cut_for(M, N, K, cus).chunks;
}

// x: bfloat16 [M, K] (ldx elements a row).  W: bfloat16 [N, K].  out: float32 [chunks][M][N], chunks =
// qvl_gemm_split_chunks(M, N, K, cus); the product is the sum of the slabs.  K a multiple of 8.
extern "C" int qvl_gemm_split(const void* x, int ldx, const void* W, int ldw, void* out, int M, int N, int K, int cus,
                              hipStream_t stream) {
  if (M <= 0 || N <= 0) return QVL_OK;
  if (K <= 0 || K % 8 || ldw % 8 || ldw < K || ldx % 8 || ldx < K || cus <= 0 || !x || !W || !out) return QVL_ERR_SHAPE;
  if (!fits_descriptors(M, N, K, ldw, ldx, 0, 0)) return QVL_ERR_LIMIT;
  if (qvl_gemm_split_chunks(M, N, K, cus) == 0) return QVL_ERR_LIMIT;
  const Cut c = cut_for(M, N, K, cus);
  ResidentArgs p;
  p.X = (const bf16_t*)x; p.ldx = ldx; p.H = nullptr; p.ldh = 0; p.norm_w = nullptr; p.eps = 0.f; p.W = (const bf16_t*)W;
  p.ldw = ldw; p.bias = nullptr; p.out = out; p.ldo = N; p.M = M; p.N = N; p.K = c.chunk_k; p.gelu = 0; p.groups = 1;
  p.cs = nullptr; p.slot = nullptr;
  p.q_out = nullptr; p.kc = nullptr; p.vc = nullptr; p.nq = p.nkv = p.hd = p.ps = 0; p.pair_tiles = 0;
  p.rows = c.rows; p.ntiles = c.ntiles; p.whole_tiles = c.ntiles; p.parts = 1; p.pairs = 8;
  p.stack_blocks = c.per_chunk; p.stack_x = p.stack_w = c.chunk_k; p.stack_o = (long long)M * N; p.all_k = K;
  const dim3 grid(c.chunks * c.per_chunk), block(64 * RW);
  hipLaunchKernelGGL((gemm_resident_kernel<float, PRO_PLAIN, EPI_STORE, true, 1>), grid, block, 0, stream, p);
  return qvl_launch_status();
}

// The stacked query | key | value projection of at most 32 tokens with rotation and cache write
// folded in (EPI_ROPE).  x / h / norm_w / eps as in qvl_gemm_resident.  W: [(nq + 2 nkv) hd, K];
// bias: float32 [(nq + 2 nkv) hd] or null.  cs: float32 [M, hd / 2, 2], cosine and sine of every
// token's angle at every frequency (1 and 0 where a frequency is not rotated);
// slot: int32 [M] flat cache slot of each token (null with nkv == 0: queries only);
// q_out: bfloat16 [M, nq hd]; kc: [pages, nkv, ps, hd]; vc: [pages, nkv, hd, ps].
// hd must be a multiple of 16 (the rotation covers the whole head, channel f with f + hd / 2).
extern "C" int qvl_gemm_resident_rope(const void* x, int ldx, const void* h, int ldh, const void* norm_w, float eps,
                                      const void* W, int ldw, const void* bias, int M, int K, const void* cs,
                                      const void* slot, void* q_out, void* kc, void* vc, int nq, int nkv, int hd, int ps,
                                      int max_blocks, hipStream_t stream) {
  if (M <= 0) return QVL_OK;
  if (M > 64) return QVL_ERR_LIMIT;
  if (M > 32 && K > PASS_K) return QVL_ERR_LIMIT;   // as in qvl_gemm_resident
  if (K <= 0 || K % 8 || ldw % 8 || ldw < K || max_blocks <= 0 || !W || !q_out) return QVL_ERR_SHAPE;
  if (nq <= 0 || nkv < 0 || hd <= 0) return QVL_ERR_SHAPE;
  if (!fits_descriptors(M, (nq + 2 * nkv) * hd, K, ldw, ldx, ldh, 0)) return QVL_ERR_LIMIT;
  if (nq <= 0 || nkv < 0 || hd <= 0 || hd % 16 || ps <= 0 || !cs) return QVL_ERR_SHAPE;
  if (nkv > 0 && (!slot || !kc || !vc)) return QVL_ERR_SHAPE;
  const bool norm = h != nullptr;
  const Plan pl = plan_for(M, K, norm, max_blocks);
  const int teams = plan_teams(pl, max_blocks);
  if (norm) {
    if (x || !norm_w || K > PASS_K || ldh % 4 || ldh < K) return QVL_ERR_SHAPE;
    if (!qvl_gemm_resident_folds_norm(M, K, max_blocks)) return QVL_ERR_LIMIT;
  } else if (!x || ldx % 8 || ldx < K) {
    return QVL_ERR_SHAPE;
  }
  ResidentArgs p;
  p.X = (const bf16_t*)x; p.ldx = ldx; p.H = (const float*)h; p.ldh = ldh; p.norm_w = (const float*)norm_w;
  p.eps = eps; p.W = (const bf16_t*)W; p.ldw = ldw; p.bias = (const float*)bias; p.out = nullptr; p.ldo = 0;
  p.M = M; p.N = (nq + 2 * nkv) * hd; p.K = K; p.gelu = 0; p.stack_blocks = 0; p.stack_x = p.stack_w = p.stack_o = 0; p.all_k = 0;
  // query and key heads in tiles of 8 + 8 rows, then the value rows in tiles as small as fills
  // the compute units evenly (36 heads of 128 on 256 units: 256 tiles of 16 and 256 of 2)
  p.pair_tiles = (nq + nkv) * (hd / 16);
  p.rows = 16;
  int value_tiles = 0;
  if (nkv > 0) {
    const long long vrows = (long long)nkv * hd, per_round = 16LL * teams;
    const long long rounds = (vrows + per_round - 1) / per_round;
    p.rows = (int)((vrows + rounds * teams - 1) / (rounds * teams));
    value_tiles = (int)((vrows + p.rows - 1) / p.rows);
  }
  p.ntiles = p.pair_tiles + value_tiles;
  p.cs = (const float*)cs; p.slot = (const int*)slot; p.q_out = (bf16_t*)q_out; p.kc = (bf16_t*)kc;
  p.vc = (bf16_t*)vc; p.nq = nq; p.nkv = nkv; p.hd = hd; p.ps = ps;
  p.whole_tiles = 0; p.parts = 1; p.pairs = 8;
  return norm ? launch<bf16_t, PRO_NORM, EPI_ROPE>(p, pl, max_blocks, stream)
              : launch<bf16_t, PRO_PLAIN, EPI_ROPE>(p, pl, max_blocks, stream);
}
