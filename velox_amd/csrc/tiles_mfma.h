// bfloat16 products of many rows in large tiles on the matrix cores of gfx950, out = a w^T: one product, whole or in parts of k, or a
// product per expert with the plan of routed.hip.
//
// What bounds such a product is power first (independent matrix instructions on random operands run at 1.8 PFLOP/s, on zeros at 2.46;
// with the reads of LDS that a tile needs 1.6) and then how evenly the matrix cores are fed.  So:
//   - Four waves, one per SIMD, 2 x 2 over the tile; a wave owns 32 RT rows x 32 CT columns as 16 x 16 accumulators in the accumulation
//     registers: the larger a wave's part, the fewer reads of LDS per product.  16x16x32 draws less power than 32x32x16 (8,192
//     cubed: 1,513 and 1,344 TFLOP/s).  The instruction is written as assembly only to pin the accumulators where they are: the
//     compiler's own allocation moves them to and fro (three moves per instruction, 703 TFLOP/s).
//   - A step is 64 indices.  Each wave works it as four quadrants (half of its rows x half of its columns); while a
//     quadrant is multiplied the operands of the next one leave LDS, each exactly once per step.  So half of a buffer is
//     free again in the middle of its step, and its loads for S steps later are asked for at once: S buffers give
//     loads S - 1/2 steps to arrive, not S - 1 (4,001 x 4,096 x 11,008: 239 us, and 332 with loads one step ahead).  Two barriers a step
//     (four, with loads up to a quarter earlier: 3 to 8% slower).
//   - Operands go straight into LDS (buffer loads, whose bounds check reads zeros behind a matrix: no clamped
//     addresses, and one set of offsets for all tiles).  A row of 64 indices is 128 bytes, eight pieces of 16; the pieces of row r are
//     exchanged by an XOR with r's low three bits: no bank conflicts.
//   - Workgroups stay and take tile after tile; a tile's last steps already load the next one's first.
//   - Tiles are dealt to the eight XCDs in contiguous runs, in blocks of 1,024 rows, column after column, so that the 32 tiles that an
//     XCD has under way share a few rows of either operand in its L2 (2,048 rows instead: 4% slower at 4,001 x 22,016 x 4,096).
// Measured on MI355X (us, the matrix library / this): 2,048 x 37,888 x 3,584 535 / 409 and with SiLU behind it 572 / 428; 836 rows 268 / 198;
// 4,001 x 22,016 x 4,096 640 / 530; 4,001 x 4,096 x 11,008 228 / 232; 1,036 x 10,368 x 2,048 49 / 38.
// An output is summed over k in one chain of 32-index instructions from zero: every tile gives the same bits.
//
// Requirements (checked by the callers): k % 8 == 0, n % 4 == 0, a_ld % 8 == 0, 16-byte aligned bases, and less than 2 GiB from a
// tile's first row of an operand to its last (tiles_fit).
#pragma once
#include <type_traits>

#include "common.h"

typedef __bf16 tl_bf16x8_t __attribute__((ext_vector_type(8)));
typedef int tl_int4_t __attribute__((ext_vector_type(4)));
typedef unsigned int tl_uint2_t __attribute__((ext_vector_type(2)));
typedef unsigned int tl_uint4_t __attribute__((ext_vector_type(4)));

// what becomes of the sums: nothing; silu(gate) * up and max(gate, 0) * up of sums that are rounded to bfloat16 first, as a product of its
// own would leave them; an expert's gated middle, silu(gate) * up or any other; a unit without a gate branch
enum { TL_PLAIN = 0, TL_SILU = 1, TL_RELU = 2, TL_SILU_UNIT = 3, TL_UNIT = 4, TL_ACT = 5 };

#define TL_XCDS 8
#define TL_WORKGROUPS 256  // one per compute unit

struct TileArgs {
  const bf16_t* a;     // element (r, k) at a[r * a_ld + k]
  long long a_ld;
  const bf16_t* w;     // [n (gated: n gate rows, then n up rows)][k]; group g's at w + g * w_group
  long long w_group;
  void* out;           // element (r, col) at out[r * n + col]; part p of a cut sum at out + p * m * n
  const float* bias;   // TL_PLAIN: float32 [n], added before the rounding (nullptr: none)
  int m, n, k;
  int splits;          // without a plan: parts of k, each with a result of its own
  const int* plan;     // nullptr: one product of m rows
  int plan_pairs, plan_groups, plan_max_tiles;
  int gather_top;      // with a plan: > 0: sorted row r is row order[r] / gather_top of `a`
  int act;             // TL_ACT: ungated_act's kind
  GluUnit unit;        // TL_UNIT
};

__device__ __forceinline__ tl_int4_t tl_resource(const void* p, long long bytes) {
  const uint64_t at = (uint64_t)p;
  return tl_int4_t{(int)at, (int)((at >> 32) & 0xffff), bytes > 0x7fffffffLL ? 0x7fffffff : (int)bytes, 0x00020000};
}

// 16 bytes per lane from `rsrc` at lane_bytes + wave_bytes into LDS, lane l's at `at` + 16 l; zeros behind the resource's end.  (In
// assembly for the reason that load_to_lds_16 gives.)
__device__ __forceinline__ void tl_load(const tl_int4_t& rsrc, uint32_t lane_bytes, uint32_t wave_bytes, uint32_t at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" : : "s"(at), "v"(lane_bytes), "s"(rsrc), "s"(wave_bytes) : "memory", "m0");
}

// `plain`: the accumulator lies in ordinary registers.
__device__ __forceinline__ void tl_mfma(float4_t& acc, const tl_bf16x8_t& x, const tl_bf16x8_t& y, bool plain) {
  if (plain) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(x), "v"(y));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(x), "v"(y));
}

typedef const __attribute__((address_space(3))) tl_bf16x8_t tl_lds_t;
__device__ __forceinline__ tl_bf16x8_t tl_read(uint32_t at) { return *(tl_lds_t*)(uintptr_t)at; }

// At most N of this wave's loads are still under way and its reads of LDS are back, then the same for the whole workgroup.
template <int N> __device__ __forceinline__ void tl_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" : : : "memory");
}

__device__ __forceinline__ uint32_t tl_pack(float x, float y) {
  return (uint32_t)(uint16_t)bf16_bits(x) | ((uint32_t)(uint16_t)bf16_bits(y) << 16);
}

// g / (1 + e^-g), as close to it as the library's exponential and division come, in half of their some forty instructions per output, which nothing
// hides here.  e^-g is 2^whole 2^rest; the rest has what the product with log2 e is rounded by, or, of a bfloat16 g (SHORT), that product with 16
// bits of log2 e is exact.  The quotient by the instruction set's reciprocal is corrected once.  Below -64, where the denominator nears float32's
// end and its reciprocal the end of what that instruction returns, both sides are 2^-8 of themselves; beyond +-88.7 the correction would
// multiply an infinity.  Every bfloat16 g has the library's bits; of 2e8 float32 ones from 0.01 to 20 and from -20 to -0.01 five have not, and either is
// 3.6e-08 and 4.4e-08 off 64 bits (the exponential and the reciprocal of the instruction set alone 4.6e-08 and 2.4e-07, and 0 below -87.3).  2,048 x 37,888 x
// 3,584: 428 us, with those two 417, with the library's 479, a product and a kernel behind it 446.
template <bool SHORT>
__device__ __forceinline__ float tl_silu(float g) {
#pragma clang fp contract(off)  // (what `power` is rounded by is added back)
  const float z = __builtin_amdgcn_fmed3f(g, -104.f, 104.f);
  const float power = z * (SHORT ? -1.44268799f : -1.44269502f), whole = rintf(power);
  const float rest = SHORT ? fmaf(z, -7.05260771e-06f, power - whole) : power - whole + fmaf(z, -1.92596303e-08f, fmaf(z, -1.44269502f, -power));
  const float e = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(rest), (int)whole);
  const float part = g < -64.f ? 0x1p-8f : 1.f;
  const float below = fmaf(e, part, part), above = g * part, inverse = __builtin_amdgcn_rcpf(below), near = above * inverse;
  return fabsf(g) <= 88.7f ? fmaf(-fmaf(near, below, -above), inverse, near) : near;
}

// A gated unit's middle.
template <int EPI>
__device__ __forceinline__ float tl_middle(float gate, float up, const TileArgs& args) {
  if (EPI == TL_UNIT) return glu_middle(gate, up, args.unit);
  if (EPI != TL_SILU_UNIT) {
    gate = to_f32(from_f32<bf16_t>(gate));
    up = to_f32(from_f32<bf16_t>(up));
  }
  if (EPI == TL_RELU) return fmaxf(gate, 0.f) * up;
  return tl_silu<EPI == TL_SILU>(gate) * up;
}

// RT, CT: tiles of 32 rows and 32 columns per wave; S: buffers.  GATHER: rows through the plan's order.  TAIL: k % 64 != 0.
template <int RT, int CT, int S, int EPI, typename TO, bool PLAN, bool GATHER, bool TAIL>
__device__ __forceinline__ void tiles_work(const TileArgs& args, char* smem) {
  static_assert(PLAN || !GATHER, "only a plan has an order");
  constexpr int WAVES = 4, TM = 64 * RT, TN = 64 * CT, STAGE = (TM + TN) * 128;
  constexpr int RH0 = (RT + 1) / 2, RH1 = RT - RH0, CH0 = (CT + 1) / 2, CH1 = CT - CH0;  // halves of a wave's tiles
  constexpr int LA0 = 2 * RH0, LC0 = 2 * CH0, LC1 = 2 * CH1, LA1 = 2 * RH1, LOADS = LA0 + LC0 + LC1 + LA1;  // loads of a wave in a step, in this order
  constexpr bool GLU = EPI == TL_SILU || EPI == TL_RELU || EPI == TL_SILU_UNIT || EPI == TL_UNIT;
  constexpr int OUT_COLS = GLU ? TN / 2 : TN;  // output columns of the tile
  constexpr int BLOCK_ROWS = 1024 / TM;        // row tiles of a block

  const int n = args.n, k = args.k;
  const int cols = (n + OUT_COLS - 1) / OUT_COLS;
  const int row_tiles = PLAN ? args.plan[0] : (args.m + TM - 1) / TM;
  const int total = row_tiles * cols * (PLAN ? 1 : args.splits), share = (total + TL_XCDS - 1) / TL_XCDS, per_xcd = gridDim.x / TL_XCDS;
  const int first_work = (int)(blockIdx.x % TL_XCDS) * share, last_work = min(total, first_work + share);
  int work = first_work + (int)(blockIdx.x / TL_XCDS);
  if (work >= last_work) return;  // (uniform over the workgroup)

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, h = lane >> 4, wm = wave >> 1, wn = wave & 1;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const uint32_t w_bytes = 2 * (uint32_t)k;
  const uint32_t piece = 8 * ((lane & 7) ^ (lane >> 3));  // first index of the piece this lane asks for, in every load
  const int* order = PLAN ? args.plan + 1 + args.plan_groups + 1 : nullptr;

  // load j of a step brings eight rows of one half of the waves' rows (of `a`) or columns (rows of W): the tile's row or column of the first
  auto of_a = [](int j) { return j < LA0 || j >= LA0 + LC0 + LC1; };
  auto place_of = [&](int j) {
    int count, stride, begin, base;
    if (j < LA0) count = RH0 * 32, stride = RT * 32, begin = 0, base = 0;
    else if (j < LA0 + LC0) count = CH0 * 32, stride = CT * 32, begin = 0, base = LA0;
    else if (j < LA0 + LC0 + LC1) count = CH1 * 32, stride = CT * 32, begin = CH0 * 32, base = LA0 + LC0;
    else count = RH1 * 32, stride = RT * 32, begin = RH0 * 32, base = LA0 + LC0 + LC1;
    const int at = 8 * (wave + WAVES * (j - base));
    return at / count * stride + begin + at % count;
  };

  struct Tile {
    int row0, end, col0, split, whole, steps;  // rows [row0, end), steps with indices of its own, steps worked (even, at least four)
    tl_int4_t a, w;
  };
  const int all_steps = (k + 63) / 64, split_steps = PLAN ? all_steps : (all_steps + args.splits - 1) / args.splits;
  auto tile_of = [&](int at) {
    Tile t;
    int begin = 0, end = args.m, tiles = row_tiles, group = 0;
    t.split = 0;
    if (PLAN) {
      const int* starts = args.plan + 1;
      const int* tile_group = order + 2 * (size_t)args.plan_pairs;
      const int* tile_row = tile_group + args.plan_max_tiles;
      // (a group's tiles follow one another, so at / cols lies among the tiles of the right one)
      const int near = at / cols;
      group = __builtin_amdgcn_readfirstlane(tile_group[near]);
      begin = __builtin_amdgcn_readfirstlane(starts[group]);
      end = __builtin_amdgcn_readfirstlane(starts[group + 1]);
      tiles = (end - begin + TM - 1) / TM;
      at -= (near - (__builtin_amdgcn_readfirstlane(tile_row[near]) - begin) / TM) * cols;
    } else {
      t.split = at / (row_tiles * cols);
      at -= t.split * row_tiles * cols;
    }
    const int block = at / (BLOCK_ROWS * cols), in_block = at % (BLOCK_ROWS * cols), block_rows = min(BLOCK_ROWS, tiles - block * BLOCK_ROWS);
    t.row0 = begin + (block * BLOCK_ROWS + in_block % block_rows) * TM;
    t.end = end;
    t.col0 = in_block / block_rows * OUT_COLS;
    const int step0 = t.split * split_steps;
    t.whole = max(0, min(split_steps, all_steps - step0));  // (a last part may be empty: zeros)
    t.steps = max(4, (t.whole + 1) / 2 * 2);
    const long long a_rows = GATHER ? args.plan_pairs / args.gather_top : PLAN ? args.plan_pairs : args.m;
    const long long a_from = (GATHER ? 0 : t.row0 * args.a_ld) + 64LL * step0, w_from = (long long)t.col0 * k + 64LL * step0;
    t.a = tl_resource(args.a + a_from, 2 * ((a_rows - 1) * args.a_ld + k - a_from));
    t.w = tl_resource(args.w + group * args.w_group + w_from, 2 * ((GLU ? 2LL * n : (long long)n) * k - w_from));
    return t;
  };

  uint32_t off[LOADS], a_off_next[GATHER ? LA0 + LA1 : 1];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    int r = place_of(j) + (lane >> 3);
    if (of_a(j)) {
      off[j] = (uint32_t)r * (2 * (uint32_t)args.a_ld) + 2 * piece;  // (GATHER: set per tile)
    } else {
      if (GLU) {  // a wave's columns: half gate rows, half the up rows of the same outputs
        const int u = r % (CT * 32);
        r = r / (CT * 32) * (CT * 16) + u % (CT * 16) + (u >= CT * 16 ? n : 0);
      }
      off[j] = (uint32_t)r * w_bytes + 2 * piece;
    }
  }
  auto gather = [&](const Tile& t) {
    if constexpr (GATHER) {
#pragma unroll
      for (int j = 0; j < LOADS; ++j)
        if (of_a(j)) {
          const int row = order[min(t.row0 + place_of(j) + (lane >> 3), t.end - 1)] / args.gather_top;
          a_off_next[j < LA0 ? j : j - LC0 - LC1] = (uint32_t)row * (2 * (uint32_t)args.a_ld) + 2 * piece;
        }
    }
  };
  auto take_gathered = [&] {
    if constexpr (GATHER) {
#pragma unroll
      for (int j = 0; j < LOADS; ++j)
        if (of_a(j)) off[j] = a_off_next[j < LA0 ? j : j - LC0 - LC1];
    }
  };

  Tile tile = tile_of(work), next;
  gather(tile);
  take_gathered();
  auto find_next = [&] {
    if (work + per_xcd < last_work) {
      next = tile_of(work + per_xcd);
      gather(next);
    } else {  // nothing is read behind the last tile
      next = tile;
      next.whole = 0;
    }
  };
  find_next();

  // where step `at` of this tile (behind its end: of the next one) comes from
  struct Source { tl_int4_t a, w; uint32_t at; bool next, tail; };
  auto source = [&](int at) {
    Source s;
    s.next = at >= tile.steps;
    const int in = s.next ? at - tile.steps : at, whole = s.next ? next.whole : tile.whole;
    s.a = s.next ? next.a : tile.a;
    s.w = s.next ? next.w : tile.w;
    if (in >= whole) s.a[2] = s.w[2] = 0;  // zeros: no indices of its own
    s.at = 128 * in;
    s.tail = TAIL && ((s.next ? next.split : tile.split) * split_steps + in == all_steps - 1);
    return s;
  };
  auto load = [&](int j, const Source& s, uint32_t stage) {
    uint32_t from = off[j];
    if (GATHER && of_a(j)) from = s.next ? a_off_next[j < LA0 ? j : j - LC0 - LC1] : from;
    if (TAIL && s.tail && (int)piece >= k % 64) from = 0x80000000u;  // (behind any resource's end: zeros)
    tl_load(of_a(j) ? s.a : s.w, from, s.at, lds0 + (place_of(j) + (of_a(j) ? 0 : TM)) * 128 + stage);
  };

  // operands: halves of the rows and of the columns, [16 x 16 tile][half of the 64 indices]; the column halves change places every step
  tl_bf16x8_t rows0[2 * RH0][2], rows1[2 * RH1][2], cols_x[2 * CH0][2], cols_y[2 * CH0][2];
  float4_t acc[2 * CT][2 * RT];
  // 64 accumulators would fill the accumulation registers to the last one, which the compiler answers with moves between them: the
  // first columns' lie in ordinary ones
  constexpr int PLAIN_TILES = RT * CT == 16 ? 1 : 0;
  auto clear = [&] {
#pragma unroll
    for (int c = 0; c < 2 * CT; ++c)
#pragma unroll
      for (int r = 0; r < 2 * RT; ++r) acc[c][r] = float4_t{0.f, 0.f, 0.f, 0.f};
  };
  // where this lane reads LDS: S == 2: in buffer 0 and 1, S == 3: in this step's and the next one's
  uint32_t a_read[2][2], w_read[2][2], stage_now = 0, stage_next = STAGE;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const uint32_t place = ((4 * q + h) ^ (i & 7)) * 16;
      a_read[b][q] = lds0 + b * STAGE + (wm * RT * 32 + i) * 128 + place;
      w_read[b][q] = lds0 + b * STAGE + (TM + wn * CT * 32 + i) * 128 + place;
      asm volatile("" : "+v"(a_read[b][q]), "+v"(w_read[b][q]));  // (kept, not worked out again at every read)
    }
#define TL_ROWS(HALF, T, Q, B) tl_read(a_read[B][Q] + (HALF) * RH0 * 4096 + (T) * 2048)
#define TL_COLS(HALF, T, Q, B) tl_read(w_read[B][Q] + (HALF) * CH0 * 4096 + (T) * 2048)

#pragma unroll
  for (int b = 0; b < S; ++b) {
    const Source s = source(b);
#pragma unroll
    for (int j = 0; j < LOADS; ++j) load(j, s, b * STAGE);
  }
  clear();
  tl_wait<LC1 + LA1 + (S - 1) * LOADS>();
#pragma unroll
  for (int t = 0; t < 2 * RH0; ++t)
#pragma unroll
    for (int q = 0; q < 2; ++q) rows0[t][q] = TL_ROWS(0, t, q, 0);
#pragma unroll
  for (int t = 0; t < 2 * CH0; ++t)
#pragma unroll
    for (int q = 0; q < 2; ++q) cols_x[t][q] = TL_COLS(0, t, q, 0);

  // NR x NC tiles of 32 x 32 at (RO, CO): the READS reads of the next quadrant among the first five eighths of the matrix instructions,
  // loads [FROM, TO) of a later step evenly between them
#define TL_QUADRANT(NR, NC, R, C, RO, CO, READS, READ, FROM, UPTO)                                                              \
  {                                                                                                                             \
    constexpr int COUNT = 8 * (NR) * (NC), ASKED = (UPTO) - (FROM);                                                             \
    __builtin_amdgcn_sched_barrier(0);                                                                                          \
    _Pragma("unroll") for (int j = 0; j < COUNT; ++j) {                                                                         \
      _Pragma("unroll") for (int u = 0; u < (READS); ++u) if (u * COUNT * 5 / ((READS) * 8) == j) { READ; }                     \
      _Pragma("unroll") for (int u = 0; u < ASKED; ++u) if (u * COUNT / ASKED == j) load((FROM) + u, from, stage);              \
      const int q = j / (4 * (NR) * (NC)), t = j % (4 * (NR) * (NC)), c = t / (2 * (NR)), z = t % (2 * (NR)), r = c & 1 ? 2 * (NR) - 1 - z : z; \
      tl_mfma(acc[2 * (CO) + c][2 * (RO) + r], C[c][q], R[r][q], 2 * (CO) + c < PLAIN_TILES);                                   \
      __builtin_amdgcn_sched_barrier(0);                                                                                        \
    }                                                                                                                           \
  }
  // A step: X holds the first column half.  In front of the first quadrant the second halves of this step have landed, in front of
  // the third the first halves of the next one; (S - 1) LOADS younger loads are under way either time, and what the quadrants
  // before have read is free for the loads that follow.
#define TL_STEP(X, Y, B)                                                                                                        \
  {                                                                                                                             \
    constexpr int NOW = S == 2 ? (B) : 0, THEN = S == 2 ? 1 - (B) : 1;                                                          \
    const uint32_t stage = S == 2 ? (B) * STAGE : stage_now;                                                                    \
    const Source from = source(s + S);                                                                                          \
    tl_wait<(S - 1) * LOADS>();                                                                                                 \
    TL_QUADRANT(RH0, CH0, rows0, X, 0, 0, 4 * CH1, (Y[u / 2][u % 2] = TL_COLS(1, u / 2, u % 2, NOW)), 0, LA0)                   \
    TL_QUADRANT(RH0, CH1, rows0, Y, 0, CH0, 4 * RH1, (rows1[u / 2][u % 2] = TL_ROWS(1, u / 2, u % 2, NOW)), LA0, LA0 + LC0)     \
    tl_wait<(S - 1) * LOADS>();                                                                                                 \
    TL_QUADRANT(RH1, CH1, rows1, Y, RH0, CH0, 4 * RH0, (rows0[u / 2][u % 2] = TL_ROWS(0, u / 2, u % 2, THEN)), LA0 + LC0, LA0 + LC0 + LC1) \
    TL_QUADRANT(RH1, CH0, rows1, X, RH0, 0, 4 * CH0, (Y[u / 2][u % 2] = TL_COLS(0, u / 2, u % 2, THEN)), LA0 + LC0 + LC1, LOADS) \
    if (S == 3) {                                                                                                               \
      stage_now = stage_next;                                                                                                   \
      const uint32_t move = stage_next == 2 * STAGE ? (uint32_t)(-2 * STAGE) : (uint32_t)STAGE;                                 \
      stage_next += move;                                                                                                       \
      _Pragma("unroll") for (int q = 0; q < 2; ++q) {                                                                           \
        a_read[0][q] = a_read[1][q];                                                                                            \
        w_read[0][q] = w_read[1][q];                                                                                            \
        a_read[1][q] += move;                                                                                                   \
        w_read[1][q] += move;                                                                                                   \
      }                                                                                                                         \
    }                                                                                                                           \
    ++s;                                                                                                                        \
  }

  for (;;) {
    int s = 0;
    for (int pair = 0; pair < tile.steps / 2; ++pair) {
      TL_STEP(cols_x, cols_y, 0)
      TL_STEP(cols_y, cols_x, 1)
    }
    asm volatile("s_nop 15\n\ts_nop 15" : : : "memory");  // the last products are in their registers,
#pragma unroll
    for (int c = 0; c < PLAIN_TILES; ++c)
#pragma unroll
      for (int r = 0; r < 2 * RT; ++r) asm volatile("" : "+v"(acc[c][r]));  // and none is read before that
    // lane (h, i) holds outputs 4 h .. + 3 of row i of every 16 x 16 tile.  float32: a 16-byte store each.  bfloat16: two tiles side by
    // side change places between the groups of 16 lanes until a lane holds eight neighbours, again 16 bytes.
    constexpr int OUT_TILES = GLU ? CT : 2 * CT;
    const int wave_col = tile.col0 + wn * OUT_TILES * 16;
    TO* out = reinterpret_cast<TO*>(args.out) + (PLAN ? (size_t)0 : (size_t)tile.split * args.m * n);
    float4_t bias[OUT_TILES];
    if (EPI == TL_PLAIN && !PLAN && args.bias != nullptr) {
#pragma unroll
      for (int c = 0; c < OUT_TILES; ++c)
#pragma unroll
        for (int u = 0; u < 4; ++u) bias[c][u] = args.bias[min(wave_col + 16 * c + 4 * h + u, n - 1)];
    }
    auto finished = [&](int c, int r) {
      float4_t v = acc[c][r];
      if (GLU) {
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = tl_middle<EPI>(v[u], acc[c + CT][r][u], args);
      }
      if (EPI == TL_ACT) {
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = ungated_act(v[u], args.act);
      }
      if (EPI == TL_PLAIN && !PLAN && args.bias != nullptr) v += bias[c];
      return v;
    };
    auto write = [&](auto whole_tile) {  // (a whole tile stores without conditions)
#pragma unroll
      for (int r = 0; r < 2 * RT; ++r) {
#pragma unroll
        for (int c = PLAIN_TILES; c < 2 * CT; ++c) asm volatile("" : "+a"(acc[c][r]));  // (nor these; a row of tiles at a time leaves the accumulation registers)
        const int row = tile.row0 + wm * RT * 32 + r * 16 + i;
        const bool mine = whole_tile.value || row < tile.end;
        TO* out_row = out + (size_t)row * n;
        auto store_four = [&](int c, const float4_t& v) {
          const int col = wave_col + 16 * c + 4 * h;
          if (!whole_tile.value && !(mine && col < n)) return;
          if constexpr (sizeof(TO) == 4) *reinterpret_cast<float4_t*>(out_row + col) = v;
          else *reinterpret_cast<tl_uint2_t*>(out_row + col) = tl_uint2_t{tl_pack(v[0], v[1]), tl_pack(v[2], v[3])};
        };
#pragma unroll
        for (int c = 0; c < OUT_TILES; c += 2) {
          const float4_t v0 = finished(c, r);
          if (c + 1 == OUT_TILES) {
            store_four(c, v0);
            continue;
          }
          const float4_t v1 = finished(c + 1, r);
          if (sizeof(TO) == 2 && (whole_tile.value || n % 8 == 0)) {
            const tl_uint2_t low = __builtin_amdgcn_permlane16_swap(tl_pack(v0[0], v0[1]), tl_pack(v1[0], v1[1]), false, false);
            const tl_uint2_t high = __builtin_amdgcn_permlane16_swap(tl_pack(v0[2], v0[3]), tl_pack(v1[2], v1[3]), false, false);
            const int col = wave_col + 16 * (c + (h & 1)) + 8 * (h >> 1);
            if (whole_tile.value || (mine && col < n)) *reinterpret_cast<tl_uint4_t*>(out_row + col) = tl_uint4_t{low[0], high[0], low[1], high[1]};
          } else {
            store_four(c, v0);
            store_four(c + 1, v1);
          }
        }
      }
    };
    const bool whole_tile = tile.row0 + TM <= tile.end && tile.col0 + OUT_COLS <= n && n % 8 == 0;
    if (whole_tile) write(std::true_type{});
    else write(std::false_type{});
    work += per_xcd;
    if (work >= last_work) break;
    tile = next;
    take_gathered();
    find_next();
    clear();
  }
  tl_wait<0>();  // (nothing is under way into LDS when the workgroup ends)
#undef TL_STEP
#undef TL_QUADRANT
#undef TL_COLS
#undef TL_ROWS
}

constexpr int tiles_lds(int rt, int ct, int s) { return s * (rt + ct) * 64 * 128; }

template <int RT, int CT, int S, int EPI, typename TO, bool PLAN, bool GATHER, bool TAIL>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) tiles_kernel(const TileArgs args) {
  static_assert(tiles_lds(RT, CT, S) <= 160 * 1024, "LDS of a compute unit");
  __shared__ __attribute__((aligned(1024))) char smem[tiles_lds(RT, CT, S)];
  tiles_work<RT, CT, S, EPI, TO, PLAN, GATHER, TAIL>(args, smem);
}

// Columns of a plan's tiles, in 64: the fewest whose tiles take no more rounds over the compute units than those of 256 do.  A tile's order of
// additions is the same at any width; a step of a narrower one is shorter, and where 256 columns leave compute units without a tile, W
// comes through more of them (each gets some 40 GB/s of it).
__host__ __device__ inline int plan_tile_cols(int row_tiles, int w_rows) {
  auto rounds = [&](int ct) { return (row_tiles * ((w_rows + 64 * ct - 1) / (64 * ct)) + TL_WORKGROUPS - 1) / TL_WORKGROUPS; };
  int ct = 4;
  while (ct > 2 && rounds(ct - 1) <= rounds(4)) --ct;
  return ct;
}

// The plan's products in tiles as wide as its number of row tiles asks for, which only the device knows: the host can expect it, but a tile more
// than makes whole rounds is a round more, and routers do not spread tokens evenly.  Measured on MI355X, us of a layer's routed experts with
// 256 columns / with the widths that evenly spread rows would ask for / like this: 2,072 pairs over 16 experts of 2,048 -> 1,408, evenly
// spread 96.9 / 89.1 / 89.8, by Zipf's law 97.8 / 125.7 / 95.4, all on two 78.1 / 64.7 / 67.8; 600 pairs, a quarter of the experts with nearly all
// 86.0 / 100.7 / 82.1; 32 of 4,096 -> 1,408, 1,340 pairs 253 / 235 / 235, by the law's square 263 / 278 / 262, 10,000 pairs 439 / 429 /
// 435; 64 of 2,048 -> 768, 8,192 pairs over experts that differ by a factor of four 216 / 234 / 207.
template <int RT, int EPI, typename TO, bool GATHER>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) plan_tiles_kernel(const TileArgs args) {
  constexpr int S4 = RT == 3 ? 2 : 3;
  constexpr int LDS = tiles_lds(RT, 4, S4) > tiles_lds(RT, 3, 3) ? tiles_lds(RT, 4, S4) : tiles_lds(RT, 3, 3);
  static_assert(LDS <= 160 * 1024, "LDS of a compute unit");
  __shared__ __attribute__((aligned(1024))) char smem[LDS];
  const int ct = plan_tile_cols(args.plan[0], (EPI == TL_UNIT || EPI == TL_SILU_UNIT ? 2 : 1) * args.n);  // (uniform over the grid)
  if (ct == 4) tiles_work<RT, 4, S4, EPI, TO, true, GATHER, false>(args, smem);
  else if (ct == 3) tiles_work<RT, 3, 3, EPI, TO, true, GATHER, false>(args, smem);
  else tiles_work<RT, 2, 3, EPI, TO, true, GATHER, false>(args, smem);
}

// Whether a tile's operands lie within the reach of its resources.
static inline bool tiles_fit(long long a_rows_reached, long long a_ld, long long w_rows_reached, int k) {
  return 2 * a_rows_reached * a_ld < 0x7fffffffLL && 2 * w_rows_reached * k < 0x7fffffffLL;
}

// The tile of one product, as TM * 1,000 + TN.  `w_rows`: rows of W.  What a tile costs, fitted to 432 products (27 shapes of 1,536 x 1,536 to
// 37,888 x 3,584, 65 to 4,001 rows; mean error of the fit 2 to 5%, the tile chosen 0.5% slower than the best one on average, 14% at worst): a
// launch, then for every round of one tile per compute unit the tile's beginning and end and its steps, which take the longer the
// more compute units work (power, and the way from L2).  us:
struct TileCost { int rt, ct; float launch, round, step, step_alone; };
static constexpr TileCost TILE_COSTS[] = {{2, 2, 3.2f, 0.9f, 0.492f, 0.347f}, {2, 3, 2.8f, 2.2f, 0.639f, 0.461f}, {2, 4, 2.0f, 3.9f, 0.776f, 0.576f}, {3, 3, 1.9f, 4.7f, 0.814f, 0.613f},
                                          {3, 4, 0.4f, 6.7f, 0.990f, 0.745f}, {4, 3, 0.0f, 7.0f, 0.985f, 0.737f}, {4, 4, -0.2f, 8.6f, 1.253f, 0.943f}};

static inline float tiles_cost_of(const TileCost& t, float tiles, int k, int splits) {
  const int steps = (((k + 63) / 64 + splits - 1) / splits + 1) / 2 * 2;
  const float full = floorf(tiles / TL_WORKGROUPS), rest = tiles / TL_WORKGROUPS - full;
  return t.launch + full * (t.round + steps * t.step) + (rest > 0.f ? t.round + steps * (t.step_alone + (t.step - t.step_alone) * rest) : 0.f);
}

static inline float tiles_cost(const TileCost& t, long long m, long long w_rows, int k, int splits) {
  const long long tiles = (m + 64 * t.rt - 1) / (64 * t.rt) * ((w_rows + 64 * t.ct - 1) / (64 * t.ct)) * splits;
  return tiles_cost_of(t, (float)tiles, k, splits);
}

static inline const TileCost& tiles_best(long long m, long long w_rows, int k, int splits) {
  const TileCost* best = TILE_COSTS;
  for (const TileCost& t : TILE_COSTS)
    if (tiles_cost(t, m, w_rows, k, splits) < tiles_cost(*best, m, w_rows, k, splits)) best = &t;
  return *best;
}

static inline int tiles_pick(long long m, long long w_rows, int k, int splits) {
  if (k % 64 != 0) return 128256;
  const TileCost& t = tiles_best(m, w_rows, k, splits);
  return 64 * t.rt * 1000 + 64 * t.ct;
}

// In how many parts, up to `most`, a sum is cut: what the tiles cost and the parts, written and read again in float32 (one part: in
// bfloat16) at 4.5 TB/s.
static inline int tiles_splits(long long m, long long n, int k, int most) {
  int best = 1;
  float least = INFINITY;
  for (int s = 1; s <= most; ++s) {
    const float cost = tiles_cost(tiles_best(m, n, k, s), m, n, k, s) + (float)(m * n) * (s > 1 ? 8.f * s : 4.f) / 4.5e6f;
    if (cost < least) {
      least = cost;
      best = s;
    }
  }
  return best;
}

// One product in tiles of `tile`.
template <int EPI, typename TO, bool TAIL>
static int tiles_launch(const TileArgs& args, int tile, hipStream_t stream) {
  constexpr int BRANCHES = EPI == TL_SILU || EPI == TL_RELU ? 2 : 1;
#define TILES(RT, CT, S)                                                                                                              \
  case 64 * RT * 1000 + 64 * CT: {                                                                                                    \
    const long long cols = (args.n + 64 * CT / BRANCHES - 1) / (64 * CT / BRANCHES);                                                  \
    const long long tiles = (args.m + 64LL * RT - 1) / (64 * RT) * cols * args.splits;                                                \
    if (tiles > (1 << 30)) return -1;                                                                                                 \
    const int workgroups = (int)(tiles < TL_WORKGROUPS ? (tiles + TL_XCDS - 1) / TL_XCDS * TL_XCDS : TL_WORKGROUPS);                  \
    tiles_kernel<RT, CT, S, EPI, TO, false, false, TAIL><<<workgroups, 256, 0, stream>>>(args);                                       \
    return (int)hipGetLastError();                                                                                                    \
  }
  if constexpr (TAIL) {
    switch (tile) { TILES(2, 4, 3) }
  } else {
    switch (tile) { TILES(2, 2, 3) TILES(2, 3, 3) TILES(2, 4, 3) TILES(3, 3, 3) TILES(3, 4, 2) TILES(4, 3, 2) TILES(4, 4, 2) }
  }
#undef TILES
  return -1;
}
