// out[M, N] = A[M, K] * W[N, K]^T (+ bias[N]) of float32 operands on the bfloat16 matrix instructions of gfx950, which multiply 16 times as
// fast as the float32 ones, with no bit of an operand left out: a float32 number, times 2^24, is the sum of three bfloat16 ones (hi + mid +
// lo, each the nearest to what is left: 8 + 8 + 8 significant bits; without the factor, parts of a number below 2^-109 are beyond bfloat16's
// smallest ones, and 1e-36 times 1e20 came out with an error of 3e-5, 1e-38 with 3e-3; the multiplication costs no time), their products are exact in float32, and of the nine products
// of parts six count, hi hi + hi mid + mid hi + hi lo + mid mid + lo hi (the other three are 2^-26 of a term; the method is that of
// Henry, Tang, Heinecke: Leveraging the bfloat16 artificial intelligence datatype for higher-precision computations, 2019).
//
// Precision: the instruction rounds down where it adds 32 products to the sum so far, which one long chain would show (1,536 terms: 6e-7
// of the result's norm; 8,960: 1.5e-6).  So an output is built from sums of 128 terms (24 instructions from zero), added in float32
// with rounding to sums of up to 2,048, which are added up in the result's place.  Every other one of them is of the negative terms (the rows
// times -2^24) and subtracted: rounded down throughout, all of a layer's outputs were too small by the same 3e-8 (1,536 terms) or 8e-8 (8,960) of
// their norm, which added up from layer to layer, and a model's logits were 3% further from 64 bits than with the float32 instructions,
// although each product was closer (eight layers of width 1,536, six seeds: 1.64 to 1.94e-06, 1.68 to 2.00e-06; so 1.59 to 1.90e-06).  Error against float64, float32 matrix
// instructions / this: 512 terms 2.1e-07 / 1.6e-07, 1,536 2.1e-07 / 1.7e-07, 8,960 2.3e-07 / 1.7e-07, 18,944 2.6e-07 / 1.8e-07; of terms of one
// sign 9.5e-08 / 7.3e-08, 6.2e-08 / 6.2e-08, 7.5e-08 / 5.3e-08, 9.8e-08 / 5.8e-08.  (Inner sums of 64 terms: 1.3e-07 at 1,536 terms, 2% slower;
// sums of 1,024 in the result's place: 190 instead of 180 us where 1,536 terms are added, for the passes over the result.)
//
// What bounds it: the matrix cores (six instructions of 16 cycles for 16 x 16 x 32 terms: at most 2,500 / 6 = 417 TFLOP/s of float32
// products, 250 at the rate that power leaves them), and beside them the splitting: 52 vector instructions for eight numbers.
//   - Eight waves own 32 RT x 64 CT outputs.  A step is 32 indices: operands come into registers a step ahead, are split ONCE per
//     workgroup on their way into LDS (not by each wave that reads them: half of the vector work) and lie there as three planes, two buffers.
//   - Half of the waves split before they multiply and half behind it, so that the vector units and the matrix cores have work at the
//     same time.  (All of them first: 4% slower.  The two waves of a SIMD at different times is better with two tiles of rows,
//     both at one time with four.)
//   - One barrier a step; a wave's operands leave LDS once per step, those of a column of tiles behind the products of the one before.
// Measured on MI355X (us, float32 matrix instructions / this): 616 rows, 1,536 -> 17,920: 330 / 203 (167 TFLOP/s); 8,960 -> 1,536 in parts 206 /
// 94; 4,000 rows, 2,048 -> 11,264: 1,560 / 970 (191); 64 rows, 8,960 -> 1,536 in eight parts 69 / 25.  Without the splitting (stale operands)
// 4,000 rows take 0.74 of the time: what is left to gain.
#include "common.h"

typedef __bf16 sp_bf16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned int sp_uint4_t __attribute__((ext_vector_type(4)));
typedef float sp_float8_t __attribute__((ext_vector_type(8)));

#define SPLIT_FOLD 4    // steps of 32 terms per inner sum
#define SPLIT_LEVEL 64  // steps whose inner sums are added up in registers, at most
#define SPLIT_SCALE 0x1p24f  // of either operand
#define SPLIT_XCDS 8
#define SPLIT_CUS 256

struct SplitArgs {
  const float* a;
  const float* w;
  const float* bias;  // nullptr: none
  float* out;         // part p of a cut sum at out + p * m * n
  int m, n, k;
  int splits, split_steps;  // parts of k and steps of 32 of each (a multiple of SPLIT_FOLD)
};

// Outputs of one wave with the float32 matrix instruction, from memory: those four of a lane's row in tile t that bit t of its `wanted` asks for, so
// that no row's bits depend on another's numbers.  It is taken where a sum is no finite number: an operand is an infinity, NaN or
// beyond 2^104, or the sum is beyond 2^80, where the factors leave float32's range.  Slow and
// seldom: a row of NaN among 616 takes 17,920 x 1,536 from 213 to 510 us, 8,960 -> 1,536 in eight parts from 95 to 331.
template <int RT, int CT>
__device__ __forceinline__ void split_outputs_in_float32(const SplitArgs& args, int row0, int col0, int part, uint32_t wanted) {
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int begin = part * args.split_steps * 32, end = min(args.k, begin + args.split_steps * 32);
  float* out = args.out + (size_t)part * args.m * args.n;
  for (int t = 0; t < RT * CT; ++t) {
    const bool mine = (wanted >> t & 1) != 0;
    if (!__any(mine)) continue;  // (the whole wave)
    const int row = row0 + t / CT * 16 + i, col = col0 + t % CT * 16;
    const float* a_row = args.a + (size_t)min(row, args.m - 1) * args.k + g;
    const float* w_row = args.w + (size_t)min(col + i, args.n - 1) * args.k + g;
    float4_t total = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = begin; k0 < end; k0 += 32 * SPLIT_FOLD) {
      float4_t acc = {0.f, 0.f, 0.f, 0.f};
      const int stop = min(end, k0 + 32 * SPLIT_FOLD);
      for (int at = k0; at < stop; at += 32) {
#pragma unroll
        for (int e = 0; e < 32; e += 4) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w_row[at + e], a_row[at + e], acc, 0, 0, 0);
      }
      total += acc;
    }
    if (!mine) continue;
    if (args.bias != nullptr) {
#pragma unroll
      for (int u = 0; u < 4; ++u) total[u] += args.bias[col + 4 * g + u];
    }
    *reinterpret_cast<float4_t*>(out + (size_t)row * args.n + col + 4 * g) = total;
  }
}

// RT, CT: 16 x 16 tiles of a wave; eight waves, 2 x 4.
template <int RT, int CT>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) split_f32_kernel(const SplitArgs args) {
  constexpr int TM = 32 * RT, TN = 64 * CT, BLOCKS = (TM + TN) / 16, PLANE = BLOCKS * 1024, STAGE = 3 * PLANE;
  constexpr int PIECES = (TM + TN) * 4, J = (PIECES + 511) / 512;
  static_assert(2 * STAGE <= 160 * 1024 && PIECES % 64 == 0 && TM * 4 % 64 == 0, "LDS of a compute unit; whole waves of pieces, of rows or columns");
  __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE];
  const int m = args.m, n = args.n, k = args.k;
  const int row_tiles = (m + TM - 1) / TM, tiles = row_tiles * ((n + TN - 1) / TN), total_tiles = tiles * args.splits;
  const int share = (total_tiles + SPLIT_XCDS - 1) / SPLIT_XCDS, mine = (int)(blockIdx.x / SPLIT_XCDS), work = (int)(blockIdx.x % SPLIT_XCDS) * share + mine;
  if (mine >= share || work >= total_tiles) return;  // (uniform over the workgroup)
  const int part = work / tiles, tile = work % tiles, m0 = tile % row_tiles * TM, n0 = tile / row_tiles * TN;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 15, h = lane >> 4;
  // a row of a step is 32 terms, four pieces of eight; 16 rows of one part are a kilobyte, [piece][row], the rows of a piece exchanged so
  // that neither the four pieces of four rows (written) nor 16 rows of one piece (read) meet in a bank
  auto place = [](int row, int piece) { return (row >> 4) * 1024 + (piece * 16 + ((row & 15) ^ (4 * piece + (piece >> 1) * 2))) * 16; };
  const float* from[J];
  uint32_t to[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int idx = min(tid + 512 * j, PIECES - 1), r = idx >> 2, piece = idx & 3;
    from[j] = (r < TM ? args.a + (size_t)min(m0 + r, m - 1) * k : args.w + (size_t)min(n0 + r - TM, n - 1) * k) + 8 * piece + (size_t)part * args.split_steps * 32;
    to[j] = place(r, piece);
  }
  const int steps = min(args.split_steps, k / 32 - part * args.split_steps);
  float4_t raw[J][2];
  auto ask = [&](int s) {
#pragma unroll
    for (int j = 0; j < J; ++j)
      if ((j + 1) * 512 <= PIECES || wave * 64 + 512 * j < PIECES) {
        raw[j][0] = *reinterpret_cast<const float4_t*>(from[j] + 32 * s);
        raw[j][1] = *reinterpret_cast<const float4_t*>(from[j] + 32 * s + 4);
      }
  };
  auto put = [&](char* stage, int s) {
    const float row_scale = s / SPLIT_FOLD % 2 != 0 ? -SPLIT_SCALE : SPLIT_SCALE;
#pragma unroll
    for (int j = 0; j < J; ++j)
      if ((j + 1) * 512 <= PIECES || wave * 64 + 512 * j < PIECES) {
        sp_float8_t x = __builtin_shufflevector(raw[j][0], raw[j][1], 0, 1, 2, 3, 4, 5, 6, 7) * (wave * 64 + 512 * j < 4 * TM ? row_scale : SPLIT_SCALE);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          sp_uint4_t bits;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(bits[e]) : "v"(x[2 * e]), "v"(x[2 * e + 1]));
            x[2 * e] -= __uint_as_float(bits[e] << 16);
            x[2 * e + 1] -= __uint_as_float(bits[e] & 0xffff0000u);
          }
          *reinterpret_cast<sp_uint4_t*>(stage + p * PLANE + to[j]) = bits;
        }
      }
  };

  const int wm = wave & 1, wn = wave >> 1;
  const bool splits_first = RT == 4 ? wm != 0 : wave < 4;
  const int a_at = place(i, h) + wm * RT * 1024, w_at = place(i, h) + (TM / 16 + wn * CT) * 1024;
  float4_t acc[CT][RT], total[CT][RT];
#pragma unroll
  for (int c = 0; c < CT; ++c)
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[c][r] = total[c][r] = float4_t{0.f, 0.f, 0.f, 0.f};
  auto fold = [&](int s) {  // the inner sum that step s belongs to
    const float sign = s / SPLIT_FOLD % 2 != 0 ? -1.f : 1.f;
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int r = 0; r < RT; ++r) {
#pragma unroll
        for (int u = 0; u < 4; ++u) total[c][r][u] = fmaf(acc[c][r][u], sign, total[c][r][u]);
        acc[c][r] = float4_t{0.f, 0.f, 0.f, 0.f};
      }
  };
  auto multiply = [&](const char* stage) {
    sp_bf16x8_t a_op[RT][3];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int p = 0; p < 3; ++p) a_op[r][p] = *reinterpret_cast<const sp_bf16x8_t*>(stage + a_at + p * PLANE + r * 1024);
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      sp_bf16x8_t w_op[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) w_op[p] = *reinterpret_cast<const sp_bf16x8_t*>(stage + w_at + p * PLANE + c * 1024);
      // the smallest products first
#pragma unroll
      for (int sum = 2; sum >= 0; --sum)
#pragma unroll
        for (int p = 0; p <= sum; ++p)
#pragma unroll
          for (int r = 0; r < RT; ++r) acc[c][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w_op[p], a_op[r][sum - p], acc[c][r], 0, 0, 0);
    }
  };

  ask(0);
  put(smem, 0);
  if (steps > 1) ask(1);
  // lane (h, i) holds outputs 4 h .. + 3 of row i of every tile
  float* out = args.out + (size_t)part * m * n;
  const int row0 = m0 + wm * 16 * RT, col0 = n0 + wn * 16 * CT;
  auto place_of = [&](int r, int c) -> float* {
    const int row = row0 + 16 * r + i, col = col0 + 16 * c + 4 * h;
    return row < m && col < n ? out + (size_t)row * n + col : nullptr;
  };
  bool begun = false;  // sums of earlier terms lie in `out`
  const int levels = (steps + SPLIT_LEVEL - 1) / SPLIT_LEVEL, level_steps = ((steps + levels - 1) / levels + SPLIT_FOLD - 1) / SPLIT_FOLD * SPLIT_FOLD;
  for (int s = 0;;) {
    const int end = min(steps, s + level_steps);
    for (; s < end; ++s) {
      char* now = smem + (s & 1) * STAGE;
      char* then = smem + (~s & 1) * STAGE;
      asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");  // what this step reads has been written, and what is written in this step has been read
      __builtin_amdgcn_s_barrier();
      asm volatile("" : : : "memory");
      auto next = [&] {
        if (s + 1 < steps) put(then, s + 1);
        if (s + 2 < steps) ask(s + 2);
        __builtin_amdgcn_sched_barrier(0);
      };
      if (splits_first) next();
      multiply(now);
      if (!splits_first) next();
      if (s % SPLIT_FOLD == SPLIT_FOLD - 1) fold(s);
    }
    fold(s);  // (a last inner sum of fewer terms, or zeros)
    if (s >= steps) break;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        if (float4_t* p = reinterpret_cast<float4_t*>(place_of(r, c))) *p = begun ? *p + total[c][r] : total[c][r];
        total[c][r] = float4_t{0.f, 0.f, 0.f, 0.f};
      }
    begun = true;
  }

  uint32_t beyond = 0;  // bit r CT + c
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      float4_t* p = reinterpret_cast<float4_t*>(place_of(r, c));
      if (p == nullptr) continue;
      float4_t v = total[c][r];
      if (begun) v += *p;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (!(fabsf(v[u]) < INFINITY)) beyond |= 1u << (r * CT + c);
        v[u] *= 1.f / (SPLIT_SCALE * SPLIT_SCALE);
        if (args.bias != nullptr) v[u] += args.bias[col0 + 16 * c + 4 * h + u];
      }
      *p = v;
    }
  if (__any(beyond != 0)) split_outputs_in_float32<RT, CT>(args, row0, col0, part, beyond);
}

// The tile of a product as rows * 1,000 + columns, by what it costs, fitted to 129 products of 512 to 37,888 columns, 1,024 to 8,960 terms and 17 to
// 4,000 rows in up to eight parts (mean error 2 to 4%; the tile and number of parts chosen are 0.3% slower than the best on average, 9% at
// worst).  us: a launch; for every round of tiles their beginning and end and their steps, which take the longer the more
// compute units work; of the small tiles two share a compute unit from 257 on.
struct SplitCost { int rt, ct, slots; float launch, round, step, step_alone; };
static constexpr SplitCost SPLIT_COSTS[] = {{4, 4, 256, 4.0f, 5.1f, 2.381f, 2.002f}, {4, 3, 256, 4.1f, 4.2f, 1.909f, 1.645f}, {3, 3, 256, 3.5f, 3.3f, 1.512f, 1.285f}, {2, 4, 256, 2.6f, 3.8f, 1.406f, 1.186f},
                                            {2, 2, 512, 2.9f, 2.4f, 1.747f, 0.780f}, {2, 1, 512, 4.1f, 0.4f, 1.127f, 0.503f}, {1, 2, 512, 3.1f, 1.2f, 1.336f, 0.609f}};

static int split_steps_of(int k, int splits) { return ((k / 32 + SPLIT_FOLD - 1) / SPLIT_FOLD + splits - 1) / splits * SPLIT_FOLD; }

static float split_cost(const SplitCost& t, long long m, long long n, int k, int splits) {
  const int steps = split_steps_of(k, splits);
  const long long tiles = (m + 32 * t.rt - 1) / (32 * t.rt) * ((n + 64 * t.ct - 1) / (64 * t.ct)) * splits;
  const float full = (float)(tiles / t.slots);
  const int rest = (int)(tiles % t.slots);
  const float busy = t.slots == SPLIT_CUS ? (float)rest / SPLIT_CUS : rest > SPLIT_CUS ? 1.f : 0.f;
  return t.launch + full * (t.round + steps * t.step) + (rest > 0 ? t.round + steps * (t.step_alone + (t.step - t.step_alone) * busy) : 0.f);
}

static const SplitCost& split_best(long long m, long long n, int k, int splits) {
  const SplitCost* best = SPLIT_COSTS;
  for (const SplitCost& t : SPLIT_COSTS)
    if (split_cost(t, m, n, k, splits) < split_cost(*best, m, n, k, splits)) best = &t;
  return *best;
}

extern "C" int velox_split_f32_tile(int m, int n, int k, int splits) {
  const SplitCost& t = split_best(m, n, k, splits);
  return 32 * t.rt * 1000 + 64 * t.ct;
}

// In how many parts, up to `most`, a sum is cut: what the tiles cost, and each further part written and read again at 4.5 TB/s.
extern "C" int velox_split_f32_parts(int m, int n, int k, int most) {
  int best = 1;
  float least = INFINITY;
  for (int s = 1; s <= most; ++s) {
    if ((s - 1) * split_steps_of(k, s) >= k / 32) continue;  // (an empty part)
    const float cost = split_cost(split_best(m, n, k, s), m, n, k, s) + (s - 1) * 8.f * m * n / 4.5e6f;
    if (cost < least) {
      least = cost;
      best = s;
    }
  }
  return best;
}

// Needs k % 32 == 0, n % 4 == 0 and 16-byte aligned operands and results.  `splits` parts of k, each with a result of its own (no bias then);
// `tile`: rows * 1,000 + columns (0: velox_split_f32_tile's).
extern "C" int velox_split_f32(const float* a, const float* w, const float* bias, float* out, int m, int n, int k, int splits, int tile, hipStream_t stream) {
  if (m <= 0 || n <= 0) return 0;
  if (k < 32 || k % 32 != 0 || n % 4 != 0 || splits < 1 || (splits > 1 && bias != nullptr) || (((uintptr_t)a | (uintptr_t)w | (uintptr_t)out) & 15) != 0) return -1;
  const int split_steps = split_steps_of(k, splits);
  if ((splits - 1) * split_steps >= k / 32) return -1;  // (an empty part)
  if (tile == 0) tile = velox_split_f32_tile(m, n, k, splits);
  SplitArgs args = {a, w, bias, out, m, n, k, splits, split_steps};
#define SPLIT(RT, CT)                                                                                                       \
  case 32 * RT * 1000 + 64 * CT: {                                                                                          \
    const long long tiles = (m + 32LL * RT - 1) / (32 * RT) * ((n + 64LL * CT - 1) / (64 * CT)) * splits;                   \
    if (tiles > (1 << 30)) return -1;                                                                                       \
    split_f32_kernel<RT, CT><<<(unsigned)((tiles + SPLIT_XCDS - 1) / SPLIT_XCDS * SPLIT_XCDS), 512, 0, stream>>>(args);     \
    VELOX_RETURN_LAUNCH_STATUS();                                                                                           \
  }
  switch (tile) { SPLIT(4, 4) SPLIT(4, 3) SPLIT(3, 3) SPLIT(2, 4) SPLIT(2, 2) SPLIT(2, 1) SPLIT(1, 2) }
#undef SPLIT
  return -1;
}
