// Many small bfloat16 products in one launch on the matrix cores of gfx950: a product per group (an expert, a head), each
// over its own rows, out[r, g, :] = W_g a[r, g, :].  Shared by the routed experts and the per-head products of
// attention over a latent.
//
// A workgroup of four waves of the kernel without a plan owns 64 rows and 64 NT output columns of one group (NT = 2 or 4 tiles of W
// per wave); a wave owns 16 NT of the columns and all 64 rows: 4 NT 16x16 accumulators.  W comes straight from global memory in the layout of
// v_mfma_f32_16x16x32_bf16 (lane = 16 g + i holds indices 8 g .. 8 g + 7 of row i: 16 bytes) and is the left operand, so
// acc[j] of lane (g, i) is out[row i][column 4 g + j]; no two waves read the same W.  The rows of `a`, which all four
// waves need, pass through LDS: a step is 64 indices, 8 KB for the 64 rows, two 16-byte pieces per thread, laid out [piece][row] so
// that the 16 lanes of a lane group read 256 contiguous bytes (no bank conflicts on the reads, which are four times as many
// as the writes); two buffers, one barrier per step, the
// next step's pieces and W operands asked for before this step's matrix instructions.  Rows and columns beyond a tile's
// own read a valid row again and are never stored.  A row's sum is built in the order of k whatever else is in the tile.
//
// Requirements (checked by the callers): K % 8 == 0, row strides and offsets of `a` multiples of 8 elements, 16-byte
// aligned bases.
#pragma once
#include "common.h"
#include "tiles_mfma.h"

typedef __bf16 gm_bf16x8_t __attribute__((ext_vector_type(8)));

#define GM_ROWS 64       // rows of a tile without a plan (a plan's tiles hold 64, 128 or 192)
#define GM_FEW_COLS 32   // output columns of a workgroup of the kernel for few rows (GLU: 16)

enum { GM_PLAIN = 0, GM_GLU = 1, GM_GATE = 2, GM_ACT = 3 };

struct GroupedArgs {
  const bf16_t* a;     // element (row r, group g, k) at a[r * a_ld + g * a_group + k]
  long long a_ld, a_group;
  const bf16_t* w;     // group g's matrix at w + g * w_group: [n (GLU: 2 n)][k]
  long long w_group;
  void* out;           // element (row r, group g, col) at out[r * out_ld + g * out_group + col]
  long long out_ld, out_group;
  int n, k;
  // rows: either every group runs rows [0, m) (plan == nullptr: blockIdx.y = row tile, blockIdx.z = group), or the plan's tiles say
  // which group runs which rows
  int m;
  const int* plan;
  int plan_pairs, plan_groups, plan_max_tiles;
  const bf16_t* gate;  // GM_GATE: times sigmoid(gate[r * gate_ld + g * gate_group + col * gate_col]); (n, 1) is a number per output, (1, 0) one per group
  long long gate_ld, gate_group, gate_col;
  int act = 0;         // GM_ACT: the result goes through ungated_act(., act)
  const float* row_scale;  // grouped_mfma_few_rows_kernel: row r of `a` times row_scale[order[r]], rounded to bfloat16, takes its place (nullptr: none)
  int gather_top = 0;      // with a plan: > 0: sorted row r is row order[r] / gather_top of `a`
  GluUnit unit = {1.f, INFINITY, 0.f};  // GM_GLU: the unit's middle (see glu_middle)
};

__device__ __forceinline__ gm_bf16x8_t gm_load(const bf16_t* p, bool ok) {
  if (!ok) {
    const float4_t z = {0.f, 0.f, 0.f, 0.f};
    return __builtin_bit_cast(gm_bf16x8_t, z);
  }
  return __builtin_bit_cast(gm_bf16x8_t, *reinterpret_cast<const float4_t*>(p));
}

template <int EPI, typename TO, int GM_NT>
__global__ void __launch_bounds__(256) grouped_mfma_kernel(const GroupedArgs args) {
  static_assert(EPI == GM_PLAIN || EPI == GM_GATE, "no other epilogue here");
  constexpr int GM_COLS = 64 * GM_NT;    // output columns of the workgroup
  constexpr int MT = GM_ROWS / 16, HALVES = 2, STEP = 32 * HALVES;
  __shared__ float4_t a_lds[2][HALVES][4 * GM_ROWS];
  const int group = blockIdx.z, row0 = blockIdx.y * GM_ROWS, rows = min(GM_ROWS, args.m - row0);
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int i = lane & 15, g4 = lane >> 4;
  const int n = args.n, k = args.k;
  int col0[GM_NT];  // the first output columns of the tiles of W this wave owns
#pragma unroll
  for (int t = 0; t < GM_NT; ++t) col0[t] = blockIdx.x * GM_COLS + wave * (16 * GM_NT) + t * 16;
  const bf16_t* w_base = args.w + (size_t)group * args.w_group;
  const bf16_t* w_row[GM_NT];
#pragma unroll
  for (int t = 0; t < GM_NT; ++t) {
    const int col = min(col0[t] + i, n - 1);
    w_row[t] = w_base + (size_t)col * k + 8 * g4;
  }
  // this thread's piece of the rows of `a`: row tid / 4, indices 8 (tid % 4) .. + 7 of a half; in LDS [part][row], so that a
  // row tile's operand reads are 256 contiguous bytes per 16 lanes
  const int a_part = 8 * (tid & 3);
  const bf16_t* a_piece = args.a + (size_t)(row0 + min(tid >> 2, rows - 1)) * args.a_ld + (size_t)group * args.a_group + a_part;
  const int a_slot = (tid & 3) * GM_ROWS + (tid >> 2);
  float4_t acc[GM_NT][MT];
#pragma unroll
  for (int t = 0; t < GM_NT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = float4_t{0.f, 0.f, 0.f, 0.f};

  gm_bf16x8_t w_cur[HALVES][GM_NT], w_next[HALVES][GM_NT];
#pragma unroll
  for (int u = 0; u < HALVES; ++u) {
#pragma unroll
    for (int t = 0; t < GM_NT; ++t) w_cur[u][t] = gm_load(w_row[t] + 32 * u, 32 * u + 8 * g4 < k);
    a_lds[0][u][a_slot] = __builtin_bit_cast(float4_t, gm_load(a_piece + 32 * u, 32 * u + a_part < k));
  }
  __syncthreads();
  int buffer = 0;
  for (int k0 = 0; k0 < k; k0 += STEP) {
    gm_bf16x8_t a_next[HALVES];
#pragma unroll
    for (int u = 0; u < HALVES; ++u) {
      const int at = k0 + STEP + 32 * u;
#pragma unroll
      for (int t = 0; t < GM_NT; ++t) w_next[u][t] = gm_load(w_row[t] + at, at + 8 * g4 < k);
      a_next[u] = gm_load(a_piece + at, at + a_part < k);
    }
#pragma unroll
    for (int u = 0; u < HALVES; ++u) {
      gm_bf16x8_t a_cur[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) a_cur[mt] = __builtin_bit_cast(gm_bf16x8_t, a_lds[buffer][u][g4 * GM_ROWS + mt * 16 + i]);
#pragma unroll
      for (int t = 0; t < GM_NT; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w_cur[u][t], a_cur[mt], acc[t][mt], 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < HALVES; ++u) a_lds[buffer ^ 1][u][a_slot] = __builtin_bit_cast(float4_t, a_next[u]);
    __syncthreads();
    buffer ^= 1;
#pragma unroll
    for (int u = 0; u < HALVES; ++u)
#pragma unroll
      for (int t = 0; t < GM_NT; ++t) w_cur[u][t] = w_next[u][t];
  }

  // A lane holds four neighbouring outputs of a row: one store, and one load of their gates, where the rows are laid out for it.
  // (Element by element the per-head products were bound by their stores and gates, not by what they move.  Measured on
  // MI355X, 2,500 rows, 32 heads: 224 -> 128 with a gate per output 53.5 -> 28.2 us, 96 -> 224 45.9 -> 23.7; 16 rows 7.4 -> 5.8 and
  // 6.1 -> 4.9.)
  typedef TO Four __attribute__((ext_vector_type(4)));
  TO* out = reinterpret_cast<TO*>(args.out);
  const bool vec = ((n | args.out_ld | args.out_group) & 3) == 0 && ((uintptr_t)args.out & (sizeof(Four) - 1)) == 0;
  const bool gate_vec = EPI == GM_GATE && args.gate_col == 1 && ((args.gate_ld | args.gate_group) & 3) == 0 && ((uintptr_t)args.gate & 7) == 0;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int r = mt * 16 + i;
    if (r >= rows) continue;
    const size_t out_row = (size_t)(row0 + r) * args.out_ld + (size_t)group * args.out_group;
#pragma unroll
    for (int t = 0; t < GM_NT; ++t) {
      const int col = col0[t] + 4 * g4;
      if (col >= n) continue;
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = acc[t][mt][j];
      if (EPI == GM_GATE) {
        const bf16_t* gate = args.gate + (size_t)(row0 + r) * args.gate_ld + (size_t)group * args.gate_group;
        float z[4];
        if (gate_vec && vec) {
          const short4_t held = *reinterpret_cast<const short4_t*>(gate + col);
#pragma unroll
          for (int j = 0; j < 4; ++j) z[j] = __uint_as_float(((uint32_t)(uint16_t)held[j]) << 16);
        } else if (args.gate_col == 0) {
          z[0] = z[1] = z[2] = z[3] = to_f32(gate[0]);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) z[j] = to_f32(gate[(size_t)min(col + j, n - 1) * args.gate_col]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] *= 1.f / (1.f + expf(-z[j]));
      }
      if (vec) {
        Four four;
#pragma unroll
        for (int j = 0; j < 4; ++j) four[j] = from_f32<TO>(v[j]);
        *reinterpret_cast<Four*>(out + out_row + col) = four;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (col + j < n) out[out_row + col + j] = from_f32<TO>(v[j]);
      }
    }
  }
}

// The same products when no tile has more than 64 rows (a decode step's pairs, with a plan): then a product is bound by reading
// W once, and what counts is how many loads are in flight.  A workgroup owns 32 output columns (GLU: 16 gate columns and
// their up columns) of one tile; its four waves split K into quarters, each wave asks for four steps' operands at once, W's a
// round ahead, and the waves' sums are added through LDS in the order of the waves (no atomics: the same result on every
// run).  A tile works as many 16-row tiles as it has rows, whatever the step's number of pairs would allow.  With `row_scale` the
// rows are scaled in registers, behind the wait for them and before that for W: the same bits as a scaled copy.  Measured on MI355X, us of a
// layer's routed experts with W in pieces of 64 bytes through the caches / in lines past them / with every wave's quarter of K beginning on a
// line (1,408 indices: 384, 384, 384 and 256 instead of four times 352, which begins two of them in the middle of a line): 64 pairs over 32 experts of
// 4,096 -> 1,408 -> 4,096 (W: 650 + 325 MB) 202 / 190 / 181, 24 pairs over 16 of 2,048 -> 1,408 -> 2,048 61.0 / 56.5 / 53.9.
template <int EPI, typename TO, int MT, bool LINES>
__device__ __forceinline__ void few_rows_tile(const GroupedArgs& args, const int group, const int row0, const int rows, const int* order,
                                              float4_t (*partial)[8][64]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = lane & 15, g4 = lane >> 4;
  const int n = args.n, k = args.k;
  int col0[2];
  col0[0] = blockIdx.x * (EPI == GM_GLU ? GM_FEW_COLS / 2 : GM_FEW_COLS);
  col0[1] = EPI == GM_GLU ? col0[0] : col0[0] + 16;
  const bf16_t* w_base = args.w + (size_t)group * args.w_group;
  // LINES (k % 64 == 0): W in whole cache lines, see rows_from_lines; a pair of loads is two steps of 32 indices
  const int piece = LINES ? 8 * (g4 + 4 * (i >> 3)) : 8 * g4;
  const bf16_t* w_row[2][LINES ? 2 : 1];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int half = 0; half < (LINES ? 2 : 1); ++half) {
      const int col = min(col0[t] + (LINES ? 8 * half + (i & 7) : i), n - 1);
      w_row[t][half] = w_base + (size_t)(EPI == GM_GLU && t == 1 ? n + col : col) * k + piece;
    }
  const int quarter = LINES ? (k + 255) / 256 * 64 : (k + 127) / 128 * 32;  // indices per wave: whole steps, with LINES whole lines of W
  const int k_begin = wave * quarter, k_end = min(k, k_begin + quarter);
  // W is what there is to read: its next step is asked for before the current one is multiplied, and its first before the rows of
  // `a` have been looked up
  gm_bf16x8_t wv[2][4], w_next[2][4];
  auto ask = [&](int k0) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if constexpr (LINES) {
          const int at = k0 + 64 * (u / 2);
          w_next[t][u] = at + piece < k_end ? __builtin_bit_cast(gm_bf16x8_t, __builtin_nontemporal_load(reinterpret_cast<const float4_t*>(w_row[t][u % 2] + at)))
                                            : __builtin_bit_cast(gm_bf16x8_t, float4_t{0.f, 0.f, 0.f, 0.f});
        } else {
          w_next[t][u] = gm_load(w_row[t][0] + k0 + 32 * u, k0 + 32 * u + 8 * g4 < k_end);
        }
      }
  };
  auto take = [&](int t, int u) {  // steps u and u + 1
    if constexpr (LINES) {
      float4_t first = __builtin_bit_cast(float4_t, w_next[t][u]), second = __builtin_bit_cast(float4_t, w_next[t][u + 1]);
      rows_from_lines(first, second);
      wv[t][u] = __builtin_bit_cast(gm_bf16x8_t, first);
      wv[t][u + 1] = __builtin_bit_cast(gm_bf16x8_t, second);
    } else {
      wv[t][u] = w_next[t][u];
      wv[t][u + 1] = w_next[t][u + 1];
    }
  };
  ask(k_begin);
  const bf16_t* a_row[MT];
  float factor[MT];
  const bool scaled = EPI != GM_PLAIN && args.row_scale != nullptr;  // (uniform)
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    int r = row0 + min(mt * 16 + i, rows - 1);
    factor[mt] = scaled ? args.row_scale[order[r]] : 1.f;
    if (args.gather_top > 0) r = order[r] / args.gather_top;
    a_row[mt] = args.a + (size_t)r * args.a_ld + (size_t)group * args.a_group + 8 * g4;
  }
  float4_t acc[2][MT];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = float4_t{0.f, 0.f, 0.f, 0.f};
  for (int k0 = k_begin; k0 < k_end; k0 += 128) {
    gm_bf16x8_t av[MT][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (u % 2 == 0) {
#pragma unroll
        for (int t = 0; t < 2; ++t) take(t, u);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) av[mt][u] = gm_load(a_row[mt] + k0 + 32 * u, k0 + 32 * u + 8 * g4 < k_end);
    }
    ask(k0 + 128);
    if (scaled) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (k0 + 32 * u + 8 * g4 >= k_end) continue;  // (zeros stay zeros, whatever the factor is)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int e = 0; e < 8; ++e) av[mt][u][e] = from_f32<bf16_t>(to_f32(av[mt][u][e]) * factor[mt]);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[t][u], av[mt][u], acc[t][mt], 0, 0, 0);
  }
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) partial[wave - 1][t * MT + mt][lane] = acc[t][mt];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int other = 0; other < 3; ++other)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const float4_t p = partial[other][t * MT + mt][lane];
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[t][mt][j] += p[j];
      }
  TO* out = reinterpret_cast<TO*>(args.out);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int r = mt * 16 + i;
    if (r >= rows) continue;
    const size_t out_row = (size_t)(row0 + r) * args.out_ld + (size_t)group * args.out_group;
#pragma unroll
    for (int t = 0; t < (EPI == GM_GLU ? 1 : 2); ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int col = col0[t] + 4 * g4 + j;
        if (col >= n) continue;
        float v = acc[t][mt][j];
        if (EPI == GM_GLU) v = glu_middle(v, acc[1][mt][j], args.unit);
        if (EPI == GM_ACT) v = ungated_act(v, args.act);
        out[out_row + col] = from_f32<TO>(v);
      }
  }
}

template <int EPI, typename TO, bool LINES>
__global__ void __launch_bounds__(256) grouped_mfma_few_rows_kernel(const GroupedArgs args) {
  static_assert(EPI == GM_PLAIN || EPI == GM_GLU || EPI == GM_ACT, "no gate here");
  __shared__ float4_t partial[3][8][64];
  const int tile = blockIdx.y;
  if (tile >= args.plan[0]) return;  // (uniform over the workgroup)
  const int* starts = args.plan + 1;
  const int* order = starts + args.plan_groups + 1;
  const int* tile_group = order + 2 * (size_t)args.plan_pairs;
  const int* tile_row = tile_group + args.plan_max_tiles;
  const int group = tile_group[tile], row0 = tile_row[tile];
  const int rows = min(64, starts[group + 1] - row0);
  // (the same for the whole workgroup)
  if (rows <= 16) few_rows_tile<EPI, TO, 1, LINES>(args, group, row0, rows, order, partial);
  else if (rows <= 32) few_rows_tile<EPI, TO, 2, LINES>(args, group, row0, rows, order, partial);
  else few_rows_tile<EPI, TO, 4, LINES>(args, group, row0, rows, order, partial);
}

// Tiles of the plan, as far as the host can tell: an expert's rows taken to lie evenly between 0.65 and 1.35 of their mean (16 experts, 2,072
// pairs in tiles of 128 and 192 rows: 24 and 16, found 23 to 26 and 16 to 17; 32 experts, 10,000 pairs 94 and 69, found 94 to 98 and 64 to 68).
static inline float plan_tiles_expected(int pairs, int experts, int tile_rows) {
  const float mean = (float)pairs / experts, low = 0.65f * mean, high = 1.35f * mean;
  float tiles = 1.f;  // sum over t of the chance of more than t tiles
  for (int t = 1; t * tile_rows < high; ++t) tiles += fminf(1.f, (high - t * tile_rows) / (high - low));
  return experts * tiles;
}

// The rows of a tile of the plan's products: 64 up to 64 pairs, above 128 or 192 (tiles_mfma.h's kernel), whichever is likely to cost less with as many
// tiles as are expected, as wide as they are then taken.  (Where a router sends all tokens to as few experts as it can the other one may be the
// quicker: 8,192 pairs on 8 of 64 experts 118 and 129 us.)  (us of the two products in tiles of 128 and 192 rows: 16 experts of 2,048 -> 1,408, 600
// pairs 70.2 and 75.6, 2,072 96 and 82, 3,000 99 and 112, 4,000 117 and 113, 6,000 153 and 139; 32 of 4,096 -> 1,408, 1,340 pairs 230 and 242, 4,000 316 and
// 288, 10,000 517 and 466).  k % 64 != 0 is built for 128.  Experts with 2 GiB or more from a gate row to its up row, which the large tiles' loads do not
// reach, stay with 64 rows at any number of pairs.  (Tiles of 64 rows were no quicker at any number of pairs above 64: 12 rows per expert
// 66 us either way, 56: 80 / 81, 75: 100 / 83, 130: 127 / 125, 256: 187 / 155, 16 experts of 2,048 -> 1,408 -> 2,048.)
static inline int grouped_tile_rows(int pairs, int experts, int inter, int hidden, int branches) {
  if (pairs <= 64 || !tiles_fit(256, hidden, branches == 2 ? inter + 256LL : 256, hidden) || !tiles_fit(256, inter, 256, inter)) return 64;
  if (inter % 64 != 0 || hidden % 64 != 0) return 128;
  float cost[2];
  for (int rt = 2; rt <= 3; ++rt) {
    const float tiles = plan_tiles_expected(pairs, experts, 64 * rt);
    auto product = [&](int w_rows, int k) {
      const int ct = plan_tile_cols((int)(tiles + 0.5f), w_rows), least = ct < rt ? ct : rt, most = ct < rt ? rt : ct;  // (3 x 2 costs what 2 x 3 does)
      const TileCost* t = TILE_COSTS;
      while (t->rt != least || t->ct != most) ++t;
      return tiles_cost_of(*t, tiles * ((w_rows + 64 * ct - 1) / (64 * ct)), k, 1);
    };
    cost[rt - 2] = product(branches * inter, hidden) + product(hidden, inter);
  }
  return cost[1] < cost[0] ? 192 : 128;
}

template <int EPI, typename TO>
static void grouped_tiles_launch(const TileArgs& tiles, int tile_rows, int workgroups, hipStream_t stream) {
#define SHAPES(GATHER)                                                                                                                 \
  if (tiles.k % 64 != 0) tiles_kernel<2, 4, 3, EPI, TO, true, GATHER, true><<<workgroups, 256, 0, stream>>>(tiles);                  \
  else if (tile_rows == 192) plan_tiles_kernel<3, EPI, TO, GATHER><<<workgroups, 256, 0, stream>>>(tiles);                           \
  else plan_tiles_kernel<2, EPI, TO, GATHER><<<workgroups, 256, 0, stream>>>(tiles);
  if constexpr (EPI != TL_PLAIN) {
    if (tiles.gather_top > 0) {
      SHAPES(true)
      return;
    }
  }
  SHAPES(false)
#undef SHAPES
}

template <int EPI, typename TO>
static int grouped_plan_launch(const GroupedArgs& args, int tile_rows, int most_tiles, hipStream_t stream) {
  if (tile_rows == 64) {
    constexpr int COLS = EPI == GM_GLU ? GM_FEW_COLS / 2 : GM_FEW_COLS;
    const dim3 grid((args.n + COLS - 1) / COLS, most_tiles);
    if (args.k % 64 == 0) grouped_mfma_few_rows_kernel<EPI, TO, true><<<grid, 256, 0, stream>>>(args);
    else grouped_mfma_few_rows_kernel<EPI, TO, false><<<grid, 256, 0, stream>>>(args);
    return (int)hipGetLastError();
  }
  TileArgs tiles = {};
  tiles.a = args.a;
  tiles.a_ld = args.a_ld;
  tiles.w = args.w;
  tiles.w_group = args.w_group;
  tiles.out = args.out;
  tiles.n = args.n;
  tiles.k = args.k;
  tiles.splits = 1;
  tiles.plan = args.plan;
  tiles.plan_pairs = args.plan_pairs;
  tiles.plan_groups = args.plan_groups;
  tiles.plan_max_tiles = args.plan_max_tiles;
  tiles.gather_top = args.gather_top;
  tiles.act = args.act;
  tiles.unit = args.unit;
  if (!tiles_fit(args.gather_top > 0 ? args.plan_pairs / args.gather_top : 256, args.a_ld, EPI == GM_GLU ? args.n + 256LL : 256, args.k)) return -1;
  const long long most = (long long)most_tiles * (((EPI == GM_GLU ? 2LL : 1LL) * args.n + 127) / 128);  // (of the narrowest)
  const int workgroups = (int)(most < TL_WORKGROUPS ? (most + TL_XCDS - 1) / TL_XCDS * TL_XCDS : TL_WORKGROUPS);
  if constexpr (EPI == GM_GLU) {
    if (args.unit.alpha == 1.f && args.unit.limit == INFINITY && args.unit.shift == 0.f) grouped_tiles_launch<TL_SILU_UNIT, TO>(tiles, tile_rows, workgroups, stream);
    else grouped_tiles_launch<TL_UNIT, TO>(tiles, tile_rows, workgroups, stream);
  } else {
    grouped_tiles_launch<EPI == GM_ACT ? TL_ACT : TL_PLAIN, TO>(tiles, tile_rows, workgroups, stream);
  }
  return (int)hipGetLastError();
}

// The products of `groups` groups that all run the same rows, where a group's matrix fits the registers of four waves: a wave keeps its 16 NT
// rows of W whole (up to 32 KC indices, asked for once) and walks 16 rows of `a` at a time, straight from memory into matrix operands, the
// next rows and their gates asked for before this step's products; no LDS and no barrier.  Bound by what it reads and writes and by the
// loads in flight: rows are dealt out so that a compute unit has about two workgroups, which reads W rarely and leaves each several
// steps.  The order of additions is that of grouped_mfma_kernel (indices beyond k are zeros).
// Measured on MI355X, 2,500 rows, 32 heads of 224 x 96: 24.2 -> 17.9 us (51 MB: 2.1 -> 2.9 TB/s).
// Needs k <= 32 KC and four outputs of a row and of its gates on 8-byte boundaries (GM_GATE with gate_col == 0: any).
template <int EPI>
__global__ void __launch_bounds__(256) head_rows_kernel(const GroupedArgs args, int rows_each) {
  static_assert(EPI == GM_PLAIN || EPI == GM_GATE, "no other epilogue here");
  constexpr int NT = 4, KC = 4;
  const int group = blockIdx.z, first = blockIdx.y * rows_each, last = min(args.m, first + rows_each);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, g4 = lane >> 4;
  const int n = args.n, k = args.k, col0 = (blockIdx.x * 4 + wave) * (16 * NT);
  if (col0 >= n) return;  // (the whole wave)
  const bf16_t* w = args.w + (size_t)group * args.w_group + 8 * g4;
  const bf16_t* a = args.a + (size_t)group * args.a_group + 8 * g4;
  const bf16_t* gate = EPI == GM_GATE ? args.gate + (size_t)group * args.gate_group : nullptr;
  bf16_t* out = reinterpret_cast<bf16_t*>(args.out) + (size_t)group * args.out_group;
  gm_bf16x8_t w_op[NT][KC], a_next[KC], a_op[KC];
  short4_t gate_next[NT], gate_now[NT];
  auto ask = [&](int row0) {
    const size_t row = min(row0 + i, last - 1);
#pragma unroll
    for (int c = 0; c < KC; ++c) a_next[c] = gm_load(a + row * args.a_ld + 32 * c, 32 * c + 8 * g4 < k);
    if constexpr (EPI == GM_GATE) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const bf16_t* from = gate + row * args.gate_ld + (args.gate_col == 0 ? 0 : min(col0 + 16 * t + 4 * g4, n - 4));
        if (args.gate_col == 0) gate_next[t][0] = __builtin_bit_cast(short, *from);
        else gate_next[t] = *reinterpret_cast<const short4_t*>(from);
      }
    }
  };
  ask(first);
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int c = 0; c < KC; ++c) w_op[t][c] = gm_load(w + (size_t)min(col0 + 16 * t + i, n - 1) * k + 32 * c, 32 * c + 8 * g4 < k);
  for (int row0 = first; row0 < last; row0 += 16) {
#pragma unroll
    for (int c = 0; c < KC; ++c) a_op[c] = a_next[c];
    if constexpr (EPI == GM_GATE) {
#pragma unroll
      for (int t = 0; t < NT; ++t) gate_now[t] = gate_next[t];
    }
    if (row0 + 16 < last) ask(row0 + 16);
    float4_t acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w_op[t][c], a_op[c], acc[t], 0, 0, 0);
    if (row0 + i >= last) continue;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int col = col0 + 16 * t + 4 * g4;
      if (col >= n) continue;
      typedef bf16_t Four __attribute__((ext_vector_type(4)));
      Four four;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v = acc[t][j];
        if (EPI == GM_GATE) {
          const float z = __uint_as_float(((uint32_t)(uint16_t)gate_now[t][args.gate_col == 0 ? 0 : j]) << 16);
          v *= 1.f / (1.f + expf(-z));
        }
        four[j] = from_f32<bf16_t>(v);
      }
      *reinterpret_cast<Four*>(out + (size_t)(row0 + i) * args.out_ld + col) = four;
    }
  }
}

// The products of `groups` groups that all run rows [0, m).
template <int EPI, typename TO>
static void grouped_rows_launch(const GroupedArgs& args, int groups, hipStream_t stream) {
  const bool fours = ((args.n | args.out_ld | args.out_group) & 3) == 0 && ((uintptr_t)args.out & 7) == 0;
  const bool gates = EPI != GM_GATE || args.gate_col == 0 || (args.gate_col == 1 && ((args.gate_ld | args.gate_group) & 3) == 0 && ((uintptr_t)args.gate & 7) == 0);
  // wide outputs of short sums, with rows enough for several steps of 16 a workgroup (us, grouped_mfma_kernel / head_rows_kernel: 32 heads of
  // 224 x 96: 200 rows 7.6 / 8.1, 1,000 10.6 / 10.1, 2,500 24.2 / 17.9, 4,096 33.4 / 25.6; 128 of 512 x 128: 64 rows 9.9 / 11.2, 200 27.2 / 20.5, 1,000 75 /
  // 62, 4,096 382 / 315.  Longer sums or up to 128 outputs were not quicker in it: 32 of 128 x 224 with gates, 2,500 rows 28.0 / 30.4, 16 of 256 x 256
  // 24.7 / 27.0, 64 of 128 x 64 with gates 32.2 / 32.8)
  if (sizeof(TO) == 2 && fours && gates && args.n > 128 && args.k > 64 && args.k <= 128 && (long long)args.m * groups >= 16384) {
    const int columns = (args.n + 255) / 256, parts = max(1, 2 * TL_WORKGROUPS / (columns * groups)), rows_each = ((args.m + parts - 1) / parts + 15) / 16 * 16;
    head_rows_kernel<EPI><<<dim3(columns, (args.m + rows_each - 1) / rows_each, groups), 256, 0, stream>>>(args, rows_each);
    return;
  }
  const int row_tiles = (args.m + GM_ROWS - 1) / GM_ROWS;
  if (args.n <= 128) grouped_mfma_kernel<EPI, TO, 2><<<dim3(1, row_tiles, groups), 256, 0, stream>>>(args);
  else grouped_mfma_kernel<EPI, TO, 4><<<dim3((args.n + 255) / 256, row_tiles, groups), 256, 0, stream>>>(args);
}

// Whether the operands meet what the kernels' 16-byte loads need.
static inline bool grouped_mfma_fits(const void* a, long long a_ld, long long a_group, long long a_offset, const void* w, int k) {
  return k % 8 == 0 && a_ld % 8 == 0 && a_group % 8 == 0 && a_offset % 8 == 0 && ((uintptr_t)a) % 16 == 0 && ((uintptr_t)w) % 16 == 0;
}
