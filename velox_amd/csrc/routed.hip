// Routed experts for gfx950: nothing about a step's routing is known to the host.
//
//   route_top:       scores of the router's float32 logits and the `top` largest per token
//   routed_plan:     the step's (token, choice) pairs sorted by expert, and the list of row tiles that the grouped products
//                    run: one workgroup, counters in LDS
//   grouped_glu:     act[p, :] = silu(Wgate_e a_p) * (Wup_e a_p) for every sorted pair p of expert e, a_p = x[token of p]
//                    (times the pair's weight when the weight scales the input)
//   grouped_down:    y[p, :] = Wdown_e act[p, :] (times the pair's weight when it scales the output), float32
//   routed_combine:  out[t, :] = sum_k y[place of pair (t, k), :] (+ shared[t, :]), the choices in order
//
// The grouped products are launched for the most tiles a step of its size can have; a workgroup beyond the step's own
// number of tiles (read from the plan) exits at once.  A row's result is summed over k in one fixed order by one thread,
// whatever other rows share its tile, so a token's output does not depend on which tokens go to the same experts or on
// the order in which the plan's atomic counters placed them.
#include "common.h"
#include "grouped_mfma.h"

#define RT_BM 64  // rows of a tile (sorted pairs of one expert)
#define RT_BN 64
#define RT_BK 16
#define RT_PAD 4
#define RT_FOLD 128

// ---------------------------------------------------------------------------------------------
// route_top: one wave per token, its lanes over the experts.  score = sigmoid(z) or softmax(z) over all experts; the `top`
// largest scores, ties to the lower index; weights are the chosen scores, divided by their sum when `renormalize`.
// Every round the wave takes the largest score that is not yet taken (value first, then the lower index), so the choices
// come out in descending order of score.  With `correction` (float32 [experts]) the choice goes by score + correction and
// the weights stay the scores themselves.  With `group_count` > 0 the experts form that many equal groups of neighbours; a
// group's score is the sum of its two largest choice scores (of its one, if it has one expert), and only experts of the
// `group_keep` best groups (ties to the lower index) can be chosen: the others' choice scores become minus infinity.
// `norm_floor` is added to the sum that renormalised weights are divided by.
// ---------------------------------------------------------------------------------------------
#define ROUTE_PER_LANE 32  // experts per lane held in registers: up to 2,048 experts

__global__ void __launch_bounds__(256) route_top_kernel(const float* __restrict__ logits, int* __restrict__ choice, float* __restrict__ weight, int tokens,
                                                        int experts, int top, int softmax, int renormalize, const float* __restrict__ correction,
                                                        int group_count, int group_keep, float norm_floor) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= tokens) return;  // (a whole wave; nothing below crosses waves)
  const float* z = logits + (size_t)t * experts;
  float shift = 0.f, denom = 1.f;
  if (softmax) {
    float m = -INFINITY;
    for (int e = lane; e < experts; e += 64) m = fmaxf(m, z[e]);
    shift = wave_max(m);
    float sum = 0.f;
    for (int e = lane; e < experts; e += 64) sum += expf(z[e] - shift);
    denom = wave_sum(sum);
  }
  const int used = (experts + 63) >> 6;  // registers of `score` that hold experts at all: the loops below stop there
  float score[ROUTE_PER_LANE];
#pragma unroll
  for (int u = 0; u < ROUTE_PER_LANE; ++u) {
    const int e = lane + 64 * u;
    score[u] = -INFINITY;  // ("no such expert" and "taken")
    if (e < experts) {
      score[u] = softmax ? expf(z[e] - shift) / denom : 1.f / (1.f + expf(-z[e]));
      if (correction) score[u] += correction[e];
    }
  }
  if (group_count > 0) {
    // lane g ends up with group g's score (group_count <= 64); every group's two largest by two rounds over the wave
    const int per = experts / group_count;
    float mine = -INFINITY;  // (lanes beyond the groups never win)
    if (used == 1 && (per & (per - 1)) == 0) {
      // one expert per lane and groups that are aligned runs of a power of two of lanes: all groups at once, the two
      // largest of a run by exchanges inside the run
      float first = score[0], second = -INFINITY;
      for (int offset = 1; offset < per; offset <<= 1) {
        const float of = __shfl_xor(first, offset, 64), os = __shfl_xor(second, offset, 64);
        second = fmaxf(fminf(first, of), fmaxf(second, os));
        first = fmaxf(first, of);
      }
      const float sum = per > 1 ? first + second : first;
      const float of_group = __shfl(sum, (lane * per) & 63, 64);
      if (lane < group_count) mine = of_group;
    } else
    for (int gidx = 0; gidx < group_count; ++gidx) {
      const int lo = gidx * per, hi = lo + per;
      float first = -INFINITY, second = -INFINITY;  // this lane's two largest inside the group
#pragma unroll
      for (int u = 0; u < ROUTE_PER_LANE; ++u) {
        if (u >= used) break;
        const int e = lane + 64 * u;
        if (e >= lo && e < hi) {
          const float v = score[u];
          if (v > first) { second = first; first = v; }
          else if (v > second) second = v;
        }
      }
      // the wave's two largest: merge (first, second) pairs
#pragma unroll
      for (int offset = 32; offset > 0; offset >>= 1) {
        const float of = __shfl_xor(first, offset, 64), os = __shfl_xor(second, offset, 64);
        const float hi1 = fmaxf(first, of);
        const float lo1 = fminf(first, of);
        second = fmaxf(lo1, fmaxf(second, os));
        first = hi1;
      }
      const float sum = per > 1 ? first + second : first;
      if (lane == gidx) mine = sum;
    }
    unsigned long long allowed = 0ull;
    for (int k = 0; k < group_keep; ++k) {
      float best = mine;
      int best_g = lane < group_count ? lane : 0x7fffffff;
      if (lane >= group_count || ((allowed >> lane) & 1ull)) { best = -INFINITY; best_g = 0x7fffffff; }
#pragma unroll
      for (int offset = 32; offset > 0; offset >>= 1) {
        const float other = __shfl_xor(best, offset, 64);
        const int other_g = __shfl_xor(best_g, offset, 64);
        if (other > best || (other == best && other_g < best_g)) { best = other; best_g = other_g; }
      }
      if (best_g < group_count) allowed |= 1ull << best_g;
      else {  // (every group left scores minus infinity or NaN: take the lowest group not yet taken)
        for (int gidx = 0; gidx < group_count; ++gidx)
          if (!((allowed >> gidx) & 1ull)) { allowed |= 1ull << gidx; break; }
      }
    }
#pragma unroll
    for (int u = 0; u < ROUTE_PER_LANE; ++u) {
      if (u >= used) break;
      const int e = lane + 64 * u;
      if (e < experts && !((allowed >> (e / per)) & 1ull)) score[u] = -INFINITY;
    }
  }
  float total = 0.f;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int best_e = 0x7fffffff;
#pragma unroll
    for (int u = 0; u < ROUTE_PER_LANE; ++u) {
      if (u >= used) break;
      if (score[u] > best) { best = score[u]; best_e = lane + 64 * u; }  // (ascending e within a lane: the first of equals stays)
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
      const float other = __shfl_xor(best, offset, 64);
      const int other_e = __shfl_xor(best_e, offset, 64);
      if (other > best || (other == best && other_e < best_e)) { best = other; best_e = other_e; }
    }
#pragma unroll
    for (int u = 0; u < ROUTE_PER_LANE; ++u) {
      if (u >= used) break;
      if (lane + 64 * u == best_e) score[u] = -INFINITY;
    }
    // (the weight is the score without the correction: the same expression as above, so the same value)
    if (best_e >= experts) best_e = 0;  // (only when every score left is a NaN: stay inside the row)
    if (correction) best = softmax ? expf(z[best_e] - shift) / denom : 1.f / (1.f + expf(-z[best_e]));
    total += best;
    if (lane == 0) {
      choice[(size_t)t * top + k] = best_e;
      weight[(size_t)t * top + k] = best;
    }
  }
  if (renormalize && lane == 0)  // (the lane that wrote them)
    for (int k = 0; k < top; ++k) weight[(size_t)t * top + k] /= (total + norm_floor);
}

extern "C" int velox_route_top(const float* logits, int* choice, float* weight, int tokens, int experts, int top, int softmax, int renormalize,
                               const float* correction, int group_count, int group_keep, float norm_floor, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (experts < 1 || experts > 64 * ROUTE_PER_LANE || top < 1 || top > experts) return -1;
  if (group_count < 0 || group_count > 64 ||
      (group_count > 0 && (experts % group_count != 0 || group_keep < 1 || group_keep > group_count || group_keep * (experts / group_count) < top)))
    return -1;
  route_top_kernel<<<(tokens + 3) / 4, 256, 0, stream>>>(logits, choice, weight, tokens, experts, top, softmax, renormalize, correction, group_count,
                                                         group_keep, norm_floor);
  VELOX_RETURN_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------------------------
// The plan, int32: [0] number of tiles, [1 .. 1 + E] first sorted row of every expert and the total, then order[P]
// (sorted row -> pair = token * top + k), place[P] (pair -> sorted row), tile_expert[max_tiles], tile_row[max_tiles]; a tile
// is up to tile_rows consecutive sorted rows of one expert.
// ---------------------------------------------------------------------------------------------
#define PLAN_MAX_EXPERTS 2048

// One workgroup, bound by the latency of its few passes over LDS and memory: every pair takes its place among its expert's rows
// from one LDS atomic (kept in `place` until the experts' first rows are known), and the experts' first rows and tiles come from
// one scan over the experts, two a thread.  Measured on MI355X: 10,000 pairs over 32 experts 14.0 us, 64 pairs 4.7 (a serial walk
// over the experts and a second round of atomics 15.2; with the rows of x copied in the same kernel, 64 pairs of 4,096, 23.8).
__global__ void __launch_bounds__(1024) routed_plan_kernel(const int* __restrict__ choice, int pairs, int experts, int max_tiles, int tile_rows,
                                                           int* __restrict__ plan) {
  __shared__ int count[PLAN_MAX_EXPERTS];
  __shared__ int first[PLAN_MAX_EXPERTS];
  __shared__ int wave_rows[16], wave_tiles[16];
  constexpr int BATCH = 4;
  int* starts = plan + 1;
  int* order = starts + experts + 1;
  int* place = order + pairs;
  int* tile_expert = place + pairs;
  int* tile_row = tile_expert + max_tiles;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int e = tid; e < experts; e += 1024) count[e] = 0;
  __syncthreads();
  for (int p0 = tid; p0 < pairs; p0 += 1024 * BATCH) {
    int e[BATCH];
#pragma unroll
    for (int j = 0; j < BATCH; ++j) e[j] = p0 + 1024 * j < pairs ? choice[p0 + 1024 * j] : -1;
#pragma unroll
    for (int j = 0; j < BATCH; ++j)
      if (p0 + 1024 * j < pairs) place[p0 + 1024 * j] = e[j] >= 0 && e[j] < experts ? atomicAdd(&count[e[j]], 1) : -1;
  }
  __syncthreads();
  {
    int rows[2], tiles[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      rows[j] = 2 * tid + j < experts ? count[2 * tid + j] : 0;
      tiles[j] = (rows[j] + tile_rows - 1) / tile_rows;
    }
    int row_at = rows[0] + rows[1], tile_at = tiles[0] + tiles[1];  // inclusive sums over the wave, then exclusive over the workgroup
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) {
      const int r = __shfl_up(row_at, offset, VELOX_WAVE), t = __shfl_up(tile_at, offset, VELOX_WAVE);
      if (lane >= offset) {
        row_at += r;
        tile_at += t;
      }
    }
    if (lane == 63) {
      wave_rows[wave] = row_at;
      wave_tiles[wave] = tile_at;
    }
    __syncthreads();
    for (int w = 0; w < wave; ++w) {
      row_at += wave_rows[w];
      tile_at += wave_tiles[w];
    }
    if (tid == 1023) {
      plan[0] = min(tile_at, max_tiles);
      starts[experts] = row_at;
    }
    row_at -= rows[0] + rows[1];
    tile_at -= tiles[0] + tiles[1];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int e = 2 * tid + j;
      if (e < experts) {
        first[e] = row_at;
        starts[e] = row_at;
        for (int t = 0; t < tiles[j] && tile_at + t < max_tiles; ++t) {
          tile_expert[tile_at + t] = e;
          tile_row[tile_at + t] = row_at + t * tile_rows;
        }
      }
      row_at += rows[j];
      tile_at += tiles[j];
    }
  }
  __syncthreads();
  for (int p0 = tid; p0 < pairs; p0 += 1024 * BATCH) {
    int e[BATCH], rank[BATCH];
#pragma unroll
    for (int j = 0; j < BATCH; ++j) {
      const int p = p0 + 1024 * j < pairs ? p0 + 1024 * j : p0;
      e[j] = choice[p];
      rank[j] = place[p];
    }
#pragma unroll
    for (int j = 0; j < BATCH; ++j) {
      const int p = p0 + 1024 * j;
      if (p >= pairs || rank[j] < 0) continue;
      const int row = first[e[j]] + rank[j];
      order[row] = p;
      place[p] = row;
    }
  }
}

extern "C" long long velox_routed_plan_elems(int pairs, int experts) {
  const long long max_tiles = (pairs + RT_BM - 1) / RT_BM + experts;
  return 1 + (experts + 1) + 2LL * pairs + 2 * max_tiles;
}

extern "C" int velox_routed_max_tiles(int pairs, int experts) { return (pairs + RT_BM - 1) / RT_BM + experts; }

// tile_rows: 64, or what velox_routed_tile_rows says for the matrix-core products.  The plan's layout is that of 64-row tiles either way
// (the most tiles there can be).
extern "C" int velox_routed_plan(const int* choice, int pairs, int experts, int* plan, int tile_rows, hipStream_t stream) {
  if (pairs <= 0) return 0;
  if (experts < 1 || experts > PLAN_MAX_EXPERTS || (tile_rows != RT_BM && tile_rows != 2 * RT_BM && tile_rows != 3 * RT_BM)) return -1;
  routed_plan_kernel<<<1, 1024, 0, stream>>>(choice, pairs, experts, velox_routed_max_tiles(pairs, experts), tile_rows, plan);
  VELOX_RETURN_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------------------------
// The grouped products.  GLU: two tiles of W (gate rows and the up rows of the same columns), the activation as the
// epilogue.  Rows of A: GLU gathers x[token] (scaled by the pair's weight and rounded to T, as a product on T operands
// would read it); the down product reads the sorted rows of act.  FIRST = 2: a unit without a gate branch, one tile of
// W (the up rows), rows gathered as for GLU, ungated_act(., act_kind) as the epilogue.
// ---------------------------------------------------------------------------------------------
template <typename T, typename TO, int FIRST>
__global__ void __launch_bounds__(256) grouped_product_kernel(const T* __restrict__ a, const T* __restrict__ w, TO* __restrict__ out,
                                                              const int* __restrict__ plan, const float* __restrict__ pair_weight, int pairs, int experts,
                                                              int max_tiles, int top, int n, int k, int scale_rows, int a_vec, int w_vec, GluUnit unit,
                                                              int act_kind) {
  constexpr bool GLU = FIRST == 1;       // two tiles of W and the gated epilogue
  constexpr bool GATHERS = FIRST != 0;   // rows are x[token of the pair], not sorted rows
  __shared__ float a_tile[RT_BK][RT_BM + RT_PAD];
  __shared__ float w_tile[GLU ? 2 : 1][RT_BK][RT_BN + RT_PAD];
  __shared__ int row_pair[RT_BM];
  const int tile = blockIdx.y;
  if (tile >= plan[0]) return;  // (uniform over the workgroup)
  const int* starts = plan + 1;
  const int* order = starts + experts + 1;
  const int* tile_expert = order + 2 * (size_t)pairs;
  const int* tile_row = tile_expert + max_tiles;
  const int e = tile_expert[tile];
  const int row0 = tile_row[tile];
  const int rows = min(RT_BM, starts[e + 1] - row0);
  const int tid = threadIdx.x;
  const int tx = tid % 16, ty = tid / 16;
  const int n0 = blockIdx.x * RT_BN;
  const int load_row = tid / 4, load_k = (tid % 4) * 4;
  if (tid < RT_BM) row_pair[tid] = tid < rows ? order[row0 + tid] : -1;
  __syncthreads();
  const bool a_row_ok = load_row < rows;
  const int my_pair = row_pair[load_row];
  size_t a_off = 0;
  float a_scale = 1.f;
  if (a_row_ok) {
    if (GATHERS) {
      a_off = (size_t)(my_pair / top) * k;
      if (scale_rows) a_scale = pair_weight[my_pair];
    } else {
      a_off = (size_t)(row0 + load_row) * k;
    }
  }
  const bool w_row_ok = n0 + load_row < n;
  const size_t w_rows = GLU ? 2 * (size_t)n : (size_t)n;  // rows of one expert's matrix
  const size_t w_off = ((size_t)e * w_rows + n0 + load_row) * k;
  const size_t up_off = w_off + (size_t)n * k;

  constexpr int NW = GLU ? 2 : 1;
  float acc[NW][4][4], total[NW][4][4];
#pragma unroll
  for (int u = 0; u < NW; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[u][i][j] = total[u][i][j] = 0.f;

  for (int k0 = 0; k0 < k; k0 += RT_BK) {
    if (k0 % RT_FOLD == 0) {
#pragma unroll
      for (int u = 0; u < NW; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            total[u][i][j] += acc[u][i][j];
            acc[u][i][j] = 0.f;
          }
    }
    float av[4], wv[NW][4];
    load4<T>(a, a_off, k0 + load_k, k, a_row_ok, a_vec != 0, av);
    if (GATHERS && scale_rows) {
#pragma unroll
      for (int i = 0; i < 4; ++i) av[i] = to_f32(from_f32<T>(av[i] * a_scale));
    }
    load4<T>(w, w_off, k0 + load_k, k, w_row_ok, w_vec != 0, wv[0]);
    if (GLU) load4<T>(w, up_off, k0 + load_k, k, w_row_ok, w_vec != 0, wv[NW - 1]);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a_tile[load_k + i][load_row] = av[i];
#pragma unroll
      for (int u = 0; u < NW; ++u) w_tile[u][load_k + i][load_row] = wv[u][i];
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < RT_BK; ++kk) {
      const float4_t ar = *reinterpret_cast<const float4_t*>(&a_tile[kk][ty * 4]);
#pragma unroll
      for (int u = 0; u < NW; ++u) {
        const float4_t wr = *reinterpret_cast<const float4_t*>(&w_tile[u][kk][tx * 4]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[u][i][j] = fmaf(ar[i], wr[j], acc[u][i][j]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = ty * 4 + i;
    if (r >= rows) continue;
    const float row_scale = (!GATHERS && scale_rows) ? pair_weight[row_pair[r]] : 1.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = n0 + tx * 4 + j;
      if (col >= n) continue;
      float v = total[0][i][j] + acc[0][i][j];
      if (GLU) {
        const float up = total[NW - 1][i][j] + acc[NW - 1][i][j];
        v = glu_middle(v, up, unit);  // (float32 throughout, one rounding at the store)
      } else if (FIRST == 2) {
        v = ungated_act(v, act_kind);
      } else {
        v *= row_scale;
      }
      out[(size_t)(row0 + r) * n + col] = from_f32<TO>(v);
    }
  }
}

extern "C" int velox_grouped_glu(const void* x, const void* gate_up, void* act, const int* plan, const float* pair_weight, int pairs, int experts, int top,
                                 int inter, int hidden, int scale_input, int dtype, float alpha, float limit, float shift, int ungated, hipStream_t stream) {
  // `ungated` > 0: `gate_up` holds [experts * inter, hidden] (up rows only) and the unit is ungated_act(up, ungated)
  if (pairs <= 0) return 0;
  const GluUnit unit = {alpha, limit, shift};
  const int max_tiles = velox_routed_max_tiles(pairs, experts);
  dim3 grid((inter + RT_BN - 1) / RT_BN, max_tiles);
  if (grid.y > 65535) return -1;
  const int size = dtype == VELOX_BF16 ? 2 : 4;
  const int a_vec = hidden % 4 == 0 && ((uintptr_t)x) % (4 * size) == 0;
  const int w_vec = hidden % 4 == 0 && ((uintptr_t)gate_up) % (4 * size) == 0;
  if (ungated > 0) {
    if (dtype == VELOX_BF16)
      grouped_product_kernel<bf16_t, bf16_t, 2><<<grid, 256, 0, stream>>>((const bf16_t*)x, (const bf16_t*)gate_up, (bf16_t*)act, plan, pair_weight, pairs, experts,
                                                                          max_tiles, top, inter, hidden, scale_input, a_vec, w_vec, unit, ungated);
    else
      grouped_product_kernel<float, float, 2><<<grid, 256, 0, stream>>>((const float*)x, (const float*)gate_up, (float*)act, plan, pair_weight, pairs, experts,
                                                                        max_tiles, top, inter, hidden, scale_input, a_vec, w_vec, unit, ungated);
    VELOX_RETURN_LAUNCH_STATUS();
  }
  if (dtype == VELOX_BF16)
    grouped_product_kernel<bf16_t, bf16_t, 1><<<grid, 256, 0, stream>>>((const bf16_t*)x, (const bf16_t*)gate_up, (bf16_t*)act, plan, pair_weight, pairs, experts,
                                                                        max_tiles, top, inter, hidden, scale_input, a_vec, w_vec, unit, 0);
  else
    grouped_product_kernel<float, float, 1><<<grid, 256, 0, stream>>>((const float*)x, (const float*)gate_up, (float*)act, plan, pair_weight, pairs, experts,
                                                                      max_tiles, top, inter, hidden, scale_input, a_vec, w_vec, unit, 0);
  VELOX_RETURN_LAUNCH_STATUS();
}

extern "C" int velox_grouped_down(const void* act, const void* down, float* y, const int* plan, const float* pair_weight, int pairs, int experts, int top,
                                  int hidden, int inter, int scale_output, int dtype, hipStream_t stream) {
  if (pairs <= 0) return 0;
  const int max_tiles = velox_routed_max_tiles(pairs, experts);
  dim3 grid((hidden + RT_BN - 1) / RT_BN, max_tiles);
  if (grid.y > 65535) return -1;
  const int size = dtype == VELOX_BF16 ? 2 : 4;
  const int a_vec = inter % 4 == 0 && ((uintptr_t)act) % (4 * size) == 0;
  const int w_vec = inter % 4 == 0 && ((uintptr_t)down) % (4 * size) == 0;
  if (dtype == VELOX_BF16)
    grouped_product_kernel<bf16_t, float, 0><<<grid, 256, 0, stream>>>((const bf16_t*)act, (const bf16_t*)down, y, plan, pair_weight, pairs, experts, max_tiles,
                                                                       top, hidden, inter, scale_output, a_vec, w_vec, GluUnit{1.f, INFINITY, 0.f}, 0);
  else
    grouped_product_kernel<float, float, 0><<<grid, 256, 0, stream>>>((const float*)act, (const float*)down, y, plan, pair_weight, pairs, experts, max_tiles,
                                                                      top, hidden, inter, scale_output, a_vec, w_vec, GluUnit{1.f, INFINITY, 0.f}, 0);
  VELOX_RETURN_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------------------------
// bfloat16 on the matrix cores: the first product fetches the rows of x through the plan, the second reads sorted rows.  When the
// pair's weight scales the expert's input, the scaled row is rounded to bfloat16 (a float32 product, one rounding) on every path:
// a router behind it that stands near a tie then chooses alike however many pairs a step has.  Up to 64 pairs are scaled where the
// first product loads them; more are copied into the plan's order by the kernel below, 16 bytes a thread.  Bound by what it moves: a
// step of 2,500 tokens of 4 x 4,096 is about 28 us longer per layer with it than with unscaled rows, one of 64 pairs about 3 us.
// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) routed_scale_kernel(const bf16_t* __restrict__ x, const int* __restrict__ order, const float* __restrict__ pair_weight,
                                                           bf16_t* __restrict__ sorted, int top, int hidden, const int* __restrict__ placed) {
  const int row = blockIdx.x;
  if (row >= *placed) return;  // (pairs whose expert the plan leaves out have no row: `order` ends at the placed ones)
  const int pair = order[row];
  const float w = pair_weight != nullptr ? pair_weight[pair] : 1.f;
  typedef bf16_t Pieces __attribute__((ext_vector_type(8)));
  const Pieces* src = reinterpret_cast<const Pieces*>(x + (size_t)(pair / top) * hidden);
  Pieces* dst = reinterpret_cast<Pieces*>(sorted + (size_t)row * hidden);
  for (int at = threadIdx.x; at < hidden / 8; at += 256) {
    Pieces piece = src[at];
#pragma unroll
    for (int e = 0; e < 8; ++e) piece[e] = from_f32<bf16_t>(to_f32(piece[e]) * w);
    dst[at] = piece;
  }
}

static GroupedArgs routed_args(const void* a, const void* w, void* out, const int* plan, int pairs, int experts, int n, int k, int w_rows) {
  GroupedArgs args = {};
  args.a = (const bf16_t*)a;
  args.a_ld = k;
  args.w = (const bf16_t*)w;
  args.w_group = (long long)w_rows * k;
  args.out = out;
  args.out_ld = n;
  args.n = n;
  args.k = k;
  args.plan = plan;
  args.plan_pairs = pairs;
  args.plan_groups = experts;
  args.plan_max_tiles = velox_routed_max_tiles(pairs, experts);
  return args;
}

// x [T, hidden] -> (`sorted` [pairs, hidden], where velox_routed_copies_rows says so) -> act [pairs, inter] -> y [pairs, hidden]
// float32.  Needs hidden % 8 == 0, inter % 8 == 0 and x and `sorted` on 16-byte boundaries (the caller checks).  The plan's tiles hold `tile_rows` rows: 64, 128 or, of
// sizes that are multiples of 64, 192 (velox_routed_tile_rows says which is likely to be the quickest).
extern "C" int velox_routed_tile_rows(int pairs, int experts, int inter, int hidden, int branches) { return grouped_tile_rows(pairs, experts, inter, hidden, branches); }

// Whether the products read sorted copies of the rows: rows that their pair's weight scales (tiles of 64 rows do that themselves), and rows further
// apart than the large tiles' loads reach through the plan (2 GiB: from 131,072 tokens of 8,192 channels on).
extern "C" int velox_routed_copies_rows(int pairs, int top, int hidden, int tile_rows, int scale_input) {
  return tile_rows != RT_BM && (scale_input || !tiles_fit(pairs / top, hidden, 256, hidden));
}

extern "C" int velox_routed_products_bf16(const void* x, const void* gate_up, const void* down, void* sorted, void* act, float* y, const int* plan,
                                          const float* pair_weight, int pairs, int experts, int top, int inter, int hidden, int scale_input,
                                          float alpha, float limit, float shift, int ungated, int tile_rows, hipStream_t stream) {
  // `ungated` > 0: `gate_up` holds [experts * inter, hidden] (up rows only) and the unit is ungated_act(up, ungated)
  if (pairs <= 0) return 0;
  if (tile_rows != RT_BM && tile_rows != 2 * RT_BM && (tile_rows != 3 * RT_BM || hidden % 64 != 0 || inter % 64 != 0)) return -1;
  if (hidden % 8 != 0 || inter % 8 != 0 || top < 1 || ((uintptr_t)x | (uintptr_t)sorted) % 16 != 0) return -1;
  const int max_tiles = velox_routed_max_tiles(pairs, experts);
  const bool copied = velox_routed_copies_rows(pairs, top, hidden, tile_rows, scale_input);
  if (copied && sorted == nullptr) return -1;
  if (max_tiles > 65535) return -1;
  if (copied)
    routed_scale_kernel<<<pairs, 256, 0, stream>>>((const bf16_t*)x, plan + 1 + (experts + 1), scale_input ? pair_weight : nullptr, (bf16_t*)sorted, top, hidden, plan + 1 + experts);
  GroupedArgs first = routed_args(copied ? sorted : x, gate_up, act, plan, pairs, experts, inter, hidden, ungated > 0 ? inter : 2 * inter);
  first.gather_top = copied ? 0 : top;
  first.row_scale = scale_input && !copied ? pair_weight : nullptr;  // (read by the kernel for tiles of 64 rows alone)
  first.act = ungated;
  first.unit = GluUnit{alpha, limit, shift};
  const int status = ungated > 0 ? grouped_plan_launch<GM_ACT, bf16_t>(first, tile_rows, max_tiles, stream) : grouped_plan_launch<GM_GLU, bf16_t>(first, tile_rows, max_tiles, stream);
  if (status != 0) return status;
  GroupedArgs last = routed_args(act, down, y, plan, pairs, experts, hidden, inter, hidden);
  // (a weight on the experts' OUTPUT is applied where the results are added up, routed_combine with scale_rows: the product
  // itself is the same kernel either way)
  return grouped_plan_launch<GM_PLAIN, float>(last, tile_rows, max_tiles, stream);
}

// ---------------------------------------------------------------------------------------------
// out[t, :] = (sum_k y[place[t * top + k], :]) + shared[t, :], the choices added in order, one rounding at the store.
// With `x`: a choice that the plan has not placed (an identity expert, whose index lies behind the real ones) adds
// pair_weight[t * top + k] * x[t, :] in its turn.  With `scale_rows` every row of y is multiplied with its pair's weight here
// (the products then left it out).
// ---------------------------------------------------------------------------------------------
// V neighbouring entries a thread (4: rows in 16-byte pieces, the choices' rows all asked for before the first is added), a
// workgroup per token and 256 V entries.  Bound by what it moves: 2,500 tokens of 4 x 4,096 float32 and a shared row, 205 MB,
// 34 us (one entry a thread and a workgroup per token: 100); 16 tokens 4.6 us (34).  With the norms, 1,036 tokens of 2 x 2,048: 9.8 (18.5).
template <int V> struct Entries { float v[V]; };
template <typename T, int V>
__device__ __forceinline__ Entries<V> entries_of(const T* p) {
  Entries<V> out;
  typedef T Pieces __attribute__((ext_vector_type(V)));
  if constexpr (V == 1) {
    out.v[0] = to_f32(*p);
  } else {
    const Pieces x = *reinterpret_cast<const Pieces*>(p);
#pragma unroll
    for (int e = 0; e < V; ++e) out.v[e] = to_f32(x[e]);
  }
  return out;
}
template <typename T, int V>
__device__ __forceinline__ void store_entries(T* p, const Entries<V>& in) {
  typedef T Pieces __attribute__((ext_vector_type(V)));
  if constexpr (V == 1) {
    *p = from_f32<T>(in.v[0]);
  } else {
    Pieces x;
#pragma unroll
    for (int e = 0; e < V; ++e) x[e] = from_f32<T>(in.v[e]);
    *reinterpret_cast<Pieces*>(p) = x;
  }
}

// A token's sum at V entries from i on, in float32.
template <typename T, int V>
__device__ __forceinline__ Entries<V> combined(const float* __restrict__ y, const int* mine, const T* __restrict__ shared, int t, int top, int hidden,
                                               const T* __restrict__ x, const float* __restrict__ pair_weight, int scale_rows, int i) {
  constexpr int BATCH = 4;
  Entries<V> sum = {};
  for (int k0 = 0; k0 < top; k0 += BATCH) {
    Entries<V> part[BATCH];
    float factor[BATCH];
#pragma unroll
    for (int j = 0; j < BATCH; ++j) {
      const int row = k0 + j < top ? mine[k0 + j] : -1;
      part[j] = Entries<V>{};
      factor[j] = 1.f;
      if (row >= 0) {
        part[j] = entries_of<float, V>(y + (size_t)row * hidden + i);
        if (scale_rows) factor[j] = pair_weight[(size_t)t * top + k0 + j];
      } else if (x && k0 + j < top) {
        part[j] = entries_of<T, V>(x + (size_t)t * hidden + i);
        factor[j] = pair_weight[(size_t)t * top + k0 + j];
      }
    }
#pragma unroll
    for (int j = 0; j < BATCH; ++j)
#pragma unroll
      for (int e = 0; e < V; ++e) sum.v[e] += factor[j] * part[j].v[e];
  }
  if (shared) {
    const Entries<V> s = entries_of<T, V>(shared + (size_t)t * hidden + i);
#pragma unroll
    for (int e = 0; e < V; ++e) sum.v[e] += s.v[e];
  }
  return sum;
}

template <typename T, int V>
__global__ void __launch_bounds__(256) routed_combine_kernel(const float* __restrict__ y, const int* __restrict__ place, const T* __restrict__ shared,
                                                             T* __restrict__ out, int top, int hidden, const T* __restrict__ x,
                                                             const float* __restrict__ pair_weight, int scale_rows) {
  const int t = blockIdx.x, i = (blockIdx.y * 256 + threadIdx.x) * V;
  if (i >= hidden) return;
  store_entries<T, V>(out + (size_t)t * hidden + i, combined<T, V>(y, place + (size_t)t * top, shared, t, top, hidden, x, pair_weight, scale_rows, i));
}

// The same sum, handed straight to a norm on the experts' output: residual[t, :] += mult * v * rsqrt(mean(v^2) + eps) * w, with v the
// sum above in float32 (never rounded to T), and `copy` (nullable) the updated residual in T; with `next_weight` `copy` is instead
// what the norm that reads the residual next makes of it, r * rsqrt(mean(r^2) + next_eps) * next_weight.  One workgroup per
// token holds the row in registers: hidden <= 16 * blockDim.x.
template <typename T, int V>
__global__ void routed_combine_norm_kernel(const float* __restrict__ y, const int* __restrict__ place, const T* __restrict__ shared, int top, int hidden,
                                           const T* __restrict__ x, const float* __restrict__ pair_weight, int scale_rows, float* __restrict__ residual,
                                           const float* __restrict__ norm_weight, float eps, float mult, T* __restrict__ copy,
                                           const float* __restrict__ next_weight, float next_eps) {
  constexpr int HELD = 16 / V;
  __shared__ float scratch[16];
  const int t = blockIdx.x;
  const int* mine = place + (size_t)t * top;
  Entries<V> held[HELD];
  float sumsq = 0.f;
#pragma unroll
  for (int c = 0; c < HELD; ++c) {
    const int i = (threadIdx.x + c * blockDim.x) * V;
    held[c] = Entries<V>{};
    if (i < hidden) held[c] = combined<T, V>(y, mine, shared, t, top, hidden, x, pair_weight, scale_rows, i);
#pragma unroll
    for (int e = 0; e < V; ++e) sumsq += held[c].v[e] * held[c].v[e];
  }
  const float total = block_sum(sumsq, scratch);
  const float inv = 1.f / sqrtf(total / (float)hidden + eps);
  sumsq = 0.f;
#pragma unroll
  for (int c = 0; c < HELD; ++c) {
    const int i = (threadIdx.x + c * blockDim.x) * V;
    if (i < hidden) {
      const Entries<V> w = entries_of<float, V>(norm_weight + i);
      Entries<V> r = entries_of<float, V>(residual + (size_t)t * hidden + i);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        r.v[e] = r.v[e] + mult * (held[c].v[e] * inv * w.v[e]);
        sumsq += r.v[e] * r.v[e];
      }
      store_entries<float, V>(residual + (size_t)t * hidden + i, r);
      if (copy && !next_weight) store_entries<T, V>(copy + (size_t)t * hidden + i, r);
      held[c] = r;
    }
  }
  if (!next_weight) return;
  const float next_inv = 1.f / sqrtf(block_sum(sumsq, scratch) / (float)hidden + next_eps);
#pragma unroll
  for (int c = 0; c < HELD; ++c) {
    const int i = (threadIdx.x + c * blockDim.x) * V;
    if (i < hidden) {
      const Entries<V> w = entries_of<float, V>(next_weight + i);
      Entries<V> r = held[c];
#pragma unroll
      for (int e = 0; e < V; ++e) r.v[e] = r.v[e] * next_inv * w.v[e];
      store_entries<T, V>(copy + (size_t)t * hidden + i, r);
    }
  }
}

// Whether all rows start on the boundaries that four entries at a time need.
static bool combine_in_fours(int hidden, int dtype, const void* y, const void* shared, const void* x, const void* a, const void* b, const void* c, const void* d) {
  const uintptr_t narrow = (uintptr_t)shared | (uintptr_t)x | (uintptr_t)d, wide = (uintptr_t)y | (uintptr_t)a | (uintptr_t)b | (uintptr_t)c;
  return hidden % 4 == 0 && wide % 16 == 0 && narrow % (dtype == VELOX_BF16 ? 8 : 16) == 0;
}

// copy: nullptr in a float32 run (the residual is its own copy).  Returns -1 when the row does not fit the registers
// (hidden > 16,384): the caller then runs the two kernels one after the other.
extern "C" int velox_routed_combine_norm(const float* y, const int* plan, const void* shared, int tokens, int top, int experts, int hidden, int dtype,
                                         const void* x, const float* pair_weight, int scale_rows, float* residual, const float* norm_weight, float eps,
                                         float mult, void* copy, const float* next_weight, float next_eps, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (next_weight && !copy) return (int)hipErrorInvalidValue;
  if (hidden > 16 * 1024) return -1;
  const int* place = plan + 1 + (experts + 1) + (size_t)tokens * top;
  int threads = tokens <= 64 ? 512 : 256;  // (few rows: more threads each with less to do)
  while (16 * threads < hidden) threads *= 2;
#define COMBINE(T, V)                                                                                                                              \
  routed_combine_norm_kernel<T, V><<<tokens, threads, 0, stream>>>(y, place, (const T*)shared, top, hidden, (const T*)x, pair_weight, scale_rows, residual, \
                                                                   norm_weight, eps, mult, (T*)copy, next_weight, next_eps)
  const bool fours = combine_in_fours(hidden, dtype, y, shared, x, residual, norm_weight, next_weight, copy);
  if (dtype == VELOX_BF16) {
    if (fours) COMBINE(bf16_t, 4);
    else COMBINE(bf16_t, 1);
  } else {
    if (fours) COMBINE(float, 4);
    else COMBINE(float, 1);
  }
#undef COMBINE
  VELOX_RETURN_LAUNCH_STATUS();
}

extern "C" int velox_routed_combine(const float* y, const int* plan, const void* shared, void* out, int tokens, int top, int experts, int hidden, int dtype,
                                    const void* x, const float* pair_weight, int scale_rows, hipStream_t stream) {
  if (tokens <= 0) return 0;
  const int* place = plan + 1 + (experts + 1) + (size_t)tokens * top;
#define COMBINE(T, V)                                                                                                                              \
  routed_combine_kernel<T, V><<<dim3(tokens, (hidden + 256 * V - 1) / (256 * V)), 256, 0, stream>>>(y, place, (const T*)shared, (T*)out, top, hidden, (const T*)x, \
                                                                                                    pair_weight, scale_rows)
  const bool fours = combine_in_fours(hidden, dtype, y, shared, x, nullptr, nullptr, nullptr, out);
  if (dtype == VELOX_BF16) {
    if (fours) COMBINE(bf16_t, 4);
    else COMBINE(bf16_t, 1);
  } else {
    if (fours) COMBINE(float, 4);
    else COMBINE(float, 1);
  }
#undef COMBINE
  VELOX_RETURN_LAUNCH_STATUS();
}
