// out[M, N] = A[M, K] * W[N, K]^T (+ bias[N]) with float32 accumulation, for gfx950.
//
// `gemm_fma_kernel` widens its operands to float32 (exactly, for bfloat16) and multiplies them with
// plain fused multiply-adds.  It serves operand mixes no library call covers (bfloat16 activations with
// weights a checkpoint stores in float32), float32 rows that are not whole 16-byte pieces and sums of
// fewer than GEMM_FOLD terms; other float32 products run on the float32 matrix instructions (gemm_mfma_f32_kernel) or, larger ones,
// on exactly split operands (split_f32.hip), whose error against 64 bits is below the float32 instructions' for operands of any size.  Each output element is summed over k in one fixed
// order by one thread, so a row's result does not depend on what the other rows of the batch hold (their number chooses the
// kernel: up to 16 rows have one of their own, with an order of its own).  The sum
// is built from sums of GEMM_FOLD consecutive terms, each started at zero: the rounding error of a
// long sum (the down projection adds 18944 terms) then grows with the square roots of the two
// lengths and not with that of their product, which keeps the float32 path as close to the exact
// result as a blocked library product on a CPU is.
#include "common.h"
#include "tiles_mfma.h"

#define GEMM_BM 64
#define GEMM_BN 64
#define GEMM_BK 16
#define GEMM_PAD 4
#define GEMM_FOLD 128  // terms per inner sum (a multiple of GEMM_BK)

template <typename TA, typename TW, typename TO>
__global__ void __launch_bounds__(256) gemm_fma_kernel(const TA* __restrict__ a, const TW* __restrict__ w, const float* __restrict__ bias,
                                                       TO* __restrict__ out, int m, int n, int k, int a_vec, int w_vec) {
  __shared__ float a_tile[GEMM_BK][GEMM_BM + GEMM_PAD];
  __shared__ float w_tile[GEMM_BK][GEMM_BN + GEMM_PAD];
  const int tid = threadIdx.x;
  const int tx = tid % 16, ty = tid / 16;
  const int m0 = blockIdx.y * GEMM_BM, n0 = blockIdx.x * GEMM_BN;
  const int load_row = tid / 4;          // 0..63
  const int load_k = (tid % 4) * 4;      // 0, 4, 8, 12
  const bool a_row_ok = m0 + load_row < m;
  const bool w_row_ok = n0 + load_row < n;
  const size_t a_off = (size_t)(m0 + load_row) * k;
  const size_t w_off = (size_t)(n0 + load_row) * k;

  float acc[4][4], total[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = total[i][j] = 0.f;

  for (int k0 = 0; k0 < k; k0 += GEMM_BK) {
    if (k0 % GEMM_FOLD == 0) {  // (also at 0: adds zeros)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          total[i][j] += acc[i][j];
          acc[i][j] = 0.f;
        }
    }
    float av[4], wv[4];
    load4<TA>(a, a_off, k0 + load_k, k, a_row_ok, a_vec != 0, av);
    load4<TW>(w, w_off, k0 + load_k, k, w_row_ok, w_vec != 0, wv);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a_tile[load_k + i][load_row] = av[i];
      w_tile[load_k + i][load_row] = wv[i];
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GEMM_BK; ++kk) {
      const float4_t ar = *reinterpret_cast<const float4_t*>(&a_tile[kk][ty * 4]);
      const float4_t wr = *reinterpret_cast<const float4_t*>(&w_tile[kk][tx * 4]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(ar[i], wr[j], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = m0 + ty * 4 + i;
    if (row >= m) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = n0 + tx * 4 + j;
      if (col >= n) continue;
      float v = total[i][j] + acc[i][j];
      if (bias) v += bias[col];
      out[(size_t)row * n + col] = from_f32<TO>(v);
    }
  }
}

// The float32 product of more than 16 rows on the matrix cores (v_mfma_f32_16x16x4_f32: float32 operands, products and sums, twice
// the rate of scalar multiply-adds).  A set of four waves owns 32 RT x 32 CT outputs, a wave 16 RT x 16 CT of them; a step is 32
// indices, so a row of either operand is 128 bytes of LDS, eight pieces of 16, exchanged by an XOR with the row's low three
// bits (no bank conflicts), filled by loads that write LDS directly, STAGES - 1 steps ahead, with one barrier per step.  Lane
// (g, i) takes indices 4 g .. 4 g + 3 of every 16 of row i as one 16-byte read and feeds one of them to each of four matrix
// instructions: both operands in the same order of k.  As in the kernel above an output is built from sums of GEMM_FOLD terms;
// here those of either half of k are added up first.  Where a step has too few tiles to fill the card, two sets of waves take
// the halves (SETS = 2), otherwise one set takes both in turn: an output's order of additions depends on k alone, whichever
// kernel a batch size leads to.
// Bound by the matrix instructions (157 TFLOP/s) where there are tiles enough, by how far ahead the loads are where there are
// few.  Tiles follow one another along the rows of A on the same XCD, so the rows of W that they share leave its L2.
// Measured on MI355X (us, multiply-adds -> this): 616 rows, 1,536 -> 17,920: 593 -> 360 (94 TFLOP/s); 616 rows, 8,960 -> 1,536: 590 ->
// 182; 2,048 rows, 1,536 -> 17,920: 1,576 -> 986 (114 TFLOP/s); 64 rows, 8,960 -> 1,536: 582 -> 70; error against float64 1.5e-07 to
// 1.7e-07 of the result's norm (before 1.5e-07 to 1.8e-07).
static __device__ __attribute__((aligned(16))) const unsigned int gemm_zero_piece[4] = {0u, 0u, 0u, 0u};

#define GEMM_XCDS 8

template <int RT, int CT, int SETS, int STAGES>
__global__ void __launch_bounds__(256 * SETS) __attribute__((amdgpu_waves_per_eu(2, 4))) gemm_mfma_f32_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                                                                              const float* __restrict__ bias, float* __restrict__ out, int m, int n, int k) {
  constexpr int ROWS = 32 * RT, COLS = 32 * CT, WAVES = 4;
  constexpr int A_LOADS = ROWS / 8 / WAVES, W_LOADS = COLS / 8 / WAVES, LOADS = A_LOADS + W_LOADS;
  constexpr int BYTES = (ROWS + COLS) * 128;
  __shared__ __attribute__((aligned(1024))) char smem_all[SETS][STAGES][BYTES];
  const int row_tiles = (m + ROWS - 1) / ROWS, total_tiles = row_tiles * ((n + COLS - 1) / COLS);
  const int share = (total_tiles + GEMM_XCDS - 1) / GEMM_XCDS;
  const int mine = (int)(blockIdx.x / GEMM_XCDS), tile = (int)(blockIdx.x % GEMM_XCDS) * share + mine;
  if (mine >= share || tile >= total_tiles) return;  // (uniform over the workgroup)
  const int m0 = tile % row_tiles * ROWS, n0 = tile / row_tiles * COLS;

  const int set = SETS == 2 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
  char (*const smem)[BYTES] = smem_all[set];
  const int i = lane & 15, g = lane >> 4;
  const int piece = 4 * ((lane & 7) ^ (lane >> 3));  // first index of the piece this lane asks for, in every load
  const float* a_at[A_LOADS];
  const float* w_at[W_LOADS];
#pragma unroll
  for (int q = 0; q < A_LOADS; ++q) a_at[q] = a + (size_t)min(m0 + 8 * (wave + WAVES * q) + (lane >> 3), m - 1) * k + piece;
#pragma unroll
  for (int q = 0; q < W_LOADS; ++q) w_at[q] = w + (size_t)min(n0 + 8 * (wave + WAVES * q) + (lane >> 3), n - 1) * k + piece;
  const int wm = wave >> 1, wn = wave & 1;
  const int a_byte = (wm * 16 * RT + i) * 128, w_byte = ROWS * 128 + (wn * 16 * CT + i) * 128;
  // k in two halves that meet at a multiple of GEMM_FOLD: two sets of waves take one each, or one set both in turn.  (The first is
  // the longer one, and two sets run its number of steps.)
  const int middle = min(k, (k + 2 * GEMM_FOLD - 1) / (2 * GEMM_FOLD) * GEMM_FOLD);

  float4_t sum[CT][RT], acc[CT][RT], total[CT][RT];
  auto half_of_k = [&](int begin, int end, int steps) {
    auto ask = [&](int s, int buffer) {
      const int k0 = begin + 32 * s;
      const bool beyond = k0 + piece >= end;  // (zeros behind the end of the half)
#pragma unroll
      for (int q = 0; q < A_LOADS; ++q) load_to_lds_16(beyond ? reinterpret_cast<const float*>(gemm_zero_piece) : a_at[q] + k0, smem[buffer] + 1024 * (wave + WAVES * q));
#pragma unroll
      for (int q = 0; q < W_LOADS; ++q) load_to_lds_16(beyond ? reinterpret_cast<const float*>(gemm_zero_piece) : w_at[q] + k0, smem[buffer] + ROWS * 128 + 1024 * (wave + WAVES * q));
    };
    float4_t a_op[2][RT], w_op[2][CT];
    auto fetch = [&](int part, int buffer) {
      const char* base = smem[buffer];
      const int place = ((4 * part + g) ^ (i & 7)) * 16;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) w_op[part][ct] = *reinterpret_cast<const float4_t*>(base + w_byte + ct * 2048 + place);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) a_op[part][rt] = *reinterpret_cast<const float4_t*>(base + a_byte + rt * 2048 + place);
    };
    auto multiply = [&](int part) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) acc[ct][rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(w_op[part][ct][e], a_op[part][rt][e], acc[ct][rt], 0, 0, 0);
    };
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) acc[ct][rt] = total[ct][rt] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
      if (s < steps) ask(s, s);
    // the first step's loads have landed when at most those of the later steps that were asked for are under way
    if (steps >= STAGES - 1) wait_for_loads<(STAGES - 2) * LOADS>();
    else wait_for_loads<0>();
    __syncthreads();
    fetch(0, 0);
    int buffer = 0;
    for (int s = 0; s < steps; ++s) {
      fetch(1, buffer);
      int freed = buffer + STAGES - 1;
      if (freed >= STAGES) freed -= STAGES;
      if (s + STAGES - 1 < steps) ask(s + STAGES - 1, freed);  // (the buffer that everybody was done with at the last barrier)
      __builtin_amdgcn_sched_barrier(0);
      multiply(0);
      __builtin_amdgcn_sched_barrier(0);
      buffer = buffer + 1 == STAGES ? 0 : buffer + 1;
      if (s + 1 < steps) {
        if (s + STAGES <= steps) wait_for_loads<(STAGES - 2) * LOADS>();
        else wait_for_loads<0>();
        __syncthreads();
        fetch(0, buffer);
      }
      __builtin_amdgcn_sched_barrier(0);
      multiply(1);
      if ((s + 1) % (GEMM_FOLD / 32) == 0) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) {
            total[ct][rt] += acc[ct][rt];
            acc[ct][rt] = float4_t{0.f, 0.f, 0.f, 0.f};
          }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) total[ct][rt] += acc[ct][rt];
    __syncthreads();  // (everybody is done with the buffers)
  };
  if (SETS == 2) {
    half_of_k(set == 0 ? 0 : middle, set == 0 ? middle : k, (middle + 31) / 32);
    float4_t* joined = reinterpret_cast<float4_t*>(smem_all[0]) + (threadIdx.x & 255);
    if (set == 1) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) joined[256 * (ct * RT + rt)] = total[ct][rt];
    }
    __syncthreads();
    if (set == 1) return;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) sum[ct][rt] = total[ct][rt] + joined[256 * (ct * RT + rt)];
  } else {
    half_of_k(0, middle, (middle + 31) / 32);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) sum[ct][rt] = total[ct][rt];
    if (middle < k) {
      half_of_k(middle, k, (k - middle + 31) / 32);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) sum[ct][rt] += total[ct][rt];
    }
  }
  // lane (g, i) holds outputs 4 g .. + 3 of row i of every tile
  const bool vec = n % 4 == 0 && ((uintptr_t)out & 15) == 0;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int row = m0 + wm * 16 * RT + rt * 16 + i;
    if (row >= m) continue;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const int col = n0 + wn * 16 * CT + ct * 16 + 4 * g;
      float4_t v = sum[ct][rt];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (bias != nullptr && col + j < n) v[j] += bias[col + j];
      if (vec && col < n) {
        *reinterpret_cast<float4_t*>(out + (size_t)row * n + col) = v;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (col + j < n) out[(size_t)row * n + col + j] = v[j];
      }
    }
  }
}

// Which tile, by the number of tiles.  Measured on MI355X (us; 128 x 64 and 64 x 64 by one set | 64 x 64, 32 x 64, 32 x 32 by two):
//   4,096 rows, 2,048 -> 11,264   1588  1690 | 1900  1960  2900        2,048 rows, 8,960 -> 1,536   614  515 | 532  586  802
//   616 rows, 1,536 -> 17,920      359   370 |  393   432   583        300 rows, 1,536 -> 17,920    242  197 | 218  212  290
//   616 rows, 8,960 -> 1,536       329   210 |  182   214   268        616 rows, 1,536 -> 2,048      65   65 |  70   58   66
//   300 rows, 8,960 -> 1,536       331   204 |  182   119   139        64 rows, 8,960 -> 1,536      330  200 | 178  111   70
// so: from two workgroups per compute unit on one set, in tiles of 128 rows if few of them stay empty; with about one workgroup
// per compute unit 64 x 64 by two sets; with fewer the largest tile that still gives most compute units a workgroup.
// The tile as rows * 10,000 + columns * 10 + sets (an entry point so that a test can tell which one a size takes).
extern "C" int velox_gemm_f32_tile(int m, int n) {
  auto tiles = [&](int rt, int ct) { return (long long)((m + 32 * rt - 1) / (32 * rt)) * ((n + 32 * ct - 1) / (32 * ct)); };
  if (tiles(4, 2) >= 512 && (m + 127) / 128 * 128 * 10 <= m * 11) return 1280641;
  if (tiles(2, 2) >= 512) return 640641;
  if (tiles(2, 2) >= 200 && tiles(2, 2) <= 256) return 640642;
  return tiles(1, 2) >= 200 ? 320642 : 320322;
}

static void launch_mfma_f32(const void* a, const void* w, const float* bias, void* out, int m, int n, int k, hipStream_t stream) {
#define MFMA(RT, CT, SETS, STAGES)                                                                                                  \
  {                                                                                                                                 \
    const long long tiles = (long long)((m + 32 * RT - 1) / (32 * RT)) * ((n + 32 * CT - 1) / (32 * CT));                           \
    gemm_mfma_f32_kernel<RT, CT, SETS, STAGES><<<(unsigned)((tiles + GEMM_XCDS - 1) / GEMM_XCDS * GEMM_XCDS), 256 * SETS, 0, stream>>>( \
        (const float*)a, (const float*)w, bias, (float*)out, m, n, k);                                                              \
  }
  switch (velox_gemm_f32_tile(m, n)) {
    case 1280641: MFMA(4, 2, 1, 2) break;
    case 640641: MFMA(2, 2, 1, 3) break;
    case 640642: MFMA(2, 2, 2, 3) break;
    case 320642: MFMA(1, 2, 2, 3) break;
    default: MFMA(1, 1, 2, 3) break;
  }
#undef MFMA
}

// The same product for few rows (M <= 16), where it is bound by reading W once: the decode steps of a float32 run.
// A wave owns ROWS consecutive rows of W and all of K; lane l takes indices 4 l .. 4 l + 3 of every block of
// 256, so a wave's load of a row's block is one contiguous kilobyte (float32) and the activations (from L2) are used
// for ROWS rows of W at once.  A lane adds its terms in the order of k, the 64 lanes' sums are added in a fixed
// tree: an element's sum depends on nothing but its own row of A and row of W, whatever ROWS is.
// Measured on MI355X, us, with four rows, a tree through LDS for every sum, ordinary loads and 8 or 16 rows of A where there are 5 or more / like this:
// 1,536 -> 151,936, 1 row 153 / 133, 6 rows 225 / 143, 16 391 / 207; 1,536 -> 17,920, 1, 6 and 16 rows 22 / 19, 38 / 23, 59 / 35; 1,536 -> 2,048 7.6 /
// 5.8, 15.2 / 7.3, 24.7 / 10.1; 8,960 -> 1,536 31 / 26, 50 / 33, 71 / 47.
// (All of W is read once and in whole lines: non-temporal.)
template <typename T>
__device__ __forceinline__ void load4_once(const T* __restrict__ p, float (&v)[4]) {
  if constexpr (sizeof(T) == 4) {
    const float4_t x = __builtin_nontemporal_load(reinterpret_cast<const float4_t*>(p));
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = x[i];
  } else {
    const short4_t x = __builtin_nontemporal_load(reinterpret_cast<const short4_t*>(p));
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(((uint32_t)(uint16_t)x[i]) << 16);
  }
}

// The wave's sums of COUNT values, in the tree of wave_sum (lanes 32 apart first, then 16, 8, ..), to its bits: at every level half of the values
// are finished in one half of the lanes and half in the other, so that a level moves half as many as the one before.  Value i's sum lies
// in the lanes whose bit 5 is i's bit 0, bit 4 its bit 1 and so on.  32 values: 32 moves, 24 of them between registers, instead of 192 through LDS.
template <int COUNT>
__device__ __forceinline__ float wave_sums(float (&v)[COUNT]) {
  const int lane = threadIdx.x & 63;
  int left = COUNT;
#pragma unroll
  for (int offset = 32; offset > 0; offset >>= 1) {
    const bool upper = (lane & offset) != 0;
    if (left == 1) {
      v[0] += __shfl_xor(v[0], offset, VELOX_WAVE);
      continue;
    }
#pragma unroll
    for (int i = 0; i < left / 2; ++i) {
      const float low = v[2 * i], high = v[2 * i + 1];
      if (offset >= 16) {  // (the two registers' halves, or their rows of 16 lanes, change places: both then hold one value's two parts)
        typedef unsigned int Two __attribute__((ext_vector_type(2)));
        const Two both = offset == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(low), __float_as_uint(high), false, false)
                                      : __builtin_amdgcn_permlane16_swap(__float_as_uint(low), __float_as_uint(high), false, false);
        v[i] = __uint_as_float(both[0]) + __uint_as_float(both[1]);
      } else {
        const float mine = upper ? high : low, other = upper ? low : high;
        v[i] = mine + __shfl_xor(other, offset, VELOX_WAVE);
      }
    }
    left /= 2;
  }
  return v[0];
}

template <typename TA, typename TW, typename TO, int MT, int ROWS>
__global__ void __launch_bounds__(256) skinny_fma_kernel(const TA* __restrict__ a, const TW* __restrict__ w, const float* __restrict__ bias,
                                                         TO* __restrict__ out, int m, int n, int k) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n0 = (blockIdx.x * 4 + wave) * ROWS;
  if (n0 >= n) return;
  float acc[ROWS][MT];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[r][i] = 0.f;
  size_t w_off[ROWS], a_off[MT];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) w_off[r] = (size_t)(n0 + r < n ? n0 + r : n0) * k;  // (a row beyond N: row n0 again, never stored)
#pragma unroll
  for (int i = 0; i < MT; ++i) a_off[i] = (size_t)(i < m ? i : 0) * k;
  for (int k0 = 4 * lane; k0 < k; k0 += 256) {
    float wv[ROWS][4], av[MT][4];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) load4_once<TW>(w + w_off[r] + k0, wv[r]);
#pragma unroll
    for (int i = 0; i < MT; ++i) load4<TA>(a, a_off[i], k0, k, true, true, av[i]);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[r][i] = fmaf(av[i][e], wv[r][e], acc[r][i]);
  }
  // 64 values at a time and what is left, filled up to a power of two with zeros
  constexpr int BATCH = 64 / ROWS;  // rows of A
  const int mine = (int)(__brev((unsigned)lane << 26) & 63u);  // the lane's six bits the other way round: which value it holds
#pragma unroll
  for (int i0 = 0; i0 < MT; i0 += BATCH) {
    constexpr int LEFT = MT < BATCH ? MT : BATCH;
    constexpr int COUNT = LEFT * ROWS <= 4 ? 4 : LEFT * ROWS <= 8 ? 8 : LEFT * ROWS <= 16 ? 16 : LEFT * ROWS <= 32 ? 32 : 64;
    float values[COUNT];
#pragma unroll
    for (int v = 0; v < COUNT; ++v) values[v] = i0 + v / ROWS < MT ? acc[v % ROWS][i0 + v / ROWS < MT ? i0 + v / ROWS : 0] : 0.f;
    const float total = wave_sums<COUNT>(values);
    const int row = i0 + mine / ROWS, col = n0 + mine % ROWS;
    if (mine < COUNT && row < m && col < n) out[(size_t)row * n + col] = from_f32<TO>(total + (bias ? bias[col] : 0.f));
  }
}

// Rows of W per wave.  Eight, which halve the loads of A, where so many outputs leave enough waves (us, four / eight rows: 1,536 -> 151,936, 2 rows 134 / 136,
// 3 137 / 136, 6 161 / 143; 2,048 -> 32,000, 8 rows 53 / 55, 12 64 / 60; 1,536 -> 17,920, 16 rows 35 / 37); two where four leave compute units without a
// workgroup (four / two rows: 1,536 -> 2,048, 6 rows 8.5 / 7.3, 8,960 -> 1,536 39 / 33).  (Other types than float32 alone: four.)
template <typename TA, typename TW, typename TO>
static void launch_skinny_fma(const void* a, const void* w, const float* bias, void* out, int m, int n, int k, hipStream_t stream) {
#define SKINNY_ROWS(MT, ROWS) \
  skinny_fma_kernel<TA, TW, TO, MT, ROWS><<<(n + 4 * ROWS - 1) / (4 * ROWS), 256, 0, stream>>>((const TA*)a, (const TW*)w, bias, (TO*)out, m, n, k)
#define SKINNY(MT)                                                              \
  {                                                                             \
    if constexpr (sizeof(TA) == 4 && sizeof(TW) == 4 && sizeof(TO) == 4) {      \
      if (MT >= 3 && (long long)n * m >= 360000) SKINNY_ROWS(MT, (MT >= 3 ? 8 : 4)); \
      else if (n < 16 * TL_WORKGROUPS) SKINNY_ROWS(MT, 2);                      \
      else SKINNY_ROWS(MT, 4);                                                  \
    } else {                                                                    \
      SKINNY_ROWS(MT, 4);                                                       \
    }                                                                           \
  }
  if (m <= 1) SKINNY(1)
  else if (m <= 2) SKINNY(2)
  else if (m <= 3) SKINNY(3)
  else if (m <= 4) SKINNY(4)
  else if (m <= 6) SKINNY(6)
  else if (m <= 8) SKINNY(8)
  else if (m <= 12) SKINNY(12)
  else SKINNY(16)
#undef SKINNY
#undef SKINNY_ROWS
}

extern "C" int velox_gemm_fma(const void* a, const void* w, const float* bias, void* out, int m, int n, int k,
                              int a_dtype, int w_dtype, int out_dtype, hipStream_t stream) {
  if (m <= 0 || n <= 0) return 0;
  dim3 grid((n + GEMM_BN - 1) / GEMM_BN, (m + GEMM_BM - 1) / GEMM_BM);
  const int a_size = a_dtype == VELOX_BF16 ? 2 : 4, w_size = w_dtype == VELOX_BF16 ? 2 : 4;
  const int a_vec = (k % 4 == 0) && (((uintptr_t)a) % (4 * a_size) == 0);
  const int w_vec = (k % 4 == 0) && (((uintptr_t)w) % (4 * w_size) == 0);
#define LAUNCH(TA, TW, TO) \
  gemm_fma_kernel<TA, TW, TO><<<grid, 256, 0, stream>>>((const TA*)a, (const TW*)w, bias, (TO*)out, m, n, k, a_vec, w_vec)
  const int key = a_dtype * 4 + w_dtype * 2 + out_dtype;
  if (m <= 16 && a_vec && w_vec) {  // (rows of whole 16-byte pieces: every load is a vector)
    switch (key) {
      case 0: launch_skinny_fma<float, float, float>(a, w, bias, out, m, n, k, stream); break;
      case 1: launch_skinny_fma<float, float, bf16_t>(a, w, bias, out, m, n, k, stream); break;
      case 2: launch_skinny_fma<float, bf16_t, float>(a, w, bias, out, m, n, k, stream); break;
      case 3: launch_skinny_fma<float, bf16_t, bf16_t>(a, w, bias, out, m, n, k, stream); break;
      case 4: launch_skinny_fma<bf16_t, float, float>(a, w, bias, out, m, n, k, stream); break;
      case 5: launch_skinny_fma<bf16_t, float, bf16_t>(a, w, bias, out, m, n, k, stream); break;
      case 6: launch_skinny_fma<bf16_t, bf16_t, float>(a, w, bias, out, m, n, k, stream); break;
      case 7: launch_skinny_fma<bf16_t, bf16_t, bf16_t>(a, w, bias, out, m, n, k, stream); break;
      default: return -1;
    }
    VELOX_RETURN_LAUNCH_STATUS();
  }
  // Sums of fewer terms than one inner sum stay with the multiply-adds, whose order of additions is that of k.  The matrix
  // instructions are quicker there too (64 terms, us, multiply-adds / matrix instructions: 417 x 256 outputs 6.4 / 3.4, 2,048 x 2,048
  // 14.8 / 10.7; 256 terms 17.7 / 4.3 and 39.1 / 27.3) and no less exact on average: the line is here because a small model with
  // sharp weights, whose recurrences blow a rounding up a thousandfold, left its tolerance in the other order of additions.
  if (key == 0 && a_vec && w_vec && k >= GEMM_FOLD) {
    launch_mfma_f32(a, w, bias, out, m, n, k, stream);
    VELOX_RETURN_LAUNCH_STATUS();
  }
  switch (key) {
    case 0: LAUNCH(float, float, float); break;
    case 1: LAUNCH(float, float, bf16_t); break;
    case 2: LAUNCH(float, bf16_t, float); break;
    case 3: LAUNCH(float, bf16_t, bf16_t); break;
    case 4: LAUNCH(bf16_t, float, float); break;
    case 5: LAUNCH(bf16_t, float, bf16_t); break;
    case 6: LAUNCH(bf16_t, bf16_t, float); break;
    case 7: LAUNCH(bf16_t, bf16_t, bf16_t); break;
    default: return -1;
  }
#undef LAUNCH
  VELOX_RETURN_LAUNCH_STATUS();
}

// out[M, N] (bfloat16, + bias; or float32 partial sums [splits, M, N] of `splits` parts of k) = A[M, K] * W[N, K]^T, bfloat16, in tiles_mfma.h's tiles of
// `tile` = rows * 1,000 + columns (0: the one that tiles_pick takes).  Needs k % 8 == 0, n % 4 == 0 and 16-byte aligned bases; k % 64 != 0 has 128 x 256 alone.
extern "C" int velox_tiles_bf16(const void* a, const void* w, const float* bias, void* out, int m, int n, int k, int splits, int out_dtype, int tile, hipStream_t stream) {
  if (m <= 0 || n <= 0) return 0;
  if (k < 1 || k % 8 != 0 || n % 4 != 0 || splits < 1 || (splits != 1 && (out_dtype == VELOX_BF16 || bias != nullptr)) ||
      (((uintptr_t)a | (uintptr_t)w | (uintptr_t)out) & 15) != 0 || !tiles_fit(256, k, 256, k))
    return -1;
  TileArgs args = {};
  args.a = (const bf16_t*)a;
  args.a_ld = k;
  args.w = (const bf16_t*)w;
  args.bias = bias;
  args.out = out;
  args.m = m;
  args.n = n;
  args.k = k;
  args.splits = splits;
  if (tile == 0) tile = tiles_pick(m, n, k, splits);
  if (k % 64 == 0) return out_dtype == VELOX_BF16 ? tiles_launch<TL_PLAIN, bf16_t, false>(args, tile, stream) : tiles_launch<TL_PLAIN, float, false>(args, tile, stream);
  return out_dtype == VELOX_BF16 ? tiles_launch<TL_PLAIN, bf16_t, true>(args, tile, stream) : tiles_launch<TL_PLAIN, float, true>(args, tile, stream);
}

// out[M, N] = act(A Wgate^T) * (A Wup^T) in bfloat16 for W = [Wgate; Wup] [2 N, K], both sums rounded to bfloat16 in front of it; act 0: SiLU, 2: the
// rectifier (the tanh form of GELU stays a kernel of its own: its tangent costs more than the pass).  Needs k % 64 == 0, n % 4 == 0 and 16-byte aligned bases.
extern "C" int velox_tiles_glu_bf16(const void* a, const void* w, void* out, int m, int n, int k, int act, int tile, hipStream_t stream) {
  if (m <= 0 || n <= 0) return 0;
  if (k < 1 || k % 64 != 0 || n % 4 != 0 || (act != 0 && act != 2) || (((uintptr_t)a | (uintptr_t)w | (uintptr_t)out) & 15) != 0 || !tiles_fit(256, k, n + 256LL, k)) return -1;
  TileArgs args = {};
  args.a = (const bf16_t*)a;
  args.a_ld = k;
  args.w = (const bf16_t*)w;
  args.out = out;
  args.m = m;
  args.n = n;
  args.k = k;
  args.splits = 1;
  if (tile == 0) tile = tiles_pick(m, 2LL * n, k, 1);
  return act == 0 ? tiles_launch<TL_SILU, bf16_t, false>(args, tile, stream) : tiles_launch<TL_RELU, bf16_t, false>(args, tile, stream);
}

extern "C" int velox_tiles_splits(int m, int n, int k, int most) { return tiles_splits(m, n, k, most); }
