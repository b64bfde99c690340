// The generalized delta rule over long portions of prompts, in chunks of 16 tokens on the float32 matrix instructions.
//
// Per head, with decay w_t, unit key u_t, removal vector b_t = a_t * u_t, key k_t, value v_t and read vector r_t:
//     S_t = diag(w_t) S_(t-1) - b_t (u_t^T S_(t-1)) + k_t v_t^T,   o_t = S_t^T r_t.
// Inside a chunk let P_t = w_1 * .. * w_t (per channel, P_0 = 1) and S_t = diag(P_t) Z_t.  With
//     U_t = u_t * P_(t-1),  R_t = r_t * P_t,  B_t = b_t / P_t,  K_t = k_t / P_t       (rows of 16 x dim matrices)
// the rule reads Z_t = Z_(t-1) - B_t d_t + K_t v_t^T with the removed rows d_t = U_t Z_(t-1), so that
//     D = U Z_0 + M1 V - M2 D,   O = R Z_0 + M3 V - M4 D,   Z_16 = Z_0 + K^T V - B^T D,
// M1 = U K^T and M2 = U B^T below the diagonal, M3 = R K^T and M4 = R B^T with it.  With T = (I + M2)^-1 (unit lower
// triangular, by substitution) everything that does not touch the state is worked for all chunks at the same time:
//     U' = T U,   Dv = T M1 V,   R' = R - M4 T U,   Ov = M3 V - M4 Dv,
// and what is left of the dependent chain is, per chunk,   D = U' Z_0 + Dv,   O = R' Z_0 + Ov,   S = diag(P_16) (Z_0 + K^T V - B^T D).
// All of it is float32.  A decay is at least exp(-scale), so P_16 is at least exp(-16 scale); the host takes these kernels only while
// 16 scale < 13 (P_16 > 2e-6), and products of rows hold P_t / P_j <= 1 for j <= t: nothing overflows and nothing cancels.
//
//   removal_chunk_prepare_kernel   a workgroup per chunk and head: unit keys, removal vectors, the decay's low-rank map, the four
//                                  products, T, and the matrices above into `scratch`
//   removal_chunk_scan_kernel      a workgroup per 16 value columns, head and sequence; a wave holds 16 rows of the state in the
//                                  matrix instructions' result layout, which is also their operand layout, so that the state
//                                  never leaves the registers; the waves exchange their parts of D and O through LDS
#include <type_traits>

#include "common.h"

#define CHUNK 16
#define CHUNK_STRIDE 20  // floats between the rows of a 16 x 16 matrix in LDS (16-byte aligned, rows on different banks)

struct RemovalChunkArgs {
  const void* main;  // [T, ld]
  int ld, r_at, k_at, v_at, a_at, low_at, rank, heads, dim, vdim;
  const float* a_bias;
  const void* w2;
  const float* w0;
  float scale;
  float* scratch;
  float* state;  // [slots, heads, dim, vdim]
  const int* slots;
  const int* cu_q;
  float* out;  // [T, heads * vdim]
  bool ordered;  // the scan's sequences by their length, see sequence_by_length
};

// A chunk and head in `scratch`, in floats: U' | R' | -B | K (each 16 * dim), P_16 (dim), Dv | Ov | V (each 16 * columns).  U' and R' as
// [dim / 16][16 tokens][16 channels], B and K as [dim][16 tokens], Dv, Ov and V as [columns][16 tokens]: what a wave reads of one
// of them is one contiguous kilobyte, 16 bytes a lane.
__host__ __device__ __forceinline__ int removal_columns(int vdim) { return (vdim + 15) / 16 * 16; }
__host__ __device__ __forceinline__ size_t removal_record(int dim, int vdim) { return (size_t)65 * dim + 48 * removal_columns(vdim); }
// the first record of a sequence (chunks are a step's items, see step_item)
__device__ __forceinline__ int removal_first_chunk(int first_token, int sequence) { return first_token / CHUNK + sequence; }

__device__ __forceinline__ float removal_sigmoid(float z) { return 1.f / (1.f + expf(-z)); }
__device__ __forceinline__ float4_t mfma4(float a, float b, float4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ float4_t four(const float* p) { return *reinterpret_cast<const float4_t*>(p); }

template <typename T>
__global__ void __launch_bounds__(256) removal_chunk_prepare_kernel(const RemovalChunkArgs a, int num_seqs) {
  extern __shared__ float4_t lds_pieces[];
  float* lds = reinterpret_cast<float*>(lds_pieces);
  const int h = blockIdx.x % a.heads, record_at = blockIdx.x / a.heads;
  const StepItem item = step_item(a.cu_q, num_seqs, CHUNK, record_at);
  const int hi = item.hi, t0 = item.lo + item.piece * CHUNK;
  if (t0 >= hi) return;  // (the whole workgroup)
  const int count = hi - t0 < CHUNK ? hi - t0 : CHUNK;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, g = lane >> 4;  // column and group of four rows in the matrix instructions' layouts
  const int dim = a.dim, rank = a.rank, row = dim + 4;
  const int padded_rank = (rank + 15) / 16 * 16, inner_row = padded_rank + 4;
  // four matrices of 16 rows (U, R, B, K), the decays, the map's inner rows, and 16 x 16 matrices: M1..M4, T, M4 T, T M1
  float* matrix[4] = {lds, lds + CHUNK * row, lds + 2 * CHUNK * row, lds + 3 * CHUNK * row};
  float* decays = lds + 4 * CHUNK * row;
  float* inner = decays + CHUNK * row;
  float* small = decays;  // (the decays and the inner rows are of no use behind the running products)
  const T* rows = (const T*)a.main + (size_t)t0 * a.ld;

  // a wave takes four tokens and a lane two channels of each (dim <= 128): all of a wave's loads are asked for before the first
  // is used (tokens beyond the portion: zeros, with decays of 1)
  float r[4][2], k[4][2], al[4][2];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int j = wave + 4 * q;
    const T* mine = rows + (size_t)j * a.ld + (size_t)h * dim;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int c = lane + 64 * p;
      const bool there = j < count && c < dim;
      r[q][p] = there ? to_f32(mine[a.r_at + c]) : 0.f;
      k[q][p] = there ? to_f32(mine[a.k_at + c]) : 0.f;
      al[q][p] = there ? to_f32(mine[a.a_at + c]) : 0.f;
    }
  }
  const float bias[2] = {lane < dim ? a.a_bias[(size_t)h * dim + lane] : 0.f, lane + 64 < dim ? a.a_bias[(size_t)h * dim + lane + 64] : 0.f};
#pragma unroll 4
  for (int i = tid; i < CHUNK * padded_rank; i += 256) {
    const int j = i / padded_rank, m = i - j * padded_rank;
    inner[j * inner_row + m] = j < count && m < rank ? tanhf(to_f32(rows[(size_t)j * a.ld + a.low_at + m])) : 0.f;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int j = wave + 4 * q;
    const float inv = 1.f / sqrtf(wave_sum(k[q][0] * k[q][0] + k[q][1] * k[q][1]) + 1e-6f);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int c = lane + 64 * p;
      if (c < dim) {
        const float u = k[q][p] * inv;
        matrix[0][j * row + c] = u;
        matrix[1][j * row + c] = r[q][p];
        matrix[2][j * row + c] = removal_sigmoid(al[q][p] + bias[p]) * u;
        matrix[3][j * row + c] = k[q][p];
      }
    }
  }
  __syncthreads();
  // the decays: 16 channels x 16 tokens at a time, w2 [channel, m] times the inner rows; a lane ends with four neighbouring channels
  // of token n
  for (int tile = wave; tile < dim / 16; tile += 4) {
    const size_t channel = (size_t)h * dim + tile * 16;
    const T* w = (const T*)a.w2 + (channel + n) * rank;
    float4_t z = {0.f, 0.f, 0.f, 0.f};
    if (rank % 16 == 0 && ((uintptr_t)a.w2 & 15) == 0) {  // (then four neighbours of a row are one access)
#pragma unroll 4
      for (int m = 4 * g; m < padded_rank; m += 16) {
        float y[4];
        load4<T>(w, 0, m, rank, true, true, y);
        const float4_t x = four(inner + n * inner_row + m);
#pragma unroll
        for (int e = 0; e < 4; ++e) z = mfma4(y[e], x[e], z);
      }
    } else {
      for (int m = 4 * g; m < padded_rank; m += 16) {
        const float4_t x = four(inner + n * inner_row + m);
#pragma unroll
        for (int e = 0; e < 4; ++e) z = mfma4(m + e < rank ? to_f32(w[m + e]) : 0.f, x[e], z);
      }
    }
    float4_t dec;
#pragma unroll
    for (int i = 0; i < 4; ++i) dec[i] = n < count ? expf(-a.scale * removal_sigmoid(a.w0[channel + 4 * g + i] + z[i])) : 1.f;
    *reinterpret_cast<float4_t*>(decays + n * row + tile * 16 + 4 * g) = dec;
  }
  __syncthreads();
  // the running products and the scaled rows; a lane walks one channel of one of the four matrices
  float* record = a.scratch + ((size_t)record_at * a.heads + h) * removal_record(dim, a.vdim);
  float* record_b = record + 32 * dim;
  float* record_k = record + 48 * dim;
  float* record_p = record + 64 * dim;
  for (int i = tid; i < 4 * dim; i += 256) {
    const int which = i / dim, c = i - which * dim;
    float* column = matrix[which] + c;
    float p = 1.f;
    float4_t kept[4];
#pragma unroll
    for (int t = 0; t < CHUNK; ++t) {
      const float before = p;
      p *= decays[t * row + c];
      const float v = column[t * row] * (which == 0 ? before : which == 1 ? p : 1.f / p);
      column[t * row] = v;
      kept[t >> 2][t & 3] = which == 2 ? -v : v;
    }
    if (which >= 2) {
      float* to = (which == 2 ? record_b : record_k) + (size_t)c * CHUNK;
#pragma unroll
      for (int q = 0; q < 4; ++q) *reinterpret_cast<float4_t*>(to + 4 * q) = kept[q];
    }
    if (which == 0) record_p[c] = p;
  }
  __syncthreads();
  // M1 = U K^T, M2 = U B^T (below the diagonal), M3 = R K^T, M4 = R B^T (with it): a wave each
  {
    const float* left = matrix[wave < 2 ? 0 : 1] + n * row;
    const float* right = matrix[(wave & 1) ? 2 : 3] + n * row;
    float4_t m = {0.f, 0.f, 0.f, 0.f};
    for (int c = 4 * g; c < dim; c += 16) {
      const float4_t x = four(left + c), y = four(right + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) m = mfma4(x[e], y[e], m);
    }
    float* to = small + wave * CHUNK * CHUNK_STRIDE;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 4 * g + i;
      to[t * CHUNK_STRIDE + n] = n < t || (wave >= 2 && n == t) ? m[i] : 0.f;
    }
  }
  __syncthreads();
  const float* M1 = small;
  const float* M2 = small + CHUNK * CHUNK_STRIDE;
  const float* M3 = small + 2 * CHUNK * CHUNK_STRIDE;
  const float* M4 = small + 3 * CHUNK * CHUNK_STRIDE;
  float* inverse = small + 4 * CHUNK * CHUNK_STRIDE;
  float* M4T = small + 5 * CHUNK * CHUNK_STRIDE;
  float* TM1 = small + 6 * CHUNK * CHUNK_STRIDE;
  if (wave == 0) {  // column n of T, by substitution (the four groups of lanes do the same)
    float x[CHUNK];
#pragma unroll
    for (int t = 0; t < CHUNK; ++t) {
      float v = t == n ? 1.f : 0.f;
#pragma unroll
      for (int q = 0; q < (t + 3) / 4; ++q) {
        const float4_t m = four(M2 + t * CHUNK_STRIDE + 4 * q);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (4 * q + e < t) v -= m[e] * x[4 * q + e];
      }
      x[t] = v;
    }
    if (g == 0) {
#pragma unroll
      for (int t = 0; t < CHUNK; ++t) inverse[t * CHUNK_STRIDE + n] = x[t];
    }
  }
  __syncthreads();
  if (wave < 2) {  // M4 T and T M1
    const float4_t x = four((wave == 0 ? M4 : inverse) + n * CHUNK_STRIDE + 4 * g);
    const float* y = (wave == 0 ? inverse : M1) + 4 * g * CHUNK_STRIDE + n;
    float4_t m = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) m = mfma4(x[e], y[e * CHUNK_STRIDE], m);
    float* to = wave == 0 ? M4T : TM1;
#pragma unroll
    for (int i = 0; i < 4; ++i) to[(4 * g + i) * CHUNK_STRIDE + n] = m[i];
  }
  __syncthreads();
  const float4_t t4 = four(inverse + n * CHUNK_STRIDE + 4 * g), m4t = four(M4T + n * CHUNK_STRIDE + 4 * g);
  for (int tile = wave; tile < dim / 16; tile += 4) {  // U' and R', 16 channels at a time
    float4_t up = {0.f, 0.f, 0.f, 0.f}, rp;
#pragma unroll
    for (int i = 0; i < 4; ++i) rp[i] = matrix[1][(4 * g + i) * row + tile * 16 + n];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float y = matrix[0][(4 * g + e) * row + tile * 16 + n];
      up = mfma4(t4[e], y, up);
      rp = mfma4(-m4t[e], y, rp);
    }
    float* to = record + tile * 256 + n;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      to[(4 * g + i) * 16] = up[i];
      to[16 * dim + (4 * g + i) * 16] = rp[i];
    }
  }
  const float4_t m3 = four(M3 + n * CHUNK_STRIDE + 4 * g), m4 = four(M4 + n * CHUNK_STRIDE + 4 * g), tm1 = four(TM1 + n * CHUNK_STRIDE + 4 * g);
  const int columns = removal_columns(a.vdim);
  float* record_d = record + 65 * dim;
  for (int tile = wave; tile < columns / 16; tile += 4) {  // Dv and Ov, 16 columns of values at a time
    const int column = tile * 16 + n;
    const T* values = rows + a.v_at + (size_t)h * a.vdim + (column < a.vdim ? column : a.vdim - 1);
    float4_t v, dv = {0.f, 0.f, 0.f, 0.f}, ov = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = 4 * g + e < count ? to_f32(values[(size_t)(4 * g + e) * a.ld]) : 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      dv = mfma4(tm1[e], v[e], dv);
      ov = mfma4(m3[e], v[e], ov);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) ov = mfma4(-m4[e], dv[e], ov);
    *reinterpret_cast<float4_t*>(record_d + (size_t)column * CHUNK + 4 * g) = dv;
    *reinterpret_cast<float4_t*>(record_d + (size_t)(columns + column) * CHUNK + 4 * g) = ov;
    *reinterpret_cast<float4_t*>(record_d + (size_t)(2 * columns + column) * CHUNK + 4 * g) = v;
  }
}

// What a wave reads of one chunk, in registers: loaded SCAN_AHEAD chunks before it is worked.
struct RemovalOperands { float4_t up, nb, k, p, dv, v; };
// Up to 64 channels the read-outs have waves of their own.
__host__ __device__ constexpr bool removal_readers(int waves) { return waves <= 4; }
template <int WAVES>
struct RemovalReads {
  static constexpr int EACH = WAVES >= 4 ? 1 : (4 + WAVES - 1) / WAVES;  // read-outs of a chunk that a lane finishes
  float4_t rp;
  float before[EACH];  // of the chunk before, whose read-outs are finished one chunk later
};
#define SCAN_AHEAD 4

// Bound by the chain of chunks on the few compute units that have a workgroup: per chunk the four dependent products that make a wave's part of D,
// its way through LDS and a barrier, and the four that take it from the state.  So nothing else is in that chain's way: with READERS a second
// set of waves, on the same SIMDs, gets the state in front of every chunk through LDS, makes O of it and finishes the read-outs a chunk
// later (without, the chain's waves do so while D's parts are under way), and buffer loads and stores leave the vector unit no addresses
// to add up.  One barrier a chunk: a buffer of `removed` or `states` is written again behind the next chunk's barrier, one of `reads` behind the
// one that follows its readers'.  Measured on MI355X, 64 chunks, 32 heads of 64 x 64: 41.0 us with everything in one chain, 35.8 with the read-outs
// a chunk later and buffer operations, 31.0 with waves of their own for them.
// (At most 256 registers a wave: the matrix instructions then keep the state in ordinary registers.  There is no bound from above on a SIMD's waves: for
// one the compiler asks for registers that nothing uses, and many short chains wait.)  Prepared and scanned, with everything in one chain / like this (with
// one workgroup a compute unit and loads ahead for single tokens), us: 32 heads of 64 x 64, 64 portions of 64 276 / 269 (390), 60 single tokens beside
// 1,024 150 / 109 (242), 200 beside 300 309 / 249 (409); 16 heads of 128 x 128 456 / 453 (549), 259 / 185 (333), 589 / 435 (649), 100 portions
// of 40 tokens 530 / 520 (560, and 561 where they asked for loads ahead and finished read-outs of no chunk).
template <int WAVES>
__global__ void __launch_bounds__(64 * WAVES * (removal_readers(WAVES) ? 2 : 1)) __attribute__((amdgpu_waves_per_eu(2))) removal_chunk_scan_kernel(const RemovalChunkArgs a) {
  constexpr bool READERS = removal_readers(WAVES);
  __shared__ float4_t removed[2][WAVES][64], reads[2][WAVES][64], states[READERS ? 2 : 1][READERS ? WAVES : 1][64];  // the waves' parts of D and O, [buffer][wave][lane]
  // (heads lie along the grid fastest in both kernels: with a multiple of 8 heads the workgroups that read a record run
  // on the XCD that wrote it and share it in that XCD's L2)
  // (the long chains begin first, not when the single tokens in front of them are done: 12 beside 1,024, 32 heads of 64 x 64, 49 -> 38 us;
  // prepared and scanned 94 -> 83, and 76 since those ask for their own chunk alone)
  const int h = blockIdx.x, tile = blockIdx.y, b = __builtin_amdgcn_readfirstlane(sequence_by_length(a.cu_q, gridDim.z, blockIdx.z, a.ordered));
  const int lo = __builtin_amdgcn_readfirstlane(a.cu_q[b]), hi = __builtin_amdgcn_readfirstlane(a.cu_q[b + 1]);
  if (hi <= lo) return;  // (the whole workgroup)
  const int lane = threadIdx.x & 63, any_wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = any_wave % WAVES, tid = wave * 64 + lane;
  const int n = lane & 15, g = lane >> 4;
  constexpr int dim = 16 * WAVES;
  constexpr int EACH = RemovalReads<WAVES>::EACH;
  const int vdim = a.vdim, columns = removal_columns(vdim);
  const int column = tile * 16 + n;
  const bool live = column < vdim;
  const int chunks = (hi - lo + CHUNK - 1) / CHUNK;
  const size_t stride = (size_t)a.heads * removal_record(dim, vdim);  // between a sequence's records of this head
  // a lane's places in a record, in bytes (the record's own address is the same for the whole wave and moves from chunk to chunk)
  const uint32_t rows_at = 4 * (wave * 256 + n * 16 + 4 * g), decays_at = 4 * (64 * dim + wave * 16 + 4 * g), column_at = 4 * (65 * dim + column * CHUNK + 4 * g);
  uint32_t reads_at[EACH], out_at[EACH];
#pragma unroll
  for (int q = 0; q < EACH; ++q) {
    const int i = tid + q * 64 * WAVES, t = ((i >> 6) & 3) * 4 + (i & 3), e = (i >> 2) & 15;  // a read-out's place in the order in which the parts lie in LDS
    reads_at[q] = 4 * (65 * dim + (columns + tile * 16 + e) * CHUNK + t);
    out_at[q] = i < 256 && tile * 16 + e < vdim ? 4u * (t * (uint32_t)a.heads * vdim + e) : 0x80000000u;  // (behind any row: not stored)
  }
  const float* next = a.scratch + ((size_t)removal_first_chunk(lo, b) * a.heads + h) * removal_record(dim, vdim);
  const float* before = next;
  const int record_bytes = 4 * (int)removal_record(dim, vdim);
  auto record_of = [&](const float* at) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(at), 0, record_bytes, 0x00020000); };
  auto load_reads = [&](float (&ov)[EACH], const float* at) {
    const auto record = record_of(at);
#pragma unroll
    for (int q = 0; q < EACH; ++q) ov[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(record, reads_at[q], 0, 0));
  };
  float* S = a.state + (((size_t)a.slots[b] * a.heads + h) * dim + wave * 16 + 4 * g) * vdim + (live ? column : vdim - 1);
  const size_t out_row = (size_t)a.heads * vdim;
  float* out = a.out + (size_t)lo * out_row + (size_t)h * vdim + tile * 16;
  const int row_bytes = 4 * (int)out_row;
  int pending = 0, left = hi - lo;  // tokens whose parts of O lie in LDS, tokens behind them

  // What a wave does: CHAINS the chain, READS the read-outs.  (A loop each, so that no load sits behind a branch.)
  auto run = [&](auto chains_too, auto reads_too) {
    constexpr bool CHAINS = decltype(chains_too)::value, READS = decltype(reads_too)::value;
    float last_reads[EACH];
    if constexpr (READS) load_reads(last_reads, next + (size_t)(chunks - 1) * stride);
    int asked = 0;  // chunks asked for so far
    auto load = [&](RemovalOperands& o, RemovalReads<WAVES>& r) {
      __builtin_amdgcn_sched_barrier(0);  // (in this order on every path: a wait counts the loads that are younger)
      const auto record = record_of(next);
      auto piece = [&](uint32_t at, int from) { return __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(record, at, 4 * from, 0)); };
      if constexpr (CHAINS) {
        o.up = piece(rows_at, 0);
        o.nb = piece(rows_at, 32 * dim);
        o.k = piece(rows_at, 48 * dim);
        o.p = piece(decays_at, 0);
        o.dv = piece(column_at, 0);
        o.v = piece(column_at, 32 * columns);
      }
      if constexpr (READS) {
        r.rp = piece(rows_at, 16 * dim);
        load_reads(r.before, before);
        before = next;
      }
      __builtin_amdgcn_sched_barrier(0);
      ++asked;
      if (asked < chunks) next += stride;  // (beyond the last chunk the last one is asked for again)
    };
    // The read-outs of a chunk, 256 over the readers' lanes, behind the barrier that follows their parts.
    auto read_out = [&](int buffer, const float (&ov)[EACH]) {
      const float* sums = reinterpret_cast<const float*>(reads[buffer]);
      const auto rows = __builtin_amdgcn_make_buffer_rsrc(out, 0, pending * row_bytes, 0x00020000);  // (what lies behind the last token is not stored)
#pragma unroll
      for (int q = 0; q < EACH; ++q) {
        float v = ov[q];
#pragma unroll
        for (int w = 0; w < WAVES; ++w) v += sums[w * 256 + ((tid + q * 64 * WAVES) & 255)];
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), rows, out_at[q], 0, 0);
      }
      out += pending * out_row;
      pending = left < CHUNK ? left : CHUNK;
      left -= pending;
    };
    auto meet = [&] {  // (what every wave has written to LDS is there; each loop comes here as often)
      asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" : : : "memory");
    };
    float4_t z = {0.f, 0.f, 0.f, 0.f};
    if constexpr (CHAINS) {
#pragma unroll
      for (int i = 0; i < 4; ++i) z[i] = S[(size_t)i * vdim];
    }
    // `first`: no read-outs of a chunk before it are finished beside it
    auto work = [&](auto first, int buffer, const RemovalOperands& o, const RemovalReads<WAVES>& r) {
      auto finish_before = [&] {
        if constexpr (decltype(first)::value) {
          pending = left < CHUNK ? left : CHUNK;
          left -= pending;
        } else {
          read_out(1 - buffer, r.before);
        }
      };
      float4_t d = {0.f, 0.f, 0.f, 0.f}, read = d, kept = z;
      if constexpr (CHAINS) {
        if constexpr (!READS) states[buffer][wave][lane] = z;
#pragma unroll
        for (int e = 0; e < 4; ++e) d = mfma4(o.up[e], z[e], d);
        __builtin_amdgcn_sched_barrier(0);
        removed[buffer][wave][lane] = d;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (READS) read = mfma4(r.rp[e], z[e], read);
          else kept = mfma4(o.k[e], o.v[e], kept);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      meet();
      if constexpr (CHAINS) {
        d = o.dv;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) d += removed[buffer][w][lane];
        if constexpr (READS) {
          reads[buffer][wave][lane] = read;
#pragma unroll
          for (int e = 0; e < 4; ++e) kept = mfma4(o.k[e], o.v[e], kept);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) kept = mfma4(o.nb[e], d[e], kept);
        if constexpr (READS) finish_before();
        z = kept * o.p;
      } else {
        const float4_t state = states[buffer][wave][lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) read = mfma4(r.rp[e], state[e], read);
        finish_before();
        reads[buffer][wave][lane] = read;
      }
    };
    // Loads are asked for whether or not there is a chunk that far ahead (then the last one's again): the same number of them lies
    // between a chunk's loads and its work on every path, so that waiting for the one does not wait for the others.
    RemovalOperands ops[SCAN_AHEAD];
    RemovalReads<WAVES> of_reads[SCAN_AHEAD];
    if (chunks < SCAN_AHEAD) {  // (single tokens and short portions ask for their own chunks alone)
#pragma unroll
      for (int j = 0; j < SCAN_AHEAD - 1; ++j)
        if (j < chunks) load(ops[j], of_reads[j]);
      work(std::true_type{}, 0, ops[0], of_reads[0]);
#pragma unroll
      for (int j = 1; j < SCAN_AHEAD - 1; ++j)
        if (j < chunks) work(std::false_type{}, j & 1, ops[j], of_reads[j]);
    } else {
#pragma unroll
      for (int j = 0; j < SCAN_AHEAD; ++j) load(ops[j], of_reads[j]);
      int c = 0;
      for (; c + SCAN_AHEAD <= chunks; c += SCAN_AHEAD) {
#pragma unroll
        for (int j = 0; j < SCAN_AHEAD; ++j) {
          work(std::false_type{}, j & 1, ops[j], of_reads[j]);
          load(ops[j], of_reads[j]);
        }
      }
#pragma unroll
      for (int j = 0; j < SCAN_AHEAD - 1; ++j)
        if (c + j < chunks) work(std::false_type{}, j & 1, ops[j], of_reads[j]);  // (the same for the whole workgroup)
    }
    meet();
    if constexpr (READS) read_out((chunks - 1) & 1, last_reads);
    if constexpr (CHAINS) {
      if (live) {
#pragma unroll
        for (int i = 0; i < 4; ++i) S[(size_t)i * vdim] = z[i];
      }
    }
  };
  if constexpr (!READERS) run(std::true_type{}, std::true_type{});
  else if (any_wave < WAVES) run(std::true_type{}, std::false_type{});
  else run(std::false_type{}, std::true_type{});
}

// LDS of removal_chunk_prepare_kernel.  Its time is that of its dependent steps, so workgroups per compute unit count: with the small
// matrices where the decays were six instead of four of them hold 64 channels and an inner size of 64 (26 KB, not 35).
static size_t removal_prepare_lds(int dim, int rank) {
  const int row = dim + 4, inner_row = (rank + 15) / 16 * 16 + 4;
  return (size_t)CHUNK * (4 * row + (row + inner_row > 7 * CHUNK_STRIDE ? row + inner_row : 7 * CHUNK_STRIDE)) * sizeof(float);
}

// float32 elements of the scratch of a step; 0: these sizes are not for these kernels
extern "C" long long velox_removal_chunk_scratch_elems(int tokens, int num_seqs, int heads, int dim, int vdim, int rank) {
  if (dim % 16 != 0 || dim < 16 || dim > 128 || vdim < 1 || rank < 1 || removal_prepare_lds(dim, rank) > 55 * 1024) return 0;
  return (step_items(tokens, num_seqs, CHUNK) + 1) * heads * (long long)removal_record(dim, vdim);
}

template <typename T>
static void removal_chunk_launch(RemovalChunkArgs a, int tokens, int num_seqs, hipStream_t stream) {
  // (1,024 tokens beside 12 single ones, 32 heads of 64 x 64, us: with the longest portion's chunks for every sequence 55.4, so 51.0, and six workgroups per
  // compute unit 44.4)
  const dim3 grid(a.heads, removal_columns(a.vdim) / 16, num_seqs);
  const long long workgroups = (long long)grid.x * grid.y * grid.z;
  a.ordered = orders_sequences(workgroups, num_seqs);
  const size_t alone = workgroups <= ALONE_WORKGROUPS ? ALONE_LDS : 0;
  removal_chunk_prepare_kernel<T><<<(unsigned)(a.heads * step_items(tokens, num_seqs, CHUNK)), 256, removal_prepare_lds(a.dim, a.rank), stream>>>(a, num_seqs);
  switch (a.dim / 16) {
    case 1: removal_chunk_scan_kernel<1><<<grid, 128, alone, stream>>>(a); break;
    case 2: removal_chunk_scan_kernel<2><<<grid, 256, alone, stream>>>(a); break;
    case 3: removal_chunk_scan_kernel<3><<<grid, 384, alone, stream>>>(a); break;
    case 4: removal_chunk_scan_kernel<4><<<grid, 512, alone, stream>>>(a); break;
    case 5: removal_chunk_scan_kernel<5><<<grid, 320, alone, stream>>>(a); break;
    case 6: removal_chunk_scan_kernel<6><<<grid, 384, alone, stream>>>(a); break;
    case 7: removal_chunk_scan_kernel<7><<<grid, 448, alone, stream>>>(a); break;
    default: removal_chunk_scan_kernel<8><<<grid, 512, alone, stream>>>(a); break;
  }
}

extern "C" int velox_removal_chunk_scan(const void* main, int dtype, int ld, int r_at, int k_at, int v_at, int a_at, int low_at, int rank, int heads, int dim,
                                        int vdim, const float* a_bias, const void* w2, const float* w0, float scale, float* scratch, float* state,
                                        const int* slots, const int* cu_q, float* out, int tokens, int num_seqs, hipStream_t stream) {
  if (num_seqs <= 0 || tokens <= 0) return 0;
  if (velox_removal_chunk_scratch_elems(tokens, num_seqs, heads, dim, vdim, rank) == 0 || heads < 1 || heads > 65535 || num_seqs > 65535 ||
      heads * step_items(tokens, num_seqs, CHUNK) > 0x7fffffff || !scratch || !(scale * CHUNK < 13.f))
    return (int)hipErrorInvalidValue;
  RemovalChunkArgs a{main, ld, r_at, k_at, v_at, a_at, low_at, rank, heads, dim, vdim, a_bias, w2, w0, scale, scratch, state, slots, cu_q, out, false};
  if (dtype == VELOX_BF16) removal_chunk_launch<bf16_t>(a, tokens, num_seqs, stream);
  else removal_chunk_launch<float>(a, tokens, num_seqs, stream);
  VELOX_RETURN_LAUNCH_STATUS();
}
