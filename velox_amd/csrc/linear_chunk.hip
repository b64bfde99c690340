// The gated delta rule and gated linear attention over long portions of prompts, in chunks of 16 tokens on the float32 matrix
// instructions.
//
// Per head, with decays g_t (a number or one per key channel, at most 1), key k_t, query q_t, value v_t and update gate b_t:
//     S <- diag(g_t) S;   u_t = b_t (v_t - S^T k_t)  ("delta")  or  u_t = v_t  ("additive");   S <- S + k_t u_t^T;   o_t = S^T q_t.
// Inside a chunk let P_t = g_1 .. g_t and P(j, t) = g_(j+1) .. g_t, all per channel.  From the state Z before the chunk
//     u_t = b_t (v_t - (k_t P_t)^T Z - sum_(j<t) M1_tj u_j),   M1_tj = sum_c k_tc k_jc P(j, t)_c,
//     o_t = (q_t P_t)^T Z + sum_(j<=t) M3_tj u_j,              M3_tj = sum_c q_tc k_jc P(j, t)_c,
//     S' = diag(P_16) Z + sum_j (k_j P(j, 16)) u_j^T.
// With T = (I + diag(b) M1)^-1 diag(b) (unit lower triangular, by substitution; M1 below the diagonal, M3 with it) everything that
// does not touch the state is worked for all chunks at the same time:
//     U' = T (k P),  Dv = T V,  R' = q P - M3 U',  Ov = M3 Dv          (additive: Dv = V, R' = q P, Ov = M3 V)
// and what is left of the dependent chain is, per chunk,   D = Dv - U' Z,   O = R' Z + Ov,   S' = diag(P_16) Z + K'^T D.
// All of it is float32 and no quotient of decays is ever formed: a decay may underflow to 0 and nothing else does.  M1 and M3 are
// built from products of rows whose factors are at most 1: at the level of blocks of 2 h tokens (h = 8, 4, 2, 1) a token t of a
// block's second half and a token j of its first meet as k_t P(m, t) and k_j P(j, m) with m the last token of the first half, so
// every pair below the diagonal belongs to exactly one level, and a level is one 16 x 16 product over the channels.
// What T, M3 and M3 T have above the diagonal is zero, but zero times an infinity or a NaN of a later token is not: a tile that
// holds one is multiplied without those terms (lower_times), so that such a value reaches its own token and later ones only.
//
// Sequences of fewer than `long_from` tokens are left to the kernels that go token by token, whatever else is in the step, and a
// step whose records would not fit the scratch is worked some heads at a time: a sequence's bits depend on its own tokens alone.
//
//   linear_chunk_prepare_kernel   a workgroup per chunk and head: a wave per level, then T and the matrices above into `scratch`
//   linear_chunk_scan_kernel      a workgroup per 16 value columns, head and sequence; a wave holds 16 rows of the state in the
//                                 matrix instructions' result layout, which is also their operand layout; the waves exchange
//                                 their parts of D through LDS with one barrier a chunk, others make O, loads four chunks ahead
// The first is bound by what it moves (41 KB of records a chunk and head of 128 x 128), the second by the chain: per chunk four
// matrix instructions, a barrier, a sum over the waves' parts, four more: 0.67 us.  Measured on MI355X, three prompts of 400 to
// 1,300 tokens (2,421 in all), 8 heads of 128 x 128: 31 + 55 us against 377 us token by token (a column of the state per wave);
// 16 heads 52 + 58 against 447; additive, 8 heads of 128 x 256: 35 + 41 against 370.
#include "common.h"

#define CHUNK 16
#define CHUNK_STRIDE 20  // floats between the rows of a 16 x 16 matrix in LDS (16-byte aligned, rows on different banks)

struct LinearChunkArgs {
  const float* qk;     // [T, kv_heads, 2, dim]
  const void* v;       // values of a token's head h at v_at + h * vdim of its row
  int v_bf16, v_ld, v_at;
  const float* decay;  // [T, heads] or [T, heads * dim]
  int decay_per_channel;
  const float* beta;   // [T, heads] (delta)
  float* scratch;
  float* state;        // [slots, heads, dim, vdim]
  const int* slots;
  const int* cu_q;
  float* out;          // [T, heads * vdim]
  int heads, kv_heads, dim, vdim;
  int num_seqs, long_from;      // sequences of at least long_from tokens are worked
  int first_head, head_count;   // the heads that this launch works; their records lie side by side in `scratch`
  bool ordered;                 // the scan's sequences by their length, see sequence_by_length
};

// A chunk and head in `scratch`, in floats: -U' | R' | K' (each 16 * dim), P_16 (dim), Dv | Ov (each 16 * columns).  U' and R' as
// [dim / 16][16 tokens][16 channels], K' as [dim][16 tokens], Dv and Ov as [columns][16 tokens]: what a wave reads of one of them is
// one contiguous kilobyte, 16 bytes a lane.
__host__ __device__ __forceinline__ int chunk_columns(int vdim) { return (vdim + 15) / 16 * 16; }
__host__ __device__ __forceinline__ size_t chunk_record(int dim, int vdim) { return (size_t)49 * dim + 32 * chunk_columns(vdim); }
// the first record of a sequence: sequences' chunks never overlap, because floor((a + n) / 16) + 1 >= floor(a / 16) + ceil(n / 16)
__device__ __forceinline__ int first_chunk(int first_token, int sequence) { return first_token / CHUNK + sequence; }

__device__ __forceinline__ float4_t mfma4(float a, float b, float4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ float4_t four(const float* p) { return *reinterpret_cast<const float4_t*>(p); }

// acc + L y for a lower triangular L (16 x 16, in LDS; `l`: row n's entries 4 g .. + 3) and a tile y of which lane (n, g) holds rows
// 4 g .. + 3 of column n; the result in the same layout.  The same for the whole wave.
__device__ __forceinline__ float4_t lower_times(const float4_t l, const float* L, const float4_t y, float4_t acc, int n, int g) {
  const float zero = y[0] * 0.f + y[1] * 0.f + y[2] * 0.f + y[3] * 0.f;
  if (__ballot(!(zero == 0.f)) == 0ull) {
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = mfma4(l[e], y[e], acc);
    return acc;
  }
#pragma unroll
  for (int j = 0; j < CHUNK; ++j) {
    const float yj = __shfl(y[j & 3], n + 16 * (j >> 2), VELOX_WAVE);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (j <= 4 * g + i) acc[i] += L[(4 * g + i) * CHUNK_STRIDE + j] * yj;
  }
  return acc;
}

// The grid counts records, of which there are about as many as chunks: one per longest portion's chunk and sequence would be a hundred
// thousand workgroups that only end, for 60 single tokens beside 1,000.  Measured on MI355X (us a step with the kernels for the short ones
// behind it; token by token / everything in chunks with such a grid / this): 60 single tokens beside 1,000, 16 heads of 128 x 128 519 / 195 /
// 149, 32 heads 677 / 359 / 238; beside 64 131 / 141 / 87, 240 / 239 / 147; 12 beside 300 142 / 62 / 56; 1 beside 300 92 / 35 / 41.
template <bool DELTA>
__global__ void __launch_bounds__(256) linear_chunk_prepare_kernel(const LinearChunkArgs a) {
  extern __shared__ float4_t lds_pieces[];
  float* lds = reinterpret_cast<float*>(lds_pieces);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int record_at = blockIdx.x / a.head_count, local_head = blockIdx.x % a.head_count, h = a.first_head + local_head;
  const StepItem item = step_item(a.cu_q, a.num_seqs, CHUNK, record_at);
  const int lo = item.lo, hi = item.hi, t0 = lo + item.piece * CHUNK;
  if (t0 >= hi || hi - lo < a.long_from) return;  // (the whole workgroup)
  const int count = hi - t0 < CHUNK ? hi - t0 : CHUNK;
  const int n = lane & 15, g = lane >> 4;  // column and group of four rows in the matrix instructions' layouts
  const int dim = a.dim, row = dim + 4;
  // rows of q, k and the decays (16 x dim each), and 16 x 16 matrices: M1, M3, T, M3 T
  float* q = lds;
  float* k = lds + CHUNK * row;
  float* decays = lds + 2 * CHUNK * row;
  float* M1 = lds + 3 * CHUNK * row;
  float* M3 = M1 + CHUNK * CHUNK_STRIDE;
  float* T = M1 + 2 * CHUNK * CHUNK_STRIDE;
  float* M3T = M1 + 3 * CHUNK * CHUNK_STRIDE;

  // the rows, four channels a lane at a time (tokens beyond the portion: zeros, with decays of 1)
  const int quads = dim / 4;
  const int kv = h / (a.heads / a.kv_heads);
  for (int at = tid; at < CHUNK * quads; at += 256) {
    const int j = at / quads, c = 4 * (at - j * quads);
    const bool there = j < count;
    const size_t t = t0 + (there ? j : 0);
    const float* qk = a.qk + (t * a.kv_heads + kv) * 2 * dim + c;
    const float4_t zero = {0.f, 0.f, 0.f, 0.f}, one = {1.f, 1.f, 1.f, 1.f};
    float4_t dec;
    if (a.decay_per_channel) {
      dec = four(a.decay + (t * a.heads + h) * dim + c);
    } else {
      const float d = a.decay[t * a.heads + h];
      dec = float4_t{d, d, d, d};
    }
    *reinterpret_cast<float4_t*>(q + j * row + c) = there ? four(qk) : zero;
    *reinterpret_cast<float4_t*>(k + j * row + c) = there ? four(qk + dim) : zero;
    *reinterpret_cast<float4_t*>(decays + j * row + c) = there ? dec : one;
  }
  __syncthreads();

  // M1 and M3 level by level, a wave each: half = 8, 4, 2, 1; lane (n, g) scales channels 4 g + 16 m .. + 3 of token n's rows
  {
    const int half = 8 >> wave;
    const int middle = (n & ~(2 * half - 1)) + half - 1;  // the last token of the first half of n's block
    const bool second = (n & half) != 0;
    const int first = second ? middle + 1 : n + 1, last = second ? n : middle;
    float4_t m1 = {0.f, 0.f, 0.f, 0.f}, m3 = m1, diagonal = m1;
    for (int c = 4 * g; c < dim; c += 16) {
      const float4_t kn = four(k + n * row + c), qn = four(q + n * row + c);
      float4_t f = {1.f, 1.f, 1.f, 1.f};
      for (int s = 0; s < half; ++s) {
        const int t = first + s <= last ? first + s : last;
        const float4_t d = four(decays + (t < 0 ? 0 : t) * row + c);
        if (first + s <= last) f *= d;
      }
      const float4_t ks = kn * f, qs = qn * f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (DELTA) m1 = mfma4(ks[e], ks[e], m1);
        m3 = mfma4(qs[e], ks[e], m3);
      }
      if (wave == 3) {
#pragma unroll
        for (int e = 0; e < 4; ++e) diagonal = mfma4(qn[e], kn[e], diagonal);
      }
    }
    // lane (n, g) holds rows 4 g + i of column n; a level owns the pairs (second half, first half) of its blocks
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 4 * g + i;
      const bool same = (t & ~(2 * half - 1)) == (n & ~(2 * half - 1));
      if (same && (t & half) != 0 && (n & half) == 0) {
        if (DELTA) M1[t * CHUNK_STRIDE + n] = m1[i];
        M3[t * CHUNK_STRIDE + n] = m3[i];
      }
      if (wave == 3 && t == n) M3[t * CHUNK_STRIDE + n] = diagonal[i];
      if (wave == 2 && t < n) M3[t * CHUNK_STRIDE + n] = 0.f;
    }
  }
  // the running products: a lane walks one channel forwards (k P and q P, in place behind the barrier) or backwards (K')
  __syncthreads();
  float* record = a.scratch + ((size_t)record_at * a.head_count + local_head) * chunk_record(dim, a.vdim);
  float* record_k = record + 32 * dim;
  float* record_p = record + 48 * dim;
  for (int c = tid; c < dim; c += 256) {
    float p = 1.f;
    float4_t kept[4];
#pragma unroll
    for (int t = CHUNK - 1; t >= 0; --t) {
      kept[t >> 2][t & 3] = k[t * row + c] * p;
      p *= decays[t * row + c];
    }
    record_p[c] = p;
#pragma unroll
    for (int s = 0; s < 4; ++s) *reinterpret_cast<float4_t*>(record_k + (size_t)c * CHUNK + 4 * s) = kept[s];
    p = 1.f;
#pragma unroll
    for (int t = 0; t < CHUNK; ++t) {
      p *= decays[t * row + c];
      k[t * row + c] *= p;
      q[t * row + c] *= p;
    }
  }
  if (DELTA && wave == 3) {  // column n of T, by substitution (the four groups of lanes do the same)
    float x[CHUNK];
    const float own = n < count ? a.beta[(size_t)(t0 + n) * a.heads + h] : 0.f;
#pragma unroll
    for (int t = 0; t < CHUNK; ++t) {
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < t; ++j) sum += M1[t * CHUNK_STRIDE + j] * x[j];
      const float bt = __shfl(own, t, VELOX_WAVE);
      x[t] = (t == n ? 1.f : 0.f) - bt * sum;
    }
    if (g == 0) {
#pragma unroll
      for (int t = 0; t < CHUNK; ++t) T[t * CHUNK_STRIDE + n] = t < n ? 0.f : x[t] * own;
    }
  }
  __syncthreads();
  if (DELTA && wave == 0) {  // M3 T
    float4_t t4;
#pragma unroll
    for (int e = 0; e < 4; ++e) t4[e] = T[(4 * g + e) * CHUNK_STRIDE + n];
    const float4_t m = lower_times(four(M3 + n * CHUNK_STRIDE + 4 * g), M3, t4, float4_t{0.f, 0.f, 0.f, 0.f}, n, g);
#pragma unroll
    for (int i = 0; i < 4; ++i) M3T[(4 * g + i) * CHUNK_STRIDE + n] = m[i];
  }
  if (DELTA) __syncthreads();
  const float4_t t4 = DELTA ? four(T + n * CHUNK_STRIDE + 4 * g) : float4_t{}, m3t = DELTA ? four(M3T + n * CHUNK_STRIDE + 4 * g) : float4_t{};
  for (int tile = wave; tile < dim / 16; tile += 4) {  // -U' and R', 16 channels at a time
    float4_t up = {0.f, 0.f, 0.f, 0.f}, rp;
#pragma unroll
    for (int i = 0; i < 4; ++i) rp[i] = q[(4 * g + i) * row + tile * 16 + n];
    if (DELTA) {
      float4_t minus_k;
#pragma unroll
      for (int e = 0; e < 4; ++e) minus_k[e] = -k[(4 * g + e) * row + tile * 16 + n];
      up = lower_times(t4, T, minus_k, up, n, g);
      rp = lower_times(m3t, M3T, minus_k, rp, n, g);
    }
    float* to = record + tile * 256 + n;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (DELTA) to[(4 * g + i) * 16] = up[i];
      to[16 * dim + (4 * g + i) * 16] = rp[i];
    }
  }
  const float4_t m3 = four(M3 + n * CHUNK_STRIDE + 4 * g);
  const int columns = chunk_columns(a.vdim);
  float* record_d = record + 49 * dim;
  for (int tile = wave; tile < columns / 16; tile += 4) {  // Dv and Ov, 16 columns of values at a time
    const int column = tile * 16 + n;
    const size_t at = (size_t)t0 * a.v_ld + a.v_at + (size_t)h * a.vdim + (column < a.vdim ? column : a.vdim - 1);
    float4_t v, dv = {0.f, 0.f, 0.f, 0.f}, ov = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const size_t token = at + (size_t)(4 * g + e < count ? 4 * g + e : 0) * a.v_ld;
      const float x = a.v_bf16 ? to_f32(((const bf16_t*)a.v)[token]) : ((const float*)a.v)[token];
      v[e] = 4 * g + e < count ? x : 0.f;
    }
    dv = DELTA ? lower_times(t4, T, v, dv, n, g) : v;
    ov = lower_times(m3, M3, dv, ov, n, g);
    *reinterpret_cast<float4_t*>(record_d + (size_t)column * CHUNK + 4 * g) = dv;
    *reinterpret_cast<float4_t*>(record_d + (size_t)(columns + column) * CHUNK + 4 * g) = ov;
  }
}

// What a wave reads of one chunk, in registers: loaded SCAN_AHEAD chunks before it is worked.
struct ChunkOperands { float4_t up, k, p, dv; };
struct ChunkReads {
  float4_t rp;
  float before;  // of the chunk before, whose read-outs are finished one chunk later
};
#define SCAN_AHEAD 4

// Bound by the chain of chunks on the few compute units that have a workgroup: per chunk the four dependent products that make a wave's part of D,
// its way through LDS and a barrier, and the four that add it to the state.  Nothing else is in that chain's way: the first WAVES waves
// work it, and as many others, on the same SIMDs, get the state in front of every chunk through LDS, make O of it and finish the
// read-outs a chunk later; buffer loads and stores leave the vector unit no addresses to add up.  One barrier a chunk: a buffer of `removed`
// or `states` is written again behind the next chunk's barrier, one of `reads` behind the one that follows its readers'.  Measured on MI355X,
// 82 chunks of the longest of three sequences, us, with everything in one chain / this: 8 heads of 128 x 128 72 / 55, 16 heads 77 / 58, additive, 8
// heads of 128 x 256, 46 / 41.  Many short chains, prepared and scanned (with one workgroup a compute unit): 32 heads of 64 x 64, 64 portions of 64
// 189 / 184 (288), of 200 488 / 477 (592); 32 heads of 128 x 128 613 / 530 (710), additive, 8 heads of 128 x 256, 202 / 183 (282): there is no bound from
// above on a SIMD's waves, and the additive rule's fit the registers of eight.
template <int WAVES, bool DELTA>
__global__ void __launch_bounds__(128 * WAVES) __attribute__((amdgpu_waves_per_eu(DELTA ? WAVES / 2 : 8))) linear_chunk_scan_kernel(const LinearChunkArgs a) {
  static_assert(WAVES == 4 || WAVES == 8, "a chunk's 256 read-outs are finished by 256 lanes of the readers");
  __shared__ float4_t removed[2][DELTA ? WAVES : 1][64], reads[2][WAVES][64], states[2][WAVES][64];  // [buffer][wave][lane]
  // (heads lie along the grid's first dimension in both kernels: with a multiple of 8 heads the workgroups that read a record run
  // on the XCD that wrote it and share it in that XCD's L2)
  const int h = a.first_head + blockIdx.x, tile = blockIdx.y, b = __builtin_amdgcn_readfirstlane(sequence_by_length(a.cu_q, a.num_seqs, blockIdx.z, a.ordered));
  const int lo = __builtin_amdgcn_readfirstlane(a.cu_q[b]), hi = __builtin_amdgcn_readfirstlane(a.cu_q[b + 1]);
  if (hi - lo < a.long_from || hi <= lo) return;  // (the whole workgroup)
  const int lane = threadIdx.x & 63, any_wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = any_wave % WAVES, tid = wave * 64 + lane;
  const int n = lane & 15, g = lane >> 4;
  constexpr int dim = 16 * WAVES;
  const int vdim = a.vdim, columns = chunk_columns(vdim);
  const int column = tile * 16 + n;
  const bool live = column < vdim;
  const int chunks = (hi - lo + CHUNK - 1) / CHUNK;
  const size_t stride = (size_t)a.head_count * chunk_record(dim, vdim);  // between a sequence's records of this head
  const size_t out_row = (size_t)a.heads * vdim;
  const float* next = a.scratch + ((size_t)first_chunk(lo, b) * a.head_count + blockIdx.x) * chunk_record(dim, vdim);
  const int record_bytes = 4 * (int)chunk_record(dim, vdim);
  // a lane's places in a record, in bytes (the record's own address is the same for the whole wave and moves from chunk to chunk)
  const uint32_t rows_at = 4 * (wave * 256 + n * 16 + 4 * g);
  auto record_of = [&](const float* at) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(at), 0, record_bytes, 0x00020000); };
  auto piece = [&](const __amdgpu_buffer_rsrc_t& record, uint32_t at, int from) { return __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(record, at, 4 * from, 0)); };
  auto meet = [&] {  // (what every wave has written to LDS is there; both loops come here as often)
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
  };
  // Loads are asked for whether or not there is a chunk that far ahead (then the last one's again), in this order on every path: a wait
  // counts the loads that are younger.  A loop per set of waves, so that none sits behind a branch.
  auto walk = [&](auto& ops, auto load, auto work) {
#pragma unroll
    for (int j = 0; j < SCAN_AHEAD; ++j) {
      load(ops[j]);
      if (j + 1 < chunks) next += stride;
      __builtin_amdgcn_sched_barrier(0);
    }
    int c = 0;
    for (; c + SCAN_AHEAD <= chunks; c += SCAN_AHEAD) {
#pragma unroll
      for (int j = 0; j < SCAN_AHEAD; ++j) {
        work(j & 1, ops[j]);
        __builtin_amdgcn_sched_barrier(0);
        load(ops[j]);
        if (c + j + SCAN_AHEAD + 1 < chunks) next += stride;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int j = 0; j < SCAN_AHEAD - 1; ++j)
      if (c + j < chunks) work(j & 1, ops[j]);  // (the same for the whole workgroup)
    meet();
  };

  if (any_wave < WAVES) {
    const uint32_t decays_at = 4 * (48 * dim + wave * 16 + 4 * g), column_at = 4 * (49 * dim + column * CHUNK + 4 * g);
    float* S = a.state + (((size_t)a.slots[b] * a.heads + h) * dim + wave * 16 + 4 * g) * vdim + (live ? column : vdim - 1);
    float4_t z;
#pragma unroll
    for (int i = 0; i < 4; ++i) z[i] = S[(size_t)i * vdim];
    ChunkOperands ops[SCAN_AHEAD];
    walk(ops, [&](ChunkOperands& o) {
      const auto record = record_of(next);
      if (DELTA) o.up = piece(record, rows_at, 0);
      o.k = piece(record, rows_at, 32 * dim);
      o.p = piece(record, decays_at, 0);
      o.dv = piece(record, column_at, 0);
    }, [&](int buffer, const ChunkOperands& o) {
      states[buffer][wave][lane] = z;
      float4_t d = o.dv;
      if constexpr (DELTA) {
        d = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) d = mfma4(o.up[e], z[e], d);
        removed[buffer][wave][lane] = d;
      }
      z *= o.p;
      if constexpr (DELTA) {
        meet();
        d = o.dv;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) d += removed[buffer][w][lane];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) z = mfma4(o.k[e], d[e], z);
      if constexpr (!DELTA) meet();
    });
    if (live) {
#pragma unroll
      for (int i = 0; i < 4; ++i) S[(size_t)i * vdim] = z[i];
    }
  } else {
    // the read-out that a lane finishes, by its place in the order in which the parts lie in LDS
    const int out_t = ((tid >> 6) & 3) * 4 + (tid & 3), out_e = (tid >> 2) & 15;
    const uint32_t read_at = 4 * (49 * dim + (columns + tile * 16 + out_e) * CHUNK + out_t);
    const uint32_t out_at = tid < 256 && tile * 16 + out_e < vdim ? 4u * (out_t * (uint32_t)out_row + out_e) : 0x80000000u;  // (behind any row: not stored)
    float* out = a.out + (size_t)lo * out_row + (size_t)h * vdim + tile * 16;
    const int row_bytes = 4 * (int)out_row;
    int pending = 0, left = hi - lo;  // tokens whose parts of O lie in LDS, tokens behind them
    auto read_of = [&](const float* at) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(record_of(at), read_at, 0, 0)); };
    const float last_read = read_of(next + (size_t)(chunks - 1) * stride);
    const float* before = next;
    auto read_out = [&](int buffer, float v) {
      const auto rows = __builtin_amdgcn_make_buffer_rsrc(out, 0, pending * row_bytes, 0x00020000);  // (what lies behind the last token is not stored)
      const float* sums = reinterpret_cast<const float*>(reads[buffer]);
#pragma unroll
      for (int w = 0; w < WAVES; ++w) v += sums[w * 256 + (tid & 255)];
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), rows, out_at, 0, 0);
      out += pending * out_row;
      pending = left < CHUNK ? left : CHUNK;
      left -= pending;
    };
    ChunkReads ops[SCAN_AHEAD];
    walk(ops, [&](ChunkReads& o) {
      o.rp = piece(record_of(next), rows_at, 16 * dim);
      o.before = read_of(before);
      before = next;
    }, [&](int buffer, const ChunkReads& o) {
      meet();
      const float4_t z = states[buffer][wave][lane];
      float4_t read = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; ++e) read = mfma4(o.rp[e], z[e], read);
      if (WAVES == 4 || wave < 4) read_out(1 - buffer, o.before);  // (uniform over the wave)
      reads[buffer][wave][lane] = read;
    });
    if (WAVES == 4 || wave < 4) read_out((chunks - 1) & 1, last_read);
  }
}

static int records_of_step(int tokens, int num_seqs) { return tokens / CHUNK + num_seqs + 1; }

// float32 elements of scratch that a head takes in a step; 0: these sizes are not for these kernels.  Key heads of 64 and 128 channels:
// the sizes whose long portions ran a column of the state per wave, in an order of sums of their own.  (Other sizes are worked in one
// order whether a portion is long or short, and larger ones would need more than a workgroup's waves for a column tile.)
extern "C" long long velox_linear_chunk_scratch_elems(int tokens, int num_seqs, int dim, int vdim) {
  if ((dim != 64 && dim != 128) || vdim < 1) return 0;
  return (long long)records_of_step(tokens, num_seqs) * (long long)chunk_record(dim, vdim);
}

template <bool DELTA>
static void linear_chunk_launch(LinearChunkArgs a, int tokens, int long_seqs, int long_span, hipStream_t stream) {
  const size_t lds = (size_t)CHUNK * (3 * (a.dim + 4) + 4 * CHUNK_STRIDE) * sizeof(float);
  linear_chunk_prepare_kernel<DELTA><<<(unsigned)records_of_step(tokens, a.num_seqs) * (unsigned)a.head_count, 256, lds, stream>>>(a);
  const int tiles = chunk_columns(a.vdim) / 16;
  a.ordered = orders_sequences((long long)a.head_count * tiles * long_seqs, a.num_seqs);
  const dim3 grid(a.head_count, tiles, a.ordered ? long_seqs : long_span);
  const size_t alone = (long long)grid.x * grid.y * grid.z <= ALONE_WORKGROUPS ? ALONE_LDS : 0;
  if (a.dim == 64) linear_chunk_scan_kernel<4, DELTA><<<grid, 512, alone, stream>>>(a);
  else linear_chunk_scan_kernel<8, DELTA><<<grid, 1024, alone, stream>>>(a);
}

extern "C" int velox_linear_scan(const float* qk, const void* v, int v_dtype, int v_ld, int v_at, const float* decay, int decay_per_channel, const float* beta,
                                 float* state, const int* slots, const int* cu_q, float* out, int num_seqs, int max_q_len, int heads, int kv_heads, int dim,
                                 int vdim, int rule, int from_tokens, int below_tokens, hipStream_t stream);

// The sequences of at least `long_from` tokens, then the shorter ones token by token: `shorter` says which kernels they may need (0: there
// are none, 1: single tokens and pairs, 2: longer ones too).  Launched from here, since a call costs the host more than a launch.
// There are at most `long_seqs` of the former, all among the last `long_span` sequences: a scan's workgroup of another sequence finds nothing to do,
// but 60 single tokens beside a portion of 1,024 have 15,360 of them with 32 heads of 128 x 128 (319 us with them, 224 without).
// beta: nullptr for the additive rule.  `scratch` holds the records of `heads_at_once`
// heads (velox_linear_chunk_scratch_elems each), which are worked one such group after the other.  qk and a decay per channel are
// read in 16-byte pieces (dim is a multiple of 16; the caller checks that the bases are aligned).
extern "C" int velox_linear_chunk_scan(const float* qk, const void* v, int v_dtype, int v_ld, int v_at, const float* decay, int decay_per_channel,
                                       const float* beta, float* scratch, float* state, const int* slots, const int* cu_q, float* out, int num_seqs,
                                       int tokens, int long_from, int long_seqs, int long_span, int shorter, int heads_at_once, int heads, int kv_heads, int dim, int vdim, hipStream_t stream) {
  if (num_seqs <= 0 || tokens <= 0) return 0;
  if (velox_linear_chunk_scratch_elems(tokens, num_seqs, dim, vdim) == 0 || heads < 1 || heads > 65535 || num_seqs > 65535 || heads_at_once < 1 ||
      (long long)records_of_step(tokens, num_seqs) * (heads_at_once < heads ? heads_at_once : heads) > (1 << 23) || vdim > 65535 * 16 || kv_heads < 1 || long_seqs < 1 || long_seqs > long_span || long_span > num_seqs ||
      heads % kv_heads != 0 || !scratch)
    return (int)hipErrorInvalidValue;
  for (int first = 0; first < heads; first += heads_at_once) {
    LinearChunkArgs a{qk, v, v_dtype == VELOX_BF16, v_ld, v_at, decay, decay_per_channel, beta, scratch, state, slots, cu_q, out, heads, kv_heads, dim, vdim,
                      num_seqs, long_from, first, heads - first < heads_at_once ? heads - first : heads_at_once, false};
    if (beta) linear_chunk_launch<true>(a, tokens, long_seqs, long_span, stream);
    else linear_chunk_launch<false>(a, tokens, long_seqs, long_span, stream);
  }
  const int status = (int)hipGetLastError();
  if (status != 0 || shorter == 0) return status;
  auto token_by_token = [&](int longest, int from, int below) {
    return velox_linear_scan(qk, v, v_dtype, v_ld, v_at, decay, decay_per_channel, beta, state, slots, cu_q, out, num_seqs, longest, heads, kv_heads, dim, vdim, beta ? 1 : 0, from,
                             below, stream);
  };
  // (1: what is neither long nor a single token or a pair can only be there beside empty sequences, and this kernel takes it too)
  const int singles = token_by_token(1, 1, shorter == 1 ? long_from : 3);
  return singles != 0 || shorter == 1 ? singles : token_by_token(3, 3, long_from);
}
