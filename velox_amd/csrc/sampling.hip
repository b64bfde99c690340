// Sampling kernels for gfx950: row argmax, the per-row sampler (temperature, top-k, top-p, exponential
// race with a counter-based generator) and the repetition / presence / frequency penalties.
// One workgroup per row; every reduction runs in a fixed order, so a row's result depends on that
// row alone.
#include "common.h"
#include "no_alloc.h"

#include <mutex>

#define SAMPLE_THREADS 1024

struct Best { float value; int index; };

__device__ __forceinline__ Best better(Best a, Best b) {
  // larger value wins; equal values: the smaller index
  if (b.value > a.value || (b.value == a.value && b.index < a.index)) return b;
  return a;
}

__device__ __forceinline__ Best block_best(Best v, Best* scratch) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int waves = (blockDim.x + 63) / 64;
#pragma unroll
  for (int offset = 32; offset > 0; offset >>= 1) {
    Best other;
    other.value = __shfl_xor(v.value, offset, VELOX_WAVE);
    other.index = __shfl_xor(v.index, offset, VELOX_WAVE);
    v = better(v, other);
  }
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  Best total = scratch[0];
  for (int w = 1; w < waves; ++w) total = better(total, scratch[w]);
  return total;
}

__device__ __forceinline__ float block_max(float v, float* scratch) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int waves = (blockDim.x + 63) / 64;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = scratch[0];
  for (int w = 1; w < waves; ++w) total = fmaxf(total, scratch[w]);
  return total;
}

// the best of row[lo .. hi), indices counted from the start of the row
__device__ __forceinline__ Best best_of_range(const float* __restrict__ row, int lo, int hi, Best* scratch) {
  Best best{-INFINITY, 0x7fffffff};
  // 16-byte loads over the aligned middle of the range, single elements at its ends
  const float* start = row + lo;
  const int count = hi - lo;
  const int head = (int)((16 - ((uintptr_t)start & 15)) & 15) / 4;
  const int first = head < count ? head : count;
  const int quads = (count - first) / 4;
  for (int i = threadIdx.x; i < first; i += blockDim.x) best = better(best, Best{start[i], lo + i});
  const float4_t* body = reinterpret_cast<const float4_t*>(start + first);
  for (int q = threadIdx.x; q < quads; q += blockDim.x) {
    const float4_t v = body[q];
#pragma unroll
    for (int j = 0; j < 4; ++j) best = better(best, Best{v[j], lo + first + 4 * q + j});
  }
  for (int i = first + 4 * quads + threadIdx.x; i < count; i += blockDim.x) best = better(best, Best{start[i], lo + i});
  return block_best(best, scratch);
}

// One workgroup per (row, chunk of the vocabulary).  With one chunk the index goes straight to `out`; with several, each
// chunk's best goes to `partial[row][chunk]` and argmax_merge_kernel picks among them (few rows alone would leave most
// of the GPU idle while 600 KB per row are read).
__global__ void __launch_bounds__(SAMPLE_THREADS) argmax_kernel(const float* __restrict__ logits, int* __restrict__ out,
                                                               Best* __restrict__ partial, int vocab, int chunk) {
  __shared__ Best scratch[16];
  const float* row = logits + (size_t)blockIdx.x * vocab;
  const int lo = blockIdx.y * chunk;
  const int hi = lo + chunk < vocab ? lo + chunk : vocab;
  const Best best = best_of_range(row, lo, hi, scratch);
  if (threadIdx.x != 0) return;
  if (gridDim.y == 1) out[blockIdx.x] = best.index;
  else partial[blockIdx.x * gridDim.y + blockIdx.y] = best;
}

__global__ void __launch_bounds__(64) argmax_merge_kernel(const Best* __restrict__ partial, int* __restrict__ out, int chunks) {
  Best best{-INFINITY, 0x7fffffff};
  for (int c = threadIdx.x; c < chunks; c += 64) best = better(best, partial[blockIdx.x * chunks + c]);
#pragma unroll
  for (int offset = 32; offset > 0; offset >>= 1) {
    Best other;
    other.value = __shfl_xor(best.value, offset, VELOX_WAVE);
    other.index = __shfl_xor(best.index, offset, VELOX_WAVE);
    best = better(best, other);
  }
  if (threadIdx.x == 0) out[blockIdx.x] = best.index;
}

// partial: room for rows * chunks (value, index) pairs of 8 bytes, used when chunks > 1.
extern "C" int velox_argmax(const float* logits, int* out, void* partial, int rows, int vocab, int chunks, hipStream_t stream) {
  if (rows <= 0) return 0;
  if (chunks < 1 || (chunks > 1 && partial == nullptr)) return -1;
  const int chunk = (vocab + chunks - 1) / chunks;
  argmax_kernel<<<dim3(rows, chunks), SAMPLE_THREADS, 0, stream>>>(logits, out, (Best*)partial, vocab, chunk);
  if (chunks > 1) argmax_merge_kernel<<<rows, 64, 0, stream>>>((const Best*)partial, out, chunks);
  VELOX_RETURN_LAUNCH_STATUS();
}

// ---- the entry point that allocates nothing (declared in no_alloc.h) ----------------------------------------------
// The chunks' best pairs of velox_argmax_static.  In host code this name is only a stand-in for the symbol: each GPU
// holds its own copy at its own address, which hipGetSymbolAddress gives with that GPU current; host code passes
// that address on, never the name.
static __device__ __align__(256) unsigned char argmax_static_scratch[VELOX_ARGMAX_STATIC_BYTES];

#define VELOX_MAX_DEVICES 64
static void* argmax_scratch_of_device[VELOX_MAX_DEVICES];  // the address of each GPU's copy, looked up once
static std::mutex argmax_scratch_lock;

static int argmax_scratch_of_current_device(void** address) {
  int device = -1;
  hipError_t status = hipGetDevice(&device);
  if (status != hipSuccess) return (int)status;
  if (device < 0 || device >= VELOX_MAX_DEVICES) return VELOX_NO_ALLOC_NO_SCRATCH;
  std::lock_guard<std::mutex> guard(argmax_scratch_lock);
  if (argmax_scratch_of_device[device] == nullptr) {
    void* found = nullptr;
    status = hipGetSymbolAddress(&found, HIP_SYMBOL(argmax_static_scratch));
    if (status != hipSuccess) return (int)status;
    if (found == nullptr) return VELOX_NO_ALLOC_NO_SCRATCH;
    argmax_scratch_of_device[device] = found;
  }
  *address = argmax_scratch_of_device[device];
  return 0;
}

extern "C" int velox_argmax_static_init(void) {
  void* address = nullptr;
  return argmax_scratch_of_current_device(&address);
}

extern "C" int velox_argmax_static(const float* logits, int* out, int rows, int vocab, int chunks, hipStream_t stream) {
  if (rows < 0 || vocab < 1 || chunks < 1 || chunks > vocab || logits == nullptr || out == nullptr) return VELOX_NO_ALLOC_BAD_ARGUMENT;
  if (rows == 0) return 0;
  if (rows > 65535 || chunks > 65535 || (long long)rows * chunks > VELOX_ARGMAX_STATIC_MAX_PAIRS) return VELOX_NO_ALLOC_TOO_LARGE;
  void* scratch = nullptr;
  const int found = argmax_scratch_of_current_device(&scratch);
  if (found != 0) return found;
  const int chunk = (vocab + chunks - 1) / chunks;
  // every pair that the merge reads is written by this launch first: what an earlier call left is never read
  argmax_kernel<<<dim3(rows, chunks), SAMPLE_THREADS, 0, stream>>>(logits, out, (Best*)scratch, vocab, chunk);
  if (chunks > 1) argmax_merge_kernel<<<rows, 64, 0, stream>>>((const Best*)scratch, out, chunks);
  VELOX_RETURN_LAUNCH_STATUS();
}

extern "C" const char* velox_no_alloc_error_text(int code) {
  switch (code) {
    case 0: return "success";
    case VELOX_NO_ALLOC_BAD_ARGUMENT: return "bad argument: rows >= 0, vocab >= 1, 1 <= chunks <= vocab and non-null pointers are required";
    case VELOX_NO_ALLOC_TOO_LARGE: return "rows * chunks exceeds VELOX_ARGMAX_STATIC_MAX_PAIRS (65536), the size of the static scratch array";
    case VELOX_NO_ALLOC_NO_SCRATCH: return "the static scratch array of this GPU could not be found";
    default: return hipGetErrorString((hipError_t)code);
  }
}

// Philox 4x32 with 10 rounds.
__device__ __forceinline__ void philox4x32(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0, uint32_t k1, uint32_t (&out)[4]) {
#pragma unroll
  for (int round = 0; round < 10; ++round) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
    const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0;
    const uint32_t n1 = (uint32_t)p1;
    const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
    const uint32_t n3 = (uint32_t)p0;
    c0 = n0; c1 = n1; c2 = n2; c3 = n3;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}

// order-preserving map from float to unsigned
__device__ __forceinline__ uint32_t sort_key(float v) {
  const uint32_t bits = __float_as_uint(v);
  return (bits & 0x80000000u) ? ~bits : (bits | 0x80000000u);
}

// ---- the threshold of top-k / top-p: a radix search over the ordered keys ------------------------------------------
// A token is kept iff fewer than top_k tokens have a larger x and the tokens with a larger x hold less than top_p of the
// probability.  Both conditions only get harder to meet as x falls, so the kept tokens are those whose key is at least
// some threshold.  The threshold is found digit by digit (11, 11 and 10 bits of the 32-bit key): one pass over the row
// fills, for the tokens that match the digits found so far, a table per value of the next digit (how many tokens, how
// much probability); a scan down the table from the largest digit finds the last digit whose largest member is still
// kept.  Probabilities are summed as 40-bit fixed-point integers, so a sum does not depend on the order in which the
// threads add and a row's threshold is the same in every run and every batch.
#define SELECT_BINS 2048
__device__ __forceinline__ unsigned long long fixed_point_mass(float p) { return (unsigned long long)(p * 1099511627776.f); }  // p in [0, 1], 2^40

struct Above { unsigned int count; unsigned long long mass; };

// Visits the elements of quads [q_lo, q_hi) of a row (quad q = elements 4q .. 4q + 3, those below vocab): f(index, value).
// Whole quads come as 16-byte loads when the row starts at a 16-byte boundary, four loads in flight per thread (with one
// load at a time a pass would take as many trips to the caches as a thread has quads).
template <typename F> __device__ __forceinline__ void for_each_in_quads(const float* __restrict__ row, int vocab, int q_lo, int q_hi, F f) {
  const bool aligned = (reinterpret_cast<uintptr_t>(row) & 15) == 0;
  int whole = aligned ? vocab / 4 : q_lo;  // quads below `whole` are complete and can be loaded as one
  whole = whole < q_hi ? whole : q_hi;
  whole = whole > q_lo ? whole : q_lo;
  const float4_t* body = reinterpret_cast<const float4_t*>(row);
  const int stride = blockDim.x;
  int q = q_lo + threadIdx.x;
  for (; q + 3 * stride < whole; q += 4 * stride) {
    const float4_t v0 = body[q], v1 = body[q + stride], v2 = body[q + 2 * stride], v3 = body[q + 3 * stride];
#pragma unroll
    for (int e = 0; e < 4; ++e) f(4 * q + e, v0[e]);
#pragma unroll
    for (int e = 0; e < 4; ++e) f(4 * (q + stride) + e, v1[e]);
#pragma unroll
    for (int e = 0; e < 4; ++e) f(4 * (q + 2 * stride) + e, v2[e]);
#pragma unroll
    for (int e = 0; e < 4; ++e) f(4 * (q + 3 * stride) + e, v3[e]);
  }
  for (; q < whole; q += stride) {
    const float4_t v = body[q];
#pragma unroll
    for (int e = 0; e < 4; ++e) f(4 * q + e, v[e]);
  }
  const int end = 4 * q_hi < vocab ? 4 * q_hi : vocab;
  for (int i = 4 * whole + threadIdx.x; i < end; i += stride) f(i, row[i]);
}

// One digit of the search.  Every thread brings its share of the digit's table, the largest digits in thread 0: digits
// hi, hi - 1, .. with hi = bins - 1 - per_thread * threadIdx.x (`c`: tokens, `m`: probability); `above` is what lies above
// every token that matches the digits found so far.  A scan over the workgroup finds what lies above each digit; every
// thread gets the digit found, and `above` grows by what lies above that digit's tokens.  `top_p` below 1 with
// `first`: the table holds all tokens, so its sum is the row's whole probability and gives the limit for this level and
// (left in `mass_limit`) the next ones.
// One wave that walked the table out of LDS, 32 entries a lane, had all 64 lanes on one bank at every step: about 6 us a
// digit, against 1 us for the scan (MI355X, three digits a row).
struct SelectScratch {
  unsigned long long wave_mass[SAMPLE_THREADS / 64];
  unsigned int wave_count[SAMPLE_THREADS / 64];
  int digit;
  Above above;
};

__device__ __forceinline__ int select_digit(const unsigned int (&c)[2], const unsigned long long (&m)[2], int per_thread, int bins, int top_k, bool use_mass,
                                            bool first, float top_p, unsigned long long& mass_limit, Above& above, SelectScratch& scratch) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned int c_before = c[0] + (per_thread > 1 ? c[1] : 0u);
  unsigned long long m_before = m[0] + (per_thread > 1 ? m[1] : 0ull);
  const unsigned int c_own = c_before;
  const unsigned long long m_own = m_before;
#pragma unroll
  for (int offset = 1; offset < 64; offset <<= 1) {
    const unsigned int oc = __shfl_up(c_before, offset, VELOX_WAVE);
    const unsigned long long om = __shfl_up(m_before, offset, VELOX_WAVE);
    if (lane >= offset) { c_before += oc; m_before += om; }
  }
  if (lane == 63) { scratch.wave_count[wave] = c_before; scratch.wave_mass[wave] = m_before; }
  if (threadIdx.x == 0) scratch.digit = 0x7fffffff;
  __syncthreads();
  c_before += above.count - c_own;
  m_before += above.mass - m_own;
  unsigned long long total = 0ull;
#pragma unroll
  for (int w = 0; w < SAMPLE_THREADS / 64; ++w) {
    const unsigned long long wave_mass = scratch.wave_mass[w];
    total += wave_mass;
    if (w < wave) { c_before += scratch.wave_count[w]; m_before += wave_mass; }
  }
  // (at least 1: the largest token is kept however small top_p is)
  if (first) mass_limit = max(1ull, (unsigned long long)((double)top_p * (double)total));
  // the smallest digit of this thread whose members' top is still kept
  const int hi = bins - 1 - (int)threadIdx.x * per_thread;
  int lowest = 0x7fffffff;
  Above lowest_above{0u, 0ull};
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (j < per_thread) {
      const bool kept = (top_k <= 0 || c_before < (unsigned int)top_k) && (!use_mass || m_before < mass_limit);
      if (kept) { lowest = hi - j; lowest_above = Above{c_before, m_before}; }
      c_before += c[j];
      m_before += m[j];
    }
  }
  // over the workgroup: kept digits form a run from the top, so the smallest one overall is the answer
  int best = lowest;
#pragma unroll
  for (int offset = 32; offset > 0; offset >>= 1) {
    const int other = __shfl_xor(best, offset, VELOX_WAVE);
    best = other < best ? other : best;
  }
  if (lane == 0 && best != 0x7fffffff) atomicMin(&scratch.digit, best);
  __syncthreads();
  int digit = scratch.digit;
  if (digit == 0x7fffffff) digit = bins - 1;  // (cannot happen: the largest digit's top is always kept)
  else if (lowest == digit) scratch.above = lowest_above;
  if (scratch.digit == 0x7fffffff && threadIdx.x == 0) scratch.above = above;
  __syncthreads();
  above = scratch.above;
  return digit;
}

// options per row, int32[6]: temperature (float bits), top_p (float bits), top_k, seed low 31 bits, seed high 31 bits, counter
//   temperature == 0: argmax.
//   otherwise x = logit / max(T, 1e-5); p = softmax(x); token i is kept iff fewer than top_k tokens have a larger x
//   (top_k > 0) and the tokens with a larger x hold less than top_p of the probability; among the kept tokens the
//   draw is argmax(x - max - log(e)), e = max(-log(u), 1e-10), u uniform from Philox(key = seed, counter = (i / 4, counter)).
// Passes over the row (from the caches: a row is a few hundred kilobytes): the maximum; with a filter, the sum and three
// digits of the threshold; the draw.  Either one workgroup walks the whole row (sample_kernel), or, when the rows are
// too few to fill the GPU that way, the row is cut into chunks of quads with a workgroup each (the sample_chunk_* kernels
// and sample_finish_kernel): the same functions over a range of quads, the tables added up in global memory
// as integers, so both ways give the same token.
struct RowOptions {
  float temperature, top_p, inv_t;
  int top_k;
  uint32_t seed_lo, seed_hi, counter;
  bool use_mass, filter;
};

__device__ __forceinline__ RowOptions read_options(const int* __restrict__ opt, int vocab) {
  RowOptions o;
  o.temperature = __int_as_float(opt[0]);
  o.top_p = __int_as_float(opt[1]);
  o.top_k = opt[2];
  o.seed_lo = (uint32_t)opt[3];
  o.seed_hi = (uint32_t)opt[4];
  o.counter = (uint32_t)opt[5];
  o.inv_t = 1.f / fmaxf(o.temperature, 1e-5f);
  o.use_mass = o.top_p < 1.f;
  o.filter = (o.top_k > 0 && o.top_k < vocab) || o.use_mass;
  return o;
}

// digits of the threshold: bits 31..21, 20..10, 9..0
__device__ __forceinline__ int level_shift(int level) { return level == 0 ? 21 : level == 1 ? 10 : 0; }
__device__ __forceinline__ int level_bins(int level) { return level == 2 ? 1024 : 2048; }

// A level's table in LDS: what it needs of counts (top-k) and probabilities (top-p) is kept, the other is neither cleared
// nor added to.  The first digit is sign, exponent and two bits of the mantissa: the tokens of a row share a few dozen
// values, and lanes of a wave that add to one entry wait for each other.  Its entries are therefore kept in
// TABLE_COPIES copies next to each other (other banks), a lane's number picks the copy.
#define TABLE_COPIES 4
template <int COPIES> struct LevelTables {
  unsigned long long masses[SELECT_BINS * COPIES];
  unsigned int counts[SELECT_BINS * COPIES];
};
__device__ __forceinline__ int level_copies(int level) { return level == 0 ? TABLE_COPIES : 1; }

template <int C> __device__ __forceinline__ void clear_tables(LevelTables<C>& t, int level, const RowOptions& o) {
  const int entries = level_bins(level) * level_copies(level);
  for (int b = threadIdx.x; b < entries; b += blockDim.x) {
    if (o.top_k > 0) t.counts[b] = 0u;
    if (o.use_mass) t.masses[b] = 0ull;
  }
}

template <int C> __device__ __forceinline__ void add_token(LevelTables<C>& t, int entry, float x, const RowOptions& o, float mx) {
  if (o.top_k > 0) atomicAdd(&t.counts[entry], 1u);
  if (o.use_mass) {
    const unsigned long long mass = fixed_point_mass(expf(x - mx));
    if (mass != 0ull) atomicAdd(&t.masses[entry], mass);
  }
}

// Adds the tokens of quads [q_lo, q_hi) that match the digits found so far (`prefix`) to the tables of digit `level`
// (cleared by the caller, barrier behind the clearing).
template <int C>
__device__ __forceinline__ void add_to_tables(const float* __restrict__ row, int vocab, int q_lo, int q_hi, const RowOptions& o, float mx,
                                              int level, uint32_t prefix, LevelTables<C>& t) {
  const int shift = level_shift(level);
  const int bins = level_bins(level);
  const int copies = level_copies(level);
  const int copy = threadIdx.x & (copies - 1);
  const uint32_t known = level == 0 ? 0u : ~((1u << (shift + (level == 2 ? 10 : 11))) - 1u);  // mask of the digits found so far
  const float inv_t = o.inv_t;
  for_each_in_quads(row, vocab, q_lo, q_hi, [&](int, float v) {
    const float x = v * inv_t;
    const uint32_t key = sort_key(x);
    if ((key & known) == prefix) add_token(t, (int)((key >> shift) & (uint32_t)(bins - 1)) * copies + copy, x, o, mx);
  });
}

// the sums of digit `bin` over the copies
template <int C> __device__ __forceinline__ void table_entry(const LevelTables<C>& t, int level, int bin, const RowOptions& o, unsigned int& c, unsigned long long& m) {
  const int copies = level_copies(level);
  c = 0u;
  m = 0ull;
  for (int e = bin * copies; e < (bin + 1) * copies; ++e) {
    if (o.top_k > 0) c += t.counts[e];
    if (o.use_mass) m += t.masses[e];
  }
}

// quad q of a row; elements beyond the vocabulary: -inf
__device__ __forceinline__ float4_t load_quad(const float* __restrict__ row, int vocab, int q, bool aligned) {
  float4_t v;
  if (aligned && 4 * q + 3 < vocab) {
    v = *reinterpret_cast<const float4_t*>(row + 4 * q);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = 4 * q + e < vocab ? row[4 * q + e] : -INFINITY;
  }
  return v;
}

// A wave's kept quads, waiting until there are as many as lanes.
#define DRAW_QUEUE 128
struct DrawQueue {
  float4_t values[SAMPLE_THREADS / 64][DRAW_QUEUE];
  int quads[SAMPLE_THREADS / 64][DRAW_QUEUE];
};

// what a token's word of the noise makes of it
__device__ __forceinline__ float token_score(float x, uint32_t bits, float mx) {
  const float u = ((float)(bits >> 8) + 0.5f) * (1.0f / 16777216.0f);
  const float noise = fmaxf(-logf(u), 1e-10f);
  const float raw = (x - mx) - logf(noise);
  // A score that is no number (of a NaN among the logits, or where the row's largest is infinite) counts as -inf: it would otherwise
  // win or lose by the order in which threads meet it, and could leave a row without any token.
  return raw > -INFINITY ? raw : -INFINITY;
}

// token i with its word of the noise
__device__ __forceinline__ void draw_token(int i, float x, uint32_t bits, float mx, Best& best) {
  const float score = token_score(x, bits, mx);
  // (a thread's tokens come in no order: equal scores go to the smaller index here too)
  if (score > best.value || best.index == 0x7fffffff || (score == best.value && i < best.index)) best = Best{score, i};
}

// The draw among the kept tokens of quads [q_lo, q_hi): this thread's best (score, index).
// Behind a filter a token or two of 256 are kept, yet nearly every wave of quads has one: the noise (ten rounds of Philox
// and eight logarithms a quad) would be worked out by whole waves for a lane or two.  The kept quads are therefore queued
// in LDS first and taken up 64 at a time (48 rows of 152,064, top-p 0.9: the pass with the digit before it 19.7 us
// without the queue, 13.4 with it).
// open(i, x, bits): whether a token at or above the threshold is taken care of elsewhere.
template <typename F>
__device__ __forceinline__ Best draw_in_quads(const float* __restrict__ row, int vocab, int q_lo, int q_hi, const RowOptions& o, float mx, uint32_t threshold,
                                              DrawQueue& queue, F open) {
  Best best{-INFINITY, 0x7fffffff};
  const bool aligned = (reinterpret_cast<uintptr_t>(row) & 15) == 0;
  const bool filter = o.filter;
  const float inv_t = o.inv_t;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  auto draw_quad = [&](int q, const float4_t& v) {
    uint32_t bits[4];
    philox4x32((uint32_t)q, o.counter, 0u, 0u, o.seed_lo, o.seed_hi, bits);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 4 * q + e;
      if (i >= vocab) break;
      const float x = v[e] * inv_t;
      if (filter && (sort_key(x) < threshold || open(i, x, bits[e]))) continue;
      draw_token(i, x, bits[e], mx, best);
    }
  };
  constexpr int AHEAD = 4;  // quads in flight per thread
  int queued = 0;           // of this wave
  for (int base = q_lo + wave * 64; base < q_hi; base += AHEAD * (int)blockDim.x) {  // (the same for all lanes of a wave)
    float4_t ahead[AHEAD];
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
      const int qa = base + lane + a * (int)blockDim.x;
      ahead[a] = load_quad(row, vocab, qa < q_hi ? qa : q_hi - 1, aligned);
    }
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
      const int q = base + lane + a * (int)blockDim.x;
      const float4_t v = ahead[a];
      if (!filter) {
        if (q < q_hi) draw_quad(q, v);
        continue;
      }
      bool any = false;
#pragma unroll
      for (int e = 0; e < 4; ++e) any = any || (4 * q + e < vocab && sort_key(v[e] * inv_t) >= threshold);
      any = any && q < q_hi;
      const unsigned long long kept = __ballot(any);
      if (any) {
        const int at = queued + __popcll(kept & ((1ull << lane) - 1ull));  // below 63 + 64
        queue.values[wave][at] = v;
        queue.quads[wave][at] = q;
      }
      queued += __popcll(kept);
      if (queued >= 64) {
        queued -= 64;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        draw_quad(queue.quads[wave][queued + lane], queue.values[wave][queued + lane]);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
    }
  }
  if (queued > 0) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane < queued) draw_quad(queue.quads[wave][lane], queue.values[wave][lane]);
  }
  return best;
}

// One workgroup per row.
__global__ void __launch_bounds__(SAMPLE_THREADS) sample_kernel(const float* __restrict__ logits, const int* __restrict__ options,
                                                                int* __restrict__ out, int vocab) {
  __shared__ Best best_scratch[16];
  __shared__ float scratch[16];
  __shared__ union { LevelTables<TABLE_COPIES> tables; DrawQueue queue; } shared;  // (the draw comes when the search is over)
  __shared__ SelectScratch select;
  const float* row = logits + (size_t)blockIdx.x * vocab;
  const RowOptions o = read_options(options + (size_t)blockIdx.x * 6, vocab);
  const int tid = threadIdx.x;
  const int quads = (vocab + 3) / 4;

  if (o.temperature == 0.f) {
    Best best{-INFINITY, 0x7fffffff};
    for_each_in_quads(row, vocab, 0, quads, [&](int i, float v) { best = better(best, Best{v, i}); });
    best = block_best(best, best_scratch);
    if (tid == 0) out[blockIdx.x] = best.index;
    return;
  }
  float mx = -INFINITY;
  for_each_in_quads(row, vocab, 0, quads, [&](int, float v) { mx = fmaxf(mx, v * o.inv_t); });
  mx = block_max(mx, scratch);

  // smallest key whose tokens are kept
  uint32_t threshold = 0u;
  if (o.filter) {
    Above above{0u, 0ull};
    unsigned long long mass_limit = 0ull;
    uint32_t prefix = 0u;  // the digits found so far, in place
#pragma unroll 1
    for (int level = 0; level < 3; ++level) {
      const int bins = level_bins(level), per_thread = bins / SAMPLE_THREADS;
      clear_tables(shared.tables, level, o);
      __syncthreads();
      add_to_tables(row, vocab, 0, quads, o, mx, level, prefix, shared.tables);
      __syncthreads();
      unsigned int c[2] = {0u, 0u};
      unsigned long long m[2] = {0ull, 0ull};
      for (int j = 0; j < per_thread; ++j) table_entry(shared.tables, level, bins - 1 - tid * per_thread - j, o, c[j], m[j]);
      const int digit = select_digit(c, m, per_thread, bins, o.top_k, o.use_mass, level == 0, o.top_p, mass_limit, above, select);
      prefix |= (uint32_t)digit << level_shift(level);
      __syncthreads();  // the tables and the scratch are free again
    }
    threshold = prefix;
  }

  Best best = draw_in_quads(row, vocab, 0, quads, o, mx, threshold, shared.queue, [](int, float, uint32_t) { return false; });
  best = block_best(best, best_scratch);
  if (tid == 0) out[blockIdx.x] = best.index;
}

extern "C" int velox_sample(const float* logits, const int* options, int* out, int rows, int vocab, hipStream_t stream) {
  if (rows <= 0) return 0;
  sample_kernel<<<rows, SAMPLE_THREADS, 0, stream>>>(logits, options, out, vocab);
  VELOX_RETURN_LAUNCH_STATUS();
}

// ---- a row cut into chunks ------------------------------------------------------------------------------------------
// What the chunks of a row share, in global memory: each chunk's maximum and best pair, the tables of the first two digits
// (cleared by the first kernel, added to with integer atomics) and what the search has found so far.  A row with a filter goes
// through four kernels: its maximum; the tables of the first digit; the tokens that this digit does not rule out, as a list per
// chunk (of a row with top-p 0.9 or top-k 50 about one token in a hundred); and from the lists, in one workgroup, the other digits,
// the draw and the token.  What bounds a pass is its few dependent steps (a launch, two trips to memory, a scan over the table), not
// the row: with a kernel per digit, one for the draw and one to merge the chunks, 48 rows of 152,064 took 55 us; see
// sample_finish_kernel.  A chunk with more such tokens than its share of FINISH_TOKENS, which is what one workgroup is quick with, adds
// them to the tables of the second digit instead, and the row's chunks are drawn from by a workgroup each: from its list, or from
// the row where a wave has found more than LIST_ENTRIES.
struct RowSearch {
  unsigned long long mass_limit;  // top_p of the row's whole probability
  unsigned long long above_mass;  // what lies above the first digit's tokens
  unsigned int above_count;
  unsigned int prefix;            // the first digit, in place
  unsigned long long best;        // of a row that is shared out, above the second digit's tokens (in_order of the pair)
  int shared_out;                 // some chunk has more than its share of tokens
  unsigned int drawn;             // chunks of such a row that have drawn
};

#define LIST_ENTRIES 256
#define FINISH_TOKENS 6144
#define NOT_LISTED ((int)0x80000000)
#define OPEN_BINS 1024  // values of the third digit
struct Listed { float logit; int index; };

struct ChunkedScratch {
  Listed* lists;               // [rows, chunks, list_room]
  int* list_lengths;           // [rows, chunks]; ~length: more than the chunk's share; NOT_LISTED
  float* chunk_max;            // [rows, chunks]
  Best* chunk_best;            // [rows, chunks]
  RowSearch* search;           // [rows]
  unsigned int* counts;        // [rows, 2, SELECT_BINS]
  unsigned long long* masses;  // [rows, 2, SELECT_BINS]
  unsigned int* open_counts;       // [rows, OPEN_BINS]: see sample_finish_kernel
  unsigned long long* open_best;   // [rows, OPEN_BINS]
  int list_room, share;        // tokens that a chunk has room for; that it may have for one workgroup to finish its row
};

static size_t chunked_scratch_layout(int rows, int vocab, int chunks, void* base, ChunkedScratch* scratch) {
  auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
  size_t at = 0;
  char* p = (char*)base;
  auto take = [&](size_t bytes) { char* here = p + at; at += up(bytes); return here; };
  ChunkedScratch s;
  s.masses = (unsigned long long*)take((size_t)rows * 2 * SELECT_BINS * sizeof(unsigned long long));
  s.counts = (unsigned int*)take((size_t)rows * 2 * SELECT_BINS * sizeof(unsigned int));
  s.search = (RowSearch*)take((size_t)rows * sizeof(RowSearch));
  s.chunk_best = (Best*)take((size_t)rows * chunks * sizeof(Best));
  s.chunk_max = (float*)take((size_t)rows * chunks * sizeof(float));
  const int chunk_tokens = 4 * (((vocab + 3) / 4 + chunks - 1) / chunks);
  s.list_room = chunk_tokens < LIST_ENTRIES * (SAMPLE_THREADS / 64) ? chunk_tokens : LIST_ENTRIES * (SAMPLE_THREADS / 64);
  s.share = FINISH_TOKENS / chunks;
  s.lists = (Listed*)take((size_t)rows * chunks * s.list_room * sizeof(Listed));
  s.list_lengths = (int*)take((size_t)rows * chunks * sizeof(int));
  s.open_best = (unsigned long long*)take((size_t)rows * OPEN_BINS * sizeof(unsigned long long));
  s.open_counts = (unsigned int*)take((size_t)rows * OPEN_BINS * sizeof(unsigned int));
  if (scratch != nullptr) *scratch = s;
  return at;
}

__device__ __forceinline__ void chunk_quads(int vocab, int chunk, int& q_lo, int& q_hi) {
  const int quads = (vocab + 3) / 4;
  const int per_chunk = (quads + gridDim.y - 1) / gridDim.y;
  q_lo = chunk * per_chunk;
  q_hi = q_lo + per_chunk < quads ? q_lo + per_chunk : quads;
  if (q_lo > quads) q_lo = quads;
}

// pass 1: clears the row's tables, leaves the chunk's maximum (or, for a greedy row, its best pair)
__global__ void __launch_bounds__(SAMPLE_THREADS) sample_chunk_max_kernel(const float* __restrict__ logits, const int* __restrict__ options,
                                                                          ChunkedScratch s, int vocab) {
  __shared__ Best best_scratch[16];
  __shared__ float scratch[16];
  const int r = blockIdx.x, c = blockIdx.y, chunks = gridDim.y;
  const float* row = logits + (size_t)r * vocab;
  const RowOptions o = read_options(options + (size_t)r * 6, vocab);
  int q_lo, q_hi;
  chunk_quads(vocab, c, q_lo, q_hi);
  if (o.temperature == 0.f) {
    Best best{-INFINITY, 0x7fffffff};
    for_each_in_quads(row, vocab, q_lo, q_hi, [&](int i, float v) { best = better(best, Best{v, i}); });
    best = block_best(best, best_scratch);
    if (threadIdx.x == 0) s.chunk_best[r * chunks + c] = best;
    return;
  }
  if (o.filter) {
    if (c == 0 && threadIdx.x == 0) s.search[r].best = 0ull, s.search[r].shared_out = 0, s.search[r].drawn = 0u;
    for (int e = c * blockDim.x + threadIdx.x; e < OPEN_BINS; e += chunks * blockDim.x) {
      s.open_counts[(size_t)r * OPEN_BINS + e] = 0u;
      s.open_best[(size_t)r * OPEN_BINS + e] = 0ull;
    }
    const int entries = 2 * SELECT_BINS;
    for (int e = c * blockDim.x + threadIdx.x; e < entries; e += chunks * blockDim.x) {
      if (o.top_k > 0) s.counts[(size_t)r * entries + e] = 0u;
      if (o.use_mass) s.masses[(size_t)r * entries + e] = 0ull;
    }
  }
  float mx = -INFINITY;
  for_each_in_quads(row, vocab, q_lo, q_hi, [&](int, float v) { mx = fmaxf(mx, v * o.inv_t); });
  mx = block_max(mx, scratch);
  if (threadIdx.x == 0) s.chunk_max[r * chunks + c] = mx;
}

__device__ __forceinline__ float row_max_of_chunks(const float* __restrict__ chunk_max, int chunks) {
  float mx = -INFINITY;
  for (int c = threadIdx.x & 63; c < chunks; c += 64) mx = fmaxf(mx, chunk_max[c]);
  return wave_max(mx);
}

// The digit of `level`, in place behind `prefix`, from table_of(bin, count, mass).
template <typename F>
__device__ __forceinline__ uint32_t digit_of_table(int level, const RowOptions& o, uint32_t prefix, unsigned long long& mass_limit, Above& above, SelectScratch& select,
                                                   F table_of) {
  const int bins = level_bins(level), per_thread = bins / SAMPLE_THREADS;
  unsigned int c[2] = {0u, 0u};
  unsigned long long m[2] = {0ull, 0ull};
  for (int j = 0; j < per_thread; ++j) table_of(bins - 1 - (int)threadIdx.x * per_thread - j, c[j], m[j]);
  return prefix | ((uint32_t)select_digit(c, m, per_thread, bins, o.top_k, o.use_mass, level == 0, o.top_p, mass_limit, above, select) << level_shift(level));
}

// adds a workgroup's tables of `level` (0 or 1) to the row's
template <int C> __device__ __forceinline__ void add_to_row_tables(const ChunkedScratch& s, int r, int level, const LevelTables<C>& tables, const RowOptions& o) {
  const size_t base = ((size_t)r * 2 + level) * SELECT_BINS;
  for (int b = threadIdx.x; b < level_bins(level); b += blockDim.x) {
    unsigned int count;
    unsigned long long mass;
    table_entry(tables, level, b, o, count, mass);
    if (count != 0u) atomicAdd(&s.counts[base + b], count);
    if (mass != 0ull) atomicAdd(&s.masses[base + b], mass);
  }
}

// Lists this wave's tokens of quads [q_lo, q_hi) whose key is at least `floor`: up to LIST_ENTRIES of them in `mine` (LDS).  Returns how
// many there are (some number above LIST_ENTRIES if there are more).
__device__ __forceinline__ int list_tokens(const float* __restrict__ row, int vocab, int q_lo, int q_hi, const RowOptions& o, uint32_t floor, Listed* mine) {
  constexpr int AHEAD = 4;  // quads in flight per thread
  const bool aligned = (reinterpret_cast<uintptr_t>(row) & 15) == 0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int found = 0;
  for (int base = q_lo + wave * 64; base < q_hi && found <= LIST_ENTRIES; base += AHEAD * (int)blockDim.x) {  // (the same for all lanes of a wave)
    float4_t ahead[AHEAD];
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
      const int qa = base + lane + a * (int)blockDim.x;
      ahead[a] = load_quad(row, vocab, qa < q_hi ? qa : q_hi - 1, aligned);
    }
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
      if (found > LIST_ENTRIES) break;
      const int q = base + lane + a * (int)blockDim.x;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool in = q < q_hi && 4 * q + e < vocab && sort_key(ahead[a][e] * o.inv_t) >= floor;
        const unsigned long long all = __ballot(in);
        if (all == 0ull) continue;
        const int at = found + __popcll(all & ((1ull << lane) - 1ull));
        if (in && at < LIST_ENTRIES) mine[at] = Listed{ahead[a][e], 4 * q + e};
        found += __popcll(all);
      }
    }
  }
  return found;
}

// pass 2 of a row with a filter: the tables of the first digit
__global__ void __launch_bounds__(SAMPLE_THREADS) sample_chunk_tables_kernel(const float* __restrict__ logits, const int* __restrict__ options,
                                                                             ChunkedScratch s, int vocab) {
  __shared__ LevelTables<TABLE_COPIES> tables;
  const int r = blockIdx.x, c = blockIdx.y, chunks = gridDim.y;
  const float* row = logits + (size_t)r * vocab;
  const RowOptions o = read_options(options + (size_t)r * 6, vocab);
  if (o.temperature == 0.f || !o.filter) return;
  int q_lo, q_hi;
  chunk_quads(vocab, c, q_lo, q_hi);
  clear_tables(tables, 0, o);
  const float mx = row_max_of_chunks(s.chunk_max + r * chunks, chunks);
  __syncthreads();
  add_to_tables(row, vocab, q_lo, q_hi, o, mx, 0, 0u, tables);
  __syncthreads();
  add_to_row_tables(s, r, 0, tables, o);
}

// a chunk's draw where the row has no filter
__device__ __forceinline__ void draw_among_all(const float* __restrict__ row, int vocab, int q_lo, int q_hi, const RowOptions& o, float mx, DrawQueue& queue,
                                               Best* best_scratch, Best* chunk_best) {
  const Best best = block_best(draw_in_quads(row, vocab, q_lo, q_hi, o, mx, 0u, queue, [](int, float, uint32_t) { return false; }), best_scratch);
  if (threadIdx.x == 0) *chunk_best = best;
}

// pass 3: the first digit, and the chunk's tokens that it does not rule out (a row without a filter: the chunk's draw)
__global__ void __launch_bounds__(SAMPLE_THREADS) sample_chunk_list_kernel(const float* __restrict__ logits, const int* __restrict__ options,
                                                                           ChunkedScratch s, int vocab) {
  constexpr int WAVES = SAMPLE_THREADS / 64;
  __shared__ union { Listed listed[WAVES][LIST_ENTRIES]; DrawQueue queue; } shared;
  __shared__ LevelTables<1> tables;
  __shared__ SelectScratch select;
  __shared__ Best best_scratch[16];
  __shared__ int found_of_wave[WAVES];
  const int r = blockIdx.x, c = blockIdx.y, chunks = gridDim.y;
  const float* row = logits + (size_t)r * vocab;
  const RowOptions o = read_options(options + (size_t)r * 6, vocab);
  if (o.temperature == 0.f) return;  // (its chunks' best pairs are there since the first pass)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int q_lo, q_hi;
  chunk_quads(vocab, c, q_lo, q_hi);
  const float mx = row_max_of_chunks(s.chunk_max + r * chunks, chunks);
  if (!o.filter) {
    draw_among_all(row, vocab, q_lo, q_hi, o, mx, shared.queue, best_scratch, s.chunk_best + r * chunks + c);
    return;
  }
  Above above{0u, 0ull};
  unsigned long long mass_limit = 0ull;
  const size_t base = (size_t)r * 2 * SELECT_BINS;
  const uint32_t prefix = digit_of_table(0, o, 0u, mass_limit, above, select, [&](int bin, unsigned int& count, unsigned long long& mass) {
    if (o.top_k > 0) count = s.counts[base + bin];
    if (o.use_mass) mass = s.masses[base + bin];
  });
  if (c == 0 && tid == 0) {
    s.search[r].mass_limit = mass_limit;
    s.search[r].above_mass = above.mass;
    s.search[r].above_count = above.count;
    s.search[r].prefix = prefix;
  }
  const int found = list_tokens(row, vocab, q_lo, q_hi, o, prefix, shared.listed[wave]);
  if (lane == 0) found_of_wave[wave] = found;
  __syncthreads();
  int before = 0, total = 0;
  bool whole = true;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    const int of_wave = found_of_wave[w];
    before += w < wave ? of_wave : 0;
    total += of_wave;
    whole = whole && of_wave <= LIST_ENTRIES;
  }
  const bool own_share = whole && total <= s.share;
  if (tid == 0) s.list_lengths[r * chunks + c] = own_share ? total : whole ? ~total : NOT_LISTED;
  if (whole) {
    Listed* mine = s.lists + ((size_t)r * chunks + c) * s.list_room + before;
    for (int j = lane; j < found; j += 64) mine[j] = shared.listed[wave][j];
  }
  if (own_share) return;
  if (tid == 0) s.search[r].shared_out = 1;
  clear_tables(tables, 1, o);
  __syncthreads();
  if (whole) {
    for (int j = lane; j < found; j += 64) {
      const float x = shared.listed[wave][j].logit * o.inv_t;
      const uint32_t key = sort_key(x);
      if ((key >> level_shift(0)) == (prefix >> level_shift(0))) add_token(tables, (int)((key >> level_shift(1)) & (uint32_t)(level_bins(1) - 1)), x, o, mx);
    }
  } else {
    add_to_tables(row, vocab, q_lo, q_hi, o, mx, 1, prefix, tables);
  }
  __syncthreads();
  add_to_row_tables(s, r, 1, tables, o);
}

// A (score, index) as one number, in the order of `better`; never 0.
__device__ __forceinline__ unsigned long long in_order(const Best& v) {
  return ((unsigned long long)sort_key(v.value + 0.f) << 32) | (unsigned int)~v.index;  // (a score of -0 is as good as one of 0)
}
__device__ __forceinline__ float value_of_key(uint32_t key) { return __uint_as_float((key & 0x80000000u) ? key ^ 0x80000000u : ~key); }
__device__ __forceinline__ Best of_order(unsigned long long v) {
  return v == 0ull ? Best{-INFINITY, 0x7fffffff} : Best{value_of_key((uint32_t)(v >> 32)), (int)~(unsigned int)v};
}
// What other workgroups of the same kernel have left by atomics: past the caches that only some of the card's compute units share.
template <typename T> __device__ __forceinline__ T load_shared(const T* p) { return __hip_atomic_load(const_cast<T*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename T> __device__ __forceinline__ void add_shared(T* p, T v) { __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename T> __device__ __forceinline__ void max_shared(T* p, T v) { __hip_atomic_fetch_max(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// this wave's stores and atomics have arrived
__device__ __forceinline__ void wait_for_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// a token's word of the noise
__device__ __forceinline__ uint32_t token_bits(int i, const RowOptions& o) {
  uint32_t bits[4];
  philox4x32((uint32_t)(i >> 2), o.counter, 0u, 0u, o.seed_lo, o.seed_hi, bits);
  return (i & 2) ? ((i & 1) ? bits[3] : bits[2]) : ((i & 1) ? bits[1] : bits[0]);
}

// A thread's open tokens of one value of the third digit, added to the workgroup's table when another value turns up: a row of equal logits
// would otherwise queue up at one entry, token by token.
struct OpenRun {
  unsigned long long best;
  unsigned int count, bin;
};
__device__ __forceinline__ void settle(const OpenRun& run, unsigned int* counts, unsigned long long* best) {
  if (run.count == 0u) return;
  atomicAdd(&counts[run.bin], run.count);
  atomicMax(&best[run.bin], run.best);
}

// pass 4 of a row with a filter: the other digits, the draw and the token.  No chunk beyond its share: the workgroup of chunk 0 does it alone.
// Otherwise each chunk's workgroup finds the second digit and draws among its tokens above that digit's.  Which of those that share
// it ("open") are kept the third digit still decides: they are counted, and the best of them kept, per value of that digit, and the
// last of the row's workgroups to come that far finds the digit in these tables and with it the token, without another look at the
// row.  (A table of the 1,024 values and not a list: logits that are equal, or masked to -inf, may all be open.)
// The six kernels before (one for each digit, one for the draw, one to merge the chunks) and these four, us: 48 rows of 152,064 with
// top-p 0.9 46.3 -> 42.1, top-k 50 37.8 -> 32.6; one row 35.0 -> 32.3 and 33.3 -> 26.7; 48 rows of 32,000 34.7 -> 30.4.  Shared out, 8 rows of
// 152,064: standard deviation 0.4 and top-p 0.9 44.9 -> 40.6, 1.5 44.0 -> 40.4, top-k 20,000 36.8 -> 33.5, equal logits 55.7 -> 45.2 (one
// workgroup for all listed tokens took 164 us for the second, a list of the open tokens 325 for the last).
__global__ void __launch_bounds__(SAMPLE_THREADS) sample_finish_kernel(const float* __restrict__ logits, const int* __restrict__ options, int* __restrict__ out,
                                                                       ChunkedScratch s, int vocab) {
  __shared__ union { Listed tokens[FINISH_TOKENS]; DrawQueue queue; } shared;
  __shared__ LevelTables<1> tables;
  __shared__ SelectScratch select;
  __shared__ Best best_scratch[16];
  __shared__ int before[1024 + 1], sum_of_wave[SAMPLE_THREADS / 64], kept_count, last;
  const int r = blockIdx.x, c = blockIdx.y, chunks = gridDim.y;
  const float* row = logits + (size_t)r * vocab;
  const RowOptions o = read_options(options + (size_t)r * 6, vocab);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool filtered = o.temperature != 0.f && o.filter;
  // (asked for together: the kernel's time is that of its trips to memory)
  const RowSearch search = s.search[r];
  const int length = tid < chunks ? s.list_lengths[r * chunks + tid] : 0, listed = s.list_lengths[r * chunks + c];
  const float mx = row_max_of_chunks(s.chunk_max + r * chunks, chunks);
  const bool shared_out = filtered && search.shared_out != 0;
  if (c != 0 && !shared_out) return;
  if (!filtered) {
    Best best{-INFINITY, 0x7fffffff};
    for (int q = tid; q < chunks; q += SAMPLE_THREADS) best = better(best, s.chunk_best[r * chunks + q]);
    best = block_best(best, best_scratch);
    if (tid == 0) out[r] = best.index;
    return;
  }
  Above above{search.above_count, search.above_mass};
  unsigned long long mass_limit = search.mass_limit;
  uint32_t prefix = search.prefix;
  const Listed* lists = s.lists + (size_t)r * chunks * s.list_room;
  auto listed_at = [&](int j) {  // the row's listed token j
    int lo = 0, hi = chunks;     // before[lo] <= j < before[hi]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (before[mid] <= j) lo = mid;
      else hi = mid;
    }
    return lists + (size_t)lo * s.list_room + (j - before[lo]);
  };
  if (tid == 0) kept_count = 0;
  // where each chunk's list begins among the row's
  const int own_tokens = max(length, 0);
  int upto = own_tokens;
#pragma unroll
  for (int offset = 1; offset < 64; offset <<= 1) {
    const int other = __shfl_up(upto, offset, VELOX_WAVE);
    if (lane >= offset) upto += other;
  }
  if (lane == 63) sum_of_wave[wave] = upto;
  __syncthreads();
  int total = 0;  // at most FINISH_TOKENS
  for (int w = 0; w < SAMPLE_THREADS / 64; ++w) {
    const int of_wave = sum_of_wave[w];
    upto += w < wave ? of_wave : 0;
    total += of_wave;
  }
  if (tid < chunks) before[tid] = upto - own_tokens;
  __syncthreads();
  for (int j = tid; j < total; j += SAMPLE_THREADS) shared.tokens[j] = *listed_at(j);  // (each thread reads back what it wrote itself)
#pragma unroll 1
  for (int level = 1; level <= (shared_out ? 1 : 2); ++level) {  // (one loop: code that runs once is fetched while it runs)
    if (total > 0) {
      clear_tables(tables, level, o);
      __syncthreads();
      const int known = level_shift(level - 1), shift = level_shift(level);
      for (int j = tid; j < total; j += SAMPLE_THREADS) {
        const float x = shared.tokens[j].logit * o.inv_t;
        const uint32_t key = sort_key(x);
        if ((key >> known) == (prefix >> known)) add_token(tables, (int)((key >> shift) & (uint32_t)(level_bins(level) - 1)), x, o, mx);
      }
      __syncthreads();
    }
    const size_t base = ((size_t)r * 2 + 1) * SELECT_BINS;
    prefix = digit_of_table(level, o, prefix, mass_limit, above, select, [&](int bin, unsigned int& count, unsigned long long& mass) {
      if (total > 0) table_entry(tables, level, bin, o, count, mass);
      if (shared_out && o.top_k > 0) count += s.counts[base + bin];
      if (shared_out && o.use_mass) mass += s.masses[base + bin];
    });
    __syncthreads();
  }
  if (!shared_out) {
    // The kept tokens are a part of the listed ones, in no order: gathered in the tables' place, so that few waves work out noise.
    constexpr int ROOM = (int)(sizeof(tables) / sizeof(Listed));
    Listed* kept = reinterpret_cast<Listed*>(&tables);
    for (int j = tid; j < total; j += SAMPLE_THREADS) {
      const Listed token = shared.tokens[j];
      const float x = token.logit * o.inv_t;
      if (sort_key(x) >= prefix) {
        const int at = atomicAdd(&kept_count, 1);
        if (at < ROOM) kept[at] = token;
      }
    }
    __syncthreads();
    const bool all = kept_count <= ROOM;
    Best best{-INFINITY, 0x7fffffff};
    for (int j = tid; j < (all ? kept_count : total); j += SAMPLE_THREADS) {
      const Listed token = all ? kept[j] : shared.tokens[j];
      const float x = token.logit * o.inv_t;
      if (sort_key(x) >= prefix) draw_token(token.index, x, token_bits(token.index, o), mx, best);
    }
    best = block_best(best, best_scratch);
    if (tid == 0) out[r] = best.index;
    return;
  }
  unsigned int* open_counts = tables.counts;
  unsigned long long* open_best = tables.masses;
  static_assert(OPEN_BINS == SAMPLE_THREADS && OPEN_BINS <= SELECT_BINS, "an entry each, in the tables' place");
  open_counts[tid] = 0u;
  open_best[tid] = 0ull;
  __syncthreads();
  OpenRun run{0ull, 0u, 0u};
  auto take_open = [&](int i, float x, uint32_t bits) {
    const uint32_t key = sort_key(x);
    if ((key >> 10) != (prefix >> 10)) return false;
    const unsigned int bin = key & (OPEN_BINS - 1);
    const unsigned long long score = in_order(Best{token_score(x, bits, mx), i});
    if (bin != run.bin) {
      settle(run, open_counts, open_best);
      run = OpenRun{0ull, 0u, bin};
    }
    run.best = max(run.best, score);
    ++run.count;
    return true;
  };
  Best best{-INFINITY, 0x7fffffff};
  if (listed != NOT_LISTED) {
    const Listed* own = lists + (size_t)c * s.list_room;
    for (int j = tid; j < (listed >= 0 ? listed : ~listed); j += SAMPLE_THREADS) {
      const Listed token = own[j];
      const float x = token.logit * o.inv_t;
      if (sort_key(x) < prefix) continue;
      const uint32_t bits = token_bits(token.index, o);
      if (!take_open(token.index, x, bits)) draw_token(token.index, x, bits, mx, best);
    }
  } else {
    int q_lo, q_hi;
    chunk_quads(vocab, c, q_lo, q_hi);
    best = draw_in_quads(row, vocab, q_lo, q_hi, o, mx, prefix, shared.queue, take_open);
  }
  settle(run, open_counts, open_best);
  best = block_best(best, best_scratch);  // (and a barrier behind the tables)
  // (fences that write back and drop whole caches, in every wave, took 40 to 70 us here: what the last workgroup reads goes past them)
  const size_t own_bin = (size_t)r * OPEN_BINS + tid;
  const unsigned int own_count = open_counts[tid];
  if (own_count != 0u) {
    add_shared(s.open_counts + own_bin, own_count);
    max_shared(s.open_best + own_bin, open_best[tid]);
  }
  if (tid == 0 && best.index != 0x7fffffff) max_shared(&s.search[r].best, in_order(best));
  wait_for_stores();
  __syncthreads();
  if (tid == 0) last = __hip_atomic_fetch_add(&s.search[r].drawn, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u == (unsigned int)chunks ? 1 : 0;
  __syncthreads();
  if (last == 0) return;
  const size_t bin_of_thread = (size_t)r * OPEN_BINS + (OPEN_BINS - 1 - tid);
  const unsigned int open_count = load_shared(s.open_counts + bin_of_thread);
  const Best of_bin = of_order(load_shared(s.open_best + bin_of_thread));
  best = of_order(tid == 0 ? load_shared(&s.search[r].best) : 0ull);
  const uint32_t own_key = prefix | (uint32_t)(OPEN_BINS - 1 - tid);
  prefix = digit_of_table(2, o, prefix, mass_limit, above, select, [&](int, unsigned int& count, unsigned long long& mass) {
    count = open_count;
    if (o.use_mass && open_count != 0u) mass = open_count * fixed_point_mass(expf(value_of_key(own_key) - mx));  // (the entry's tokens are all alike)
  });
  if (own_key >= prefix) best = better(best, of_bin);
  best = block_best(best, best_scratch);
  if (tid == 0) out[r] = best.index;
}

// Rows of a batch without any filter: the draw behind the maximum, among all of a chunk's tokens.
__global__ void __launch_bounds__(SAMPLE_THREADS) sample_chunk_draw_kernel(const float* __restrict__ logits, const int* __restrict__ options,
                                                                           ChunkedScratch s, int vocab) {
  __shared__ Best best_scratch[16];
  __shared__ DrawQueue queue;
  const int r = blockIdx.x, c = blockIdx.y, chunks = gridDim.y;
  const RowOptions o = read_options(options + (size_t)r * 6, vocab);
  if (o.temperature == 0.f) return;  // (its chunks' best pairs are there since the first pass)
  if (o.filter) {
    // the caller promised that no row has a filter, and this one has: the kernels of the digits did not run.  No token
    // rather than one drawn from the wrong set: the row's result is -1.
    if (threadIdx.x == 0) s.chunk_best[r * chunks + c] = Best{INFINITY, -1};
    return;
  }
  int q_lo, q_hi;
  chunk_quads(vocab, c, q_lo, q_hi);
  const float mx = row_max_of_chunks(s.chunk_max + r * chunks, chunks);
  draw_among_all(logits + (size_t)r * vocab, vocab, q_lo, q_hi, o, mx, queue, best_scratch, s.chunk_best + r * chunks + c);
}

extern "C" long long velox_sample_chunked_scratch_bytes(int rows, int vocab, int chunks) {
  if (rows < 1 || vocab < 1 || chunks < 1) return 0;
  return (long long)chunked_scratch_layout(rows, vocab, chunks, nullptr, nullptr);
}

// The same tokens as velox_sample, every row cut into `chunks` chunks.  scratch: velox_sample_chunked_scratch_bytes(rows,
// vocab, chunks) bytes at a 256-byte boundary, contents arbitrary.  with_filter = 0 promises that no row has top-k or top-p (the
// kernels of the digits are then left out; a row that has one all the same gets the token -1).
extern "C" int velox_sample_chunked(const float* logits, const int* options, int* out, int rows, int vocab, int chunks, void* scratch,
                                    long long scratch_bytes, int with_filter, hipStream_t stream) {
  if (rows <= 0) return 0;
  if (chunks < 2 || chunks > 1024 || rows > 65535 || scratch == nullptr || ((uintptr_t)scratch & 255) != 0) return -1;
  ChunkedScratch s;
  if ((long long)chunked_scratch_layout(rows, vocab, chunks, scratch, &s) > scratch_bytes) return -1;
  const dim3 grid(rows, chunks);
  sample_chunk_max_kernel<<<grid, SAMPLE_THREADS, 0, stream>>>(logits, options, s, vocab);
  if (with_filter) {
    sample_chunk_tables_kernel<<<grid, SAMPLE_THREADS, 0, stream>>>(logits, options, s, vocab);
    sample_chunk_list_kernel<<<grid, SAMPLE_THREADS, 0, stream>>>(logits, options, s, vocab);
    sample_finish_kernel<<<grid, SAMPLE_THREADS, 0, stream>>>(logits, options, out, s, vocab);
  } else {
    sample_chunk_draw_kernel<<<grid, SAMPLE_THREADS, 0, stream>>>(logits, options, s, vocab);
    argmax_merge_kernel<<<rows, 64, 0, stream>>>(s.chunk_best, out, chunks);
  }
  VELOX_RETURN_LAUNCH_STATUS();
}

// Penalties over the tokens a request has seen (prompt and output), each distinct token once:
//   v = logit - frequency * count;  v = v > 0 ? v / repetition : v * repetition;  v -= presence
// One workgroup per row.  The vocabulary is taken a range of PENALTY_RANGE token ids at a time: the history's tokens
// inside the range are counted into a table in LDS, then the history is walked again and whoever takes a token's count
// out of the table (leaving zero behind, so the table is clean for the next range) applies it.  Work grows with the
// history's length times the number of ranges, never with its square.
#define PENALTY_RANGE 8192
__global__ void __launch_bounds__(256) penalties_kernel(float* __restrict__ logits, const int* __restrict__ tokens, const int* __restrict__ lengths,
                                                        const float* __restrict__ coeffs, int vocab, int width) {
  __shared__ int table[PENALTY_RANGE];
  __shared__ unsigned int touched[(1 << 20) / PENALTY_RANGE / 32 + 1];  // one bit per range (vocabularies up to 2^20 ids and beyond: see below)
  const int r = blockIdx.x;
  const int n = lengths[r] < width ? lengths[r] : width;
  const int* seen = tokens + (size_t)r * width;
  const float repetition = coeffs[3 * r], presence = coeffs[3 * r + 1], frequency = coeffs[3 * r + 2];
  float* row = logits + (size_t)r * vocab;
  const int ranges = (vocab + PENALTY_RANGE - 1) / PENALTY_RANGE;
  const bool track = ranges <= (1 << 20) / PENALTY_RANGE;  // (a larger vocabulary visits every range)
  for (int i = threadIdx.x; i < PENALTY_RANGE; i += blockDim.x) table[i] = 0;
  for (int i = threadIdx.x; i < (int)(sizeof(touched) / sizeof(touched[0])); i += blockDim.x) touched[i] = 0u;
  __syncthreads();
  if (track) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
      const int token = seen[i];
      if (token >= 0 && token < vocab) atomicOr(&touched[(token / PENALTY_RANGE) >> 5], 1u << ((token / PENALTY_RANGE) & 31));
    }
    __syncthreads();
  }
  for (int range = 0; range < ranges; ++range) {
    if (track && !((touched[range >> 5] >> (range & 31)) & 1u)) continue;  // (the same for every thread)
    const int lo = range * PENALTY_RANGE;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
      const int token = seen[i];
      if (token >= lo && token < lo + PENALTY_RANGE && token < vocab) atomicAdd(&table[token - lo], 1);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
      const int token = seen[i];
      if (token < lo || token >= lo + PENALTY_RANGE || token >= vocab) continue;
      const int count = atomicExch(&table[token - lo], 0);
      if (count == 0) continue;  // another occurrence of the token took the count
      float v = row[token] - frequency * (float)count;
      v = v > 0.f ? v / repetition : v * repetition;
      row[token] = v - presence;
    }
    __syncthreads();
  }
}

extern "C" int velox_apply_penalties(float* logits, const int* tokens, const int* lengths, const float* coeffs, int rows, int vocab,
                                     int width, hipStream_t stream) {
  if (rows <= 0) return 0;
  penalties_kernel<<<rows, 256, 0, stream>>>(logits, tokens, lengths, coeffs, vocab, width);
  VELOX_RETURN_LAUNCH_STATUS();
}

// ---- penalties from a table of counts that lives on the device -------------------------------------------------------
// counts: int32 [table rows, vocab], one row per request with penalties: how often the request has seen each token
// (prompt and output).  The row is built once from the request's tokens and then kept up to date from the sampler's
// output, on the device: a step's penalties need neither the history nor the value of the token before it on the host.
__global__ void __launch_bounds__(256) count_tokens_kernel(int* __restrict__ counts_row, const int* __restrict__ tokens, int n, int vocab) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int token = tokens[i];
    if (token >= 0 && token < vocab) atomicAdd(&counts_row[token], 1);
  }
}

// row_of[r]: the table row of batch row r, or -1 (no penalties)
__global__ void __launch_bounds__(64) count_sampled_kernel(int* __restrict__ counts, const int* __restrict__ row_of, const int* __restrict__ tokens, int rows,
                                                           int vocab) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows || row_of[r] < 0) return;
  const int token = tokens[r];
  if (token >= 0 && token < vocab) atomicAdd(&counts[(size_t)row_of[r] * vocab + token], 1);  // (one request may not sit in two rows; atomic all the same)
}

// v = logit - frequency * count;  v = v > 0 ? v / repetition : v * repetition;  v -= presence, where count > 0
__global__ void __launch_bounds__(256) penalties_from_counts_kernel(float* __restrict__ logits, const int* __restrict__ counts, const int* __restrict__ row_of,
                                                                    const float* __restrict__ coeffs, int vocab) {
  const int r = blockIdx.x;
  const int table_row = row_of[r];
  if (table_row < 0) return;
  const float repetition = coeffs[3 * r], presence = coeffs[3 * r + 1], frequency = coeffs[3 * r + 2];
  float* row = logits + (size_t)r * vocab;
  const int* seen = counts + (size_t)table_row * vocab;
  for (int i = blockIdx.y * blockDim.x + threadIdx.x; i < vocab; i += gridDim.y * blockDim.x) {
    const int count = seen[i];
    if (count == 0) continue;
    float v = row[i] - frequency * (float)count;
    v = v > 0.f ? v / repetition : v * repetition;
    row[i] = v - presence;
  }
}

extern "C" int velox_count_tokens(int* counts_row, const int* tokens, int n, int vocab, hipStream_t stream) {
  if (n <= 0) return 0;
  const int blocks = (n + 255) / 256 < 256 ? (n + 255) / 256 : 256;
  count_tokens_kernel<<<blocks, 256, 0, stream>>>(counts_row, tokens, n, vocab);
  VELOX_RETURN_LAUNCH_STATUS();
}

extern "C" int velox_count_sampled(int* counts, const int* row_of, const int* tokens, int rows, int vocab, hipStream_t stream) {
  if (rows <= 0) return 0;
  count_sampled_kernel<<<(rows + 63) / 64, 64, 0, stream>>>(counts, row_of, tokens, rows, vocab);
  VELOX_RETURN_LAUNCH_STATUS();
}

extern "C" int velox_penalties_from_counts(float* logits, const int* counts, const int* row_of, const float* coeffs, int rows, int vocab, int chunks,
                                           hipStream_t stream) {
  if (rows <= 0) return 0;
  if (chunks < 1 || chunks > 65535 || rows > 65535) return -1;
  penalties_from_counts_kernel<<<dim3(rows, chunks), 256, 0, stream>>>(logits, counts, row_of, coeffs, vocab);
  VELOX_RETURN_LAUNCH_STATUS();
}
