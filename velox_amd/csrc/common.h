// Shared helpers of the gfx950 kernels: element types, conversions, reductions, launch checks.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

// Element type codes used across the C interface.
#define VELOX_F32 0
#define VELOX_BF16 1

typedef __bf16 bf16_t;
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef short short4_t __attribute__((ext_vector_type(4)));

#define VELOX_WAVE 64

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16_t v) { return (float)v; }

template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16_t from_f32<bf16_t>(float v) { return (bf16_t)v; }

__device__ __forceinline__ short bf16_bits(float v) { return __builtin_bit_cast(short, (bf16_t)v); }

// Sum over the 64 lanes of a wave; every lane gets the result.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int offset = 32; offset > 0; offset >>= 1) v += __shfl_xor(v, offset, VELOX_WAVE);
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int offset = 32; offset > 0; offset >>= 1) v = fmaxf(v, __shfl_xor(v, offset, VELOX_WAVE));
  return v;
}

// Sum over a block of up to 1024 threads; `scratch` holds one float per wave (16 at most).
// Every thread gets the result.  The order of the additions is fixed, so the result does not
// depend on anything but the values.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & (VELOX_WAVE - 1);
  const int wave = threadIdx.x / VELOX_WAVE;
  const int waves = (blockDim.x + VELOX_WAVE - 1) / VELOX_WAVE;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int w = 0; w < waves; ++w) total += scratch[w];
  return total;
}

// 16 bytes per lane from global memory straight into LDS: lane l's piece lands at dst + 16 l, so one instruction fills a
// contiguous kilobyte.  `dst` must be the same for the whole wave.  Written as assembly on purpose: of a load that the
// compiler knows to write LDS it assumes that any later LDS read may touch what is still in flight, and waits for ALL
// outstanding loads before the first read, which undoes a load issued ahead into another buffer.  The caller orders
// things itself: `wait_for_loads<N>()` (at most N of the wave's loads still in flight) and a barrier before the reads.
__device__ __forceinline__ void load_to_lds_16(const void* src, void* dst) {
  const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)dst;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(at), "v"(src) : "memory", "m0");
}
// The same with the address as a base that is the same for the whole wave (it travels in scalar registers) plus 32 bits of
// byte offset per lane: no 64-bit vector arithmetic per load.
__device__ __forceinline__ void load_to_lds_16(const void* wave_base, uint32_t lane_bytes, void* dst) {
  const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)dst;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(at), "v"(lane_bytes), "s"(wave_base) : "memory", "m0");
}
template <int N> __device__ __forceinline__ void wait_for_loads() {
  static_assert(N >= 0 && N < 64, "the counter of loads in flight has six bits");
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// Work item `item` of a step whose sequence b has items of `size` tokens from item cu_q[b] / size + b on: those of two sequences never overlap,
// floor((a + n) / size) + 1 >= floor(a / size) + ceil(n / size), so `step_items` of them hold all.  Gives the sequence with its tokens [lo, hi)
// and the item's place in it (sequence -1: none, and lo == hi; pieces behind a sequence's end are the caller's to skip).  The whole wave
// takes part.  For a grid of one workgroup per item and not of the longest sequence's items for each: 12 single tokens beside 1,024 are
// 77 chunks of 16 and not 832, of which the empty ones held compute units while they read their sequence's ends.
struct StepItem { int sequence, lo, hi, piece; };
__host__ __device__ __forceinline__ long long step_items(int tokens, int num_seqs, int size) { return (long long)(tokens / size) + num_seqs; }
__device__ __forceinline__ StepItem step_item(const int* cu_q, int num_seqs, int size, int item) {
  const int lane = threadIdx.x & (VELOX_WAVE - 1);
  StepItem found = {-1, 0, 0, 0};
  for (int base = 0; base < num_seqs; base += VELOX_WAVE) {
    const int b = base + lane;
    const int lo = b < num_seqs ? cu_q[b] : 0, hi = b < num_seqs ? cu_q[b + 1] : 0;
    const int first = lo / size + b, here = __popcll(__ballot(b < num_seqs && first <= item));
    if (here == 0) break;
    const int last = here - 1;  // (first items rise with the sequence)
    found = {base + last, __builtin_amdgcn_readlane(lo, last), __builtin_amdgcn_readlane(hi, last), item - __builtin_amdgcn_readlane(first, last)};
    if (here < VELOX_WAVE) break;
  }
  return found;
}

// Rows of a matrix as the left operand of v_mfma_f32_16x16x32_bf16 want them, lane (g, i) two pieces of 16 bytes of row i, from loads of whole
// cache lines: what a lane asks for is `first` of row i & 7 and `second` of row 8 + (i & 7), the lanes with i >= 8 the other of the two
// pieces, so that a load covers eight rows of 128 bytes and not sixteen of 64.  Lanes eight apart then change places.  (Read once and
// in whole lines W streams at up to 7 TB/s past the caches; sixteen half lines a load, at 5.3 to 6.3, and the hint costs speed there.)
__device__ __forceinline__ void rows_from_lines(float4_t& first, float4_t& second) {
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const int a = __float_as_int(first[d]), b = __float_as_int(second[d]);
    first[d] = __int_as_float(__builtin_amdgcn_update_dpp(a, b, 0x128, 0xf, 0xc, false));   // lanes 8 .. 15 of 16 from eight lanes down,
    second[d] = __int_as_float(__builtin_amdgcn_update_dpp(b, a, 0x128, 0xf, 0x3, false));  // lanes 0 .. 7 from eight lanes up
  }
}

// Grids of a workgroup per sequence, head and tile whose time is the longest chain's: it has to begin with the first workgroups.  With up to
// ORDERED_WORKGROUPS of them each looks for the sequence with the `rank`-th most tokens (ties in their order); with more, where that would cost more than
// it gives, or beyond 64 sequences, it goes from the back, since a step's single tokens come before its portions of prompts.  (Chunks' read-outs of
// 32 heads of 64 x 64, us, searched / from the back: 60 single tokens beside 1,024 119 / 109, 64 portions of 64 282 / 269.)  The whole wave takes
// part; the lengths are gone through from their highest bit down, a few scalar instructions each.
constexpr long long ORDERED_WORKGROUPS = 1024;
static inline bool orders_sequences(long long workgroups, int num_seqs) { return num_seqs <= VELOX_WAVE && workgroups <= ORDERED_WORKGROUPS; }

__device__ __forceinline__ int sequence_by_length(const int* cu_q, int num_seqs, int rank, bool ordered) {
  if (!ordered) return num_seqs - 1 - rank;
  const int lane = threadIdx.x & (VELOX_WAVE - 1), at = lane < num_seqs ? lane : 0;
  const int begin = cu_q[at], mine = cu_q[at + 1] - begin;
  const int total = __builtin_amdgcn_readlane(begin + mine, num_seqs - 1);
  uint64_t among = __ballot(lane < num_seqs);
  for (int bit = 31 - __builtin_clz(total | 1); bit >= 0; --bit) {
    const uint64_t more = among & __ballot((mine >> bit) & 1);
    const int count = __popcll((unsigned long long)more);
    if (rank < count) {
      among = more;
    } else {
      rank -= count;
      among &= ~more;
    }
  }
  const int before = __builtin_amdgcn_mbcnt_hi((unsigned)(among >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)among, 0));  // of the lanes before this one
  return __ffsll((unsigned long long)__ballot(before == rank && ((among >> lane) & 1))) - 1;
}

// Grids of chains of up to ALONE_WORKGROUPS workgroups have a compute unit each to themselves: with ALONE_LDS bytes of LDS more no second one fits.  (Two
// chains on a compute unit slow each other down, many short ones hide each other's waits.  Three portions of 400 to 1,300 tokens, 32 heads of 64 x 64,
// 384 workgroups, us, up to two a compute unit / one: 134 / 124; eight of 300, 16 heads of 64 x 64, 512: 48 / 52; 32 heads, 1,024: 84 / 90.)
constexpr size_t ALONE_WORKGROUPS = 384, ALONE_LDS = 80 * 1024;

// Four consecutive elements of a row, widened to float32: one 8- or 16-byte access when `vec_ok` (the row starts on such a
// boundary and k is a multiple of 4) and all four lie below k_limit, else element by element with zeros beyond k_limit.
template <typename T>
__device__ __forceinline__ void load4(const T* __restrict__ base, size_t row_offset, int k, int k_limit, bool row_ok, bool vec_ok, float (&v)[4]) {
  if (!row_ok) { v[0] = v[1] = v[2] = v[3] = 0.f; return; }
  const T* p = base + row_offset + k;
  if (vec_ok && k + 3 < k_limit) {
    if constexpr (sizeof(T) == 4) {
      const float4_t x = *reinterpret_cast<const float4_t*>(p);
      v[0] = x[0]; v[1] = x[1]; v[2] = x[2]; v[3] = x[3];
    } else {
      const short4_t x = *reinterpret_cast<const short4_t*>(p);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(((uint32_t)(uint16_t)x[i]) << 16);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (k + i < k_limit) ? to_f32(p[i]) : 0.f;
  }
}

// The middle of a gated unit: g sigmoid(alpha g) (u + shift) with g = min(gate, limit), u = clamp(up, -limit, limit);
// (1, inf, 0) is silu(gate) * up.
struct GluUnit { float alpha, limit, shift; };
__device__ __forceinline__ float glu_middle(float gate, float up, const GluUnit& unit) {
  const float g = fminf(gate, unit.limit);
  const float u = fminf(fmaxf(up, -unit.limit), unit.limit);
  return g / (1.f + expf(-unit.alpha * g)) * (u + unit.shift);
}

// The middle of a unit without a gate branch, act(up): kind 1 is relu(up)^2 (any other kind passes the value).
#define VELOX_ACT_RELU2 1
__device__ __forceinline__ float ungated_act(float v, int kind) {
  const float r = fmaxf(v, 0.f);
  return kind == VELOX_ACT_RELU2 ? r * r : v;
}

#define VELOX_RETURN_LAUNCH_STATUS() return (int)hipGetLastError()
