// resident.h — lane and memory helpers shared by the resident recurrences (recurrent weights in the
// registers of one workgroup, or of a small cluster of workgroups).
#pragma once

#include <hip/hip_runtime.h>

namespace rxmet {

// A buffer offset past every buffer: a load returns 0, a store is dropped.
constexpr unsigned kResSkip = 0x80000000u;

// All of the workgroup's LDS accesses are complete; memory accesses stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__device__ __forceinline__ void buf_f32(__amdgpu_buffer_rsrc_t r, float v, unsigned off) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, 0, 0);
}
__device__ __forceinline__ void buf_u16(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned off) {
  __builtin_amdgcn_raw_buffer_store_b16(static_cast<unsigned short>(v), r, off, 0, 0);
}
__device__ __forceinline__ void buf_u8(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned off) {
  __builtin_amdgcn_raw_buffer_store_b8(static_cast<unsigned char>(v), r, off, 0, 0);
}
__device__ __forceinline__ float buf_load_f32(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
__device__ __forceinline__ unsigned buf_load_u32(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return static_cast<unsigned>(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
__device__ __forceinline__ unsigned buf_load_u16(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return static_cast<unsigned short>(__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0));
}
__device__ __forceinline__ unsigned buf_load_u8(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return static_cast<unsigned char>(__builtin_amdgcn_raw_buffer_load_b8(r, off, 0, 0));
}

// A value from the lane's quad partner (lane ^ 1, lane ^ 2).
__device__ __forceinline__ unsigned quad_xor1(unsigned v) {
  return static_cast<unsigned>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), 0xB1, 0xf, 0xf, true));
}
__device__ __forceinline__ unsigned quad_xor2(unsigned v) {
  return static_cast<unsigned>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), 0x4E, 0xf, 0xf, true));
}

// Largest of the 16 lanes of a row, in every lane of it.
__device__ __forceinline__ unsigned row16_max(unsigned v) {
  v = max(v, quad_xor1(v));
  v = max(v, quad_xor2(v));
  v = max(v, static_cast<unsigned>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), 0x141, 0xf, 0xf, true)));
  return max(v, static_cast<unsigned>(
                    __builtin_amdgcn_mov_dpp(static_cast<int>(v), 0x140, 0xf, 0xf, true)));
}

// Byte i of the quad's four words, to its lane i (byte k from lane k).
__device__ __forceinline__ unsigned quad_transpose8(unsigned v, int lane) {
  v = __builtin_amdgcn_perm(quad_xor1(v), v, lane & 1 ? 0x03070105u : 0x06020400u);
  return __builtin_amdgcn_perm(quad_xor2(v), v, lane & 2 ? 0x03020706u : 0x05040100u);
}

typedef unsigned v2u __attribute__((ext_vector_type(2)));

// 16-bit value i of the quad's lanes (values 0, 1 in a, 2, 3 in b, low half first), to its lane i
// (from lanes 0, 1 in the first word, 2, 3 in the second).
__device__ __forceinline__ v2u quad_transpose16(unsigned a, unsigned b, int lane) {
  const unsigned s = lane & 1 ? 0x03020706u : 0x05040100u;
  const unsigned p = __builtin_amdgcn_perm(quad_xor1(a), a, s);
  const unsigned q = __builtin_amdgcn_perm(quad_xor1(b), b, s);
  const unsigned r = quad_xor2(lane & 2 ? p : q);
  return lane & 2 ? v2u{r, q} : v2u{p, r};
}

// Block fixed point: with `top` the bits of the largest magnitude (below 2^(ex - 126), ex its
// exponent field), every value scaled by 2^fixed_exp(top) is below 2^30.
__device__ __forceinline__ int fixed_exp(unsigned top) { return 156 - static_cast<int>(top >> 23); }
__device__ __forceinline__ bool fixed_bad(unsigned top) { return top >= 0x7f800000u; }

// A value at exponent ex as four signed byte digits (digit k in byte k): adding 128 to the three
// low bytes carries into the next, and flipping their top bits subtracts it again.
__device__ __forceinline__ unsigned fixed_digits(float v, int ex) {
  const int q = static_cast<int>(rintf(ldexpf(v, ex)));
  return (static_cast<unsigned>(q) + 0x00808080u) ^ 0x00808080u;
}

// Two neighbouring digit sums over at most 256 products of bytes (each within 2^22) as one integer.
__device__ __forceinline__ int fixed_pair(int s0, int s1) { return s1 * 256 + s0; }

// The sum of products from the pairs of its four digit sums, back at the values' scale; exact (47
// bits).  In fp32 the pairs would be rounded, an error that stays where they cancel.
__device__ __forceinline__ double fixed_sum(int lo, int hi, int ex) {
  return __builtin_ldexp(__builtin_fma(static_cast<double>(hi), 65536.0, static_cast<double>(lo)), -ex);
}

}  // namespace rxmet
