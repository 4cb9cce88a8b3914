// FP32 products on the FP16 matrix cores, for the 8x256 NeRF MLP.
//
// An FP32 operand x, scaled by a power of two into the FP16 range, is split into
// h = fp16(x) and l = fp16(x - h): 22 significant bits and the sign of l, within
// 2^-23 of x.  A product is ah bh, summed in one FP32 accumulator, plus al bh +
// ah bl, summed in a second one (they are 2^-11 of it; al bl is dropped at 2^-22
// of it, on average 2^-24.6); the two are added once per output.
// v_mfma_f32_32x32x16_f16 does 16 times the work per cycle of the FP32
// instruction, so the three products take 3/16 of its time; and the large
// products' sum is rounded once per 16 terms, not once per term.  Error against
// 64 bits of a K-term dot product (norm of the error over norm of the result,
// weights uniform, inputs normal / after a ReLU):
//   K = 256: 1.3e-7 / 1.3e-7, v_mfma_f32_16x16x4f32 2.9e-7 / 2.0e-7
//   K =  64: 9.9e-8 / 9.9e-8, v_mfma_f32_16x16x4f32 1.4e-7 / 1.0e-7
// (all three products in one accumulator: 1.9e-7 at K = 256).  The scale puts the
// largest input of a sample (weights: of an output block of 32) into [2^14,
// 2^15); inputs down to 2^-16 of it keep all their split's bits, smaller ones
// have an error of 2^-40 of it, so no FP32 value overflows or vanishes that would
// not in FP32.
#pragma once
#include "mlp_fwd_bf16ws.h"

namespace f32s {

using ws::u32x4;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2_ __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) half8 lds_h8;
typedef __attribute__((address_space(3))) floatx4 lds_f4;
typedef __attribute__((address_space(3))) float lds_f;

constexpr int kWaves = 8;     // waves per workgroup: wave w owns output block w of every layer
constexpr int kUnit = 2048;   // bytes of one (output block, k-step): two planes of 1 KB
constexpr int kTH = 16;       // k-steps of a hidden input

struct Planes {  // one k-step of an operand: high and low parts
  half8 h, l;
};

// Exponent s that brings m (the largest magnitude) to [2^14, 2^15) as m 2^s; 15 for m = 0.
// At most 126, so that 2^s is a normal number: inputs that are all below 2^-112 come out
// smaller than that.  (Weights: at most 60, see inv_scale.)
__device__ __forceinline__ int scale_exp(float m, int most = 126) {
  const int s = 15 - __builtin_amdgcn_frexp_expf(m);
  return s < most ? s : most;
}
__device__ __forceinline__ float pow2(int e) { return __builtin_ldexpf(1.f, e); }

// The factor that takes sums of inputs scaled by 2^se and weights scaled by 2^we back; where
// it leaves the FP32 range, so does what it scales.
__device__ __forceinline__ float inv_scale(int se, int we) {
  const int e = -(se + we);
  return pow2(e < -126 ? -126 : (e > 127 ? 127 : e));
}

// a s and b s split (s a power of two): the remainder a s - h is exact in one v_fma_mix_f32.
__device__ __forceinline__ void split2(float a, float b, float s, uint32_t& h, uint32_t& l) {
  const half2_ hv = __builtin_convertvector((floatx2_){fmul(a, s), fmul(b, s)}, half2_);
  const float ra = __builtin_fmaf(a, s, -(float)hv[0]), rb = __builtin_fmaf(b, s, -(float)hv[1]);
  h = __builtin_bit_cast(uint32_t, hv);
  l = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2_){ra, rb}, half2_));
}

__device__ __forceinline__ Planes split8(const float (&v)[8], float s) {
  uint32_t h[4], l[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) split2(v[2 * k], v[2 * k + 1], s, h[k], l[k]);
  return {__builtin_bit_cast(half8, u32x4{h[0], h[1], h[2], h[3]}),
          __builtin_bit_cast(half8, u32x4{l[0], l[1], l[2], l[3]})};
}

__device__ __forceinline__ void mfma3(const Planes& a, const Planes& b, floatx16& hi, floatx16& lo) {
  lo = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.l, b.h, lo, 0, 0, 0);
  hi = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.h, b.h, hi, 0, 0, 0);
  lo = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.h, b.l, lo, 0, 0, 0);
}

// Workgroup barrier that orders LDS only (global loads and stores stay in flight).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ half8 ldh(__amdgpu_buffer_rsrc_t r, uint32_t voff, int64_t soff) {
  return __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(r, voff, (int)soff, 0));
}

__device__ __forceinline__ Planes load_unit(__amdgpu_buffer_rsrc_t rs, uint32_t lane_off, int64_t off) {
  return {ldh(rs, lane_off, off), ldh(rs, lane_off, off + 1024)};
}

// Per-lane LDS pointer to element `lane` of a half8 array, opaque to the optimiser.
__device__ __forceinline__ lds_h8* lds_lane(const half8* arr, int lane) {
  uint32_t a = (uint32_t)(uintptr_t)(const lds_h8*)arr + 16u * (uint32_t)lane;
  asm volatile("" : "+v"(a));
  return (lds_h8*)(uintptr_t)a;
}

// hi, lo += the products of this wave's output block with N sample blocks over T
// k-steps, B operands from the tile (per-lane pointer per sample block).  The
// weights of the first AR - 1 k-steps are in a[R ..]; every step loads the unit
// AR - 1 steps ahead, past the end those that follow at `next`.  R is the ring
// position of the first k-step.  BR: k-steps' B operands in registers (BR - 1 are
// read ahead).
template <int N, int T, int R, int AR, int BR>
__device__ __forceinline__ void steps(Planes (&a)[AR], floatx16 (&hi)[N], floatx16 (&lo)[N],
                                      lds_h8* const (&tile)[N], __amdgpu_buffer_rsrc_t rs, uint32_t lane_off,
                                      int64_t cur, int64_t next) {
  Planes b[BR][N];
  auto read = [&](int t) {
#pragma unroll
    for (int n = 0; n < N; ++n) b[t % BR][n] = {tile[n][t * 128], tile[n][t * 128 + 64]};
  };
#pragma unroll
  for (int t = 0; t < BR - 1; ++t) read(t);
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int ta = t + AR - 1;
    a[(R + ta) % AR] = load_unit(rs, lane_off, ta < T ? cur + ta * kUnit : next + (ta - T) * kUnit);
    if (t + BR - 1 < T) read(t + BR - 1);
    if (BR > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < N; ++n) mfma3(a[(R + t) % AR], b[t % BR][n], hi[n], lo[n]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <int N>
__device__ __forceinline__ void zero(floatx16 (&v)[N]) {
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) v[n][i] = 0.f;
}

// The largest of a sample's 256 magnitudes: mx over this lane's 16, then over the lane halves
// and (LDS, [block][sample]) the waves.  put, a barrier, get.
__device__ __forceinline__ void put_max(lds_f* s, int wv, int j, int g, float mx) {
  mx = fmaxf(mx, shfl_xor(mx, 32));
  if (g == 0) s[wv * 32 + j] = mx;
}
__device__ __forceinline__ float get_max(const lds_f* s, int j) {
  float m = 0.f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) m = fmaxf(m, s[w * 32 + j]);
  return m;
}

// A 32 x 32 block of FP32 rows (v: lane (j, g) holds features 8 q + 4 g + r of row j) to a
// row-major buffer, through this wave's 4 KB of LDS: each store instruction then writes eight
// whole 128-byte lines, non-temporally, instead of 32-byte pieces of 32 rows (786,432 samples:
// forward with stash 3,560 -> 3,190 us with two layers' ReLU words per store, dX chain 3,180 ->
// 2,850; the pieces stored non-temporally took twice the time).  off: byte offset of feature 0 of the
// block's row 0 in the resource, whose range drops rows past the batch.  (The 16-byte pieces of
// a row are XORed with the row in LDS, so neither pass has bank conflicts.)
__device__ __forceinline__ void store_rows(const floatx16& v, lds_h8* slot, int lane, __amdgpu_buffer_rsrc_t r,
                                           uint32_t off, uint32_t row_bytes) {
  lds_f4* s = (lds_f4*)(slot - lane);  // (slot is this lane's pointer)
  const int j = lane & 31, g = lane >> 5;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    s[8 * j + ((2 * q + g) ^ (j & 7))] = floatx4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
  wave_sync();
  const int r0 = lane >> 3, c = lane & 7;
  floatx4 x[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = s[64 * i + 8 * r0 + (c ^ r0)];
  uint32_t o = off + r0 * row_bytes + 16u * (uint32_t)c;
#pragma unroll
  for (int i = 0; i < 4; ++i, o += 8 * row_bytes)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x[i]), r, o, 0, kNT);
  wave_sync();
}

}  // namespace f32s
