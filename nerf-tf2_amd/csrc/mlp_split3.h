// FP32 products on the BF16 matrix cores, for the 8x256 NeRF MLP.
//
// An FP32 operand is held exactly, as three bf16 numbers x = h + m / 2^6 + l / 2^12: h the top
// half of x's bits (so that an infinity stays one and no finite x becomes one), m and l the
// rounded remainders, 24 significant bits.  m and l are stored scaled up, so that all three have
// about the exponent of x: every finite x of at least 2^-122 in magnitude is exact, whatever
// stands beside it (below that the last bits of l reach under bf16's range), and no scale is
// needed for a sample, a feature or a block.  A product is the six partial products that reach
// 2^-23 of it, in three FP32 accumulators of one order each, h h; m h + h m; l h + h l + m m,
// added once per output, the small ones first (the three that are left out are below 2^-22 of
// the product, 2^-25 on average).  An infinite or NaN operand makes the small sums NaN; the
// large one alone is then what FP32's sum is.
//
// v_mfma_f32_32x32x16_bf16 does 16 times the work per cycle of the FP32 instruction, so the
// six products take 3/8 of its time; and a sum is rounded once per 16 terms, not once per term.
// Two FP16 parts and three products are faster still (render launch below: 18.7 ms), but their
// 22 bits lie within 2^-40 of the largest value that shares the scale: nets with features or
// weights of very unlike size, which FP32 computes as well as any other, came out wrong.
#pragma once
#include "mlp_fwd_bf16ws.h"

namespace split3 {

using ws::lds_b8;
using ws::u32x4;

typedef __attribute__((address_space(3))) floatx4 lds_f4;

constexpr int kWaves = 8;       // waves per workgroup: wave w owns output block w of every layer
constexpr int kUnit = 3072;     // bytes of one (output block, k-step): three planes of 1 KB
constexpr int kStep = 3 * 64;   // bf16x8 of one k-step of a tile
constexpr int kTH = 16;         // k-steps of a hidden input
constexpr float kScale = 64.f;  // of m against h and of l against m: both stay below h, their sums in its range

struct Planes {  // one k-step of an operand
  bf16x8 h, m, l;
};

// a and b in three parts.
__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  auto lo = [](uint32_t p) { return __builtin_bit_cast(float, p << 16); };
  auto up = [](uint32_t p) { return __builtin_bit_cast(float, p & 0xFFFF0000u); };
  const uint32_t ua = __builtin_bit_cast(uint32_t, a), ub = __builtin_bit_cast(uint32_t, b);
  h = __builtin_amdgcn_perm(ub, ua, 0x07060302u);
  const float ra = fmul(fsub(a, up(ua)), kScale), rb = fmul(fsub(b, up(ub)), kScale);
  m = pack_bf16x2(ra, rb);
  l = pack_bf16x2(fmul(fsub(ra, lo(m)), kScale), fmul(fsub(rb, up(m)), kScale));
}

__device__ __forceinline__ Planes split8(const float (&v)[8]) {
  uint32_t h[4], m[4], l[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) split2(v[2 * k], v[2 * k + 1], h[k], m[k], l[k]);
  return {__builtin_bit_cast(bf16x8, u32x4{h[0], h[1], h[2], h[3]}),
          __builtin_bit_cast(bf16x8, u32x4{m[0], m[1], m[2], m[3]}),
          __builtin_bit_cast(bf16x8, u32x4{l[0], l[1], l[2], l[3]})};
}

// The accumulators of a block's products, by order.
struct Acc {
  floatx16 h, m, l;
};

__device__ __forceinline__ void mfma6(const Planes& a, const Planes& b, Acc& c) {
  c.l = mfma_bf16(a.l, b.h, c.l);
  c.m = mfma_bf16(a.m, b.h, c.m);
  c.h = mfma_bf16(a.h, b.h, c.h);
  c.l = mfma_bf16(a.m, b.m, c.l);
  c.m = mfma_bf16(a.h, b.m, c.m);
  c.l = mfma_bf16(a.h, b.l, c.l);
}

__device__ __forceinline__ void zero(Acc& c) {
#pragma unroll
  for (int i = 0; i < 16; ++i) c.h[i] = c.m[i] = c.l[i] = 0.f;
}

__device__ __forceinline__ float sum_finite(const Acc& c, int i) {  // NaN or infinite where FP32's sum is either
  constexpr float k = 1.f / kScale;
  return __builtin_fmaf(__builtin_fmaf(c.l[i], k, c.m[i]), k, c.h[i]);
}
__device__ __forceinline__ float sum(const Acc& c, int i) {
  return __builtin_fabsf(c.h[i]) < __builtin_inff() ? sum_finite(c, i) : c.h[i];
}

// Workgroup barrier that orders LDS only (global loads and stores stay in flight).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ Planes load_unit(__amdgpu_buffer_rsrc_t rs, uint32_t lane_off, int64_t off) {
  return {ws::ldw(rs, lane_off, off), ws::ldw(rs, lane_off, off + 1024), ws::ldw(rs, lane_off, off + 2048)};
}

__device__ __forceinline__ void put_step(lds_b8* o, const Planes& p) {
  o[0] = p.h;
  o[64] = p.m;
  o[128] = p.l;
}

// acc += the products of this wave's output block with N sample blocks over T k-steps, the
// first TH with B operands from the tile, the others from ex (per-lane pointers per sample
// block).  The weights of the first AR - 1 k-steps are in a[R ..]; every step loads the unit
// AR - 1 steps ahead, past the end those that follow at `next`.  R is the ring position of the
// first k-step.  BR: k-steps' B operands in registers (BR - 1 are read ahead).
template <int N, int T, int TH, int R, int AR, int BR>
__device__ __forceinline__ void steps(Planes (&a)[AR], Acc (&acc)[N], lds_b8* const (&tile)[N],
                                      lds_b8* const (&ex)[N], __amdgpu_buffer_rsrc_t rs, uint32_t lane_off,
                                      int64_t cur, int64_t next) {
  Planes b[BR][N];
  auto read = [&](int t) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const lds_b8* p = t < TH ? tile[n] + t * kStep : ex[n] + (t - TH) * kStep;
      b[t % BR][n] = {p[0], p[64], p[128]};
    }
  };
#pragma unroll
  for (int t = 0; t < BR - 1 && t < T; ++t) read(t);
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int ta = t + AR - 1;
    a[(R + ta) % AR] = load_unit(rs, lane_off, ta < T ? cur + ta * kUnit : next + (ta - T) * kUnit);
    if (t + BR - 1 < T) read(t + BR - 1);
    if (BR > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < N; ++n) mfma6(a[(R + t) % AR], b[t % BR][n], acc[n]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// A 32 x 32 block of FP32 rows (v: lane (j, g) holds features 8 q + 4 g + r of row j) to a
// row-major buffer, through 4 KB of this wave's LDS: each store instruction then writes eight
// whole 128-byte lines, non-temporally, instead of 32-byte pieces of 32 rows (786,432 samples:
// forward with stash 3,560 -> 3,190 us, dX chain 3,180 -> 2,850 on the two-part kernels; the
// pieces stored non-temporally took twice the time).  off: byte offset of feature 0 of the
// block's row 0 in the resource, whose range drops rows past the batch.  (The 16-byte pieces of
// a row are XORed with the row in LDS, so neither pass has bank conflicts.)
__device__ __forceinline__ void store_rows(const floatx16& v, lds_b8* slot, int lane, __amdgpu_buffer_rsrc_t r,
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

}  // namespace split3
