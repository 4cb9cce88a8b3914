// FP32 weight gradients dW = X^T dz on the BF16 matrix cores.
//
// Each FP32 operand is split exactly into three bf16 numbers x = h + m + l (each
// the rounded remainder; 24 significant bits in all, FP32's range), and a product
// is the six partial products that reach 2^-24 of it: xh zh in one FP32
// accumulator, xl zh + xh zl + xm zm + xm zh + xh zm in a second one, added at the
// end.  Six v_mfma_f32_32x32x16_bf16 take 0.375 of the FP32 instruction's time,
// and the large products' sum is rounded once per 16 samples instead of once per
// sample (K = 4,096: error 3.0e-7 .. 3.8e-7 of the result's norm against 64 bits,
// v_mfma_f32_16x16x4f32 8.0e-7 .. 1.1e-6).  The sum runs over samples whose
// gradients differ by many powers of two, so the forward's two FP16 parts with one
// scale per sample do not serve here.
//
// A workgroup owns one sample range of one tile of KB x NB blocks of 32 x 32.  It
// stages 32-sample chunks: a thread loads 8 samples of one feature, splits them
// and writes one 16-byte unit per plane, [plane][8-sample group][feature], which
// is a lane's MFMA operand; reads and writes are free of bank conflicts.  Two LDS
// buffers, one barrier per chunk; half of the waves stage chunk c + 1 before they
// multiply chunk c, the others after it, so that on each SIMD one wave splits
// while the other multiplies.  The loads of chunk c + 2 are in flight meanwhile.
// The 256 x 256 layers run as two 256 x 128 tiles (both accumulators fit), placed
// on one XCD, so that the rows of X they share come from its L2.  Tiles of one
// shape share a launch and one launch sums every split.
//
// Measured for the 8x256 net, all weight gradients of a call, against one FP32 GEMM
// (128 x 128 tiles, v_mfma_f32_32x32x2_f32) and one reduction per layer:
//   M = 786,432: 10,200 -> 5,490 us; the 256 x 128 tiles take 4,690 of them at 1,121
//     TFLOP/s of BF16 work, where a bare stream of the six products with random
//     operands, LDS and L2 reads runs at 1,250 to 1,450 (power)
//   M = 192,064: 4,860 -> 1,380 us;  M = 4,096: 2,880 -> 92 us (12 reductions of 192
//     to 256 splits, one thread per output, were 240 us each)
#pragma once
#include "mlp_kernels.h"

namespace wg32 {

constexpr int kChunk = 32;     // samples per LDS chunk
constexpr int kMaxTiles = 32;  // per launch

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

struct Tile {
  int xoff, zoff;  // X / dz column offsets of the layer
  int K, N, n0;    // layer size, first column of the tile
  float* part;     // [splits][K][N]
  float* bpart;    // [splits][N] or null
};
struct Args {
  const float* X;
  const float* Z;
  int64_t ldx, ldz, M;
  int m_per_split, splits;  // m_per_split: a multiple of kChunk
  int pairs, singles;       // tiles 2 p and 2 p + 1 (p < pairs) share X rows
  Tile tile[kMaxTiles];
};

// x = h + m + l exactly (round to nearest each; non-finite x gives NaN in m and l).
__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = pack_bf16x2(a, b);
  const float ra = fsub(a, __builtin_bit_cast(float, h << 16));
  const float rb = fsub(b, __builtin_bit_cast(float, h & 0xffff0000u));
  m = pack_bf16x2(ra, rb);
  l = pack_bf16x2(fsub(ra, __builtin_bit_cast(float, m << 16)), fsub(rb, __builtin_bit_cast(float, m & 0xffff0000u)));
}

struct Planes {
  bf16x8 h, m, l;
};

__device__ __forceinline__ void mfma6(const Planes& a, const Planes& b, floatx16& hi, floatx16& lo) {
  lo = mfma_bf16(a.l, b.h, lo);
  hi = mfma_bf16(a.h, b.h, hi);
  lo = mfma_bf16(a.h, b.l, lo);
  lo = mfma_bf16(a.m, b.m, lo);
  lo = mfma_bf16(a.m, b.h, lo);
  lo = mfma_bf16(a.h, b.m, lo);
}

// KB x NB blocks; a wave owns RK x RN of them.
template <int KB, int NB, int RK, int RN>
__global__ __launch_bounds__(64 * (KB / RK) * (NB / RN)) void wgrad_f32s_kernel(Args a) {
  constexpr int NWN = NB / RN, NW = (KB / RK) * NWN, NT = 64 * NW;
  constexpr int XU = KB * 128, U = (KB + NB) * 128;  // units (8 samples of a feature) per chunk: X, all
  constexpr int UT = (U + NT - 1) / NT;              // per thread; whole waves of X or of Z
  __shared__ u32x4 s_x[2][3][4][KB * 32];
  __shared__ u32x4 s_z[2][3][4][NB * 32];
  // workgroup -> (tile, split); the two tiles of a pair are 8 apart: one XCD
  int ti, split;
  {
    const int P = a.pairs * a.splits, b0 = 16 * ((P + 7) / 8), b = blockIdx.x;
    if (b < b0) {
      const int q = (b >> 4) * 8 + (b & 7);
      if (q >= P) return;
      ti = 2 * (q % a.pairs) + ((b >> 3) & 1);
      split = q / a.pairs;
    } else {
      ti = 2 * a.pairs + (b - b0) % a.singles;
      split = (b - b0) / a.singles;
    }
  }
  const Tile T = a.tile[ti];
  const int64_t mb = (int64_t)split * a.m_per_split;
  const int64_t me = mb + a.m_per_split < a.M ? mb + a.m_per_split : a.M;
  const int rows = me > mb ? (int)(me - mb) : 0;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, g = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rk0 = (wv / NWN) * RK, rn0 = (wv % NWN) * RN;
  // rows of the split as buffer resources: rows past it read as zero
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(a.X) + mb * a.ldx, 0, (int)(rows * a.ldx * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(a.Z) + mb * a.ldz, 0, (int)(rows * a.ldz * 4), 0x00020000);
  const uint32_t sx = (uint32_t)a.ldx * 4u, sz = (uint32_t)a.ldz * 4u;  // row bytes

  floatx16 hi[RK][RN], lo[RK][RN];
#pragma unroll
  for (int x = 0; x < RK; ++x)
#pragma unroll
    for (int y = 0; y < RN; ++y)
#pragma unroll
      for (int i = 0; i < 16; ++i) hi[x][y][i] = lo[x][y][i] = 0.f;

  float v[UT][8];   // the loaded unit(s) of this thread
  float bsum[UT];   // bias sums of its Z features
#pragma unroll
  for (int k = 0; k < UT; ++k) bsum[k] = 0.f;
  // unit u of the chunk: X for u < XU (u % 32 KB the feature, u / 32 KB the 8-sample group), then Z
  auto is_x = [&](int k) { return 64 * wv + k * NT < XU; };      // wave-uniform
  auto on = [&](int k) { return 64 * wv + k * NT < U; };
  auto load = [&](int c) {
#pragma unroll
    for (int k = 0; k < UT; ++k) {
      if (!on(k)) continue;
      const int u = tid + k * NT;
      if (is_x(k)) {
        const int f = u % (KB * 32), mg = u / (KB * 32);
        uint32_t vo = (uint32_t)(c * kChunk + 8 * mg) * sx + 4u * (uint32_t)(T.xoff + f);
#pragma unroll
        for (int e = 0; e < 8; ++e, vo += sx)
          v[k][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, vo, 0, 0));
      } else {
        const int f = (u - XU) % (NB * 32), mg = (u - XU) / (NB * 32);
        uint32_t vo = (uint32_t)(c * kChunk + 8 * mg) * sz + 4u * (uint32_t)(T.zoff + T.n0 + f);
#pragma unroll
        for (int e = 0; e < 8; ++e, vo += sz)
          v[k][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rz, vo, 0, 0));
      }
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int k = 0; k < UT; ++k) {
      if (!on(k)) continue;
      u32x4 p[3];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t h, m, l;
        split2(v[k][2 * e], v[k][2 * e + 1], h, m, l);
        p[0][e] = h;
        p[1][e] = m;
        p[2][e] = l;
      }
      const int u = tid + k * NT;
      if (is_x(k)) {
#pragma unroll
        for (int q = 0; q < 3; ++q) (&s_x[buf][q][0][0])[u] = p[q];
      } else {
#pragma unroll
        for (int q = 0; q < 3; ++q) (&s_z[buf][q][0][0])[u - XU] = p[q];
#pragma unroll
        for (int e = 0; e < 8; ++e) bsum[k] += v[k][e];
      }
    }
  };
  auto operand = [&](const auto& s, int buf, int blk, int t) -> Planes {
    const int f = 32 * blk + r, mg = 2 * t + g;
    return {__builtin_bit_cast(bf16x8, s[buf][0][mg][f]), __builtin_bit_cast(bf16x8, s[buf][1][mg][f]),
            __builtin_bit_cast(bf16x8, s[buf][2][mg][f])};
  };
  auto compute = [&](int buf) {
#pragma unroll
    for (int t = 0; t < kChunk / 16; ++t) {
      Planes z[RN];
#pragma unroll
      for (int y = 0; y < RN; ++y) z[y] = operand(s_z, buf, rn0 + y, t);
#pragma unroll
      for (int x = 0; x < RK; ++x) {
        const Planes p = operand(s_x, buf, rk0 + x, t);
#pragma unroll
        for (int y = 0; y < RN; ++y) mfma6(p, z[y], hi[x][y], lo[x][y]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  const int nchunks = (rows + kChunk - 1) / kChunk;
  load(0);
  stage(0);
  load(1);
  __syncthreads();
  const bool early = wv < NW / 2 || NW == 1;
  for (int c = 0; c < nchunks; ++c) {
    // (chunks past the end read as zeros and are never multiplied)
    if (early) {
      stage((c + 1) & 1);
      load(c + 2);
      __builtin_amdgcn_sched_barrier(0);
    }
    compute(c & 1);
    if (!early) {
      __builtin_amdgcn_sched_barrier(0);
      stage((c + 1) & 1);
      load(c + 2);
    }
    __syncthreads();
  }

  float* out = T.part + (int64_t)split * T.K * T.N;
#pragma unroll
  for (int x = 0; x < RK; ++x)
#pragma unroll
    for (int y = 0; y < RN; ++y) {
      const int nn = T.n0 + 32 * (rn0 + y) + r;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int kk = 32 * (rk0 + x) + 8 * (i / 4) + 4 * g + (i % 4);
        if (kk < T.K && nn < T.N) out[(int64_t)kk * T.N + nn] = hi[x][y][i] + lo[x][y][i];
      }
    }
  if (T.bpart) {
    // the four 8-sample groups of a feature, in order (the loop ended with a barrier)
    float* red = reinterpret_cast<float*>(s_z);
#pragma unroll
    for (int k = 0; k < UT; ++k)
      if (on(k) && !is_x(k)) red[tid + k * NT - XU] = bsum[k];
    __syncthreads();
    for (int f = tid; f < NB * 32; f += NT)
      if (T.n0 + f < T.N)
        T.bpart[(int64_t)split * T.N + T.n0 + f] =
            ((red[f] + red[f + NB * 32]) + red[f + 2 * NB * 32]) + red[f + 3 * NB * 32];
  }
}

// Heads (at most 4 output columns): dW[k][c] = sum_m X[m][k] dz[m][c].  Thread k of a
// workgroup owns feature k (two or more row groups where K < 256): FP32 FMAs, bounded
// by reading X once.  The bias, a single sum that may cancel, is summed with compensation
// by one wave of each row group.
struct HeadArgs {
  const float* X;
  const float* Z;
  int64_t ldx, ldz, M;
  int m_per_split, splits, njobs;
  Tile tile[4];
};

__global__ __launch_bounds__(256) void wgrad_head_kernel(HeadArgs a) {
  __shared__ float red[256][4];
  const Tile T = a.tile[blockIdx.x / a.splits];
  const int split = blockIdx.x % a.splits;
  const int64_t mb = (int64_t)split * a.m_per_split;
  const int64_t me = mb + a.m_per_split < a.M ? mb + a.m_per_split : a.M;
  const int KP = T.K > 128 ? 256 : (T.K > 64 ? 128 : 64), R = 256 / KP;  // threads per row group, row groups
  const int k = threadIdx.x % KP, rg = threadIdx.x / KP;                  // rg is wave-uniform
  const float* x = a.X + T.xoff + (k < T.K ? k : 0);
  const float* z = a.Z + T.zoff;
  float s[4] = {0.f, 0.f, 0.f, 0.f}, b[4] = {0.f, 0.f, 0.f, 0.f}, bl[4] = {0.f, 0.f, 0.f, 0.f};
  const bool sums = T.bpart && k < 64;  // wave-uniform
  auto add_bias = [&](int c, float zc) {
    float e;
    two_sum(b[c], zc, b[c], e);
    bl[c] += e;
  };
  constexpr int B = 16;  // rows in flight
  int64_t m = mb + rg;
  for (; m + (int64_t)(B - 1) * R < me; m += B * R) {
    float xv[B], zv[B][4];
#pragma unroll
    for (int e = 0; e < B; ++e) xv[e] = x[(m + e * R) * a.ldx];
#pragma unroll
    for (int e = 0; e < B; ++e)
#pragma unroll
      for (int c = 0; c < 4; ++c) zv[e][c] = c < T.N ? z[(m + e * R) * a.ldz + c] : 0.f;
#pragma unroll
    for (int e = 0; e < B; ++e)
#pragma unroll
      for (int c = 0; c < 4; ++c) s[c] = __builtin_fmaf(xv[e], zv[e][c], s[c]);
    if (sums)
#pragma unroll
      for (int e = 0; e < B; ++e)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (c < T.N) add_bias(c, zv[e][c]);
  }
  for (; m < me; m += R)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float zc = c < T.N ? z[m * a.ldz + c] : 0.f;
      s[c] = __builtin_fmaf(x[m * a.ldx], zc, s[c]);
      if (sums) add_bias(c, zc);
    }
#pragma unroll
  for (int c = 0; c < 4; ++c) b[c] += bl[c];
  auto combine = [&](float (&q)[4]) {  // over the row groups, in order
#pragma unroll
    for (int c = 0; c < 4; ++c) red[threadIdx.x][c] = q[c];
    __syncthreads();
    if (rg == 0)
      for (int i = 1; i < R; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) q[c] += red[k + i * KP][c];
    __syncthreads();
  };
  combine(s);
  combine(b);
  if (rg == 0) {
    if (k < T.K)
      for (int c = 0; c < T.N; ++c) T.part[((int64_t)split * T.K + k) * T.N + c] = s[c];
    if (k == 0 && T.bpart)
      for (int c = 0; c < T.N; ++c) T.bpart[(int64_t)split * T.N + c] = b[c];
  }
}

}  // namespace wg32
