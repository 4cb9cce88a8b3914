// FP32 weight gradients dW = X^T dz on the BF16 matrix cores (mlp_split3.h): both operands
// held exactly, in three bf16 parts each, a product six partial products.
//
// The sum runs over samples whose gradients differ by any number of powers of two, and ReLU
// zeros can leave an element small terms only, so no scale of a feature or a sample serves
// here (two FP16 parts under a scale per feature were faster, 4,695 us at 786,432 samples, but
// 2^-47 below a feature's largest value nothing was left of them).  32 samples are summed
// from zero, in an accumulator for each order of size, and added to the running sums by the
// vector unit: the matrix core drops what an addend holds below the products' last bits,
// always towards minus infinity, so small sums carried into larger products add up an offset
// (1.2e-6 of the result's norm at 786,432 samples, 0.87 of it the same for all elements).
// Error against 64 bits, X normal behind a ReLU, dz normal, of the result's norm:
// M = 786,432 5.2e-7, 192,064 2.7e-7, 65,536 2.3e-7, 4,096 0.9e-7, where
// v_mfma_f32_32x32x2_f32 had 8.6e-7, 6.9e-7, 6.8e-7, 5.8e-7.
//
// A workgroup owns one sample range of one tile of KB x NB blocks of 32 x 32.  It
// stages 32-sample chunks: a thread loads 8 samples of one feature, splits them
// and writes one 16-byte unit per plane, [plane][8-sample group][feature], which
// is a lane's MFMA operand; reads and writes are free of bank conflicts.  Two LDS
// buffers, one barrier per chunk; half of the waves stage chunk c + 1 before they
// multiply chunk c, the others after it, so that on each SIMD one wave splits
// while the other multiplies.  The loads of chunk c + 2 are in flight meanwhile.
// The 256 x 256 layers run as two 256 x 128 tiles (two buffers of the whole would not
// fit), placed on one XCD, so that the rows of X they share come from its L2.  Tiles of
// one shape share a launch and one launch sums every split.
//
// Measured for the 8x256 net, all weight gradients of a call, against one FP32 GEMM
// (128 x 128 tiles, v_mfma_f32_32x32x2_f32) and one reduction per layer:
//   M = 786,432: 10,170 -> 6,460 us; the 256 x 128 tiles take 5,680 of them at 925 TFLOP/s
//     of BF16 work (the vector unit's sums beside them; accumulated in place 4,690 us, with
//     an error of 9.5e-7)
//   M = 192,064: 4,860 -> 1,610 us;  65,536: 3,670 -> 568;  4,096: 2,890 -> 85
#pragma once
#include "mlp_split3.h"

namespace wg32 {

constexpr int kChunk = 32;     // samples per LDS chunk
constexpr int kMaxTiles = 32;  // per launch

using split3::Planes;

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

// KB x NB blocks; a wave owns RK x RN of them.
template <int KB, int NB, int RK, int RN>
__global__ __launch_bounds__(64 * (KB / RK) * (NB / RN)) void wgrad_f32s_kernel(Args a) {
  constexpr int NWN = NB / RN, NW = (KB / RK) * NWN, NT = 64 * NW;
  constexpr int KF = KB * 32, F = (KB + NB) * 32;  // features of the tile: X's, then dz's
  constexpr int U = F * (kChunk / 8);              // units (8 samples of a feature) per chunk
  constexpr int UT = (U + NT - 1) / NT;            // per thread; a wave's 64 are of one 8-sample group, all X or all dz
  static_assert(KF % 64 == 0 && F % 64 == 0);
  __shared__ bf16x8 s_op[2][3][kChunk / 8][F];  // [buffer][plane][8-sample group][feature]
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

  // Unit k of this thread: features f0 + lane of the tile, samples 8 mg to 8 mg + 7 of a chunk, all
  // of it but the lane wave-uniform.  The rows of the split are a buffer resource: rows past it
  // read as zero.
  struct Unit {
    __amdgpu_buffer_rsrc_t rows;
    uint32_t pitch, at;  // bytes of a row; of the unit's first value from the split's first row
    int place;           // in a plane
    bool on, z;
  };
  auto unit = [&](int k) {
    const int u0 = 64 * wv + k * NT, mg = u0 / F, f0 = u0 % F;
    Unit u;
    u.on = U % NT == 0 || u0 < U;
    u.z = f0 >= KF;
    const int64_t ld = u.z ? a.ldz : a.ldx;
    u.rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(u.z ? a.Z : a.X) + mb * ld, 0, (int)(rows * ld * 4),
                                               0x00020000);
    u.pitch = (uint32_t)ld * 4u;
    u.at = 8u * (uint32_t)mg * u.pitch + 4u * (uint32_t)(u.z ? T.zoff + T.n0 + f0 - KF : T.xoff + f0);
    u.place = u0;
    return u;
  };

  floatx16 acc[RK][RN];
#pragma unroll
  for (int x = 0; x < RK; ++x)
#pragma unroll
    for (int y = 0; y < RN; ++y)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[x][y][i] = 0.f;
  float v[UT][8];  // the loaded units
  float bsum[UT];  // sums over the samples (the bias, for units of dz)
#pragma unroll
  for (int k = 0; k < UT; ++k) bsum[k] = 0.f;
  auto load = [&](int c) {
#pragma unroll
    for (int k = 0; k < UT; ++k) {
      const Unit u = unit(k);
      if (!u.on) continue;
      uint32_t vo = (uint32_t)(c * kChunk) * u.pitch + u.at + 4u * (uint32_t)lane;
#pragma unroll
      for (int e = 0; e < 8; ++e, vo += u.pitch)
        v[k][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(u.rows, vo, 0, 0));
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int k = 0; k < UT; ++k) {
      const Unit u = unit(k);
      if (!u.on) continue;
      const Planes p = split3::split8(v[k]);
      bf16x8* o = &s_op[buf][0][0][0] + u.place + lane;
      o[0] = p.h;
      o[U] = p.m;
      o[2 * U] = p.l;
      bsum[k] += ((v[k][0] + v[k][1]) + (v[k][2] + v[k][3])) + ((v[k][4] + v[k][5]) + (v[k][6] + v[k][7]));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto operand = [&](int buf, int blk, int t) -> Planes {
    const bf16x8* o = &s_op[buf][0][2 * t + g][32 * blk + r];
    return {o[0], o[U], o[2 * U]};
  };
  auto compute = [&](int buf) {
    constexpr int KS = kChunk / 16;
    const floatx16 zero = {};
#pragma unroll
    for (int y = 0; y < RN; ++y) {
      Planes z[KS];
#pragma unroll
      for (int t = 0; t < KS; ++t) z[t] = operand(buf, KB + rn0 + y, t);
#pragma unroll
      for (int x = 0; x < RK; ++x) {
        Planes p[KS];
#pragma unroll
        for (int t = 0; t < KS; ++t) p[t] = operand(buf, rk0 + x, t);
        split3::Acc c;
#pragma unroll
        for (int t = 0; t < KS; ++t) {
          c.l = mfma_bf16(p[t].l, z[t].h, t ? c.l : zero);
          c.m = mfma_bf16(p[t].m, z[t].h, t ? c.m : zero);
          c.h = mfma_bf16(p[t].h, z[t].h, t ? c.h : zero);
          c.l = mfma_bf16(p[t].m, z[t].m, c.l);
          c.m = mfma_bf16(p[t].h, z[t].m, c.m);
          c.l = mfma_bf16(p[t].h, z[t].l, c.l);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[x][y][i] += split3::sum_finite(c, i);
        asm volatile("" : "+v"(acc[x][y]));  // (added here, not sunk past the next block)
        __builtin_amdgcn_sched_barrier(0);
      }
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
        if (kk < T.K && nn < T.N) out[(int64_t)kk * T.N + nn] = acc[x][y][i];
      }
    }
  if (T.bpart) {
    // the four 8-sample groups of a feature (the loop ended with a barrier)
    float* red = reinterpret_cast<float*>(s_op);
#pragma unroll
    for (int k = 0; k < UT; ++k) {
      const Unit u = unit(k);
      if (u.on) red[u.place + lane] = bsum[k];
    }
    __syncthreads();
    for (int f = tid; f < NB * 32; f += NT)
      if (T.n0 + f < T.N) {
        const float* b = red + KF + f;
        T.bpart[(int64_t)split * T.N + T.n0 + f] = (b[0] + b[F]) + (b[2 * F] + b[3 * F]);
      }
  }
}

struct HeadArgs {
  const float* X;
  const float* Z;
  int64_t ldx, ldz, M;
  int m_per_split, splits;
  Tile tile[4];
};

// Rows m, m + R, .. of this split (up to me) into a head's sums s (FP32 FMAs in row order) and,
// where `sums`, the bias sums b + bl; N columns, B rows in flight.  Everything but column xk of X
// is wave-uniform: dz comes through scalar loads.
template <int N, int B>
__device__ __forceinline__ void head_rows(const float* __restrict__ x, int xk, const float* __restrict__ z, int64_t ldx,
                                          int64_t ldz, int64_t m, int64_t me, int R, bool sums, float (&s)[3],
                                          float (&b)[3], float (&bl)[3]) {
  const int64_t sx = R * ldx, sz = R * ldz;
  x += m * ldx;
  z += m * ldz;
  auto add_bias = [&](int c, float zc) {
    float e;
    two_sum(b[c], zc, b[c], e);
    bl[c] += e;
  };
  for (; m + (int64_t)(B - 1) * R < me; m += B * R) {
    float xv[B], zv[B][N];
#pragma unroll
    for (int e = 0; e < B; ++e, x += sx) xv[e] = x[xk];
#pragma unroll
    for (int e = 0; e < B; ++e, z += sz)
#pragma unroll
      for (int c = 0; c < N; ++c) zv[e][c] = z[c];
#pragma unroll
    for (int e = 0; e < B; ++e)
#pragma unroll
      for (int c = 0; c < N; ++c) s[c] = __builtin_fmaf(xv[e], zv[e][c], s[c]);
    if (sums)
#pragma unroll
      for (int e = 0; e < B; ++e)
#pragma unroll
        for (int c = 0; c < N; ++c) add_bias(c, zv[e][c]);
  }
  for (; m < me; m += R, x += sx, z += sz)
#pragma unroll
    for (int c = 0; c < N; ++c) {
      s[c] = __builtin_fmaf(x[xk], z[c], s[c]);
      if (sums) add_bias(c, z[c]);
    }
}

// Heads (1 or 3 output columns): dW[k][c] = sum_m X[m][k] dz[m][c].  Thread k of a
// workgroup owns feature k (two or more row groups where K < 256): FP32 FMAs, bounded
// by reading X once, so by how many rows are in flight: the single column has a loop of its
// own, for the registers and so the waves (786,432 samples, both heads: 430 -> 255 us, 5.5 TB/s).
// The bias, a single sum that may cancel, is summed with compensation
// by one wave of each row group.
__global__ __launch_bounds__(256) void wgrad_head_kernel(HeadArgs a) {
  __shared__ float red[256][3];
  const Tile T = a.tile[blockIdx.x / a.splits];
  const int split = blockIdx.x % a.splits;
  const int64_t mb = (int64_t)split * a.m_per_split;
  const int64_t me = mb + a.m_per_split < a.M ? mb + a.m_per_split : a.M;
  const int KP = T.K > 128 ? 256 : (T.K > 64 ? 128 : 64), R = 256 / KP;  // threads per row group, row groups
  const int k = threadIdx.x % KP, rg = __builtin_amdgcn_readfirstlane(threadIdx.x / KP);  // rg is wave-uniform
  const int xk = k < T.K ? k : 0;
  const float* x = a.X + T.xoff;
  const float* z = a.Z + T.zoff;
  float s[3] = {0.f, 0.f, 0.f}, b[3] = {0.f, 0.f, 0.f}, bl[3] = {0.f, 0.f, 0.f};
  const bool sums = T.bpart && k < 64;  // wave-uniform
  if (T.N == 1) head_rows<1, 16>(x, xk, z, a.ldx, a.ldz, mb + rg, me, R, sums, s, b, bl);
  else head_rows<3, 16>(x, xk, z, a.ldx, a.ldz, mb + rg, me, R, sums, s, b, bl);
#pragma unroll
  for (int c = 0; c < 3; ++c) b[c] += bl[c];
  auto combine = [&](float (&q)[3]) {  // over the row groups, in order
#pragma unroll
    for (int c = 0; c < 3; ++c) red[threadIdx.x][c] = q[c];
    __syncthreads();
    if (rg == 0)
      for (int i = 1; i < R; ++i)
#pragma unroll
        for (int c = 0; c < 3; ++c) q[c] += red[k + i * KP][c];
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
