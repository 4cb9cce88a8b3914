// FP32 weight gradients dW = X^T dz on the FP16 matrix cores.
//
// Each FP32 operand is split into two FP16 numbers x 2^s = h + l / 2^11 (l the rounded
// remainder; 22 significant bits and more) under a power of two per feature, and a product is
// xh zl + xl zh, scaled, + xh zh.  The sum runs over samples whose gradients differ by many
// powers of two, and ReLU zeros can leave an element small terms only, so the parts have to
// reach far down: a scale belongs to a feature over the samples of a split, starts where the
// first chunk's largest value needs it, with kRoom powers of two to spare, and falls when a
// later chunk's largest passes that (the sums so far are then taken along, which is exact);
// all 22 bits last down to 2^-24 of the feature's largest, the last one to 2^-46.  The matrix
// core drops what an addend holds below its accumulator's last bits, which adds up over a long
// sum (1,000 chunks accumulated in place: 7.2e-7 of the result's norm), so 32 samples are
// summed from zero, small products first, and added to the running sums by the vector unit.
// Error against 64 bits, 786,432 samples of the 8x256 net, of the result's norm: 1.1e-7; three
// bf16 parts and six products 1.7e-7; v_mfma_f32_32x32x2_f32 2.1e-7.  Element by element, of
// sum |x| |z|, with gradients spread over 2^20: at most 3.3e-7 (v_mfma_f32_32x32x2_f32:
// 2.1e-6; without the 2^11: 9e-6).
//
// A workgroup owns one sample range of one layer.  Rows come into LDS by direct loads in
// slots of SR samples, RING of them, 1 KB of whole lines per instruction; a lane then takes
// 16 samples of two features, splits them and writes 16-byte units, [plane][8-sample
// group][position], each a lane's MFMA operand (no bank conflicts).  A wave multiplies RK x RN
// blocks of 32 x 32 and issues the next chunk's loads in between.  One workgroup of 8 waves
// holds the whole 256 x 256 layer, so every row of X and dz is read once; narrower layers of
// the same net run in the same launch with part of the tile, where what they do not have is
// neither read nor multiplied.
//
// What bounds it (256 x 256, clocks per 32 samples at 1.9 GHz): splitting 2,500 by vector
// instructions, multiplying 4,500 (3,072 by the matrix cores, 2,000 by vector adds), barriers
// 400; the loads are hidden (3.3 TB/s).  Measured for the 8x256 net, all weight gradients of a
// call, against one v_mfma_f32_32x32x2_f32 GEMM (128 x 128) and one reduction per layer, and
// then three bf16 parts and six products with 256 x 128 tiles and a launch per tile shape:
//   M = 786,432: 10,200 -> 5,490 -> 5,090 us;  M = 192,064: 4,860 -> 1,380 -> 1,245 us
//   M = 65,536: 540 -> 450 us;  M = 4,096: 2,880 -> 92 -> 63 us
// Loads through registers are slower (a chunk in flight takes the 32 registers that let blocks
// overlap), and so are all loads at once (1,350 clocks until the last is taken).
#pragma once
#include "mlp_f32s.h"

namespace wg32 {

using f32s::half8;
using f32s::Planes;

constexpr int kChunk = 32;     // samples per LDS chunk
constexpr int kMaxTiles = 32;  // per launch
constexpr int kRoom = 4;       // powers of two that a feature may grow before its scale falls again
constexpr float kLow = 1.f / 2048;  // scale of the low parts, which then reach as far down as the high ones
constexpr int kTop = 126;      // the largest exponent of a scale

struct Tile {
  int xoff, zoff;  // X / dz column offsets of the layer
  int K, N;        // layer size
  int first;       // its first workgroup; one per split
  int m_per_split; // whole chunks (but for the heads)
  float* part;     // [splits][K][N]
  float* bpart;    // [splits][N] or null
};
struct Args {
  const float* X;
  const float* Z;
  int64_t ldx, ldz, M;
  int tiles;
  Tile tile[kMaxTiles];
};

__device__ __forceinline__ int tile_of(const Args& a, int block) {
  int t = 0;
  while (t + 1 < a.tiles && block >= a.tile[t + 1].first) ++t;
  return t;
}

__device__ __forceinline__ floatx16 mfma_f16(half8 a, half8 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// a s = h + l / 2^11 (s a power of two), each part rounded once.
__device__ __forceinline__ Planes split8(const float (&a)[8], float s) {
  Planes p;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const floatx2_ u = {a[2 * k] * s, a[2 * k + 1] * s};
    const f32s::half2_ h = __builtin_convertvector(u, f32s::half2_);
    const floatx2_ d = {__builtin_fmaf(a[2 * k], s, -(float)h[0]), __builtin_fmaf(a[2 * k + 1], s, -(float)h[1])};
    const f32s::half2_ l = __builtin_convertvector((floatx2_){d[0] * (1.f / kLow), d[1] * (1.f / kLow)}, f32s::half2_);
    p.h[2 * k] = h[0];
    p.h[2 * k + 1] = h[1];
    p.l[2 * k] = l[0];
    p.l[2 * k + 1] = l[1];
  }
  return p;
}

// KB x NB blocks; a wave owns RK x RN of them.
template <int KB, int NB, int RK, int RN, int SR, int RING>
__global__ __launch_bounds__(64 * (KB / RK) * (NB / RN)) void wgrad_f32s_kernel(Args a) {
  constexpr int NWN = NB / RN, NW = (KB / RK) * NWN;
  constexpr int KF = KB * 32, F = (KB + NB) * 32;  // features of the tile: X's, then dz's
  constexpr int SLOTS = kChunk / SR;               // per chunk
  constexpr int PX = SR * KF / 256, PT = SR * F / 256, PW = PT / NW;  // loads (1 KB) per slot: X, all, per wave
  static_assert(PT % NW == 0 && PX % NW == 0 && F / 64 <= NW && RING >= SLOTS);
  __shared__ float s_raw[RING][SR * F];  // [slot][X rows, dz rows]
  __shared__ half8 s_op[2][4][F];        // [plane][8-sample group][position]
  __shared__ int s_e[F];                 // by how many powers of two a feature's scale fell with the chunk
  __shared__ int s_fell[F / 64];         // whether any did, of the features that a wave stages
  const Tile T = a.tile[tile_of(a, blockIdx.x)];
  const int split = blockIdx.x - T.first;
  const int64_t mb = (int64_t)split * T.m_per_split;
  const int64_t me = mb + T.m_per_split < a.M ? mb + T.m_per_split : a.M;
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

  // Load i of a slot takes 256 / (row's features) rows of X or dz, 16 bytes per lane; features
  // past the layer's are out of range: they read as zero and cost no memory traffic.
  auto lane_offset = [&](int width, int used, int off, uint32_t rb) -> uint32_t {
    const int p = 256 * wv + 4 * lane, f = p % width;
    return f < used ? (uint32_t)(p / width) * rb + 4u * (uint32_t)(off + f) : 0x80000000u;
  };
  const uint32_t ox = lane_offset(KF, T.K, T.xoff, sx), oz = lane_offset(F - KF, T.N, T.zoff, sz);
  auto load = [&](int slot, int pos, int i) {
    const bool x = i * NW < PX;
    const int width = x ? KF : F - KF, j = x ? i : i - PX / NW;
    const uint32_t rb = x ? sx : sz;
    const uint32_t vo = (x ? ox : oz) + (uint32_t)(slot * SR + j * NW * 256 / width) * rb;
    float* dst = &s_raw[pos][(i * NW + wv) * 256];
    __builtin_amdgcn_raw_ptr_buffer_load_lds(x ? rx : rz, (__attribute__((address_space(3))) void*)dst, 16, vo, 0, 0, 0);
  };

  floatx16 acc[RK][RN];
#pragma unroll
  for (int x = 0; x < RK; ++x)
#pragma unroll
    for (int y = 0; y < RN; ++y)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[x][y][i] = 0.f;
  // Wave w < F / 64 stages features 64 w to 64 w + 63: a lane features 2 r and 2 r + 1 of them
  // in the 8-sample groups g and 2 + g.  They go to positions r and 32 + r (no bank
  // conflicts), so that a 32 x 32 block of MFMA holds every second feature of 64.
  auto feat = [](int blk, int pos) { return 64 * (blk >> 1) + 2 * pos + (blk & 1); };
  float bsum[2] = {0.f, 0.f};  // bias sums of the two features
  int se[2] = {kTop, kTop};    // exponents of their scales
  auto stage = [&](int first) {  // first: the ring position of the chunk's first slot
    floatx2_ v[2][8];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int m = 16 * j + 8 * g;  // of the chunk
      int pos = first + m / SR;
      pos -= pos >= RING ? RING : 0;
      const float* p = 64 * wv < KF ? &s_raw[pos][(m % SR) * KF + 64 * wv] : &s_raw[pos][SR * KF + (m % SR) * (F - KF) + 64 * wv - KF];
      const int pitch = 64 * wv < KF ? KF : F - KF;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[j][e] = *reinterpret_cast<const floatx2_*>(p + e * pitch + 2 * r);
    }
    bool fell = false;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float mx = 0.f;  // the feature's largest of the chunk
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(fmaxf(mx, fabsf(v[0][e][h])), fabsf(v[1][e][h]));
      mx = fmaxf(mx, shfl_xor(mx, 32));
      const int s0 = mx > 0.f ? f32s::scale_exp(mx, kTop) : kTop, s = s0 < se[h] ? s0 - kRoom : se[h], f = 64 * wv + r + 32 * h;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        float u[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) u[e] = v[j][e][h];
        const Planes p = split8(u, f32s::pow2(s));
        s_op[0][2 * j + g][f] = p.h;
        s_op[1][2 * j + g][f] = p.l;
        if (64 * wv >= KF) bsum[h] += ((u[0] + u[1]) + (u[2] + u[3])) + ((u[4] + u[5]) + (u[6] + u[7]));
      }
      if (g == 0) s_e[f] = s - se[h];
      fell |= s != se[h];
      se[h] = s;
    }
    const bool any = __any(fell);
    if (lane == 0) s_fell[wv] = any;
  };
  auto operand = [&](int blk, int t) -> Planes {
    return {s_op[0][2 * t + g][32 * blk + r], s_op[1][2 * t + g][32 * blk + r]};
  };
  auto row = [&](int x, int i) { return 32 * (rk0 + x) + 8 * (i / 4) + 4 * g + i % 4; };
  auto col = [&](int y) { return 32 * (KB + rn0 + y) + r; };
  // (the next loads are issued between the blocks: in one go they take 1,350 clocks)
  auto compute = [&](auto&& next) {
    int fell = 0;
#pragma unroll
    for (int i = 0; i < (RK + 1) / 2; ++i) fell |= s_fell[rk0 / 2 + i];
#pragma unroll
    for (int i = 0; i < (RN + 1) / 2; ++i) fell |= s_fell[(KB + rn0) / 2 + i];
    if (__builtin_amdgcn_readfirstlane(fell)) {
#pragma unroll
      for (int x = 0; x < RK; ++x)
#pragma unroll
        for (int y = 0; y < RN; ++y)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            acc[x][y][i] = __builtin_ldexpf(acc[x][y][i], s_e[row(x, i)] + s_e[col(y)]);
    }
    // Per block: the small products from zero, their scale, the large products; the block before
    // is added to the running sums, and operands and rows are fetched, while the small ones run.
    constexpr int KS = kChunk / 16, B = RK * RN;
    Planes z[KS], p[2][KS];
    floatx16 w[2];
    auto fetch = [&](int b) {
#pragma unroll
      for (int t = 0; t < KS; ++t) p[b & 1][t] = operand(rk0 + b % RK, t);
    };
    auto add = [&](int b) {
      floatx16& c = acc[b % RK][b / RK];
#pragma unroll
      for (int i = 0; i < 16; ++i) c[i] += w[b & 1][i];
      asm volatile("" : "+v"(c));  // added here, not sunk past the next block
    };
    fetch(0);
#pragma unroll
    for (int b = 0; b < B; ++b) {
      floatx16& c = w[b & 1];
      if (b % RK == 0)
#pragma unroll
        for (int t = 0; t < KS; ++t) z[t] = operand(KB + rn0 + b / RK, t);
      __builtin_amdgcn_sched_barrier(0);
      if (b + 1 < B) fetch(b + 1);
      next(b);
#pragma unroll
      for (int i = 0; i < 16; ++i) c[i] = 0.f;
#pragma unroll
      for (int t = 0; t < KS; ++t) {
        c = mfma_f16(p[b & 1][t].h, z[t].l, c);
        c = mfma_f16(p[b & 1][t].l, z[t].h, c);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (b > 0) add(b - 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 16; ++i) c[i] *= kLow;
#pragma unroll
      for (int t = 0; t < KS; ++t) c = mfma_f16(p[b & 1][t].h, z[t].h, c);
    }
    __builtin_amdgcn_sched_barrier(0);
    add(B - 1);
  };

  const int nchunks = (rows + kChunk - 1) / kChunk;
  // a barrier for LDS alone: the loads of the newest slots stay in flight across it
  auto sync = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  // this wave's loads but those of the RING - SLOTS newest slots have landed
  auto landed = [] { asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RING - SLOTS) * PW) : "memory"); };
#pragma unroll
  for (int i = 0; i < RING * PW; ++i) load(i / PW, i / PW, i % PW);
  landed();
  sync();
  const bool has = 64 * (rk0 / 2) < T.K && 64 * (rn0 / 2) < T.N;  // both blocks of 64 features hold some of each
  int first = 0;
  for (int c = 0; c < nchunks; ++c) {
    if (64 * wv < F) stage(first);
    sync();
    auto next = [&](int b) {
      constexpr int L = SLOTS * PW, B = RK * RN;
#pragma unroll
      for (int l = b * L / B; l < (b + 1) * L / B; ++l) {
        const int i = l / PW;
        load(c * SLOTS + RING + i, first + i - (first + i >= RING ? RING : 0), l % PW);
      }
    };
    if (has) {
      compute(next);
    } else {
#pragma unroll
      for (int b = 0; b < RK * RN; ++b) next(b);
    }
    first += SLOTS - (first + SLOTS >= RING ? RING : 0);
    landed();
    sync();
  }
  // (no load may still write when the workgroup's LDS is given back)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  if (64 * wv < F && g == 0) {
    s_e[64 * wv + r] = -se[0];
    s_e[64 * wv + 32 + r] = -se[1];
  }
  __syncthreads();
  float* out = T.part + (int64_t)split * T.K * T.N;
#pragma unroll
  for (int x = 0; x < RK; ++x)
#pragma unroll
    for (int y = 0; y < RN; ++y) {
      const int nn = feat(rn0 + y, r);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int kk = feat(rk0 + x, 8 * (i / 4) + 4 * g + i % 4);
        if (kk < T.K && nn < T.N) out[(int64_t)kk * T.N + nn] = __builtin_ldexpf(acc[x][y][i], s_e[row(x, i)] + s_e[col(y)]);
      }
    }
  if (T.bpart && 64 * wv >= KF && 64 * wv < F) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float b = bsum[h] + shfl_xor(bsum[h], 32);
      const int f = 64 * wv - KF + 2 * r + h;
      if (g == 0 && f < T.N) T.bpart[(int64_t)split * T.N + f] = b;
    }
  }
}

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
__global__ __launch_bounds__(256) void wgrad_head_kernel(Args a) {
  __shared__ float red[256][3];
  const Tile T = a.tile[tile_of(a, blockIdx.x)];
  const int split = blockIdx.x - T.first;
  const int64_t mb = (int64_t)split * T.m_per_split;
  const int64_t me = mb + T.m_per_split < a.M ? mb + T.m_per_split : a.M;
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
