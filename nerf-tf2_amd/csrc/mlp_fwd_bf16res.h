// BF16 forward of the density-only net with 64-wide layers (the proposal network), with or
// without the training stash: the whole net's weights stay in LDS.
//
// The per-wave kernel (mlp_fwd_bf16.h) read all 28 KB of weights from L2 for each 32 samples
// and passed every layer through an LDS slab: at 1,572,864 samples 12 TB/s of L2 traffic
// bounded it.  Here a workgroup copies the operands, biases and the head to LDS once (33 KB,
// four workgroups a CU) and its waves walk over blocks of 32 samples; a layer's accumulators
// become the next layer's B operands in registers (the weights' order is packed for that),
// and the same packed values leave as the stash's 16-byte row chunks.  Every operation and its order is the
// per-wave kernel's, so the outputs and the stash are the same bits.
// 1,572,864 samples: 122 -> 103 us, with the stash 244 -> 211 (1.0 GB written); 196,608: 21.5 ->
// 16.3 and 31.5 -> 29.4 us.  Vector instruction issue bounds it now, half of it the sines.  Four waves a
// SIMD (128 registers, accumulators in VGPRs): 104.3 us with the next block's points loaded
// ahead, 108.5 us with three waves.
#pragma once
#include "mlp_fwd_bf16ws.h"

template <int W, int D, int SKIP, int LX, int LD>
__global__ __launch_bounds__(256, 4) void mlp_fwd_bf16res_kernel(
    MlpPlan P, const char* __restrict__ pk, int64_t M, const float* __restrict__ xyz,
    const float* __restrict__ dirs, const float* __restrict__ ro, const float* __restrict__ rd,
    const float* __restrict__ tv, int spr, float* __restrict__ sig_out, __bf16* __restrict__ stash) {
  using C = NetC<W, D, SKIP, LX, LD>;
  using ws::u32x4;
  static_assert(W == 64 && !C::RGB && SKIP < 0 && C::KX == 32, "four k-steps of encoding and of each hidden layer");
  constexpr int T = 4, NB = 2, U = T * NB * 64;  // bf16x8 per layer
  __shared__ bf16x8 s_w[D * U];
  __shared__ floatx4 s_b[D * W / 4];
  __shared__ floatx4 s_h[W / 4 + 1];             // the sigma head's weights by lane half, its bias
#pragma unroll
  for (int l = 0; l < D; ++l)
#pragma unroll
    for (int i = 0; i < U / 256; ++i)
      s_w[l * U + 256 * i + threadIdx.x] = reinterpret_cast<const bf16x8*>(pk + P.p_fwd[l])[256 * i + threadIdx.x];
  if (threadIdx.x < D * W / 4)
    s_b[threadIdx.x] = reinterpret_cast<const floatx4*>(pk + P.p_bias[threadIdx.x / (W / 4)])[threadIdx.x % (W / 4)];
  if (threadIdx.x < W / 4 + 1) s_h[threadIdx.x] = reinterpret_cast<const floatx4*>(pk + P.p_head_sigma)[threadIdx.x];
  __syncthreads();

  const int lane = threadIdx.x & 63, j = lane & 31, g = lane >> 5;
  const int64_t nblk = (M + 31) / 32, step = (int64_t)gridDim.x * 4;
  int64_t blk = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float x[3], d[3];
  auto load = [&](int64_t b) {
    const int64_t m = b * 32 + j;
    load_sample(m < M ? m : M - 1, xyz, dirs, ro, rd, tv, spr, x, d);
  };
  for (; blk < nblk; blk += step) {
    load(blk);
    const int64_t m = blk * 32 + j;
    const bool valid = m < M, st = stash && valid;
    const BlkRow<__bf16> srow{stash ? stash + blk * 32 * P.stash_per_sample : nullptr,
                              (int)(M - blk * 32 < 32 ? M - blk * 32 : 32), j};
    auto put = [&](bf16x8 v, int64_t el) {
      __builtin_nontemporal_store(__builtin_bit_cast(u32x4, v), reinterpret_cast<u32x4*>(srow.at(el)));
    };
    bf16x8 b[T];
    {
      float ex[C::KX];
      encode_slots<LX, C::KX>(x, g, ex);
      slots_to_bf16(ex, b);
    }
    if (st) {
#pragma unroll
      for (int t = 0; t < T; ++t) put(b[t], P.st_encx + g * C::KX + 8 * t);
    }
    ws::static_for<0, D>([&](auto Lc) {
      constexpr int l = decltype(Lc)::value;
      floatx16 acc[NB];
      zero_acc(acc);
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[nb] = mfma_bf16(s_w[l * U + (t * NB + nb) * 64 + lane], b[t], acc[nb]);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx4 bv = s_b[l * (W / 4) + 8 * nb + 2 * q + g];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = acc[nb][4 * q + r] + bv[r];
            acc[nb][4 * q + r] = v > 0.f ? v : 0.f;
          }
        }
        b[2 * nb] = acc_to_bf16(acc[nb], 0);
        b[2 * nb + 1] = acc_to_bf16(acc[nb], 1);
      }
      if (stash) {
        bf16x8 row[T];  // (both lane halves take part in the swap)
#pragma unroll
        for (int t = 0; t < T; ++t) row[t] = ws::swap_halves(b[t]);
        if (st) {
#pragma unroll
          for (int t = 0; t < T; ++t) put(row[t], P.st_h[l] + 16 * t + 8 * g);
        }
      }
    });
    // sigma head on the rounded activations
    float zs = 0.f;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const floatx4 w = s_h[g * (W / 8) + 2 * t + h];
#pragma unroll
        for (int r = 0; r < 4; ++r) zs = zs + (float)b[t][4 * h + r] * w[r];
      }
    zs = zs + shfl_xor(zs, 32);
    zs = zs + s_h[W / 4][0];
    if (valid && g == 0) sig_out[m] = softplus(zs);
  }
}

template <int W, int D, int SKIP, int LX, int LD>
void launch_fwd_bf16res(const MlpPlan& P, const void* packed, int64_t M, const float* xyz, const float* dirs,
                        const float* ro, const float* rd, const float* tv, int spr, float* sigma, void* stash,
                        hipStream_t s) {
  // four workgroups a CU (LDS), each over as many blocks as that leaves it
  int64_t grid = (M + 127) / 128;
  const int64_t most = (int64_t)4 * nerf_num_cus();
  if (grid > most) grid = most;
  mlp_fwd_bf16res_kernel<W, D, SKIP, LX, LD><<<(unsigned)grid, 256, 0, s>>>(
      P, reinterpret_cast<const char*>(packed), M, xyz, dirs, ro, rd, tv, spr, sigma,
      reinterpret_cast<__bf16*>(stash));
}
