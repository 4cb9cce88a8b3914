// FP32 dX chain of the reference topology (W = 256 with the rgb branch) on the BF16
// matrix cores (mlp_split3.h): the backward twin of mlp_fwd_f32s.h.
//
// dh_{l-1} = W_l[:W] dz_l: wave w of a workgroup owns input block w (32 features)
// of every layer, the k-steps run over the layer's outputs, dz_l sits in LDS as
// split B operands, the transposed weights stream from L2.  The ReLU masks are the
// forward's 16-bit words, one 16-byte load per lane and sample block for the whole
// trunk; every dz row is written in FP32 for the weight GEMMs through a buffer
// resource over the workgroup's rows (rows past M fall outside it).  One workgroup
// fills a CU with N = 2; N = 1 where the samples do not fill the chip, the forward's
// rule.
//
// Bound by the matrix cores (0.58 busy at 1.69 GHz) and the dz stores (9.9 KB a sample).  Against the register-resident
// v_mfma_f32_16x16x4f32 kernel that it replaced: 6,570 -> 4,580 us at 786,432 samples
// (1,150 TFLOP/s of BF16 work), 1,665 -> 1,110 at 192,064, 188 -> 53 at 8,192, 142 -> 39 at
// 1,000; the dz rows' error against 64 bits 5.5e-7 -> 1.9e-7 of their norm at the last layer
// (h0), 1.6e-7 -> 0.8e-7 at the first of 256 inputs.  (Two FP16 parts under a scale per sample
// took 2,800 us and were at 3.5e-7; cotangents below 2^-93 came out too large, and features
// of unlike size lost the small ones.)
//   rgb = sigmoid(z):  dz_rgb = d_rgb * rgb (1 - rgb)
//   sigma = relu(z):   dz_sigma = d_sigma * [sigma > 0]
//   dz = dh * [h > 0] for the ReLU layers; the bottleneck is linear.
#pragma once
#include "mlp_split3.h"

template <int W, int D, int SKIP, int LX, int LD, int N>
__global__ __launch_bounds__(512, 2) void mlp_bwd_f32s_kernel(
    MlpPlan P, const char* __restrict__ pk, int64_t M, const float* __restrict__ d_rgb,
    const float* __restrict__ d_sigma, const float* __restrict__ rgb, const float* __restrict__ sigma,
    const float* __restrict__ stash, float* __restrict__ dz) {
  using namespace split3;
  using C = NetC<W, D, SKIP, LX, LD>;
  static_assert(W == 256 && D == 8 && C::NBR == 4 && (N == 1 || N == 2), "split kernel is for the 8x256 NeRF MLP");
  constexpr int AR = N == 1 ? 6 : 4, BR = 2;               // as in the forward
  constexpr int TR = 2 * C::NBR;                           // k-steps over the rgb branch's outputs
  __shared__ bf16x8 s_tile[N][kTH * kStep];  // 48 KB per sample block: dz of the layer above
  const int lane = threadIdx.x & 63, j = lane & 31, g = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t base = (int64_t)blockIdx.x * (32 * N);
  const __amdgpu_buffer_rsrc_t rs = ws::packed_rsrc(pk + P.p_bs[1], P.bs_bytes);
  const uint32_t lane_off = 16u * (uint32_t)lane;
  auto unit0 = [&](int l) -> int64_t { return P.p_bs[l] - P.p_bs[1] + (int64_t)wv * (l == D + 1 ? TR : kTH) * kUnit; };
  Planes a[AR];
#pragma unroll
  for (int t = 0; t < AR - 1; ++t) a[t] = load_unit(rs, lane_off, unit0(D + 1) + t * kUnit);

  const int64_t w_rows = M - base < 32 * N ? M - base : 32 * N;
  const __amdgpu_buffer_rsrc_t rst = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(stash) + base * P.stash_per_sample, 0, (int)(w_rows * P.stash_per_sample * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t rdz =
      __builtin_amdgcn_make_buffer_rsrc(dz + base * P.dz_per_sample, 0, (int)(w_rows * P.dz_per_sample * 4), 0x00020000);
  const uint32_t row_bytes = (uint32_t)(P.dz_per_sample * 4), row_z = j * row_bytes, blk_z = 32 * row_bytes;
  auto store_block = [&](const floatx16& v, int n, int64_t el) {  // features 8 q + 4 g + r of a block
#pragma unroll
    for (int q = 0; q < 4; ++q)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, floatx4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]}),
                                             rdz, row_z + n * blk_z + (uint32_t)(4 * (el + 8 * q + 4 * g)), 0, 0);
  };
  // the forward's ReLU words of this wave's block, all trunk layers (8 words, one load)
  const uint32_t row_s = (uint32_t)((j * P.stash_per_sample + P.st_mask) * 4), blk_s = (uint32_t)(32 * P.stash_per_sample * 4);
  u32x4 mw[N];
  float dzs[N];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    mw[n] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                          rst, row_s + n * blk_s + (uint32_t)(2 * D * (2 * wv + g)), 0, 0));
    const int64_t m = base + 32 * n + j;
    dzs[n] = m < M && sigma[m] > 0.f ? d_sigma[m] : 0.f;
  }
  lds_b8* tile[N];
#pragma unroll
  for (int n = 0; n < N; ++n) tile[n] = ws::lds_lane(s_tile[n], 0, lane);
  Acc acc[N];

  // v = this wave's block of dz for a sample block: k-steps 2 blk, 2 blk + 1 of its tile
  auto put_tile = [&](const floatx16& v, lds_b8* to, int blk) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = v[8 * h + i];
      put_step(to + (2 * blk + h) * kStep, split8(x));
    }
  };

  // ---- rgb head: dh_rbr[f] = sum_c W_rgb[f][c] dz_rgb[c], masked; wave w does output block
  // w % 4 of sample block w / 4
  {
    const int n = N == 1 ? 0 : wv >> 2, nb = wv & 3;
    const bool own = wv < 4 * N;
    if (own) {
      floatx16 v;
      const int64_t m = base + 32 * n + j;
      float dzr[3] = {0.f, 0.f, 0.f};
      if (m < M) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const float y = rgb[3 * m + c];
          dzr[c] = d_rgb[3 * m + c] * y * (1.f - y);  // sigmoid'
        }
      }
      if (nb == 0 && g == 0) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, dzr[c]), rdz,
                                                row_z + n * blk_z + (uint32_t)((P.dz_rgb + c) * 4), 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, n ? dzs[N - 1] : dzs[0]), rdz,
                                              row_z + n * blk_z + (uint32_t)(P.dz_sigma * 4), 0, 0);
      }
      const uint32_t mr = __builtin_amdgcn_raw_buffer_load_b16(
          rst, row_s + n * blk_s + (uint32_t)(2 * (16 * D + 2 * nb + g)), 0, 0);
      const floatx4* hr4 = reinterpret_cast<const floatx4*>(pk + P.p_head_rgb) + g * 16 * C::NBR + 16 * nb;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const floatx4 w = hr4[i];
        const float d = dzr[0] * w[0] + dzr[1] * w[1] + dzr[2] * w[2];
        v[i] = (mr >> i) & 1u ? d : 0.f;
      }
      store_block(v, n, P.dz_rbr + 32 * nb);
      put_tile(v, n ? tile[N - 1] : tile[0], nb);
    }
    lds_barrier();
  }

  // ---- layers D + 1 (to the bottleneck, linear), D (to h_{D-1}, with the density head's part)
  // and D - 1 .. 1 (to h_{l-1})
  constexpr auto ring0 = [](int s) { return s == 0 ? 0 : (TR + (s - 1) * kTH) % AR; };
  ws::static_for<0, D + 1>([&](auto Sc) {
    constexpr int s = decltype(Sc)::value, l = D + 1 - s, R = ring0(s);
#pragma unroll
    for (int n = 0; n < N; ++n) zero(acc[n]);
    constexpr int T = s == 0 ? TR : kTH;
    steps<N, T, T, R, AR, BR>(a, acc, tile, tile, rs, lane_off, unit0(l), unit0(l > 1 ? l - 1 : 1));
    const int64_t el = (l == D + 1 ? P.dz_bott : P.dz_h[l - 1]) + 32 * wv;
#pragma unroll
    for (int n = 0; n < N; ++n) {
      floatx16& v = acc[n].h;
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = sum(acc[n], i);
      if constexpr (l == D) {  // + W_sigma dz_sigma
        const floatx4* hs = reinterpret_cast<const floatx4*>(pk + P.p_head_sigma) + (g * C::KH + 16 * wv) / 4;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx4 w = hs[q];
#pragma unroll
          for (int r = 0; r < 4; ++r) v[4 * q + r] = v[4 * q + r] + w[r] * dzs[n];
        }
      }
      if constexpr (l <= D) {
        const uint32_t w = mw[n][(l - 1) >> 1];
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = (w >> (16 * ((l - 1) & 1) + i)) & 1u ? v[i] : 0.f;
      }
    }
    lds_barrier();  // every wave has read the tile
#pragma unroll
    for (int n = 0; n < N; ++n)
      store_rows(acc[n].h, tile[n] + 2 * wv * kStep, lane, rdz, n * blk_z + (uint32_t)(4 * el), row_bytes);
    if constexpr (l > 1) {
#pragma unroll
      for (int n = 0; n < N; ++n) put_tile(acc[n].h, tile[n], wv);
      lds_barrier();
    }
  });
}

template <int W, int D, int SKIP, int LX, int LD>
void launch_bwd_f32s(const MlpPlan& P, const void* packed, int64_t M, const float* d_rgb, const float* d_sigma,
                     const float* rgb, const float* sigma, const void* stash, void* dz, hipStream_t s) {
  auto go = [&](auto Nc) {
    constexpr int N = decltype(Nc)::value;
    mlp_bwd_f32s_kernel<W, D, SKIP, LX, LD, N><<<(unsigned)((M + 32 * N - 1) / (32 * N)), 64 * split3::kWaves, 0, s>>>(
        P, reinterpret_cast<const char*>(packed), M, d_rgb, d_sigma, rgb, sigma,
        reinterpret_cast<const float*>(stash), reinterpret_cast<float*>(dz));
  };
  if (M <= (int64_t)32 * nerf_num_cus())
    go(std::integral_constant<int, 1>{});
  else
    go(std::integral_constant<int, 2>{});
}
