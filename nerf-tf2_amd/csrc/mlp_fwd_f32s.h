// FP32 forward of the reference topology (W = 256 with the rgb branch), with or
// without the training stash, on the BF16 matrix cores (mlp_split3.h).
//
// A workgroup of eight waves carries 32 N samples through every layer.  Wave w
// owns output block w (32 features); a layer's input sits in LDS as split B
// operands (48 KB per sample block), the encodings beside it, the weights, split
// when they are packed, stream from L2 as 1 KB loads three k-steps ahead.  A layer
// ends with the bias, the ReLU and, behind a barrier, the split values' stores
// over the old tile.  One workgroup fills a CU with N = 2.
//
// What bounds it: the matrix cores at the clock that they are held at (0.65 busy at 1.89 GHz).
// At 6,291,456 samples it takes 32.9 to 34.1 ms (219 to 227 TFLOP/s of FP32 work, 1,310 to 1,360
// of BF16 work, where a bare stream of the six products with random operands, LDS and
// L2 reads runs at 1,250 to 1,450), against 51.0 ms of the register-resident
// v_mfma_f32_16x16x4f32 kernel that it replaced.  (Two FP16 parts and three products took
// 18.7 ms, without FP32's range: mlp_split3.h.)  Error against 64 bits, of the norm over 4,096
// samples: a layer by itself 0.7e-7 (FP32 instruction 1.9e-7), densities 1.2e-7 (3.3e-7), colours
// 0.45e-7 (0.73e-7).
//
// N = 1 halves a workgroup's serial time where the samples do not fill the chip, and doubles
// the weights' traffic: M = 1,000 189 us (FP32 instruction) -> 39.8; N = 1 / 2: 38.3 / 70.9 us
// at M = 4,096, 51.2 / 71.3 at 8,192, 87.4 / 74.9 at 12,000, 100.7 / 89.3 at 16,384, and with
// the stash 59.7 / 82.0 at 8,192, 103.5 / 88.4 at 12,000, so N = 1 up to 32 samples per CU.
#pragma once
#include "mlp_split3.h"

// N sample blocks of 32 per workgroup.
template <int W, int D, int SKIP, int LX, int LD, int N, bool STASH>
__global__ __launch_bounds__(512, 2) void mlp_fwd_f32s_kernel(
    MlpPlan P, const char* __restrict__ pk, int64_t M, const float* __restrict__ xyz,
    const float* __restrict__ dirs, const float* __restrict__ ro, const float* __restrict__ rd,
    const float* __restrict__ tv, int spr, float* __restrict__ rgb_out, float* __restrict__ sig_out,
    float* __restrict__ stash) {
  using namespace split3;
  using C = NetC<W, D, SKIP, LX, LD>;
  static_assert(W == 256 && C::KX == 32 && C::KD == 16 && D % 2 == 0 && SKIP >= 0 && SKIP + 1 < D,
                "split kernel is for the 8x256 NeRF MLP");
  static_assert(N == 1 || N == 2, "the rgb branch's 4 N output blocks go to waves 0 .. 4 N - 1");
  constexpr int TX = C::KX / 8, TD = C::KD / 8;
  // weight units and k-steps of B operands in registers
  constexpr int AR = N == 1 ? 6 : 4, BR = 2;
  constexpr int NBIAS = (D + 1) * C::NB + C::NBR;
  __shared__ bf16x8 s_tile[N][kTH * kStep];      // 48 KB per sample block: a layer's input
  __shared__ bf16x8 s_ex[N][TX * kStep];         // 12 KB: the xyz encoding
  __shared__ bf16x8 s_ed[N][TD * kStep];         // 6 KB: the direction encoding
  __shared__ floatx4 s_bias[NBIAS * 8];          // 9.5 KB: [block][lane half][16]
  __shared__ float s_sig[N][kWaves * 32];        // sigma-head partials per block and sample
  __shared__ float s_pt[N][6][32];               // sample points and directions
  const int lane = threadIdx.x & 63, j = lane & 31, g = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t base = (int64_t)blockIdx.x * (32 * N);
  const __amdgpu_buffer_rsrc_t rs = ws::packed_rsrc(pk + P.p_fs[0], P.fs_bytes);
  const uint32_t lane_off = 16u * (uint32_t)lane;
  // this wave's units of layer l start here (rgb branch: output block wv % 4)
  auto unit0 = [&](int l) -> int64_t {
    const int T = l == 0 ? TX : (l == SKIP + 1 ? kTH + TX : (l <= D ? kTH : kTH + TD));
    return P.p_fs[l] - P.p_fs[0] + (int64_t)(l <= D ? wv : wv & 3) * T * kUnit;
  };
  Planes a[AR];
#pragma unroll
  for (int t = 0; t < AR - 1; ++t)
    a[t] = load_unit(rs, lane_off, t < TX ? unit0(0) + t * kUnit : unit0(1) + (t - TX) * kUnit);

  // the stash rows of this workgroup as a buffer resource (rows past M fall outside it)
  const int64_t w_rows = M - base < 32 * N ? M - base : 32 * N;
  const __amdgpu_buffer_rsrc_t rst =
      STASH ? __builtin_amdgcn_make_buffer_rsrc(stash + base * P.stash_per_sample, 0,
                                                (int)(w_rows * P.stash_per_sample * 4), 0x00020000)
            : rs;
  const uint32_t row_bytes = (uint32_t)(P.stash_per_sample * 4), row = j * row_bytes, blk_row = 32 * row_bytes;
  auto st4 = [&](floatx4 v, int n, int64_t el) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rst, row + n * blk_row + (uint32_t)(4 * el), 0, 0);
  };

  if (threadIdx.x < 32 * N) {
    const int64_t m = base + threadIdx.x;
    float x[3], d[3];
    load_sample(m < M ? m : M - 1, xyz, dirs, ro, rd, tv, spr, x, d);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      s_pt[threadIdx.x >> 5][c][threadIdx.x & 31] = x[c];
      s_pt[threadIdx.x >> 5][3 + c][threadIdx.x & 31] = d[c];
    }
  }
  // k-step t of an encoding of L frequencies (K slots per lane half) of sample block n
  auto encode = [&](auto Lc, int c0, int n, int t, bf16x8* to, int64_t st_off) {
    constexpr int L = decltype(Lc)::value, K = L == LX ? C::KX : C::KD;
    const float x[3] = {s_pt[n][c0][j], s_pt[n][c0 + 1][j], s_pt[n][c0 + 2][j]};
    float v[8];
    encode_kstep<L>(x, g, t, v);
    put_step((lds_b8*)to + lane, split8(v));
    if constexpr (STASH) {
      st4(floatx4{v[0], v[1], v[2], v[3]}, n, st_off + g * K + 8 * t);
      st4(floatx4{v[4], v[5], v[6], v[7]}, n, st_off + g * K + 8 * t + 4);
    }
  };
  // biases of every layer in accumulator order (element 4 a + r of half g: feature 8 a + 4 g + r)
  {
    const __amdgpu_buffer_rsrc_t rp = ws::packed_rsrc(pk, P.packed_bytes);
    for (int e = threadIdx.x; e < NBIAS * 8; e += 64 * kWaves) {
      const int blk = e >> 3, h = (e >> 2) & 1, q = e & 3;
      const int l = blk / C::NB < D + 1 ? blk / C::NB : D + 1;
      s_bias[e] = ws::ldf4(rp, 4u * (uint32_t)(32 * (blk - C::NB * l) + 8 * q + 4 * h) + (uint32_t)P.p_bias[l], 0);
    }
  }
  lds_b8 *tile[N], *ex[N], *ed[N];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    tile[n] = ws::lds_lane(s_tile[n], 0, lane);
    ex[n] = ws::lds_lane(s_ex[n], 0, lane);
    ed[n] = ws::lds_lane(s_ed[n], 0, lane);
  }
  const lds_f4* bias = (const lds_f4*)&s_bias[8 * wv + 4 * g];
  Acc acc[N];
  uint32_t mw[N];
  lds_barrier();
  // the encodings, a k-step of a sample block at a time (wave u % 8)
  for (int u = wv; u < (TX + TD) * N; u += kWaves) {
    if (u < TX * N)
      encode(std::integral_constant<int, LX>{}, 0, u / TX, u % TX, &s_ex[u / TX][u % TX * kStep], P.st_encx);
    else
      encode(std::integral_constant<int, LD>{}, 3, (u - TX * N) / TD, u % TD, &s_ed[(u - TX * N) / TD][u % TD * kStep],
             P.st_encd);
  }
  lds_barrier();

  // ring position of layer l's first weight unit
  constexpr auto ring0 = [](int l) {
    int u = 0;
    for (int i = 0; i < l; ++i) u += i == 0 ? TX : (i == SKIP + 1 ? kTH + TX : kTH);
    return u % AR;
  };
  ws::static_for<0, D + 1>([&](auto Lc) {
    constexpr int l = decltype(Lc)::value, R = ring0(l);
#pragma unroll
    for (int n = 0; n < N; ++n) zero(acc[n]);
    constexpr int TH = l == 0 ? 0 : kTH, T = TH + (l == 0 || l == SKIP + 1 ? TX : 0);
    steps<N, T, TH, R, AR, BR>(a, acc, tile, ex, rs, lane_off, unit0(l), unit0(l + 1));
    const int64_t st_off = (l < D ? P.st_h[l] : P.st_bott) + 32 * wv;
#pragma unroll
    for (int n = 0; n < N; ++n) {
      floatx16& v = acc[n].h;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const floatx4 b = bias[8 * C::NB * l + q];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 4 * q + r;
          v[i] = sum(acc[n], i) + b[r];
          if constexpr (l < D) v[i] = v[i] > 0.f ? v[i] : 0.f;
        }
      }
      if constexpr (STASH && l < D) {
        // ReLU words of this block and lane half, two layers per store
        uint32_t w = 0u;
#pragma unroll
        for (int i = 0; i < 16; ++i) w |= (v[i] > 0.f ? 1u : 0u) << i;
        if constexpr ((l & 1) == 0)
          mw[n] = w;
        else
          __builtin_amdgcn_raw_buffer_store_b32(mw[n] | (w << 16), rst,
                                                row + n * blk_row + (uint32_t)(4 * P.st_mask + 2 * ((2 * wv + g) * D + l - 1)), 0, 0);
      }
      if constexpr (l == D - 1) {
        // sigma head on h_{D-1} (model.py:374-375): this block's part of the dot product
        const floatx4* hs = reinterpret_cast<const floatx4*>(pk + P.p_head_sigma) + (g * C::KH + 16 * wv) / 4;
        float z = 0.f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx4 w = hs[q];
#pragma unroll
          for (int r = 0; r < 4; ++r) z = z + v[4 * q + r] * w[r];
        }
        z = z + shfl_xor(z, 32);
        if (g == 0) s_sig[n][wv * 32 + j] = z;
      }
    }
    lds_barrier();  // every wave has read the tile
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const floatx16& u = acc[n].h;
      lds_b8* o = tile[n] + 2 * wv * kStep;
      if constexpr (STASH) store_rows(u, o, lane, rst, n * blk_row + (uint32_t)(4 * st_off), row_bytes);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = u[8 * h + i];
        put_step(o + h * kStep, split8(v));
      }
    }
    lds_barrier();
  });

  // ---- dense_{D+1} on concat(bottleneck, direction encoding) (model.py:380-384): wave w
  // does output block w % 4 of sample block w / 4
  constexpr int RR = ring0(D + 1);
  const bool own = wv < 4 * N;
  const int n = N == 1 ? 0 : wv >> 2, nb = wv & 3;
  Acc c1[1];
  lds_b8* t1[1];
  lds_b8* e1[1];
  t1[0] = n ? tile[N - 1] : tile[0];
  e1[0] = n ? ed[N - 1] : ed[0];
  zero(c1[0]);
  float p0 = 0.f, p1 = 0.f, p2 = 0.f;
  if (own) {
    steps<1, kTH + TD, kTH, RR, AR, BR>(a, c1, t1, e1, rs, lane_off, unit0(D + 1), unit0(D + 1));
    const floatx4* hr4 = reinterpret_cast<const floatx4*>(pk + P.p_head_rgb) + g * 16 * C::NBR + 16 * nb;
    floatx16& v = c1[0].h;
    const lds_f4* br = (const lds_f4*)&s_bias[8 * (C::NB * (D + 1) + nb) + 4 * g];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const floatx4 b = br[q];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 4 * q + r;
        const float z = sum(c1[0], i) + b[r];
        v[i] = z > 0.f ? z : 0.f;
        const floatx4 w = hr4[i];  // rgb head (model.py:386-387)
        p0 = p0 + v[i] * w[0];
        p1 = p1 + v[i] * w[1];
        p2 = p2 + v[i] * w[2];
      }
      if constexpr (STASH)
        st4(floatx4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]}, n,
            P.st_rbr + 32 * nb + 8 * q + 4 * g);
    }
    if constexpr (STASH) {
      uint32_t w = 0u;
#pragma unroll
      for (int i = 0; i < 16; ++i) w |= (v[i] > 0.f ? 1u : 0u) << i;
      __builtin_amdgcn_raw_buffer_store_b16((unsigned short)w, rst,
                                            row + n * blk_row + (uint32_t)(4 * P.st_mask + 2 * (16 * D + 2 * nb + g)), 0, 0);
    }
    p0 = p0 + shfl_xor(p0, 32);
    p1 = p1 + shfl_xor(p1, 32);
    p2 = p2 + shfl_xor(p2, 32);
  }
  lds_barrier();  // the tile is free: rgb-head partials per output block and sample
  float* s_red = reinterpret_cast<float*>(s_tile);  // [nb][n][3][32]
  if (own && g == 0) {
    float* o = s_red + (nb * N + n) * 96 + j;
    o[0] = p0;
    o[32] = p1;
    o[64] = p2;
  }
  lds_barrier();
  // outputs: thread 4 q + c of the first 128 N finishes colour c (c < 3) or sigma of sample q
  if (threadIdx.x < 128 * N) {
    const int q = threadIdx.x >> 2, c = threadIdx.x & 3, nn = q >> 5, jj = q & 31;
    const int64_t m = base + q;
    if (m < M) {
      if (c < 3) {
        const float* r = s_red + nn * 96 + c * 32 + jj;
        const float z = ((r[0] + r[N * 96]) + (r[2 * N * 96] + r[3 * N * 96])) +
                        reinterpret_cast<const float*>(pk + P.p_head_rgb)[2 * 16 * C::NBR * 4 + c];
        rgb_out[3 * m + c] = sigmoidf(z);
      } else {
        float z = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) z = z + s_sig[nn][w * 32 + jj];
        sig_out[m] = relu(z + reinterpret_cast<const float*>(pk + P.p_head_sigma)[2 * C::KH]);
      }
    }
  }
}

template <int W, int D, int SKIP, int LX, int LD>
void launch_fwd_f32s(const MlpPlan& P, const void* packed, int64_t M, const float* xyz, const float* dirs,
                     const float* ro, const float* rd, const float* tv, int spr, float* rgb, float* sigma,
                     void* stash, hipStream_t s) {
  auto go = [&](auto Nc, auto St) {
    constexpr int N = decltype(Nc)::value;
    mlp_fwd_f32s_kernel<W, D, SKIP, LX, LD, N, decltype(St)::value>
        <<<(unsigned)((M + 32 * N - 1) / (32 * N)), 64 * split3::kWaves, 0, s>>>(
            P, reinterpret_cast<const char*>(packed), M, xyz, dirs, ro, rd, tv, spr, rgb, sigma,
            reinterpret_cast<float*>(stash));
  };
  const bool small = M <= (int64_t)32 * nerf_num_cus();  // (figures at the top)
  if (stash) {
    if (small) go(std::integral_constant<int, 1>{}, std::true_type{});
    else go(std::integral_constant<int, 2>{}, std::true_type{});
  } else {
    if (small) go(std::integral_constant<int, 1>{}, std::false_type{});
    else go(std::integral_constant<int, 2>{}, std::false_type{});
  }
}
