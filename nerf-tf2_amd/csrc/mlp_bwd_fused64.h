// BF16 backward of the density-only net with 64-wide layers (the proposal network) in
// one kernel: the dX chain and every layer's weight gradient, from the stash alone.
//
// As a chain kernel and weight GEMMs the backward wrote dz (576 B per sample) and read
// it and the stash (640 B) again, in five launches of which the GEMMs' tiles are too
// small to fill the chip: memory and launches, not arithmetic, took the time.  Here a
// workgroup of eight waves walks over 256 samples at a time, 32 to a wave.  A wave loads
// a layer's activations once, as 16-byte row chunks; turns them to the accumulator
// layout for the ReLU mask; and keeps its dz in registers, where an MFMA's accumulators
// are the next one's B operand (the weights' order is packed for that).  For the
// gradients, which sum over samples, both go through LDS transposed, as [feature][sample]
// rows of sample pairs (the 16-byte units of row f at u ^ f: no bank conflicts on either
// side), double-buffered, one barrier a layer; wave w then owns block (w / 2 % 2, w % 2)
// of the 64 x 64 gradient over half of the samples (w / 4), 16 accumulators per layer,
// kept over all of the workgroup's samples.  At the end the halves are added and each
// workgroup writes one partial tile per layer (67 KB); wgrad_reduce_batch_kernel sums
// those.  One workgroup a CU (153 KB of LDS, two waves a SIMD).
//
// dz is bit for bit that of mlp_bwd_bf16_kernel; the sums over samples differ in order.
// 196,608 samples: 46 us of chain and 54 us of GEMMs and sums before, now 39 us here
// (3.2 TB/s of stash) and 9 us of sums; a forward and backward pass 142 -> 96 us, of
// which the host's part is 90; a training step of the learned form 4.11 -> 4.05 ms.
#pragma once
#include "mlp_bwd_bf16ws.h"

namespace fb64 {

constexpr int kD = 4, kTiles = 5;        // trunk layers; tiles h3, h2, h1, h0, encoding
constexpr int kSamples = 256;            // per chunk: 32 for each of eight waves
constexpr int kRow = 2 * kSamples;       // bytes of a transposed row
constexpr int kTile = 64 * kRow;         // bytes of a transposed tile
constexpr int kMaxGroups = 256;          // one workgroup per CU

struct Args {
  const char* pk;                        // packed operands
  int64_t p_bwd[kD], p_sigma;            // their offsets (p_bwd[0] is not read)
  int64_t M, ld;                         // samples; stash elements per sample
  int chunk0[kTiles];                    // first 8-element chunk of each tile in a stash row
  const __bf16* stash;
  const float *d_sigma, *sigma;
  float* part[kD + 1];                   // partial tiles [group][64 x 64] of dense_0 .. 3, [group][64] of sigma
  float* bpart[kD + 1];                  // their bias sums [group][64], [group][1]
};

// Halves with 0 < h <= infinity (as `h > 0`: a NaN counts as not positive) as 0xFFFF,
// others 0: the sign of min(h - 1, 0x7F80) - 0x7F80, in packed 16-bit steps.
__device__ __forceinline__ uint32_t positive_mask(uint32_t h) {
  typedef short shortx2 __attribute__((ext_vector_type(2)));
  const ws::ushortx2 one = {1, 1}, lim = {0x7F80, 0x7F80};
  ws::ushortx2 t = __builtin_elementwise_min((ws::ushortx2)(__builtin_bit_cast(ws::ushortx2, h) - one), lim);
  uint32_t m = __builtin_bit_cast(uint32_t, (ws::ushortx2)(t - lim));
  asm volatile("" : "+v"(m));  // (or it becomes a compare and a select for each half)
  return __builtin_bit_cast(uint32_t, (shortx2)(__builtin_bit_cast(shortx2, m) >> 15));
}

__device__ __forceinline__ float sum8(bf16x8 v) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) s += (float)v[i];
  return s;
}

__global__ __launch_bounds__(512, 2) void mlp_bwd_fused64_kernel(Args a) {
  using ws::u32x4;
  __shared__ __align__(1024) char s_buf[4 * kTile];  // X, Z of the even stages, X, Z of the odd ones
  __shared__ bf16x8 s_w[(kD - 1) * 8 * 64];          // transposed weights of layers 1 .. 3, 24 KB
  __shared__ __align__(16) __bf16 s_dzs[kSamples];
  __shared__ floatx4 s_sig[16];                      // the sigma head's weights, by lane half
  const int lane = threadIdx.x & 63, j = lane & 31, g = lane >> 5, odd = j & 1;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int xb = (wv >> 1) & 1, zb = wv & 1, kh = wv >> 2;
#pragma unroll
  for (int l = 1; l < kD; ++l)
    s_w[(l - 1) * 512 + threadIdx.x] = reinterpret_cast<const bf16x8*>(a.pk + a.p_bwd[l])[threadIdx.x];

  if (threadIdx.x < 16) s_sig[threadIdx.x] = reinterpret_cast<const floatx4*>(a.pk + a.p_sigma)[threadIdx.x];
  __syncthreads();

  // byte offsets of this lane's stores into a transposed tile: feature 16 q + i + 8 g + 4 odd,
  // sample pair 16 wv + j / 2; the (q, i) part of the row is an immediate
  uint32_t st_off[2][4];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t f = 8u * g + 4u * odd, unit = 4u * wv + (j >> 3);
      st_off[q][i] = f * kRow + ((unit ^ (f + 16u * q + i)) << 4) + 4u * ((j >> 1) & 3);
    }
  auto store_t = [&](char* tile, const u32x4& v, int q) {
    const auto r = pair_rows<true>(__builtin_bit_cast(u32x4_, v), odd);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<uint32_t*>(tile + st_off[q & 1][i] + (16 * q + i) * kRow) = r[i];
    __builtin_amdgcn_sched_barrier(0);  // (a stage's conversions all at once would spill)
  };
  // operand of k-step t (16 samples) of feature 32 b + j: at (this ^ (t << 5)) of the tile
  uint32_t ld_off = (uint32_t)(j * kRow + ((g ^ j) << 4));
  auto operand = [&](const char* tile, int b, int t) {
    return *reinterpret_cast<const bf16x8*>(tile + b * (32 * kRow) + (ld_off ^ (uint32_t)(t << 5)));
  };

  const int64_t nchunk = (a.M + kSamples - 1) / kSamples;
  // tile k of this wave's 32 samples of chunk c as row chunks: chunk 2 q + g of the tile's
  // eight; through a buffer resource over the chunk's samples, zeros past M
  auto load_tile = [&](u32x4 (&v)[4], int64_t c, int k) {
    const int64_t m0 = c * kSamples, left = a.M - m0;
    const int rows = left >= kSamples ? kSamples : (left > 0 ? (int)left : 0);
    const int n = __builtin_amdgcn_readfirstlane(rows < 32 * wv ? 0 : rows - 32 * wv < 32 ? rows - 32 * wv : 32);
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<__bf16*>(a.stash + (rows > 0 ? m0 * a.ld : 0)), 0, (int)(rows * a.ld * 2), 0x00020000);
    const uint32_t off = j < n ? (uint32_t)(64 * wv * a.ld) + 16u * (uint32_t)(g * n + j) : 0x80000000u;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      v[q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 16 * (a.chunk0[k] + 2 * q) * n, 0));
  };
  float sg = 0.f, ds = 0.f;
  auto load_sigma = [&](int64_t c) {
    const int64_t m = c * kSamples + 32 * wv + j;
    sg = m < a.M ? a.sigma[m] : 0.f;
    ds = m < a.M ? a.d_sigma[m] : 0.f;
  };

  floatx16 wacc[kD], sacc;   // dense gradients by layer, the sigma head's column
  float bsum[kD], dsum = 0.f;
  zero_acc(wacc);
#pragma unroll
  for (int i = 0; i < 16; ++i) sacc[i] = 0.f;
#pragma unroll
  for (int l = 0; l < kD; ++l) bsum[l] = 0.f;

  u32x4 x[3][4];             // tiles k, k + 1, k + 2 in slots k % 3, ...: 5 tiles a chunk, so
  int64_t c = blockIdx.x;    // the slots are renamed at its end
  load_tile(x[0], c, 0);
  load_tile(x[1], c, 1);
  load_sigma(c);
  int buf = 0;
  for (; c < nchunk; c += gridDim.x) {
    const float dzs = ds * (1.f - expf(-sg));  // softplus' derivative
    const __bf16 dzb = (__bf16)dzs;
    dsum += g == 0 ? (float)dzb : 0.f;
    floatx16 acc[2];
    {
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const floatx4 w = s_sig[g * 8 + 4 * nb + i];
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[nb][4 * i + r] = 0.f + w[r] * dzs;
        }
    }
    const int64_t cn = c + gridDim.x;
    bf16x8 z[4];             // dz of the stage as B operands (k-step q: features 16 q ..)
    ws::static_for<0, kTiles>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      asm volatile("" : "+v"(ld_off));  // (or its sixteen variants are kept in registers, and spill)
      char* const tx = s_buf + buf * (2 * kTile);
      char* const tz = tx + kTile;
      if constexpr (k > 0) {  // dz of layer 4 - k: rounded, masked by that layer's output (tile k - 1)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const u32x4 h = __builtin_bit_cast(u32x4, ws::swap_halves(__builtin_bit_cast(bf16x8, x[(k - 1) % 3][q])));
          u32x4 d = __builtin_bit_cast(u32x4, acc_to_bf16(acc[q >> 1], q & 1));
#pragma unroll
          for (int i = 0; i < 4; ++i) d[i] &= positive_mask(h[i]);
          z[q] = __builtin_bit_cast(bf16x8, d);
          store_t(tz, __builtin_bit_cast(u32x4, ws::swap_halves(z[q])), q);
        }
      } else {
        if (g == 0) s_dzs[32 * wv + j] = dzb;
      }
      if constexpr (k + 2 < kTiles) load_tile(x[(k + 2) % 3], c, k + 2);
      else load_tile(x[(k + 2) % 3], cn, k + 2 - kTiles);
      if constexpr (k == kTiles - 1) load_sigma(cn);
#pragma unroll
      for (int q = 0; q < 4; ++q) store_t(tx, x[k % 3][q], q);
      __syncthreads();
      if constexpr (k == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // rows 32 (wv % 2) .., k-steps 4 (wv / 2) ..; column 0 is dz of sigma
          const int t = 4 * (wv >> 1) + i;
          u32x4 b = *reinterpret_cast<const u32x4*>(s_dzs + 16 * t + 8 * g);
#pragma unroll
          for (int e = 0; e < 4; ++e) b[e] = j == 0 ? b[e] : 0u;
          sacc = mfma_bf16(operand(tx, wv & 1, t), __builtin_bit_cast(bf16x8, b), sacc);
        }
      } else {
        if constexpr (k < kTiles - 1) {  // acc = W^T dz for the layer below
#pragma unroll
          for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[nb][i] = 0.f;
#pragma unroll
          for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
              acc[nb] = mfma_bf16(s_w[(kD - 1 - k) * 512 + (2 * t + nb) * 64 + lane], z[t], acc[nb]);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int t = 8 * kh + i;
          const bf16x8 zo = operand(tz, zb, t);
          wacc[kD - k] = mfma_bf16(operand(tx, xb, t), zo, wacc[kD - k]);
          if ((i & 1) == xb) bsum[kD - k] += sum8(zo);  // (both xb waves read it: they share the sum)
          if (i & 1) __builtin_amdgcn_sched_barrier(0);
        }
      }
      buf ^= 1;
    });
    // tiles 0 and 1 of the next chunk arrived in slots 2 and 0
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const u32x4 t0 = x[2][q], t1 = x[0][q];
      x[0][q] = t0;
      x[1][q] = t1;
    }
  }

  // ---- the waves' sums: halves of the samples, then this workgroup's partial tiles
  __syncthreads();
  float* const sw = reinterpret_cast<float*>(s_buf);      // [layer][block][16][64], 64 KB
  float* const ssig = sw + kD * 4 * 1024;                 // [wave][32]
  float* const sb = ssig + 8 * 32;                        // [layer][wave][64]
  float* const sd = sb + kD * 8 * 64;                     // [wave]
  dsum = wave_sum(dsum);
  if (lane == 0) sd[wv] = dsum;
#pragma unroll
  for (int l = 0; l < kD; ++l) {
    sb[(l * 8 + wv) * 64 + lane] = bsum[l];
    if (kh == 1) {
#pragma unroll
      for (int i = 0; i < 16; ++i) sw[((l * 4 + (wv & 3)) * 16 + i) * 64 + lane] = wacc[l][i];
    }
  }
  if (j == 0) {
#pragma unroll
    for (int i = 0; i < 16; ++i) ssig[wv * 32 + 8 * (i >> 2) + 4 * g + (i & 3)] = sacc[i];
  }
  __syncthreads();
  const int64_t grp = blockIdx.x;
  if (kh == 0) {
#pragma unroll
    for (int l = 0; l < kD; ++l)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float v = wacc[l][i] + sw[((l * 4 + wv) * 16 + i) * 64 + lane];
        a.part[l][grp * 4096 + (32 * xb + 8 * (i >> 2) + 4 * g + (i & 3)) * 64 + 32 * zb + j] = v;
      }
  } else {
    const int e = threadIdx.x - 256, l = e >> 6, n = e & 63;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w)  // waves zb + 2 w
      for (int h = 0; h < 2; ++h) v += sb[(l * 8 + (n >> 5) + 2 * w) * 64 + 32 * h + (n & 31)];
    a.bpart[l][grp * 64 + n] = v;
    if (e < 64) {  // sigma head: row e, waves e / 32 + 2 w
      float s = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) s += ssig[((e >> 5) + 2 * w) * 32 + (e & 31)];
      a.part[kD][grp * 64 + e] = s;
      if (e == 0) {
        float b = 0.f;
#pragma unroll
        for (int w = 0; w < 8; ++w) b += sd[w];
        a.bpart[kD][grp] = b;
      }
    }
  }
}

// Workgroups of a call.
inline int64_t groups(int64_t M) {
  const int64_t n = (M + kSamples - 1) / kSamples;
  return n < kMaxGroups ? n : kMaxGroups;
}
constexpr int64_t kGroupFloats = kD * (4096 + 64) + 64 + 1;

inline bool takes(const MlpPlan& P) {
  return P.prec == NERF_PREC_BF16 && P.W == 64 && P.D == kD && P.skip < 0 && !P.rgb && P.KX == 32 && P.sblk == 32;
}

}  // namespace fb64
