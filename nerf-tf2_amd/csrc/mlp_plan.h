// Layout plan of the fused NeRF MLP: the flat "Keras" parameter layout, the
// packed MFMA operand layout, the training stash and the per-sample gradients.
//
// Register layout (v_mfma_f32_32x32x{2f32,16_bf16}): one wave owns 32 samples.
// Lane l = j + 32 g (j = sample in the block, g = lane half).  An MFMA output
// block nb (32 features) holds in accumulator i of lane l the feature
//   F(nb, i, g) = 32 nb + 8 (i/4) + 4 g + (i%4)
// of sample j.  Those accumulators are fed back as the B operand of the next
// layer without any transpose: fp32 k-step s = 16 nb + i uses F(nb, i, g) on
// lane half g; bf16 k-step t uses slots r = 0..7 of F(t/2, 8 (t%2) + r, g).
// The packed A operand (weights) is permuted to match, so the k order of each
// dot product is the only thing that differs from a plain matmul.
//
// Positional-encoding features are produced directly in lane slots: half g
// holds slots e = 0..H-1 (H = 2 + 3L).  Half 0: x, y, z, pad, then (sin, cos)
// pairs 0..P0-1; half 1: pairs P0..3L-1 (P0 = (3L-2)/2).  Pair p encodes
// component c = p / L at frequency l = p % L, i.e. reference features
// 3 + c 2L + 2l + {0: sin, 1: cos} (model.py:323-330).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define NERF_MAX_LAYERS 16

__host__ __device__ inline int ru(int x, int m) { return (x + m - 1) / m * m; }

// Reference feature index of encoding slot e on lane half g, or -1 for a pad slot.
__host__ __device__ inline int enc_feat(int g, int e, int L) {
  const int H = 2 + 3 * L, P0 = (3 * L - 2) / 2;
  if (e < 0 || e >= H) return -1;
  int p, sc;
  if (g == 0) {
    if (e < 3) return e;
    if (e == 3) return -1;
    p = (e - 4) / 2;
    sc = (e - 4) % 2;
  } else {
    p = P0 + e / 2;
    sc = e % 2;
  }
  const int c = p / L, l = p % L;
  return 3 + c * 2 * L + 2 * l + sc;
}

// Hidden feature held by accumulator i of output block nb on lane half g.
__host__ __device__ inline int cfeat(int nb, int i, int g) { return 32 * nb + 8 * (i / 4) + 4 * g + (i % 4); }

struct MlpPlan {
  int D, W, skip, LX, LD, rgb;
  int NB, NBR, WR;      // hidden blocks, rgb-branch blocks, rgb-branch width
  int HX, HD;           // encoding slots per lane half
  int KX, KD;           // encoding slots per half padded to 8 (= fp32 k-steps)
  int KX16, KD16;       // bf16 k-steps for the encodings
  int FX, FD;           // encoding widths (3 + 6L)
  int n_keras;          // Keras layers in trainable-variable order
  int kl_sigma, kl_bott, kl_rbr, kl_rgb;  // their Keras indices (-1: absent)
  int fan_in[NERF_MAX_LAYERS], fan_out[NERF_MAX_LAYERS];
  int64_t k_off[NERF_MAX_LAYERS], b_off[NERF_MAX_LAYERS];
  int64_t n_params;
  // MFMA layers: m = 0..D-1 trunk, D bottleneck, D+1 rgb branch (index into arrays below)
  int n_mfma;
  int keras_of[NERF_MAX_LAYERS];   // Keras layer index of MFMA layer m
  int ks_hid[NERF_MAX_LAYERS];     // fp32 k-steps read from the hidden input (0 for m = 0)
  int ks_enc[NERF_MAX_LAYERS];     // fp32 k-steps from an encoding (KX / KD / 0)
  int enc_L[NERF_MAX_LAYERS];      // L of that encoding
  int nb_out[NERF_MAX_LAYERS];     // output blocks
  int relu[NERF_MAX_LAYERS];
  // packed byte offsets
  int64_t p_fwd[NERF_MAX_LAYERS], p_bwd[NERF_MAX_LAYERS], p_bias[NERF_MAX_LAYERS];
  int64_t p_head_sigma, p_head_rgb, packed_bytes;
  // fp32, the reference topology only (-1 otherwise): A operands of the forward on the
  // BF16 matrix cores, each weight in three bf16 planes (mlp_split3.h).  Per layer
  // units [output block of 32][k-step of 16][plane][lane][8], the k-steps and their
  // order as in the bf16 form; the layers follow each other without gaps (fs_bytes
  // from p_fs[0] on)
  int64_t p_fs[NERF_MAX_LAYERS], fs_bytes;
  // the same for the dX chain, layers m >= 1: A[n = input hidden feature][k = output
  // feature], units [input block of 32][k-step of 16], bs_bytes from p_bs[1] on
  int64_t p_bs[NERF_MAX_LAYERS], bs_bytes;
  int prec;
  // stash (elements per sample; fp32 or bf16 elements) and dz (floats per sample)
  int64_t st_encx, st_h[NERF_MAX_LAYERS], st_bott, st_rbr, st_encd, stash_per_sample;
  // ReLU bit masks (W = 256 with an rgb branch; -1 otherwise), written by the
  // forward for the dX chain: per 32-feature block nb and lane half g, D uint16
  // words, one per trunk layer (word (2 nb + g) D + l, bit i = accumulator i; in
  // bf16 the bit order of ws::nz_bits), then 8 words for the rgb branch (word 16 D +
  // 2 nb + g).  16 D + 8 elements of the bf16 stash, half as many of the fp32 one.
  int64_t st_mask;
  int64_t dz_h[NERF_MAX_LAYERS], dz_bott, dz_rbr, dz_sigma, dz_rgb, dz_per_sample;
  // Samples per block of the stash and dz buffers.  A buffer of M samples with S
  // elements per sample is cut into blocks of sblk consecutive samples (the last
  // one may hold fewer); a block [b, b + n) stores its rows chunk-major: the
  // 8-element chunk c of sample m at element b S + 8 (c n + m - b).  sblk = 1 is
  // the plain row-major layout (fp32); 32 (one MFMA sample block) for bf16, whose
  // row chunks of 32 consecutive samples are then 512 contiguous bytes.
  int sblk;
};

// Element offset, in a blocked stash or dz buffer (MlpPlan::sblk = B, S elements
// per sample, M samples), of element e of sample m.
__host__ __device__ inline int64_t blk_elem(int64_t m, int64_t e, int64_t S, int B, int64_t M) {
  const int64_t b = m - m % B;
  const int64_t n = M - b < B ? M - b : B;
  return b * S + 8 * ((e >> 3) * n + (m - b)) + (e & 7);
}

// Returns 0 on success, -1 if the description is not supported.
inline int mlp_make_plan(int D, int W, int skip, int LX, int LD, int prec, MlpPlan* p) {
  // skip < D-1: the sigma head and the bottleneck read the last trunk layer only
  if (D < 2 || D > 10 || W < 32 || W > 256 || (W % 32) || skip < -1 || skip >= D - 1 || LX < 2 ||
      (LX % 2) || LX > 16 || LD < 0 || (LD % 2) || LD > 16 || (prec != 0 && prec != 1))
    return -1;
  MlpPlan& P = *p;
  P = MlpPlan{};
  P.D = D; P.W = W; P.skip = skip; P.LX = LX; P.LD = LD; P.rgb = LD > 0; P.prec = prec;
  // every bf16 stash and dz is blocked (the kernels' launchers check it)
  P.sblk = prec == 1 ? 32 : 1;
  P.NB = W / 32;
  P.WR = W / 2;
  P.NBR = (P.WR + 31) / 32;
  P.HX = 2 + 3 * LX;
  P.HD = LD ? 2 + 3 * LD : 0;
  P.KX = ru(P.HX, 8);
  P.KD = LD ? ru(P.HD, 8) : 0;
  P.KX16 = P.KX / 8;
  P.KD16 = P.KD / 8;
  P.FX = 3 + 6 * LX;
  P.FD = LD ? 3 + 6 * LD : 0;
  // Keras layers in trainable-variable order.  A functional model lists its
  // layers by decreasing depth from the outputs, ties in the order a depth-first
  // walk from the outputs [rgb, sigma] first meets them (model.py:389-392).  The
  // last trunk layer feeds the bottleneck (depth 3 below rgb), so it sits at
  // depth 4; sigma and rgb are both outputs (depth 0) and the walk meets rgb
  // first: dense_0 .. dense_{D-1}, dense_D, dense_{D+1}, rgb, sigma.  A
  // density-only net is dense_0 .. dense_{D-1}, sigma.
  int n = 0;
  const int trunk_out_in = W + (skip == D - 1 ? P.FX : 0);
  for (int i = 0; i < D; ++i) {
    P.fan_in[n] = i == 0 ? P.FX : W + (i - 1 == skip ? P.FX : 0);
    P.fan_out[n] = W;
    ++n;
  }
  P.kl_bott = P.kl_rbr = P.kl_rgb = -1;
  if (P.rgb) {
    P.kl_bott = n; P.fan_in[n] = trunk_out_in; P.fan_out[n] = W; ++n;   // dense_D (bottleneck)
    P.kl_rbr = n; P.fan_in[n] = W + P.FD; P.fan_out[n] = P.WR; ++n;     // dense_{D+1}
    P.kl_rgb = n; P.fan_in[n] = P.WR; P.fan_out[n] = 3; ++n;            // rgb
  }
  P.kl_sigma = n; P.fan_in[n] = trunk_out_in; P.fan_out[n] = 1; ++n;  // sigma
  P.n_keras = n;
  int64_t off = 0;
  for (int i = 0; i < n; ++i) {
    P.k_off[i] = off;
    off += (int64_t)P.fan_in[i] * P.fan_out[i];
    P.b_off[i] = off;
    off += P.fan_out[i];
  }
  P.n_params = off;
  // MFMA layers
  int m = 0;
  for (int i = 0; i < D; ++i) {
    P.keras_of[m] = i;
    P.ks_hid[m] = i == 0 ? 0 : W / 2;
    P.ks_enc[m] = i == 0 ? P.KX : (i - 1 == skip ? P.KX : 0);
    P.enc_L[m] = LX;
    P.nb_out[m] = P.NB;
    P.relu[m] = 1;
    ++m;
  }
  if (P.rgb) {
    P.keras_of[m] = P.kl_bott;
    P.ks_hid[m] = W / 2;
    P.ks_enc[m] = skip == D - 1 ? P.KX : 0;
    P.enc_L[m] = LX;
    P.nb_out[m] = P.NB;
    P.relu[m] = 0;
    ++m;
    P.keras_of[m] = P.kl_rbr;
    P.ks_hid[m] = W / 2;
    P.ks_enc[m] = P.KD;
    P.enc_L[m] = LD;
    P.nb_out[m] = P.NBR;
    P.relu[m] = 1;
    ++m;
  }
  P.n_mfma = m;
  // packed layout (p_fwd, p_bwd: not for the split form, whose kernels read p_fs and p_bs).  The
  // split form is that of the one topology with kernels for it: other descriptions of the same
  // width have other numbers of inputs (l_xyz or l_dir from 12 on more than its packing holds)
  // and are packed as any other net.
  const bool split = prec == 0 && D == 8 && W == 256 && skip == 4 && LX == 10 && LD == 4;
  int64_t b = 0;
  auto align = [&](int64_t a) { b = (b + a - 1) / a * a; };
  for (int i = 0; i < P.n_mfma; ++i) {
    P.p_fwd[i] = -1;
    if (split) continue;
    align(256);
    P.p_fwd[i] = b;
    if (prec == 0)
      b += (int64_t)(P.ks_hid[i] + P.ks_enc[i]) * P.nb_out[i] * 64 * 4;
    else {
      const int ke16 = P.ks_enc[i] == 0 ? 0 : (P.enc_L[i] == LX ? P.KX16 : P.KD16);
      b += (int64_t)(P.ks_hid[i] / 8 + ke16) * P.nb_out[i] * 64 * 16;
    }
  }
  for (int i = 0; i < P.n_mfma; ++i) {
    P.p_bwd[i] = -1;
    if (i == 0 || split) continue;  // no dX for the encoding input
    align(256);
    P.p_bwd[i] = b;
    // A[n = input hidden feature][k = output feature]: k-steps over the outputs
    const int out_ks = P.nb_out[i] * 16;  // fp32 k-steps over 32*nb_out outputs
    if (prec == 0)
      b += (int64_t)out_ks * P.NB * 64 * 4;
    else
      b += (int64_t)(out_ks / 8) * P.NB * 64 * 16;
  }
  for (int i = 0; i < P.n_mfma; ++i) {
    align(256);
    P.p_bias[i] = b;
    b += (int64_t)P.nb_out[i] * 32 * 4;
  }
  align(256);
  P.p_head_sigma = b;  // [2][W/2] fp32 + bias (padded to 4)
  b += (int64_t)2 * (W / 2) * 4 + 16;
  align(256);
  P.p_head_rgb = b;  // [2][16*NBR][4] fp32 + bias[4]
  if (P.rgb) b += (int64_t)2 * 16 * P.NBR * 16 + 16;
  align(4096);
  const int64_t fs0 = b;
  for (int i = 0; i < P.n_mfma; ++i) {
    P.p_fs[i] = split ? b : -1;
    if (split) b += (int64_t)((P.ks_hid[i] + P.ks_enc[i]) / 8) * P.nb_out[i] * 3 * 1024;
  }
  P.fs_bytes = b - fs0;
  align(4096);
  const int64_t bs0 = b;
  for (int i = 0; i < P.n_mfma; ++i) {
    P.p_bs[i] = split && i > 0 ? b : -1;
    if (split && i > 0) b += (int64_t)P.nb_out[i] * 2 * P.NB * 3 * 1024;
  }
  P.bs_bytes = b - bs0;
  align(256);
  P.packed_bytes = b;
  // stash (elements per sample)
  int64_t s = 0;
  P.st_encx = s; s += 2 * P.KX;
  for (int i = 0; i < D; ++i) { P.st_h[i] = s; s += W; }
  P.st_bott = P.st_rbr = P.st_encd = -1;
  if (P.rgb) {
    P.st_bott = s; s += W;
    P.st_rbr = s; s += 32 * P.NBR;
    P.st_encd = s; s += 2 * P.KD;
  }
  s = ru((int)s, 8);
  P.st_mask = -1;
  if (W == 256 && P.rgb && P.NBR == 4) {
    P.st_mask = s;
    s += 16 * D + 8;
  }
  // rows padded to 64 elements: every stash row, and each 64-feature segment a
  // wave writes, starts on a 128-byte line (bf16), so the forward writes whole lines
  P.stash_per_sample = ru((int)s, 64);
  // dz (elements per sample: float32 for the fp32 form, bf16 for the bf16 form);
  // every segment starts on a multiple of 8 elements (16-byte aligned bf16 loads)
  int64_t z = 0;
  for (int i = 0; i < D; ++i) { P.dz_h[i] = z; z += W; }
  P.dz_bott = P.dz_rbr = P.dz_rgb = -1;
  if (P.rgb) {
    P.dz_bott = z; z += W;
    P.dz_rbr = z; z += 32 * P.NBR;
  }
  P.dz_sigma = z; z += 8;
  if (P.rgb) { P.dz_rgb = z; z += 8; }
  P.dz_per_sample = ru((int)z, 64);  // 128-byte rows (bf16), as the stash
  return 0;
}
