// Packing of the flat "Keras" MLP parameters into the MFMA operand layout,
// and the size queries of the MLP entry points.
#include "common.h"
#include "mlp_plan.h"
#include "mlp_split3.h"
#include "optim.h"

namespace {

typedef float floatx4_a4 __attribute__((ext_vector_type(4), aligned(4)));  // the caller's weights: any float alignment

// Input row (of the Keras kernel) fed by fp32 k-step s on lane half g of MFMA layer m.
__device__ int fwd_row_f32(const MlpPlan& P, int m, int s, int g) {
  const int kh = P.ks_hid[m];
  if (s < kh) return cfeat(s / 16, s % 16, g);
  const int e = s - kh;
  const int ef = enc_feat(g, e, P.enc_L[m]);
  if (ef < 0) return -1;
  return (m == 0 ? 0 : P.W) + ef;
}

// Same for bf16 k-step t, slot r (0..7).
__device__ int fwd_row_bf16(const MlpPlan& P, int m, int t, int r, int g) {
  const int th = P.ks_hid[m] / 8;
  if (t < th) return cfeat(t / 2, 8 * (t % 2) + r, g);
  const int e = 8 * (t - th) + r;
  const int ef = enc_feat(g, e, P.enc_L[m]);
  if (ef < 0) return -1;
  return (m == 0 ? 0 : P.W) + ef;
}

__device__ float kernel_at(const MlpPlan& P, const float* flat, int kl, int row, int col) {
  if (row < 0 || row >= P.fan_in[kl] || col < 0 || col >= P.fan_out[kl]) return 0.f;
  return flat[P.k_off[kl] + (int64_t)row * P.fan_out[kl] + col];
}

// One launch packs everything: a list of segments, each a run of workgroups.
struct PackModels {
  const float* flat[kOptModels];
  char* packed[kOptModels];
};
enum PackKind : int { kFwd, kBwd, kBias, kHeads };
constexpr int kMaxSegs = 3 * NERF_MAX_LAYERS + 1;
struct PackSegs {
  int n;
  int first[kMaxSegs + 1];  // first workgroup of each segment; [n]: their number
  unsigned char kind[kMaxSegs], layer[kMaxSegs];
};

// This lane's slots of unit w of a layer's split operands.
__device__ __forceinline__ void put_split(const float (&f)[8], char* to, int w, int lane) {
  bf16x8* o = reinterpret_cast<bf16x8*>(to) + w * split3::kStep + lane;
  const split3::Planes p = split3::split8(f);
  o[0] = p.h;
  o[64] = p.m;
  o[128] = p.l;
}

// Forward A operands of MFMA layer m: a wave writes unit w = (k-step or k-step group,
// output block; the split form: output block, k-step), 16 bytes per lane and plane.  The
// unit's number is wave-uniform and a hidden k-step's rows are two runs of four, so that what
// each lane computes is little more than eight addresses (the divisions by block and model
// sizes per thread were most of this kernel: 10.7 -> 7.9 us for the two BF16 8x256 models).
__device__ void pack_fwd(const MlpPlan& P, const float* __restrict__ flat, char* __restrict__ out, int m, int w) {
  const int kl = P.keras_of[m], NBo = P.nb_out[m], T = (P.ks_hid[m] + P.ks_enc[m]) / 8;
  const bool split = P.p_fs[m] >= 0;
  const int lane = threadIdx.x & 63, j = lane & 31, g = lane >> 5;
  const int nb = split ? w / T : w % NBo, t = split ? w % T : w / NBo;
  const int col = 32 * nb + j, FO = P.fan_out[kl];
  const float* k = flat + P.k_off[kl] + col;
  const bool in = col < FO;
  if (P.prec == 0 && !split) {
    if (t >= 2 * T) return;
    floatx4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = kernel_at(P, flat, kl, fwd_row_f32(P, m, 4 * t + r, g), col);
    reinterpret_cast<floatx4*>(out + P.p_fwd[m])[w * 64 + lane] = v;
  } else {
    const int th = P.ks_hid[m] / 8;
    if (nb >= NBo || t >= T) return;
    float f[8];
    if (t < th) {  // cfeat(t / 2, 8 (t % 2) + r, g)
      const float* q = k + (int64_t)(16 * t + 4 * g) * FO;
#pragma unroll
      for (int r = 0; r < 8; ++r) f[r] = in ? q[(r < 4 ? r : r + 4) * FO] : 0.f;
    } else {
#pragma unroll
      for (int r = 0; r < 8; ++r) f[r] = kernel_at(P, flat, kl, fwd_row_bf16(P, m, t, r, g), col);
    }
    if (split) return put_split(f, out + P.p_fs[m], w, lane);
    ushortx8 v;
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r] = f2bf(f[r]);
    reinterpret_cast<ushortx8*>(out + P.p_fwd[m])[w * 64 + lane] = v;
  }
}

// Backward (transposed) A operands: A[n = input hidden feature 32 nb + j][k = output feature],
// a unit per wave as above; a lane's outputs are one or two runs of four consecutive weights.
__device__ void pack_bwd(const MlpPlan& P, const float* __restrict__ flat, char* __restrict__ out, int m, int w) {
  const int kl = P.keras_of[m], lane = threadIdx.x & 63, j = lane & 31, g = lane >> 5, T = 2 * P.nb_out[m];
  const bool split = P.p_bs[m] >= 0;
  const int nb = split ? w / T : w % P.NB, t = split ? w % T : w / P.NB;
  const int FO = P.fan_out[kl];
  const float* k = flat + P.k_off[kl] + (int64_t)(32 * nb + j) * FO;
  auto run = [&](int c) -> floatx4 {  // (FO is a multiple of 4: a run is inside or outside)
    return c < FO ? (floatx4)*reinterpret_cast<const floatx4_a4*>(k + c) : floatx4{0.f, 0.f, 0.f, 0.f};
  };
  if (P.prec == 0 && !split) {
    if (t >= 2 * T) return;
    reinterpret_cast<floatx4*>(out + P.p_bwd[m])[w * 64 + lane] = run(cfeat(t / 4, 4 * (t % 4), g));
  } else {
    if (nb >= P.NB || t >= T) return;
    const floatx4 lo = run(16 * t + 4 * g), hi = run(16 * t + 4 * g + 8);  // cfeat(t / 2, 8 (t % 2) + r, g)
    if (split) return put_split({lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, out + P.p_bs[m], w, lane);
    ushortx8 v;
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r] = f2bf(r < 4 ? lo[r & 3] : hi[r & 3]);
    reinterpret_cast<ushortx8*>(out + P.p_bwd[m])[w * 64 + lane] = v;
  }
}

__device__ void pack_heads(const MlpPlan& P, const float* __restrict__ flat, char* __restrict__ out) {
  float* hs = reinterpret_cast<float*>(out + P.p_head_sigma);
  const int KH = P.W / 2, KS = 16 * P.NBR;
  for (int e = threadIdx.x; e < 2 * KH + 4; e += 256) {
    const int g = e / KH, s = e % KH;
    hs[e] = e < 2 * KH ? kernel_at(P, flat, P.kl_sigma, cfeat(s / 16, s % 16, g), 0)
                       : (e == 2 * KH ? flat[P.b_off[P.kl_sigma]] : 0.f);
  }
  if (!P.rgb) return;
  float* hr = reinterpret_cast<float*>(out + P.p_head_rgb);
  for (int e = threadIdx.x; e < 2 * KS * 4 + 4; e += 256) {
    const int c = e % 4, s = (e / 4) % KS, g = e / (4 * KS);
    if (e < 2 * KS * 4)
      hr[e] = c < 3 ? kernel_at(P, flat, P.kl_rgb, cfeat(s / 16, s % 16, g), c) : 0.f;
    else
      hr[e] = c < 3 ? flat[P.b_off[P.kl_rgb] + c] : 0.f;
  }
}

// blockIdx.y: the model (all of one plan).  The first thread of the last launch of an optimizer
// step also closes the step (state; null otherwise).
__global__ __launch_bounds__(256) void pack_kernel(MlpPlan P, PackSegs S, PackModels A, StepState* state,
                                                   StepEnd end) {
  const float* __restrict__ flat = A.flat[blockIdx.y];
  char* __restrict__ out = A.packed[blockIdx.y];
  if (state && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) step_end(state, end);
  int seg = 0;
  while (seg + 1 < S.n && (int)blockIdx.x >= S.first[seg + 1]) ++seg;
  const int blk = blockIdx.x - S.first[seg], m = S.layer[seg], u = 256 * blk + threadIdx.x;
  const int unit = 4 * blk + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  switch (S.kind[seg]) {
    case kFwd: return pack_fwd(P, flat, out, m, unit);
    case kBwd: return pack_bwd(P, flat, out, m, unit);
    case kBias: {
      const int kl = P.keras_of[m];
      if (u < 32 * P.nb_out[m])
        reinterpret_cast<float*>(out + P.p_bias[m])[u] = u < P.fan_out[kl] ? flat[P.b_off[kl] + u] : 0.f;
      return;
    }
    case kHeads: return pack_heads(P, flat, out);
  }
}

// The segments of a plan, the longest-running first.
PackSegs pack_segs(const MlpPlan& P) {
  PackSegs S{};
  auto add = [&](PackKind k, int m, int64_t blocks) {
    S.kind[S.n] = (unsigned char)k;
    S.layer[S.n] = (unsigned char)m;
    S.first[S.n + 1] = S.first[S.n] + (int)blocks;
    ++S.n;
  };
  auto blocks16 = [](int64_t bytes) { return (bytes + 4095) / 4096; };  // 16 bytes per thread
  for (int m = 0; m < P.n_mfma; ++m) {
    const int T = (P.ks_hid[m] + P.ks_enc[m]) / 8;
    add(kFwd, m, blocks16((int64_t)P.nb_out[m] * 64 * 16 * (P.p_fwd[m] >= 0 && P.prec == 0 ? 2 * T : T)));
    if (m > 0) add(kBwd, m, blocks16((int64_t)P.nb_out[m] * (P.p_bwd[m] >= 0 && P.prec == 0 ? 4 : 2) * P.NB * 64 * 16));
  }
  for (int m = 0; m < P.n_mfma; ++m) add(kBias, m, (32 * P.nb_out[m] + 255) / 256);
  add(kHeads, 0, 1);
  return S;
}

}  // namespace

// Packs n <= kOptModels models of one plan in one launch; state: also close the step.
void pack_models(const MlpPlan& P, int n, const float* const* flat, void* const* packed, StepState* state,
                 const StepEnd& end, hipStream_t s) {
  const PackSegs S = pack_segs(P);
  PackModels A{};
  for (int i = 0; i < n; ++i) {
    A.flat[i] = flat[i];
    A.packed[i] = reinterpret_cast<char*>(packed[i]);
  }
  pack_kernel<<<dim3((unsigned)S.first[S.n], (unsigned)n), 256, 0, s>>>(P, S, A, state, end);
}

int nerf_plan_from_desc(const nerf_mlp_desc* d, int prec, MlpPlan* p) {
  if (!d) return -1;
  return mlp_make_plan(d->depth, d->width, d->skip, d->l_xyz, d->l_dir, prec, p);
}

#define NERF_PLAN_OR_FAIL(desc, prec, P, name)                                                 \
  MlpPlan P;                                                                                   \
  NERF_CHECK_ARG(nerf_plan_from_desc(desc, prec, &P) == 0,                                     \
                 "%s: unsupported MLP description or precision", name)

extern "C" int64_t nerf_mlp_param_count(const nerf_mlp_desc* desc) {
  MlpPlan P;
  if (nerf_plan_from_desc(desc, 0, &P)) return -1;
  return P.n_params;
}
extern "C" int64_t nerf_mlp_packed_bytes(const nerf_mlp_desc* desc, int32_t precision) {
  MlpPlan P;
  if (nerf_plan_from_desc(desc, precision, &P)) return -1;
  return P.packed_bytes;
}
extern "C" int64_t nerf_mlp_stash_floats_per_sample(const nerf_mlp_desc* desc) {
  MlpPlan P;
  if (nerf_plan_from_desc(desc, 0, &P)) return -1;
  return P.stash_per_sample;
}
extern "C" int64_t nerf_mlp_dz_floats_per_sample(const nerf_mlp_desc* desc) {
  MlpPlan P;
  if (nerf_plan_from_desc(desc, 0, &P)) return -1;
  return P.dz_per_sample;
}
extern "C" int32_t nerf_mlp_sample_block(const nerf_mlp_desc* desc, int32_t precision) {
  MlpPlan P;
  if (nerf_plan_from_desc(desc, precision, &P)) return -1;
  return P.sblk;
}

extern "C" int32_t nerf_mlp_pack(const nerf_mlp_desc* desc, int32_t precision, const float* flat,
                                 void* packed, void* stream) {
  NERF_PLAN_OR_FAIL(desc, precision, P, "nerf_mlp_pack");
  NERF_CHECK_ARG(flat && packed, "nerf_mlp_pack: null pointer");
  pack_models(P, 1, &flat, &packed, nullptr, StepEnd{}, as_stream(stream));
  NERF_LAUNCH_CHECK("nerf_mlp_pack");
  return NERF_OK;
}

// Compute units of the current device (cached per device).
int nerf_num_cus() {
  static int cache[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cache[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cache[dev] = n;
  }
  return cache[dev];
}
