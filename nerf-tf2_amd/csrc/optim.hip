// Loss gradient, Adam (TF ApplyAdam form) and the finite check of the loss scaler.
//   MeanSquaredError        nerf/core/model.py:32, 157-168
//   Adam + ExponentialDecay nerf/core/model.py:413-418
#include <string.h>

#include "common.h"
#include "optim.h"

namespace {

// One block: deterministic reduction of sum((pred - true)^2), plus the gradient.
__global__ __launch_bounds__(1024) void mse_kernel(int64_t n, const float* __restrict__ pred,
                                                   const float* __restrict__ truth, float scale,
                                                   float* __restrict__ g, float* __restrict__ loss) {
  __shared__ float part[1024 / 64];
  const float inv = 1.0f / (float)(3 * n);
  float acc = 0.f;
  for (int64_t i = threadIdx.x; i < 3 * n; i += blockDim.x) {
    const float d = pred[i] - truth[i];
    acc += d * d;
    if (g) g[i] = scale * (2.0f * d * inv);
  }
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.f;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += part[w];
    if (loss) *loss = s * inv;
  }
}

__global__ void adam_kernel(int64_t n, float* __restrict__ var, float* __restrict__ m,
                            float* __restrict__ v, const float* __restrict__ grad, float lr_t,
                            float omb1, float omb2, float eps, const float* __restrict__ inv_scale,
                            const int32_t* __restrict__ skip) {
  if (skip && *skip) return;
  const float s = inv_scale ? *inv_scale : 1.0f;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const float gr = inv_scale ? fmul(grad[i], s) : grad[i];
    float mi = m[i], vi = v[i];
    mi = fadd(mi, fmul(fsub(gr, mi), omb1));                 // m += (g - m) * (1 - b1)
    vi = fadd(vi, fmul(fsub(fmul(gr, gr), vi), omb2));       // v += (g^2 - v) * (1 - b2)
    m[i] = mi;
    v[i] = vi;
    var[i] = fsub(var[i], fdiv(fmul(mi, lr_t), fadd(fsqrt(vi), eps)));
  }
}

__global__ void finite_kernel(int64_t n, const float* __restrict__ x, int32_t* __restrict__ flag) {
  int bad = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    bad |= !isfinite(x[i]);
  if (__any(bad) && (threadIdx.x & 63) == 0) *flag = 1;
}

struct StepBegin {
  float lr0, decay_steps, rate, b1, b2;
};

// float32(base ** e) with the power evaluated in float64 and rounded once.
__device__ float pow_f32(float base, float e) { return (float)pow((double)base, (double)e); }

// inv_scale and the step's coefficients from the iteration count.
__device__ __forceinline__ void step_begin(const StepState* st, const StepBegin& b, StepState* out) {
  out->inv_scale = fdiv(1.0f, st->scale);
  const int it = st->iterations;
  const float lr = fmul(b.lr0, pow_f32(b.rate, fdiv((float)it, b.decay_steps)));
  const float t = (float)(it + 1);
  const float b1p = pow_f32(b.b1, t), b2p = pow_f32(b.b2, t);
  out->lr_t = fdiv(fmul(lr, fsqrt(fsub(1.0f, b2p))), fsub(1.0f, b1p));
  out->omb1 = fsub(1.0f, b.b1);
  out->omb2 = fsub(1.0f, b.b2);
}

__global__ void step_begin_kernel(StepState* st, StepBegin b) {
  if (threadIdx.x != 0) return;
  st->overflow = 0;
  step_begin(st, b, st);
}

// Adam of one element (TF ApplyAdam): m += (g - m)(1 - b1), v += (g^2 - v)(1 - b2), var -= ...
__device__ __forceinline__ void adam_one(float gr, float lr_t, float omb1, float omb2, float eps, float& m, float& v,
                                         float& var) {
  m = fadd(m, fmul(fsub(gr, m), omb1));
  v = fadd(v, fmul(fsub(fmul(gr, gr), v), omb2));
  var = fsub(var, fdiv(fmul(m, lr_t), fadd(fsqrt(v), eps)));
}

// One optimizer step over several models (nerf_optimizer_step): blockIdx.y is the model.
struct OptArgs {
  int64_t n[kOptModels], n_check[kOptModels];
  float *var[kOptModels], *m[kOptModels], *v[kOptModels];
  const float* grad[kOptModels];
  unsigned char vec[kOptModels];  // every pointer 16-byte aligned: four elements per thread
};

// Finite check of every gradient; row n_models opens the step (its coefficients).
__global__ __launch_bounds__(256) void opt_check_kernel(OptArgs a, int n_models, StepState* st, StepBegin b) {
  const int k = blockIdx.y;
  if (k == n_models) {
    if (blockIdx.x == 0 && threadIdx.x == 0) step_begin(st, b, st);
    return;
  }
  const float* x = a.grad[k];
  const int64_t n = a.n_check[k], stride = (int64_t)gridDim.x * 256, i0 = (int64_t)blockIdx.x * 256 + threadIdx.x;
  int bad = 0;
  int64_t done = 0;
  if (a.vec[k]) {
    done = n / 4 * 4;
    for (int64_t i = i0; i < n / 4; i += stride) {
      const floatx4 g = reinterpret_cast<const floatx4*>(x)[i];
      bad |= !isfinite(g[0]) | !isfinite(g[1]) | !isfinite(g[2]) | !isfinite(g[3]);
    }
  }
  for (int64_t i = done + i0; i < n; i += stride) bad |= !isfinite(x[i]);
  if (__any(bad) && (threadIdx.x & 63) == 0) st->found = 1;
}

// Adam of every model, skipped where the check found an overflow.  begin: there is no check
// launch, each workgroup computes the step's coefficients (and the first one stores them).
__global__ __launch_bounds__(256) void opt_adam_kernel(OptArgs a, float eps, StepState* st, int begin, StepBegin b) {
  __shared__ StepState c;
  if (begin) {
    if (threadIdx.x == 0) {
      step_begin(st, b, &c);
      if (blockIdx.x == 0 && blockIdx.y == 0) {
        st->inv_scale = c.inv_scale;
        st->lr_t = c.lr_t;
        st->omb1 = c.omb1;
        st->omb2 = c.omb2;
      }
    }
    __syncthreads();
  } else {
    if (st->found) return;
    if (threadIdx.x == 0) c = *st;
    __syncthreads();
  }
  const float s = c.inv_scale, lr_t = c.lr_t, omb1 = c.omb1, omb2 = c.omb2;
  const int k = blockIdx.y;
  const int64_t n = a.n[k], stride = (int64_t)gridDim.x * 256, i0 = (int64_t)blockIdx.x * 256 + threadIdx.x;
  int64_t done = 0;
  if (a.vec[k]) {
    done = n / 4 * 4;
    for (int64_t i = i0; i < n / 4; i += stride) {
      const floatx4 g = reinterpret_cast<const floatx4*>(a.grad[k])[i];
      floatx4 m4 = reinterpret_cast<floatx4*>(a.m[k])[i], v4 = reinterpret_cast<floatx4*>(a.v[k])[i];
      floatx4 x4 = reinterpret_cast<floatx4*>(a.var[k])[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float m = m4[e], v = v4[e], x = x4[e];
        adam_one(fmul(g[e], s), lr_t, omb1, omb2, eps, m, v, x);
        m4[e] = m;
        v4[e] = v;
        x4[e] = x;
      }
      reinterpret_cast<floatx4*>(a.m[k])[i] = m4;
      reinterpret_cast<floatx4*>(a.v[k])[i] = v4;
      reinterpret_cast<floatx4*>(a.var[k])[i] = x4;
    }
  }
  for (int64_t i = done + i0; i < n; i += stride) {
    float m = a.m[k][i], v = a.v[k][i], x = a.var[k][i];
    adam_one(fmul(a.grad[k][i], s), lr_t, omb1, omb2, eps, m, v, x);
    a.m[k][i] = m;
    a.v[k][i] = v;
    a.var[k][i] = x;
  }
}

__global__ void adam_state_kernel(int64_t n, float* __restrict__ var, float* __restrict__ m,
                                  float* __restrict__ v, const float* __restrict__ grad, float eps,
                                  const StepState* __restrict__ st) {
  if (st->overflow) return;
  const float s = st->inv_scale, lr_t = st->lr_t, omb1 = st->omb1, omb2 = st->omb2;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    float mi = m[i], vi = v[i], xi = var[i];
    adam_one(fmul(grad[i], s), lr_t, omb1, omb2, eps, mi, vi, xi);
    m[i] = mi;
    v[i] = vi;
    var[i] = xi;
  }
}

__global__ void step_end_kernel(StepState* st, StepEnd e) {
  if (threadIdx.x == 0) step_end(st, e);
}

}  // namespace

extern "C" int32_t nerf_step_begin(nerf_step_state* state, float lr0, int32_t decay_steps, float decay_rate,
                                   float b1, float b2, void* stream) {
  NERF_CHECK_ARG(state && decay_steps > 0, "nerf_step_begin: bad arguments");
  step_begin_kernel<<<1, 64, 0, as_stream(stream)>>>(reinterpret_cast<StepState*>(state),
                                                    StepBegin{lr0, (float)decay_steps, decay_rate, b1, b2});
  NERF_LAUNCH_CHECK("nerf_step_begin");
  return NERF_OK;
}

extern "C" int32_t nerf_adam_tf_state(int64_t n, float* var, float* m, float* v, const float* grad, float eps,
                                      const nerf_step_state* state, void* stream) {
  NERF_CHECK_ARG(n >= 0 && var && m && v && grad && state, "nerf_adam_tf_state: bad arguments");
  if (n == 0) return NERF_OK;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  adam_state_kernel<<<(unsigned)blocks, 256, 0, as_stream(stream)>>>(
      n, var, m, v, grad, eps, reinterpret_cast<const StepState*>(state));
  NERF_LAUNCH_CHECK("nerf_adam_tf_state");
  return NERF_OK;
}

extern "C" int32_t nerf_step_end(nerf_step_state* state, int32_t interval, float factor, float min_scale,
                                 void* stream) {
  NERF_CHECK_ARG(state && interval > 0 && factor > 0.f, "nerf_step_end: bad arguments");
  step_end_kernel<<<1, 64, 0, as_stream(stream)>>>(reinterpret_cast<StepState*>(state),
                                                  StepEnd{interval, factor, min_scale, 0});
  NERF_LAUNCH_CHECK("nerf_step_end");
  return NERF_OK;
}

extern "C" int32_t nerf_mse_grad(int64_t n_rays, const float* pred_rgb, const float* true_rgb,
                                 float scale, float* g_rgb, float* loss_out, void* stream) {
  NERF_CHECK_ARG(n_rays > 0 && pred_rgb && true_rgb, "nerf_mse_grad: bad arguments");
  mse_kernel<<<1, 1024, 0, as_stream(stream)>>>(n_rays, pred_rgb, true_rgb, scale, g_rgb, loss_out);
  NERF_LAUNCH_CHECK("nerf_mse_grad");
  return NERF_OK;
}

extern "C" int32_t nerf_adam_tf(int64_t n, float* var, float* m, float* v, const float* grad,
                                float lr_t, float one_minus_b1, float one_minus_b2, float eps,
                                const float* inv_scale, const int32_t* skip_flag, void* stream) {
  NERF_CHECK_ARG(n >= 0 && var && m && v && grad, "nerf_adam_tf: bad arguments");
  if (n == 0) return NERF_OK;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  adam_kernel<<<(unsigned)blocks, 256, 0, as_stream(stream)>>>(n, var, m, v, grad, lr_t, one_minus_b1,
                                                              one_minus_b2, eps, inv_scale, skip_flag);
  NERF_LAUNCH_CHECK("nerf_adam_tf");
  return NERF_OK;
}

extern "C" int32_t nerf_check_finite(int64_t n, const float* x, int32_t* flag, void* stream) {
  NERF_CHECK_ARG(n >= 0 && x && flag, "nerf_check_finite: bad arguments");
  if (n == 0) return NERF_OK;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 2048) blocks = 2048;
  finite_kernel<<<(unsigned)blocks, 256, 0, as_stream(stream)>>>(n, x, flag);
  NERF_LAUNCH_CHECK("nerf_check_finite");
  return NERF_OK;
}

// What bounds it: launches.  The two 8x256 models' step moves 38 MB (7 us at the rate of a
// copy); as separate launches (open, a check per model, Adam and packing per model, close) it
// took 48.5 us (BF16), most of it the eight calls and launches, and takes 18 here: one check of every gradient, one
// Adam over every model, one packing launch per plan, the first opening and the last closing
// the step; without a check the Adam launch opens it.
extern "C" int32_t nerf_optimizer_step(int32_t n_models, const nerf_opt_model* models, float lr0, int32_t decay_steps,
                                       float decay_rate, float b1, float b2, float eps, nerf_step_state* state,
                                       int32_t check, int32_t interval, float factor, float min_scale,
                                       void* stream) {
  NERF_CHECK_ARG(n_models >= 0 && (models || !n_models) && state && decay_steps > 0 && interval > 0 && factor > 0.f,
                 "nerf_optimizer_step: bad arguments");
  MlpPlan P;
  for (int i = 0; i < n_models; ++i) {
    const nerf_opt_model& M = models[i];
    NERF_CHECK_ARG(M.desc && nerf_plan_from_desc(M.desc, M.precision, &P) == 0,
                   "nerf_optimizer_step: unsupported MLP description or precision");
    NERF_CHECK_ARG(M.params && M.m && M.v && M.grad && M.packed && M.grad_n >= 0,
                   "nerf_optimizer_step: null pointer");
  }
  hipStream_t s = as_stream(stream);
  StepState* st = reinterpret_cast<StepState*>(state);
  const StepBegin sb{lr0, (float)decay_steps, decay_rate, b1, b2};
  const StepEnd se{interval, factor, min_scale, 1};
  // models that share parameters or moments (one net listed twice) are updated one after the other
  auto shares = [&](int i, int j) {
    MlpPlan Pi, Pj;
    nerf_plan_from_desc(models[i].desc, models[i].precision, &Pi);
    nerf_plan_from_desc(models[j].desc, models[j].precision, &Pj);
    const float* bi[3] = {models[i].params, models[i].m, models[i].v};
    const float* bj[3] = {models[j].params, models[j].m, models[j].v};
    for (const float* x : bi)
      for (const float* y : bj)
        if (x < y + Pj.n_params && y < x + Pi.n_params) return true;
    return false;
  };
  // models first, first + 1, .. of at most kOptModels per launch
  auto args = [&](int first, OptArgs& a, int& n, unsigned& gx) {
    a = OptArgs{};
    int64_t most = 0;
    for (n = 0; n < kOptModels && first + n < n_models; ++n) {
      bool apart = true;
      for (int k = 0; k < n && apart; ++k) apart = !shares(first + k, first + n);
      if (!apart) break;
      const nerf_opt_model& M = models[first + n];
      nerf_plan_from_desc(M.desc, M.precision, &P);
      a.n[n] = P.n_params;
      a.n_check[n] = M.grad_n;
      a.var[n] = M.params;
      a.m[n] = M.m;
      a.v[n] = M.v;
      a.grad[n] = M.grad;
      a.vec[n] = (((uintptr_t)M.params | (uintptr_t)M.m | (uintptr_t)M.v | (uintptr_t)M.grad) & 15) == 0;
      if (a.n[n] > most) most = a.n[n];
      if (a.n_check[n] > most) most = a.n_check[n];
    }
    const int64_t blocks = (most + 1023) / 1024;  // four elements per thread
    gx = (unsigned)(blocks < 1 ? 1 : (blocks > 4096 ? 4096 : blocks));
  };
  OptArgs a;
  int n = 0;
  unsigned gx = 1;
  if (check)
    for (int i = 0; i == 0 || i < n_models; i += n ? n : 1) {  // (the first launch opens the step)
      args(i, a, n, gx);
      opt_check_kernel<<<dim3(gx, (unsigned)n + (i == 0)), 256, 0, s>>>(a, n, st, sb);
    }
  for (int i = 0; i < n_models; i += n) {
    args(i, a, n, gx);
    opt_adam_kernel<<<dim3(gx, (unsigned)n), 256, 0, s>>>(a, eps, st, !check, sb);
  }
  // one packing launch per plan (and kOptModels models); the last one closes the step
  auto same = [&](int i, int j) {
    return models[j].precision == models[i].precision &&
           memcmp(models[j].desc, models[i].desc, sizeof(nerf_mlp_desc)) == 0;
  };
  int left = n_models;
  for (int i = 0; i < n_models; ++i) {
    bool seen = false;
    for (int j = 0; j < i && !seen; ++j) seen = same(i, j);
    if (seen) continue;
    nerf_plan_from_desc(models[i].desc, models[i].precision, &P);
    const float* flat[kOptModels];
    void* out[kOptModels];
    n = 0;
    for (int j = i; j < n_models; ++j) {
      if (!same(i, j)) continue;
      flat[n] = models[j].params;
      out[n++] = models[j].packed;
      --left;
      if (n == kOptModels || !left) {
        pack_models(P, n, flat, out, left ? nullptr : st, se, s);
        n = 0;
      }
    }
    if (n) pack_models(P, n, flat, out, nullptr, se, s);
  }
  if (!n_models) step_end_kernel<<<1, 64, 0, s>>>(st, se);
  NERF_LAUNCH_CHECK("nerf_optimizer_step");
  return NERF_OK;
}
