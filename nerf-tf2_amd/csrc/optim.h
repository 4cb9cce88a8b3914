// Device-side state of an optimizer step, shared by the optimizer kernels and the operand packing
// (whose last launch closes the step).
#pragma once
#include "common.h"
#include "mlp_plan.h"

constexpr int kOptModels = 8;  // models per optimizer step

// Loss-scaled step state (layout of nerf_step_state).  found: set by the finite check of the
// running nerf_optimizer_step, cleared when that step closes.
struct StepState {
  float scale, inv_scale;
  int32_t overflow, good, iterations, skipped;
  float lr_t, omb1, omb2;
  int32_t found;
  int32_t reserved[6];
};
static_assert(sizeof(StepState) == 64, "nerf_step_state is 64 bytes");

struct StepEnd {
  int interval;
  float factor, min_scale;
  int found;  // take the overflow flag from state->found, and clear it
};

// Scale and iteration count after a step (see nerf_step_end).
__device__ __forceinline__ void step_end(StepState* st, const StepEnd& e) {
  if (e.found) {
    st->overflow = st->found;
    st->found = 0;
  }
  if (st->overflow) {
    const float s = fdiv(st->scale, e.factor);
    st->scale = s > e.min_scale ? s : e.min_scale;
    st->good = 0;
    st->skipped += 1;
  } else {
    st->iterations += 1;
    st->good += 1;
    if (st->good >= e.interval) {
      st->scale = fmul(st->scale, e.factor);
      st->good = 0;
    }
  }
}

void pack_models(const MlpPlan& P, int n, const float* const* flat, void* const* packed, StepState* state,
                 const StepEnd& end, hipStream_t s);
int nerf_plan_from_desc(const nerf_mlp_desc* d, int prec, MlpPlan* p);
