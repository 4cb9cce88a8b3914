// Inverse-transform fine sampling: create_input_batch_fine_model
// (nerf/utils/ray_utils.py:276-406).  One wave64 per ray.
//
// Bit-exact with the oracle: every float op is an explicitly rounded
// intrinsic and the summation orders are fixed —
//   denom = reduce_sum(w' * width)  in the order of an 8-wide Eigen packet
//           reduction (lane j sums bins j, j+8, ...; then
//           ((p0+p4)+(p2+p6)) + ((p1+p5)+(p3+p7)), plus the n mod 8 tail);
//   agg   = cumsum(pdf * width)      sequential, each lane recomputing its own
//           prefix in left-to-right order.
// searchsorted(side='right') is an upper_bound binary search; the final
// tf.sort(concat(t_coarse, t_fine)) is a rank merge (coarse values first on
// ties), so equal values land in equal slots and the output is the sorted set.
//
// Compensated mode (NERF_CDF_COMPENSATED, the BF16 and learned forms): the
// products w' * width are split exactly into (hi, lo) pairs (fma residual),
// prefix-summed as compensated pairs (TwoSum), denom is the rounded total and
// cdf_k = S_k / denom with the division's remainder carried (fma), so every
// cdf value is within about one ulp of the exact prefix ratio instead of
// accumulating one rounding per bin.  pdf = w' / denom as in the reference.
#include "common.h"
#include <type_traits>

namespace {

constexpr int kWaves = 4;
constexpr int kMaxNc = 64;
constexpr int kMaxNf = 256;

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Compensated inclusive prefix of (ph, pl) pairs over lanes 0..63 (lanes past
// the bins hold zeros): Hillis-Steele steps with compensated pair adds.
__device__ __forceinline__ void comp_prefix(float& sh, float& sl, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const float oh = shfl_up(sh, d), ol = shfl_up(sl, d);
    if (lane >= d) dd_add(oh, ol, sh, sl, sh, sl);
  }
}

// (sh + sl) / denom rounded once up to the division's own error: the exact
// remainder of the first quotient is carried into a correction term.
__device__ __forceinline__ float comp_ratio(float sh, float sl, float denom) {
  const float q = fdiv(sh, denom);
  const float r = __builtin_fmaf(-q, denom, sh);
  return fadd(q, fdiv(fadd(r, sl), denom));
}

__global__ __launch_bounds__(256) void fine_kernel(
    int64_t n_rays, int nc, int nf, const float* __restrict__ ro, const float* __restrict__ rd,
    const float* __restrict__ bin_weights, const float* __restrict__ bin_edges,
    const float* __restrict__ bin_widths, const float* __restrict__ t_c,
    const float* __restrict__ u_vals, float* __restrict__ t_out, int32_t* __restrict__ idx_out,
    float* __restrict__ tf_out, float* __restrict__ xyz, float* __restrict__ dirs, int comp,
    float* __restrict__ cdf_out) {
  __shared__ float s_agg[kWaves][kMaxNc + 1];
  __shared__ float s_pdf[kWaves][kMaxNc];
  __shared__ float s_left[kWaves][kMaxNc];
  __shared__ float s_tc[kWaves][kMaxNc];
  __shared__ float s_tf[kWaves][kMaxNf];
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int64_t ray = (int64_t)blockIdx.x * kWaves + w;
  if (ray >= n_rays) return;  // wave-uniform; no block-level barriers below
  const int S = nc + nf;

  // ---- pdf and cdf over the coarse bins (ray_utils.py:335-345)
  const bool on = lane < nc;
  const float wv = on ? bin_weights[ray * nc + lane] : 0.f;
  const float width = on ? bin_widths[ray * nc + lane] : 0.f;
  const float left = on ? bin_edges[ray * (nc + 1) + lane] : 0.f;
  const float wp = fadd(wv, 1e-5f);      // bin_weights + 1e-5
  const float prod = fmul(wp, width);    // bin_weights * bin_widths
  float pdf, agg;
  if (comp) {
    float sh = on ? prod : 0.f, sl = on ? __builtin_fmaf(wp, width, -prod) : 0.f;
    comp_prefix(sh, sl, lane);
    const float denom = shfl(sh, nc - 1);
    pdf = fdiv(wp, denom);
    agg = comp_ratio(sh, sl, denom);
  } else {
    const int nv = (nc / 8) * 8;
    float p = 0.f;
    for (int i = (lane & 7); i < nv; i += 8) p = fadd(p, shfl(prod, i));
    // every lane needs the same shuffles: loop bound is lane-independent
    float tail = 0.f;
    for (int i = nv; i < nc; ++i) tail = fadd(tail, shfl(prod, i));
    const float P0 = shfl(p, 0), P1 = shfl(p, 1), P2 = shfl(p, 2), P3 = shfl(p, 3);
    const float P4 = shfl(p, 4), P5 = shfl(p, 5), P6 = shfl(p, 6), P7 = shfl(p, 7);
    const float denom =
        fadd(tail, fadd(fadd(fadd(P0, P4), fadd(P2, P6)), fadd(fadd(P1, P5), fadd(P3, P7))));
    pdf = fdiv(wp, denom);               // ray_utils.py:339
    const float cw = fmul(pdf, width);   // pdf * bin_widths
    agg = 0.f;
    for (int k = 0; k < nc; ++k) {       // sequential inclusive cumsum (ray_utils.py:342)
      const float v = shfl(cw, k);
      if (k <= lane) agg = fadd(agg, v);
    }
  }
  if (cdf_out) {
    if (lane == 0) cdf_out[ray * (nc + 1)] = 0.f;
    if (on) cdf_out[ray * (nc + 1) + 1 + lane] = agg;
  }
  if (lane == 0) s_agg[w][0] = 0.f;      // concat 0 (ray_utils.py:345)
  if (on) {
    s_agg[w][lane + 1] = agg;
    s_pdf[w][lane] = pdf;
    s_left[w][lane] = left;
    s_tc[w][lane] = t_c[ray * nc + lane];
  }
  wave_sync();

  // ---- inverse transform (ray_utils.py:355-377)
  for (int q = lane; q < nf; q += 64) {
    const float u = u_vals[ray * nf + q];
    // searchsorted(agg[:, 1:-1], u, side='right'): first inner edge > u
    int lo = 0, hi = nc - 1;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (s_agg[w][1 + mid] <= u)
        lo = mid + 1;
      else
        hi = mid;
    }
    const int idx = lo;
    const float agg_ = s_agg[w][idx];
    float pdf_ = s_pdf[w][idx];
    const float left_ = s_left[w][idx];
    const float mask = pdf_ < 1e-8f ? 0.f : 1.f;   // ray_utils.py:372
    pdf_ = fmaxf(pdf_, 1e-8f);                      // ray_utils.py:373
    const float tf = fadd(fmul(fdiv(fsub(u, agg_), pdf_), mask), left_);  // :376
    s_tf[w][q] = tf;
    if (idx_out) idx_out[ray * nf + q] = idx;
    if (tf_out) tf_out[ray * nf + q] = tf;
  }
  wave_sync();

  // ---- sort(concat(t_coarse, t_fine)) as a rank merge (ray_utils.py:380-385)
  float o3[3] = {0.f, 0.f, 0.f}, d3[3] = {0.f, 0.f, 0.f};
  if (xyz) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      o3[c] = ro[3 * ray + c];
      d3[c] = rd[3 * ray + c];
    }
  }
  float* trow = t_out + ray * S;
  auto emit = [&](int pos, float t) {
    trow[pos] = t;
    if (xyz) {  // o + t * d                                  (ray_utils.py:389-398)
      const int64_t m = ray * S + pos;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        xyz[3 * m + c] = fadd(o3[c], fmul(t, d3[c]));
        dirs[3 * m + c] = d3[c];
      }
    }
  };
  for (int q = lane; q < nf; q += 64) {
    const float v = s_tf[w][q];
    int rank = 0;
    for (int k = 0; k < nf; ++k) {
      const float o = s_tf[w][k];
      rank += (o < v) || (o == v && k < q);
    }
    int nle = 0;  // coarse values <= v (coarse first on ties)
    for (int k = 0; k < nc; ++k) nle += (s_tc[w][k] <= v);
    emit(rank + nle, v);
  }
  for (int j = lane; j < nc; j += 64) {
    const float v = s_tc[w][j];
    int nlt = 0;
    for (int k = 0; k < nf; ++k) nlt += (s_tf[w][k] < v);
    emit(j + nlt, v);
  }
}

// Value of `v` in lane `k` (a compile-time lane after unrolling): v_readlane
// into a scalar register, no LDS round trip.
__device__ __forceinline__ float lane_value(float v, int k) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), k));
}

// Lane i - 1's value in lane i, 0 in lane 0 (DPP wave_shr:1, bound_ctrl).
__device__ __forceinline__ float lane_shift_up(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xF, 0xF, true));
}

// Lane i ^ J's value for J = 1, 2, 3, 4, 7, 8, 15, 16, 31, 63: DPP moves (quad_perm,
// row_half_mirror = ^7, row_ror:8 = ^8, row_mirror = ^15) and their products; across
// rows of 16 and halves of 32, a lane swap and a select.
template <int J>
__device__ __forceinline__ int lane_xor(int x, int lane) {
  if constexpr (J == 1) return __builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, false);
  else if constexpr (J == 2) return __builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, false);
  else if constexpr (J == 3) return __builtin_amdgcn_mov_dpp(x, 0x1B, 0xF, 0xF, false);
  else if constexpr (J == 7) return __builtin_amdgcn_mov_dpp(x, 0x141, 0xF, 0xF, false);
  else if constexpr (J == 8) return __builtin_amdgcn_mov_dpp(x, 0x128, 0xF, 0xF, false);
  else if constexpr (J == 15) return __builtin_amdgcn_mov_dpp(x, 0x140, 0xF, 0xF, false);
  else if constexpr (J == 4) return lane_xor<3>(lane_xor<7>(x, lane), lane);
  else if constexpr (J == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);  // rows (0, 0, 2, 2) and (1, 1, 3, 3)
    return lane & 16 ? r[0] : r[1];
  } else if constexpr (J == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);  // halves (0, 0) and (1, 1)
    return lane & 32 ? r[0] : r[1];
  } else if constexpr (J == 31) return lane_xor<15>(lane_xor<16>(x, lane), lane);
  else {
    static_assert(J == 63, "");
    return lane_xor<31>(lane_xor<32>(x, lane), lane);
  }
}

template <int J>
__device__ __forceinline__ float lane_xor_f(float x, int lane) {
  return __builtin_bit_cast(float, lane_xor<J>(__builtin_bit_cast(int, x), lane));
}

// The smaller of a and b where lim is INT_MIN, the larger where it is INT_MAX (v_med3_i32).
__device__ __forceinline__ int med3(int a, int b, int lim) {
  const int lo = a < b ? a : b, hi = a < b ? b : a;
  const int c = hi < lim ? hi : lim;
  return lo > c ? lo : c;
}

// Ascending sort of the wave's 64 R integers; element e = R lane + r.  Bitonic merges
// whose first step pairs e with e ^ (2 k - 1), so that every comparison puts the smaller
// value at the smaller index: which of the two a lane keeps depends on one bit of its
// number, one v_med3_i32 against that bit's limit (lim).  With two elements a lane the
// steps between neighbours stay inside the lane.
template <int R>
__device__ __forceinline__ void wave_sort(int (&v)[R], int lane) {
  static_assert(R == 1 || R == 2, "");
  int lim[6];
#pragma unroll
  for (int b = 0; b < 6; ++b) lim[b] = (int)(0x80000000u + (uint32_t)((lane << (31 - b)) >> 31));  // INT_MIN or INT_MAX
  auto in_lane = [&]() {
    if constexpr (R == 2) {
      const int a = v[0], b = v[1];
      v[0] = a < b ? a : b;
      v[1] = a < b ? b : a;
    }
  };
  auto step = [&](auto jc, auto mirror_c, int b) {
    constexpr int J = decltype(jc)::value;
    constexpr bool kMirror = decltype(mirror_c)::value;
    int o[R];
#pragma unroll
    for (int r = 0; r < R; ++r) o[r] = lane_xor<J>(v[kMirror ? R - 1 - r : r], lane);
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = med3(v[r], o[r], lim[b]);
  };
  auto merge = [&](auto bc) {  // sorted runs of 2^b lanes -> of 2^(b + 1) lanes
    constexpr int B = decltype(bc)::value;
    step(std::integral_constant<int, (2 << B) - 1>{}, std::true_type{}, B);
    if constexpr (B >= 5) step(std::integral_constant<int, 16>{}, std::false_type{}, 4);
    if constexpr (B >= 4) step(std::integral_constant<int, 8>{}, std::false_type{}, 3);
    if constexpr (B >= 3) step(std::integral_constant<int, 4>{}, std::false_type{}, 2);
    if constexpr (B >= 2) step(std::integral_constant<int, 2>{}, std::false_type{}, 1);
    if constexpr (B >= 1) step(std::integral_constant<int, 1>{}, std::false_type{}, 0);
    in_lane();
  };
  in_lane();
  merge(std::integral_constant<int, 0>{});
  merge(std::integral_constant<int, 1>{});
  merge(std::integral_constant<int, 2>{});
  merge(std::integral_constant<int, 3>{});
  merge(std::integral_constant<int, 4>{});
  merge(std::integral_constant<int, 5>{});
}

// Integers in the order of the floats (its own inverse); NaNs lie beyond the infinities.
__device__ __forceinline__ int order_key(int x) { return x ^ ((x >> 31) & 0x7FFFFFFF); }

// Count of the first N entries of the ascending row a that are <= x (LE) or < x (!LE),
// in steps of falling powers of two without a branch.  N = 2^k - 1 needs nothing more;
// N = 2^k ends with one more comparison; for any other N the row has to be continued
// to the next 2^k - 1 entries with +infinity, and the count is held to N.
template <int N, bool LE>
__device__ __forceinline__ int count_below(const float* a, float x) {
  constexpr bool kPow2 = (N & (N - 1)) == 0, kFull = (N & (N + 1)) == 0;
  constexpr int kTop = 1 << (31 - __builtin_clz(N));
  const float* p = a;  // a + the count so far
#pragma unroll
  for (int step = kPow2 ? N / 2 : kTop; step > 0; step >>= 1) {
    const float e = p[step - 1];
    p += (LE ? (e <= x) : (e < x)) ? step : 0;
  }
  if (kPow2) p += (LE ? (*p <= x) : (*p < x)) ? 1 : 0;
  const int c = (int)(p - a);
  return kPow2 || kFull ? c : (c < N ? c : N);
}

// The same computation for the shapes in use (32, 48 or 64 coarse bins, 64 or 128 fine
// samples), organised for throughput.  Instruction issue bounds it: the first form of
// this kernel issued 738 vector instructions a ray, 2,950 of the 2,900 cycles a ray took
// on its SIMD.  So: row addresses are scalar (the wave's number is made uniform); every
// cross-lane read of the cdf passes is a DPP move or a v_readlane; the sort works on
// integers (no canonicalising), two instructions a step and value; the searches have
// neither a branch nor a remainder test; and only the coarse values look up their place
// (index + the number of fine values below it, coarse first on ties): they are put down
// in a cleared row, and each remaining place takes the next fine value, found by
// counting the coarse values before it (a ballot) instead of by a search per fine value.
// Equal floats are indistinguishable, so the output equals the sorted set bit for bit.
// 32,768 rays, kernel trace: 64 + 128 samples 41.9 -> 27.7 us (84 MB with the coarse
// kernel's: 2.3 TB/s here); as calls one after another, 32 + 128, by fine_kernel before:
// 98 -> 23 us, 64 + 64: 45 -> 19 us.
template <int NC, int NF, bool COMP>
__global__ __launch_bounds__(256) void fine_wave_kernel(
    int64_t n_rays, const float* __restrict__ ro, const float* __restrict__ rd,
    const float* __restrict__ bin_weights, const float* __restrict__ bin_edges,
    const float* __restrict__ bin_widths, const float* __restrict__ t_c,
    const float* __restrict__ u_vals, float* __restrict__ t_out, int32_t* __restrict__ idx_out,
    float* __restrict__ tf_out, float* __restrict__ xyz, float* __restrict__ dirs,
    float* __restrict__ cdf_out) {
  constexpr int S = NC + NF, R = NF / 64, Q = (S + 63) / 64;
  static_assert(NC >= 2 && NC <= 64 && NC % 8 == 0 && NF == 64 * R, "one coarse bin per lane, R fine samples");
  constexpr int kFree = 0x7FC0A5A5;  // a place no coarse value has taken
  __shared__ float s_agg[kWaves][65];
  __shared__ float2 s_bin[kWaves][64];  // pdf, left edge
  __shared__ float s_sorted[kWaves][NF];
  __shared__ int s_row[kWaves][64 * Q];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t ray = (int64_t)blockIdx.x * kWaves + w;
  if (ray >= n_rays) return;  // wave-uniform; no block-level barriers below

  // ---- pdf and cdf over the coarse bins (ray_utils.py:335-345)
  const bool on = NC == 64 || lane < NC;
  const float wv = on ? (bin_weights + ray * NC)[lane] : 0.f;
  const float width = on ? (bin_widths + ray * NC)[lane] : 0.f;
  const float left = on ? (bin_edges + ray * (NC + 1))[lane] : 0.f;
  const float tc = on ? (t_c + ray * NC)[lane] : 0.f;
  float u[R];
#pragma unroll
  for (int r = 0; r < R; ++r) u[r] = (u_vals + ray * NF)[lane + 64 * r];
  const float wp = fadd(wv, 1e-5f);
  const float prod = fmul(wp, width);
  float pdf, agg;
  if constexpr (COMP) {
    float sh = on ? prod : 0.f, sl = on ? __builtin_fmaf(wp, width, -prod) : 0.f;
    comp_prefix(sh, sl, lane);
    const float denom = lane_value(sh, NC - 1);
    pdf = fdiv(wp, denom);
    agg = comp_ratio(sh, sl, denom);
  } else {
    // lane j < 8: packet sum P_j = prod_j + prod_{j+8} + ... in that order (the other
    // lanes' sums wrap round and are not used)
    float pj = prod;
#pragma unroll
    for (int i = 1; 8 * i < NC; ++i)
      pj = fadd(pj, __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(4 * lane + 32 * i, __builtin_bit_cast(int, prod))));
    // lane 0: ((P0 + P4) + (P2 + P6)) + ((P1 + P5) + (P3 + P7)); the 8-wide reduction's
    // tail is empty
    pj = fadd(pj, lane_xor_f<4>(pj, lane));
    pj = fadd(pj, lane_xor_f<2>(pj, lane));
    pj = fadd(pj, lane_xor_f<1>(pj, lane));
    const float denom = fadd(0.f, lane_value(pj, 0));
    pdf = fdiv(wp, denom);
    const float cw = fmul(pdf, width);
    // sequential inclusive prefix: after step s lane i holds cw_{i-s} + ... + cw_i added
    // left to right (lane -1 reads 0), so after NC - 1 steps every lane < NC holds
    // ((cw_0 + cw_1) + ...) + cw_i exactly
    agg = cw;
#pragma unroll
    for (int step = 1; step < NC; ++step) agg = fadd(lane_shift_up(agg), cw);
  }
  if (cdf_out) {
    if (lane == 0) cdf_out[ray * (NC + 1)] = 0.f;
    if (on) cdf_out[ray * (NC + 1) + 1 + lane] = agg;
  }
  if (lane == 0) s_agg[w][0] = 0.f;
  // the last bin's cdf is no inner edge: +infinity from there on (count_below)
  s_agg[w][lane + 1] = lane < NC - 1 ? agg : __builtin_inff();
  s_bin[w][lane] = make_float2(pdf, left);
#pragma unroll
  for (int i = 0; i < Q; ++i) s_row[w][lane + 64 * i] = kFree;
  wave_sync();

  // ---- inverse transform (ray_utils.py:355-377), fine samples lane + 64 r
  int key[R], idx[R];
#pragma unroll
  for (int r = 0; r < R; ++r) idx[r] = count_below<NC - 1, true>(&s_agg[w][1], u[r]);  // searchsorted(agg[1:-1], u, 'right')
  float v[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float agg_ = s_agg[w][idx[r]];
    const float2 bin = s_bin[w][idx[r]];
    const float mask = bin.x < 1e-8f ? 0.f : 1.f;
    const float pdf_ = fmaxf(bin.x, 1e-8f);
    v[r] = fadd(fmul(fdiv(fsub(u[r], agg_), pdf_), mask), bin.y);
    key[r] = order_key(__builtin_bit_cast(int, v[r]));
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (idx_out) (idx_out + ray * NF)[lane + 64 * r] = idx[r];
    if (tf_out) (tf_out + ray * NF)[lane + 64 * r] = v[r];
  }
  wave_sort<R>(key, lane);
#pragma unroll
  for (int r = 0; r < R; ++r) s_sorted[w][R * lane + r] = __builtin_bit_cast(float, order_key(key[r]));
  wave_sync();

  // ---- sort(concat(t_coarse, t_fine)) (ray_utils.py:380-398)
  if (on) s_row[w][lane + count_below<NF, false>(&s_sorted[w][0], tc)] = __builtin_bit_cast(int, tc);
  wave_sync();
  float o3[3] = {0.f, 0.f, 0.f}, d3[3] = {0.f, 0.f, 0.f};
  if (xyz) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      o3[c] = ro[3 * ray + c];
      d3[c] = rd[3 * ray + c];
    }
  }
  int before = 0;  // coarse values in the places below 64 i
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const int pos = lane + 64 * i;
    const int c = s_row[w][pos];
    const uint64_t taken = __ballot(c != kFree);
    int k = pos - before -
            (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(taken >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)taken, 0u));
    before += __popcll(taken);
    k = k < NF ? k : NF - 1;  // (only where coarse values were not ascending and shared a place)
    const float f = s_sorted[w][k];
    const float t = c != kFree ? __builtin_bit_cast(float, c) : f;
    if (S % 64 == 0 || pos < S) {
      (t_out + ray * S)[pos] = t;
      if (xyz) {
        const int64_t m = ray * S + pos;
#pragma unroll
        for (int c3 = 0; c3 < 3; ++c3) {
          xyz[3 * m + c3] = fadd(o3[c3], fmul(t, d3[c3]));
          dirs[3 * m + c3] = d3[c3];
        }
      }
    }
  }
}

}  // namespace

extern "C" int32_t nerf_create_input_batch_fine(int64_t n_rays, int32_t n_coarse, int32_t n_fine,
                                                const float* rays_o, const float* rays_d,
                                                const float* bin_weights, const float* bin_edges,
                                                const float* bin_widths,
                                                const float* t_vals_coarse, const float* u_vals,
                                                float* t_vals, int32_t* piece_idxs,
                                                float* t_vals_fine, float* xyz_inputs,
                                                float* dir_inputs, int32_t cdf_mode, float* cdf,
                                                void* stream) {
  NERF_CHECK_ARG(n_rays >= 0 && n_coarse >= 2 && n_coarse <= kMaxNc && n_fine >= 1 &&
                     n_fine <= kMaxNf,
                 "nerf_create_input_batch_fine: n_coarse=%d (2..%d) n_fine=%d (1..%d)", n_coarse,
                 kMaxNc, n_fine, kMaxNf);
  NERF_CHECK_ARG(cdf_mode == NERF_CDF_TF_ORDER || cdf_mode == NERF_CDF_COMPENSATED,
                 "nerf_create_input_batch_fine: cdf_mode=%d", cdf_mode);
  if (n_rays == 0) return NERF_OK;  // empty batch
  NERF_CHECK_ARG(bin_weights && bin_edges && bin_widths && t_vals_coarse && u_vals && t_vals,
                 "nerf_create_input_batch_fine: null pointer");
  NERF_CHECK_ARG((xyz_inputs == nullptr) == (dir_inputs == nullptr),
                 "nerf_create_input_batch_fine: xyz_inputs and dir_inputs go together");
  NERF_CHECK_ARG(!xyz_inputs || (rays_o && rays_d),
                 "nerf_create_input_batch_fine: xyz_inputs needs rays");
  const unsigned grid = (unsigned)((n_rays + kWaves - 1) / kWaves);
  hipStream_t s = as_stream(stream);
  const bool comp = cdf_mode == NERF_CDF_COMPENSATED;
#define NERF_FINE(NC_, NF_)                                                                       \
  if (n_coarse == NC_ && n_fine == NF_) {                                                         \
    const auto k = comp ? fine_wave_kernel<NC_, NF_, true> : fine_wave_kernel<NC_, NF_, false>;   \
    k<<<grid, 64 * kWaves, 0, s>>>(n_rays, rays_o, rays_d, bin_weights, bin_edges, bin_widths,    \
                                   t_vals_coarse, u_vals, t_vals, piece_idxs, t_vals_fine,        \
                                   xyz_inputs, dir_inputs, cdf);                                  \
  } else
  NERF_FINE(64, 128)
  NERF_FINE(48, 128)
  NERF_FINE(32, 128)
  NERF_FINE(64, 64)
  NERF_FINE(48, 64)
  NERF_FINE(32, 64)
  // other shapes: loops instead of unrolled lanes, a quadratic rank merge
  fine_kernel<<<grid, 64 * kWaves, 0, s>>>(
      n_rays, n_coarse, n_fine, rays_o, rays_d, bin_weights, bin_edges, bin_widths, t_vals_coarse,
      u_vals, t_vals, piece_idxs, t_vals_fine, xyz_inputs, dir_inputs, comp ? 1 : 0, cdf);
#undef NERF_FINE
  NERF_LAUNCH_CHECK("nerf_create_input_batch_fine");
  return NERF_OK;
}
