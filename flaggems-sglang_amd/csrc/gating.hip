// Router gating: scores -> top-k -> optional renormalisation, one wave per
// token. Produces the (topk_weights, topk_ids) pair the fused MoE consumes
// (the routing the reference's tests build with torch ops,
// tests/test_fused_moe.py:37-41, and that _standard_topk_to_triton_kernels
// converts, src/flaggems_sglang/ops/fused_moe.py:119-146).
//
// Each lane holds experts lane, lane+64, ... (VPL per lane). Selection ranks
// the logits themselves (softmax and sigmoid are monotonic, so this is the
// same set as ranking the scores, and it is exact: no rounding can reorder
// two experts); equal logits go to the lower expert id. Selected experts come
// out in rank order, like torch.topk(sorted=True).
//
// Bound: latency. A wave's chain of topk picks sets the time -- at one token
// there is nothing else, at 2048 tokens of 256 logits (2 MB) still most of
// it. A pick is a wave-wide maximum of order-preserving 32-bit keys by DPP row
// rotations and four readlanes, then one ballot per register for the lowest
// id that holds it, in place of six two-word butterfly shuffles (an LDS
// round trip each): 6.7 -> 3.0 us at one token of 128 experts, 10.0 -> 4.8 at
// 2048 tokens of 256, 9.3 -> 4.6 at 37.
#include <math.h>

#include "fgs_common.h"
#include "fgs_moe_kernels.h"

namespace fgs {

// v rotated by N lanes within each row of 16 lanes.
template <int N>
__device__ __forceinline__ uint32_t row_ror(uint32_t v) {
  return static_cast<uint32_t>(
      __builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x120 + N, 0xf, 0xf, false));
}

// f over all 64 lanes' values (f commutative and associative up to
// rounding); the result is uniform.
template <class F>
__device__ __forceinline__ uint32_t wave_reduce(uint32_t v, F f) {
  v = f(v, row_ror<8>(v));
  v = f(v, row_ror<4>(v));
  v = f(v, row_ror<2>(v));
  v = f(v, row_ror<1>(v));
  const uint32_t a = __builtin_amdgcn_readlane(v, 0), b = __builtin_amdgcn_readlane(v, 16);
  const uint32_t c = __builtin_amdgcn_readlane(v, 32), d = __builtin_amdgcn_readlane(v, 48);
  return f(f(a, b), f(c, d));
}

// Unsigned keys in the order of the floats (-0 as +0; a NaN of either sign
// beyond the infinity of its sign); 0 is below every float's key but the
// negative NaNs' lowest, which is raised to 1.
__device__ __forceinline__ uint32_t order_key(float f) {
  const uint32_t b = __float_as_uint(f + 0.0f);
  const uint32_t k = (b >> 31) ? ~b : b | 0x80000000u;
  return k > 0 ? k : 1u;
}

template <int VPL>
__global__ __launch_bounds__(256) void topk_gating_kernel(
    const void* __restrict__ logits, int bf16_in, int64_t m, int num_experts,
    int topk, int sigmoid, int renormalize, float* __restrict__ w_out,
    int32_t* __restrict__ id_out) {
  const int lane = threadIdx.x & 63;
  const int64_t row = blockIdx.x * 4LL + (threadIdx.x >> 6);
  if (row >= m) return;  // whole wave

  float v[VPL];
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int e = i * 64 + lane;
    if (e < num_experts) {
      const int64_t at = row * num_experts + e;
      v[i] = bf16_in ? bf16_bits_to_f32(static_cast<const uint16_t*>(logits)[at])
                     : static_cast<const float*>(logits)[at];
    } else {
      v[i] = -INFINITY;
    }
  }

  // scores
  float p[VPL];
  if (sigmoid) {
#pragma unroll
    for (int i = 0; i < VPL; ++i) p[i] = 1.0f / (1.0f + __expf(-v[i]));
  } else {
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < VPL; ++i) mx = fmaxf(mx, v[i]);
    mx = __uint_as_float(wave_reduce(__float_as_uint(mx), [](uint32_t a, uint32_t b) {
      return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b)));
    }));
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      p[i] = i * 64 + lane < num_experts ? __expf(v[i] - mx) : 0.f;
      sum += p[i];
    }
    sum = __uint_as_float(wave_reduce(__float_as_uint(sum), [](uint32_t a, uint32_t b) {
      return __float_as_uint(__uint_as_float(a) + __uint_as_float(b));
    }));
    const float inv = 1.0f / sum;
#pragma unroll
    for (int i = 0; i < VPL; ++i) p[i] *= inv;
  }

  // top-k by (logit desc, expert id asc); lane r keeps the r-th pick. A
  // picked or absent expert's key is 0; topk <= num_experts leaves one above
  // 0 for every pick.
  uint32_t key[VPL];
#pragma unroll
  for (int i = 0; i < VPL; ++i) key[i] = i * 64 + lane < num_experts ? order_key(v[i]) : 0u;
  float my_w = 0.f, wsum = 0.f;
  int my_id = 0;
  for (int r = 0; r < topk; ++r) {
    uint32_t best = key[0];
#pragma unroll
    for (int i = 1; i < VPL; ++i) best = max(best, key[i]);
    best = wave_reduce(best, [](uint32_t a, uint32_t b) { return max(a, b); });
    // the first register, then lane, that holds it: the lowest expert id
    int idx = -1;
    float pw = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const uint64_t hit = __ballot(key[i] == best);
      if (idx < 0 && hit != 0) {
        const int at = __ffsll(static_cast<long long>(hit)) - 1;
        idx = i * 64 + at;
        pw = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(p[i]), at));
        if (lane == at) key[i] = 0u;
      }
    }
    if (lane == r) {
      my_w = pw;
      my_id = idx;
    }
    wsum += pw;
  }
  if (lane < topk) {
    w_out[row * topk + lane] = renormalize ? my_w / wsum : my_w;
    id_out[row * topk + lane] = my_id;
  }
}

int launch_topk_gating(const void* logits, bool bf16_in, int64_t m,
                       int num_experts, int topk, bool sigmoid,
                       bool renormalize, float* w_out, int32_t* id_out,
                       hipStream_t stream) {
  if (m == 0) return FGS_OK;
  const dim3 grid(static_cast<unsigned>((m + 3) / 4));
  const int vpl = (num_experts + 63) / 64;
#define FGS_GATING_CASE(V)                                                      \
  hipLaunchKernelGGL(topk_gating_kernel<V>, grid, dim3(256), 0, stream, logits, \
                     bf16_in ? 1 : 0, m, num_experts, topk, sigmoid ? 1 : 0,     \
                     renormalize ? 1 : 0, w_out, id_out)
  if (vpl <= 1) FGS_GATING_CASE(1);
  else if (vpl <= 2) FGS_GATING_CASE(2);
  else if (vpl <= 4) FGS_GATING_CASE(4);
  else if (vpl <= 8) FGS_GATING_CASE(8);
  else FGS_GATING_CASE(16);
#undef FGS_GATING_CASE
  return check_launch("topk_gating_kernel");
}

}  // namespace fgs
