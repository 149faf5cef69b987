// Bandwidth-bound kernels of the fused-MoE path: silu_and_mul, moe_sum and
// the dynamic activation quantisers. Every thread moves 16-byte vectors;
// a row is processed by consecutive threads so each wave touches one or two
// contiguous 1 KiB spans per instruction.
#include <math.h>

#include <string>
#include <type_traits>

#include "fgs_moe_kernels.h"

namespace fgs {

// ----------------------------------------------------------- silu_and_mul ---
// out[r, c] = bf16(silu(f32(in[r, c])) * f32(in[r, n + c]))
// (ops/fused_moe.py:44-63). Requires n % 8 == 0; 8 columns per thread.
__global__ __launch_bounds__(256) void silu_and_mul_kernel(
    const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int64_t rows,
    int64_t n) {
  const int64_t vec_per_row = n / 8;
  const int64_t total = rows * vec_per_row;
  for (int64_t v = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
       v < total; v += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t r = v / vec_per_row;
    const int64_t c = (v - r * vec_per_row) * 8;
    const u32x4 g = *reinterpret_cast<const u32x4*>(in + r * 2 * n + c);
    const u32x4 u = *reinterpret_cast<const u32x4*>(in + r * 2 * n + n + c);
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float g0 = __uint_as_float(g[j] << 16);
      const float g1 = __uint_as_float(g[j] & 0xffff0000u);
      const float u0 = __uint_as_float(u[j] << 16);
      const float u1 = __uint_as_float(u[j] & 0xffff0000u);
      o[j] = pack_bf16x2(silu_mul(g0, u0), silu_mul(g1, u1));
    }
    *reinterpret_cast<u32x4*>(out + r * n + c) = o;
  }
}

// ---------------------------------------------------------------- moe_sum ---
// out[t, c] = bf16(sum_j f32(in[t, j, c])): the top-k reduction that
// matmul_ogs performs when given scatter_indx (ops/fused_moe.py:224-231).
// Requires k % 8 == 0. With `ids` given, slots whose expert id lies outside
// [0, num_experts) were never computed and contribute nothing. With
// `weights` given each slot is scaled first: out = bf16(sum_j w_j * y_j),
// product and sum each rounded in fp32 in slot order (no fused multiply-add),
// which is the gammas-on-GEMM2 reduction of ops/fused_moe.py:203,224-231.
// `out_scale` (1: none) multiplies the rounded output (scaled_bf16_bits).
__global__ __launch_bounds__(256) void moe_sum_kernel(
    const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int64_t m,
    int topk, int64_t k, const int32_t* __restrict__ ids, int num_experts,
    const float* __restrict__ weights, float out_scale) {
  const int64_t vec_per_row = k / 8;
  const int64_t total = m * vec_per_row;
  for (int64_t v = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
       v < total; v += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t t = v / vec_per_row;
    const int64_t c = (v - t * vec_per_row) * 8;
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    const uint16_t* src = in + t * topk * k + c;
    for (int j = 0; j < topk; ++j) {
      if (ids) {
        const int e = ids[t * topk + j];
        if (e < 0 || e >= num_experts) continue;
      }
      const u32x4 x = *reinterpret_cast<const u32x4*>(src + j * k);
      if (weights) {
        const float w = weights[t * topk + j];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          acc[2 * q] = __fadd_rn(acc[2 * q], __fmul_rn(w, __uint_as_float(x[q] << 16)));
          acc[2 * q + 1] =
              __fadd_rn(acc[2 * q + 1], __fmul_rn(w, __uint_as_float(x[q] & 0xffff0000u)));
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          acc[2 * q] += __uint_as_float(x[q] << 16);
          acc[2 * q + 1] += __uint_as_float(x[q] & 0xffff0000u);
        }
      }
    }
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = scaled_bf16x2(acc[2 * q], acc[2 * q + 1], out_scale);
    *reinterpret_cast<u32x4*>(out + t * k + c) = o;
  }
}

// moe_sum_kernel for a compile-time top-k: a thread issues its TK row loads
// before any of the dropped-slot checks (a runtime loop with a `continue`
// keeps each load behind the previous slot's check: TK round trips in
// series), then sums in slot order with the same roundings. Every slot has a
// row in `in`, so the loads stay in bounds whatever the ids say. The output
// scale is a template case: with the test for it in the unscaled kernel, whose
// latency it is (eight slots, 1 to 1000 tokens), the first slot's row was
// loaded last: 2.58 -> 2.81 us at one token.
template <int TK, bool SCALED>
__global__ __launch_bounds__(256) void moe_sum_tk_kernel(
    const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int64_t m,
    int64_t k, const int32_t* __restrict__ ids, int num_experts,
    const float* __restrict__ weights, float out_scale) {
  const int64_t vec_per_row = k / 8;
  const int64_t total = m * vec_per_row;
  for (int64_t v = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
       v < total; v += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t t = v / vec_per_row;
    const int64_t c = (v - t * vec_per_row) * 8;
    const uint16_t* src = in + t * TK * k + c;
    u32x4 x[TK];
#pragma unroll
    for (int j = 0; j < TK; ++j) x[j] = *reinterpret_cast<const u32x4*>(src + j * k);
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < TK; ++j) {
      if (ids) {
        const int e = ids[t * TK + j];
        if (e < 0 || e >= num_experts) continue;
      }
      if (weights) {
        const float w = weights[t * TK + j];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          acc[2 * q] = __fadd_rn(acc[2 * q], __fmul_rn(w, __uint_as_float(x[j][q] << 16)));
          acc[2 * q + 1] =
              __fadd_rn(acc[2 * q + 1], __fmul_rn(w, __uint_as_float(x[j][q] & 0xffff0000u)));
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          acc[2 * q] += __uint_as_float(x[j][q] << 16);
          acc[2 * q + 1] += __uint_as_float(x[j][q] & 0xffff0000u);
        }
      }
    }
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      o[q] = SCALED ? scaled_bf16x2(acc[2 * q], acc[2 * q + 1], out_scale)
                    : pack_bf16x2(acc[2 * q], acc[2 * q + 1]);
    *reinterpret_cast<u32x4*>(out + t * k + c) = o;
  }
}

// moe_sum over fp32 split-K partials: 4 columns per thread.
__global__ __launch_bounds__(256) void moe_sum_partials_kernel(
    const float* __restrict__ part, int nsplit, uint16_t* __restrict__ out,
    int64_t m, int topk, int64_t k, const int32_t* __restrict__ ids,
    int num_experts, const float* __restrict__ weights, float out_scale) {
  const int64_t vec_per_row = k / 4;
  const int64_t total = m * vec_per_row;
  const int64_t split_stride = m * topk * k;
  for (int64_t v = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
       v < total; v += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t t = v / vec_per_row;
    const int64_t c = (v - t * vec_per_row) * 4;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < topk; ++j) {
      const int64_t slot = t * topk + j;
      const int e = ids[slot];
      if (e < 0 || e >= num_experts) continue;
      f32x4 y = *reinterpret_cast<const f32x4*>(part + slot * k + c);
      for (int s = 1; s < nsplit; ++s)
        y += *reinterpret_cast<const f32x4*>(part + s * split_stride + slot * k + c);
      const float w = weights ? weights[slot] : 1.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float yb = bf16_bits_to_f32(f32_to_bf16_bits(y[q]));
        acc[q] = weights ? __fadd_rn(acc[q], __fmul_rn(w, yb)) : acc[q] + yb;
      }
    }
    uint2 o;
    o.x = scaled_bf16x2(acc[0], acc[1], out_scale);
    o.y = scaled_bf16x2(acc[2], acc[3], out_scale);
    *reinterpret_cast<uint2*>(out + t * k + c) = o;
  }
}

// --------------------------------------------------------- quantisers ---
// x / scale correctly rounded for a finite scale, from inv = 1 / scale
// (correctly rounded, one division for all of a scale's values): Markstein's
// scheme (P. Markstein, "Computation of elementary functions on the IBM RISC
// System/6000 processor", IBM J. Res. Dev. 1990): x * inv is within two ulps,
// one residual step brings it within one, and a second from there, with a
// correctly rounded reciprocal, gives the rounded quotient (and, with x's
// sign, its signed zero). Six FMA-rate instructions in place of a division's
// ten and its reciprocal; the quantisers were bound by those. Exact where the
// residuals are: a quotient small enough for one to lose bits rounds to code 0
// either way.
__device__ __forceinline__ float quotient(float x, float scale, float inv) {
  float q = x * inv;
  q = __builtin_fmaf(__builtin_fmaf(-scale, q, x), inv, q);
  q = __builtin_fmaf(__builtin_fmaf(-scale, q, x), inv, q);
  return __builtin_copysignf(q, x);
}

// The scale for quotient's residuals: itself, or zero for an infinite one (an
// infinity in the row or group), with which a finite x gives its signed zero
// and an infinity NaN, as the division does. (With a division as the other
// branch, per value: int8, 20000 rows of 128 columns 10.2 us, 7.3 so, 1024 of
// 8192 12.6 and 9.9, one of 14336 6.0 and 5.2; divisions alone 8.1, 11.4, 5.7.)
__device__ __forceinline__ float residual_scale(float scale) {
  return scale < INFINITY ? scale : 0.f;
}

// The row of x a quantiser's work item `i` takes: i, or the padded row given
// for it (-1: none).
__device__ __forceinline__ int64_t quant_row(const int32_t* row_of, int64_t i,
                                             int64_t row_limit) {
  if (!row_of) return i;
  const int64_t r = row_of[i];
  return r < row_limit ? r : -1;
}

// ------------------------------------------------------ fp8 group quant ---
// Each lane quantises 8 consecutive columns; the group/8 lanes of a group
// (a power of two <= 64, aligned within the wave) reduce its amax with
// butterfly shuffles, so a wave covers 512 columns. A workgroup takes
// 2048 columns of one row (grid: rows x column chunks), so the row and its
// skip test are uniform and no index is divided.
// scale = max(amax, 1e-10) / 448; q = e4m3fn(clamp(x / scale, +-448)).
// Measured (with a division per value, and padded rows a workgroup each,
// before): 16384 rows of 2048 22.0 -> 20.1 us (5.0 TB/s); DeepSeek M=4096's
// GEMM1 output, 32768 live rows of 98048, 76 -> 56 us.
constexpr int kQuantChunkCols = 256 * 8;  // columns per workgroup
__global__ __launch_bounds__(256) void quant_fp8_group_kernel(
    const uint16_t* __restrict__ x, uint8_t* __restrict__ q,
    float* __restrict__ scales, int64_t cols, int group,
    const int32_t* __restrict__ row_of, int64_t row_limit, int64_t scale_kstride) {
  const int lane = threadIdx.x & 63;
  const int lanes_per_group = group / 8;
  const int64_t r = quant_row(row_of, blockIdx.x, row_limit);
  if (r < 0) return;
  const int64_t c = (static_cast<int64_t>(blockIdx.y) * kQuantChunkCols) + threadIdx.x * 8;
  // a group lies wholly inside or outside the row (cols % group == 0)
  const bool active = c < cols;
  float f[8];
  float amax = 0.f;
  if (active) {
    const u32x4 w = *reinterpret_cast<const u32x4*>(x + r * cols + c);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f[2 * j] = __uint_as_float(w[j] << 16);
      f[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(f[j]));
  }
  for (int d = lanes_per_group / 2; d >= 1; d >>= 1)
    amax = fmaxf(amax, __shfl_xor(amax, d, 64));
  if (!active) return;
  const float scale = fmaxf(amax, 1e-10f) / 448.0f;
  const float inv = 1.0f / scale;
#pragma unroll
  for (int j = 0; j < 8; ++j) f[j] = quotient(f[j], residual_scale(scale), inv);
  uint32_t lo = 0, hi = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float a = fminf(fmaxf(f[2 * j], -448.f), 448.f);
    const float b = fminf(fmaxf(f[2 * j + 1], -448.f), 448.f);
    const uint32_t pk = cvt_pk_fp8(a, b);
    if (j < 2)
      lo |= pk << (16 * j);
    else
      hi |= pk << (16 * (j - 2));
  }
  uint2 o;
  o.x = lo;
  o.y = hi;
  *reinterpret_cast<uint2*>(q + r * cols + c) = o;
  if ((lane & (lanes_per_group - 1)) == 0) {
    const int gshift = __builtin_ctz(group);  // group is a power of two
    const int64_t g = c >> gshift;
    if (scale_kstride > 0) scales[g * scale_kstride + r] = scale;
    else scales[r * (cols >> gshift) + g] = scale;
  }
}

// Activation scales of the padded row order, k-block-major:
// out[kb * stride + r] = xs[sorted_ids[r] / topk][kb] for the rows below
// num_tokens_post_padded; a pad row takes the block's first row's scales
// (any finite value does: pad rows' outputs are never stored). A thread takes
// kGatherBlocks k blocks of one padded row, read V at a time (V = 4: 64
// consecutive bytes of the token's scales, where kblocks % 4 == 0 keeps them
// 16-byte aligned); a wave's writes of each k block are 64 consecutive rows.
// One k block per thread read the row order, divided by topk and touched a
// line of scales once per value: 98048 padded rows of 56 k blocks, 15 -> 8.3 us.
constexpr int kGatherBlocks = 16;
template <int V>
__global__ __launch_bounds__(256) void moe_scale_gather_kernel(
    const float* __restrict__ xs, int kblocks, const int32_t* __restrict__ sorted_ids,
    const int32_t* __restrict__ num_post_pad, int64_t numel, int topk, int block,
    float* __restrict__ out, int64_t stride) {
  typedef float vec __attribute__((ext_vector_type(V)));
  const int64_t r = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (r >= num_post_pad[0]) return;
  int sid = sorted_ids[r];
  if (sid >= numel) sid = sorted_ids[r - r % block];
  const float* row = xs + static_cast<int64_t>(sid / topk) * kblocks;
  const int kb0 = blockIdx.y * kGatherBlocks;
#pragma unroll
  for (int q = 0; q < kGatherBlocks; q += V) {
    const int kb = kb0 + q;
    if (kb >= kblocks) return;
    const vec v = *reinterpret_cast<const vec*>(row + kb);
#pragma unroll
    for (int j = 0; j < V; ++j) out[(kb + j) * stride + r] = v[j];
  }
}

// ----------------------------------------------------- int8 token quant ---
constexpr int64_t kInt8WaveRows = 1024;  // rows from which a wave takes a row
// Eight values of a row -> int8 codes rne(x / scale) clamped to +-127
// (`scale`: residual_scale's).
__device__ __forceinline__ uint2 quant_int8x8(const u32x4& w, float scale, float inv) {
  uint32_t packed[2] = {0, 0};
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float f = (j & 1) ? __uint_as_float(w[j / 2] & 0xffff0000u)
                            : __uint_as_float(w[j / 2] << 16);
    float rq = __builtin_rintf(quotient(f, scale, inv));
    rq = fminf(fmaxf(rq, -127.f), 127.f);
    const uint32_t b = static_cast<uint32_t>(static_cast<int32_t>(rq)) & 0xffu;
    packed[j / 4] |= b << (8 * (j & 3));
  }
  return uint2{packed[0], packed[1]};
}

// One wave per row (4 rows per workgroup), the row held in registers: NV
// vectors of 8 columns per lane (cols <= 512 * NV, cols % 8 == 0), one read
// of x. scale = max(amax, 1e-10) / 127; q = clamp(rne(x / scale), -127, 127).
// Measured as above: 8192 rows of 3584 32.8 -> 27.2 us; Qwen2 M=8192's GEMM1
// output, 65536 rows of 2560, 109 -> 97 us (5.2 TB/s), M=64's 512 live rows
// of 8640 15.4 -> 5.2 us (a workgroup per row).
template <int NV>
__global__ __launch_bounds__(256) void quant_int8_token_kernel(
    const uint16_t* __restrict__ x, int8_t* __restrict__ q,
    float* __restrict__ scales, int64_t rows, int64_t cols,
    const int32_t* __restrict__ row_of, int64_t row_limit) {
  const int lane = threadIdx.x & 63;
  const int64_t item = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item >= rows) return;
  const int64_t r = quant_row(row_of, item, row_limit);
  if (r < 0) return;
  const uint16_t* src = x + r * cols;
  int8_t* dst = q + r * cols;
  u32x4 w[NV];
  float amax = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int64_t c = (static_cast<int64_t>(v) * 64 + lane) * 8;
    if (c < cols) {
      w[v] = *reinterpret_cast<const u32x4*>(src + c);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        amax = fmaxf(amax, fabsf(__uint_as_float(w[v][j] << 16)));
        amax = fmaxf(amax, fabsf(__uint_as_float(w[v][j] & 0xffff0000u)));
      }
    }
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) amax = fmaxf(amax, __shfl_xor(amax, d, 64));
  const float scale = fmaxf(amax, 1e-10f) / 127.0f;
  const float inv = 1.0f / scale, res = residual_scale(scale);
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int64_t c = (static_cast<int64_t>(v) * 64 + lane) * 8;
    if (c < cols) *reinterpret_cast<uint2*>(dst + c) = quant_int8x8(w[v], res, inv);
  }
  if (lane == 0) scales[r] = scale;
}

// ------------------------------------------------------------- launchers ---
static unsigned grid_for(int64_t work_items, int threads) {
  int64_t g = (work_items + threads - 1) / threads;
  const int64_t cap = 256 * 64;  // enough waves to fill 256 CUs many times
  if (g > cap) g = cap;
  if (g < 1) g = 1;
  return static_cast<unsigned>(g);
}

int launch_silu_and_mul(const void* in, void* out, int64_t rows, int64_t n,
                        hipStream_t stream) {
  if (rows == 0) return FGS_OK;
  hipLaunchKernelGGL(silu_and_mul_kernel, dim3(grid_for(rows * (n / 8), 256)),
                     dim3(256), 0, stream, static_cast<const uint16_t*>(in),
                     static_cast<uint16_t*>(out), rows, n);
  return check_launch("silu_and_mul_kernel");
}

int launch_moe_sum(const void* in, void* out, int64_t m, int topk, int64_t k,
                   hipStream_t stream) {
  return launch_moe_sum_routed(in, out, m, topk, k, nullptr, 0, nullptr, stream);
}

int launch_moe_sum_routed(const void* in, void* out, int64_t m, int topk,
                          int64_t k, const int32_t* ids, int num_experts,
                          const float* weights, hipStream_t stream, float out_scale) {
  if (m == 0) return FGS_OK;
  const dim3 grid(grid_for(m * (k / 8), 256));
  const uint16_t* src = static_cast<const uint16_t*>(in);
  uint16_t* dst = static_cast<uint16_t*>(out);
  if (topk == 8 || topk == 2) {
    const bool scaled = out_scale != 1.f;
    auto kernel = topk == 8 ? (scaled ? moe_sum_tk_kernel<8, true> : moe_sum_tk_kernel<8, false>)
                            : (scaled ? moe_sum_tk_kernel<2, true> : moe_sum_tk_kernel<2, false>);
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, src, dst, m, k, ids, num_experts,
                       weights, out_scale);
    return check_launch("moe_sum_tk_kernel");
  }
  hipLaunchKernelGGL(moe_sum_kernel, dim3(grid_for(m * (k / 8), 256)),
                     dim3(256), 0, stream, static_cast<const uint16_t*>(in),
                     static_cast<uint16_t*>(out), m, topk, k, ids, num_experts,
                     weights, out_scale);
  return check_launch("moe_sum_kernel");
}

int launch_moe_sum_partials(const float* part, int nsplit, void* out, int64_t m,
                            int topk, int64_t k, const int32_t* ids,
                            int num_experts, const float* weights,
                            hipStream_t stream, float out_scale) {
  if (m == 0) return FGS_OK;
  hipLaunchKernelGGL(moe_sum_partials_kernel, dim3(grid_for(m * (k / 4), 256)),
                     dim3(256), 0, stream, part, nsplit,
                     static_cast<uint16_t*>(out), m, topk, k, ids, num_experts,
                     weights, out_scale);
  return check_launch("moe_sum_partials_kernel");
}

// Few rows (under kInt8WaveRows): a workgroup of 256 threads per row, two
// passes over the row (amax, then quantise), for parallelism at small M.
__global__ __launch_bounds__(256) void quant_int8_token_wg_kernel(
    const uint16_t* __restrict__ x, int8_t* __restrict__ q,
    float* __restrict__ scales, int64_t cols, const int32_t* __restrict__ row_of,
    int64_t row_limit) {
  const int64_t r = quant_row(row_of, blockIdx.x, row_limit);
  if (r < 0) return;
  const uint16_t* src = x + r * cols;
  int8_t* dst = q + r * cols;
  float amax = 0.f;
  for (int64_t c = threadIdx.x * 8; c < cols; c += 256 * 8) {
    const u32x4 w = *reinterpret_cast<const u32x4*>(src + c);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      amax = fmaxf(amax, fabsf(__uint_as_float(w[j] << 16)));
      amax = fmaxf(amax, fabsf(__uint_as_float(w[j] & 0xffff0000u)));
    }
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) amax = fmaxf(amax, __shfl_xor(amax, d, 64));
  __shared__ float red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float scale = fmaxf(amax, 1e-10f) / 127.0f;
  const float inv = 1.0f / scale, res = residual_scale(scale);
  for (int64_t c = threadIdx.x * 8; c < cols; c += 256 * 8)
    *reinterpret_cast<uint2*>(dst + c) =
        quant_int8x8(*reinterpret_cast<const u32x4*>(src + c), res, inv);
  if (threadIdx.x == 0) scales[r] = scale;
}

// Calls f(std::integral_constant<int, n>) for a runtime n in [0, N].
template <int N, class F>
static void dispatch_nv(int n, F&& f) {
  if constexpr (N >= 0) {
    if (n == N) {
      f(std::integral_constant<int, N>{});
      return;
    }
    dispatch_nv<N - 1>(n, f);
  }
}

int launch_quant_fp8_group(const void* x, void* q, float* scales,
                           int64_t rows, int64_t cols, int group,
                           hipStream_t stream, const int32_t* row_of, int64_t row_limit,
                           int64_t scale_kstride) {
  if (rows == 0 || cols == 0) return FGS_OK;
  const int64_t chunks = (cols + kQuantChunkCols - 1) / kQuantChunkCols;
  if (rows > 0x7fffffff || chunks > 0xffff)
    return fail(FGS_EUNSUPPORTED, "fp8 group quantiser: too many rows or columns for its grid");
  hipLaunchKernelGGL(quant_fp8_group_kernel,
                     dim3(static_cast<unsigned>(rows), static_cast<unsigned>(chunks)),
                     dim3(256), 0, stream, static_cast<const uint16_t*>(x),
                     static_cast<uint8_t*>(q), scales, cols, group, row_of, row_limit,
                     scale_kstride);
  return check_launch("quant_fp8_group_kernel");
}

int launch_scale_gather(const float* xs, int kblocks, const int32_t* sorted_ids,
                        const int32_t* num_post_pad, int64_t numel, int topk, int block,
                        int64_t max_padded, float* out, hipStream_t stream) {
  if (max_padded <= 0 || kblocks <= 0) return FGS_OK;
  const dim3 grid(static_cast<unsigned>((max_padded + 255) / 256),
                  static_cast<unsigned>((kblocks + kGatherBlocks - 1) / kGatherBlocks));
  auto kernel = kblocks % 4 == 0 ? moe_scale_gather_kernel<4> : moe_scale_gather_kernel<1>;
  hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, xs, kblocks, sorted_ids, num_post_pad,
                     numel, topk, block, out, max_padded);
  return check_launch("moe_scale_gather_kernel");
}

int launch_quant_int8_token(const void* x, int8_t* q, float* scales,
                            int64_t rows, int64_t cols, hipStream_t stream,
                            const int32_t* row_of, int64_t row_limit) {
  if (rows == 0) return FGS_OK;
  const uint16_t* xs = static_cast<const uint16_t*>(x);
  // rows too wide for a wave's registers take the workgroup-per-row kernel
  if (rows < kInt8WaveRows || cols > 512 * kInt8QuantMaxVec) {
    hipLaunchKernelGGL(quant_int8_token_wg_kernel, dim3(static_cast<unsigned>(rows)),
                       dim3(256), 0, stream, xs, q, scales, cols, row_of, row_limit);
    return check_launch("quant_int8_token_wg_kernel");
  }
  const dim3 grid(static_cast<unsigned>((rows + 3) / 4));
  const int nv = static_cast<int>((cols + 511) / 512);
  bool launched = false;
  dispatch_nv<kInt8QuantMaxVec>(nv, [&](auto nv_c) {
    constexpr int NV = decltype(nv_c)::value;
    if constexpr (NV >= 1) {
      hipLaunchKernelGGL(quant_int8_token_kernel<NV>, grid, dim3(256), 0, stream, xs, q,
                         scales, rows, cols, row_of, row_limit);
      launched = true;
    }
  });
  if (!launched) return fail(FGS_EINVAL, "int8 token quantiser: bad column count");
  return check_launch("quant_int8_token_kernel");
}

}  // namespace fgs
