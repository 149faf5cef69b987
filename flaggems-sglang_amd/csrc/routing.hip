// Routing-format conversion for gfx950, both directions.
//
// (topk_weights, topk_ids) -> the triton_kernels routing tuple of the
// reference's _standard_topk_to_triton_kernels (src/flaggems_sglang/ops/
// fused_moe.py:119-146), block metadata included. The reference sorts each
// token's ids (:130-131), takes a stable argsort of the flattened ids (:134),
// its inverse (:135), the gathered weights (:136), a histogram (:137-139) and
// compute_expt_data_torch's tile tables (:140). Here the stable argsort is
// moe_align_block_size itself (align.hip: a bit-exact stable counting sort),
// run with block size 1 over E + 1 id classes:
//   classes 0..E-1: experts 0..E-1, class E: ids outside [0, E).
// Inside a class, slots stay in flat (token-major) order. Slots with ids
// outside [0, E) (not routed here) go behind expert E-1: matmul_ogs reads
// expert e's rows at gathered positions [token_offs_raw[e],
// token_offs_raw[e+1]) with token_offs_raw starting at 0, so they must not
// sit ahead of expert 0 (where the reference's argsort would put negative
// ids; its own callers never produce them).
//
// (The alignment takes the class of an outside id and writes the histogram as
// it sorts.) Then one launch, per sorted position q (slot s = sorted[q] of
// token t):
//   topk_indx[q] = t*k + rank of s's id among token t's ids (the index the
//                  reference's per-token sort gives the slot),
//   gate_indx[topk_indx[q]] = q, gate_scal[q] = topk_weights[s],
// and in its last workgroup, from the histogram, the tile tables for block_m
// in {16, 32, 64, 128}:
//   token_offs_raw[e]      = sum of hist below e (E + 1 entries),
//   token_offs_pad[B][e]   = sum of ceil(hist/B) below e (in tiles),
//   block_pid_map[B][tile] = (b << 16) | e for expert e's b-th tile, -1 past
//                            the last tile (max_tiles entries).
//
// The routing tuple -> what the grouped GEMMs consume (routing_order_kernel,
// the direction the reference's matmul_ogs calls take, :205-231): expert e's
// gathered positions [raw[e], raw[e] + hist[e]) of gather_indx.src_indx become
// its segment of the block-padded order, and each flat slot gets back its
// expert id and gate scale.
#include <algorithm>
#include <string>

#include "fgs_moe_kernels.h"

namespace fgs {

constexpr int kRoutingBlockMs[4] = {16, 32, 64, 128};
constexpr int kRoutingThreads = 1024;

// Inclusive sums of each thread's N values over the workgroup (a thread per
// value set, whole waves): wave scans by lane shuffles, then the waves'
// totals (one barrier each way). `add` must be associative. tmp: N x 16
// words.
template <int N, class F>
__device__ __forceinline__ void block_scan(uint32_t (&v)[N], uint32_t (*tmp)[16], F add) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    uint32_t o[N];
#pragma unroll
    for (int i = 0; i < N; ++i) o[i] = __shfl_up(v[i], d, kWave);
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (lane >= d) v[i] = add(o[i], v[i]);
  }
  __syncthreads();  // (an earlier scan's readers are done with tmp)
  if (lane == kWave - 1) {
#pragma unroll
    for (int i = 0; i < N; ++i) tmp[i][wave] = v[i];
  }
  __syncthreads();
  for (int w = 0; w < wave; ++w) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = add(tmp[i][w], v[i]);
  }
}

// The per-position outputs in all workgroups but the last, which derives the
// tables from the histogram: one thread per expert (num_experts < 1024),
// the five sums scanned together. Bound by launches and latency: as class,
// finish and table kernels of their own (the table kernel finding the
// histogram by binary search in the sorted classes, its sums by 100
// barriers) 4.7 + 4.8 + 18 us at 1024 tokens, top-8 of 64; this one launch 7.9.
__global__ __launch_bounds__(kRoutingThreads) void routing_finish_kernel(
    const int32_t* __restrict__ ids, const float* __restrict__ weights, int64_t numel, int topk,
    const int32_t* __restrict__ sorted, float* __restrict__ gate_scal,
    int32_t* __restrict__ topk_indx, int32_t* __restrict__ gate_indx, int num_experts,
    const int32_t* __restrict__ hist, int32_t* __restrict__ token_offs_raw,
    int32_t* __restrict__ token_offs_pad, int32_t* __restrict__ block_pid_map,
    int64_t max_tiles) {
  if (blockIdx.x + 1 < gridDim.x) {
    const int64_t q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (q >= numel) return;
    const int64_t s = sorted[q];
    const int64_t t = s / topk;
    const int j = static_cast<int>(s - t * topk);
    const int e = ids[s];
    int rank = 0;
    for (int jj = 0; jj < topk; ++jj) {
      const int o = ids[t * topk + jj];
      rank += (o < e || (o == e && jj < j)) ? 1 : 0;
    }
    const int32_t r = static_cast<int32_t>(t * topk + rank);
    topk_indx[q] = r;
    gate_indx[r] = static_cast<int32_t>(q);
    gate_scal[q] = weights[s];
    return;
  }
  __shared__ uint32_t tmp[5][16];
  __shared__ int incl[4][kRoutingThreads];
  const int e = threadIdx.x;
  const uint32_t h = e < num_experts ? static_cast<uint32_t>(hist[e]) : 0u;
  uint32_t v[5] = {h};
#pragma unroll
  for (int bi = 0; bi < 4; ++bi)
    v[bi + 1] = (h + kRoutingBlockMs[bi] - 1) / static_cast<uint32_t>(kRoutingBlockMs[bi]);
  block_scan(v, tmp, [](uint32_t a, uint32_t b) { return a + b; });
  if (e == 0) token_offs_raw[0] = 0;
  if (e < num_experts) token_offs_raw[e + 1] = static_cast<int32_t>(v[0]);
#pragma unroll
  for (int bi = 0; bi < 4; ++bi) {
    int32_t* pad = token_offs_pad + static_cast<int64_t>(bi) * (num_experts + 1);
    if (e == 0) pad[0] = 0;
    if (e < num_experts) pad[e + 1] = static_cast<int32_t>(v[bi + 1]);
    incl[bi][e] = static_cast<int>(v[bi + 1]);
  }
  __syncthreads();
  for (int bi = 0; bi < 4; ++bi) {
    const int total = incl[bi][num_experts - 1];
    int32_t* map = block_pid_map + static_cast<int64_t>(bi) * max_tiles;
    for (int64_t t = e; t < max_tiles; t += blockDim.x) {
      int32_t x = -1;
      if (t < total) {
        // expert of tile t: the first e with incl[e] > t
        int lo = 0, hi = num_experts - 1;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (incl[bi][mid] > t) hi = mid;
          else lo = mid + 1;
        }
        const int first = lo == 0 ? 0 : incl[bi][lo - 1];
        x = (static_cast<int32_t>(t - first) << 16) | lo;
      }
      map[t] = x;
    }
  }
}

int64_t routing_max_tiles(int64_t numel, int num_experts) {
  // compute_expt_data_torch's bound for the smallest block (16): at most
  // ceil((numel - E + 1) / 16) + E - 1 tiles, or numel when numel <= E
  if (numel <= num_experts) return numel;
  return (numel - num_experts + 1 + 15) / 16 + num_experts - 1;
}

int64_t routing_workspace_bytes(int64_t numel, int num_experts) {
  auto up = [](int64_t b) { return (b + 255) / 256 * 256; };
  // sorted positions, class per position, padded total, align scratch
  return 2 * up(numel * 4) + 256 + up(align_scratch_bytes(numel, num_experts + 1));
}

int launch_topk_to_routing(const float* weights, const int32_t* ids, int64_t m, int topk,
                           int num_experts, float* gate_scal, int32_t* topk_indx,
                           int32_t* gate_indx, int32_t* hist, int32_t* token_offs_raw,
                           int32_t* token_offs_pad, int32_t* block_pid_map,
                           int64_t max_tiles, void* workspace, hipStream_t stream) {
  const int64_t numel = m * topk;
  auto up = [](int64_t b) { return (b + 255) / 256 * 256; };
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  int32_t* sorted = reinterpret_cast<int32_t*>(ws);
  int32_t* cls_sorted = reinterpret_cast<int32_t*>(ws + up(numel * 4));
  int32_t* npp = reinterpret_cast<int32_t*>(ws + 2 * up(numel * 4));
  int32_t* scratch = align_scratch_bytes(numel, num_experts + 1) > 0
                         ? reinterpret_cast<int32_t*>(ws + 2 * up(numel * 4) + 256)
                         : nullptr;
  // block size 1: sorted holds every slot, cls_sorted its class, hist the
  // experts' counts (all zero without slots)
  int rc = launch_align(ids, numel, num_experts + 1, 1, sorted, cls_sorted, npp, numel, stream,
                        scratch, nullptr, nullptr, num_experts, hist);
  if (rc) return rc;
  const int blocks = static_cast<int>((numel + kRoutingThreads - 1) / kRoutingThreads) + 1;
  hipLaunchKernelGGL(routing_finish_kernel, dim3(blocks), dim3(kRoutingThreads), 0, stream, ids,
                     weights, numel, topk, sorted, gate_scal, topk_indx, gate_indx, num_experts,
                     hist, token_offs_raw, token_offs_pad, block_pid_map, max_tiles);
  return check_launch("routing_finish_kernel");
}

// ------------------------------------------------ routing tuple -> order ---
constexpr int kOrderThreads = 1024;  // one expert per thread (E <= 1024)

// First index i in [0, n) with incl[i] > x (incl non-decreasing; n when none).
__device__ __forceinline__ int first_above(const int32_t* incl, int n, int64_t x) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (incl[mid] > x) hi = mid;
    else lo = mid + 1;
  }
  return lo;
}

// Expert e reads gathered positions [raw[e], raw[e] + h[e]) with raw the
// exclusive sums of the histogram (token_offs_raw, as matmul_ogs reads
// them); h is the histogram clamped so every range stays inside [0, numel)
// (negative counts read as 0, sums past numel are cut at numel).
//   order (sorted_ids != null): sorted_ids[pad[e] + i] = src[raw[e] + i] for
//     i < h[e], numel elsewhere (pads, and src entries outside [0, numel));
//     pad[e] = exclusive sums of ceil(h / block) * block; expert_ids[b] = the
//     expert of padded row b * block, -1 past the padded total;
//     *num_post_pad = the padded total;
//   inverse (ids_out != null): for every gathered position p with
//     v = src[p] in [0, numel): ids_out[v] = the expert whose range holds p
//     (-1 past the histogram's total: a slot no expert reads),
//     w_out[v] = gate_scal[p];
//   rows (row_of != null, with the inverse): row_of[p] = p's padded row, -1
//     past the total and where src[p] is outside. By position, so all numel
//     entries are written and each row that holds a slot has its own, also
//     where a caller's src names a slot twice and another never.
// Every workgroup (one thread per expert: blockDim >= E, a power of two up
// to 1024) derives the offsets itself (by wave scans: 5.9 us at 8192 gates
// over 64 experts, 8.5 with 64-bit sums in LDS and a barrier per step) and
// then walks its share of the positions; no atomics, so the result is
// deterministic.
__global__ __launch_bounds__(kOrderThreads) void routing_order_kernel(
    const float* __restrict__ gate_scal, const int32_t* __restrict__ src,
    const int32_t* __restrict__ hist, int64_t numel, int num_experts, int block,
    int64_t max_padded, int32_t* __restrict__ sorted_ids, int32_t* __restrict__ expert_ids,
    int32_t* __restrict__ num_post_pad, int32_t* __restrict__ ids_out,
    float* __restrict__ w_out, int32_t* __restrict__ row_of) {
  __shared__ uint32_t tmp[1][16];
  __shared__ int32_t raw_incl[kOrderThreads];
  __shared__ int32_t pad_incl[kOrderThreads];
  const int e = threadIdx.x;
  const int E = num_experts;
  // counts clamped to [0, numel], sums to numel (below 2^31, so two of them
  // add in 32 bits; min(a + b, cap) is associative for values in [0, cap])
  const uint32_t cap = static_cast<uint32_t>(numel);
  uint32_t r[1] = {e < E ? min(static_cast<uint32_t>(max(hist[e], 0)), cap) : 0u};
  block_scan(r, tmp, [cap](uint32_t a, uint32_t b) { return min(a + b, cap); });
  raw_incl[e] = static_cast<int32_t>(r[0]);
  __syncthreads();
  const uint32_t hc = e < E ? r[0] - (e > 0 ? raw_incl[e - 1] : 0) : 0;
  uint32_t pc[1] = {(hc + block - 1) / block * block};
  block_scan(pc, tmp, [](uint32_t a, uint32_t b) { return a + b; });
  pad_incl[e] = static_cast<int32_t>(pc[0]);
  __syncthreads();
  const int64_t total_raw = raw_incl[E - 1];
  const int64_t total_pad = pad_incl[E - 1];

  const int64_t tid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  if (sorted_ids) {
    for (int64_t q = tid; q < max_padded; q += stride) {
      int32_t v = static_cast<int32_t>(numel);
      if (q < total_pad) {
        const int x = first_above(pad_incl, E, q);
        const int64_t i = q - (x > 0 ? pad_incl[x - 1] : 0);
        const int64_t r0 = x > 0 ? raw_incl[x - 1] : 0;
        if (i < raw_incl[x] - r0) {
          const int32_t s = src[r0 + i];
          if (s >= 0 && s < numel) v = s;
        }
      }
      sorted_ids[q] = v;
    }
    for (int64_t b = tid; b < max_padded / block; b += stride)
      expert_ids[b] = b * block < total_pad ? first_above(pad_incl, E, b * block) : -1;
    if (tid == 0) *num_post_pad = static_cast<int32_t>(total_pad);
  }
  if (ids_out) {
    for (int64_t p = tid; p < numel; p += stride) {
      const int32_t s = src[p];
      const bool named = s >= 0 && s < numel;
      const int x = p < total_raw ? first_above(raw_incl, E, p) : -1;
      if (row_of)
        row_of[p] = !named || x < 0 ? -1
                                    : (x > 0 ? pad_incl[x - 1] : 0) + static_cast<int32_t>(p) -
                                          (x > 0 ? raw_incl[x - 1] : 0);
      if (!named) continue;
      ids_out[s] = x;
      w_out[s] = gate_scal[p];
    }
  }
}

int launch_routing_order(const float* gate_scal, const int32_t* src, const int32_t* hist,
                         int64_t numel, int num_experts, int block, int64_t max_padded,
                         int32_t* sorted_ids, int32_t* expert_ids, int32_t* num_post_pad,
                         int32_t* ids_out, float* w_out, hipStream_t stream,
                         int32_t* row_of) {
  if (num_experts < 1 || num_experts > kOrderThreads)
    return fail(FGS_EINVAL, "routing order: num_experts must be in [1, 1024]");
  // one wave for up to 64 experts (its barriers cost next to nothing)
  int threads = 64;
  while (threads < num_experts) threads *= 2;
  const int64_t work = std::max<int64_t>(sorted_ids ? max_padded : 0, numel);
  const int blocks =
      static_cast<int>(std::min<int64_t>(std::max<int64_t>((work + threads - 1) / threads, 1), 1024));
  hipLaunchKernelGGL(routing_order_kernel, dim3(blocks), dim3(threads), 0, stream,
                     gate_scal, src, hist, numel, num_experts, block, max_padded, sorted_ids,
                     expert_ids, num_post_pad, ids_out, w_out, row_of);
  return check_launch("routing_order_kernel");
}

}  // namespace fgs
