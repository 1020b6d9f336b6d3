// Cross-entropy over a vocabulary processed in column chunks, so the
// [tokens, vocab] logits never exist at once (the last pipeline stage's
// output layer + loss).
//
// zk_ce_fwd_chunk: for each row of a [rows, cols] chunk of logits (columns
// col0 .. col0 + cols of the vocabulary) update a running maximum m and a
// running sum s of exp(l - m) (online log-sum-exp, fp32), and record the
// label's logit when the label falls inside the chunk.
// zk_ce_bwd_chunk: overwrite the chunk with d loss / d logits =
// scale * (exp(l - lse) - [j == label]), rounded to the storage type.
// Rows whose label is negative (ignore_index) contribute nothing.
//
// One workgroup per row; each thread covers 8 consecutive columns per access
// (16-byte accesses for 2-byte types; the forward has four in flight and takes
// one rescale for the 32 values) and the row reductions use wave shuffles plus
// one LDS exchange.  Both passes are bound by HBM: 4096 rows of 49152 bf16
// columns (403 MB) take 81 us forward with exp_neg, 103 with expf and 107 with
// one access in flight besides, 76 with exp_neg's first line alone (2046 rows
// that the product has just left in the last-level cache 50, 40 with that); 2046
// rows 66 us backward (402 MB).
//
// zk_ce_labels and zk_ce_finish are what precedes and follows the chunks, one
// workgroup each up to kOneGroup rows: checked row labels, the number of valid rows and the initial
// accumulators; the rows' log-sum-exp and the mean loss.  As tensor operations
// they were 30 launches of 2 to 5 us and two waits of the host for the device (a
// head of 2046 tokens, 1536 wide, 49152 columns: 1098 us against 931).  One wait
// is left, for the label check before any logits are allocated; with the check
// read after the products the same head took 910.
#include "vec.h"

namespace zk {

// e^x for x <= 0 (0 for -inf, NaN for NaN): 2^p, p = x log2(e) rounded, times
// 1 + r for what the rounding left out, r = x - p ln(2).  Without r it is off by
// |p| 2^-25, several ulps at x = -10.  expf, which reduces p to its fraction and
// scales back, takes twice the instructions.  Largest and rms error of a sum
// dominated by e^-5.6 to e^-8: 9.3e-8 and 3.1e-8, with expf 8.8e-8 and 3.0e-8,
// without r 3.1e-7 and 1.0e-7 (of one sign on average).  r is kept in [-1, 1] so
// that 0 times it stays 0 where p is -inf.
__device__ __forceinline__ float exp_neg(float x) {
  constexpr float kLog2e = 1.4426950408889634f, kLn2 = 0.693147180559945309f;
  constexpr float kLn2Lo = static_cast<float>(0.693147180559945309 - kLn2);
  const float p = x * kLog2e, w = __builtin_amdgcn_exp2f(p);
  const float r = fmaf(-p, kLn2Lo, fmaf(-p, kLn2, x));
  return fmaf(w, __builtin_amdgcn_fmed3f(r, -1.0f, 1.0f), w);
}

template <int NT>
__device__ __forceinline__ void block_max_sum(float& m, float& s, float* red) {
  // combine (max, sum-of-exp relative to max) pairs across the workgroup
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float om = __shfl_xor(m, off, 64);
    const float os = __shfl_xor(s, off, 64);
    const float nm = fmaxf(m, om);
    s = (m == -INFINITY ? 0.f : s * expf(m - nm)) + (om == -INFINITY ? 0.f : os * expf(om - nm));
    m = nm;
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) {
    red[2 * wave] = m;
    red[2 * wave + 1] = s;
  }
  __syncthreads();
  m = -INFINITY;
  s = 0.f;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) {
    const float om = red[2 * w], os = red[2 * w + 1];
    const float nm = fmaxf(m, om);
    s = (m == -INFINITY ? 0.f : s * expf(m - nm)) + (om == -INFINITY ? 0.f : os * expf(om - nm));
    m = nm;
  }
}

template <typename T, int NT>
__global__ __launch_bounds__(NT) void ce_fwd_chunk(const T* __restrict__ logits, int64_t cols,
                                                   int64_t ld, const int64_t* __restrict__ labels,
                                                   int64_t col0, float* __restrict__ run_max,
                                                   float* __restrict__ run_sum,
                                                   float* __restrict__ target) {
  __shared__ float red[2 * (NT / 64)];
  const int64_t row = blockIdx.x;
  const T* lr = logits + row * ld;
  const bool vec = (cols % 8) == 0;
  float m = -INFINITY, s = 0.f;
  if (vec) {
    constexpr int U = 4;
    for (int64_t c = threadIdx.x * 8; c < cols; c += U * NT * 8) {
      float v[U][8];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (c + u * NT * 8 < cols) {
          Vec8<T>::load(lr + c + u * NT * 8, v[u]);
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) v[u][i] = -INFINITY;
        }
      }
      float nm = m;
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < 8; ++i) nm = fmaxf(nm, v[u][i]);
      if (nm == -INFINITY) continue;  // nothing but -inf so far
      float acc = m == -INFINITY ? 0.f : s * exp_neg(m - nm);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc += exp_neg(v[u][i] - nm);
      s = acc;
      m = nm;
    }
  } else {
    for (int64_t c = threadIdx.x; c < cols; c += NT) {
      const float v = to_f32(lr[c]);
      const float nm = fmaxf(m, v);
      s = (m == -INFINITY ? 0.f : s * expf(m - nm)) + expf(v - nm);
      m = nm;
    }
  }
  block_max_sum<NT>(m, s, red);
  if (threadIdx.x == 0) {
    const int64_t lab = labels[row];
    if (lab >= col0 && lab < col0 + cols) target[row] = to_f32(lr[lab - col0]);
    const float om = run_max[row], os = run_sum[row];
    const float nm = fmaxf(m, om);
    run_sum[row] = (m == -INFINITY ? 0.f : s * expf(m - nm)) +
                   (om == -INFINITY ? 0.f : os * expf(om - nm));
    run_max[row] = nm;
  }
}

template <typename T, int NT>
__global__ __launch_bounds__(NT) void ce_bwd_chunk(T* __restrict__ logits, int64_t cols, int64_t ld,
                                                   const int64_t* __restrict__ labels, int64_t col0,
                                                   const float* __restrict__ lse, float scale,
                                                   const float* __restrict__ grad,
                                                   const int64_t* __restrict__ n_valid) {
  const int64_t row = blockIdx.x;
  // scale, or the mean's share of the loss gradient from device memory
  if (grad != nullptr) scale = *grad / static_cast<float>(*n_valid > 1 ? *n_valid : 1);
  T* lr = logits + row * ld;
  const int64_t lab = labels[row];
  const float l0 = lse[row];
  const float sc = lab < 0 ? 0.f : scale;
  if ((cols % 8) == 0) {
    for (int64_t c = threadIdx.x * 8; c < cols; c += NT * 8) {
      float v[8];
      Vec8<T>::load(lr + c, v);
#pragma unroll
      for (int i = 0; i < 8; ++i)
        v[i] = lab < 0 ? 0.f : sc * (expf(v[i] - l0) - (col0 + c + i == lab ? 1.f : 0.f));
      Vec8<T>::store(lr + c, v);
    }
  } else {
    for (int64_t c = threadIdx.x; c < cols; c += NT) {
      const float v = to_f32(lr[c]);
      lr[c] = from_f32<T>(lab < 0 ? 0.f : sc * (expf(v - l0) - (col0 + c == lab ? 1.f : 0.f)));
    }
  }
}

// Sum of x over a 1024-thread workgroup, in every thread.
template <typename U>
__device__ __forceinline__ U block_sum_1024(U x, U* red) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  U t = red[0];
#pragma unroll
  for (int w = 1; w < 16; ++w) t += red[w];
  return t;
}

// One workgroup moves 80 GB/s: 262144 rows took 94 us for the labels, 11 this way.
// More rows than the two ways take alike go to a workgroup per kGroupRows and a
// second launch for the totals (integer counts; float sums in the groups' order).
constexpr int64_t kOneGroup = 16384, kGroupRows = 4096;

__global__ __launch_bounds__(1024) void ce_labels_kernel(
    const int64_t* __restrict__ labels, int64_t rows, int64_t vocab, int64_t ignore,
    int64_t* __restrict__ row_label, float* __restrict__ run_max, float* __restrict__ run_sum,
    float* __restrict__ target, int64_t* __restrict__ stats, int64_t* __restrict__ host_stats) {
  __shared__ int red[16];
  int valid = 0, bad = 0;
  const int64_t first = blockIdx.x * kGroupRows;
  const int64_t end = gridDim.x == 1 || first + kGroupRows > rows ? rows : first + kGroupRows;
  for (int64_t i = first + threadIdx.x; i < end; i += 1024) {
    const int64_t l = labels[i];
    const bool skip = l == ignore;
    valid += !skip;
    bad += !skip && (l < 0 || l >= vocab);
    row_label[i] = skip ? -1 : l;
    run_max[i] = -INFINITY;
    run_sum[i] = 0.f;
    target[i] = 0.f;
  }
  valid = block_sum_1024(valid, red);
  bad = block_sum_1024(bad, red);
  if (threadIdx.x == 0 && gridDim.x > 1) {
    unsigned long long* const total = reinterpret_cast<unsigned long long*>(stats);
    atomicAdd(total, static_cast<unsigned long long>(valid));
    atomicAdd(total + 1, static_cast<unsigned long long>(bad));
  } else if (threadIdx.x == 0) {
    stats[0] = valid;
    stats[1] = bad;
    host_stats[0] = valid;
    host_stats[1] = bad;
  }
}

// stats = {0, 0}, or its copy to the host.
__global__ void ce_stats_kernel(int64_t* stats, int64_t* host_stats) {
  if (host_stats == nullptr)
    stats[threadIdx.x] = 0;
  else
    host_stats[threadIdx.x] = stats[threadIdx.x];
}

// A workgroup of several leaves its sum in run_max at its first row.
__global__ __launch_bounds__(1024) void ce_finish_kernel(
    const int64_t* __restrict__ row_label, int64_t rows, float* run_max,
    const float* __restrict__ run_sum, const float* __restrict__ target,
    const int64_t* __restrict__ stats, float* __restrict__ lse, float* __restrict__ loss) {
  __shared__ float red[16];
  float sum = 0.f;
  const int64_t first = blockIdx.x * kGroupRows;
  const int64_t end = gridDim.x == 1 || first + kGroupRows > rows ? rows : first + kGroupRows;
  for (int64_t i = first + threadIdx.x; i < end; i += 1024) {
    const float l = run_max[i] + logf(run_sum[i]);
    lse[i] = l;
    if (row_label[i] >= 0) sum += l - target[i];
  }
  sum = block_sum_1024(sum, red);  // (its barriers: every row is read)
  if (threadIdx.x != 0) return;
  if (gridDim.x > 1)
    run_max[first] = sum;
  else
    *loss = sum / static_cast<float>(stats[0] > 1 ? stats[0] : 1);
}

__global__ __launch_bounds__(1024) void ce_mean_kernel(const float* __restrict__ run_max,
                                                       int64_t groups,
                                                       const int64_t* __restrict__ stats,
                                                       float* __restrict__ loss) {
  __shared__ float red[16];
  float sum = 0.f;
  for (int64_t i = threadIdx.x; i < groups; i += 1024) sum += run_max[i * kGroupRows];
  sum = block_sum_1024(sum, red);
  if (threadIdx.x == 0) *loss = sum / static_cast<float>(stats[0] > 1 ? stats[0] : 1);
}

static unsigned row_groups(int64_t rows) {
  return rows <= kOneGroup ? 1 : static_cast<unsigned>((rows + kGroupRows - 1) / kGroupRows);
}

}  // namespace zk

using namespace zk;

extern "C" int zk_ce_labels(const int64_t* labels, int64_t rows, int64_t vocab, int64_t ignore_index,
                            int64_t* row_label, float* run_max, float* run_sum,
                            float* target_logit, int64_t* stats, int64_t* host_stats,
                            zk_stream_t stream) {
  ZK_REQUIRE(rows >= 0 && rows <= 0x7fffffff && vocab > 0, ZK_EINVAL, "zk_ce_labels: bad shape");
  ZK_REQUIRE(stats && host_stats &&
                 (rows == 0 || (labels && row_label && run_max && run_sum && target_logit)),
             ZK_EINVAL, "zk_ce_labels: null pointer");
  hipStream_t s = as_stream(stream);
  const unsigned groups = row_groups(rows);
  int64_t* const none = nullptr;
  if (groups > 1) hipLaunchKernelGGL(ce_stats_kernel, dim3(1), dim3(2), 0, s, stats, none);
  hipLaunchKernelGGL(ce_labels_kernel, dim3(groups), dim3(1024), 0, s, labels, rows, vocab,
                     ignore_index, row_label, run_max, run_sum, target_logit, stats, host_stats);
  if (groups > 1) hipLaunchKernelGGL(ce_stats_kernel, dim3(1), dim3(2), 0, s, stats, host_stats);
  return launch_status("zk_ce_labels");
}

extern "C" int zk_ce_finish(const int64_t* row_label, int64_t rows, float* run_max,
                            const float* run_sum, const float* target_logit,
                            const int64_t* stats, float* lse, float* loss, zk_stream_t stream) {
  ZK_REQUIRE(rows >= 0 && rows <= 0x7fffffff, ZK_EINVAL, "zk_ce_finish: bad shape");
  ZK_REQUIRE(stats && loss && (rows == 0 || (row_label && run_max && run_sum && target_logit && lse)),
             ZK_EINVAL, "zk_ce_finish: null pointer");
  hipStream_t s = as_stream(stream);
  const unsigned groups = row_groups(rows);
  hipLaunchKernelGGL(ce_finish_kernel, dim3(groups), dim3(1024), 0, s, row_label, rows, run_max,
                     run_sum, target_logit, stats, lse, loss);
  if (groups > 1)
    hipLaunchKernelGGL(ce_mean_kernel, dim3(1), dim3(1024), 0, s, run_max,
                       static_cast<int64_t>(groups), stats, loss);
  return launch_status("zk_ce_finish");
}

extern "C" int zk_ce_fwd_chunk(const void* logits, int64_t rows, int64_t cols, int64_t ld,
                               const int64_t* labels, int64_t col0, float* run_max,
                               float* run_sum, float* target_logit, int dtype,
                               zk_stream_t stream) {
  ZK_REQUIRE(valid_dtype(dtype), ZK_EDTYPE, "zk_ce_fwd_chunk: bad dtype %d", dtype);
  ZK_REQUIRE(rows >= 0 && cols > 0 && ld >= cols && col0 >= 0, ZK_EINVAL,
             "zk_ce_fwd_chunk: bad shape rows=%lld cols=%lld ld=%lld col0=%lld",
             (long long)rows, (long long)cols, (long long)ld, (long long)col0);
  ZK_REQUIRE(rows <= 0x7fffffff, ZK_EINVAL, "zk_ce_fwd_chunk: too many rows");
  if (rows == 0) return ZK_OK;
  ZK_REQUIRE(logits && labels && run_max && run_sum && target_logit, ZK_EINVAL,
             "zk_ce_fwd_chunk: null pointer");
  const bool vec_ok = cols % 8 == 0 && ld % 8 == 0 && aligned(logits, 16);
  ZK_REQUIRE(vec_ok || cols % 8 != 0, ZK_EALIGN,
             "zk_ce_fwd_chunk: logits must be 16-byte aligned with ld a multiple of 8");
  hipStream_t s = as_stream(stream);
  if (dtype == ZK_BF16)
    hipLaunchKernelGGL((ce_fwd_chunk<bf16, 256>), dim3(rows), dim3(256), 0, s, (const bf16*)logits,
                       cols, ld, labels, col0, run_max, run_sum, target_logit);
  else if (dtype == ZK_F16)
    hipLaunchKernelGGL((ce_fwd_chunk<f16, 256>), dim3(rows), dim3(256), 0, s, (const f16*)logits,
                       cols, ld, labels, col0, run_max, run_sum, target_logit);
  else
    hipLaunchKernelGGL((ce_fwd_chunk<float, 256>), dim3(rows), dim3(256), 0, s,
                       (const float*)logits, cols, ld, labels, col0, run_max, run_sum,
                       target_logit);
  return launch_status("zk_ce_fwd_chunk");
}

static int ce_bwd_impl(void* logits, int64_t rows, int64_t cols, int64_t ld,
                       const int64_t* labels, int64_t col0, const float* lse, float scale,
                       const float* grad, const int64_t* n_valid, int dtype, zk_stream_t stream) {
  ZK_REQUIRE(valid_dtype(dtype), ZK_EDTYPE, "zk_ce_bwd_chunk: bad dtype %d", dtype);
  ZK_REQUIRE(rows >= 0 && cols > 0 && ld >= cols && col0 >= 0, ZK_EINVAL,
             "zk_ce_bwd_chunk: bad shape rows=%lld cols=%lld ld=%lld col0=%lld",
             (long long)rows, (long long)cols, (long long)ld, (long long)col0);
  ZK_REQUIRE(rows <= 0x7fffffff, ZK_EINVAL, "zk_ce_bwd_chunk: too many rows");
  if (rows == 0) return ZK_OK;
  ZK_REQUIRE(logits && labels && lse, ZK_EINVAL, "zk_ce_bwd_chunk: null pointer");
  const bool vec_ok = cols % 8 == 0 && ld % 8 == 0 && aligned(logits, 16);
  ZK_REQUIRE(vec_ok || cols % 8 != 0, ZK_EALIGN,
             "zk_ce_bwd_chunk: logits must be 16-byte aligned with ld a multiple of 8");
  hipStream_t s = as_stream(stream);
  if (dtype == ZK_BF16)
    hipLaunchKernelGGL((ce_bwd_chunk<bf16, 256>), dim3(rows), dim3(256), 0, s, (bf16*)logits,
                       cols, ld, labels, col0, lse, scale, grad, n_valid);
  else if (dtype == ZK_F16)
    hipLaunchKernelGGL((ce_bwd_chunk<f16, 256>), dim3(rows), dim3(256), 0, s, (f16*)logits,
                       cols, ld, labels, col0, lse, scale, grad, n_valid);
  else
    hipLaunchKernelGGL((ce_bwd_chunk<float, 256>), dim3(rows), dim3(256), 0, s, (float*)logits,
                       cols, ld, labels, col0, lse, scale, grad, n_valid);
  return launch_status("zk_ce_bwd_chunk");
}

extern "C" int zk_ce_bwd_chunk(void* logits, int64_t rows, int64_t cols, int64_t ld,
                               const int64_t* labels, int64_t col0, const float* lse,
                               float scale, int dtype, zk_stream_t stream) {
  return ce_bwd_impl(logits, rows, cols, ld, labels, col0, lse, scale, nullptr, nullptr, dtype,
                     stream);
}

extern "C" int zk_ce_bwd_chunk_mean(void* logits, int64_t rows, int64_t cols, int64_t ld,
                                    const int64_t* labels, int64_t col0, const float* lse,
                                    const float* grad, const int64_t* n_valid, int dtype,
                                    zk_stream_t stream) {
  ZK_REQUIRE(grad && n_valid, ZK_EINVAL, "zk_ce_bwd_chunk_mean: null pointer");
  return ce_bwd_impl(logits, rows, cols, ld, labels, col0, lse, 0.f, grad, n_valid, dtype, stream);
}
