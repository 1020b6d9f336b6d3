// Products whose tiles leave most CUs idle over a long reduction: the
// reduction is split over workgroups, each of which stores its partial sums in
// fp32, and one pass adds them (in order of the reduction), adds the residual
// and rounds once.
//
// Bound: a CU takes in its tiles' operands at about 55 GB/s, so a product with
// 32 tiles runs at an eighth of what 256 workgroups load; the partial sums cost
// 8 bytes an output and part.  The second launch takes 3.8 us for 64 x 4096 in 8
// parts, 5.0 for 256 x 4096 in 4, 9.7 for 1024 x 2688 in 5 and 10.9 for 2046 x
// 1536 in 5 (63 MB read, 5.8 TB/s), with no gap before it.
#include "gemm_ring.h"

namespace zk {
namespace gemm {

namespace {
template <typename T, bool BKM>
void launch_t(Tile t, int parts, const GemmArgs& ga, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(tile_count(t, ga.M, ga.N)), static_cast<unsigned>(parts));
  if (t == k256)
    hipLaunchKernelGGL((gemm_tiled_kernel<T, 3, false, BKM, true>), grid, dim3(256), 0, s, ga);
  else if (t == k128x2)
    hipLaunchKernelGGL((gemm_ring_kernel<T, 3, false, BKM, 4, 4, 4, 2, 2>), grid, dim3(512), 0, s,
                       ga);
  else
    hipLaunchKernelGGL((gemm_ring_kernel<T, 3, false, BKM, 2, 4, 4, 2, 2>), grid, dim3(512), 0, s,
                       ga);
}

// Four columns a thread; N is a multiple of 8 and rows 16-byte aligned.
template <typename T>
__global__ __launch_bounds__(256) void split_sum_kernel(const float* __restrict__ ws, int parts,
                                                        T* __restrict__ C, int64_t ldc,
                                                        const T* __restrict__ R, int64_t ldr,
                                                        int64_t M, int64_t N) {
  typedef T T4 __attribute__((ext_vector_type(4)));
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i >= M * N) return;
  const int64_t row = i / N, col = i - row * N;
  float4 v = *reinterpret_cast<const float4*>(ws + i);
#pragma unroll 4
  for (int p = 1; p < parts; ++p) {
    const float4 w = *reinterpret_cast<const float4*>(ws + p * M * N + i);
    v.x += w.x;
    v.y += w.y;
    v.z += w.z;
    v.w += w.w;
  }
  if (R != nullptr) {
    const T4 r = *reinterpret_cast<const T4*>(R + row * ldr + col);
    v.x += to_f32(r[0]);
    v.y += to_f32(r[1]);
    v.z += to_f32(r[2]);
    v.w += to_f32(r[3]);
  }
  const T4 o = {static_cast<T>(v.x), static_cast<T>(v.y), static_cast<T>(v.z), static_cast<T>(v.w)};
  *reinterpret_cast<T4*>(C + row * ldc + col) = o;
}
}  // namespace

void launch_split(bool bf16_, bool b_kmajor, Tile t, int parts, const GemmArgs& ga, hipStream_t s) {
  if (bf16_) {
    if (b_kmajor)
      launch_t<bf16, true>(t, parts, ga, s);
    else
      launch_t<bf16, false>(t, parts, ga, s);
  } else {
    if (b_kmajor)
      launch_t<f16, true>(t, parts, ga, s);
    else
      launch_t<f16, false>(t, parts, ga, s);
  }
}

void launch_split_sum(bool bf16_, const float* ws, int parts, const GemmArgs& ga, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>((ga.M * ga.N / 4 + 255) / 256));
#define ZK_SUM(T)                                                                                \
  hipLaunchKernelGGL((split_sum_kernel<T>), grid, dim3(256), 0, s, ws, parts, (T*)ga.c, ga.ldc, \
                     (const T*)ga.r, ga.ldr, ga.M, ga.N)
  if (bf16_) ZK_SUM(bf16); else ZK_SUM(f16);
#undef ZK_SUM
}

}  // namespace gemm
}  // namespace zk
