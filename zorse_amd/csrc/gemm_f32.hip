// Launches of the small-tile GEMM (gemm_ring.h) on fp32 operands, every layout.
#include "gemm_ring.h"

namespace zk {
namespace gemm {

namespace {
template <bool AKM, bool BKM>
void launch_t(bool small, const GemmArgs& ga, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(tile_count(small ? k64 : k128, ga.M, ga.N)));
  if (small)
    hipLaunchKernelGGL((gemm_ring_kernel<float, 0, AKM, BKM, 2, 2, 4, 2, 1>), grid, dim3(256), 0, s,
                       ga);
  else
    hipLaunchKernelGGL((gemm_ring_kernel<float, 0, AKM, BKM, 4, 4, 2, 2, 1>), grid, dim3(256), 0, s,
                       ga);
}
}  // namespace

void launch_ring_f32(bool a_kmajor, bool b_kmajor, const GemmArgs& ga, hipStream_t s) {
  const bool small = f32_tile(ga.M, ga.N) == k64;
  if (!a_kmajor && !b_kmajor)
    launch_t<false, false>(small, ga, s);
  else if (!a_kmajor)
    launch_t<false, true>(small, ga, s);
  else if (b_kmajor)
    launch_t<true, true>(small, ga, s);
  else
    launch_t<true, false>(small, ga, s);
}

}  // namespace gemm
}  // namespace zk
