// Launches of the tiled GEMM with a K-major operand: the input gradient
// dY W (W K-major) and the weight gradient dY^T X (both K-major, or dY^T
// row-major when a producer wrote it), compiled apart from gemm.hip for the
// register-assignment flag described in gemm_kernels.h.
#include "gemm_kernels.h"

namespace zk {
namespace gemm {

namespace {
template <typename T>
void launch_t(bool akm, bool bkm, bool ragged, bool half, const GemmArgs& ga, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(tile_count(half ? k128x256 : k256, ga.M, ga.N)));
  if (half) {
    hipLaunchKernelGGL((gemm_tiled_kernel<T, 0, false, true, false, 4>), grid, dim3(256), 0, s, ga);
    return;
  }
#define ZK_TILED(A, B, R) \
  hipLaunchKernelGGL((gemm_tiled_kernel<T, 0, A, B, R>), grid, dim3(256), 0, s, ga)
  if (akm && bkm) {
    if (ragged) ZK_TILED(true, true, true); else ZK_TILED(true, true, false);
  } else if (akm) {
    ZK_TILED(true, false, false);
  } else {
    if (ragged) ZK_TILED(false, true, true); else ZK_TILED(false, true, false);
  }
#undef ZK_TILED
}
}  // namespace

void launch_tiled_kmajor(bool bf16_, bool a_kmajor, bool b_kmajor, bool ragged, bool half,
                         const GemmArgs& ga, hipStream_t s) {
  if (bf16_)
    launch_t<bf16>(a_kmajor, b_kmajor, ragged, half, ga, s);
  else
    launch_t<f16>(a_kmajor, b_kmajor, ragged, half, ga, s);
}

}  // namespace gemm
}  // namespace zk
