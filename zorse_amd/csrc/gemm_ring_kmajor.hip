// Launches of the small-tile GEMM (gemm_ring.h) with a K-major operand,
// compiled with the register-assignment flag of the tiled K-major forms
// (gemm_kernels.h).
#include "gemm_ring.h"

namespace zk {
namespace gemm {

namespace {
template <typename T, bool AKM, bool BKM>
void launch_t(Tile t, const GemmArgs& ga, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(tile_count(t, ga.M, ga.N)));
#define ZK_RING(MB, NB, RB, WPE, KS)                                                   \
  hipLaunchKernelGGL((gemm_ring_kernel<T, 0, AKM, BKM, MB, NB, RB, WPE, KS>), grid,   \
                     dim3(256 * KS), 0, s, ga)
  if constexpr (AKM) {
    if (t == k64 && BKM)
      ZK_RING(2, 2, 4, 2, 1);
    else
      ZK_RING(4, 4, 2, 2, 1);
  } else {
    if (t == k64)
      ZK_RING(2, 2, 4, 2, 1);
    else if (t == k64x128)
      ZK_RING(2, 4, 4, 2, 2);
    else if (t == k128x2)
      ZK_RING(4, 4, 4, 2, 2);
    else
      ZK_RING(4, 4, 2, 2, 1);
  }
#undef ZK_RING
}

template <typename T>
void launch_layout(bool akm, bool bkm, Tile t, const GemmArgs& ga, hipStream_t s) {
  if (akm && bkm)
    launch_t<T, true, true>(t, ga, s);
  else if (bkm)
    launch_t<T, false, true>(t, ga, s);
  else
    launch_t<T, true, false>(t, ga, s);
}
}  // namespace

void launch_ring_kmajor(bool bf16_, bool a_kmajor, bool b_kmajor, Tile t, const GemmArgs& ga,
                        hipStream_t s) {
  if (bf16_)
    launch_layout<bf16>(a_kmajor, b_kmajor, t, ga, s);
  else
    launch_layout<f16>(a_kmajor, b_kmajor, t, ga, s);
}

}  // namespace gemm
}  // namespace zk
