// Launches of the small-tile GEMM (gemm_ring.h) with both operands along the
// reduction: plain, SwiGLU and RoPE epilogues.
#include "gemm_ring.h"

namespace zk {
namespace gemm {

namespace {
template <typename T, int EPI>
void launch_t(Tile t, const GemmArgs& ga, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(tile_count(t, ga.M, ga.N)));
#define ZK_RING(MB, NB, RB, WPE, KS)                                                       \
  hipLaunchKernelGGL((gemm_ring_kernel<T, EPI, false, false, MB, NB, RB, WPE, KS>), grid, \
                     dim3(256 * KS), 0, s, ga)
  if (t == k64)
    ZK_RING(2, 2, 4, 2, 1);
  else if (t == k64x128)
    ZK_RING(2, 4, 4, 2, 2);
  else if (t == k128x2)
    ZK_RING(4, 4, 4, 2, 2);
  else
    ZK_RING(4, 4, 2, 2, 1);
#undef ZK_RING
}

template <typename T>
void launch_epi(int epi, Tile t, const GemmArgs& ga, hipStream_t s) {
  if (epi == 1)
    launch_t<T, 1>(t, ga, s);
  else if (epi == 2)
    launch_t<T, 2>(t, ga, s);
  else
    launch_t<T, 0>(t, ga, s);
}
}  // namespace

void launch_ring(bool bf16_, int epi, bool a_kmajor, bool b_kmajor, Tile t, const GemmArgs& ga,
                 hipStream_t s) {
  if (a_kmajor || b_kmajor)
    launch_ring_kmajor(bf16_, a_kmajor, b_kmajor, t, ga, s);
  else if (bf16_)
    launch_epi<bf16>(epi, t, ga, s);
  else
    launch_epi<f16>(epi, t, ga, s);
}

}  // namespace gemm
}  // namespace zk
