// Instantiations of the lean bulk kernels (lsf_lean.h): H and E, forward and adjoint, the E ones by material mode;
// persistent or one tile per block.

#include "lsf_launch.h"
#include "lsf_lean.h"

namespace lsf {
namespace {

template <bool ADJ>
void go_h(const KLaunch& L, hipStream_t s) {
  if (L.grid < L.sc.n_pad)
    hipLaunchKernelGGL((k_lean_h<ADJ, true>), dim3(L.grid), dim3(64 * LEAN_WAVES), 0, s, L.args, L.sc);
  else
    hipLaunchKernelGGL((k_lean_h<ADJ, false>), dim3(L.sc.n_pad), dim3(64 * LEAN_WAVES), 0, s, L.args, L.sc);
}

template <bool ADJ, int MAT>
void go_e(const KLaunch& L, hipStream_t s) {
  if (L.grid < L.sc.n_pad)
    hipLaunchKernelGGL((k_lean_e<ADJ, MAT, true>), dim3(L.grid), dim3(64 * LEAN_WAVES), 0, s, L.args, L.sc);
  else
    hipLaunchKernelGGL((k_lean_e<ADJ, MAT, false>), dim3(L.sc.n_pad), dim3(64 * LEAN_WAVES), 0, s, L.args, L.sc);
}

}  // namespace

void launch_lean_h(const KLaunch& L, bool adjoint, hipStream_t s) {
  if (adjoint) go_h<true>(L, s);
  else go_h<false>(L, s);
}

void launch_lean_e(const KLaunch& L, bool adjoint, hipStream_t s) {
  if (adjoint) {
    if (L.mat) go_e<true, 1>(L, s);
    else go_e<true, 0>(L, s);
  } else {
    if (L.mat) go_e<false, 1>(L, s);
    else go_e<false, 0>(L, s);
  }
}

}  // namespace lsf
