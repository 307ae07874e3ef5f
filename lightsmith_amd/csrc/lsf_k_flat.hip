// Instantiations of the flat bulk kernels (lsf_flat.h): the H kernel by field type, the E kernel by field type and
// material mode; two cells per lane, four wavefronts per block, persistent or one tile per block.

#include "lsf_flat.h"
#include "lsf_launch.h"

namespace lsf {
namespace {

constexpr int V = FLAT_CELLS, W = FLAT_WAVES;

template <class T>
void go_h(const KLaunch& L, hipStream_t s) {
  if (L.grid < L.sc.n_pad)
    hipLaunchKernelGGL((k_flat_h<T, V, W, true>), dim3(L.grid), dim3(64 * W), 0, s, L.args, L.sc);
  else
    hipLaunchKernelGGL((k_flat_h<T, V, W, false>), dim3(L.sc.n_pad), dim3(64 * W), 0, s, L.args, L.sc);
}

template <class T, int MAT>
void go_e(const KLaunch& L, hipStream_t s) {
  if (L.grid < L.sc.n_pad)
    hipLaunchKernelGGL((k_flat_e<T, MAT, V, W, true>), dim3(L.grid), dim3(64 * W), 0, s, L.args, L.sc);
  else
    hipLaunchKernelGGL((k_flat_e<T, MAT, V, W, false>), dim3(L.sc.n_pad), dim3(64 * W), 0, s, L.args, L.sc);
}

}  // namespace

void launch_flat_h(const KLaunch& L, hipStream_t s) {
  if (L.cplx) go_h<c32>(L, s);
  else go_h<float>(L, s);
}

void launch_flat_e(const KLaunch& L, hipStream_t s) {
  if (L.cplx) {
    if (L.mat) go_e<c32, 1>(L, s);
    else go_e<c32, 0>(L, s);
  } else {
    if (L.mat) go_e<float, 1>(L, s);
    else go_e<float, 0>(L, s);
  }
}

}  // namespace lsf
