// Instantiations of the single-pass step kernel (lsf_pass.h): material mode x poles per D-form node (the slot
// stride) x the kappa term (on no axis, on every axis with CPML, on some).

#include "lsf_launch.h"
#include "lsf_pass.h"

namespace lsf {
namespace {

// The D-form chunk table: one thread per (chunk, component), from the slot bases and the material (a D-form node's
// coefficient is negative) over the E-stepped box.
__global__ void k_dform_chunks(StepArgs a, DChunk* out, long long n) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const int c = (int)(q % 3);
  const long long ch = q / 3;
  const int nchunk = a.nchunk, nx = a.g.n[0], ny = a.g.n[1];
  const int x0 = (int)(ch % nchunk) * 32;
  const long long row = ch / nchunk;  // k ny + j
  const int j = (int)(row % ny), k = (int)(row / ny);
  unsigned mask = 0u;
  for (int b = 0; b < 32 && x0 + b < nx; ++b) {
    const long long cell = row * nx + x0 + b;
    const float v = a.mid ? a.mtab[(a.mid[cell] >> (8 * c)) & 255u] : a.cbd[(long long)c * a.g.N + cell];
    if (v < 0.f && e_box<false>(a.g, c, x0 + b, j, k)) mask |= 1u << b;
  }
  out[q] = DChunk{a.chunk_base[q], mask};
}

template <int MAT, int NP>
void go(const PassLaunch& L, hipStream_t s) {
  const dim3 grid(L.sc.n_pad), block(64 * PASS_WAVES);
  if (L.kappa == 2) hipLaunchKernelGGL((k_pass<MAT, NP, 2>), grid, block, 0, s, L.args, L.sc);
  else if (L.kappa) hipLaunchKernelGGL((k_pass<MAT, NP, 1>), grid, block, 0, s, L.args, L.sc);
  else hipLaunchKernelGGL((k_pass<MAT, NP, 0>), grid, block, 0, s, L.args, L.sc);
}

template <int MAT>
void by_poles(const PassLaunch& L, hipStream_t s) {
  switch (L.np) {
    case 0: return go<MAT, 0>(L, s);
    case 1: return go<MAT, 1>(L, s);
    case 2: return go<MAT, 2>(L, s);
    case 3: return go<MAT, 3>(L, s);
    default: return go<MAT, 4>(L, s);
  }
}

}  // namespace

void launch_pass(const PassLaunch& L, hipStream_t s) {
  if (L.mat) by_poles<1>(L, s);
  else by_poles<0>(L, s);
}

void launch_dform_chunks(const StepArgs& a, void* out, long long n, hipStream_t s) {
  hipLaunchKernelGGL(k_dform_chunks, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, (DChunk*)out, n);
}

}  // namespace lsf
