// The kernels of passes whose program is decoded into LDS first: forward and reverse-sweep passes, by
// tile width.
#include "staged.hpp"

namespace cqs {

template <int L>
__global__ __launch_bounds__(TileShape<L>::NT) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_pass_staged(
    float2* __restrict__ psi, TileProg P) {
  extern __shared__ float2 lds[];
  const uint64_t base = deposit_bounded<31>((uint64_t)blockIdx.x, P.opos, P.nouter);
  pass_tile<L, RunStaged>(psi, P, P.lpos, P.lpos_out, base, lds, P.basis, P.zmask, P.zval, P.wmask, P.wval);
}

template <int L>
__global__ __launch_bounds__(TileShape<L>::NT) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_adjoint_staged(
    float2* __restrict__ psi, float2* __restrict__ phi, TileProg P, double* __restrict__ partial, int64_t stride) {
  extern __shared__ float2 lds[];
  const uint64_t base = deposit_bounded<31>((uint64_t)blockIdx.x, P.opos, P.nouter);
  adjoint_tile<L, RunStagedAdjoint>(psi, phi, P, P.lpos, base, partial, stride, blockIdx.x, lds);
}

const StagedPassKernel kPassStaged[15] = {
    nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, k_pass_staged<6>, k_pass_staged<7>, k_pass_staged<8>,
    k_pass_staged<9>, k_pass_staged<10>, k_pass_staged<11>, k_pass_staged<12>, nullptr, nullptr};

const StagedAdjKernel kAdjStaged[15] = {
    nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, k_adjoint_staged<6>, k_adjoint_staged<7>,
    k_adjoint_staged<8>, k_adjoint_staged<9>, k_adjoint_staged<10>, k_adjoint_staged<11>, nullptr, nullptr,
    nullptr};

}  // namespace cqs
