// Paired single-pass kernel instantiations for fp32 operands.
#include "wgrad_wide.hpp"

namespace fdp {
namespace wg {

hipError_t launch_pair_f32(const WideArgs& a, bool plain, hipStream_t s) {
  const void* fns[3] = {reinterpret_cast<const void*>(&wgrad_pair_kernel<F32, 0>),
                        reinterpret_cast<const void*>(&wgrad_pair_kernel<F32, 1>),
                        reinterpret_cast<const void*>(&wgrad_pair_kernel<F32, 2>)};
  if (a.bias_op < 0 || a.bias_op > 2) return hipErrorInvalidValue;
  const void* fn = fns[a.bias_op];
  if (host::occupancy(fn, kWideThreads, 0) < 1) return hipErrorNotSupported;
  WideArgs c = a;
  void* params[] = {&c};
  return plain ? hipLaunchKernel(fn, dim3(a.nwg), dim3(kWideThreads), params, 0, s)
               : hipLaunchCooperativeKernel(fn, dim3(a.nwg), dim3(kWideThreads), params, 0, s);
}

}  // namespace wg
}  // namespace fdp
