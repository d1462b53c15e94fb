// Register-fed two-pass kernels (unaligned rows, either layout) for bf16 inputs.
#include "wgrad_staged.hpp"

namespace fdp {
namespace wg {

hipError_t launch_staged_bf16(const Args& a, const StreamPlan& sp, int layout, StagedPass pass,
                              hipStream_t s) {
  return launch_staged<BF16>(a, sp, layout, pass, s);
}

}  // namespace wg
}  // namespace fdp
