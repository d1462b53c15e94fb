// Two-pass (Gram norm + streamed clipped sum) kernel instantiations for f16
// inputs.
#include "wgrad_stream.hpp"

namespace fdp {
namespace wg {

hipError_t launch_gram_norm_f16(const GramArgs& g, hipStream_t s) {
  return launch_gram_norm<F16>(g, s);
}
hipError_t launch_clipsum_f16(const Args& a, const StreamPlan& sp, int layout, hipStream_t s) {
  return launch_clipsum<F16>(a, sp, layout, s);
}
hipError_t launch_prod_norm_f16(const Args& a, const StreamPlan& sp, int layout, hipStream_t s) {
  return launch_prod_norm<F16>(a, sp, layout, s);
}

}  // namespace wg
}  // namespace fdp
