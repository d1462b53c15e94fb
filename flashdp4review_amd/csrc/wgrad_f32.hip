// fp32 two-pass clipped weight gradient: kernel instantiations and launches.
#include "wgrad_f32.hpp"

namespace fdp {
namespace wg {

namespace {

template <class C>
void set_tiles(Args& a) {
  a.tiles_m = static_cast<int>((a.M + C::TM - 1) / C::TM);
  a.tiles_n = static_cast<int>((a.N + C::TM - 1) / C::TM);
}

template <class C>
void norm(Args a, int layout, hipStream_t s) {
  set_tiles<C>(a);
  const dim3 grid(static_cast<unsigned>(a.tiles_m * a.tiles_n),
                  static_cast<unsigned>(a.B < kGridY ? a.B : kGridY));
  if (layout == FDP_LAYOUT_TN)
    hipLaunchKernelGGL((f32_norm_kernel<C, FDP_LAYOUT_TN>), grid, dim3(NT), 0, s, a);
  else
    hipLaunchKernelGGL((f32_norm_kernel<C, FDP_LAYOUT_NN>), grid, dim3(NT), 0, s, a);
}

template <class C>
void sum(Args a, int64_t rows, int layout, hipStream_t s) {
  set_tiles<C>(a);
  const dim3 grid(static_cast<unsigned>(a.tiles_m * a.tiles_n * a.groups));
  if (layout == FDP_LAYOUT_TN)
    hipLaunchKernelGGL((f32_sum_kernel<C, FDP_LAYOUT_TN>), grid, dim3(NT), 0, s, a, rows);
  else
    hipLaunchKernelGGL((f32_sum_kernel<C, FDP_LAYOUT_NN>), grid, dim3(NT), 0, s, a, rows);
}

}  // namespace

hipError_t launch_f32(Args a, const F32Plan& f, int layout, bool noclip, hipStream_t s) {
  if (!noclip) {
    const unsigned nb = static_cast<unsigned>(a.B < 65536 ? a.B : 65536);
    if (f.norm == kF32NormRow)
      hipLaunchKernelGGL(f32_row_kernel<0>, dim3(nb), dim3(NT), 0, s, a);
    else if (f.norm == kF32NormRowGram)
      hipLaunchKernelGGL(f32_rowgram_kernel<0>, dim3(nb), dim3(NT), 0, s, a);
    else if (f.norm_small)
      norm<F32Small>(a, layout, s);
    else
      norm<F32Big>(a, layout, s);
  }
  // the sum pass forms the factors itself while a workgroup's range holds few
  // enough samples and partials that this costs less than a launch
  const int64_t K = a.K > 0 ? a.K : 1;
  const int64_t nsamp = f.rows_per_split / K + 2;
  a.groups = f.splits;
  if (noclip && a.K > 0) {  // (without rows the sum pass meets no sample)
    a.fac_parts = -1;
  } else if (a.K > 0 &&
             (f.per_sample <= kF32FacThread || nsamp * f.per_sample <= 16384)) {
    a.fac_parts = f.per_sample;
  } else {
    launch_factors(a, f.per_sample, noclip, s);
    a.fac_parts = 0;
    a.norms_out = a.factors_out = nullptr;
  }
  if (f.sum_small) sum<F32Small>(a, f.rows_per_split, layout, s);
  else sum<F32Big>(a, f.rows_per_split, layout, s);
  if (a.groups > 1) launch_finalize(a, s);
  return hipGetLastError();
}

}  // namespace wg
}  // namespace fdp
