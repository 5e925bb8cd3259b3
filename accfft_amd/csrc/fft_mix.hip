// One part of the compile-time mixed-radix kernels (fft_mix.hpp) in one
// precision: AFFT_T, AFFT_PART and AFFT_PART_LIST are set by the build.
#include "fft_mix.hpp"
#include "fft_mix_list.hpp"

namespace afft {
namespace {

template <typename T, int N>
hipError_t launch_n(bool strided, int mode, unsigned flip, FftArgs<T>& a, int64_t units,
                    hipStream_t st) {
  if (strided) {
    using CF = MixS<T, N>;
    const dim3 g((unsigned)((units + CF::L - 1) / CF::L)), b(CF::TPB);
    switch (mode) {
      case M_C2C: hipLaunchKernelGGL((mix_s_kernel<T, N, M_C2C>), g, b, 0, st, a, flip); break;
      case M_MULT: hipLaunchKernelGGL((mix_s_kernel<T, N, M_MULT>), g, b, 0, st, a, flip); break;
      case M_DERIV: hipLaunchKernelGGL((mix_s_kernel<T, N, M_DERIV>), g, b, 0, st, a, flip); break;
      default: return hipErrorNotSupported;
    }
  } else {
#define AFFT_MIXZ(MODE)                                                                        \
  case MODE: {                                                                                 \
    using CF = MixZ<T, N, MODE>;                                                               \
    const dim3 g((unsigned)((units + CF::L - 1) / CF::L)), b(CF::TPB);                         \
    hipLaunchKernelGGL((mix_z_kernel<T, N, MODE>), g, b, 0, st, a, flip);                      \
    break;                                                                                     \
  }
    switch (mode) {
      AFFT_MIXZ(M_C2C)
      AFFT_MIXZ(M_R2C)
      AFFT_MIXZ(M_C2R)
      AFFT_MIXZ(M_DERIV)
      default: return hipErrorNotSupported;
    }
#undef AFFT_MIXZ
  }
  return hipGetLastError();
}

}  // namespace

template <>
hipError_t mix_launch<AFFT_T, AFFT_PART>(bool strided, int mode, int sign, FftArgs<AFFT_T>& a, int n,
                                         int64_t units, hipStream_t st) {
  const unsigned flip = sign > 0 ? 0x80000000u : 0u;
  switch (n) {
#define AFFT_CASE(N) \
  case N: return launch_n<AFFT_T, N>(strided, mode, flip, a, units, st);
    AFFT_PART_LIST(AFFT_CASE)
#undef AFFT_CASE
    default: return hipErrorNotSupported;
  }
}

}  // namespace afft
