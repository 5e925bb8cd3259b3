// One part of the compile-time mixed-radix kernels (fft_mix.hpp) in one
// precision: AFFT_T, AFFT_PART and AFFT_PART_LIST are set by the build.
#include "fft_mix.hpp"
#include "fft_mix_list.hpp"

namespace afft {
namespace {

// the powers of two have the passes that launch_fft sends here
template <typename T, int N>
constexpr bool built(bool strided, int mode) {
  return (N & (N - 1)) != 0 || mix_pow2_built<T>(N, strided, mode);
}

template <typename T, int N>
hipError_t launch_n(bool strided, int mode, unsigned flip, FftArgs<T>& a, int64_t units,
                    hipStream_t st) {
  if (strided) {
#define AFFT_MIXS(MODE)                                                                         \
  if constexpr (built<T, N>(true, MODE))                                                        \
    if (mode == MODE) {                                                                         \
      using CF = MixS<T, N>;                                                                    \
      const dim3 g((unsigned)((units + CF::L - 1) / CF::L)), b(CF::TPB);                        \
      hipLaunchKernelGGL((mix_s_kernel<T, N, MODE>), g, b, 0, st, a, flip);                     \
      return hipGetLastError();                                                                 \
    }
    AFFT_MIXS(M_C2C)
    AFFT_MIXS(M_MULT)
    AFFT_MIXS(M_DERIV)
#undef AFFT_MIXS
  } else {
#define AFFT_MIXZ(MODE)                                                                         \
  if constexpr (built<T, N>(false, MODE))                                                       \
    if (mode == MODE) {                                                                         \
      using CF = MixZ<T, N, MODE>;                                                              \
      const dim3 g((unsigned)((units + CF::L - 1) / CF::L)), b(CF::TPB);                        \
      hipLaunchKernelGGL((mix_z_kernel<T, N, MODE>), g, b, 0, st, a, flip);                     \
      return hipGetLastError();                                                                 \
    }
    AFFT_MIXZ(M_C2C)
    AFFT_MIXZ(M_R2C)
    AFFT_MIXZ(M_C2R)
    AFFT_MIXZ(M_DERIV)
#undef AFFT_MIXZ
  }
  return hipErrorNotSupported;
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
