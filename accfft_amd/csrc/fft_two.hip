// The two-pass kernels (fft_two.hpp) in one precision, AFFT_T, set by the
// build.
#include "fft_two.hpp"
#include "fft_two_launch.hpp"

namespace afft {

template <>
hipError_t launch_two_zy<AFFT_T>(int sign, int nz, int r, const FftArgs<AFFT_T>& a,
                                 const cpx<AFFT_T>* twy, hipStream_t st) {
  const dim3 g((unsigned)a.nlines);
#define AFFT_ZY(NZ, R)                                                                            \
  if (nz == NZ && r == R) {                                                                       \
    const dim3 b(ZYCfg<AFFT_T, R / 2, NZ>::TPB);                                                  \
    if (sign < 0) hipLaunchKernelGGL((two_zy_r2c_kernel<AFFT_T, NZ, R>), g, b, 0, st, a, twy);    \
    else hipLaunchKernelGGL((two_zy_c2r_kernel<AFFT_T, NZ, R>), g, b, 0, st, a, twy);             \
    return hipGetLastError();                                                                     \
  }
  AFFT_ZY(32, 32)
  AFFT_ZY(64, 32)
  AFFT_ZY(128, 32)
  AFFT_ZY(256, 32)
  AFFT_ZY(512, 32)
  AFFT_ZY(32, 64)
  AFFT_ZY(64, 64)
  AFFT_ZY(128, 64)
  AFFT_ZY(256, 64)
  AFFT_ZY(512, 64)
#undef AFFT_ZY
  return hipErrorNotSupported;
}

template <>
hipError_t launch_two_zy_c2c<AFFT_T>(int sign, int nz, int r, const FftArgs<AFFT_T>& a,
                                     const cpx<AFFT_T>* twy, hipStream_t st) {
  const dim3 g((unsigned)a.nlines);
#define AFFT_ZC(NZ, R)                                                                            \
  if constexpr (two_c2c_tile<AFFT_T>(NZ, R))                                                      \
    if (nz == NZ && r == R) {                                                                     \
      const dim3 b(ZYCfg<AFFT_T, R, NZ>::TPB);                                                    \
      if (sign < 0) hipLaunchKernelGGL((two_zy_c2c_kernel<AFFT_T, NZ, R, -1>), g, b, 0, st, a, twy); \
      else hipLaunchKernelGGL((two_zy_c2c_kernel<AFFT_T, NZ, R, +1>), g, b, 0, st, a, twy);       \
      return hipGetLastError();                                                                   \
    }
  AFFT_ZC(32, 32)
  AFFT_ZC(64, 32)
  AFFT_ZC(128, 32)
  AFFT_ZC(256, 32)
  AFFT_ZC(512, 32)
  AFFT_ZC(32, 64)
  AFFT_ZC(64, 64)
  AFFT_ZC(128, 64)
  AFFT_ZC(256, 64)
  AFFT_ZC(512, 64)
#undef AFFT_ZC
  return hipErrorNotSupported;
}

template <>
hipError_t launch_two_xy<AFFT_T>(int mode, int sign, int n0, int m, const FftArgs<AFFT_T>& a,
                                 hipStream_t st) {
#define AFFT_XY(NN, MM)                                                                           \
  if (n0 == NN && m == MM) {                                                                      \
    using CF = XYCfg<AFFT_T, NN, MM, M_C2C>;                                                      \
    using CM = XYCfg<AFFT_T, NN, MM, M_MULT>;                                                     \
    static_assert(CF::W == CM::W, "one tile width");                                              \
    if (a.nlines % CF::W) return hipErrorNotSupported;                                            \
    const dim3 g((unsigned)(a.nlines / CF::W)), b(mode == M_C2C ? CF::TPB : CM::TPB);             \
    constexpr int INV = sizeof(AFFT_T) == 4 ? +1 : -1;  /* FP64: the forward kernel, conjugated */  \
    const unsigned flip = sign > 0 ? 0x80000000u : 0u;                                            \
    if (mode == M_C2C && sign < 0) hipLaunchKernelGGL((two_xy_kernel<AFFT_T, NN, MM, M_C2C, -1>), g, b, 0, st, a, flip); \
    else if (mode == M_C2C) hipLaunchKernelGGL((two_xy_kernel<AFFT_T, NN, MM, M_C2C, INV>), g, b, 0, st, a, flip); \
    else if (mode == M_MULT) hipLaunchKernelGGL((two_xy_kernel<AFFT_T, NN, MM, M_MULT, -1>), g, b, 0, st, a, flip); \
    else return hipErrorNotSupported;                                                             \
    return hipGetLastError();                                                                     \
  }
#define AFFT_XYM(NN) AFFT_XY(NN, 2) AFFT_XY(NN, 4) AFFT_XY(NN, 8)
  AFFT_XYM(32)
  AFFT_XYM(64)
  AFFT_XYM(128)
  AFFT_XYM(256)
  AFFT_XYM(512)
#undef AFFT_XYM
#undef AFFT_XY
  return hipErrorNotSupported;
}

}  // namespace afft
