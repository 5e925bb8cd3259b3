// fft_two_launch.hpp -- when a plan takes the two-pass kernels (fft_two.hpp)
// and how they are launched (fft_two.hip).
#pragma once
#include "fft_kernels.hpp"

namespace afft {

inline bool two_pow2(int n, int lo, int hi) { return n >= lo && n <= hi && (n & (n - 1)) == 0; }
// R of N1 = R M, the rows pass 1 transforms at once (0: no two-pass form).
// M = 1 leaves pass 2 the plain x pass, which takes any length; M = 2, 4, 8
// take x lengths of 32 to 512 points.  Larger M or longer axes would need
// tiles beyond a CU's registers.
inline bool two_xy_ok(int n0, int m) { return m == 1 || (m <= 8 && two_pow2(n0, 32, 512)); }
inline int two_rows(const int* n) {
  if (!two_pow2(n[2], 32, 512) || !two_pow2(n[1], 32, 512)) return 0;
  const int r = n[1] == 32 ? 32 : 64;
  return two_xy_ok(n[0], n[1] / r) ? r : 0;
}
// Complex rows take twice the tile of real ones: at most 256 KiB.
template <typename T>
constexpr bool two_c2c_tile(int nz, int r) { return (size_t)nz * r * sizeof(cpx<T>) <= 256 * 1024; }
template <typename T>
inline int two_rows_c2c(const int* n) {
  if (!two_pow2(n[2], 32, 512) || !two_pow2(n[1], 32, 512)) return 0;
  const int r = n[1] == 32 || !two_c2c_tile<T>(n[2], 64) ? 32 : 64;
  return two_xy_ok(n[0], n[1] / r) ? r : 0;
}

// Pass 1 of `a.nlines` = planes x M blocks; sign < 0 r2c, > 0 c2r.
template <typename T>
hipError_t launch_two_zy(int sign, int nz, int r, const FftArgs<T>& a, const cpx<T>* twy, hipStream_t st);
// The same over complex rows, both signs.
template <typename T>
hipError_t launch_two_zy_c2c(int sign, int nz, int r, const FftArgs<T>& a, const cpx<T>* twy, hipStream_t st);
// Pass 2, M_C2C (either sign) or M_MULT.
template <typename T>
hipError_t launch_two_xy(int mode, int sign, int n0, int m, const FftArgs<T>& a, hipStream_t st);
#define AFFT_TWO_DECL(T)                                                                          \
  template <>                                                                                     \
  hipError_t launch_two_zy<T>(int, int, int, const FftArgs<T>&, const cpx<T>*, hipStream_t);      \
  template <>                                                                                     \
  hipError_t launch_two_zy_c2c<T>(int, int, int, const FftArgs<T>&, const cpx<T>*, hipStream_t);  \
  template <>                                                                                     \
  hipError_t launch_two_xy<T>(int, int, int, int, const FftArgs<T>&, hipStream_t);
AFFT_TWO_DECL(float)
AFFT_TWO_DECL(double)
#undef AFFT_TWO_DECL

}  // namespace afft
