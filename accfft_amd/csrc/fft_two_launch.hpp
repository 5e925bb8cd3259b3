// fft_two_launch.hpp -- when a plan takes the two-pass kernels (fft_two.hpp)
// and how they are launched (fft_two.hip).
#pragma once
#include "fft_kernels.hpp"

namespace afft {

inline bool two_pow2(int n, int lo, int hi) { return n >= lo && n <= hi && (n & (n - 1)) == 0; }
// R of N1 = R M, the rows pass 1 transforms at once (0: no two-pass form).
// M = 1 leaves pass 2 the plain x pass, which takes any length; M = 2, 4, 8
// take x lengths of 32 to 512 points.  Larger M or longer axes would need
// tiles beyond a CU's registers.  64 rows: with 128, pass 1 of 512^3 FP32
// fills a CU with one workgroup (274 / 299 us instead of 209 / 230), more
// than pass 2 gains with M = 4 (244-257 us instead of 293).  Every grid of
// the rule measured faster than with one pass per axis (round trips, FP32 /
// FP64: 64^3 40 -> 26 / 42 -> 26 us, 128^3 67 -> 40 / 86 -> 51, 256^3 148 ->
// 119 / 313 -> 214, 512^3 1121 -> 949 / 2375 -> 2060; 512 x 256 x 512 FP32
// 556 -> 479, 256 x 512 x 256 FP64 669 -> 461).
inline bool two_xy_ok(int n0, int m) { return m == 1 || (m <= 8 && two_pow2(n0, 32, 512)); }
inline int two_rows(const int* n) {
  if (!two_pow2(n[2], 32, 512) || !two_pow2(n[1], 32, 512)) return 0;
  const int r = n[1] == 32 ? 32 : 64;
  return two_xy_ok(n[0], n[1] / r) ? r : 0;
}
// Complex rows take twice the tile of real ones: at most 256 KiB.  (c2c
// pairs, FP32 / FP64: 64^3 35 -> 21 / 42 -> 26 us, 128^3 86 -> 43 / 88 -> 65,
// 256^3 279 -> 220 / 543 -> 460, 512^3 2541 -> 2053 us.)
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
