// fft_two_launch.hpp -- when a plan takes the two-pass kernels (fft_two.hpp)
// and how they are launched (fft_two.hip).
#pragma once
#include "fft_kernels.hpp"

namespace afft {

inline bool two_pow2(int n, int lo, int hi) { return n >= lo && n <= hi && (n & (n - 1)) == 0; }
// Pass 1 runs N0 M blocks; where its tiles are large, a block's chain of
// stages takes as long as a few short passes, so tiles of 128 KiB and more,
// and those of 512-point lines, need as many blocks as they have complex rows
// (r2c packs two real rows into one).  Below that line one pass per axis is
// faster, above it the two passes are (us, two passes / one per axis: r2c, c2r
// FP32 8 x 64 x 512 17.6, 20.2 / 15.8, 16.3, 48 x 64 x 512 20.3, 22.0 / 22.0,
// 23.8; FP64 8 x 64 x 512 28.1, 30.1 / 21.1, 21.3, 32 x 64 x 512 30.8, 32.7 /
// 35.0, 38.0; c2c FP32 8 x 64 x 512 23.9 / 15.1, 64 x 64 x 512 32.1 / 34.5, FP64
// 8 x 64 x 256 23.0 / 15.6, 64 x 64 x 128 20.3 / 20.8).  Smaller tiles are
// faster with any number of planes.
inline bool two_blocks_ok(const int* n, int r, int rows, size_t csz) {
  const bool large = n[2] == 512 || (size_t)rows * n[2] * csz >= 128 * 1024;
  return !large || (int64_t)n[0] * (n[1] / r) >= rows;
}
// R of N1 = R M, the rows pass 1 transforms at once (0: no two-pass form).
// M = 1 leaves pass 2 the plain x pass, which takes any length; M = 2, 4, 8
// take x lengths of 32 to 512 points.  The limit of 512 points an axis and of
// M = 8 is where the kernels that are built end: FP64 tiles beyond it exceed a
// CU's registers; FP32 ones of 1024 points (256 KiB) were not built or
// measured.  64 rows: with 128, pass 1 of 512^3 FP32
// fills a CU with one workgroup (274 / 299 us instead of 209 / 230), more
// than pass 2 gains with M = 4 (244-257 us instead of 293).  Grids of the
// rule measured faster than with one pass per axis (round trips, FP32 /
// FP64: 64^3 40 -> 26 / 42 -> 26 us, 128^3 67 -> 40 / 86 -> 51, 256^3 148 ->
// 119 / 313 -> 214, 512^3 1121 -> 949 / 2375 -> 2060; 512 x 256 x 512 FP32
// 556 -> 479, 256 x 512 x 256 FP64 669 -> 461).
inline bool two_xy_ok(int n0, int m) { return m == 1 || (m <= 8 && two_pow2(n0, 32, 512)); }
template <typename T>
inline int two_rows(const int* n) {
  if (!two_pow2(n[2], 32, 512) || !two_pow2(n[1], 32, 512)) return 0;
  const int r = n[1] == 32 ? 32 : 64;
  return two_xy_ok(n[0], n[1] / r) && two_blocks_ok(n, r, r / 2, sizeof(cpx<T>)) ? r : 0;
}
// Complex rows take twice the tile of real ones: at most 256 KiB.  (c2c
// pairs, FP32 / FP64: 64^3 35 -> 21 / 42 -> 26 us, 128^3 86 -> 43 / 88 -> 65,
// 256^3 279 -> 220 / 543 -> 460, 512^3 2541 -> 2053 us.  FP64 64 x 128 x 256 and
// 32 x 256 x 256, 128 blocks of 256 KiB, lose 3 %: 41 -> 42, 39 -> 41 us.)
template <typename T>
constexpr bool two_c2c_tile(int nz, int r) { return (size_t)nz * r * sizeof(cpx<T>) <= 256 * 1024; }
template <typename T>
inline int two_rows_c2c(const int* n) {
  if (!two_pow2(n[2], 32, 512) || !two_pow2(n[1], 32, 512)) return 0;
  const int r = n[1] == 32 || !two_c2c_tile<T>(n[2], 64) ? 32 : 64;
  return two_xy_ok(n[0], n[1] / r) && two_blocks_ok(n, r, r, sizeof(cpx<T>)) ? r : 0;
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
