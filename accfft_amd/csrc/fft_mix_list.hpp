// fft_mix_list.hpp -- the lengths with compile-time mixed-radix kernels
// (fft_mix.hpp) and the interface of their launchers: every length from 18
// to 1024 with the prime factors 2, 3 and 5, and to 512 with 7, of the
// powers of two 16 to 512.  Longer ones and other factors run the run-time
// engine.  Where the list ends is a choice of size, not a measured line: each
// length costs fourteen kernels (about 0.2 MB), and neither the lengths with a
// factor 7 above 512 nor any above 1024 were built and timed; on the run-time
// engine they reach 1.5-3 TB/s a pass, where those of the list reach 3.7-6.
// The lists are parts of about equal work, compiled as translation units of
// their own (fft_mix.hip).
#pragma once
#include "fft_kernels.hpp"

#define AFFT_MIX_0(X) \
  X(16) X(18) X(28) X(45) X(60) X(81) X(105) X(135) X(162) X(196) X(240) X(280) X(324) X(378) \
  X(432) X(490) X(625) X(750) X(960)
#define AFFT_MIX_1(X) \
  X(32) X(20) X(30) X(48) X(63) X(84) X(108) X(140) X(168) X(200) X(243) X(288) X(336) X(384) \
  X(441) X(500) X(640) X(768) X(972)
#define AFFT_MIX_2(X) \
  X(64) X(21) X(35) X(49) X(70) X(90) X(112) X(144) X(175) X(210) X(245) X(294) X(343) X(392) \
  X(448) X(504) X(648) X(800) X(1000)
#define AFFT_MIX_3(X) \
  X(128) X(24) X(36) X(50) X(72) X(96) X(120) X(147) X(180) X(216) X(250) X(300) X(350) X(400) \
  X(450) X(540) X(675) X(810)
#define AFFT_MIX_4(X) \
  X(256) X(25) X(40) X(54) X(75) X(98) X(125) X(150) X(189) X(224) X(252) X(315) X(360) X(405) \
  X(480) X(576) X(720) X(864)
#define AFFT_MIX_5(X) \
  X(512) X(27) X(42) X(56) X(80) X(100) X(126) X(160) X(192) X(225) X(270) X(320) X(375) X(420) \
  X(486) X(600) X(729) X(900)
#define AFFT_MIX_EACH(X) X(0) X(1) X(2) X(3) X(4) X(5)

namespace afft {

// Part whose translation unit holds length n, -1 for none.
inline int mix_part(int n) {
  switch (n) {
#define AFFT_MIX_N0(N) case N: return 0;
#define AFFT_MIX_N1(N) case N: return 1;
#define AFFT_MIX_N2(N) case N: return 2;
#define AFFT_MIX_N3(N) case N: return 3;
#define AFFT_MIX_N4(N) case N: return 4;
#define AFFT_MIX_N5(N) case N: return 5;
    AFFT_MIX_0(AFFT_MIX_N0)
    AFFT_MIX_1(AFFT_MIX_N1)
    AFFT_MIX_2(AFFT_MIX_N2)
    AFFT_MIX_3(AFFT_MIX_N3)
    AFFT_MIX_4(AFFT_MIX_N4)
    AFFT_MIX_5(AFFT_MIX_N5)
    default: return -1;
  }
}

// Powers of two on the mixed-radix kernels.  Strided up to 256 points: one
// or two LDS round trips instead of three or four (64^3 FP64 passes 9.0-10
// -> 6.5-7.2 us, 256^3 FP32 x pass 29 -> 26 us, multiply 47 -> 30 us,
// derivatives 38 -> 28 us, FP64 51 -> 47, 81 -> 54, 65-69 -> 52-56 us); 512
// points FP64 (multiply 569 -> 423 us, derivatives 751 / 512 -> 570 / 407
// us, C2C 401-418 -> 388-394 us) and FP32 C2C (204 / 197 -> 197 / 184 us; the
// fused FP32 passes stay with the two-level tiles, derivatives 219 against
// 240-250 us).  z up to 128 points (64^3 FP64 8.5 -> 6.6 us) and the FP32
// derivative at 256 and 512 (37 -> 32, 276 -> 217 us); the other z passes are
// faster as they are (256^3 FP64 r2c 60 against 69 us, 512^3 369 against 410
// us).  No others are built; C2C passes up to 256 points and z passes up to 128
// go here by mix_pow2 (fft_launch.hpp), the rest of these always.
template <typename T>
constexpr bool mix_pow2_built(int n, bool strided, int mode) {
  if (strided) return n <= 256 || (n == 512 && (sizeof(T) == 8 || mode == M_C2C));
  return n <= 128 || (sizeof(T) == 4 && mode == M_DERIV && n <= 512);
}

// Launches a z (strided = false) or strided pass of length n over `units`
// complex lines (pairs of real lines); hipErrorNotSupported for a mode the
// part does not hold.
template <typename T, int PART>
hipError_t mix_launch(bool strided, int mode, int sign, FftArgs<T>& a, int n, int64_t units,
                      hipStream_t st);
#define AFFT_MIX_DECL(P)                                                                       \
  template <>                                                                                  \
  hipError_t mix_launch<float, P>(bool, int, int, FftArgs<float>&, int, int64_t, hipStream_t); \
  template <>                                                                                  \
  hipError_t mix_launch<double, P>(bool, int, int, FftArgs<double>&, int, int64_t, hipStream_t);
AFFT_MIX_EACH(AFFT_MIX_DECL)
#undef AFFT_MIX_DECL

}  // namespace afft
