// The rules by which a plan's passes choose their kernels, evaluated on the
// host (no kernel is instantiated or launched): prints "name value" lines
// for tests/test_route_rules.py.
#include <stdio.h>

#include "../../accfft_amd/csrc/dispatch.hpp"
#include "../../accfft_amd/csrc/exec.hpp"
#include "../../accfft_amd/csrc/fft_two.hpp"

using namespace afft;

namespace {

const cpx<float> rootsf{};
const cpx<double> rootsd{};
const cpx<float>* roots(float) { return &rootsf; }
const cpx<double>* roots(double) { return &rootsd; }

// an axis as the plan's tables leave it (only the pointers' presence counts)
template <typename T>
AxisTab<T> axis(int n, int s4v = -1, bool forced = false) {
  AxisTab<T> t;
  t.n = n;
  t.is_static = static_length(n);
  if (mix_part(n) >= 0) t.tw_mix = roots(T());
  if (n == 512 || (sizeof(T) == 4 && (n == 1024 || n == 2048))) t.tw_sub = t.tw_subw = roots(T());
  t.s4v = s4v;
  t.forced = forced;
  return t;
}

// nlines lines; strided: rows of `row` elements
template <typename T>
FftArgs<T> pass(int n, int64_t nlines, int64_t row = 512, int64_t zcol = 0) {
  FftArgs<T> a{};
  a.zcol = zcol;
  a.nlines = nlines;
  a.C = a.Sin = a.Sout = row;
  a.Din = a.Dout = n * row;
  return a;
}
// log2 of the most points (2^15 ... 2^27) of a pass over lines of n points
// that goes to the mixed-radix kernels, 0 for none; rows of a multiple of 128
// bytes, of one element more, and (z) half-spectrum columns in blocks
template <typename T>
void most(const char* prec, int n) {
  for (int strided = 0; strided < 2; ++strided)
    for (int mode : {M_C2C, M_R2C, M_C2R, M_DERIV, M_MULT})
      for (int odd = 0; odd < 3; ++odd) {
        int lg = 27;
        while (lg >= 15 && !mix_first(pass<T>(n, ((int64_t)1 << lg) / n, 512 + odd % 2, odd / 2 * 9), axis<T>(n), strided, mode)) --lg;
        printf("most_%s_%d_%c%d_%d %d\n", prec, n, strided ? 's' : 'z', mode, odd, lg < 15 ? 0 : lg);
      }
}

// a 512-point strided axis on the mixed-radix kernels
template <typename T>
void choices(const char* prec) {
  const int modes[3] = {M_C2C, M_MULT, M_DERIV};
  const char* names[3] = {"c2c", "mult", "deriv"};
  for (int s4v = -2; s4v < 1; ++s4v)
    for (int forced = 0; forced < 2; ++forced)
      for (int m = 0; m < 3; ++m)
        printf("mix512_%s_%s_%d_%d %d\n", prec, names[m], s4v, forced,
               (int)mix_first(pass<T>(512, 512 * 512), axis<T>(512, s4v, forced), true, modes[m]));
}

// an out-of-place 1 x 1 plan (kind 1 r2c, 2 c2c)
template <typename T>
accfft_amd_plan plan(int kind, int n0, int n1, int n2) {
  accfft_amd_plan p;
  p.kind = kind;
  p.n[0] = n0;
  p.n[1] = n1;
  p.n[2] = n2;
  p.fp = sizeof(T) == 4 ? ACCFFT_AMD_F32 : ACCFFT_AMD_F64;
  for (int ax = 0; ax < 3; ++ax) const_cast<AxisTab<T>&>(Ops<T>::tab(&p, ax)) = axis<T>(p.n[ax]);
  p.two = kind == 1 ? two_rows<T>(p.n) : two_rows_c2c<T>(p.n);
  return p;
}
// two-pass form with no choice, with one on x, with one on y; timed axes
template <typename T>
void tuning(const char* prec, int kind, int n0, int n1, int n2) {
  accfft_amd_plan p = plan<T>(kind, n0, n1, n2);
  printf("tune_%s_%d_%dx%dx%d two %d", prec, kind, n0, n1, n2, (int)Ops<T>::two(&p));
  for (int ax = 0; ax < 2; ++ax) {
    auto& t = const_cast<AxisTab<T>&>(Ops<T>::tab(&p, ax));
    t.s4v = -2;
    printf(" %d", (int)Ops<T>::two(&p));
    t.s4v = -1;
  }
  printf(" axes");
  for (const auto& q : Ops<T>::tune_passes(&p)) printf(" %d", q.ax);
  printf("\n");
}

// rows of pass 1, r2c and c2c
template <typename T>
void rows(const char* prec, int n0, int n1, int n2) {
  const int n[3] = {n0, n1, n2};
  printf("rows_%s_%dx%dx%d %d %d\n", prec, n0, n1, n2, two_rows<T>(n), two_rows_c2c<T>(n));
}

// columns of pass 2 that its tiles would leave over, and bytes its offsets
// span, over every plan of x length N0 that has one
template <typename T, int N0, int M>
void pass2(const char* prec) {
  int64_t left = 0, bytes = 0;
  int plans = 0;
  for (int kind = 1; kind < 3; ++kind)
    for (int n1 = 32; n1 <= 512; n1 *= 2)
      for (int n2 = 32; n2 <= 512; n2 *= 2) {
        const int n[3] = {N0, n1, n2};
        const int r = kind == 1 ? two_rows<T>(n) : two_rows_c2c<T>(n);
        if (!r || n1 / r != M) continue;
        const int64_t nh = kind == 1 ? n2 / 2 + 1 : n2;
        left += r * nh % XYCfg<T, N0, M, M_C2C>::W;
        bytes = std::max(bytes, (int64_t)N0 * n1 * nh * (int64_t)sizeof(cpx<T>));
        ++plans;
      }
  printf("pass2_%s_%d_%d %d %lld %lld\n", prec, N0, M, plans, (long long)left, (long long)bytes);
}
template <typename T>
void pass2(const char* prec) {
#define AFFT_N0(N) pass2<T, N, 2>(prec), pass2<T, N, 4>(prec), pass2<T, N, 8>(prec)
  AFFT_N0(32);
  AFFT_N0(64);
  AFFT_N0(128);
  AFFT_N0(256);
  AFFT_N0(512);
#undef AFFT_N0
}

}  // namespace

int main() {
  pass2<float>("f32");
  pass2<double>("f64");
  printf("modes %d %d %d %d %d\n", M_C2C, M_R2C, M_C2R, M_DERIV, M_MULT);
  for (int n : {16, 32, 64, 128, 256, 512, 1024}) {
    most<float>("f32", n);
    most<double>("f64", n);
  }
  for (int n0 : {1, 15, 16, 31, 32, 63, 64, 512})
    for (int n1 : {32, 64, 128})
      for (int n2 : {32, 128, 256, 512}) {
        rows<float>("f32", n0, n1, n2);
        rows<double>("f64", n0, n1, n2);
      }
  choices<float>("f32");
  choices<double>("f64");
  tuning<float>("f32", 1, 2048, 64, 512);
  tuning<double>("f64", 1, 512, 32, 256);
  tuning<float>("f32", 2, 1024, 64, 64);
  tuning<double>("f64", 2, 512, 64, 512);
  tuning<float>("f32", 1, 512, 512, 512);
  tuning<double>("f64", 1, 512, 512, 500);
  return 0;
}
