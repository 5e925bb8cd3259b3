// The rules by which a plan's passes choose their kernels, evaluated on the
// host (no kernel is instantiated or launched): prints "name value" lines
// for tests/test_route_rules.py.
#include <stdio.h>

#include "../../accfft_amd/csrc/dispatch.hpp"
#include "../../accfft_amd/csrc/exec.hpp"

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

// a 512-point strided axis on the mixed-radix kernels
template <typename T>
void choices(const char* prec) {
  const int modes[3] = {M_C2C, M_MULT, M_DERIV};
  const char* names[3] = {"c2c", "mult", "deriv"};
  for (int s4v = -2; s4v < 1; ++s4v)
    for (int forced = 0; forced < 2; ++forced)
      for (int m = 0; m < 3; ++m)
        printf("mix512_%s_%s_%d_%d %d\n", prec, names[m], s4v, forced,
               (int)mix_first(axis<T>(512, s4v, forced), true, modes[m]));
}

}  // namespace

int main() {
  choices<float>("f32");
  choices<double>("f64");
  return 0;
}
