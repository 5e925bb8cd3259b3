// fft_mix.hpp -- compile-time mixed-radix tiles: lengths with the prime
// factors 2, 3, 5 and 7, powers of two included where they are faster than
// the tiles of fft_kernels.hpp (mix_pow2 in fft_launch.hpp).
//
// A tile is L lines of N points.  N is split at compile time into two to
// four radices of at most 16 (mix_sched); every stage is a Stockham stage
// whose butterflies live in registers:
//   first stage   global memory -> registers -> LDS
//   middle stages LDS -> registers -> the same LDS buffer
//   last stage    LDS -> registers -> global memory
// so S stages cost S-1 LDS round trips on one buffer (the run-time engine
// of fft_device.hpp takes S+1 round trips on two buffers and forms every
// index at run time).  Strided tiles keep the L columns adjacent
// ([n][L], lanes along the columns), contiguous ones whole lines
// ([line][n], lanes along the line).
//
// The passes are bound by memory: 384^3 FP32 z r2c 84, y 82-87, x 76 us (5.2
// to 6.0 TB/s, a large copy reaches 5.1 and part of the reads come from the
// memory-side cache) and z c2r 100 us (4.5 TB/s; it loads each element of the
// half spectrum twice, for k and N - k) against 207 / 81-140 / 216 us in the
// run-time engine; 768^3 FP64 z r2c 1.34, y and x 1.41-1.53 ms (4.8-5.4 TB/s).
// Small grids are bound by the latency of one block's stages and the launch
// (64^3 FP64 x passes 4.3 us).
//
// LDS layout: one pad row (element) after every R0 = first radix, when R0
// is even.  The first stage writes with a stride of R0 rows, which padded is
// odd and spreads over the banks; all later accesses move in multiples of
// R0 rows, so the padded address stays linear in the radix index.
//
// The fused modes run the inverse as the forward stages backwards: the last
// stage's outputs j + r N/R are already in the registers of the thread that
// needs them, so symbol and inverse last stage follow without an exchange,
// and the inverse of every stage writes where its forward read.
#pragma once
#include "fft_kernels.hpp"

namespace afft {

// ------------------------------------------------------------ small DFTs
// R = A B with coprime A, B by the prime-factor map: n = (B n1 + A n2) mod
// R, k = the number with k = k1 mod A, k = k2 mod B; no twiddles.
template <typename T, int A, int B, int SIGN>
__device__ __forceinline__ void dft_pfa(cpx<T>* v) {
  constexpr int R = A * B;
  cpx<T> y[B][A];
#pragma unroll
  for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) y[n2][n1] = v[(B * n1 + A * n2) % R];
    dft<T, A, SIGN>(y[n2]);
  }
#pragma unroll
  for (int k1 = 0; k1 < A; ++k1) {
    cpx<T> z[B];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) z[n2] = y[n2][k1];
    dft<T, B, SIGN>(z);
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) {
      // the k < R with k % A == k1 and k % B == k2
      int k = k1;
#pragma unroll
      for (int m = 0; m < B; ++m)
        if (k % B != k2) k += A;
      v[k] = z[k2];
    }
  }
}
template <typename T, int R, int SIGN>
__device__ __forceinline__ void mdft(cpx<T>* v) {
  if constexpr (R == 6) dft_pfa<T, 2, 3, SIGN>(v);
  else if constexpr (R == 10) dft_pfa<T, 2, 5, SIGN>(v);
  else if constexpr (R == 12) dft_pfa<T, 4, 3, SIGN>(v);
  else if constexpr (R == 14) dft_pfa<T, 2, 7, SIGN>(v);
  else if constexpr (R == 15) dft_pfa<T, 3, 5, SIGN>(v);
  else if constexpr (R == 16) dft16q<T, SIGN>(v);
  else dft<T, R, SIGN>(v);
}

// ------------------------------------------------------------- schedule
struct MixSched {
  int s;     // stages, 0: no schedule
  int r[4];  // radices, largest first
};
constexpr bool mix_radix(int r) { return (r >= 2 && r <= 10) || r == 12 || (r >= 14 && r <= 16); }
// The fewest stages whose radices are at most 16, and among those the
// smallest largest radix (fewest registers).
// `most`: the largest radix allowed.
constexpr MixSched mix_search(int n, int most) {
  MixSched best{0, {1, 1, 1, 1}};
  for (int a = 2; a <= most && !best.s; ++a) {
    if (!mix_radix(a) || n % a) continue;
    const int b = n / a;
    if (b <= a && mix_radix(b)) best = MixSched{2, {a, b, 1, 1}};
  }
  for (int a = 2; a <= most && !best.s; ++a) {
    if (!mix_radix(a) || n % a) continue;
    for (int b = a; b >= 2 && !best.s; --b) {
      if (!mix_radix(b) || (n / a) % b) continue;
      const int c = n / a / b;
      if (c <= b && c >= 2 && mix_radix(c)) best = MixSched{3, {a, b, c, 1}};
    }
  }
  for (int a = 2; a <= most && !best.s; ++a) {
    if (!mix_radix(a) || n % a) continue;
    for (int b = a; b >= 2 && !best.s; --b) {
      if (!mix_radix(b) || (n / a) % b) continue;
      for (int c = b; c >= 2 && !best.s; --c) {
        if (!mix_radix(c) || (n / a / b) % c) continue;
        const int d = n / a / b / c;
        if (d <= c && d >= 2 && mix_radix(d)) best = MixSched{4, {a, b, c, d}};
      }
    }
  }
  return best;
}
// FP64 from 256 points: radices up to 10, more stages with half the
// registers (256^3 derivative passes 83 -> 57 us, z r2c 93 -> 69 us, 960^3
// strided passes 4.2 -> 3.3 ms, 768^3 1.58-1.69 -> 1.43-1.56 ms); shorter
// lines lose by the extra exchange (240^3 derivatives 49 -> 75 us).
template <typename T>
constexpr MixSched mix_sched(int n) {
  if (sizeof(T) == 8 && n >= 256) {
    const MixSched m = mix_search(n, 10);
    if (m.s) return m;
  }
  return mix_search(n, 16);
}
constexpr int mix_ns(const MixSched& m, int s) {  // span before stage s
  int ns = 1;
  for (int i = 0; i < s; ++i) ns *= m.r[i];
  return ns;
}
constexpr int mix_twoff(const MixSched& m, int s) {  // twiddle table offset of stage s
  int off = 0;
  for (int i = 1; i < s; ++i) off += (m.r[i] - 1) * mix_ns(m, i);
  return off;
}
constexpr int mix_twn(const MixSched& m) { return mix_twoff(m, m.s); }

// Work of a block of t threads and L lines, threads without a butterfly
// included, summed over the stages.
constexpr long mix_cost(const MixSched& m, int n, int l, int t) {
  long c = 0;
  for (int s = 0; s < m.s; ++s) {
    const int b = n / m.r[s] * l;
    c += (long)((b + t - 1) / t) * t * m.r[s];
  }
  return c;
}
// Threads per block for L lines: the multiple of the wavefront up to 512 that
// holds at most `most` elements a thread and wastes least.
constexpr int mix_tpb(const MixSched& m, int n, int l, int most) {
  int best = 0;
  long cost = 0;
  for (int t = 64; t <= 512; t += 64) {
    if (t < 512 && (long)n * l > (long)most * t) continue;
    const long c = mix_cost(m, n, l, t);
    if (!best || c * 100 < cost * 97) {
      best = t;
      cost = c;
    }
  }
  return best;
}
// Lines of a contiguous tile: of l / 2 ... 4 l / 3, those that waste least.
constexpr int mix_lines(const MixSched& m, int n, int l, int most) {
  int best = l;
  for (int k = l / 2 > 2 ? l / 2 : 2; k <= l + l / 3 && k <= 32; ++k) {
    const long c = mix_cost(m, n, k, mix_tpb(m, n, k, most)) * best;
    const long b = mix_cost(m, n, best, mix_tpb(m, n, best, most)) * k;
    if (c * 100 < b * 97) best = k;
  }
  return best;
}

// Strided tiles: the widest power-of-two column count whose buffer stays
// within 52 KiB (three workgroups per CU) and whose row segments are at most
// 128 bytes, 256 for FP64 lengths from 256.  Those of three stages and more
// exchange real and imaginary parts in turn (HALF): with whole-tile
// exchanges only two workgroups fit, 384^3 FP32 y / x passes 100 / 85 ->
// 88 / 78 us, FP64 202 / 213 -> 175 / 188 us, and 151 / 175 us with 256-byte
// segments (FP32: 90 / 80 us with those); 768^3 FP64 1934 / 2055 -> 1604 /
// 1659 us, whose 64-byte segments become 128-byte ones.  Lengths below 256
// fit as they are (200^3 FP32 round trip 92 us, 97 us with HALF).
template <typename T, int N>
struct MixS {
  static constexpr bool HALF = mix_sched<T>(N).s > 2 && N >= 256;
  static constexpr int SEG = sizeof(T) == 8 && HALF ? 256 : 128;
  static constexpr int cols() {
    int w = 1;
    const int es = HALF ? sizeof(T) : sizeof(cpx<T>);
    while (w * 2 * (int)sizeof(cpx<T>) <= SEG && (long)w * 2 * N * es <= 52 * 1024) w *= 2;
    return w;
  }
  static constexpr int L = cols();
  static constexpr int TPB = mix_tpb(mix_sched<T>(N), N, L, sizeof(T) == 4 ? 24 : 12);
};
// Contiguous tiles: about 1152 elements and at least two lines above 256
// points (the staged twiddle table is about one line long: 768^3 FP64 z r2c
// 1694 us with two, 1949 with four lines a block, FP32 384^3 93 us with
// three, 103 with six), 2304 elements up to 256 (200^3 FP64 27 us with
// eleven lines, 31 with five).
// Derivative passes from 192 points, which spend their time in butterflies,
// take the line count that leaves the fewest threads idle (256 points: eight
// lines fill 128 threads, nine leave a quarter idle; FP32 32.6 -> 29.5 us,
// 240 points 31.0 -> 26.2 us); the other passes and shorter lines are up to
// 10 % faster with the idle threads, which share the loads and stores.
template <typename T, int N, int MODE>
struct MixZ {
  static constexpr int most = N > 256 ? 1152 : 2304;
  static constexpr int L0 = most / N > 2 ? (most / N > 32 ? 32 : most / N) : 2;
  static constexpr int R0 = mix_sched<T>(N).r[0], E = sizeof(T) == 4 ? 12 : 8;
  static constexpr int L = MODE == M_DERIV && N >= 192 ? mix_lines(mix_sched<T>(N), N, L0, R0 > E ? R0 : E) : L0;
  static constexpr int TPB = mix_tpb(mix_sched<T>(N), N, L, R0 > E ? R0 : E);
};

// ---------------------------------------------------------------- engine
// HALF: the exchanges move the real parts, then the imaginary parts, through
// a buffer of half the tile (twice the barriers, twice the workgroups or
// columns per CU).
template <typename T, int N, int L, int TPB, bool STR, bool HALF = false>
struct Mix {
  static constexpr MixSched SC = mix_sched<T>(N);
  static constexpr int S = SC.s;
  static_assert(S >= 2, "no schedule for this length");
  static constexpr int R0 = SC.r[0];
  static constexpr int PAD = R0 % 2 == 0 ? 1 : 0;
  static constexpr int LP = N + PAD * (N / R0);  // padded line
  static constexpr int ELEMS = L * LP;
  static constexpr int TWN = mix_twn(SC);
  template <int s>
  struct St {
    static constexpr int R = SC.r[s], NB = N / R, NS = mix_ns(SC, s), OFF = mix_twoff(SC, s);
    static constexpr int B = NB * L, PER = (B + TPB - 1) / TPB;
    static constexpr bool FULL = B % TPB == 0;
    // butterfly i of this thread -> line, j; false past the last one
    static __device__ __forceinline__ bool map(int i, int& line, int& j) {
      const int b = (int)threadIdx.x + i * TPB;
      if constexpr (STR) {
        line = b % L;
        j = b / L;
      } else {
        line = b / NB;
        j = b % NB;
      }
      return FULL || b < B;
    }
  };
  using Last = St<S - 1>;
  // padded row / element of n
  static __device__ __forceinline__ int P(int n) { return PAD ? n + n / R0 : n; }
  static __device__ __forceinline__ int at(int line, int p) { return STR ? p * L + line : line * LP + p; }
  static constexpr int ES = STR ? L : 1;

  // stage s reads x[j + r NB] (s >= 1): base and step of r
  template <int s>
  static __device__ __forceinline__ int rbase(int line, int j) { return at(line, P(j)); }
  template <int s>
  static constexpr int rstep() { return (St<s>::NB + PAD * (St<s>::NB / R0)) * ES; }
  // and writes y[(j - k) R + k + r NS], k = j mod NS
  template <int s>
  static __device__ __forceinline__ int wbase(int line, int j) {
    if constexpr (s == 0) {
      return at(line, j * (R0 + PAD));
    } else {
      constexpr int NS = St<s>::NS, R = St<s>::R;
      const int m = j / NS, k = j - m * NS;
      return at(line, m * (NS * R + PAD * (NS * R / R0)) + P(k));
    }
  }
  template <int s>
  static constexpr int wstep() {
    return s == 0 ? ES : (St<s>::NS + PAD * (St<s>::NS / R0)) * ES;
  }
  template <int s, int SIGN>
  static __device__ __forceinline__ void twiddle(cpx<T>* v, int j, const cpx<T>* tw) {
    const int k = j % St<s>::NS;
#pragma unroll
    for (int r = 1; r < St<s>::R; ++r) {
      const cpx<T> w = tw[St<s>::OFF + (r - 1) * St<s>::NS + k];
      v[r] = SIGN < 0 ? cmul(v[r], w) : cmulc(v[r], w);
    }
  }

  template <int s>
  using Regs = cpx<T>[St<s>::PER][St<s>::R];
  using BufT = typename std::conditional<HALF, T, cpx<T>>::type;

  // fn(i, p): for each butterfly i of stage s that exists, the LDS position
  // of its inputs (W = false) or outputs (W = true)
  template <int s, bool W, typename F>
  static __device__ __forceinline__ void each(F&& fn) {
#pragma unroll
    for (int i = 0; i < St<s>::PER; ++i) {
      int line, j;
      if (St<s>::map(i, line, j)) fn(i, W ? wbase<s>(line, j) : rbase<s>(line, j));
    }
  }
  template <int s, bool W, int PART>
  static __device__ __forceinline__ void write(const Regs<s>& v, BufT* buf) {
    constexpr int D = W ? wstep<s>() : rstep<s>();
    each<s, W>([&](int i, int p) {
#pragma unroll
      for (int r = 0; r < St<s>::R; ++r) {
        if constexpr (!HALF) buf[p + r * D] = v[i][r];
        else buf[p + r * D] = PART == 0 ? v[i][r].x : v[i][r].y;
      }
    });
  }
  template <int s, bool W, int PART>
  static __device__ __forceinline__ void read(Regs<s>& v, const BufT* buf) {
    constexpr int D = W ? wstep<s>() : rstep<s>();
    each<s, W>([&](int i, int p) {
#pragma unroll
      for (int r = 0; r < St<s>::R; ++r) {
        if constexpr (!HALF) v[i][r] = buf[p + r * D];
        else if constexpr (PART == 0) v[i][r].x = buf[p + r * D];
        else v[i][r].y = buf[p + r * D];
      }
    });
  }
  // a, stage s's results, to b, the operands of stage q: forward (q = s + 1)
  // through the positions stage s writes and q reads, backward (q = s - 1)
  // through those s read and q wrote.  sync: the buffer may still be read.
  template <int s, int q>
  static __device__ __forceinline__ void exchange(const Regs<s>& a, Regs<q>& b, BufT* buf, bool sync) {
    constexpr bool W = q > s;
    if (sync) __syncthreads();
    write<s, W, 0>(a, buf);
    __syncthreads();
    read<q, !W, 0>(b, buf);
    if constexpr (HALF) {
      __syncthreads();
      write<s, W, 1>(a, buf);
      __syncthreads();
      read<q, !W, 1>(b, buf);
    }
  }
  template <int s>
  static __device__ __forceinline__ void butterflies(Regs<s>& v, const cpx<T>* tw) {
#pragma unroll
    for (int i = 0; i < St<s>::PER; ++i) {
      int line, j;
      (void)St<s>::map(i, line, j);
      if constexpr (s > 0) twiddle<s, -1>(v[i], j, tw);
      mdft<T, St<s>::R, -1>(v[i]);
    }
  }
  template <int s>
  static __device__ __forceinline__ void inverse_butterflies(Regs<s>& v, const cpx<T>* tw) {
#pragma unroll
    for (int i = 0; i < St<s>::PER; ++i) {
      int line, j;
      (void)St<s>::map(i, line, j);
      mdft<T, St<s>::R, +1>(v[i]);
      if constexpr (s > 0) twiddle<s, +1>(v[i], j, tw);
    }
  }

  // Forward transform: v holds x[j + r N/R0] of the first stage, o ends with
  // the last stage's outputs X[j + r N/R].
  static __device__ __forceinline__ void forward(Regs<0>& v, Regs<S - 1>& o, BufT* buf, const cpx<T>* tw) {
    butterflies<0>(v, tw);
    if constexpr (S == 2) {
      exchange<0, 1>(v, o, buf, false);
    } else {
      Regs<1> x;
      exchange<0, 1>(v, x, buf, false);
      butterflies<1>(x, tw);
      if constexpr (S == 3) {
        exchange<1, 2>(x, o, buf, true);
      } else {
        Regs<2> y;
        exchange<1, 2>(x, y, buf, true);
        butterflies<2>(y, tw);
        exchange<2, 3>(y, o, buf, true);
      }
    }
    butterflies<S - 1>(o, tw);
  }
  // Inverse transform from the registers forward() ended in, by the forward
  // stages backwards; ends with x[j + r N/R0] in v.  (Its first exchange
  // needs no barrier: a thread writes only where it alone has read.)
  static __device__ __forceinline__ void backward(Regs<S - 1>& o, Regs<0>& v, BufT* buf, const cpx<T>* tw) {
    inverse_butterflies<S - 1>(o, tw);
    if constexpr (S == 2) {
      exchange<1, 0>(o, v, buf, false);
    } else if constexpr (S == 3) {
      Regs<1> x;
      exchange<2, 1>(o, x, buf, false);
      inverse_butterflies<1>(x, tw);
      exchange<1, 0>(x, v, buf, true);
    } else {
      Regs<2> y;
      exchange<3, 2>(o, y, buf, false);
      inverse_butterflies<2>(y, tw);
      Regs<1> x;
      exchange<2, 1>(y, x, buf, true);
      inverse_butterflies<1>(x, tw);
      exchange<1, 0>(x, v, buf, true);
    }
    inverse_butterflies<0>(v, tw);
  }
};

// The twiddle table into LDS: all of the thread's loads first (clamped, not
// conditional: a conditionally written register array goes to scratch).
template <typename T, int TWN, int TPB>
__device__ __forceinline__ void mix_twiddles(cpx<T>* dst, const cpx<T>* __restrict__ src, int t) {
  constexpr int E = (TWN + TPB - 1) / TPB;
  cpx<T> v[E];
#pragma unroll
  for (int j = 0; j < E; ++j) {
    const int i = t + j * TPB;
    v[j] = src[i < TWN ? i : TWN - 1];
  }
#pragma unroll
  for (int j = 0; j < E; ++j)
    if (t + j * TPB < TWN) dst[t + j * TPB] = v[j];
}

// The sign of the imaginary parts: conj(F(conj x)) is the inverse transform,
// so one forward kernel serves both directions (one XOR per element on the
// way in and out, exact).
template <typename T>
__device__ __forceinline__ cpx<T> conj_if(cpx<T> a, unsigned flip) {
  if constexpr (sizeof(T) == 4) {
    a.y = __uint_as_float(__float_as_uint(a.y) ^ flip);
  } else {
    const uint64_t b = (uint64_t)__double_as_longlong(a.y) ^ ((uint64_t)flip << 32);
    a.y = __longlong_as_double((long long)b);
  }
  return a;
}

// A grad or laplace-family symbol on one column of a M_MULT pass: the two
// fixed axes' part once per thread, the varying axis's wavenumber per
// element, factors in FP64 as apply_sym forms them (sums of squares below
// 2^53, so every step is exact up to the same one rounding).
struct MixSym {
  double fixed = 0;  // laplace family: w^2 of the fixed axes; grad: their w
  double scale;
  bool on_k;  // grad: along the varying axis
  template <typename T>
  __device__ __forceinline__ MixSym(const FftArgs<T>& a, int64_t col)
      : MixSym(a, (long)(col / a.Ch), (long)(col % a.Ch)) {}
  // u: wavenumber index of the other full axis, Z: along z
  template <typename T>
  __device__ __forceinline__ MixSym(const FftArgs<T>& a, long u, long Z) {
    const long Nu = a.maxis == 0 ? a.N1 : a.N0;
    scale = a.scale;
    on_k = a.sym == (a.maxis == 0 ? SYM_GRAD_X : SYM_GRAD_Y);
    if (a.sym <= SYM_GRAD_Z) {
      fixed = a.sym == SYM_GRAD_Z ? (double)wave_nyq0(Z, a.N2) : (double)wave_nyq0(u, Nu);
    } else if (a.sym == SYM_INV_BIHARMONIC) {
      const double wu = (double)(u > Nu / 2 ? u - Nu : u), wz = (double)(Z > a.N2 / 2 ? Z - a.N2 : Z);
      fixed = wu * wu + wz * wz;
    } else {
      const double wu = (double)wave_nyq0(u, Nu), wz = (double)wave_nyq0(Z, a.N2);
      fixed = wu * wu + wz * wz;
    }
  }
  template <int KIND, typename T>
  __device__ __forceinline__ cpx<T> mul(int k, int n, cpx<T> v) const {
    int w = k > n / 2 ? k - n : k;
    if (KIND != SYM_INV_BIHARMONIC && k == n / 2) w = 0;
    if constexpr (KIND == SYM_GRAD_X) {  // any grad
      const T f = (T)(scale * (on_k ? (double)w : fixed));
      return {-f * v.y, f * v.x};
    } else {
      const double wave = -(double)(w * w) - fixed;
      double f;
      if constexpr (KIND == SYM_LAPLACE) f = wave;
      else if constexpr (KIND == SYM_BIHARMONIC) f = wave * wave;
      else if constexpr (KIND == SYM_INV_LAPLACE) f = wave == 0 ? 0.0 : 1.0 / wave;
      else f = wave == 0 ? 1.0 : 1.0 / (wave * wave);
      const T g = (T)(scale * f);
      return {g * v.x, g * v.y};
    }
  }
};

// ------------------------------------------------------- strided columns
// M_C2C, M_MULT (grad and laplace-family symbols), M_DERIV (the complex view
// of adjacent real columns: even counts and strides, checked by the
// launcher).  sign: of a M_C2C transform.
template <typename T, int N, int MODE>
__global__ void __launch_bounds__((MixS<T, N>::TPB))
    mix_s_kernel(FftArgs<T> a, unsigned flip) {
  using CF = MixS<T, N>;
  using E = Mix<T, N, CF::L, CF::TPB, true, CF::HALF>;
  using S0 = typename E::template St<0>;
  using SL = typename E::Last;
  constexpr int L = CF::L, TPB = CF::TPB;
  __shared__ typename E::BufT buf[E::ELEMS];
  __shared__ cpx<T> tw[E::TWN];
  const int t = threadIdx.x;
  int64_t tile = xcd_tile(blockIdx.x, gridDim.x, (unsigned)a.xgroup);
  if (a.reverse) tile = (int64_t)gridDim.x - 1 - tile;
  // TPB is a multiple of L (both powers of two times a wavefront), so a
  // thread keeps its column
  static_assert(TPB % L == 0, "a thread keeps its column");
  const int64_t col = tile * L + t % L;
  const bool ok = col < a.nlines;
  const int64_t u = col / a.C, c = col - u * a.C;
  cpx<T> v[S0::PER][S0::R];
  {
    const cpx<T>* src = reinterpret_cast<const cpx<T>*>(a.in) + u * a.Din + c;
    const int64_t step = (int64_t)S0::NB * a.Sin;
#pragma unroll
    for (int i = 0; i < S0::PER; ++i) {
      int line, j;
      const bool in = S0::map(i, line, j) && ok;
      gptr<const cpx<T>> p = to_global(src + (int64_t)j * a.Sin);
#pragma unroll
      for (int r = 0; r < S0::R; ++r) {
        v[i][r] = in ? ld_global(p) : cpx<T>{(T)0, (T)0};
        p += step;
        asm volatile("" : "+v"(p));
      }
    }
  }
  mix_twiddles<T, E::TWN, TPB>(tw, a.tw, t);
  if constexpr (MODE == M_C2C) {
#pragma unroll
    for (int i = 0; i < S0::PER; ++i)
#pragma unroll
      for (int r = 0; r < S0::R; ++r) v[i][r] = conj_if(v[i][r], flip);
  }
  cpx<T> o[SL::PER][SL::R];
  E::forward(v, o, buf, tw);
  cpx<T>* dst = reinterpret_cast<cpx<T>*>(a.out) + u * a.Dout + c;
  if constexpr (MODE == M_C2C) {
    const int64_t step = (int64_t)SL::NB * a.Sout;
#pragma unroll
    for (int i = 0; i < SL::PER; ++i) {
      int line, j;
      if (SL::map(i, line, j) && ok) {
        gptr<cpx<T>> p = to_global(dst + (int64_t)j * a.Sout);
#pragma unroll
        for (int r = 0; r < SL::R; ++r) {
          *p = conj_if(o[i][r], flip);
          p += step;
          asm volatile("" : "+v"(p));
        }
      }
    }
    return;
  } else {
    // symbol at k = j + r N/R of this thread's column
    if constexpr (MODE == M_DERIV) {
#pragma unroll
      for (int i = 0; i < SL::PER; ++i) {
        int line, j;
        (void)SL::map(i, line, j);
#pragma unroll
        for (int r = 0; r < SL::R; ++r) {
          const T f = (T)(a.scale * (double)(int)wave_sym(j + r * SL::NB, N));
          o[i][r] = cpx<T>{-f * o[i][r].y, f * o[i][r].x};
        }
      }
    } else {
      const MixSym sym(a, col);
      auto apply = [&](auto kind) {
#pragma unroll
        for (int i = 0; i < SL::PER; ++i) {
          int line, j;
          (void)SL::map(i, line, j);
#pragma unroll
          for (int r = 0; r < SL::R; ++r)
            o[i][r] = sym.template mul<decltype(kind)::value>(j + r * SL::NB, N, o[i][r]);
        }
      };
      switch (a.sym) {  // uniform: one loop per kind
        case SYM_LAPLACE: apply(std::integral_constant<int, SYM_LAPLACE>{}); break;
        case SYM_BIHARMONIC: apply(std::integral_constant<int, SYM_BIHARMONIC>{}); break;
        case SYM_INV_LAPLACE: apply(std::integral_constant<int, SYM_INV_LAPLACE>{}); break;
        case SYM_INV_BIHARMONIC: apply(std::integral_constant<int, SYM_INV_BIHARMONIC>{}); break;
        default: apply(std::integral_constant<int, SYM_GRAD_X>{}); break;
      }
    }
    E::backward(o, v, buf, tw);
    const int64_t step = (int64_t)S0::NB * a.Sout;
#pragma unroll
    for (int i = 0; i < S0::PER; ++i) {
      int line, j;
      if (S0::map(i, line, j) && ok) {
        gptr<cpx<T>> p = to_global(dst + (int64_t)j * a.Sout);
        if (MODE == M_DERIV && a.accumulate) {
          cpx<T> w[S0::R];
          gptr<const cpx<T>> q = p;
#pragma unroll
          for (int r = 0; r < S0::R; ++r) {
            w[r] = ld_global(q);
            q += step;
            asm volatile("" : "+v"(q));
          }
#pragma unroll
          for (int r = 0; r < S0::R; ++r) v[i][r] = cadd(w[r], v[i][r]);
        }
#pragma unroll
        for (int r = 0; r < S0::R; ++r) {
          *p = v[i][r];
          p += step;
          asm volatile("" : "+v"(p));
        }
      }
    }
  }
}

// ------------------------------------------------------ contiguous lines
// M_C2C, M_R2C, M_C2R, M_DERIV of the z pass; a line of the real modes is a
// pair of real lines.
template <typename T, int N, int MODE>
__global__ void __launch_bounds__((MixZ<T, N, MODE>::TPB))
    mix_z_kernel(FftArgs<T> a, unsigned flip) {
  using CF = MixZ<T, N, MODE>;
  using E = Mix<T, N, CF::L, CF::TPB, false>;
  using S0 = typename E::template St<0>;
  using SL = typename E::Last;
  constexpr int L = CF::L, TPB = CF::TPB, NH = N / 2 + 1;
  __shared__ typename E::BufT buf[E::ELEMS];
  __shared__ cpx<T> tw[E::TWN];
  const int t = threadIdx.x;
  const int64_t bx = xcd_tile(blockIdx.x, gridDim.x, (unsigned)a.xgroup);
  const int64_t l0 = (a.reverse ? (int64_t)gridDim.x - 1 - bx : bx) * L;
  const int64_t nl = a.nlines;
  cpx<T> v[S0::PER][S0::R];
  if constexpr (MODE == M_C2R) {
    cpx<T> w[S0::PER][S0::R];
#pragma unroll
    for (int i = 0; i < S0::PER; ++i) {
      int line, j;
      const bool in = S0::map(i, line, j);
      const int64_t ga = 2 * (l0 + line), gb = ga + 1;
#pragma unroll
      for (int r = 0; r < S0::R; ++r) {
        const int n = j + r * S0::NB, k = n < NH ? n : N - n;
        v[i][r] = w[i][r] = cpx<T>{(T)0, (T)0};
        if (in && ga < nl) v[i][r] = ldc<T>(a.in, zcol_off(a, ga, a.idist, k, NH));
        if (in && gb < nl) w[i][r] = ldc<T>(a.in, zcol_off(a, gb, a.idist, k, NH));
      }
    }
    mix_twiddles<T, E::TWN, TPB>(tw, a.tw, t);
    // Z = A + i B below the middle, conj(A) + i conj(B) above; conjugated
    // (the transform is conj(F(conj Z)), whose real and imaginary parts are
    // the two lines)
#pragma unroll
    for (int i = 0; i < S0::PER; ++i) {
      int line, j;
      (void)S0::map(i, line, j);
#pragma unroll
      for (int r = 0; r < S0::R; ++r) {
        const int n = j + r * S0::NB, k = n < NH ? n : N - n;
        cpx<T> A = v[i][r], B = w[i][r];
        if (k == 0 || 2 * k == N) {
          A.y = (T)0;
          B.y = (T)0;
        } else if (a.adjw) {
          A = cscale(A, (T)0.5);
          B = cscale(B, (T)0.5);
        }
        v[i][r] = n < NH ? cpx<T>{A.x - B.y, -(A.y + B.x)} : cpx<T>{A.x + B.y, A.y - B.x};
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < S0::PER; ++i) {
      int line, j;
      const bool in = S0::map(i, line, j);
#pragma unroll
      for (int r = 0; r < S0::R; ++r) {
        const int n = j + r * S0::NB;
        v[i][r] = cpx<T>{(T)0, (T)0};
        if constexpr (MODE == M_C2C) {
          const int64_t g = l0 + line;
          if (in && g < nl) v[i][r] = ldc<T>(a.in, g * a.idist + n);
        } else {
          const int64_t ga = 2 * (l0 + line), gb = ga + 1;
          if (in && ga < nl) v[i][r].x = ldr<T>(a.in, ga * a.idist + n);
          if (in && gb < nl) v[i][r].y = ldr<T>(a.in, gb * a.idist + n);
        }
      }
    }
    mix_twiddles<T, E::TWN, TPB>(tw, a.tw, t);
    if constexpr (MODE == M_C2C) {
#pragma unroll
      for (int i = 0; i < S0::PER; ++i)
#pragma unroll
        for (int r = 0; r < S0::R; ++r) v[i][r] = conj_if(v[i][r], flip);
    }
  }
  cpx<T> o[SL::PER][SL::R];
  E::forward(v, o, buf, tw);
  if constexpr (MODE == M_C2C || MODE == M_C2R) {
#pragma unroll
    for (int i = 0; i < SL::PER; ++i) {
      int line, j;
      if (!SL::map(i, line, j)) continue;
#pragma unroll
      for (int r = 0; r < SL::R; ++r) {
        const int n = j + r * SL::NB;
        if constexpr (MODE == M_C2C) {
          const int64_t g = l0 + line;
          if (g < nl) stc<T>(a.out, g * a.odist + n, conj_if(o[i][r], flip));
        } else {
          const int64_t ga = 2 * (l0 + line), gb = ga + 1;
          if (ga < nl) str<T>(a.out, ga * a.odist + n, o[i][r].x);
          if (gb < nl) str<T>(a.out, gb * a.odist + n, -o[i][r].y);
        }
      }
    }
  } else if constexpr (MODE == M_R2C) {
    E::template write<E::S - 1, false, 0>(o, buf);
    __syncthreads();
    constexpr int EH = (2 * L * NH + TPB - 1) / TPB;
#pragma unroll
    for (int i = 0; i < EH; ++i) {
      const int e = t + i * TPB;
      if (e >= 2 * L * NH) break;
      const int rl = e / NH, k = e - rl * NH;
      const int64_t g = 2 * l0 + rl;
      if (g >= nl) continue;
      const cpx<T> z1 = buf[E::at(rl >> 1, E::P(k))];
      const cpx<T> z2 = buf[E::at(rl >> 1, E::P(k == 0 ? 0 : N - k))];
      const T h = (T)0.5;
      cpx<T> x;
      if ((rl & 1) == 0) x = {h * (z1.x + z2.x), h * (z1.y - z2.y)};
      else x = {h * (z1.y + z2.y), h * (z2.x - z1.x)};
      if (a.adjw && k != 0 && 2 * k != N) x = cscale(x, (T)2);
      stc<T>(a.out, zcol_off(a, g, a.odist, k, NH), x);
    }
  } else {  // M_DERIV
#pragma unroll
    for (int i = 0; i < SL::PER; ++i) {
      int line, j;
      (void)SL::map(i, line, j);
#pragma unroll
      for (int r = 0; r < SL::R; ++r) {
        const T f = (T)(a.scale * (double)(int)wave_sym(j + r * SL::NB, N));
        o[i][r] = cpx<T>{-f * o[i][r].y, f * o[i][r].x};
      }
    }
    E::backward(o, v, buf, tw);
#pragma unroll
    for (int i = 0; i < S0::PER; ++i) {
      int line, j;
      if (!S0::map(i, line, j)) continue;
      const int64_t ga = 2 * (l0 + line), gb = ga + 1;
      if (a.accumulate) {
        cpx<T> w[S0::R];
#pragma unroll
        for (int r = 0; r < S0::R; ++r) {
          const int n = j + r * S0::NB;
          w[r].x = ga < nl ? ldr<T>(a.out, ga * a.odist + n) : (T)0;
          w[r].y = gb < nl ? ldr<T>(a.out, gb * a.odist + n) : (T)0;
        }
#pragma unroll
        for (int r = 0; r < S0::R; ++r) v[i][r] = cadd(w[r], v[i][r]);
      }
#pragma unroll
      for (int r = 0; r < S0::R; ++r) {
        const int n = j + r * S0::NB;
        if (ga < nl) str<T>(a.out, ga * a.odist + n, v[i][r].x);
        if (gb < nl) str<T>(a.out, gb * a.odist + n, v[i][r].y);
      }
    }
  }
}

}  // namespace afft
