// fft_two.hpp -- 3-D transforms of power-of-two grids in two passes over HBM.
//
// With N1 = R M, the y transform is split R x M (y = n2 + M n1,
// ky = k1 + R k2):
//   pass 1 (two_zy)  for each (x, n2): z transform of the R rows n2 + M n1,
//                    R-point DFT over n1, twiddle exp(-2 pi i n2 k1 / N1),
//                    to the rows k1 + R n2;
//   pass 2 (two_xy)  for each column (k1, kz): the M-point DFT over n2
//                    (rows k1 + R n2 -> k1 + R k2, in place) and the x
//                    transform.
// A workgroup transforms 4 to 256 KiB of a pass at once, held in registers
// (a CU has 512 KiB of them); the LDS only exchanges real, then imaginary
// parts between stages.  Against one pass per axis this reads and writes the
// spectrum once less in each direction: R + 3 C bytes instead of R + 5 C.
//
// What bounds them (512^3 FP32, a large copy runs at 5.1 TB/s): pass 1 runs
// at 5.1 TB/s (209 / 212 us r2c / c2r, two workgroups of 512 threads per CU);
// pass 2 at 3.85-4.2 TB/s (279 / 259 us): one 256 KiB tile fills a CU, so
// its 10 us of vector and 3 us of LDS time a tile are not hidden, and a copy
// with its access pattern (64-byte segments of 4096 rows) reaches 4.5 TB/s.
// One pass per axis takes 181 + 169 + 203 us forward.  Staggered starts of
// the workgroups and 32-byte segments with two workgroups per CU measured no
// faster.
#pragma once
#include "fft_mix.hpp"

namespace afft {

// Element at 32-bit byte offset `off` of a uniform base: the base stays in
// scalar registers (scalar arithmetic for the row steps) and a thread keeps
// one offset register for all of its loads.  Pass 1 has a 64-bit base for
// each plane (at most 4 MB of offsets); in pass 2 the offsets span the grid,
// at most 1.08 GB (the 512^3 half spectrum in FP64; c2c 1.07 GB, 512^3 in
// FP32 and 512 x 256 x 512 in FP64).
template <typename V, typename B>
__device__ __forceinline__ gptr<V> at_off(B* base, uint32_t off) {
  return (gptr<V>)((gptr<typename std::conditional<std::is_const<B>::value, const char, char>::type>)base + off);
}

template <typename T, int R, int SIGN>
__device__ __forceinline__ void pdft(cpx<T>* v) {
  if constexpr (R == 1) return;
  else if constexpr (R == 16) dft16q<T, SIGN>(v);
  else if constexpr (R == 32) dft32<T, SIGN>(v);
  else dft<T, R, SIGN>(v);
}

// ------------------------------------------------------------------ pass 2
// Tile: W adjacent columns x M rows n2 x N0 rows x.  A thread's first
// butterflies are R0 values of x for each of the M values of n2, so the
// M-point y DFT runs in the same registers; two more x stages R1, R2 follow
// (R1, R2 = 1 where N0 is short).  LDS position of (x, n2, c): row x of
// L = M W values, the n2 groups rotated by XOR with x / R0: the first stage
// writes M consecutive j = x / R0 from one wavefront, which would otherwise
// fall on the same W banks.
template <typename T, int N0, int M, int MODE>
struct XYCfg {
  // 64-byte row segments for tiles of 1024 rows and more (FP64: 128 bytes
  // below 4096 rows), 128 bytes for shorter ones
  static constexpr int W = sizeof(T) == 4 ? (M * N0 >= 1024 ? 8 : 16) : (M * N0 >= 4096 ? 4 : 8);
  // elements a thread: 64 registers of data; the FP32 multiply of short
  // tiles half of that (it needs registers for the symbol and the way back:
  // 128^3 16.3 -> 13.3 us, from 1024 rows 43 us with 32, 45 with 16)
  // (and of 32-point x axes, whose blocks would fall below a wavefront)
  static constexpr int E = sizeof(T) == 8 ? (N0 * M <= 64 ? 8 : 16)
                           : N0 <= 32 || (MODE == M_MULT && M * N0 < 1024) ? 16 : 32;
  // waves per SIMD of the multiply: three leave it 168 registers, with four
  // it spills 30 to 70 (256^3 FP32 52 against 42 us)
  static constexpr int MULT_WAVES = 3;
  static constexpr int R0 = E / M;
  static constexpr int NR = N0 / R0;  // left for R1 R2
  static constexpr int R2 = NR <= 16 ? 1 : NR <= 64 ? 8 : 16;
  static constexpr int R1 = NR / R2;
  static constexpr int TPB = NR * W;
};
template <typename T, int N0, int M, int MODE>
struct XYTile {
  using CF = XYCfg<T, N0, M, MODE>;
  static constexpr int W = CF::W, TPB = CF::TPB, R0 = CF::R0, R1 = CF::R1, R2 = CF::R2, L = M * W;
  static constexpr int NB1 = N0 / R1, P1 = NB1 * L / TPB, NB2 = N0 / R2, P2 = NB2 * L / TPB;
  static constexpr int NS1 = R0, NS2 = R0 * R1;
  static constexpr int OFF2 = (R1 - 1) * NS1;
  static constexpr int TWN = OFF2 + (R2 > 1 ? (R2 - 1) * NS2 : 0);
  static constexpr int S = R2 > 1 ? 3 : 2;
  static_assert(R0 >= 2 && R1 >= 2 && R0 * R1 * R2 == N0 && TPB % 64 == 0 && TPB <= 1024, "tile shape");
  static_assert(TPB % L == 0, "a thread keeps its column and row n2 after the first stage");
  static_assert(P1 * TPB == NB1 * L && P2 * TPB == NB2 * L, "stages must split evenly");
  // the x stages' twiddles out of the full table of N0
  static __device__ __forceinline__ void stage_tw(cpx<T>* dst, const cpx<T>* __restrict__ full, int t) {
    for (int i = t; i < OFF2; i += TPB)
      dst[i] = full[(i / NS1 + 1) * (i % NS1) * (N0 / (NS1 * R1))];
    if constexpr (R2 > 1)
      for (int i = t; i < (R2 - 1) * NS2; i += TPB) dst[OFF2 + i] = full[(i / NS2 + 1) * (i % NS2)];
  }
  using V0 = cpx<T>[M][R0];
  using V1 = cpx<T>[P1][R1];
  using V2 = cpx<T>[P2][R2];
  // LDS positions f(i, r): stage 0 writes, stage 1 reads and writes, stage 2
  // reads.  x / R0 of a stage's rows is j / R0 plus a multiple of r, so the
  // rotation is the same for all r (or known at compile time) and r moves
  // the position by a constant.
  static __device__ __forceinline__ int rot(int line, int g) { return line ^ ((g % M) * W); }
  static __device__ __forceinline__ int w0(int t, int i, int r) {
    return (t / W) * (R0 * L) + rot(i * W + t % W, t / W) + r * L;
  }
  static __device__ __forceinline__ int r1(int t, int i, int r) {
    const int line = t % L, j = (t + i * TPB) / L;
    if constexpr (R2 == 1) return j * L + r * NB1 * L + rot(line, r);  // NB1 = R0
    else if constexpr (R2 % M == 0) return j * L + rot(line, j / R0) + r * NB1 * L;
    else return j * L + r * NB1 * L + rot(line, j / R0 + r * R2);
  }
  static __device__ __forceinline__ int w1(int t, int i, int r) {
    const int line = t % L, j = (t + i * TPB) / L, k = j % NS1;
    if constexpr (R1 % M == 0) return ((j - k) * R1 + k) * L + r * NS1 * L + rot(line, r);
    else return ((j - k) * R1 + k) * L + r * NS1 * L + rot(line, (j - k) / R0 * R1 + r);
  }
  static __device__ __forceinline__ int r2(int t, int i, int r) {
    const int line = t % L, j = (t + i * TPB) / L;
    if constexpr (R1 % M == 0) return j * L + rot(line, j / R0) + r * NB2 * L;
    else return j * L + r * NB2 * L + rot(line, j / R0 + r * R1);
  }
  template <int PA, int RA, int PB, int RB, typename FA, typename FB>
  static __device__ __forceinline__ void exchange(const cpx<T> (&a)[PA][RA], cpx<T> (&b)[PB][RB], T* buf,
                                                  bool sync, FA&& fa, FB&& fb) {
    if (sync) __syncthreads();
#pragma unroll
    for (int i = 0; i < PA; ++i)
#pragma unroll
      for (int r = 0; r < RA; ++r) buf[fa(i, r)] = a[i][r].x;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PB; ++i)
#pragma unroll
      for (int r = 0; r < RB; ++r) b[i][r].x = buf[fb(i, r)];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PA; ++i)
#pragma unroll
      for (int r = 0; r < RA; ++r) buf[fa(i, r)] = a[i][r].y;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PB; ++i)
#pragma unroll
      for (int r = 0; r < RB; ++r) b[i][r].y = buf[fb(i, r)];
  }
  template <int R, int NS, int SIGN>
  static __device__ __forceinline__ void twiddle(cpx<T>* v, int j, const cpx<T>* tw) {
    const int k = j % NS;
#pragma unroll
    for (int r = 1; r < R; ++r) {
      const cpx<T> w = tw[(r - 1) * NS + k];
      v[r] = SIGN < 0 ? cmul(v[r], w) : cmulc(v[r], w);
    }
  }
  // M-point DFTs over n2 and R0-point DFTs over x in the loaded registers
  template <int SIGN>
  static __device__ __forceinline__ void first(V0& v) {
#pragma unroll
    for (int r = 0; r < R0; ++r) {
      cpx<T> y[M];
#pragma unroll
      for (int i = 0; i < M; ++i) y[i] = v[i][r];
      pdft<T, M, SIGN>(y);
#pragma unroll
      for (int i = 0; i < M; ++i) v[i][r] = y[i];
    }
#pragma unroll
    for (int i = 0; i < M; ++i) pdft<T, R0, SIGN>(v[i]);
  }
  // stage 1 or 2 on the registers: twiddles then DFTs, or (BACK: a stage
  // undone) DFTs then twiddles
  template <int PER, int R, int NS, int SIGN, bool BACK>
  static __device__ __forceinline__ void stage(cpx<T> (&x)[PER][R], int t, const cpx<T>* tw) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int j = (t + i * TPB) / L;
      if constexpr (!BACK) twiddle<R, NS, SIGN>(x[i], j, tw);
      pdft<T, R, SIGN>(x[i]);
      if constexpr (BACK) twiddle<R, NS, SIGN>(x[i], j, tw);
    }
  }
};

// A grad or laplace-family symbol on one (column, row n2): the fixed axes'
// part once per thread, arithmetic in T.  The grids are powers of two, so
// scale = 1 / (N0 N1 N2) is one in T and |k|^2 < 2^24 is exact in FP32: the
// factors are the FP64 ones of apply_sym rounded to T once.
template <typename T>
struct TwoSym {
  T fixed, scale;  // -(sum of squares), grad: the wavenumber
  bool on_x;
  static __device__ __forceinline__ int wave(int k, int n) {
    const int w = k > n / 2 ? k - n : k;
    return k == n / 2 ? 0 : w;
  }
  __device__ __forceinline__ TwoSym(const FftArgs<T>& a, int ky, int kz) {
    const int wy = wave(ky, (int)a.N1), wz = wave(kz, (int)a.N2);
    scale = (T)a.scale;
    on_x = a.sym == SYM_GRAD_X;
    fixed = a.sym > SYM_GRAD_Z ? -(T)(wy * wy + wz * wz) : (T)(a.sym == SYM_GRAD_Z ? wz : wy);
  }
  template <int KIND>
  __device__ __forceinline__ cpx<T> mul(int k, int n, cpx<T> v) const {
    const int w = wave(k, n);
    if constexpr (KIND == SYM_GRAD_X) {  // any grad
      const T f = scale * (on_x ? (T)w : fixed);
      return {-f * v.y, f * v.x};
    } else {
      const T q = fixed - (T)(w * w);
      T f;
      if constexpr (KIND == SYM_LAPLACE) f = scale * q;
      else if constexpr (KIND == SYM_BIHARMONIC) f = (scale * q) * q;
      else f = q == (T)0 ? (T)0 : scale / q;
      return {f * v.x, f * v.y};
    }
  }
};

// In place or out of place over [N0][N1][Nh]: a.Sin / a.Sout the x strides,
// a.Din / a.Dout the n2 strides (R Nh), a.nlines = R Nh columns, a.tw the
// full table of N0.  M_C2C: transforms of sign SIGN; FP64 has the forward
// kernel alone, whose inverse is conj(F(conj x)) by flip as in mix_s_kernel
// (its own inverse spilled 12 registers: 547 against 512 us at 512^3; 465-487
// us since the kernel has no guard for a partial tile).
// M_MULT: forward, the
// symbol a.sym (a.Ch = Nh, a.C = R), inverse, the inverse running the
// forward stages backwards (512^3 FP32 418 us, against 171 + 232 + 181 us as
// y, fused x and y passes; 256^3 42 against 25 + 30 + 24 us).
template <typename T, int N0, int M, int MODE, int SIGN>
__global__ void __launch_bounds__((XYCfg<T, N0, M, MODE>::TPB), (MODE == M_MULT ? XYCfg<T, N0, M, MODE>::MULT_WAVES : 4))
    two_xy_kernel(FftArgs<T> a, unsigned flip) {
  using K = XYTile<T, N0, M, MODE>;
  constexpr int W = K::W, TPB = K::TPB, R0 = K::R0, R1 = K::R1, R2 = K::R2, L = K::L;
  static_assert(MODE == M_C2C || SIGN < 0, "M_MULT starts forward");
  __shared__ T buf[N0 * L];
  __shared__ cpx<T> tw[K::TWN];
  const int t = threadIdx.x;
  int64_t tile = xcd_tile(blockIdx.x, gridDim.x, (unsigned)a.xgroup);
  if (a.reverse) tile = (int64_t)gridDim.x - 1 - tile;
  const int64_t col0 = tile * W;
  // first-stage registers: column t % W, x = t / W + r N0 / R0, all n2 (every
  // tile is whole: the launcher refuses R Nh columns that W does not divide)
  typename K::V0 v;
  {
    const uint32_t off = (uint32_t)((t % W + (t / W) * a.Sin) * sizeof(cpx<T>));
    const cpx<T>* src = reinterpret_cast<const cpx<T>*>(a.in) + col0;
#pragma unroll
    for (int r = 0; r < R0; ++r)
#pragma unroll
      for (int i = 0; i < M; ++i)
        v[i][r] = ld_global(at_off<const cpx<T>>(src + r * (N0 / R0) * a.Sin + i * a.Din, off));
  }
  K::stage_tw(tw, a.tw, t);
  constexpr bool FLIP = MODE == M_C2C && sizeof(T) == 8;
  if constexpr (FLIP) {
#pragma unroll
    for (int i = 0; i < M; ++i)
#pragma unroll
      for (int r = 0; r < R0; ++r) v[i][r] = conj_if(v[i][r], flip);
  }
  auto w0 = [&](int i, int r) { return K::w0(t, i, r); };
  auto r1 = [&](int i, int r) { return K::r1(t, i, r); };
  auto w1 = [&](int i, int r) { return K::w1(t, i, r); };
  auto r2 = [&](int i, int r) { return K::r2(t, i, r); };
  K::template first<SIGN>(v);
  typename K::V1 x;
  K::exchange(v, x, buf, false, w0, r1);
  K::template stage<K::P1, R1, K::NS1, SIGN, false>(x, t, tw);
  // the last stage's outputs: row x = j + r N0 / R, row n2 -> k2 and column
  // of this thread
  const int line = t % L;
  if constexpr (MODE == M_C2C) {
    auto store = [&](auto& o, auto per, auto rad) {
      constexpr int PER = decltype(per)::value, R = decltype(rad)::value;
      cpx<T>* dst = reinterpret_cast<cpx<T>*>(a.out) + col0;
      const uint32_t off = (uint32_t)((line % W + (line / W) * a.Dout + (t / L) * a.Sout) * sizeof(cpx<T>));
#pragma unroll
      for (int i = 0; i < PER; ++i)
#pragma unroll
        for (int r = 0; r < R; ++r)
          *at_off<cpx<T>>(dst + (i * (TPB / L) + r * (N0 / R)) * a.Sout, off) =
              FLIP ? conj_if(o[i][r], flip) : o[i][r];
    };
    if constexpr (R2 > 1) {
      typename K::V2 o;
      K::exchange(x, o, buf, true, w1, r2);
      K::template stage<K::P2, R2, K::NS2, SIGN, false>(o, t, tw + K::OFF2);
      store(o, std::integral_constant<int, K::P2>{}, std::integral_constant<int, R2>{});
    } else {
      store(x, std::integral_constant<int, K::P1>{}, std::integral_constant<int, R1>{});
    }
    return;
  } else {
    const int64_t col = col0 + line % W;
    const int64_t k1 = col / a.Ch;
    const TwoSym<T> sym(a, (int)(k1 + a.C * (line / W)), (int)(col - k1 * a.Ch));
    auto symbol = [&](auto& o, auto per, auto rad) {
      constexpr int PER = decltype(per)::value, R = decltype(rad)::value;
      auto apply = [&](auto kind) {
#pragma unroll
        for (int i = 0; i < PER; ++i)
#pragma unroll
          for (int r = 0; r < R; ++r)
            o[i][r] = sym.template mul<decltype(kind)::value>((t + i * TPB) / L + r * (N0 / R), N0, o[i][r]);
      };
      switch (a.sym) {  // uniform: one loop per kind
        case SYM_LAPLACE: apply(std::integral_constant<int, SYM_LAPLACE>{}); break;
        case SYM_BIHARMONIC: apply(std::integral_constant<int, SYM_BIHARMONIC>{}); break;
        case SYM_INV_LAPLACE: apply(std::integral_constant<int, SYM_INV_LAPLACE>{}); break;
        default: apply(std::integral_constant<int, SYM_GRAD_X>{}); break;
      }
    };
    // the way back recomputes its positions: kept over the symbol they would
    // take 30 to 60 registers
    int tb = t;
    asm volatile("" : "+v"(tb));
    auto bw0 = [&](int i, int r) { return K::w0(tb, i, r); };
    auto br1 = [&](int i, int r) { return K::r1(tb, i, r); };
    auto bw1 = [&](int i, int r) { return K::w1(tb, i, r); };
    auto br2 = [&](int i, int r) { return K::r2(tb, i, r); };
    if constexpr (R2 > 1) {
      typename K::V2 o;
      K::exchange(x, o, buf, true, w1, r2);
      K::template stage<K::P2, R2, K::NS2, -1, false>(o, t, tw + K::OFF2);
      symbol(o, std::integral_constant<int, K::P2>{}, std::integral_constant<int, R2>{});
      K::template stage<K::P2, R2, K::NS2, +1, true>(o, tb, tw + K::OFF2);
      // (a thread writes where it alone has read: no barrier)
      K::exchange(o, x, buf, false, br2, bw1);
    } else {
      symbol(x, std::integral_constant<int, K::P1>{}, std::integral_constant<int, R1>{});
    }
    K::template stage<K::P1, R1, K::NS1, +1, true>(x, tb, tw);
    K::exchange(x, v, buf, R2 > 1, br1, bw0);
    K::template first<+1>(v);
    cpx<T>* dst = reinterpret_cast<cpx<T>*>(a.out) + col0;
    const uint32_t off = (uint32_t)((tb % W + (tb / W) * a.Sout) * sizeof(cpx<T>));
#pragma unroll
    for (int r = 0; r < R0; ++r)
#pragma unroll
      for (int i = 0; i < M; ++i)
        *at_off<cpx<T>>(dst + r * (N0 / R0) * a.Sout + i * a.Dout, off) = v[i][r];
  }
}

// ------------------------------------------------------------------ pass 1
// Tile: P rows x NZ points (complex lines, or pairs of real lines), a 2-D
// transform. A stage takes 2^bp rows x 2^bz points of each dimension's
// Stockham recursion into one butterfly (no twiddles between the
// dimensions), 2^e elements a thread.
struct TwoSched {
  int s;
  int bp[6], bz[6];
};
constexpr int two_log(int n) {
  int l = 0;
  while ((1 << l) < n) ++l;
  return l;
}
// As much of one dimension as fits a butterfly, then the other: few stages
// with twiddles.  rows_first: the first stage takes whole z rows (lanes along
// z: the loads of r2c), otherwise the last one does (the stores of c2r).
constexpr TwoSched two_sched(int P, int NZ, int E, bool rows_first) {
  TwoSched m{0, {}, {}};
  int h = two_log(P), z = two_log(NZ);
  const int e = two_log(E);
  while (h + z > 0) {
    int &d0 = rows_first ? h : z, &d1 = rows_first ? z : h;
    const int b0 = e < d0 ? e : d0, b1 = e - b0 < d1 ? e - b0 : d1;
    d0 -= b0;
    d1 -= b1;
    m.bp[m.s] = rows_first ? b0 : b1;
    m.bz[m.s] = rows_first ? b1 : b0;
    ++m.s;
  }
  return m;
}
template <typename T, int P, int NZ>
struct ZYCfg {
  // elements a thread: large tiles 64 registers of data, small ones fewer
  // (more threads)
  static constexpr int EM = sizeof(T) == 4 ? 32 : 16;
  static constexpr int E = P * NZ / EM >= 256 ? EM : P * NZ / (EM / 2) >= 256 ? EM / 2 : EM / 4;
  static constexpr int TPB = P * NZ / E;
};
template <typename T, int P, int NZ, bool ROWS_FIRST>
struct ZYTile {
  using CF = ZYCfg<T, P, NZ>;
  static constexpr int E = CF::E, TPB = CF::TPB;
  static constexpr TwoSched SC = two_sched(P, NZ, E, ROWS_FIRST);
  static constexpr int S = SC.s;
  static_assert(TPB >= 64 && TPB <= 1024 && TPB % 64 == 0, "tile shape");
  // LDS: rows of NZ values, five pad values after every 64: a first z stage
  // writes with a stride of its radix, a second one in groups of the first
  // radix; both spread over the banks (a CPU model of the accesses)
  static constexpr int ZP = NZ + NZ / 64 * 5;
  static __device__ __forceinline__ int at(int p, int z) { return p * ZP + z + (z >> 6) * 5; }
  template <int s>
  struct St {
    static constexpr int RP = 1 << SC.bp[s], RZ = 1 << SC.bz[s];
    static constexpr int ns(bool z) {
      int n = 1;
      for (int i = 0; i < s; ++i) n <<= z ? SC.bz[i] : SC.bp[i];
      return n;
    }
    static constexpr int NSP = ns(false), NSZ = ns(true);
    static constexpr int NBP = P / RP, NBZ = NZ / RZ, PER = E / (RP * RZ);
    static constexpr int off(bool z) {  // twiddle offsets
      int o = 0, n = 1;
      for (int i = 0; i < s; ++i) {
        const int b = z ? SC.bz[i] : SC.bp[i];
        if (n > 1) o += ((1 << b) - 1) * n;
        n <<= b;
      }
      return o;
    }
    static constexpr int OFFP = off(false), OFFZ = off(true);
    static __device__ __forceinline__ void map(int t, int i, int& pj, int& zj) {
      const int b = t + i * TPB;
      zj = b % NBZ;
      pj = b / NBZ;
    }
  };
  static constexpr int tw_size(bool z) {
    int o = 0, n = 1;
    for (int i = 0; i < S; ++i) {
      const int b = z ? SC.bz[i] : SC.bp[i];
      if (n > 1) o += ((1 << b) - 1) * n;
      n <<= b;
    }
    return o > 0 ? o : 1;
  }
  static constexpr int TWZ = tw_size(true), TWP = tw_size(false);
  template <int s>
  using Regs = cpx<T>[St<s>::PER][St<s>::RP][St<s>::RZ];
  using Last = St<S - 1>;

  // stage tables out of the length's full table (stride q between its roots)
  template <bool Z>
  static __device__ __forceinline__ void stage_tw(cpx<T>* dst, const cpx<T>* __restrict__ full, int q, int t) {
    int n = 1, o = 0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int b = Z ? SC.bz[s] : SC.bp[s], R = 1 << b;
      if (n > 1 && R > 1) {
        const int cnt = (R - 1) * n, step = (Z ? NZ : P) / (n * R) * q;
        for (int i = t; i < cnt; i += TPB) dst[o + i] = full[(i / n + 1) * (i % n) * step];
        o += cnt;
      }
      n <<= b;
    }
  }
  template <int s, int SIGN>
  static __device__ __forceinline__ void butterflies(Regs<s>& v, int t, const cpx<T>* twp, const cpx<T>* twz) {
    using X = St<s>;
#pragma unroll
    for (int i = 0; i < X::PER; ++i) {
      int pj, zj;
      X::map(t, i, pj, zj);
#pragma unroll
      for (int r = 0; r < X::RP; ++r) {
        if constexpr (X::NSZ > 1 && X::RZ > 1) {
          const int k = zj % X::NSZ;
#pragma unroll
          for (int q = 1; q < X::RZ; ++q) {
            const cpx<T> w = twz[X::OFFZ + (q - 1) * X::NSZ + k];
            v[i][r][q] = SIGN < 0 ? cmul(v[i][r][q], w) : cmulc(v[i][r][q], w);
          }
        }
        pdft<T, X::RZ, SIGN>(v[i][r]);
      }
      if constexpr (X::RP > 1) {
        const int k = pj % X::NSP;
#pragma unroll
        for (int q = 0; q < X::RZ; ++q) {
          cpx<T> y[X::RP];
#pragma unroll
          for (int r = 0; r < X::RP; ++r) {
            y[r] = v[i][r][q];
            if (X::NSP > 1 && r > 0) {
              const cpx<T> w = twp[X::OFFP + (r - 1) * X::NSP + k];
              y[r] = SIGN < 0 ? cmul(y[r], w) : cmulc(y[r], w);
            }
          }
          pdft<T, X::RP, SIGN>(y);
#pragma unroll
          for (int r = 0; r < X::RP; ++r) v[i][r][q] = y[r];
        }
      }
    }
  }
  // fn(i, r, q, position): a stage's read (W = false) or write positions
  template <int s, bool W, typename F>
  static __device__ __forceinline__ void each(int t, F&& fn) {
    using X = St<s>;
#pragma unroll
    for (int i = 0; i < X::PER; ++i) {
      int pj, zj;
      X::map(t, i, pj, zj);
      const int kp = pj % X::NSP, kz = zj % X::NSZ;
      const int p0 = W ? (pj - kp) * X::RP + kp : pj, z0 = W ? (zj - kz) * X::RZ + kz : zj;
      constexpr int dp = W ? X::NSP : X::NBP, dz = W ? X::NSZ : X::NBZ;
      const int base = at(p0, z0);
#pragma unroll
      for (int r = 0; r < X::RP; ++r)
#pragma unroll
        for (int q = 0; q < X::RZ; ++q) {
          // linear in r and q: the lowest bits of z0 stay below dz, a
          // power of two, so adding q dz carries nothing into them
          fn(i, r, q, base + r * dp * ZP + q * dz + ((q * dz) >> 6) * 5);
        }
    }
  }
  template <int s, bool W>
  static __device__ __forceinline__ void put(const Regs<s>& v, T* buf, int t, bool im) {
    each<s, W>(t, [&](int i, int r, int q, int p) { buf[p] = im ? v[i][r][q].y : v[i][r][q].x; });
  }
  template <int s, bool W>
  static __device__ __forceinline__ void get(Regs<s>& v, const T* buf, int t, bool im) {
    each<s, W>(t, [&](int i, int r, int q, int p) {
      if (im) v[i][r][q].y = buf[p];
      else v[i][r][q].x = buf[p];
    });
  }
  template <int s>
  static __device__ __forceinline__ void exchange(const Regs<s>& a, Regs<s + 1>& b, T* buf, int t, bool sync) {
    if (sync) __syncthreads();
    put<s, true>(a, buf, t, false);
    __syncthreads();
    get<s + 1, false>(b, buf, t, false);
    __syncthreads();
    put<s, true>(a, buf, t, true);
    __syncthreads();
    get<s + 1, false>(b, buf, t, true);
  }
  // stages s .. S-1 from the operands of stage s
  template <int s, int SIGN>
  static __device__ __forceinline__ void run(Regs<s>& v, Regs<S - 1>& o, T* buf, int t, bool sync,
                                             const cpx<T>* twp, const cpx<T>* twz) {
    butterflies<s, SIGN>(v, t, twp, twz);
    if constexpr (s == S - 2) {
      exchange<s>(v, o, buf, t, sync);
      butterflies<S - 1, SIGN>(o, t, twp, twz);
    } else {
      Regs<s + 1> x;
      exchange<s>(v, x, buf, t, sync);
      run<s + 1, SIGN>(x, o, buf, t, true, twp, twz);
    }
  }
};

// a b + c d and a b - c d; conj: a conj b + c conj d, a conj b - c conj d
template <typename T, int S, bool CONJ>
__device__ __forceinline__ cpx<T> cmul2(cpx<T> a, cpx<T> b, cpx<T> c, cpx<T> d) {
  const cpx<T> p = CONJ ? cmulc(a, b) : cmul(a, b);
  if constexpr (CONJ)
    return S > 0 ? cpx<T>{p.x + c.x * d.x + c.y * d.y, p.y + c.y * d.x - c.x * d.y}
                 : cpx<T>{p.x - c.x * d.x - c.y * d.y, p.y - c.y * d.x + c.x * d.y};
  else
    return S > 0 ? cpx<T>{p.x + c.x * d.x - c.y * d.y, p.y + c.x * d.y + c.y * d.x}
                 : cpx<T>{p.x - c.x * d.x + c.y * d.y, p.y - c.x * d.y - c.y * d.x};
}

// Factors of the split: te[k1] = w^(n2 k1) for the even rows' part of row k1,
// to[k1] = te[k1] w_R^(k1 mod P) for the odd rows', w = exp(-2 pi i / N1) (one
// table entry each: one rounding instead of two products in a row), times
// scale.
template <typename T, int R, int TPB>
__device__ __forceinline__ void split_factors(cpx<T>* te, cpx<T>* to, const cpx<T>* __restrict__ twy,
                                              int n2, int M, T scale, int t) {
  for (int k = t; k < R; k += TPB) {
    const int e = n2 * k, o = e + M * (k & (R / 2 - 1));
    te[k] = cscale(twy[e], scale);
    to[k] = cscale(twy[o < M * R ? o : o - M * R], scale);
  }
}

// Real rows n2 + M n1 of plane x (n1 < R) -> rows k1 + R n2 of the half
// spectrum, transformed along z and over n1.  The rows 2p, 2p+1 are packed as
// real and imaginary parts, P = R/2 complex rows; with U the 2-D transform of
// the packed rows,
//   E_q[k] = (U_q[k] + conj U_-q[-k]) / 2, O_q[k] = -i (U_q[k] - conj U_-q[-k]) / 2
// are the transforms of the even and odd rows, and the last radix-2 level
//   X_q = E_q + w_R^q O_q, X_{q+P} = E_q - w_R^q O_q
// rides on the split, with the twiddles of the M-point level in its factors.
// a.idist / a.odist: row pitches, a.Din / a.Dout plane strides, a.C = M,
// a.tw / twy the full tables of NZ and N1.
template <typename T, int NZ, int R>
__global__ void __launch_bounds__((ZYCfg<T, R / 2, NZ>::TPB))
    two_zy_r2c_kernel(FftArgs<T> a, const cpx<T>* __restrict__ twy) {
  constexpr int P = R / 2, NH = NZ / 2 + 1;
  using K = ZYTile<T, P, NZ, true>;
  constexpr int TPB = K::TPB, I = P * (NZ / 2) / TPB;
  __shared__ T buf[P * K::ZP];
  __shared__ cpx<T> twz[K::TWZ], twp[K::TWP], te[R], to[R];
  const int t = threadIdx.x;
  const int64_t blk = xcd_tile(blockIdx.x, gridDim.x, (unsigned)a.xgroup);
  const int64_t M = a.C, x = blk / M, n2 = blk - x * M;
  using S0 = typename K::template St<0>;
  typename K::template Regs<0> v;
  {
    const T* src = reinterpret_cast<const T*>(a.in) + x * a.Din + n2 * a.idist;
    const int64_t row = M * a.idist;
#pragma unroll
    for (int i = 0; i < S0::PER; ++i) {
      int pj, zj;
      S0::map(t, i, pj, zj);
      const uint32_t off = (uint32_t)((2 * pj * row + zj) * sizeof(T));
#pragma unroll
      for (int r = 0; r < S0::RP; ++r)
#pragma unroll
        for (int q = 0; q < S0::RZ; ++q) {
          v[i][r][q].x = *at_off<const T>(src + 2 * r * S0::NBP * row + q * S0::NBZ, off);
          v[i][r][q].y = *at_off<const T>(src + (2 * r * S0::NBP + 1) * row + q * S0::NBZ, off);
        }
    }
  }
  K::template stage_tw<true>(twz, a.tw, 1, t);
  K::template stage_tw<false>(twp, twy, 2 * (int)M, t);  // roots of P = N1 / (2 M)
  split_factors<T, R, TPB>(te, to, twy, (int)n2, (int)M, (T)0.5, t);
  typename K::template Regs<K::S - 1> o;
  K::template run<0, -1>(v, o, buf, t, false, twp, twz);
  // U in natural order through the LDS (each thread writes where it alone
  // has read); item: U_q[k] and U_-q[-k], k < NZ / 2, and the column NZ / 2
  T ax[I + 1], ay[I + 1], bx[I + 1], by[I + 1];
  auto item = [&](int i, int& q, int& k) {
    if (i < I) {
      const int b = t + i * TPB;
      k = b % (NZ / 2);
      q = b / (NZ / 2);
    } else {
      k = NZ / 2;
      q = t & (P - 1);
    }
  };
  auto grab = [&](T* f, T* g) {
#pragma unroll
    for (int i = 0; i <= I; ++i) {
      int q, k;
      item(i, q, k);
      f[i] = buf[K::at(q, k)];
      g[i] = buf[K::at((P - q) & (P - 1), (NZ - k) & (NZ - 1))];
    }
  };
  K::template put<K::S - 1, false>(o, buf, t, false);
  __syncthreads();
  grab(ax, bx);
  __syncthreads();
  K::template put<K::S - 1, false>(o, buf, t, true);
  __syncthreads();
  grab(ay, by);
  cpx<T>* dst = reinterpret_cast<cpx<T>*>(a.out) + x * a.Dout + n2 * R * a.odist;
#pragma unroll
  for (int i = 0; i <= I; ++i) {
    if (i == I && t >= P) break;
    int q, k;
    item(i, q, k);
    cpx<T> e = {ax[i] + bx[i], ay[i] - by[i]}, d = {ay[i] + by[i], bx[i] - ax[i]};
    if (a.adjw && k != 0 && k != NZ / 2) {  // (the factors carry the 1/2)
      e = cscale(e, (T)2);
      d = cscale(d, (T)2);
    }
    cpx<T>* p = dst + q * a.odist + k;
    p[0] = cmul2<T, 1, false>(e, te[q], d, to[q]);
    p[P * a.odist] = cmul2<T, -1, false>(e, te[q + P], d, to[q + P]);
  }
}

// Pass 1 of a c2c transform, either sign: the complex rows n2 + M n1 -> rows
// k1 + R n2, transformed along z and over n1 and twiddled for the M-point
// level.  (The inverse c2c runs the two passes in the same order with the
// other sign.)  Arguments as above.
template <typename T, int NZ, int R, int SIGN>
__global__ void __launch_bounds__((ZYCfg<T, R, NZ>::TPB))
    two_zy_c2c_kernel(FftArgs<T> a, const cpx<T>* __restrict__ twy) {
  using K = ZYTile<T, R, NZ, true>;
  constexpr int TPB = K::TPB;
  __shared__ T buf[R * K::ZP];
  __shared__ cpx<T> twz[K::TWZ], twp[K::TWP], te[R];
  const int t = threadIdx.x;
  const int64_t blk = xcd_tile(blockIdx.x, gridDim.x, (unsigned)a.xgroup);
  const int64_t M = a.C, x = blk / M, n2 = blk - x * M;
  using S0 = typename K::template St<0>;
  using SL = typename K::Last;
  typename K::template Regs<0> v;
  const cpx<T>* src = reinterpret_cast<const cpx<T>*>(a.in) + x * a.Din + n2 * a.idist;
  const int64_t row = M * a.idist;
#pragma unroll
  for (int i = 0; i < S0::PER; ++i) {
    int pj, zj;
    S0::map(t, i, pj, zj);
    const uint32_t off = (uint32_t)((pj * row + zj) * sizeof(cpx<T>));
#pragma unroll
    for (int r = 0; r < S0::RP; ++r)
#pragma unroll
      for (int q = 0; q < S0::RZ; ++q)
        v[i][r][q] = ld_global(at_off<const cpx<T>>(src + r * S0::NBP * row + q * S0::NBZ, off));
  }
  K::template stage_tw<true>(twz, a.tw, 1, t);
  K::template stage_tw<false>(twp, twy, (int)M, t);  // roots of R = N1 / M
  for (int k = t; k < R; k += TPB) te[k] = twy[n2 * k];
  typename K::template Regs<K::S - 1> o;
  K::template run<0, SIGN>(v, o, buf, t, false, twp, twz);
  cpx<T>* dst = reinterpret_cast<cpx<T>*>(a.out) + x * a.Dout + n2 * R * a.odist;
#pragma unroll
  for (int i = 0; i < SL::PER; ++i) {
    int pj, zj;
    SL::map(t, i, pj, zj);
    const uint32_t off = (uint32_t)((pj * a.odist + zj) * sizeof(cpx<T>));
#pragma unroll
    for (int r = 0; r < SL::RP; ++r) {
      const cpx<T> w = te[pj + r * SL::NBP];
#pragma unroll
      for (int q = 0; q < SL::RZ; ++q)
        *at_off<cpx<T>>(dst + r * SL::NBP * a.odist + q * SL::NBZ, off) =
            SIGN < 0 ? cmul(o[i][r][q], w) : cmulc(o[i][r][q], w);
    }
  }
}

// The inverse: rows k1 + R n2 -> real rows n2 + M n1, the steps above
// backwards (E_q = Y_q conj te_q + Y_{q+P} conj te_{q+P}, O_q = Y_q conj to_q -
// Y_{q+P} conj to_{q+P} of the rows Y, U_q[k] = E + i O, U_-q[-k] = conj E + i conj O).  c2r
// drops the imaginary parts of the row spectra at k = 0 and NZ / 2: there
// E_q becomes (E_q + conj E_-q) / 2, O alike.
template <typename T, int NZ, int R>
__global__ void __launch_bounds__((ZYCfg<T, R / 2, NZ>::TPB))
    two_zy_c2r_kernel(FftArgs<T> a, const cpx<T>* __restrict__ twy) {
  constexpr int P = R / 2;
  using K = ZYTile<T, P, NZ, false>;
  constexpr int TPB = K::TPB, I = P * (NZ / 2) / TPB;
  __shared__ T buf[P * K::ZP];
  __shared__ cpx<T> twz[K::TWZ], twp[K::TWP], te[R], to[R], edge[2][2][P];
  const int t = threadIdx.x;
  const int64_t blk = xcd_tile(blockIdx.x, gridDim.x, (unsigned)a.xgroup);
  const int64_t M = a.C, x = blk / M, n2 = blk - x * M;
  const cpx<T>* src = reinterpret_cast<const cpx<T>*>(a.in) + x * a.Din + n2 * R * a.idist;
  cpx<T> y0[I], y1[I];
#pragma unroll
  for (int i = 0; i < I; ++i) {
    const int b = t + i * TPB;
    const cpx<T>* p = src + (int64_t)(b / (NZ / 2)) * a.idist + b % (NZ / 2);
    y0[i] = p[0];
    y1[i] = p[P * a.idist];
  }
  // the column NZ / 2: one item each for the first P threads
  cpx<T> z0 = {(T)0, (T)0}, z1 = z0;
  if (t < P) {
    const cpx<T>* p = src + (int64_t)t * a.idist + NZ / 2;
    z0 = p[0];
    z1 = p[P * a.idist];
  }
  K::template stage_tw<true>(twz, a.tw, 1, t);
  K::template stage_tw<false>(twp, twy, 2 * (int)M, t);
  split_factors<T, R, TPB>(te, to, twy, (int)n2, (int)M, (T)1, t);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < I; ++i) {
    const int b = t + i * TPB, k = b % (NZ / 2), q = b / (NZ / 2);
    const cpx<T> e = cmul2<T, 1, true>(y0[i], te[q], y1[i], te[q + P]);
    const cpx<T> d = cmul2<T, -1, true>(y0[i], to[q], y1[i], to[q + P]);
    if (k == 0) {
      edge[0][0][q] = e;
      edge[0][1][q] = d;
    }
    y0[i] = {e.x - d.y, e.y + d.x};
    y1[i] = {e.x + d.y, d.x - e.y};
  }
  if (a.adjw) {
#pragma unroll
    for (int i = 0; i < I; ++i) {
      y0[i] = cscale(y0[i], (T)0.5);
      y1[i] = cscale(y1[i], (T)0.5);
    }
  }
  if (t < P) {
    edge[1][0][t] = cmul2<T, 1, true>(z0, te[t], z1, te[t + P]);
    edge[1][1][t] = cmul2<T, -1, true>(z0, to[t], z1, to[t + P]);
  }
  __syncthreads();
  // edge items (column ec, row eq), one for each of the first 2 P threads
  static_assert(2 * P <= TPB, "one edge item a thread");
  const int eq = t & (P - 1), ec = t / P;
  cpx<T> eu = {(T)0, (T)0};
  if (t < 2 * P) {
    const int en = (P - eq) & (P - 1);
    const cpx<T> e0 = edge[ec][0][eq], e1 = edge[ec][0][en], d0 = edge[ec][1][eq], d1 = edge[ec][1][en];
    const T h = (T)0.5;
    const cpx<T> e = {h * (e0.x + e1.x), h * (e0.y - e1.y)}, d = {h * (d0.x + d1.x), h * (d0.y - d1.y)};
    eu = {e.x - d.y, e.y + d.x};
  }
  typename K::template Regs<0> v;
  auto scatter = [&](bool im) {
#pragma unroll
    for (int i = 0; i < I; ++i) {
      const int b = t + i * TPB, k = b % (NZ / 2), q = b / (NZ / 2);
      if (k != 0) {
        buf[K::at(q, k)] = im ? y0[i].y : y0[i].x;
        buf[K::at((P - q) & (P - 1), NZ - k)] = im ? y1[i].y : y1[i].x;
      }
    }
    if (t < 2 * P) buf[K::at(eq, ec * (NZ / 2))] = im ? eu.y : eu.x;
  };
  scatter(false);
  __syncthreads();
  K::template get<0, false>(v, buf, t, false);
  __syncthreads();
  scatter(true);
  __syncthreads();
  K::template get<0, false>(v, buf, t, true);
  typename K::template Regs<K::S - 1> o;
  K::template run<0, +1>(v, o, buf, t, true, twp, twz);
  using SL = typename K::Last;
  T* dst = reinterpret_cast<T*>(a.out) + x * a.Dout + n2 * a.odist;
  const int64_t row = M * a.odist;
#pragma unroll
  for (int i = 0; i < SL::PER; ++i) {
    int pj, zj;
    SL::map(t, i, pj, zj);
    const uint32_t off = (uint32_t)((2 * pj * row + zj) * sizeof(T));
#pragma unroll
    for (int r = 0; r < SL::RP; ++r)
#pragma unroll
      for (int q = 0; q < SL::RZ; ++q) {
        *at_off<T>(dst + 2 * r * SL::NBP * row + q * SL::NBZ, off) = o[i][r][q].x;
        *at_off<T>(dst + (2 * r * SL::NBP + 1) * row + q * SL::NBZ, off) = o[i][r][q].y;
      }
  }
}

}  // namespace afft
