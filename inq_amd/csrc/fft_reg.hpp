// fft_reg.hpp -- mixed-radix FFT of one line held in registers (gfx950).
//
// A line of N complex values lives in a register array x[N] of one lane.
// The transform is a recursive decimation-in-time split N = R*M, fully
// unrolled at compile time: every index and every twiddle is a constant, so
// the array is promoted to VGPRs and the twiddles become instruction
// immediates.  Twiddles come from a constexpr table evaluated by the
// compiler (Taylor series after quadrant reduction, exact at multiples of
// pi/2), so there is no table in memory and no sincos at run time.
//
// SIGN = -1: forward, unnormalised, exp(-2 pi i j k / N)
// SIGN = +1: backward, unnormalised, exp(+2 pi i j k / N)
// These are the conventions of the reference's to_fourier / to_real before
// its separate 1/N pass (src/operations/transform.hpp:79,141,175-181).
#pragma once

#include <hip/hip_runtime.h>

namespace inqx {

// plain aggregate complex (trivially copyable, so it can be loaded and
// stored through address-space-qualified pointers)
template <typename T> struct alignas(2 * sizeof(T)) cplx_pod {
  T x, y;
};
template <typename T> using cplx = cplx_pod<T>;

template <typename C> __device__ __forceinline__ C cadd(C a, C b) { return C{a.x + b.x, a.y + b.y}; }
template <typename C> __device__ __forceinline__ C csub(C a, C b) { return C{a.x - b.x, a.y - b.y}; }
template <typename C> __device__ __forceinline__ C cmul(C a, C b) {
  return C{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename C> __device__ __forceinline__ C cmulc(C a, C b) {  // conj(a) * b
  return C{a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x};
}
template <typename C, typename S> __device__ __forceinline__ C cscale(C a, S s) { return C{a.x * s, a.y * s}; }

// ---------------------------------------------------------------- twiddles
struct tw_cs {
  double c, s;
};

// exp(+2 pi i k / n), evaluated at compile time
constexpr tw_cs tw_value(long k, long n) {
  k %= n;
  if (k < 0) k += n;
  long q = (4 * k) / n;
  long r = 4 * k - q * n;  // angle = pi/2 * (q + r/n)
  double phi = 1.5707963267948966 * (double)r / (double)n;
  double p2 = phi * phi;
  double c = 1.0, s = phi, tc = 1.0, ts = phi;
  for (int m = 1; m < 24; ++m) {
    tc *= -p2 / (double)((2 * m - 1) * (2 * m));
    ts *= -p2 / (double)((2 * m) * (2 * m + 1));
    c += tc;
    s += ts;
  }
  if (r == 0) {
    c = 1.0;
    s = 0.0;
  }
  switch (q) {
    case 0: return tw_cs{c, s};
    case 1: return tw_cs{-s, c};
    case 2: return tw_cs{-c, -s};
    default: return tw_cs{s, -c};
  }
}

template <int N> struct tw_table {
  double c[N], s[N];
  constexpr tw_table() : c(), s() {
    for (int k = 0; k < N; ++k) {
      tw_cs v = tw_value(k, N);
      c[k] = v.c;
      s[k] = v.s;
    }
  }
};
template <int N> inline constexpr tw_table<N> kTw{};

// multiply by exp(SIGN * 2 pi i e / N); e is a constant after unrolling and
// the exact 0 / +-1 cases fold to moves and negations.
template <int N, int SIGN, typename C>
__device__ __forceinline__ C twmul(C v, int e) {
  using T = decltype(v.x);
  const int k = ((e % N) + N) % N;
  const double dc = kTw<N>.c[k];
  const double ds = SIGN * kTw<N>.s[k];
  if (ds == 0.0) {
    if (dc == 1.0) return v;
    if (dc == -1.0) return C{-v.x, -v.y};
  }
  if (dc == 0.0) {
    if (ds == 1.0) return C{-v.y, v.x};
    if (ds == -1.0) return C{v.y, -v.x};
  }
  const T c = (T)dc, s = (T)ds;
  return C{v.x * c - v.y * s, v.x * s + v.y * c};
}

// ---------------------------------------------------------------- small DFTs
template <int R, int SIGN, typename C> struct dft_small {
  // generic R-point DFT, t[q] = sum_r W_R^{SIGN r q} t[r]
  static __device__ __forceinline__ void run(C (&t)[R]) {
    C o[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      C acc = t[0];
#pragma unroll
      for (int r = 1; r < R; ++r) acc = cadd(acc, twmul<R, SIGN>(t[r], r * q));
      o[q] = acc;
    }
#pragma unroll
    for (int q = 0; q < R; ++q) t[q] = o[q];
  }
};

template <int SIGN, typename C> struct dft_small<2, SIGN, C> {
  static __device__ __forceinline__ void run(C (&t)[2]) {
    C a = t[0], b = t[1];
    t[0] = cadd(a, b);
    t[1] = csub(a, b);
  }
};

template <int SIGN, typename C> struct dft_small<4, SIGN, C> {
  static __device__ __forceinline__ void run(C (&t)[4]) {
    C a0 = cadd(t[0], t[2]), a1 = csub(t[0], t[2]);
    C b0 = cadd(t[1], t[3]), b1 = csub(t[1], t[3]);
    // b1 * (SIGN i)
    C jb1 = (SIGN > 0) ? C{-b1.y, b1.x} : C{b1.y, -b1.x};
    t[0] = cadd(a0, b0);
    t[2] = csub(a0, b0);
    t[1] = cadd(a1, jb1);
    t[3] = csub(a1, jb1);
  }
};

template <int SIGN, typename C> struct dft_small<3, SIGN, C> {
  static __device__ __forceinline__ void run(C (&t)[3]) {
    using T = decltype(t[0].x);
    const T c = (T)-0.5, s = (T)(SIGN * 0.86602540378443864676);
    C a = t[0];
    C u = cadd(t[1], t[2]);
    C v = csub(t[1], t[2]);
    C m = C{a.x + c * u.x, a.y + c * u.y};
    C js = C{-s * v.y, s * v.x};
    t[0] = cadd(a, u);
    t[1] = cadd(m, js);
    t[2] = csub(m, js);
  }
};

template <int SIGN, typename C> struct dft_small<5, SIGN, C> {
  static __device__ __forceinline__ void run(C (&t)[5]) {
    using T = decltype(t[0].x);
    const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
    const T s1 = (T)(SIGN * 0.95105651629515357212), s2 = (T)(SIGN * 0.58778525229247312917);
    C a = t[0];
    C u1 = cadd(t[1], t[4]), v1 = csub(t[1], t[4]);
    C u2 = cadd(t[2], t[3]), v2 = csub(t[2], t[3]);
    C m1 = C{a.x + c1 * u1.x + c2 * u2.x, a.y + c1 * u1.y + c2 * u2.y};
    C m2 = C{a.x + c2 * u1.x + c1 * u2.x, a.y + c2 * u1.y + c1 * u2.y};
    // i*(s1 v1 + s2 v2) and i*(s2 v1 - s1 v2)
    C n1 = C{-(s1 * v1.y + s2 * v2.y), s1 * v1.x + s2 * v2.x};
    C n2 = C{-(s2 * v1.y - s1 * v2.y), s2 * v1.x - s1 * v2.x};
    t[0] = cadd(a, cadd(u1, u2));
    t[1] = cadd(m1, n1);
    t[4] = csub(m1, n1);
    t[2] = cadd(m2, n2);
    t[3] = csub(m2, n2);
  }
};

// ---------------------------------------------------------------- radix choice
constexpr int fft_radix(int n) {
  if (n % 4 == 0 && n != 8) return 4;
  if (n % 2 == 0) return 2;
  if (n % 3 == 0) return 3;
  if (n % 5 == 0) return 5;
  if (n % 7 == 0) return 7;
  return n;
}

constexpr bool fft_supported(int n) {
  if (n < 1) return false;
  while (n % 2 == 0) n /= 2;
  while (n % 3 == 0) n /= 3;
  while (n % 5 == 0) n /= 5;
  while (n % 7 == 0) n /= 7;
  return n == 1;
}

// ---------------------------------------------------------------- recursive FFT
template <int N, int SIGN, typename C> struct fft_line {
  static_assert(fft_supported(N), "FFT length must be a product of 2, 3, 5, 7");
  static __device__ __forceinline__ void run(C (&x)[N]) {
    constexpr int R = fft_radix(N);
    constexpr int M = N / R;
    if constexpr (M == 1) {
      dft_small<R, SIGN, C>::run(x);
    } else {
      C sub[R][M];
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) sub[r][m] = x[r + R * m];
#pragma unroll
      for (int r = 0; r < R; ++r) fft_line<M, SIGN, C>::run(sub[r]);
#pragma unroll
      for (int k1 = 0; k1 < M; ++k1) {
        C t[R];
        t[0] = sub[0][k1];
#pragma unroll
        for (int r = 1; r < R; ++r) t[r] = twmul<N, SIGN>(sub[r][k1], r * k1);
        dft_small<R, SIGN, C>::run(t);
#pragma unroll
        for (int k2 = 0; k2 < R; ++k2) x[k1 + M * k2] = t[k2];
      }
    }
  }
};

// ---------------------------------------------------------------- lines split over lanes
// A line of N values is shared by S lanes of a wave, N/S values each, so a lane
// holds 1/S of the registers of fft_line: S = 2, lanes l and l + 32 (part 0 and
// 1), or S = 4, lanes l + 16 q (part q).  Radix-2 stages cross the lanes through
// v_permlane32_swap and v_permlane16_swap, which exchange the upper part's value
// of one register with the lower part's value of another: swapping v[k] with
// v[k + M/2] (M values per lane) hands each lane BOTH operands of a butterfly for
// half of the butterflies.  A stage then costs one swap per two registers and
// one full butterfly per two values.  Giving both lanes both operands of every
// butterfly, as the stages for odd M below still do, costs a swap and a move per
// register and a half butterfly with its own twiddle per value.  The transforms
// are VALU bound as much as memory bound, so this shows in every pass: H on 128
// states at 72^3 418.9 -> 395.6 us in complex64 and 1065 -> 927 us in complex128
// (whose plane passes also lose the 16-lane shuffles through the LDS crossbar).
//
// Order of the values, dit in / dif out: part q holds x[S n + q].  dit out / dif
// in: register j of part q holds X[line_out_j<N, S>(j) + line_out_q<N, S>(q)].

__host__ __device__ constexpr int quad_rev(int q) { return ((q & 1) << 1) | (q >> 1); }

// even values per lane: the swapped stages run
template <int N, int S> __host__ __device__ constexpr bool line_swapped() { return (N / S) % 2 == 0; }
template <int N, int S> __host__ __device__ constexpr int line_out_j(int j) {
  constexpr int M = N / S;
  return line_swapped<N, S>() && j >= M / 2 ? j - M / 2 + N / 2 : j;
}
template <int N, int S> __host__ __device__ constexpr int line_out_q(int q) {
  constexpr int M = N / S;
  if (!line_swapped<N, S>()) return M * (S == 2 ? q : quad_rev(q));
  return S == 2 ? q * (M / 2) : (q >> 1) * (M / 2) + (q & 1) * M;
}

// parts 32 lanes apart: a <- (lower part's a, lower part's b), b <- (upper part's a, upper part's b)
__device__ __forceinline__ void swap32(float &a, float &b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
// the same for parts 16 lanes apart (even and odd rows of 16 lanes)
__device__ __forceinline__ void swap16(float &a, float &b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap32(double &a, double &b) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(a), v = (unsigned long long)__double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)v, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(u >> 32), (unsigned)(v >> 32), false, false);
  a = __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0]));
  b = __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
}
__device__ __forceinline__ void swap16(double &a, double &b) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(a), v = (unsigned long long)__double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)u, (unsigned)v, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(u >> 32), (unsigned)(v >> 32), false, false);
  a = __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0]));
  b = __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
}
template <typename C> __device__ __forceinline__ void cswap32(C &a, C &b) {
  swap32(a.x, b.x);
  swap32(a.y, b.y);
}
template <typename C> __device__ __forceinline__ void cswap16(C &a, C &b) {
  swap16(a.x, b.x);
  swap16(a.y, b.y);
}
// the values held by the lower and the upper part, on both
template <typename C> __device__ __forceinline__ void pair_vals(C v, C &lo, C &hi) {
  lo = hi = v;
  cswap32(lo, hi);
}
template <typename C> __device__ __forceinline__ void pair_vals16(C v, C &lo, C &hi) {
  lo = hi = v;
  cswap16(lo, hi);
}

// up ? (SIGN i) t : t
template <int SIGN, typename C> __device__ __forceinline__ C quarter_if(C t, bool up) {
  return SIGN > 0 ? C{up ? -t.y : t.x, up ? t.x : t.y} : C{up ? t.y : t.x, up ? -t.x : t.y};
}

template <int N, int SIGN, typename C> struct fft_split {
  static_assert(N % 2 == 0, "split lines need an even length");
  static constexpr int H = N / 2;
  using T = decltype(C{}.x);
  // decimation in time: lower lanes hold x[2n], upper lanes x[2n+1] (n < H)
  static __device__ __forceinline__ void dit(C (&v)[H], bool upper) {
    fft_line<H, SIGN, C>::run(v);
    if constexpr (H % 2 == 0) {
      // lower lanes take the butterflies k < H/2, upper lanes k + H/2, whose
      // twiddle W^(k + N/4) is a quarter turn further
#pragma unroll
      for (int k = 0; k < H / 2; ++k) {
        C e = v[k], o = v[k + H / 2];
        cswap32(e, o);
        const C t = quarter_if<SIGN>(twmul<N, SIGN>(o, k), upper);
        v[k] = cadd(e, t);
        v[k + H / 2] = csub(e, t);
      }
    } else {
      const T sg = upper ? (T)-1 : (T)1;
#pragma unroll
      for (int k = 0; k < H; ++k) {
        C a, b;
        pair_vals(v[k], a, b);
        const C t = twmul<N, SIGN>(b, k);
        v[k] = C{a.x + sg * t.x, a.y + sg * t.y};
      }
    }
  }
  // decimation in frequency, the mirror: afterwards lower lanes hold X[2k], upper lanes X[2k + 1]
  static __device__ __forceinline__ void dif(C (&v)[H], bool upper) {
    if constexpr (H % 2 == 0) {
#pragma unroll
      for (int k = 0; k < H / 2; ++k) {
        C s = cadd(v[k], v[k + H / 2]);
        C d = quarter_if<SIGN>(twmul<N, SIGN>(csub(v[k], v[k + H / 2]), k), upper);
        cswap32(s, d);
        v[k] = s;
        v[k + H / 2] = d;
      }
    } else {
      const T sg = upper ? (T)-1 : (T)1;
#pragma unroll
      for (int n = 0; n < H; ++n) {
        C a, b;
        pair_vals(v[n], a, b);
        const C d{a.x + sg * b.x, a.y + sg * b.y};
        const C t = twmul<N, SIGN>(d, n);
        v[n] = upper ? t : d;
      }
    }
    fft_line<H, SIGN, C>::run(v);
  }
};

// ONE: dit's last butterflies take W_N^k part_turn(q) as one rounded factor (complex64)
template <int N, int SIGN, typename C, bool ONE = false> struct fft_quad {
  static_assert(N % 4 == 0, "four-lane lines need a length divisible by 4");
  static constexpr int Q = N / 4;
  using T = decltype(C{}.x);
  // W_8^(q >> 1) (SIGN i)^(q & 1): what part q's last butterflies turn by beyond W_N^k
  static __device__ __forceinline__ C part_turn(int q) {
    const T r = (T)0.70710678118654752440;
    const C w = q >= 2 ? C{r, (T)SIGN * r} : C{(T)1, (T)0};
    return quarter_if<SIGN>(w, (q & 1) != 0);
  }
  // v W_N^k part_turn(q).  Two factors round once more than one that is chosen from the
  // two a part's half may have.  Density in complex64, rms error with two factors, with
  // one and with two lanes per line: 1.49e-7, 1.43e-7 and 1.38e-7 at 24^3, 1.93e-7,
  // 1.87e-7 and 1.82e-7 at 64^3 (the choice costs its line pass 0 to 6 %).  The pair
  // planes, bound by VALU issue, keep two: the choice cost 9 to 36 % there, and their
  // solves' error is the same either way within 4 % (2.57e-7 and 2.47e-7 at 72^3, 2.08e-7
  // and 2.14e-7 at 80^3; 2.48e-7 and 2.17e-7 with two lanes)
  static __device__ __forceinline__ C part_twmul(C v, int k, int q, C rho) {
    if constexpr (ONE && sizeof(T) == 4) {
      const bool hi = q >= 2;
      const T c = hi ? (T)kTw<N>.c[k + N / 8] : (T)kTw<N>.c[k];
      const T s = hi ? (T)SIGN * (T)kTw<N>.s[k + N / 8] : (T)SIGN * (T)kTw<N>.s[k];
      return quarter_if<SIGN>(C{v.x * c - v.y * s, v.x * s + v.y * c}, (q & 1) != 0);
    } else {
      return twmul<N, SIGN>(cmul(v, rho), k);
    }
  }
  // decimation in time: part q holds x[4n + q] (n < Q)
  static __device__ __forceinline__ void dit(C (&v)[Q], int q) {
    fft_line<Q, SIGN, C>::run(v);  // Y_q[k], the transform of x[4n + q]
    const bool odd = (q & 1) != 0, hi = q >= 2;
    if constexpr (Q % 2 == 0) {
      // parts q, q ^ 2 hold the even and odd samples of x[2m + (q & 1)]: their
      // length-N/2 transform at m = k + (Q/2)(q >> 1) and at m + Q
#pragma unroll
      for (int k = 0; k < Q / 2; ++k) {
        C e = v[k], o = v[k + Q / 2];
        cswap32(e, o);
        const C t = quarter_if<SIGN>(twmul<N / 2, SIGN>(o, k), hi);
        v[k] = cadd(e, t);
        v[k + Q / 2] = csub(e, t);
      }
      // parts q, q ^ 1 hold those of the even and the odd samples, E[m] and O[m]:
      // X[m] = E + W_N^m O and X[m + N/2] = E - W_N^m O, m now plus Q on odd parts
      const C rho = part_turn(q);
#pragma unroll
      for (int k = 0; k < Q / 2; ++k) {
        C e = v[k], o = v[k + Q / 2];
        cswap16(e, o);
        const C t = part_twmul(o, k, q, rho);
        v[k] = cadd(e, t);
        v[k + Q / 2] = csub(e, t);
      }
    } else {
      const T sa = hi ? (T)-1 : (T)1, sb = odd ? (T)-1 : (T)1;
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        C a, b;
        pair_vals(v[k], a, b);
        const C t = twmul<N / 2, SIGN>(b, k);
        v[k] = C{a.x + sa * t.x, a.y + sa * t.y};
      }
      // part q: X[k + Q quad_rev(q)]
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        C e, o;
        pair_vals16(v[k], e, o);
        const C t = quarter_if<SIGN>(twmul<N, SIGN>(o, k), hi);  // W^(k + N/4) = W^k (SIGN i)
        v[k] = C{e.x + sb * t.x, e.y + sb * t.y};
      }
    }
  }
  // decimation in frequency, the mirror: afterwards part q holds X[4k + q] (k < Q)
  static __device__ __forceinline__ void dif(C (&v)[Q], int q) {
    const bool odd = (q & 1) != 0, hi = q >= 2;
    if constexpr (Q % 2 == 0) {
      // even parts take the sums x[m] + x[m + N/2] (the even frequencies), odd
      // parts the differences times W_N^m
      const C rho = part_turn(q);
#pragma unroll
      for (int k = 0; k < Q / 2; ++k) {
        C s = cadd(v[k], v[k + Q / 2]);
        C d = twmul<N, SIGN>(cmul(csub(v[k], v[k + Q / 2]), rho), k);
        cswap16(s, d);
        v[k] = s;
        v[k + Q / 2] = d;
      }
#pragma unroll
      for (int k = 0; k < Q / 2; ++k) {
        C s = cadd(v[k], v[k + Q / 2]);
        C d = quarter_if<SIGN>(twmul<N / 2, SIGN>(csub(v[k], v[k + Q / 2]), k), hi);
        cswap32(s, d);
        v[k] = s;
        v[k + Q / 2] = d;
      }
    } else {
      // part q holds x[m + Q quad_rev(q)]; with chunk p = p0 + 2 p1 in part q (p0 =
      // q >> 1, p1 = q & 1) and frequency t = t0 + 2 t1,
      // X[4k + t] = sum_m W_Q^(mk) W_N^(mt) sum_p x[m + Q p] W_4^(pt), the inner sum
      // taken over p1 (parts q, q ^ 1) and then over p0 (parts q, q ^ 2)
      // u = x[m + Q p0] + (-1)^t0 x[m + Q (p0 + 2)], t0 = q & 1
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        C a, b;
        pair_vals16(v[k], a, b);
        v[k] = odd ? C{a.x - b.x, a.y - b.y} : C{a.x + b.x, a.y + b.y};
      }
      // z = u(p0 = 0) + (-1)^t1 W_4^t0 u(p0 = 1), t1 = q >> 1
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        C a, b;
        pair_vals(v[k], a, b);
        b = quarter_if<SIGN>(b, odd);  // W_4 = SIGN i
        v[k] = hi ? C{a.x - b.x, a.y - b.y} : C{a.x + b.x, a.y + b.y};
      }
      // W_N^(m q), then the length-Q transform
#pragma unroll
      for (int m = 0; m < Q; ++m) {
        const T c = q == 0 ? (T)1 : q == 1 ? (T)kTw<N>.c[m % N] : q == 2 ? (T)kTw<N>.c[(2 * m) % N] : (T)kTw<N>.c[(3 * m) % N];
        const T sn = q == 0 ? (T)0
                            : (T)SIGN * (q == 1   ? (T)kTw<N>.s[m % N]
                                         : q == 2 ? (T)kTw<N>.s[(2 * m) % N]
                                                  : (T)kTw<N>.s[(3 * m) % N]);
        v[m] = C{v[m].x * c - v[m].y * sn, v[m].x * sn + v[m].y * c};
      }
    }
    fft_line<Q, SIGN, C>::run(v);
  }
};

}  // namespace inqx
