// Two-pass register FFT for any 5-smooth length that splits into two radices
// of at most 32 (all up to 1024 but 2, 3, 5, 972 and 1000), with the radices
// chosen at run time.
//
// A length N = A B is transformed in two passes.  In the first, B threads per
// line each take one radix-A butterfly on x[j + t B] in registers; one LDS
// exchange; in the second, A threads per line each take one radix-B butterfly
// (twiddles exp(dir 2 pi i t j / N)) and hold X[j + t A].  That is the input
// order of a transform with the radices swapped, so the fused z pass runs
// forward, multiplies by the kernel spectrum and comes back with two exchanges
// in all.  A kernel carries the code of every radix and branches on the plan's
// two (wave-uniform) radices, so one kernel serves all lengths.
//
// This replaced a pass per radix 2, 3, 4, 5 or 8 over lines held in LDS (four
// to five LDS sweeps and barriers a transform), which remains for the lengths
// without such a split.  Measured per launch,
// before and after: x inverse with the quotient, rows of 360 samples, 263 x 149
// rows: 126 -> 54 us; x forward there 108 -> 33 us; y of 150 points, 76 columns
// x 96 planes: 15 -> 8 us.  Ten iterations of three 128x128x64 views (150 x 150
// x 96 points) 5.94 -> 3.60 ms, of four 311x263x149 views (360 x 288 x 192)
// 32.5 -> 18.7 ms.  What bounds the kernels: at a few thousand workgroups the
// HBM traffic (2.5 to 3.5 TB/s) and VALU issue together; below a thousand the
// latency of one workgroup's load, two butterflies and store (6 us or so).
//
// Exchange layout: the value t of butterfly j sits at slot j P + t, P the
// radix made odd.  The stores of neighbouring butterflies are an odd number of
// slots apart and the loads (slot t P + j) one slot, so neither conflicts.
#pragma once

#include <type_traits>

#include "mvd_internal.h"

namespace mvd {

// cos and sin of 2 pi m / n at compile time (Taylor series on [0, pi / 4] in
// double, reduced by symmetry; the float constants are their roundings).
namespace trig {
constexpr double kTwoPi = 6.283185307179586476925286766559;
constexpr double cos_small(double x) {
  double t = 1.0, s = 1.0;
  for (int i = 1; i < 14; ++i) {
    t *= -x * x / ((2.0 * i - 1.0) * (2.0 * i));
    s += t;
  }
  return s;
}
constexpr double sin_small(double x) {
  double t = x, s = x;
  for (int i = 1; i < 14; ++i) {
    t *= -x * x / ((2.0 * i) * (2.0 * i + 1.0));
    s += t;
  }
  return s;
}
// m / n of a turn, 0 <= m < n
constexpr double cos_turn(int m, int n);
constexpr double sin_turn(int m, int n) {
  if (2 * m > n) return -sin_turn(n - m, n);
  if (4 * m > n) return sin_turn(n - 2 * m, 2 * n);  // sin(pi - x)
  if (8 * m > n) return cos_small(kTwoPi * (n - 4 * m) / (4.0 * n));
  return sin_small(kTwoPi * m / n);
}
constexpr double cos_turn(int m, int n) {
  if (2 * m > n) return cos_turn(n - m, n);
  if (4 * m > n) return -cos_turn(n - 2 * m, 2 * n);  // cos(pi - x)
  if (8 * m > n) return sin_small(kTwoPi * (n - 4 * m) / (4.0 * n));
  return cos_small(kTwoPi * m / n);
}
template <int N>
struct Table {
  float c[N], s[N];
  constexpr Table() : c(), s() {
    for (int m = 0; m < N; ++m) {
      c[m] = (float)cos_turn(m, N);
      s[m] = (float)sin_turn(m, N);
    }
  }
};
}  // namespace trig

template <int DIR>
__device__ __forceinline__ float2 mul_i(float2 a) {  // a times DIR * i
  return DIR > 0 ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
}

// a exp(DIR 2 pi i m / N), m a constant once the loops around it are unrolled
template <int N, int DIR>
__device__ __forceinline__ float2 mul_root(float2 a, int m) {
  constexpr trig::Table<N> T{};
  if (m == 0) return a;
  if (4 * m == N) return mul_i<DIR>(a);
  if (2 * m == N) return make_float2(-a.x, -a.y);
  if (4 * m == 3 * N) return mul_i<-DIR>(a);
  const float c = T.c[m], s = DIR > 0 ? T.s[m] : -T.s[m];
  return make_float2(a.x * c - a.y * s, a.y * c + a.x * s);
}

// DFT of R values in registers, direction DIR (-1 forward, +1 inverse).
template <int R, int DIR>
struct Dft;

// R = P Q: n = n1 + P n2, k = k1 + Q k2
template <int P, int Q, int DIR>
__device__ __forceinline__ void dft_pq(float2* v) {
  constexpr int N = P * Q;
  float2 a[P][Q];
#pragma unroll
  for (int n1 = 0; n1 < P; ++n1) {
    float2 t[Q];
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) t[n2] = v[n1 + P * n2];
    Dft<Q, DIR>::run(t);
#pragma unroll
    for (int k1 = 0; k1 < Q; ++k1) a[n1][k1] = mul_root<N, DIR>(t[k1], (n1 * k1) % N);
  }
#pragma unroll
  for (int k1 = 0; k1 < Q; ++k1) {
    float2 t[P];
#pragma unroll
    for (int n1 = 0; n1 < P; ++n1) t[n1] = a[n1][k1];
    Dft<P, DIR>::run(t);
#pragma unroll
    for (int k2 = 0; k2 < P; ++k2) v[k1 + Q * k2] = t[k2];
  }
}

template <int DIR>
struct Dft<2, DIR> {
  static __device__ __forceinline__ void run(float2* v) { butterfly<2>(v, (float)DIR); }
};
template <int DIR>
struct Dft<3, DIR> {
  static __device__ __forceinline__ void run(float2* v) {
    const float s1 = 0.866025403784438646763723f;
    const float2 a = v[0], sum = cadd(v[1], v[2]), dif = csub(v[1], v[2]);
    const float2 m = make_float2(a.x - 0.5f * sum.x, a.y - 0.5f * sum.y), d = mul_i<DIR>(dif);
    v[0] = cadd(a, sum);
    v[1] = make_float2(m.x + s1 * d.x, m.y + s1 * d.y);
    v[2] = make_float2(m.x - s1 * d.x, m.y - s1 * d.y);
  }
};
template <int DIR>
struct Dft<4, DIR> {
  static __device__ __forceinline__ void run(float2* v) {
    const float2 a0 = cadd(v[0], v[2]), a1 = csub(v[0], v[2]);
    const float2 a2 = cadd(v[1], v[3]), a3 = mul_i<DIR>(csub(v[1], v[3]));
    v[0] = cadd(a0, a2);
    v[2] = csub(a0, a2);
    v[1] = cadd(a1, a3);
    v[3] = csub(a1, a3);
  }
};
template <int DIR>
struct Dft<5, DIR> {
  static __device__ __forceinline__ void run(float2* v) {
    const float c1 = 0.309016994374947424102293f, c2 = -0.809016994374947424102293f;
    const float s1 = 0.951056516295153572116439f, s2 = 0.587785252292473129168706f;
    const float2 a = v[0];
    const float2 p14 = cadd(v[1], v[4]), m14 = mul_i<DIR>(csub(v[1], v[4]));
    const float2 p23 = cadd(v[2], v[3]), m23 = mul_i<DIR>(csub(v[2], v[3]));
    const float2 r1 = make_float2(a.x + c1 * p14.x + c2 * p23.x, a.y + c1 * p14.y + c2 * p23.y);
    const float2 r2 = make_float2(a.x + c2 * p14.x + c1 * p23.x, a.y + c2 * p14.y + c1 * p23.y);
    const float2 i1 = make_float2(s1 * m14.x + s2 * m23.x, s1 * m14.y + s2 * m23.y);
    const float2 i2 = make_float2(s2 * m14.x - s1 * m23.x, s2 * m14.y - s1 * m23.y);
    v[0] = make_float2(a.x + p14.x + p23.x, a.y + p14.y + p23.y);
    v[1] = cadd(r1, i1);
    v[4] = csub(r1, i1);
    v[2] = cadd(r2, i2);
    v[3] = csub(r2, i2);
  }
};
template <int DIR>
struct Dft<8, DIR> {
  static __device__ __forceinline__ void run(float2* v) {
    float2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    Dft<4, DIR>::run(e);
    Dft<4, DIR>::run(o);
    const float h = 0.707106781186547524400844f;
    const float2 j1 = mul_i<DIR>(o[1]), j3 = mul_i<DIR>(o[3]);
    const float2 t1 = cadd(o[1], j1), t2 = mul_i<DIR>(o[2]), t3 = csub(j3, o[3]);
    v[0] = cadd(e[0], o[0]);
    v[4] = csub(e[0], o[0]);
    v[1] = make_float2(e[1].x + h * t1.x, e[1].y + h * t1.y);
    v[5] = make_float2(e[1].x - h * t1.x, e[1].y - h * t1.y);
    v[2] = cadd(e[2], t2);
    v[6] = csub(e[2], t2);
    v[3] = make_float2(e[3].x + h * t3.x, e[3].y + h * t3.y);
    v[7] = make_float2(e[3].x - h * t3.x, e[3].y - h * t3.y);
  }
};
#define MVD_DFT(R, P, Q)                                                              \
  template <int DIR>                                                                  \
  struct Dft<R, DIR> {                                                                \
    static __device__ __forceinline__ void run(float2* v) { dft_pq<P, Q, DIR>(v); }   \
  };
MVD_DFT(6, 2, 3)
MVD_DFT(9, 3, 3)
MVD_DFT(10, 2, 5)
MVD_DFT(12, 4, 3)
MVD_DFT(15, 3, 5)
MVD_DFT(16, 4, 4)
MVD_DFT(18, 2, 9)
MVD_DFT(20, 4, 5)
MVD_DFT(24, 8, 3)
MVD_DFT(25, 5, 5)
MVD_DFT(27, 3, 9)
MVD_DFT(30, 2, 15)
MVD_DFT(32, 4, 8)
#undef MVD_DFT

// Runs f(integral_constant<int, R>) for the run-time radix r of a plan.  RC is
// the radix class of a kernel (any_class): a kernel takes the registers of its
// largest radix, so the plans are served by four kernels, with radices up to
// 16 (72 VGPRs in the y pass), 20, 27 and 32.  with_radix_a takes a plan's
// first radix a, with_radix_b its second, b <= a.
#define MVD_R(R) \
  case R: f(std::integral_constant<int, R>{}); break;
#define MVD_LAST(R) \
  default: f(std::integral_constant<int, R>{}); break;
template <int RC, class F>
__device__ __forceinline__ void with_radix_a(int r, F f) {
  if constexpr (RC == 0) {
    switch (r) {
      MVD_R(2) MVD_R(3) MVD_R(4) MVD_R(5) MVD_R(6) MVD_R(8) MVD_R(9) MVD_R(10) MVD_R(12) MVD_R(15) MVD_LAST(16)
    }
  } else if constexpr (RC == 1) {
    switch (r) { MVD_R(18) MVD_LAST(20) }
  } else if constexpr (RC == 2) {
    switch (r) { MVD_R(24) MVD_R(25) MVD_LAST(27) }
  } else {
    switch (r) { MVD_R(30) MVD_LAST(32) }
  }
}
template <int RC, class F>
__device__ __forceinline__ void with_radix_b(int r, F f) {
  if constexpr (RC == 0) {
    with_radix_a<0>(r, f);
  } else if constexpr (RC == 1) {
    switch (r) { MVD_R(9) MVD_R(10) MVD_R(12) MVD_R(15) MVD_R(16) MVD_R(18) MVD_LAST(20) }
  } else if constexpr (RC == 2) {
    switch (r) {
      MVD_R(5) MVD_R(9) MVD_R(10) MVD_R(15) MVD_R(16) MVD_R(18) MVD_R(20) MVD_R(24) MVD_R(25) MVD_LAST(27)
    }
  } else {
    switch (r) { MVD_R(16) MVD_R(20) MVD_R(24) MVD_R(25) MVD_R(27) MVD_R(30) MVD_LAST(32) }
  }
}
#undef MVD_R
#undef MVD_LAST
// Calls with a class as a constant: MVD_ANY_CLASS(rc, CALL) runs CALL(0) .. CALL(3).
#define MVD_ANY_CLASS(rc, CALL) \
  switch (rc) {                 \
    case 0: CALL(0) break;      \
    case 1: CALL(1) break;      \
    case 2: CALL(2) break;      \
    default: CALL(3) break;     \
  }

// Two-pass plan in kernel parameters.
struct AnyFft {
  int n, a, b;    // n = a b, a >= b
  int pa, pb;     // a, b made odd: slots per butterfly in the exchanges
  unsigned ma;    // ceil(2^32 / a), ceil(2^32 / b): i / a = umulhi(i, ma) for i < 65536
  unsigned mb;
};
inline AnyFft any_fft(const FftPlan& p) {
  AnyFft f;
  f.n = p.n;
  f.a = p.a;
  f.b = p.b;
  f.pa = p.a | 1;
  f.pb = p.b | 1;
  f.ma = (unsigned)((((uint64_t)1 << 32) + p.a - 1) / p.a);
  f.mb = (unsigned)((((uint64_t)1 << 32) + p.b - 1) / p.b);
  return f;
}
inline int any_class(const FftPlan& p) { return p.a <= 16 ? 0 : p.a <= 20 ? 1 : p.a <= 27 ? 2 : 3; }
// slots of one line in either exchange
__host__ __device__ inline int any_slots(const AnyFft& f) {
  return f.b * f.pa > f.a * f.pb ? f.b * f.pa : f.a * f.pb;
}

// v[t] *= exp(DIR 2 pi i t j / n) from the forward table tw of n STEP entries
template <int R, int DIR, int STEP = 1>
__device__ __forceinline__ void any_twiddle(float2 (&v)[R], const float2* tw, int j) {
  const float2* p = tw;
#pragma unroll
  for (int t = 1; t < R; ++t) {
    p += STEP * j;
    float2 w = *p;
    if (DIR > 0) w.y = -w.y;
    v[t] = cmul(v[t], w);
  }
}

// Sums of squares of values v + shift (x) and v (y), in one order wherever the
// energies of an image are taken.
__device__ __forceinline__ float2 add_squares(float2 s, float v, float shift) {
  const float w = v + shift;
  return make_float2(fmaf(w, w, s.x), fmaf(v, v, s.y));
}
// Sum over each half of a wavefront, in lanes 31 and 63 only: within rows of 16
// lanes by shifts, then from row 0 to 1 and 2 to 3 by a broadcast of the last
// lane, all in the VALU.
template <int CTRL, int ROWS>
__device__ __forceinline__ float add_lanes(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ float half_wave_sum(float v) {
  v = add_lanes<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
  v = add_lanes<0x112, 0xf>(v);
  v = add_lanes<0x114, 0xf>(v);
  v = add_lanes<0x118, 0xf>(v);
  return add_lanes<0x142, 0xa>(v);  // row_bcast:15 to rows 1 and 3
}
// The energy of a half wavefront's pairs of columns x and x + 1 (a, b) within
// [0, nx), in its last lane.
__device__ __forceinline__ float2 energy_of_pair(float2 a, float2 b, int x, int nx) {
  const bool in_a = (unsigned)x < (unsigned)nx, in_b = (unsigned)(x + 1) < (unsigned)nx;
  const float2 s = make_float2((in_a ? a.x : 0.f) + (in_b ? b.x : 0.f), (in_a ? a.y : 0.f) + (in_b ? b.y : 0.f));
  return make_float2(half_wave_sum(s.x), half_wave_sum(s.y));
}

// Exchange accesses of butterfly j: the first pass's stores (values of one
// butterfly, P slots apart between butterflies) and the second pass's loads.
// ls: log2 of the lines, 0 for a line per row of LDS.
template <int R>
__device__ __forceinline__ void any_put(const float2 (&v)[R], float2* buf, int P, int ls, int line, int j) {
  float2* p = buf + ((j * P) << ls) + line;
  const int step = 1 << ls;
#pragma unroll
  for (int t = 0; t < R; ++t) p[t * step] = v[t];
}
template <int R>
__device__ __forceinline__ void any_take(float2 (&v)[R], const float2* buf, int P, int ls, int line, int j) {
  const float2* p = buf + (j << ls) + line;
  const int step = P << ls;
#pragma unroll
  for (int t = 0; t < R; ++t) v[t] = p[t * step];
}

}  // namespace mvd
