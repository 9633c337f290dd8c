// Column passes (y and z) of the two-pass register FFT: pieces shared by
// fft_any_yz.hip and fft_rows.hip.
#pragma once

#include "fft_any.h"

namespace mvd {

// Lines per workgroup: 16 columns make every row segment a whole 128-byte
// line; lengths whose lines do not fit 64 KB of LDS that way take 8 or 4.
struct LineGroup {
  int ls;  // log2 of the lines
  int nt;  // threads: one butterfly of the pass with more of them each
  size_t lds;
};
inline LineGroup line_group_of(const FftPlan& p, int sets = 1) {
  const AnyFft f = any_fft(p);
  LineGroup g;
  for (g.ls = 4;; --g.ls) {
    g.lds = sizeof(float2) * (f.n + ((size_t)sets * any_slots(f) << g.ls));
    if (g.lds <= 64 * 1024 || g.ls == 2) break;
  }
  g.nt = ((p.a << g.ls) + 63) / 64 * 64;
  return g;
}

// line groups along a row of the spectrum, its padding included
inline int line_groups(const ShapePlan& sp, int ls) { return (sp.pitch + (1 << ls) - 1) >> ls; }

// Last pass of an inverse transform along z whose first one (radix b) is in
// the exchange: store(p, value), p = out + z plane, for the rows z in [lo, hi).
template <int RC, class Ptr, class Store>
__device__ __forceinline__ void z_any_last(const AnyFft& f, const float2* tw, const float2* buf, int ls, int line,
                                           int j, int lo, int hi, Ptr out, int64_t plane, Store store) {
  if (j < f.b) {
    with_radix_a<RC>(f.a, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      float2 v[R];
      any_take<R>(v, buf, f.pb, ls, line, j);
      any_twiddle<R, 1>(v, tw, j);
      Dft<R, 1>::run(v);
      const auto p = out + j * plane;
      const int64_t step = f.b * plane;
#pragma unroll
      for (int t = 0; t < R; ++t) {
        const int z = j + t * f.b;
        if (z >= lo && z < hi) store(p + t * step, v[t]);
      }
    });
  }
}

// R rows of a column, `step` apart; zero for the lanes past the spectrum.
template <int R>
__device__ __forceinline__ void z_any_rows(float2 (&v)[R], const float2* in, int64_t off, int64_t step, bool valid) {
  const auto p = gmem(in) + off;
#pragma unroll
  for (int t = 0; t < R; ++t) {
    v[t] = make_float2(0.f, 0.f);
    if (valid) v[t] = p[t * step];
  }
}

}  // namespace mvd
