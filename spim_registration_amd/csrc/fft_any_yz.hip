// y and z passes of the two-pass register FFT (fft_any.h): any length with a
// plan of two radices, one launch for one spectrum or for a batch of items.
#include <cstring>

#include "fft_columns.h"

namespace mvd {

struct YAnyParams {
  float2* spec;
  const float2* tw;
  AnyFft f;
  int hx, pitch, ls, zlo, ylo, yhi;
  // input rows outside [iylo, iyhi) of planes outside [izlo, izhi) read as zero
  int iylo, iyhi, izlo, izhi;
};


template <int RC, int DIR>
__device__ __forceinline__ void y_any_body(const YAnyParams& P, int bx, int by, float2* smem) {
  const AnyFft& f = P.f;
  float2* tw = smem;
  float2* buf = smem + f.n;
  const int ls = P.ls, line = threadIdx.x & ((1 << ls) - 1), j = threadIdx.x >> ls;
  for (int i = threadIdx.x; i < f.n; i += blockDim.x) tw[i] = gmem(P.tw)[i];
  // lanes of the row padding [hx, pitch) transform zeros and store them, so
  // that every 128-byte line of a row is written whole
  const int col = (bx << ls) + line;
  const bool valid = col < P.hx, store_col = col < P.pitch;
  const int z = P.zlo + by;
  const auto base = gmem(P.spec) + (int64_t)z * f.n * P.pitch + col;
  const bool plane_in = valid && z >= P.izlo && z < P.izhi;
  if (j < f.b) {
    with_radix_a<RC>(f.a, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      float2 v[R];
      const auto p = base + j * P.pitch;
      const int step = f.b * P.pitch;
#pragma unroll
      for (int t = 0; t < R; ++t) {
        const int y = j + t * f.b;
        v[t] = make_float2(0.f, 0.f);
        if (plane_in && y >= P.iylo && y < P.iyhi) v[t] = p[t * step];
      }
      Dft<R, DIR>::run(v);
      any_put<R>(v, buf, f.pa, ls, line, j);
    });
  }
  __syncthreads();
  if (j < f.a) {
    with_radix_b<RC>(f.b, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      float2 v[R];
      any_take<R>(v, buf, f.pa, ls, line, j);
      any_twiddle<R, DIR>(v, tw, j);
      Dft<R, DIR>::run(v);
      if (store_col) {
        const auto p = base + j * P.pitch;
        const int step = f.a * P.pitch;
#pragma unroll
        for (int t = 0; t < R; ++t) {
          const int y = j + t * f.a;
          if (y >= P.ylo && y < P.yhi) p[t * step] = v[t];
        }
      }
    });
  }
}

// One kernel for single launches (items null: P) and batches (the item of the
// workgroup; the parameters are copied into registers first).
template <int RC, int DIR>
__global__ __launch_bounds__(512) void k_y_any(YAnyParams P, const YAnyParams* items, const int* prefix, const int* gx,
                                               int nitems) {
  extern __shared__ float2 smem[];
  int bx = blockIdx.x, by = blockIdx.y;
  if (items) {
    int item;
    batch_locate(prefix, gx, nitems, item, bx, by);
    P = items[item];
  }
  y_any_body<RC, DIR>(P, bx, by, smem);
}

// z pass: forward, product with the kernel spectrum, inverse (kspec), rows
// [zlo, zhi) written; or one transform in direction DIR times scale.
struct ZAnyParams {
  float2* spec;
  const float2* kspec;
  float2* aux;        // with kspec: also the forward spectrum, all rows (nullable)
  const float2* pre;  // with kspec: the lines already transformed along z (nullable)
  const double* wsum;  // with pre: the product's zero-frequency value is *wsum kdc (nullable)
  double kdc;
  const float2* tw;
  AnyFft f;
  float scale;
  int hx, pitch, qy, ls, zlo, zhi;
};

// First pass of a line set along z: loads and the exchange's stores.
template <int RC, int DIR>
__device__ __forceinline__ void z_any_first(const AnyFft& f, const float2* in, int64_t off, int64_t plane, bool valid,
                                            float2* buf, int ls, int line, int j) {
  if (j < f.b) {
    with_radix_a<RC>(f.a, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      float2 v[R];
      z_any_rows<R>(v, in, off + j * plane, f.b * plane, valid);
      Dft<R, DIR>::run(v);
      any_put<R>(v, buf, f.pa, ls, line, j);
    });
  }
}

template <int RC>
__device__ __forceinline__ void z_any_conv_body(const ZAnyParams& P, int bx, int by, float2* smem) {
  const AnyFft& f = P.f;
  float2* tw = smem;
  float2* buf = smem + f.n;
  const int ls = P.ls, line = threadIdx.x & ((1 << ls) - 1), j = threadIdx.x >> ls;
  for (int i = threadIdx.x; i < f.n; i += blockDim.x) tw[i] = gmem(P.tw)[i];
  const int col = (bx << ls) + line;
  const bool valid = col < P.hx, store_col = col < P.pitch;
  const int64_t plane = (int64_t)P.qy * P.pitch, off = (int64_t)by * P.pitch + col;
  if (!P.pre) z_any_first<RC, -1>(f, P.spec, off, plane, valid, buf, ls, line, j);
  __syncthreads();
  with_radix_b<RC>(f.b, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    float2 v[R], kv[R];
    if (j < f.a) {
      // the kernel spectrum is loaded first, so that it arrives during the transform
      const int64_t at = off + j * plane, step = f.a * plane;
      z_any_rows<R>(kv, P.kspec, at, step, valid);
      if (P.pre) {
        z_any_rows<R>(v, P.pre, at, step, valid);
      } else {
        any_take<R>(v, buf, f.pa, ls, line, j);
        any_twiddle<R, -1>(v, tw, j);
        Dft<R, -1>::run(v);
      }
      if (P.aux && valid) {
#pragma unroll
        for (int t = 0; t < R; ++t) (gmem(P.aux) + at)[t * step] = v[t];
      }
#pragma unroll
      for (int t = 0; t < R; ++t) v[t] = cmul(v[t], kv[t]);
      if (P.wsum && by == 0 && col == 0 && j == 0) v[0] = make_float2((float)(*gmem(P.wsum) * P.kdc), 0.f);
      Dft<R, 1>::run(v);
    }
    __syncthreads();
    if (j < f.a) any_put<R>(v, buf, f.pb, ls, line, j);
  });
  __syncthreads();
  z_any_last<RC>(f, tw, buf, ls, line, j, P.zlo, store_col ? P.zhi : P.zlo, gmem(P.spec) + off, plane,
                 [](auto p, float2 x) { *p = x; });
}

template <int RC>
__global__ __launch_bounds__(512) void k_z_any_conv(ZAnyParams P, const ZAnyParams* items, const int* prefix,
                                                    const int* gx, int nitems) {
  extern __shared__ float2 smem[];
  int bx = blockIdx.x, by = blockIdx.y;
  if (items) {
    int item;
    batch_locate(prefix, gx, nitems, item, bx, by);
    P = items[item];
  }
  z_any_conv_body<RC>(P, bx, by, smem);
}

template <int RC, int DIR>
__global__ __launch_bounds__(512) void k_z_any(ZAnyParams P) {
  extern __shared__ float2 smem[];
  const AnyFft& f = P.f;
  float2* tw = smem;
  float2* buf = smem + f.n;
  const int ls = P.ls, line = threadIdx.x & ((1 << ls) - 1), j = threadIdx.x >> ls;
  for (int i = threadIdx.x; i < f.n; i += blockDim.x) tw[i] = gmem(P.tw)[i];
  const int col = (blockIdx.x << ls) + line;
  const bool valid = col < P.hx, store_col = col < P.pitch;
  const int64_t plane = (int64_t)P.qy * P.pitch, off = (int64_t)blockIdx.y * P.pitch + col;
  z_any_first<RC, DIR>(f, P.spec, off, plane, valid, buf, ls, line, j);
  __syncthreads();
  if (j < f.a) {
    with_radix_b<RC>(f.b, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      float2 v[R];
      any_take<R>(v, buf, f.pa, ls, line, j);
      any_twiddle<R, DIR>(v, tw, j);
      Dft<R, DIR>::run(v);
      if (store_col) {
        const auto p = gmem(P.spec) + off + j * plane;
        const int64_t step = f.a * plane;
#pragma unroll
        for (int t = 0; t < R; ++t) p[t * step] = cscale(v[t], P.scale);
      }
    });
  }
}

// z pass of the likelihood gradient, after the x and y transforms of a block's
// residual R.  Per line: the forward transform R^ (z), then
//   adjoint     A = R^ conj(P^)  -> inverse z -> rows [zlo, zhi) of spec (in
//               place) or adj; skipped when zhi <= zlo;
//   correlation C = conj(R^) W^ e(-2 pi i <k, s> / q), the lag shift s moving
//               the lags the kernel needs, c - j for j in the kernel box, to
//               [0, kd): accumulated into corr over the blocks (mode 0), or
//               inverse-transformed along z with rows [0, kz) stored (mode 1);
//               skipped when corr is null.
struct ZAnyGradParams {
  float2* spec;
  const float2* what;
  const float2* khat;
  float2* corr;
  const float2* tw;
  const float2* twx;   // exp(-2 pi i m / q.x), m < q.x
  const float2* twy;   // exp(-2 pi i m / q.y), m < q.y
  const double* rsum;  // R^(0) from the residual's double sum (nullable)
  float2* adj;         // the adjoint rows' destination (nullable: spec, in place)
  AnyFft f;
  int mode, first, adj_add;  // adj_add: add the adjoint rows to adj
  Int3 shift, q;
  int hx, pitch, ls, zlo, zhi, kz;
};

template <int RC>
__global__ __launch_bounds__(512) void k_z_any_grad(ZAnyGradParams P) {
  extern __shared__ float2 smem[];
  const AnyFft& f = P.f;
  float2* tw = smem;
  float2* buf = smem + f.n;                              // R^, then the correlation
  float2* abuf = buf + ((size_t)any_slots(f) << P.ls);   // the adjoint
  const int ls = P.ls, line = threadIdx.x & ((1 << ls) - 1), j = threadIdx.x >> ls;
  for (int i = threadIdx.x; i < f.n; i += blockDim.x) tw[i] = gmem(P.tw)[i];
  const int ky = blockIdx.y, col = (blockIdx.x << ls) + line;
  const bool valid = col < P.hx;
  const int64_t plane = (int64_t)P.q.y * P.pitch, off = (int64_t)ky * P.pitch + col;
  z_any_first<RC, -1>(f, P.spec, off, plane, valid, buf, ls, line, j);
  __syncthreads();
  const bool corr = P.corr != nullptr, back = corr && P.mode == 1, adj = P.zhi > P.zlo;
  with_radix_b<RC>(f.b, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    float2 v[R], c[R];
    const int64_t at = off + j * plane, step = f.a * plane;
    if (j < f.a) {
      any_take<R>(v, buf, f.pa, ls, line, j);
      any_twiddle<R, -1>(v, tw, j);
      Dft<R, -1>::run(v);
      // R^(0): kz = 0 is v[0] of thread j = 0, of the line (kx, ky) = (0, 0)
      if (P.rsum && ky == 0 && col == 0 && j == 0) v[0] = make_float2((float)*gmem(P.rsum), 0.f);
      if (corr) {
        // lag-shift phase: the (kx, ky) part is one factor per line; index
        // times shift stays below 1024^2 (32-bit remainders)
        const int tx = (int)(((uint32_t)(valid ? col : 0) * (uint32_t)P.shift.x) % (uint32_t)P.q.x);
        const int ty = (int)(((uint32_t)ky * (uint32_t)P.shift.y) % (uint32_t)P.q.y);
        const float2 pl = cmul(gmem(P.twx)[tx], gmem(P.twy)[ty]);
#pragma unroll
        for (int t = 0; t < R; ++t) {
          const int z = j + t * f.a;
          float2 w = make_float2(0.f, 0.f);
          if (valid) w = (gmem(P.what) + at)[t * step];
          const float2 ph = cmul(pl, tw[((uint32_t)z * (uint32_t)P.shift.z) % (uint32_t)f.n]);
          c[t] = cmul(cmul(cconj(v[t]), w), ph);
        }
        if (!back && valid) {
#pragma unroll
          for (int t = 0; t < R; ++t) {
            const auto p = gmem(P.corr) + at + t * step;
            *p = P.first ? c[t] : cadd(c[t], *p);
          }
        }
        if (back) Dft<R, 1>::run(c);
      }
    }
    if (back) {
      __syncthreads();  // the first exchange is read
      if (j < f.a) any_put<R>(c, buf, f.pb, ls, line, j);
    }
    if (adj && j < f.a) {
#pragma unroll
      for (int t = 0; t < R; ++t) {
        float2 p = make_float2(0.f, 0.f);
        if (valid) p = (gmem(P.khat) + at)[t * step];
        v[t] = cmul(v[t], cconj(p));
      }
      Dft<R, 1>::run(v);
      any_put<R>(v, abuf, f.pb, ls, line, j);
    }
  });
  __syncthreads();
  // one run of the last pass for each of the two line sets
#pragma unroll 1
  for (int set = 0; set < 2; ++set) {
    if (set == 0 ? !back : !adj) continue;
    float2* dst = set == 0 ? P.corr : P.adj ? P.adj : P.spec;
    const bool add = set == 1 && P.adj_add;
    const int lo = set == 0 ? 0 : P.zlo, hi = !valid ? lo : set == 0 ? P.kz : P.zhi;
    z_any_last<RC>(f, tw, set == 0 ? buf : abuf, ls, line, j, lo, hi, gmem(dst) + off, plane,
                   [add](auto p, float2 x) { *p = add ? cadd(*p, x) : x; });
  }
}

// ---------------------------------------------------------------------------
// launchers

static YAnyParams y_any_params(const ShapePlan& sp, float2* spec, int zlo, int ylo, int yhi, Int3 in_lo, Int3 in_hi) {
  return YAnyParams{spec, sp.tw_y, any_fft(sp.py), sp.hx, sp.pitch, line_group_of(sp.py).ls, zlo, ylo, yhi,
                    in_lo.y, in_hi.y, in_lo.z, in_hi.z};
}

static void enqueue_y(int rc, bool forward, dim3 grid, dim3 block, size_t lds, hipStream_t stream, const YAnyParams& P,
                      const YAnyParams* items, const int* prefix, const int* gx, int nitems) {
#define MVD_Y(RC)                                                                                                  \
  if (forward) hipLaunchKernelGGL((k_y_any<RC, -1>), grid, block, lds, stream, P, items, prefix, gx, nitems);      \
  else hipLaunchKernelGGL((k_y_any<RC, 1>), grid, block, lds, stream, P, items, prefix, gx, nitems);
  MVD_ANY_CLASS(rc, MVD_Y)
#undef MVD_Y
}

static void enqueue_z_conv(int rc, dim3 grid, dim3 block, size_t lds, hipStream_t stream, const ZAnyParams& P,
                           const ZAnyParams* items, const int* prefix, const int* gx, int nitems) {
#define MVD_Z(RC) hipLaunchKernelGGL((k_z_any_conv<RC>), grid, block, lds, stream, P, items, prefix, gx, nitems);
  MVD_ANY_CLASS(rc, MVD_Z)
#undef MVD_Z
}

hipError_t launch_y_any(const ShapePlan& sp, float2* spec, int zlo, int zhi, int ylo, int yhi, float dir, Int3 in_lo,
                        Int3 in_hi, hipStream_t stream) {
  const LineGroup g = line_group_of(sp.py);
  const YAnyParams P = y_any_params(sp, spec, zlo, ylo, yhi, in_lo, in_hi);
  const dim3 grid(line_groups(sp, g.ls), zhi - zlo), block(g.nt);
  (void)hipGetLastError();
  enqueue_y(any_class(sp.py), dir < 0, grid, block, g.lds, stream, P, nullptr, nullptr, nullptr, 0);
  return hipGetLastError();
}

static ZAnyParams z_any_params(const ShapePlan& sp, float2* spec, const float2* kspec, float scale, int zlo, int zhi,
                               float2* aux, const float2* pre, const double* wsum, double kdc) {
  return ZAnyParams{spec, kspec, aux, pre, wsum, kdc, sp.tw_z, any_fft(sp.pz), scale, sp.hx, sp.pitch, sp.q.y,
                    line_group_of(sp.pz).ls, zlo, zhi};
}

hipError_t launch_z_any(const ShapePlan& sp, float2* spec, const float2* kspec, float scale, int zlo, int zhi,
                        hipStream_t stream, float dir, float2* aux, const float2* pre, const double* wsum,
                        double kdc) {
  const LineGroup g = line_group_of(sp.pz);
  const ZAnyParams P = z_any_params(sp, spec, kspec, scale, zlo, zhi, aux, pre, pre ? wsum : nullptr, kdc);
  const dim3 grid(line_groups(sp, g.ls), sp.q.y), block(g.nt);
  (void)hipGetLastError();
  const int rc = any_class(sp.pz);
  if (kspec) {
    enqueue_z_conv(rc, grid, block, g.lds, stream, P, nullptr, nullptr, nullptr, 0);
  } else {
#define MVD_Z(RC)                                                                            \
  if (dir < 0) hipLaunchKernelGGL((k_z_any<RC, -1>), grid, block, g.lds, stream, P);         \
  else hipLaunchKernelGGL((k_z_any<RC, 1>), grid, block, g.lds, stream, P);
    MVD_ANY_CLASS(rc, MVD_Z)
#undef MVD_Z
  }
  return hipGetLastError();
}

hipError_t launch_z_any_grad(const ShapePlan& sp, float2* spec, const float2* what, const float2* khat, float2* corr,
                             int mode, int first, Int3 shift, int zlo, int zhi, int kz, const double* rsum,
                             float2* adj, bool adj_add, hipStream_t stream) {
  const LineGroup g = line_group_of(sp.pz, 2);
  ZAnyGradParams P{spec, what, khat, corr, sp.tw_z, sp.tw_x, sp.tw_y, rsum, adj, any_fft(sp.pz), mode, first,
                   adj_add ? 1 : 0, shift, sp.q, sp.hx, sp.pitch, g.ls, zlo, zhi, kz};
  const dim3 grid(line_groups(sp, g.ls), sp.q.y), block(g.nt);
  (void)hipGetLastError();
#define MVD_ZG(RC) hipLaunchKernelGGL((k_z_any_grad<RC>), grid, block, g.lds, stream, P);
  MVD_ANY_CLASS(any_class(sp.pz), MVD_ZG)
#undef MVD_ZG
  return hipGetLastError();
}

int build_any_yz_params(const PassDesc& d, void* out, int* gx, int* gy, int* cls, int* threads, size_t* lds) {
  const ShapePlan& sp = *d.sp;
  const FftPlan& p = d.kind == kPassZConv ? sp.pz : sp.py;
  const LineGroup g = line_group_of(p);
  *gx = line_groups(sp, g.ls);
  *cls = any_class(p);
  *threads = g.nt;
  *lds = g.lds;
  if (d.kind == kPassZConv) {
    const ZAnyParams P = z_any_params(sp, d.spec, d.kspec, d.scale, d.zlo, d.zhi, nullptr, nullptr, nullptr, 0.0);
    *gy = sp.q.y;
    std::memcpy(out, &P, sizeof(P));
    return sizeof(P);
  }
  const YAnyParams P = y_any_params(sp, d.spec, d.zlo, d.ylo, d.yhi, {0, 0, 0}, {1 << 30, 1 << 30, 1 << 30});
  *gy = d.zhi - d.zlo;
  std::memcpy(out, &P, sizeof(P));
  return sizeof(P);
}

hipError_t launch_batch_any_yz(int kind, int cls, const void* items, const int* prefix, const int* gx, int nitems,
                               int nwg, int threads, size_t lds, hipStream_t stream) {
  if (nwg <= 0) return hipSuccess;
  (void)hipGetLastError();
  const dim3 grid(nwg), block(threads);
  if (kind == kPassZConv) {
    enqueue_z_conv(cls, grid, block, lds, stream, ZAnyParams{}, static_cast<const ZAnyParams*>(items), prefix, gx, nitems);
  } else if (kind == kPassYForward || kind == kPassYInverse) {
    enqueue_y(cls, kind == kPassYForward, grid, block, lds, stream, YAnyParams{}, static_cast<const YAnyParams*>(items),
              prefix, gx, nitems);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace mvd
