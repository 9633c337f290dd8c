// x passes of the two-pass register FFT (fft_any.h): rows of 2M real samples
// <-> M + 1 complex values for any M with a plan of two radices, with the
// window gather of the forward pass and the epilogues of the inverse one.
#include <cstring>

#include "fft_any.h"
#include "pointwise_math.h"

namespace mvd {

namespace {

// Rows per workgroup: as many as give each thread of 256 one butterfly of the
// pass with more of them, within 64 KB of LDS.
struct RowGroup {
  int rows, nt, slots;  // slots: float2 per row in LDS (an exchange, or M + 1 values)
  size_t lds;
};
RowGroup row_group_of(const FftPlan& p) {
  const AnyFft f = any_fft(p);
  RowGroup g;
  // rows start a slots apart modulo the 32 slots of a full set of banks, so that
  // the second pass's loads (a neighbouring slots of each row) run through them
  const int ex = f.b * f.pa, least = ex > p.n + 1 ? ex : p.n + 1;
  g.slots = least + ((p.a - least) % 32 + 32) % 32;
  g.rows = 256 / p.a;
  while (g.rows > 1 && sizeof(float2) * (2 * p.n + (size_t)g.rows * g.slots) > 64 * 1024) --g.rows;
  g.nt = (g.rows * p.a + 63) / 64 * 64;
  g.lds = sizeof(float2) * (2 * p.n + (size_t)g.rows * g.slots);
  return g;
}

}  // namespace

struct XAnyFwdParams {
  ConvGeom g;
  const float* src;
  float2* spec;
  const float2* tw;  // 2M entries
  AnyFft f;
  int pitch, rows, slots;
  float fill;  // constant gathers: the value outside the source
  const float2* center;  // (nullable) y: subtracted from the samples of the source
};

// Second pass of the workgroup's rows after the first pass's exchange, natural
// order into LDS: Z[k] of row l at buf[l slots + k].  Ends synchronised.
template <int RC, int DIR>
__device__ __forceinline__ void x_any_second(const AnyFft& f, const float2* tw, float2* buf, int rows, int slots) {
  const int l = (int)__umulhi((unsigned)threadIdx.x, f.ma), j = threadIdx.x - l * f.a;
  float2* row = buf + l * slots;
  __syncthreads();
  with_radix_b<RC>(f.b, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    float2 v[R];
    if (l < rows) {
      any_take<R>(v, row, f.pa, 0, 0, j);
      any_twiddle<R, DIR, 2>(v, tw, j);
      Dft<R, DIR>::run(v);
    }
    __syncthreads();
    if (l < rows) {
#pragma unroll
      for (int t = 0; t < R; ++t) row[j + t * f.a] = v[t];
    }
  });
  __syncthreads();
}

// Z = FFT(even + i odd) of the rows in LDS unpacked into X[0, M] and the row
// padding [M + 1, pitch) as zeros; a wave takes whole rows.  row_out(l): the
// row's place in global memory, or null.
template <class RowOut>
__device__ __forceinline__ void x_any_unpack(const AnyFft& f, const float2* tw, const float2* buf, int rows, int slots,
                                             int pitch, RowOut row_out) {
  const int M = f.n, lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  for (int l = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); l < rows; l += nw) {
    const auto out = row_out(l);
    if (!out) continue;
    const float2* z = buf + l * slots;
    for (int k = lane; 2 * k <= M; k += 64) {
      const float2 a = z[k], b = z[k ? M - k : 0];
      const float2 E = make_float2(0.5f * (a.x + b.x), 0.5f * (a.y - b.y));
      const float2 O = make_float2(0.5f * (a.y + b.y), 0.5f * (b.x - a.x));  // -i (a - conj b) / 2
      const float2 t = cmul(tw[k], O);
      out[k] = cadd(E, t);
      // X[M - k] = conj(E - t): its twiddle is -conj(tw[k])
      if (2 * k != M) out[M - k] = make_float2(E.x - t.x, t.y - E.y);
    }
    for (int k = M + 1 + lane; k < pitch; k += 64) out[k] = make_float2(0.f, 0.f);
  }
}

// Gathers of the forward pass.
enum XGather : int {
  kXMirror = 0,     // mirror-single, the window reaches past a face by less than the image: one reflection
  kXMirrorAny = 1,  // mirror-single, any number of reflections
  kXConst = 2,      // P.fill out of bounds
  kXWrap = 3,       // the kernel wrapped so that its centre sits at index 0
};
XGather x_gather_of(const ConvGeom& g, int gather) {
  if (gather == kGatherKernelWrap) return kXWrap;
  if (gather != kGatherMirror) return kXConst;
  return g.off.x > -g.src.x && g.off.x + g.win.x <= 2 * g.src.x - 1 ? kXMirror : kXMirrorAny;
}

// Every load is made, from a clamped position where the sample is a constant,
// and the constant selected afterwards: a branch per sample would cut the
// loads in flight into pieces.
template <int RC, int MODE>
__device__ __forceinline__ void x_any_forward_body(const XAnyFwdParams& P, int bx, float2* smem) {
  const AnyFft& f = P.f;
  const ConvGeom& g = P.g;
  float2* tw = smem;
  float2* buf = smem + 2 * f.n;
  for (int i = threadIdx.x; i < 2 * f.n; i += blockDim.x) tw[i] = gmem(P.tw)[i];
  const int nrows = g.q.y * g.q.z, row0 = bx * P.rows;
  {
    const int l = (int)__umulhi((unsigned)threadIdx.x, f.mb), j = threadIdx.x - l * f.b;
    const int row = row0 + l;
    if (l < P.rows) {
      const int z = row / g.q.y, y = row - z * g.q.y;
      const bool live = row < nrows && y < g.win.y && z < g.win.z;
      // the row of the source, and whether it lies in it
      int gy, gz;
      bool in = live;
      if (MODE == kXWrap) {
        gy = y + g.src.y / 2;
        gz = z + g.src.z / 2;
        if (gy >= g.q.y) gy -= g.q.y;
        if (gz >= g.q.z) gz -= g.q.z;
        in = live && gy < g.src.y && gz < g.src.z;
      } else {
        gy = g.off.y + y;
        gz = g.off.z + z;
        if (MODE != kXConst) {
          gy = mirror_single(gy, g.src.y);
          gz = mirror_single(gz, g.src.z);
        } else {
          in = live && gy >= 0 && gy < g.src.y && gz >= 0 && gz < g.src.z;
        }
      }
      const auto srow = gmem(P.src) + (in ? (int64_t)g.src.x * (gy + (int64_t)g.src.y * gz) : 0);
      const int sx = MODE == kXWrap ? g.src.x / 2 : g.off.x, last = g.src.x - 1;
      const int nx = live ? g.win.x : 0;
      const float fill = MODE == kXConst ? P.fill : 0.f, shift = P.center ? gmem(P.center)->y : 0.f;
      auto sample = [&](int x) -> float {
        int gx = sx + x;
        if (MODE == kXWrap) gx = gx >= g.q.x ? gx - g.q.x : gx;
        if (MODE == kXMirror) {
          gx = gx < 0 ? -gx : gx;
          gx = min(gx, 2 * last - gx);
        }
        if (MODE == kXMirrorAny) gx = mirror_single(gx, last + 1);
        const int at = MODE == kXMirrorAny ? gx : min(max(gx, 0), last);
        const bool keep = x < nx && (MODE == kXMirror || MODE == kXMirrorAny || (in && at == gx));
        // (bit masks: a conditional use would let the compiler move the load into a branch)
        const unsigned m = keep ? ~0u : 0u, v = __float_as_uint(srow[at]) & m;
        return __uint_as_float(v | (x < nx && !keep ? __float_as_uint(fill) : 0u)) -
               __uint_as_float(__float_as_uint(shift) & m);
      };
      with_radix_a<RC>(f.a, [&](auto rc) {
        constexpr int R = decltype(rc)::value;
        float2 v[R];
#pragma unroll
        for (int t = 0; t < R; ++t) {
          const int x = 2 * (j + t * f.b);
          v[t] = make_float2(sample(x), sample(x + 1));
        }
        Dft<R, -1>::run(v);
        any_put<R>(v, buf + l * P.slots, f.pa, 0, 0, j);
      });
    }
  }
  x_any_second<RC, -1>(f, tw, buf, P.rows, P.slots);
  x_any_unpack(f, tw, buf, P.rows, P.slots, P.pitch, [&](int l) {
    const int row = row0 + l;
    return row < nrows ? gmem(P.spec) + (int64_t)row * P.pitch : nullptr;
  });
}

template <int RC, int MODE>
__global__ __launch_bounds__(256) void k_x_any_forward(XAnyFwdParams P, const XAnyFwdParams* items, const int* prefix,
                                                       const int* gx, int nitems) {
  extern __shared__ float2 smem[];
  int bx = blockIdx.x, by = 0;
  if (items) {
    int item;
    batch_locate(prefix, gx, nitems, item, bx, by);
    P = items[item];
  }
  x_any_forward_body<RC, MODE>(P, bx, smem);
}

struct XAnyInvParams {
  ConvGeom g;
  const float2* spec;
  EpilogueArgs e;
  const float2* tw;  // 2M entries
  AnyFft f;
  int pitch, rows, slots;
};

template <int RC, int EPI>
__device__ __forceinline__ void x_any_inverse_body(const XAnyInvParams& P, int bx, float2* smem) {
  __shared__ double red_sum[4], red_rsum[4];
  __shared__ float red_max[4];
  const AnyFft& f = P.f;
  const ConvGeom& g = P.g;
  float2* tw = smem;
  float2* buf = smem + 2 * f.n;
  for (int i = threadIdx.x; i < 2 * f.n; i += blockDim.x) tw[i] = gmem(P.tw)[i];
  const int M = f.n, ny = g.eff_size.y, nrows = ny * g.eff_size.z, row0 = bx * P.rows;
  __syncthreads();
  {
    const int l = (int)__umulhi((unsigned)threadIdx.x, f.mb), j = threadIdx.x - l * f.b;
    const int row = row0 + l;
    if (l < P.rows) {
      const bool live = row < nrows;
      const int zo = live ? row / ny : 0, yo = live ? row - zo * ny : 0;
      const auto srow =
          gmem(P.spec) + ((int64_t)(g.eff_local.z + zo) * g.q.y + (g.eff_local.y + yo)) * P.pitch;
      with_radix_a<RC>(f.a, [&](auto rc) {
        constexpr int R = decltype(rc)::value;
        float2 v[R];
        // Z[k] = E + i O from X[k] and X[M - k], read from global memory for
        // both (the second read of a value hits the cache)
        float2 u[R];
#pragma unroll
        for (int t = 0; t < R; ++t) {
          const int k = j + t * f.b;
          v[t] = u[t] = make_float2(0.f, 0.f);
          if (live) {
            v[t] = srow[k];
            u[t] = srow[M - k];
          }
        }
#pragma unroll
        for (int t = 0; t < R; ++t) {
          const float2 b = cconj(u[t]);
          v[t] = cadd(cadd(v[t], b), mul_i<1>(cmul(csub(v[t], b), cconj(tw[j + t * f.b]))));
        }
        Dft<R, 1>::run(v);
        any_put<R>(v, buf + l * P.slots, f.pa, 0, 0, j);
      });
    }
  }
  x_any_second<RC, 1>(f, tw, buf, P.rows, P.slots);
  float* fbuf = reinterpret_cast<float*>(buf);
  const EpilogueArgs& e = P.e;
  const int nx = g.eff_size.x, lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const double inv_lambda = rl_inv_lambda(e.lambda);
  double my_sum = 0.0, my_rsum = 0.0;
  float my_max = -1.f;
  const bool r_rows = EPI != kEpiStore && e.rspec != nullptr;
  // (less = 0 and shift = 0 change no bit of any value they are subtracted from)
  float less = 0.f, shift = 0.f;
  if ((EPI == kEpiQuotient || EPI == kEpiUpdate) && e.center) {
    less = -gmem(e.center)->x;
    shift = gmem(e.center)->y;
  }
  // A wave takes whole rows in pieces of 64 voxels; the inputs of four pieces
  // are loaded before the first is computed (piece by piece, the memory
  // latency of each would follow on the one before).
  constexpr int U = 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int live_rows = min(P.rows, nrows - row0);
  int l = wave, x0 = 0;
  // the row's place in the destination (wave-uniform, one division in all);
  // images hold fewer than 2^31 voxels (checked by the host)
  int zo = (row0 + l) / ny, yo = row0 + l - zo * ny;
  while (l < live_rows) {
    int base[U], vofs[U];
    bool on[U];
    float in0[U], in1[U], in2[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int x = x0 + lane;
      on[u] = l < live_rows && x < nx;
      base[u] = g.eff_offset.x + g.dst.x * ((g.eff_offset.y + yo) + g.dst.y * (g.eff_offset.z + zo)) + x;
      vofs[u] = 2 * l * P.slots + g.eff_local.x + x;
      in0[u] = in2[u] = 0.f;
      in1[u] = EPI == kEpiUpdate ? e.wconst : 1.f;
      if (on[u]) {
        if (EPI == kEpiQuotient || EPI == kEpiResidual) in0[u] = gmem(e.img)[base[u]];
        if (EPI == kEpiUpdate) in0[u] = gmem(e.dst)[base[u]];
        if (EPI == kEpiResidual && e.weight_mode == kWeightArray) in1[u] = gmem(e.weight)[base[u]];
        if (EPI == kEpiUpdate && e.weight_mode != kWeightNone) in1[u] = gmem(e.weight)[base[u]];
        if (EPI == kEpiUpdate && e.weight_mode == kWeightVirtual) in2[u] = gmem(e.wsum)[base[u]];
      }
      x0 += 64;
      if (x0 >= nx) {
        x0 = 0;
        l += nw;
        for (yo += nw; yo >= ny; yo -= ny) ++zo;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (!on[u]) continue;
      const float val = fbuf[vofs[u]];
      const auto dst = gmem(e.dst) + base[u];
      if (EPI == kEpiStore) {
        *dst = val;
      } else if (EPI == kEpiQuotient) {
        const float ratio = rl_quotient(val - less, in0[u]);
        if (r_rows) fbuf[vofs[u]] = ratio - shift;
        else *dst = ratio;
      } else if (EPI == kEpiResidual) {
        float rv = 0.f;
        if (val > 0.f) {
          my_sum += nll_term(in1[u], val, in0[u]);
          rv = nll_residual(in1[u], val, in0[u]);
        }
        if (r_rows) {
          fbuf[vofs[u]] = rv;
          my_rsum += (double)rv;
        } else {
          *dst = rv;
        }
      } else {
        float w = in1[u];
        if (e.weight_mode == kWeightVirtual) w = (float)java_min(1.0, (double)w / (double)in2[u] * e.osem);
        const float next = rl_next_value(in0[u], val - less, w, e.lambda, inv_lambda);
        if (e.keep) gmem(e.keep)[base[u]] = in0[u];
        *dst = next;
        if (r_rows) fbuf[vofs[u]] = next - shift;
        const float change = fabsf(next - in0[u]);
        my_sum += (double)change;
        my_max = java_maxf(my_max, change);
      }
    }
  }
  if (r_rows) {
    // the window rows: the effective row at eff_local; outside it the residual
    // is zero, the ratio one and the estimate mirrored, up to the window's end
    if (EPI == kEpiUpdate) __syncthreads();
    for (int r = wave; r < live_rows; r += nw) {
      float* wrow = fbuf + 2 * r * P.slots;
      for (int h = lane; h < 2 * M - nx; h += 64) {  // the row's positions outside the image
        const int x = h < g.eff_local.x ? h : h + nx, p = x - g.eff_local.x;
        float v = 0.f;
        if (EPI == kEpiQuotient && x < g.win.x) v = 1.f - shift;
        if (EPI == kEpiUpdate && x < g.win.x) v = wrow[g.eff_local.x + mirror_single(p, nx)];
        wrow[x] = v;
      }
    }
  }
  if (EPI == kEpiUpdate || EPI == kEpiResidual) {
    for (int o = 32; o > 0; o >>= 1) {
      my_sum += __shfl_xor(my_sum, o);
      my_max = java_maxf(my_max, __shfl_xor(my_max, o));
      if (EPI == kEpiResidual) my_rsum += __shfl_xor(my_rsum, o);
    }
    if (lane == 0) {
      red_sum[threadIdx.x >> 6] = my_sum;
      red_max[threadIdx.x >> 6] = my_max;
      if (EPI == kEpiResidual) red_rsum[threadIdx.x >> 6] = my_rsum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      double s = 0.0, rs = 0.0;
      float m = -1.f;
      for (int i = 0; i < nw; ++i) {
        s += red_sum[i];
        m = java_maxf(m, red_max[i]);
        if (EPI == kEpiResidual) rs += red_rsum[i];
      }
      gmem(e.part_sum)[bx] = s;
      gmem(e.part_max)[bx] = m;
      if (EPI == kEpiResidual && r_rows) gmem(e.part_rsum)[bx] = rs;
    }
  }
  if constexpr (EPI != kEpiStore) {
    if (!r_rows) return;  // uniform
    // the x transform of the window rows
    const int l = (int)__umulhi((unsigned)threadIdx.x, f.mb), j = threadIdx.x - l * f.b;
    __syncthreads();
    if ((EPI == kEpiQuotient || EPI == kEpiUpdate) && e.part_sq) {
      // the rows' energies from LDS, two neighbouring values of every row a
      // thread, a piece per half wavefront: the quotient of 880x880x440 1459 ->
      // 1538 us (1614 with single values and shuffles through LDS)
      const int pieces = energy_pieces(2 * M);
      for (int c = threadIdx.x; c < pieces * 32; c += blockDim.x) {
        const float2* q = buf + min(c, M - 1);
        float2 a = make_float2(0.f, 0.f), b = a;
#pragma unroll 4
        for (int r = 0; r < live_rows; ++r) {
          const float2 v = q[r * P.slots];
          a = add_squares(a, v.x, shift);
          b = add_squares(b, v.y, shift);
        }
        const float2 s = energy_of_pair(a, b, 2 * c - g.eff_local.x, nx);
        if ((lane & 31) == 31) gmem(e.part_sq)[(int64_t)bx * pieces + (c >> 5)] = s;
      }
    }
    with_radix_a<RC>(f.a, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      float2 v[R];
      if (l < P.rows) {
#pragma unroll
        for (int t = 0; t < R; ++t) v[t] = buf[l * P.slots + j + t * f.b];
        Dft<R, -1>::run(v);
      }
      __syncthreads();
      if (l < P.rows) any_put<R>(v, buf + l * P.slots, f.pa, 0, 0, j);
    });
    x_any_second<RC, -1>(f, tw, buf, P.rows, P.slots);
    x_any_unpack(f, tw, buf, P.rows, P.slots, e.rpitch, [&](int r) {
      const int row = row0 + r;
      return row < nrows ? gmem(e.rspec) + ((int64_t)(g.eff_local.z + row / ny) * g.q.y + g.eff_local.y + row % ny) *
                                               e.rpitch
                         : nullptr;
    });
  }
}

template <int RC, int EPI>
__global__ __launch_bounds__(256) void k_x_any_inverse(XAnyInvParams P, const XAnyInvParams* items, const int* prefix,
                                                       const int* gx, int nitems) {
  extern __shared__ float2 smem[];
  int bx = blockIdx.x, by = 0;
  if (items) {
    int item;
    batch_locate(prefix, gx, nitems, item, bx, by);
    P = items[item];
  }
  x_any_inverse_body<RC, EPI>(P, bx, smem);
}

// ---------------------------------------------------------------------------
// launchers

int x_any_rows_per_wg(const FftPlan& p) { return row_group_of(p).rows; }

static XAnyFwdParams x_any_fwd_params(const ShapePlan& sp, const ConvGeom& g, const float* src, int gather,
                                      float2* spec, const float2* center = nullptr) {
  const RowGroup r = row_group_of(sp.px);
  return XAnyFwdParams{g, src, spec, sp.tw_x, any_fft(sp.px), sp.pitch, r.rows, r.slots,
                       gather == kGatherOne ? 1.f : 0.f, center};
}

static hipError_t enqueue_x_forward(int rc, int mode, dim3 grid, dim3 block, size_t lds, hipStream_t stream,
                                    const XAnyFwdParams& P, const XAnyFwdParams* items, const int* prefix,
                                    const int* gx, int nitems) {
  (void)hipGetLastError();
#define MVD_XG(RC, MODE) \
  case MODE: hipLaunchKernelGGL((k_x_any_forward<RC, MODE>), grid, block, lds, stream, P, items, prefix, gx, nitems); break;
#define MVD_XF(RC)                                                                                                   \
  switch (mode) {                                                                                                    \
    MVD_XG(RC, kXMirror) MVD_XG(RC, kXMirrorAny) MVD_XG(RC, kXConst) MVD_XG(RC, kXWrap)                              \
    default: return hipErrorInvalidValue;                                                                            \
  }
  MVD_ANY_CLASS(rc, MVD_XF)
#undef MVD_XF
#undef MVD_XG
  return hipGetLastError();
}

hipError_t launch_x_forward_any(const ShapePlan& sp, const ConvGeom& g, const float* src, int gather, float2* spec,
                                hipStream_t stream, const float2* center) {
  const RowGroup r = row_group_of(sp.px);
  const int nrows = g.q.y * g.q.z;
  return enqueue_x_forward(any_class(sp.px), x_gather_of(g, gather), dim3((nrows + r.rows - 1) / r.rows), dim3(r.nt), r.lds, stream,
                           x_any_fwd_params(sp, g, src, gather, spec, center), nullptr, nullptr, nullptr, 0);
}

static hipError_t enqueue_x_inverse(int rc, int epi, dim3 grid, dim3 block, size_t lds, hipStream_t stream,
                                    const XAnyInvParams& P, const XAnyInvParams* items, const int* prefix,
                                    const int* gx, int nitems) {
  (void)hipGetLastError();
#define MVD_XE(RC, EPI) \
  case EPI: hipLaunchKernelGGL((k_x_any_inverse<RC, EPI>), grid, block, lds, stream, P, items, prefix, gx, nitems); break;
#define MVD_XI(RC)                                                                                       \
  switch (epi) {                                                                                         \
    MVD_XE(RC, kEpiStore) MVD_XE(RC, kEpiQuotient) MVD_XE(RC, kEpiUpdate) MVD_XE(RC, kEpiResidual)       \
    default: return hipErrorInvalidValue;                                                                \
  }
  MVD_ANY_CLASS(rc, MVD_XI)
#undef MVD_XI
#undef MVD_XE
  return hipGetLastError();
}

hipError_t launch_x_inverse_any(const ShapePlan& sp, const ConvGeom& g, const float2* spec, const EpilogueArgs& e,
                                hipStream_t stream, int nwg) {
  const RowGroup r = row_group_of(sp.px);
  const XAnyInvParams P{g, spec, e, sp.tw_x, any_fft(sp.px), sp.pitch, r.rows, r.slots};
  return enqueue_x_inverse(any_class(sp.px), e.mode, dim3(nwg), dim3(r.nt), r.lds, stream, P, nullptr, nullptr,
                           nullptr, 0);
}

int build_any_x_params(const PassDesc& d, void* out, int* gx, int* gy, int* cls, int* threads, size_t* lds) {
  const ShapePlan& sp = *d.sp;
  const RowGroup r = row_group_of(sp.px);
  *gy = 1;
  *threads = r.nt;
  *lds = r.lds;
  if (d.kind == kPassXForward) {
    const XAnyFwdParams P = x_any_fwd_params(sp, d.g, d.src, d.gather, d.spec);
    *gx = (d.g.q.y * d.g.q.z + r.rows - 1) / r.rows;
    *cls = any_class(sp.px) + 4 * x_gather_of(d.g, d.gather);
    std::memcpy(out, &P, sizeof(P));
    return sizeof(P);
  }
  const XAnyInvParams P{d.g, d.spec, d.e, sp.tw_x, any_fft(sp.px), sp.pitch, r.rows, r.slots};
  *gx = (d.g.eff_size.y * d.g.eff_size.z + r.rows - 1) / r.rows;
  *cls = any_class(sp.px);
  std::memcpy(out, &P, sizeof(P));
  return sizeof(P);
}

hipError_t launch_batch_any_x(int kind, int cls, int epi, const void* items, const int* prefix, const int* gx,
                              int nitems, int nwg, int threads, size_t lds, hipStream_t stream) {
  if (nwg <= 0) return hipSuccess;
  if (kind == kPassXForward)
    return enqueue_x_forward(cls & 3, cls >> 2, dim3(nwg), dim3(threads), lds, stream, XAnyFwdParams{},
                             static_cast<const XAnyFwdParams*>(items), prefix, gx, nitems);
  return enqueue_x_inverse(cls, epi, dim3(nwg), dim3(threads), lds, stream, XAnyInvParams{},
                           static_cast<const XAnyInvParams*>(items), prefix, gx, nitems);
}

}  // namespace mvd
