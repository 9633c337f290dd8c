// Whole-image convolution by rows (RowConv in mvd_internal.h): the y and z
// passes between an array of x-transformed image rows, one per (y, z) of the
// image, and tiles of planes.  The window's rows and planes outside the image
// are never stored: the y pass reads a mirrored row from the row that it
// mirrors, the z pass a mirrored plane likewise, and the constant ones come
// from one row and one plane.

#include <algorithm>
#include <cstring>

#include "fft_columns.h"
#include "pointwise_math.h"

namespace mvd {

constexpr int kRowsThreads = 320;  // at most, per workgroup

// What lies outside the image.
enum RowsMode : int {
  kRowsMirror = 0,     // mirror-single, one reflection
  kRowsMirrorAny = 1,  // mirror-single, any number of reflections
  kRowsConst = 2,      // the constant row / plane
};

// Index in [0, n) that position p of the extended axis shows, and whether it
// shows one (kRowsConst: else the constant).
template <int MODE>
__device__ __forceinline__ int rows_index(int p, int n, bool& in) {
  in = true;
  if (MODE == kRowsMirrorAny) return mirror_single(p, n);
  if (MODE == kRowsMirror) {
    p = p < 0 ? -p : p;
    return min(p, 2 * n - 2 - p);
  }
  in = (unsigned)p < (unsigned)n;
  return in ? p : 0;
}

// v, or zero: by masks, so that the load of v stays where it is (a conditional
// use lets the compiler move it into a branch)
__device__ __forceinline__ float2 keep_if(float2 v, bool keep) {
  const unsigned m = keep ? ~0u : 0u;
  return make_float2(__uint_as_float(__float_as_uint(v.x) & m), __uint_as_float(__float_as_uint(v.y) & m));
}

// Planes are stored in slabs of eight rows, [(q.y + 7) / 8][planes][8][pitch]:
// the z pass then walks a column in steps of eight rows instead of a whole
// plane (0.7 MB at 288 x 304), and the y pass writes 36 runs of eight rows
// instead of 288 of one; with whole planes every access of a column is on
// another page, and the z pass ran between 267 and 390 us on different machines.
//
// Every access is a 32-bit byte offset from a wave-uniform base (the host keeps
// the arrays below 4 GiB): 64-bit addresses of a butterfly's loads would take
// two registers each.
struct YRowsParams {
  float2* rows;        // [nz][ny][pitch], then the constant row
  float2* planes;      // slabs of this tile
  const float2* tw;
  AnyFft f;
  int hx, pitch, ls, ny;
  int off, win;        // image row of tile row 0; tile rows that hold the window
  int lo, cnt, eoff;   // inverse: tile rows [lo, lo + cnt) are the image rows from eoff
  int nrows;           // ny nz: the constant row's index
  int nplanes;         // of the tile
};

// Byte offset in a slab array of row y of plane 0 (row: bytes of a row, a
// multiple of 128; slab: bytes of a slab).
__device__ __forceinline__ uint32_t slab_row(int y, uint32_t row, uint32_t slab) {
  return (__umul24((unsigned)y >> 3, slab >> 7) << 7) + __umul24((unsigned)y & 7, row);
}

// The butterflies of a pass of a line group, `count` per line, over the threads
// of a workgroup: body(j).  Where there are more butterflies than threads, the
// rest of them go to a wave that depends on the workgroup.
template <class F>
__device__ __forceinline__ void for_butterflies(int count, int ls, F body) {
  const int total = count << ls, nt = blockDim.x;
#pragma unroll 1
  for (int r = 0; r < total; r += nt) {
    int i = threadIdx.x;
    if (r > 0) i = r + (nt == 256 ? (i + (blockIdx.x & 3) * 64) & 255 : i);
    if (i < total) body(i >> ls);
  }
}

template <int RC, int MODE>
__global__ __launch_bounds__(kRowsThreads) void k_y_rows_forward(const YRowsParams* items, const int* prefix, const int* gx,
                                                        int nitems) {
  extern __shared__ float2 smem[];
  int item, bx, z;
  batch_locate(prefix, gx, nitems, item, bx, z);
  const YRowsParams P = items[item];
  const AnyFft& f = P.f;
  float2* tw = smem;
  float2* buf = smem + f.n;
  const int ls = P.ls, line = threadIdx.x & ((1 << ls) - 1);
  for (int i = threadIdx.x; i < f.n; i += blockDim.x) tw[i] = gmem(P.tw)[i];
  const int col = (bx << ls) + line;
  const bool valid = col < P.hx, store_col = col < P.pitch;
  const float2* in_base = P.rows + (int64_t)z * P.ny * P.pitch;
  const uint32_t row = (uint32_t)P.pitch * 8u, at = (uint32_t)(valid ? col : 0) * 8u;
  const uint32_t crow = (uint32_t)(P.nrows - z * P.ny) * row + at;
  for_butterflies(f.b, ls, [&](int j) {
    with_radix_a<RC>(f.a, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      float2 v[R];
#pragma unroll
      for (int t = 0; t < R; ++t) {
        const int y = j + t * f.b;
        bool in;
        const int g = rows_index<MODE>(min(y, P.win - 1) + P.off, P.ny, in);
        const uint32_t o = MODE == kRowsConst && !in ? crow : (uint32_t)g * row + at;
        v[t] = keep_if(*gbyte(in_base, o), valid && y < P.win);
      }
      Dft<R, -1>::run(v);
      any_put<R>(v, buf, f.pa, ls, line, j);
    });
  });
  __syncthreads();
  const uint32_t slab = (uint32_t)P.nplanes * 8u * row;
  float2* out_base = P.planes + (int64_t)z * 8 * P.pitch;
  for_butterflies(f.a, ls, [&](int j) {
    with_radix_b<RC>(f.b, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      float2 v[R];
      any_take<R>(v, buf, f.pa, ls, line, j);
      any_twiddle<R, -1>(v, tw, j);
      Dft<R, -1>::run(v);
      if (store_col) {
#pragma unroll
        for (int t = 0; t < R; ++t) *gbyte(out_base, slab_row(j + t * f.a, row, slab) + (uint32_t)col * 8u) = v[t];
      }
    });
  });
}

template <int RC>
__global__ __launch_bounds__(kRowsThreads) void k_y_rows_inverse(const YRowsParams* items, const int* prefix, const int* gx,
                                                        int nitems) {
  extern __shared__ float2 smem[];
  int item, bx, z;
  batch_locate(prefix, gx, nitems, item, bx, z);
  const YRowsParams P = items[item];
  const AnyFft& f = P.f;
  float2* tw = smem;
  float2* buf = smem + f.n;
  const int ls = P.ls, line = threadIdx.x & ((1 << ls) - 1);
  for (int i = threadIdx.x; i < f.n; i += blockDim.x) tw[i] = gmem(P.tw)[i];
  const int col = (bx << ls) + line;
  const bool store_col = col < P.pitch;
  const uint32_t row = (uint32_t)P.pitch * 8u, at = (uint32_t)(store_col ? col : 0) * 8u;
  const uint32_t slab = (uint32_t)P.nplanes * 8u * row;
  const float2* in_base = P.planes + (int64_t)z * 8 * P.pitch;
  for_butterflies(f.b, ls, [&](int j) {
    with_radix_a<RC>(f.a, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      float2 v[R];
#pragma unroll
      for (int t = 0; t < R; ++t) v[t] = *gbyte(in_base, slab_row(j + t * f.b, row, slab) + at);
      Dft<R, 1>::run(v);
      any_put<R>(v, buf, f.pa, ls, line, j);
    });
  });
  __syncthreads();
  if (!store_col) return;
  float2* out_base = P.rows + ((int64_t)z * P.ny + P.eoff) * P.pitch;
  for_butterflies(f.a, ls, [&](int j) {
    with_radix_b<RC>(f.b, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      float2 v[R];
      any_take<R>(v, buf, f.pa, ls, line, j);
      any_twiddle<R, 1>(v, tw, j);
      Dft<R, 1>::run(v);
      const uint32_t step = (uint32_t)f.a * row;
      uint32_t o = (uint32_t)(j - P.lo) * row + at;  // (wraps below row lo, where nothing is stored)
#pragma unroll
      for (int t = 0; t < R; ++t, o += step)
        if ((unsigned)(j + t * f.a - P.lo) < (unsigned)P.cnt) *gbyte(out_base, o) = v[t];
    });
  });
}

struct ZRowsParams {
  float2* planes;        // the tiles' slabs, then those of the constant plane
  const float2* kspec;   // [qz][qy][pitch], or slabs of qz planes
  const float2* tw;
  AnyFft f;
  int hx, pitch, qy, ls, nz, off, win;  // off: the window's first plane is image plane -off
  int tiles, gxl, groups;               // line groups along a row; line groups of a tile
  int kslabs;                           // the kernel spectrum is stored in slabs
};

// The tiles of one line group run on one XCD one after another (workgroup w of
// a launch runs on XCD w mod 8), so the second and later ones find the kernel
// spectrum in its L2.
//
// The second pass, the product and the inverse's first pass of a butterfly stay
// in one thread's registers, and its values go back to the slots that it read
// (slot t pa + j, value t of butterfly j): no other butterfly reads those, so no
// barrier stands between, and the last pass reads pa neighbouring slots.
template <int RC, int MODE>
__global__ __launch_bounds__(kRowsThreads) void k_z_rows(const ZRowsParams* items, const int* prefix, const int* gx,
                                                int nitems) {
  extern __shared__ float2 smem[];
  int item, w, unused;
  batch_locate(prefix, gx, nitems, item, w, unused);
  const ZRowsParams P = items[item];
  const int rest = w >> 3, tile = rest % P.tiles, group = rest / P.tiles * 8 + (w & 7);
  if (group >= P.groups) return;  // uniform
  const AnyFft& f = P.f;
  float2* tw = smem;
  float2* buf = smem + f.n;
  const int ls = P.ls, line = threadIdx.x & ((1 << ls) - 1);
  for (int i = threadIdx.x; i < f.n; i += blockDim.x) tw[i] = gmem(P.tw)[i];
  const int by = group / P.gxl, bx = group - by * P.gxl;
  const int col = (bx << ls) + line;
  const bool store_col = col < P.pitch;
  // byte offsets: from plane to plane, and of the workgroup's column
  const uint32_t row = (uint32_t)P.pitch * 8u, plane = 8u * row, in_row = (uint32_t)(store_col ? col : 0) * 8u;
  const uint32_t tile_bytes = (uint32_t)((P.qy + 7) >> 3) * (uint32_t)P.nz * plane;
  const uint32_t at = slab_row(by, row, (uint32_t)P.nz * plane) + in_row;
  const uint32_t kplane = P.kslabs ? plane : (uint32_t)P.qy * row;
  const uint32_t kat = (P.kslabs ? slab_row(by, row, (uint32_t)f.n * plane) : (uint32_t)by * row) + in_row;
  float2* base = P.planes + (int64_t)tile * (tile_bytes >> 3);
  const uint32_t cplane = (uint32_t)(P.tiles - tile) * tile_bytes + (uint32_t)by * row + in_row;
  for_butterflies(f.b, ls, [&](int j) {
    with_radix_a<RC>(f.a, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      float2 v[R];
#pragma unroll
      for (int t = 0; t < R; ++t) {
        const int z = j + t * f.b;
        bool in;
        const int g = rows_index<MODE>(min(z, P.win - 1) - P.off, P.nz, in);
        const uint32_t o = MODE == kRowsConst && !in ? cplane : (uint32_t)g * plane + at;
        v[t] = keep_if(*gbyte(base, o), z < P.win);
      }
      Dft<R, -1>::run(v);
      any_put<R>(v, buf, f.pa, ls, line, j);
    });
  });
  __syncthreads();
  for_butterflies(f.a, ls, [&](int j) {
    with_radix_b<RC>(f.b, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      float2 v[R];
      any_take<R>(v, buf, f.pa, ls, line, j);
      any_twiddle<R, -1>(v, tw, j);
      Dft<R, -1>::run(v);
      uint32_t o = (uint32_t)j * kplane + kat;
      const uint32_t step = (uint32_t)f.a * kplane;
#pragma unroll
      for (int t = 0; t < R; ++t, o += step) v[t] = cmul(v[t], *gbyte(P.kspec, o));
      Dft<R, 1>::run(v);
      float2* p = buf + (j << ls) + line;
      const int slots = f.pa << ls;
#pragma unroll
      for (int t = 0; t < R; ++t) p[t * slots] = v[t];
    });
  });
  __syncthreads();
  if (!store_col) return;
  for_butterflies(f.b, ls, [&](int j) {
    with_radix_a<RC>(f.a, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      float2 v[R];
      const float2* p = buf + ((j * f.pa) << ls) + line;
#pragma unroll
      for (int t = 0; t < R; ++t) v[t] = p[t << ls];
      any_twiddle<R, 1>(v, tw, j);
      Dft<R, 1>::run(v);
      const uint32_t step = (uint32_t)f.b * plane;
      uint32_t o = (uint32_t)(j - P.off) * plane + at;  // (wraps below plane off, where nothing is stored)
#pragma unroll
      for (int t = 0; t < R; ++t, o += step)
        if ((unsigned)(j + t * f.b - P.off) < (unsigned)P.nz) *gbyte(base, o) = v[t];
    });
  });
}

// Lines per workgroup: sixteen (whole 128-byte lines of a row) in up to 80 KB
// of LDS, which still holds two workgroups per CU; longer lengths take fewer.
// Threads: 256 where the first radix's butterflies fit them, although the
// second radix then has up to 320 or 384 (a wave for each would make five or six
// waves, two of them on one SIMD, whose registers two such workgroups fill: 1.5
// were resident on average; 288 points along y 136 -> 119 us and 320 along z
// 280 -> 267 us for 6 views of 512x512x256).  Where neither pass fits (360 =
// 20 x 18) both would run twice as long for a few butterflies: 320 threads
// (ten stacks of 96^3 to 384^3: z passes of these lengths 66 -> 48 ms).
static LineGroup rows_group_of(const FftPlan& p) {
  const AnyFft f = any_fft(p);
  LineGroup g;
  for (g.ls = 4;; --g.ls) {
    g.lds = sizeof(float2) * (f.n + ((size_t)f.b * f.pa << g.ls));
    if (g.lds <= 80 * 1024 || g.ls == 2) break;
  }
  g.nt = ((p.a << g.ls) + 63) / 64 * 64;
  if (g.nt > kRowsThreads || (p.b << g.ls) <= 256) g.nt = std::min(256, g.nt);
  return g;
}

// A spectrum [qz][qy][pitch] into slabs (the rows past qy are left as they are).
__global__ __launch_bounds__(256) void k_to_slabs(const float2* in, float2* out, int qy, int pitch) {
  const int y = blockIdx.x, z = blockIdx.y, qz = gridDim.y;
  const auto src = gmem(in) + ((int64_t)z * qy + y) * pitch;
  const auto dst = gmem(out) + (((int64_t)(y >> 3) * qz + z) * 8 + (y & 7)) * pitch;
  for (int x = threadIdx.x; x < pitch; x += 256) dst[x] = src[x];
}

int64_t slab_elems(const ShapePlan& sp, int planes) { return (int64_t)((sp.q.y + 7) / 8) * planes * 8 * sp.pitch; }

hipError_t launch_to_slabs(const ShapePlan& sp, const float2* in, float2* out, hipStream_t stream) {
  (void)hipGetLastError();
  hipLaunchKernelGGL(k_to_slabs, dim3(sp.q.y, sp.q.z), dim3(256), 0, stream, in, out, sp.q.y, sp.pitch);
  return hipGetLastError();
}

int build_rows_params(const RowsPass& d, void* out, int* gx, int* gy, int* cls, int* threads, size_t* lds) {
  const ShapePlan& sp = *d.sp;
  const FftPlan& p = d.kind == kPassZConv ? sp.pz : sp.py;
  const LineGroup g = rows_group_of(p);
  *threads = g.nt;
  *lds = g.lds;
  const int gxl = line_groups(sp, g.ls);
  auto mode_of = [&](int lo, int hi, int n) {  // extended positions [lo, hi) of an axis of n
    return !d.mirror ? kRowsConst : lo > -n && hi <= 2 * n - 1 ? kRowsMirror : kRowsMirrorAny;
  };
  if (d.kind == kPassZConv) {
    const int groups = gxl * sp.q.y;
    const ZRowsParams P{d.planes, d.kspec, sp.tw_z, any_fft(p), sp.hx, sp.pitch, sp.q.y, g.ls, d.n.z,
                        d.off_z, d.win_z, d.tiles, gxl, groups, d.kslabs ? 1 : 0};
    *gx = (groups + 7) / 8 * 8 * d.tiles;
    *gy = 1;
    *cls = any_class(p) + 4 * mode_of(-d.off_z, d.win_z - d.off_z, d.n.z);
    std::memcpy(out, &P, sizeof(P));
    return sizeof(P);
  }
  const YRowsParams P{d.rows, d.planes, sp.tw_y, any_fft(p), sp.hx, sp.pitch, g.ls, d.n.y, d.off_y, d.win_y,
                      d.lo_y, d.cnt_y, d.eoff_y, d.n.y * d.n.z, d.nplanes};
  *gx = gxl;
  *gy = d.nplanes;
  *cls = any_class(p) + (d.kind == kPassYForward ? 4 * mode_of(d.off_y, d.off_y + d.win_y, d.n.y) : 0);
  std::memcpy(out, &P, sizeof(P));
  return sizeof(P);
}

hipError_t launch_rows(int kind, int cls, const void* items, const int* prefix, const int* gx, int nitems, int nwg,
                       int threads, size_t lds, hipStream_t stream) {
  if (nwg <= 0) return hipSuccess;
  (void)hipGetLastError();
  const dim3 grid(nwg), block(threads);
  const YRowsParams* yi = static_cast<const YRowsParams*>(items);
  const ZRowsParams* zi = static_cast<const ZRowsParams*>(items);
  const int mode = cls >> 2;
#define MVD_ROWS(K, RC, IT)                                                                                       \
  if (mode == kRowsMirror) hipLaunchKernelGGL((K<RC, kRowsMirror>), grid, block, lds, stream, IT, prefix, gx, nitems); \
  else if (mode == kRowsConst) hipLaunchKernelGGL((K<RC, kRowsConst>), grid, block, lds, stream, IT, prefix, gx, nitems); \
  else hipLaunchKernelGGL((K<RC, kRowsMirrorAny>), grid, block, lds, stream, IT, prefix, gx, nitems);
#define MVD_YF(RC) MVD_ROWS(k_y_rows_forward, RC, yi)
#define MVD_Z(RC) MVD_ROWS(k_z_rows, RC, zi)
#define MVD_YI(RC) hipLaunchKernelGGL((k_y_rows_inverse<RC>), grid, block, lds, stream, yi, prefix, gx, nitems);
  if (kind == kPassZConv) {
    MVD_ANY_CLASS(cls & 3, MVD_Z)
  } else if (kind == kPassYForward) {
    MVD_ANY_CLASS(cls & 3, MVD_YF)
  } else if (kind == kPassYInverse) {
    MVD_ANY_CLASS(cls & 3, MVD_YI)
  } else {
    return hipErrorInvalidValue;
  }
#undef MVD_ROWS
#undef MVD_YF
#undef MVD_Z
#undef MVD_YI
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// energies of what an iteration transforms

__global__ __launch_bounds__(256) void k_rows_energy(const float* img, int nx, int nrows, int ex, int pieces, int per,
                                                     const float2* center, float2* part) {
  const int row0 = blockIdx.x * per, rows = min(per, nrows - row0);
  const float shift = center ? gmem(center)->y : 0.f;
  for (int c = threadIdx.x; c < pieces * 32; c += 256) {
    const int x = 2 * c - ex;
    const auto src = gmem(img) + (int64_t)row0 * nx;
    const int xa = min(max(x, 0), nx - 1), xb = min(max(x + 1, 0), nx - 1);
    float2 a = make_float2(0.f, 0.f), b = a;
#pragma unroll 4
    for (int r = 0; r < rows; ++r) {
      a = add_squares(a, src[(int64_t)r * nx + xa] - shift, shift);
      b = add_squares(b, src[(int64_t)r * nx + xb] - shift, shift);
    }
    const float2 s = energy_of_pair(a, b, x, nx);
    if ((threadIdx.x & 31) == 31) gmem(part)[(int64_t)blockIdx.x * pieces + (c >> 5)] = s;
  }
}

constexpr int kEnergyThreads = 256;

// Sums of a workgroup's threads, valid in all of them.
template <int N>
__device__ __forceinline__ void block_sums(double (&v)[N], double* lds) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __syncthreads();
    lds[threadIdx.x] = v[i];
    __syncthreads();
    for (int o = kEnergyThreads / 2; o > 0; o >>= 1) {
      if (threadIdx.x < o) lds[threadIdx.x] += lds[threadIdx.x + o];
      __syncthreads();
    }
    v[i] = lds[0];
  }
}

// A workgroup per convolution, region and slice of the region's planes.  A
// cell (one piece of one workgroup's rows) counts towards every region that it
// overlaps, and its energy as transformed towards the one that holds its first
// voxel.
__global__ __launch_bounds__(kEnergyThreads) void k_energy_sums(const EnergyItem* items) {
  __shared__ double lds[kEnergyThreads];
  const EnergyItem E = items[blockIdx.z];
  const int conv = blockIdx.y, at = blockIdx.x;
  if (conv >= E.convs || at >= E.regions * E.slices) return;  // uniform
  const int region = at / E.slices, slice = at - region * E.slices;
  const auto box = gmem(E.boxes) + region * 6;
  const int x0 = box[0], x1 = box[1], y0 = box[2], y1 = box[3], z0 = box[4], z1 = box[5];
  // workgroups that hold a row of planes [z0, z1), and pieces with a voxel of [x0, x1)
  const int w0 = (int)((int64_t)z0 * E.ny / E.per), w1 = (int)(((int64_t)z1 * E.ny - 1) / E.per) + 1;
  const int p0 = (x0 + E.ex) / kEnergyPiece, np = (x1 - 1 + E.ex) / kEnergyPiece + 1 - p0;
  const int lo = w0 + (int)((int64_t)(w1 - w0) * slice / E.slices);
  const int hi = w0 + (int)((int64_t)(w1 - w0) * (slice + 1) / E.slices);
  const auto part = gmem(E.part) + (int64_t)conv * E.nwg * E.pieces;
  double v[3] = {0.0, 0.0, 0.0};
#pragma unroll 2
  for (int i = threadIdx.x; i < (hi - lo) * np; i += kEnergyThreads) {
    const int w = lo + i / np, p = p0 + i % np;
    const float2 s = part[(int64_t)w * E.pieces + p];
    const int r0 = w * E.per, r1 = min(r0 + E.per, E.nrows) - 1;
    const int za = r0 / E.ny, ya = r0 - za * E.ny, zb = r1 / E.ny, yb = r1 - zb * E.ny;
    const bool in_a = za >= z0 && za < z1, in_b = zb >= z0 && zb < z1;
    const bool over = za == zb       ? in_a && ya < y1 && yb >= y0
                      : zb == za + 1 ? (in_a && ya < y1) || (in_b && yb >= y0)
                                     : za < z1 && zb >= z0;
    const int xa = max(p * kEnergyPiece - E.ex, 0), xb = min((p + 1) * kEnergyPiece - E.ex, E.nx);
    if (over) {
      v[0] += (double)s.x;
      v[1] += (double)((r1 - r0 + 1) * (xb - xa));
    }
    if (in_a && ya >= y0 && ya < y1 && xa >= x0) v[2] += (double)s.y;
  }
  block_sums(v, lds);
  if (threadIdx.x < 3)
    gmem(E.sums)[((int64_t)conv * E.regions * E.slices + at) * 3 + threadIdx.x] = v[threadIdx.x];
}

__global__ __launch_bounds__(kEnergyThreads) void k_energy_check(const EnergyItem* items) {
  __shared__ double lds[kEnergyThreads];
  const EnergyItem E = items[blockIdx.x];
  int refuse = 0;
  for (int c = 0; c < E.convs; ++c) {
    const auto sums = gmem(E.sums) + (int64_t)c * E.regions * E.slices * 3;
    double all[1] = {0.0};
    for (int i = threadIdx.x; i < E.regions * E.slices; i += kEnergyThreads) all[0] += sums[3 * i + 2];
    block_sums(all, lds);
    if (!(all[0] < INFINITY)) refuse = 1;  // (also where squares pass the largest float)
    const double mean = all[0] / ((double)E.nx * E.nrows);
    for (int r = threadIdx.x; E.limit > 0.0 && r < E.regions; r += kEnergyThreads) {
      double sq = 0.0, n = 0.0;
      for (int i = r * E.slices; i < (r + 1) * E.slices; ++i) {
        sq += sums[3 * i];
        n += sums[3 * i + 1];
      }
      if (!(mean * n < E.limit * sq)) refuse = 1;
    }
  }
  refuse = __syncthreads_or(refuse);
  if (threadIdx.x == 0) *gmem(E.refuse) = refuse;
}

hipError_t launch_rows_energy(const float* img, Int3 n, int ex, int pieces, int per, const float2* center,
                              float2* part, hipStream_t stream) {
  const int nrows = n.y * n.z;
  (void)hipGetLastError();
  hipLaunchKernelGGL(k_rows_energy, dim3((nrows + per - 1) / per), dim3(256), 0, stream, img, n.x, nrows, ex, pieces,
                     per, center, part);
  return hipGetLastError();
}

hipError_t launch_energy_check(const EnergyItem* items, int nitems, int max_convs, int max_sums, hipStream_t stream) {
  (void)hipGetLastError();
  hipLaunchKernelGGL(k_energy_sums, dim3(max_sums, max_convs, nitems), dim3(kEnergyThreads), 0, stream, items);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_energy_check, dim3(nitems), dim3(kEnergyThreads), 0, stream, items);
  return hipGetLastError();
}

}  // namespace mvd
