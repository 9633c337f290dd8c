// Input preparation on the GPU: one view resampled into the fused bounding box
// and its blending weight evaluated at the same position
// (deconv/TransformInputAndWeights.java:100-135, deconv/TransformInput.java:69-95,
//  spim/process/fusion/weights/BlendingRealRandomAccess.java:44-121).
//
// A wavefront takes 64 voxels along x or a tile of 16 x 4 (whichever reads fewer
// raw lines), four output rows per thread.  The arithmetic
// keeps the reference's types and order so that results are bit-identical to
// the CPU restatement: the inverse affine map in double, evaluated left to
// right without fused multiply-adds and rounded to float; trilinear weights in
// double; each corner term rounded to float and summed in float in the
// interpolator's corner order; blending distances in float and the lookup
// table in double.  The inputs are read through the texture-less vector path:
// the eight corners of neighbouring voxels overlap, so they hit L1/L2 and the
// HBM traffic is about one read of the raw view plus the two outputs.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/mvdecon.h"
#include "mvd_internal.h"

namespace mvd {

namespace {

constexpr int kTfThreads = 256;
constexpr float kMinValueF = 0.0001f;  // deconv/MVDeconvolution.java:70

// BlendingRealRandomAccess.java:47-53: d accumulated in double in steps of
// 0.001 while d <= 1.0001; entry round(d * 1000) = (cos((1 - d) pi) + 1) / 2.
std::vector<double> blend_lut_host() {
  std::vector<double> t(kBlendLutSize, 0.0);
  for (double d = 0; d <= 1.0001; d = d + 0.001) t[(int)std::floor(d * 1000.0 + 0.5)] = (std::cos((1 - d) * M_PI) + 1) / 2;
  return t;
}

std::mutex g_lut_mu;
std::vector<double*> g_lut;  // per device, held until the process ends

__device__ __forceinline__ float blend_weight(const float t[3], const int size[3], const float border[3],
                                              const float range[3], const double* __restrict__ lut) {
#pragma clang fp contract(off)
  float m = 1.f;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float l = t[d];
    const float a = l - border[d], b = (float)(size[d] - 1) - l - border[d];
    // Math.max(0, Math.min(a, b)), NaN propagating as in Java
    const float lo = a != a ? a : (b != b ? b : (a < b ? a : b));
    const float dist = (lo != lo || lo > 0.f) ? lo : 0.f;
    if (dist == 0.f) return 0.f;
    // dist >= range gives a rounded quotient >= 1 (no factor): the division
    // is only needed inside the blending band
    if (!(dist >= range[d])) {
      const float rel = __fdiv_rn(dist, range[d]);
      if (rel < 1.f) {
        const double x = (double)rel * 1000.0;
        m = (float)((double)m * gmem(lut)[(int)floor(x + 0.5)]);
      }
    }
  }
  return m;
}

// Two neighbouring values of a raw row, at any multiple of four bytes.
struct __attribute__((packed, aligned(4))) RawPair {
  float a, b;
};

// Trilinear interpolation over the mirror-single extension, for 0 <= t < size
// (the caller checks): the lower corner is in range and the upper one only
// leaves it at the far face, where the mirror maps n to n - 2 (n = 1: 0).
// The two corners of a row are one 8-byte load; at the far face it starts one
// voxel lower and its values change places (the mirror of n is n - 2).  The
// integer and fractional parts are taken in float: t >= 0, so both are exact.
// kOff32: the raw view spans fewer than 2^32 bytes, so corner addresses are
// 32-bit byte offsets from the (uniform) base.
struct Corners {
  RawPair q00, q10, q01, q11;  // rows (y0, z0), (y1, z0), (y0, z1), (y1, z1)
  bool far;                    // pairs that start one voxel lower
};

template <bool kOff32>
__device__ __forceinline__ Corners gather(const float* __restrict__ raw, const int size[3], const float t[3]) {
  Corners c;
  const int x0 = (int)t[0], y0 = (int)t[1], z0 = (int)t[2];
  const int y1 = y0 + 1 < size[1] ? y0 + 1 : (size[1] > 1 ? size[1] - 2 : 0);
  const int z1 = z0 + 1 < size[2] ? z0 + 1 : (size[2] > 1 ? size[2] - 2 : 0);
  const bool pairs = size[0] > 1;
  c.far = pairs && x0 + 1 == size[0];
  const int xb = c.far ? x0 - 1 : x0;
  if constexpr (kOff32) {
    const uint32_t sx = (uint32_t)size[0], sxy = (uint32_t)size[0] * (uint32_t)size[1];
    const uint32_t at = (uint32_t)xb * 4u;
    const uint32_t r00 = (y0 * sx + z0 * sxy) * 4u + at, r10 = (y1 * sx + z0 * sxy) * 4u + at;
    const uint32_t r01 = (y0 * sx + z1 * sxy) * 4u + at, r11 = (y1 * sx + z1 * sxy) * 4u + at;
    if (pairs) {
      c.q00 = *gbyte((const RawPair*)raw, r00);
      c.q10 = *gbyte((const RawPair*)raw, r10);
      c.q01 = *gbyte((const RawPair*)raw, r01);
      c.q11 = *gbyte((const RawPair*)raw, r11);
    } else {
      c.q00.a = c.q00.b = *gbyte(raw, r00);
      c.q10.a = c.q10.b = *gbyte(raw, r10);
      c.q01.a = c.q01.b = *gbyte(raw, r01);
      c.q11.a = c.q11.b = *gbyte(raw, r11);
    }
  } else {
    const int64_t sx = size[0], sxy = (int64_t)size[0] * size[1];
    const auto g = gmem(raw) + xb;
    const int64_t r00 = y0 * sx + z0 * sxy, r10 = y1 * sx + z0 * sxy;
    const int64_t r01 = y0 * sx + z1 * sxy, r11 = y1 * sx + z1 * sxy;
    const int n = pairs ? 1 : 0;
    c.q00 = {g[r00], g[r00 + n]};
    c.q10 = {g[r10], g[r10 + n]};
    c.q01 = {g[r01], g[r01 + n]};
    c.q11 = {g[r11], g[r11 + n]};
  }
  return c;
}

__device__ __forceinline__ float trilinear(Corners c, const float t[3]) {
#pragma clang fp contract(off)
  const double w0 = (double)(t[0] - floorf(t[0])), w0i = 1.0 - w0;
  const double w1 = (double)(t[1] - floorf(t[1])), w1i = 1.0 - w1;
  const double w2 = (double)(t[2] - floorf(t[2])), w2i = 1.0 - w2;
  // NLinearInterpolator3D weights: products in the order x, y, z
  const double a00 = w0i * w1i, a10 = w0 * w1i, a01 = w0i * w1, a11 = w0 * w1;
  const double w000 = a00 * w2i, w100 = a10 * w2i, w010 = a01 * w2i, w110 = a11 * w2i;
  const double w001 = a00 * w2, w101 = a10 * w2, w011 = a01 * w2, w111 = a11 * w2;
  if (c.far) {
    c.q00 = {c.q00.b, c.q00.a};
    c.q10 = {c.q10.b, c.q10.a};
    c.q01 = {c.q01.b, c.q01.a};
    c.q11 = {c.q11.b, c.q11.a};
  }
  const float v000 = c.q00.a, v100 = c.q00.b, v010 = c.q10.a, v110 = c.q10.b;
  const float v001 = c.q01.a, v101 = c.q01.b, v011 = c.q11.a, v111 = c.q11.b;
  // FloatType accumulation in the interpolator's corner order
  float acc = (float)((double)v000 * w000);
  acc = acc + (float)((double)v100 * w100);
  acc = acc + (float)((double)v110 * w110);
  acc = acc + (float)((double)v010 * w010);
  acc = acc + (float)((double)v011 * w011);
  acc = acc + (float)((double)v111 * w111);
  acc = acc + (float)((double)v101 * w101);
  acc = acc + (float)((double)v001 * w001);
  return acc;
}

// A wavefront covers LX x LY x LZ output voxels, a workgroup four of them along
// x, each thread kTfVox of them LY rows apart (same z), so the raw rows that
// neighbouring output rows share are fetched once into this CU's cache.
//
// A gather costs the cache one cycle per raw line that the wavefront's 64 voxels
// touch: 64 voxels along x of a view turned by 60 degrees lie in about 30 raw
// rows, 16 x 4 of them in 11.  512x512x256 with weights from 512x512x128 at 60
// degrees: 535 us with 64 voxels along x and eight 4-byte loads each (the L1 busy
// 93 % of the time), 435 us now.  What is left is arithmetic, 70 FP64 instructions
// a voxel; two or four rows in flight per thread (70 VGPRs) measured 430 to 445,
// eight or sixteen rows per thread 450 to 466.
constexpr int kTfVox = 4;

template <bool kOff32, int LX, int LY, int LZ>
__global__ __launch_bounds__(kTfThreads) void k_transform_view(TransformArgs a, int chunks, int ygroups) {
#pragma clang fp contract(off)
  static_assert(LX * LY * LZ == 64, "one wavefront");
  const int zy = blockIdx.x / chunks;  // z group * ygroups + y group
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int x = ((blockIdx.x - zy * chunks) * 4 + wave) * LX + lane % LX;
  const int zg = zy / ygroups, y0 = (zy - zg * ygroups) * (kTfVox * LY) + lane / LX % LY;
  const int z = zg * LZ + lane / (LX * LY);
  if (x >= a.nx || z >= a.nz) return;
  // cursor position (float) + offset (int): TransformInput.java:79-83;
  // AffineTransform3D.applyInverse: (float)(m0*s0 + m1*s1 + m2*s2 + m3), left
  // to right in double -- m0*s0 and m2*s2 are the column's terms
  const double s0 = (double)((float)x + a.off[0]), s2 = (double)((float)z + a.off[2]);
  double ra[3], rc[3];
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    ra[r] = a.inv[4 * r] * s0;
    rc[r] = a.inv[4 * r + 2] * s2;
  }
#pragma unroll 1
  for (int k = 0; k < kTfVox; ++k) {
    const int y = y0 + k * LY;
    if (y >= a.ny) break;
    const double s1 = (double)((float)y + a.off[1]);
    float t[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) t[r] = (float)(((ra[r] + a.inv[4 * r + 1] * s1) + rc[r]) + a.inv[4 * r + 3]);
    const int64_t o = ((int64_t)z * a.ny + y) * a.nx + x;
    // FusionHelper.intersects
    const bool in = a.out_img && t[0] >= 0.f && t[1] >= 0.f && t[2] >= 0.f && t[0] < a.rlim[0] && t[1] < a.rlim[1] &&
                    t[2] < a.rlim[2];
    Corners c;
    if (in) c = gather<kOff32>(a.raw, a.rsize, t);  // in flight under the weight's arithmetic
    if (a.out_w) gmem(a.out_w)[o] = blend_weight(t, a.rsize, a.border, a.range, a.lut);
    if (a.out_img) {
      float v = 0.f;  // outside the view: the reference's new image keeps 0
      if (in) {
        const float r = trilinear(c, t);
        v = r != r ? r : (r > kMinValueF ? r : kMinValueF);  // Math.max(minValue, r)
      }
      gmem(a.out_img)[o] = v;
    }
  }
}

}  // namespace

const double* blend_lut_device(int device) {
  std::lock_guard<std::mutex> lk(g_lut_mu);
  if ((int)g_lut.size() <= device) g_lut.resize(device + 1, nullptr);
  if (!g_lut[device]) {
    const auto t = blend_lut_host();
    double* p = nullptr;
    if (hipMalloc(&p, sizeof(double) * kBlendLutSize) != hipSuccess) return nullptr;
    if (hipMemcpy(p, t.data(), sizeof(double) * kBlendLutSize, hipMemcpyHostToDevice) != hipSuccess) {
      (void)hipFree(p);
      return nullptr;
    }
    g_lut[device] = p;
  }
  return g_lut[device];
}

const char* check_transform_args(const TransformArgs& a) {
  if (a.nx <= 0 || a.ny <= 0 || a.nz <= 0) return "output size must be positive";
  if ((int64_t)((a.ny + kTfVox - 1) / kTfVox) * a.nz * ((a.nx + kTfThreads - 1) / kTfThreads) >= (int64_t(1) << 31))
    return "output too large for one launch";
  if (!a.out_img && !a.out_w) return "no output requested";
  if (a.rsize[0] <= 0 || a.rsize[1] <= 0 || a.rsize[2] <= 0) return "raw view size must be positive";
  if (a.out_img && !a.raw) return "raw view missing";
  if ((int64_t)a.rsize[0] * a.rsize[1] * a.rsize[2] >= (int64_t(1) << 40)) return "raw view too large";
  if (a.out_w) {
    if (!a.lut) return "blending table missing";
    for (int d = 0; d < 3; ++d)
      if (!(a.range[d] > 0.f)) return "blending range must be positive";
  }
  for (int d = 0; d < 12; ++d)
    if (!std::isfinite(a.inv[d])) return "affine map must be finite";
  return nullptr;
}

namespace {

template <int LX, int LY, int LZ>
int64_t tile_wgs(const TransformArgs& a, int* chunks, int* ygroups) {
  *chunks = (a.nx + 4 * LX - 1) / (4 * LX);
  *ygroups = (a.ny + kTfVox * LY - 1) / (kTfVox * LY);
  return (int64_t)*chunks * *ygroups * ((a.nz + LZ - 1) / LZ);
}

// Lines that the wavefront's loads (four of raw pairs) and store touch: a row of
// voxels along x enters a new raw row with every step in the raw y and z, and
// the tile as a whole cannot touch more than its bounding box holds.
template <int LX, int LY, int LZ>
double tile_lines(const TransformArgs& a) {
  auto m = [&](int r, int c) { return std::fabs(a.inv[4 * r + c]); };
  double box = 1, path = 1;
  for (int r = 0; r < 3; ++r) {
    const double per_line = r == 0 ? 32.0 : 1.0;
    box *= 1 + ((LX - 1) * m(r, 0) + (LY - 1) * m(r, 1) + (LZ - 1) * m(r, 2)) / per_line;
    path += (LX - 1) * m(r, 0) / per_line;
  }
  return 4 * std::min({64.0, box, LY * LZ * path}) + LY * LZ * std::max(1.0, LX / 32.0);
}

template <int LX, int LY, int LZ>
void launch_tile(const TransformArgs& a, hipStream_t stream) {
  int chunks, ygroups;
  const int64_t wgs = tile_wgs<LX, LY, LZ>(a, &chunks, &ygroups);
  if ((int64_t)a.rsize[0] * a.rsize[1] * a.rsize[2] * 4 < (int64_t(1) << 32))
    hipLaunchKernelGGL((k_transform_view<true, LX, LY, LZ>), dim3((unsigned)wgs), dim3(kTfThreads), 0, stream, a,
                       chunks, ygroups);
  else
    hipLaunchKernelGGL((k_transform_view<false, LX, LY, LZ>), dim3((unsigned)wgs), dim3(kTfThreads), 0, stream, a,
                       chunks, ygroups);
}

}  // namespace

hipError_t launch_transform_view(const TransformArgs& args, hipStream_t stream) {
  TransformArgs a = args;
  for (int d = 0; d < 3; ++d) {  // the smallest float >= size: t < size for a float t
    a.rlim[d] = (float)a.rsize[d];
    if ((double)a.rlim[d] < (double)a.rsize[d]) a.rlim[d] = std::nextafterf(a.rlim[d], INFINITY);
  }
  // The tile of fewest lines, counting the work of lanes outside the output.
  // Rows also without an image (nothing is gathered), and where a step in x hardly
  // moves along the raw x: there the tile's planes, a power of two apart in many
  // views, compete for the same cache sets.  512x512x256 from 512x512x128, turned
  // about y, rows against 16 x 4: 0 degrees 375 and 390 us, 20 401 and 400, 60 456
  // and 435, 70 457 and 450, 80 455 and 468, 90 427 and 558; 500x490x250 from
  // 500x490x125: 20 439 and 375, 45 526 and 416, 60 500 and 433, 90 443 and 434.
  int c, g;
  const double rows = (double)tile_wgs<64, 1, 1>(a, &c, &g);
  double best = tile_lines<64, 1, 1>(a) * rows;
  int tile = 0;
  if (a.out_img && std::fabs(a.inv[0]) >= 0.2) {
    if (const double n = (double)tile_wgs<16, 1, 4>(a, &c, &g); n < 2147483648.0 && tile_lines<16, 1, 4>(a) * n < best)
      best = tile_lines<16, 1, 4>(a) * n, tile = 1;
    if (const double n = (double)tile_wgs<16, 4, 1>(a, &c, &g); n < 2147483648.0 && tile_lines<16, 4, 1>(a) * n < best)
      tile = 2;
  }
  (void)hipGetLastError();
  if (tile == 1)
    launch_tile<16, 1, 4>(a, stream);
  else if (tile == 2)
    launch_tile<16, 4, 1>(a, stream);
  else
    launch_tile<64, 1, 1>(a, stream);
  return hipGetLastError();
}

}  // namespace mvd

using namespace mvd;

extern "C" int mvd_transform_view(int device, const float* raw, int rx, int ry, int rz, const double* inverse_affine,
                                  const long long* offset, int nx, int ny, int nz, const float* border,
                                  const float* range, float* out_img, float* out_weight) {
  if (!inverse_affine || !offset) {
    set_error("NULL affine map or offset");
    return -1;
  }
  if ((border == nullptr) != (range == nullptr) || (out_weight && !border)) {
    set_error("weights need both border and range");
    return -1;
  }
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) {
    set_error("invalid device");
    return -1;
  }
  int prev = 0;
  (void)hipGetDevice(&prev);
  if (hipSetDevice(device) != hipSuccess) {
    set_error("hipSetDevice failed");
    return -2;
  }
  TransformArgs a{};
  a.rsize[0] = rx;
  a.rsize[1] = ry;
  a.rsize[2] = rz;
  for (int i = 0; i < 12; ++i) a.inv[i] = inverse_affine[i];
  for (int d = 0; d < 3; ++d) a.off[d] = (float)offset[d];
  a.nx = nx;
  a.ny = ny;
  a.nz = nz;
  if (border)
    for (int d = 0; d < 3; ++d) {
      a.border[d] = border[d];
      a.range[d] = range[d];
    }
  a.lut = out_weight ? blend_lut_device(device) : nullptr;
  const int64_t n = (int64_t)nx * ny * nz, nr = (int64_t)rx * ry * rz;
  float *d_raw = nullptr, *d_img = nullptr, *d_w = nullptr;
  int rc = 0;
  auto fail = [&](const std::string& m, int code) {
    set_error(m);
    rc = code;
  };
  a.raw = out_img ? raw : nullptr;
  a.out_img = out_img;
  a.out_w = out_weight;
  if (const char* msg = check_transform_args(a)) {
    fail(msg, -1);
  } else if (out_img && hipMalloc(&d_raw, sizeof(float) * nr) != hipSuccess) {
    fail("out of device memory (raw view)", -2);
  } else if (out_img && hipMalloc(&d_img, sizeof(float) * n) != hipSuccess) {
    fail("out of device memory (image)", -2);
  } else if (out_weight && hipMalloc(&d_w, sizeof(float) * n) != hipSuccess) {
    fail("out of device memory (weight)", -2);
  } else if (out_img && staged_h2d(d_raw, raw, sizeof(float) * nr, nullptr) != hipSuccess) {
    fail("copy of the raw view failed", -2);
  } else {
    a.raw = d_raw;
    a.out_img = d_img;
    a.out_w = d_w;
    hipError_t e = launch_transform_view(a, nullptr);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e == hipSuccess && out_img) e = staged_d2h(out_img, d_img, sizeof(float) * n, nullptr);
    if (e == hipSuccess && out_weight) e = staged_d2h(out_weight, d_w, sizeof(float) * n, nullptr);
    if (e != hipSuccess) fail(std::string("transform failed: ") + hipGetErrorString(e), -2);
  }
  if (d_raw) (void)hipFree(d_raw);
  if (d_img) (void)hipFree(d_img);
  if (d_w) (void)hipFree(d_w);
  (void)hipSetDevice(prev);
  return rc;
}

extern "C" int mvd_transform_view_device(int device, const float* raw, int rx, int ry, int rz,
                                         const double* inverse_affine, const long long* offset, int nx, int ny,
                                         int nz, const float* border, const float* range, float* out_img,
                                         float* out_weight, void* stream) {
  if (!inverse_affine || !offset) {
    set_error("NULL affine map or offset");
    return -1;
  }
  if ((border == nullptr) != (range == nullptr) || (out_weight && !border)) {
    set_error("weights need both border and range");
    return -1;
  }
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) {
    set_error("invalid device");
    return -1;
  }
  int prev = 0;
  (void)hipGetDevice(&prev);
  if (hipSetDevice(device) != hipSuccess) {
    set_error("hipSetDevice failed");
    return -2;
  }
  TransformArgs a{};
  a.raw = raw;
  a.rsize[0] = rx;
  a.rsize[1] = ry;
  a.rsize[2] = rz;
  for (int i = 0; i < 12; ++i) a.inv[i] = inverse_affine[i];
  for (int d = 0; d < 3; ++d) a.off[d] = (float)offset[d];
  a.nx = nx;
  a.ny = ny;
  a.nz = nz;
  if (border)
    for (int d = 0; d < 3; ++d) {
      a.border[d] = border[d];
      a.range[d] = range[d];
    }
  a.out_img = out_img;
  a.out_w = out_weight;
  a.lut = out_weight ? blend_lut_device(device) : nullptr;
  int rc = 0;
  if (const char* msg = check_transform_args(a)) {
    set_error(msg);
    rc = -1;
  } else {
    const hipError_t e = launch_transform_view(a, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) {
      set_error(std::string("transform launch failed: ") + hipGetErrorString(e));
      rc = -2;
    }
  }
  (void)hipSetDevice(prev);
  return rc;
}
