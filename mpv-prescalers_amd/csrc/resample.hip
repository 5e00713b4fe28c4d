// The scaler after a prescaler: resamples a prescaled plane to the display size and
// consumes the prescaler's OFFSET (mpv applies a hook's accumulated OFFSET in the next
// scaling pass, e.g. nnedi3-nns256-win8x6.hook:349-352 `//!OFFSET 0.000000 -0.500000`).
//
// Geometry: display pixel j (centre j + 1/2) sits at u = (j + 1/2) * in_w / out_w in the
// prescaled plane's continuous coordinate; the prescaled content is shifted by the
// offset, so the sample point is t = u + offset, and taps run over the texels whose
// centres lie within the filter radius of t (texel i has its centre at i + 1/2).  Weights
// are normalised to sum 1; reads are clamped to the plane (clamp-to-edge).
// Separable filters: bilinear (tent, r = 1), Catmull-Rom and Mitchell-Netravali cubics
// (r = 2), spline36 and Lanczos-3 (r = 3).  No widening when downscaling.
#include <math.h>

#include "common.h"
#include "launch.h"

namespace mpx {

__device__ __forceinline__ float filter_w(int filter, float x) {
  x = fabsf(x);
  switch (filter) {
    case 0: return fmaxf(0.f, 1.f - x);
    case 1:
    case 2: {  // cubic, (B, C) = (0, 1/2) Catmull-Rom, (1/3, 1/3) Mitchell
      const float B = filter == 1 ? 0.f : 1.f / 3.f, C = filter == 1 ? 0.5f : 1.f / 3.f;
      if (x < 1.f) return ((12.f - 9.f * B - 6.f * C) * x * x * x + (-18.f + 12.f * B + 6.f * C) * x * x + (6.f - 2.f * B)) / 6.f;
      if (x < 2.f)
        return ((-B - 6.f * C) * x * x * x + (6.f * B + 30.f * C) * x * x + (-12.f * B - 48.f * C) * x + (8.f * B + 24.f * C)) / 6.f;
      return 0.f;
    }
    case 3: {  // spline36
      if (x < 1.f) return ((13.f / 11.f * x - 453.f / 209.f) * x - 3.f / 209.f) * x + 1.f;
      if (x < 2.f) {
        x -= 1.f;
        return ((-6.f / 11.f * x + 270.f / 209.f) * x - 156.f / 209.f) * x;
      }
      if (x < 3.f) {
        x -= 2.f;
        return ((1.f / 11.f * x - 45.f / 209.f) * x + 26.f / 209.f) * x;
      }
      return 0.f;
    }
    default: {  // Lanczos-3: sinc(x) sinc(x/3)
      if (x >= 3.f) return 0.f;
      if (x < 1e-6f) return 1.f;
      const float px = 3.14159265358979f * x;
      return 3.f * sinf(px) * sinf(px / 3.f) / (px * px);
    }
  }
}

constexpr int kMaxTaps = 6;
constexpr int kResX = 64;        // output columns per block
constexpr int kResMaxY = 32;     // most output rows per block
constexpr int kResMaxRows = 96;  // most source rows a block keeps filtered in LDS (24 KB)

struct Taps {
  int base;
  float w[kMaxTaps];
};

// taps for display coordinate j along one axis
template <int R>
__device__ __forceinline__ Taps axis_taps(int filter, int j, int in_n, int out_n, float off) {
  const float t = (static_cast<float>(j) + 0.5f) * static_cast<float>(in_n) / static_cast<float>(out_n) + off;
  const float p = t - 0.5f;  // in texel-index units
  Taps r;
  const float fl = floorf(p);
  r.base = static_cast<int>(fl) - R + 1;
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < 2 * R; ++i) {
    r.w[i] = filter_w(filter, p - (fl - R + 1 + i));
    sum += r.w[i];
  }
  const float inv = 1.f / sum;
#pragma unroll
  for (int i = 0; i < 2 * R; ++i) r.w[i] *= inv;
  return r;
}

template <int DT> struct Elem;
template <> struct Elem<DT_U8> { typedef uint8_t T; };
template <> struct Elem<DT_U16> { typedef uint16_t T; };
template <> struct Elem<DT_F16> { typedef _Float16 T; };
template <> struct Elem<DT_F32> { typedef float T; };

template <int DT>
__device__ __forceinline__ float to_float(typename Elem<DT>::T v, float in_max, float in_rmax) {
  if constexpr (DT == DT_U8 || DT == DT_U16) return unorm_quotient(static_cast<float>(v), in_max, in_rmax);
  return static_cast<float>(v);
}

// One block per kResX x ty output tile (ty rows, 8 to kResMaxY), one column per lane.
// Each column's and each row's taps are computed once per tile into LDS; a thread keeps its
// column's taps in registers, filters the source rows the tile reads along x into LDS
// (`rows` of them, taken in turn by the four waves) and then filters the kept rows along y.
// Where the rows a tile reads do not fit in LDS, or overlap so little that keeping them saves
// nothing (strong downscaling), each output row filters its own 2R rows directly.  Both
// orders of work add the same products in the same order.
// A block that evaluated both axes' weights per output pixel and loaded (2R)^2 samples for it
// was bound by VALU issue (2160p -> 1440p FP16 Catmull-Rom: 73.9 us); with the weights per
// tile and the rows shared the same call takes 12.9 us, mostly the call itself.
template <int R, int DT>
__global__ __launch_bounds__(256) void resample_kernel(Io io, int out_w, int out_h, int planes, int filter,
                                                       float off_x, float off_y, int ty, int cap) {
  typedef typename Elem<DT>::T T;
  __shared__ Taps taps[kResX + kResMaxY];  // the tile's columns, then its rows
  extern __shared__ float kept[];  // cap rows of kResX filtered samples
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int x0 = blockIdx.x * kResX, y0 = blockIdx.y * ty;
  const int fc = blockIdx.z;  // frame * planes + plane
  const int f = fc / planes, c = fc - f * planes;
  const int ny = min(ty, out_h - y0);
  if (static_cast<int>(threadIdx.x) < kResX + ny) {
    const bool col = threadIdx.x < kResX;
    const int j = col ? min(x0 + lane, out_w - 1) : y0 + static_cast<int>(threadIdx.x) - kResX;
    taps[threadIdx.x] = axis_taps<R>(filter, j, col ? io.W : io.H, col ? out_w : out_h, col ? off_x : off_y);
  }
  __syncthreads();
  const Taps* ytap = taps + kResX;
  const int x = x0 + lane;
  const Taps tx = taps[lane];
  const T* in = reinterpret_cast<const T*>(static_cast<const char*>(frame_in(io, f)) +
                                           c * io.in_cstride * static_cast<int64_t>(sizeof(T)));
  // this column's 2R samples: contiguous, or clamped to the plane's edge columns
  int xo[2 * R];
#pragma unroll
  for (int i = 0; i < 2 * R; ++i) xo[i] = min(max(tx.base + i, 0), io.W - 1);
  const bool inner = __all(tx.base >= 0 && tx.base + 2 * R <= io.W);
  // source row yy filtered along x at this lane's column
  auto filter_row = [&](int yy) {
    const T* p = in + static_cast<int64_t>(min(max(yy, 0), io.H - 1)) * io.in_pitch;
    T v[2 * R];
    if (inner) {
      __builtin_memcpy(v, p + tx.base, sizeof(v));
    } else {
#pragma unroll
      for (int i = 0; i < 2 * R; ++i) v[i] = p[xo[i]];
    }
    float row = 0.f;
#pragma unroll
    for (int i = 0; i < 2 * R; ++i) row = fmaf(tx.w[i], to_float<DT>(v[i], io.in_max, io.in_rmax), row);
    return row;
  };
  const int r0 = ytap[0].base, rows = ytap[ny - 1].base - r0 + 2 * R;
  char* out = static_cast<char*>(frame_out(io, f)) + c * io.out_cstride * elem_bytes(io.out_dt);
  if (rows <= cap && rows < 2 * R * ny) {  // (uniform over the block)
#pragma unroll 4
    for (int i = wave; i < rows; i += 4) kept[i * kResX + lane] = filter_row(r0 + i);
    __syncthreads();
    if (x >= out_w) return;
    for (int j = wave; j < ny; j += 4) {
      const float* k = kept + (ytap[j].base - r0) * kResX + lane;
      float acc = 0.f;
#pragma unroll
      for (int i = 0; i < 2 * R; ++i) acc = fmaf(ytap[j].w[i], k[i * kResX], acc);
      store_elem(out, static_cast<int64_t>(y0 + j) * io.out_pitch + x, io.out_dt, acc);
    }
    return;
  }
  for (int j = wave; j < ny; j += 4) {
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < 2 * R; ++i) acc = fmaf(ytap[j].w[i], filter_row(ytap[j].base + i), acc);
    if (x < out_w) store_elem(out, static_cast<int64_t>(y0 + j) * io.out_pitch + x, io.out_dt, acc);
  }
}

template <int R>
static hipError_t launch_resample_r(const Io& io, int out_w, int out_h, int planes, int filter, float off_x,
                                    float off_y, hipStream_t st) {
  // Tall tiles share more filtered rows; small outputs take short ones so that every compute
  // unit has a few blocks.
  const int nx = (out_w + kResX - 1) / kResX;
  const int64_t nz = static_cast<int64_t>(io.batch) * planes;
  int ty = kResMaxY;
  while (ty > 8 && nx * nz * ((out_h + ty - 1) / ty) < 4 * device_cu_count()) ty /= 2;
  const double need = static_cast<double>(ty - 1) * io.H / out_h + 2 * R + 2;  // rows of a tile, at most
  const int cap = need <= kResMaxRows ? static_cast<int>(need) : 0;
  const dim3 grid(nx, (out_h + ty - 1) / ty, static_cast<unsigned>(nz));
  const size_t lds = static_cast<size_t>(cap) * kResX * sizeof(float);
#define MPX_RES(DT)                                                                                                  \
  case DT:                                                                                                           \
    hipLaunchKernelGGL((resample_kernel<R, DT>), grid, dim3(256), lds, st, io, out_w, out_h, planes, filter, off_x, \
                       off_y, ty, cap);                                                                              \
    break;
  switch (io.in_dt) {
    MPX_RES(DT_U8) MPX_RES(DT_U16) MPX_RES(DT_F16) MPX_RES(DT_F32)
    default: return hipErrorInvalidValue;
  }
#undef MPX_RES
  return hipGetLastError();
}

hipError_t launch_resample(const Io& io, int out_w, int out_h, int planes, int filter, float off_x, float off_y,
                           hipStream_t st) {
  if (filter == 0) return launch_resample_r<1>(io, out_w, out_h, planes, filter, off_x, off_y, st);
  if (filter <= 2) return launch_resample_r<2>(io, out_w, out_h, planes, filter, off_x, off_y, st);
  return launch_resample_r<3>(io, out_w, out_h, planes, filter, off_x, off_y, st);
}

}  // namespace mpx
