// Shared device code for the RAVU family: element I/O, the structure tensor, the
// eigen-analysis hash with its FP64 re-decision near bucket boundaries.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gauss_tables.h"

namespace mpx {

enum DType : int { DT_U8 = 0, DT_U16 = 1, DT_F16 = 2, DT_F32 = 3 };

constexpr int kMaxTab = 16;  // frames per launch through a pointer table

// Device-side description of one launch's planes (strides in elements).  Frames are
// either `bstride` apart from `in` / `out`, or (ntab > 0) at the addresses of the
// pointer tables, which travel by value in the kernel arguments.
struct Io {
  const void* in;
  void* out;
  const void* tab_in[kMaxTab];
  void* tab_out[kMaxTab];
  int ntab;
  int64_t in_pitch, in_cstride, in_bstride;
  int64_t out_pitch, out_cstride, out_bstride;
  int32_t* buckets;   // optional, [batch][sites] rows
  int64_t bucket_bstride;
  int in_dt, out_dt;
  float in_max;       // integer full-scale value for U8/U16 inputs (255, 1023, ...)
  float in_rmax;      // RN(1 / in_max), computed on the host
  int W, H;           // input plane size
  int batch;
  // Frames of different sizes in one launch (sized != 0; ntab frames through the pointer
  // tables): each frame's input size and row pitches, planes contiguous.  `tiles` is the
  // prefix sum of the launch's tiles per frame, filled by the launcher for its tile shape.
  int sized;
  int fw[kMaxTab], fh[kMaxTab];
  int64_t fin_pitch[kMaxTab], fout_pitch[kMaxTab];
  int tiles[kMaxTab + 1];
  int sx, sy;         // output scale of the launch (for the output plane stride)
  // intermediates (NNEDI3's double_y plane, RAVU's int11) rounded to FP16 as mpv's
  // default rgba16f FBOs store them (MPX_STORE_FP16)
  int store16;
};

// One tile of a launch: its frame, origin and that frame's geometry.
struct FrameTile {
  int f, x0, y0;
  int W, H;
  int64_t in_pitch, out_pitch, in_cstride, out_cstride;
};

__device__ __host__ __forceinline__ int elem_bytes(int dt) { return dt == DT_F32 ? 4 : (dt == DT_U8 ? 1 : 2); }

__device__ __forceinline__ const void* frame_in(const Io& io, int f) {
  if (io.ntab) return io.tab_in[f];
  return static_cast<const char*>(io.in) + static_cast<int64_t>(f) * io.in_bstride * elem_bytes(io.in_dt);
}
__device__ __forceinline__ void* frame_out(const Io& io, int f) {
  if (io.ntab) return io.tab_out[f];
  return static_cast<char*>(io.out) + static_cast<int64_t>(f) * io.out_bstride * elem_bytes(io.out_dt);
}

// Each of the 8 XCDs (own L2 each) takes thread blocks round-robin in launch order.
// xcd_tile maps launch-order block L of T to a tile so that every XCD walks one contiguous
// range of tiles: neighbouring tiles, which share halo rows, then meet in the same L2.
// A bijection on [0, T) for any T.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_tile(int L, int T) {
  const int q = T / kXcds, r = T % kXcds;
  const int x = L % kXcds, j = L / kXcds;
  return x * q + min(x, r) + j;
}

// Tile (x, y) and frame z of this block in a 1-D launch of nx * ny * nz blocks.
struct BlockXYZ {
  int x, y, z;
};
__device__ __forceinline__ BlockXYZ block_xyz(int nx, int ny, int nz) {
  const int per = nx * ny;
  const int t = xcd_tile(static_cast<int>(blockIdx.x), per * nz);
  const int z = t / per, r = t - z * per;
  return {r % nx, r / nx, z};
}

// The TX x TY input tile of block L (launch order, XCD-aware) among `total` tiles.
template <int TX, int TY>
__device__ __forceinline__ FrameTile frame_tile(const Io& io, int L, int total) {
  const int t = xcd_tile(L, total);
  FrameTile ft;
  if (!io.sized) {
    const int nx = (io.W + TX - 1) / TX, per = nx * ((io.H + TY - 1) / TY);
    ft.f = t / per;
    const int r = t - ft.f * per;
    ft.x0 = (r % nx) * TX;
    ft.y0 = (r / nx) * TY;
    ft.W = io.W;
    ft.H = io.H;
    ft.in_pitch = io.in_pitch;
    ft.out_pitch = io.out_pitch;
    ft.in_cstride = io.in_cstride;
    ft.out_cstride = io.out_cstride;
    return ft;
  }
  int f = 0;
  while (f + 1 < io.ntab && t >= io.tiles[f + 1]) ++f;
  const int r = t - io.tiles[f];
  const int nx = (io.fw[f] + TX - 1) / TX;
  ft.f = f;
  ft.x0 = (r % nx) * TX;
  ft.y0 = (r / nx) * TY;
  ft.W = io.fw[f];
  ft.H = io.fh[f];
  ft.in_pitch = io.fin_pitch[f];
  ft.out_pitch = io.fout_pitch[f];
  ft.in_cstride = io.fin_pitch[f] * io.fh[f];
  ft.out_cstride = io.fout_pitch[f] * io.fh[f] * io.sy;
  return ft;
}

// Host: tiles of a launch for a TX x TY tile (fills the per-frame prefix of sized launches).
template <int TX, int TY>
inline int launch_tiles(Io& io) {
  if (!io.sized) return ((io.W + TX - 1) / TX) * ((io.H + TY - 1) / TY) * io.batch;
  io.tiles[0] = 0;
  for (int f = 0; f < io.ntab; ++f)
    io.tiles[f + 1] = io.tiles[f] + ((io.fw[f] + TX - 1) / TX) * ((io.fh[f] + TY - 1) / TY);
  return io.tiles[io.ntab];
}

// v / m for an integer sample v (0..65535) and full scale m = 2^bits - 1, rounded exactly
// as the division rounds, given rm = RN(1/m): q0 = v * rm lies within one ulp of v/m, the
// residual v - m*q0 is exact under fma, and one corrected step gives RN(v/m) (Markstein's
// theorem).  Three operations instead of the division's ten; equal to the division for
// every 16-bit v and every bits 1..16 (checked exhaustively).
__device__ __forceinline__ float unorm_quotient(float v, float m, float rm) {
  const float q0 = v * rm;
  return fmaf(fmaf(-q0, m, v), rm, q0);
}

__device__ __forceinline__ float load_elem(const void* p, int64_t idx, int dt, float in_max) {
  switch (dt) {
    case DT_F32: return static_cast<const float*>(p)[idx];
    case DT_F16: return __half2float(static_cast<const __half*>(p)[idx]);
    case DT_U8: return static_cast<float>(static_cast<const uint8_t*>(p)[idx]) / in_max;
    default: return static_cast<float>(static_cast<const uint16_t*>(p)[idx]) / in_max;
  }
}

// Halo tile of P planes, PH x PW samples each (PW a multiple of 4), taken at (ox + col,
// oy + r) clamped to the W x H plane (clamp-to-edge sampling) and staged to LDS as
// tile[c][r][col], by NT threads.  A thread takes items of V = 4 neighbouring samples of a
// row (2 where items of four would leave half the threads idle and the block waiting for the
// others): `issue` starts one load per item (V samples at the samples' own alignment),
// moved inwards where the item reaches past the plane's left or right edge; `commit` converts
// the samples, repeats the edge ones in such items (tiles at a side edge only) and writes each
// item to LDS at once.  A tile therefore costs one memory latency, and a persistent block
// can issue its next tile while it computes this one.  Loads cover exactly V samples of the
// plane's row: nothing outside the frame is read (planes under V samples wide: sample by
// sample).
// Bound by VALU issue: one address and one LDS write per sample took about 19 instructions
// per sample, 8-17 % of a kernel.  Measured with items: ravu-r4-yuv 2 x 1080p 254.0 -> 240.8
// us, r3 1366x768 38.1 -> 37.3, nnedi3 nns32 1080p 94.4 -> 93.0 (fewer registers held for
// the next tile: 123 -> 96 VGPRs, five waves per SIMD), lite and 3x (small tiles) unchanged.
// Sample addresses are 32-bit element offsets from the frame (plane c * cstride + row *
// pitch + column, the row term a 24-bit multiply): the host refuses frames that span 2^32
// elements or more, or whose pitch reaches 2^24 elements (kMaxSpan, kMaxPitch).
// Pointers into global memory (address space 1): loads through them are global loads, never
// flat ones (which would also count against the LDS wait counter).
#define MPX_GLOBAL __attribute__((address_space(1)))
typedef const MPX_GLOBAL uint32_t* GlobalU32;

template <int P, int PH, int PW, int NT>
struct HaloTile {
  static_assert(PW % 4 == 0, "rows are staged in whole items");
  static constexpr int V = P * PH * PW / 4 * 2 <= NT ? 2 : 4;  // samples per item
  static constexpr int Q = PW / V;       // items per row
  static constexpr int N = P * PH * Q;   // items of the tile
  static constexpr int E = (N + NT - 1) / NT;
  typedef uint32_t Raw __attribute__((ext_vector_type(V)));  // V dwords, or V samples packed into the first ones
  typedef float Val __attribute__((ext_vector_type(V)));
  Raw v[E];

  // samples col .. col + V - 1 of the row at p (LSH: log2 element bytes); W < V: 0 .. W - 1, the last repeated
  template <int LSH>
  __device__ __forceinline__ static Raw load(uintptr_t p, int col, int W) {
    constexpr int D = (V << LSH) / 4;  // dwords of an item (0: two bytes)
    typedef uint32_t Dwords __attribute__((ext_vector_type(D > 1 ? D : 2)));
    typedef Dwords DwordsA __attribute__((aligned(1 << LSH)));
    typedef uint32_t DwordA __attribute__((aligned(1)));
    typedef uint16_t HalfA __attribute__((aligned(1)));
    Raw w;
#pragma unroll
    for (int k = 0; k < V; ++k) w[k] = 0;
    if (W >= V) {
      const uintptr_t a = p + (static_cast<uintptr_t>(static_cast<uint32_t>(col)) << LSH);
      if constexpr (D > 1) {
        const Dwords x = *reinterpret_cast<const MPX_GLOBAL DwordsA*>(a);
#pragma unroll
        for (int k = 0; k < D; ++k) w[k] = x[k];
      } else if constexpr (D == 1) {
        w[0] = *reinterpret_cast<const MPX_GLOBAL DwordA*>(a);
      } else {
        w[0] = *reinterpret_cast<const MPX_GLOBAL HalfA*>(a);
      }
      return w;
    }
#pragma unroll
    for (int k = 0; k < V; ++k) {
      const uintptr_t a = p + (static_cast<uintptr_t>(static_cast<uint32_t>(min(k, W - 1))) << LSH);
      if constexpr (LSH == 2) w[k] = *reinterpret_cast<GlobalU32>(a);
      else if constexpr (LSH == 1) w[k / 2] |= static_cast<uint32_t>(*reinterpret_cast<const MPX_GLOBAL uint16_t*>(a)) << (16 * (k % 2));
      else w[0] |= static_cast<uint32_t>(*reinterpret_cast<const MPX_GLOBAL uint8_t*>(a)) << (8 * k);
    }
    return w;
  }

  // first sample of the load of the item at column col: its own, moved into the row
  __device__ __forceinline__ static int load_col(int col, int W) { return max(min(col, W - V), 0); }

  template <int LSH>
  __device__ __forceinline__ void issue_as(const void* base, int64_t pitch, int64_t cstride, int W, int H, int ox,
                                           int oy) {
    const uintptr_t b = reinterpret_cast<uintptr_t>(base);
    const uint32_t ps = static_cast<uint32_t>(pitch), cs = static_cast<uint32_t>(cstride);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = min(static_cast<int>(threadIdx.x) + e * NT, N - 1);  // tail lanes repeat the last item
      const int c = P == 1 ? 0 : i / (PH * Q);
      const int j = i - c * (PH * Q);
      const int r = j / Q, col = ox + V * (j - r * Q);
      const int gy = min(max(oy + r, 0), H - 1);
      const uint32_t off = static_cast<uint32_t>(c) * cs + __umul24(static_cast<uint32_t>(gy), ps);
      v[e] = load<LSH>(b + (static_cast<uintptr_t>(off) << LSH), load_col(col, W), W);
    }
  }

  __device__ __forceinline__ void issue(const void* base, int dt, int64_t pitch, int64_t cstride, int W, int H,
                                        int ox, int oy) {
    if (dt == DT_F32) issue_as<2>(base, pitch, cstride, W, H, ox, oy);
    else if (dt == DT_U8) issue_as<0>(base, pitch, cstride, W, H, ox, oy);
    else issue_as<1>(base, pitch, cstride, W, H, ox, oy);
  }

  // in_rmax = RN(1 / in_max) (from the host): integer samples cost three operations each
  __device__ __forceinline__ static Val convert(Raw w, int dt, float in_max, float in_rmax) {
    Val f;
    switch (dt) {
      case DT_F32:
#pragma unroll
        for (int k = 0; k < V; ++k) f[k] = __uint_as_float(w[k]);
        break;
      case DT_F16:
#pragma unroll
        for (int k = 0; k < V; ++k)
          f[k] = __half2float(__ushort_as_half(static_cast<unsigned short>(w[k / 2] >> (16 * (k % 2)))));
        break;
      case DT_U8:
#pragma unroll
        for (int k = 0; k < V; ++k) f[k] = unorm_quotient(static_cast<float>((w[0] >> (8 * k)) & 0xffu), in_max, in_rmax);
        break;
      default:
#pragma unroll
        for (int k = 0; k < V; ++k)
          f[k] = unorm_quotient(static_cast<float>((w[k / 2] >> (16 * (k % 2))) & 0xffffu), in_max, in_rmax);
        break;
    }
    return f;
  }

  // `tile`: 16-byte aligned, P * PH * PW floats; W, ox as issued; `each(i, f)` sees item i's values
  template <typename Each>
  __device__ __forceinline__ void commit(float* tile, int dt, float in_max, float in_rmax, int W, int ox,
                                         Each each) const {
    const bool whole = ox >= 0 && ox + PW <= W;  // (uniform) every item lies inside its row
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = static_cast<int>(threadIdx.x) + e * NT;
      if (E * NT == N || i < N) {
        Val f = convert(v[e], dt, in_max, in_rmax);
        if (!whole) {
          // sample k wanted sits at position k + d of the loaded ones, clamped: the edge sample repeats
          const int col = ox + V * (i % Q), d = col - load_col(col, W);
          const Val g = f;
#pragma unroll
          for (int k = 0; k < V; ++k) {
            f[k] = g[V - 1];
#pragma unroll
            for (int j = V - 2; j >= 0; --j) f[k] = d <= j - k ? g[j] : f[k];
          }
        }
        reinterpret_cast<Val*>(tile)[i] = f;
        each(i, f);
      }
    }
  }
  __device__ __forceinline__ void commit(float* tile, int dt, float in_max, float in_rmax, int W, int ox) const {
    commit(tile, dt, in_max, in_rmax, W, ox, [](int, const Val&) {});
  }
};

// Row length of a staged tile: n samples, rounded up to whole items.
constexpr int staged_width(int n) { return (n + 3) / 4 * 4; }

__device__ __forceinline__ void store_elem(void* p, int64_t idx, int dt, float v) {
  if (dt == DT_F32)
    static_cast<float*>(p)[idx] = v;
  else
    static_cast<__half*>(p)[idx] = __float2half_rn(v);
}

// Two horizontally adjacent outputs (idx even-aligned by construction of the callers).
__device__ __forceinline__ void store_pair(void* p, int64_t idx, int dt, float v0, float v1) {
  if (dt == DT_F32) {
    float* q = static_cast<float*>(p) + idx;
    q[0] = v0;
    q[1] = v1;
  } else {
    __half* q = static_cast<__half*>(p) + idx;
    q[0] = __float2half_rn(v0);
    q[1] = __float2half_rn(v1);
  }
}

// two FP16 values packed in one dword (low half first)
__device__ __forceinline__ __half2 bits_h2(uint32_t v) {
  __half2 h;
  __builtin_memcpy(&h, &v, sizeof(h));
  return h;
}

__device__ __forceinline__ float4 load_lut4(const __half* lut, int64_t texel) {
  const __half2* p = reinterpret_cast<const __half2*>(lut + 4 * texel);
  float2 lo = __half22float2(p[0]);
  float2 hi = __half22float2(p[1]);
  return make_float4(lo.x, lo.y, hi.x, hi.y);
}

template <int N>
__device__ __host__ constexpr double gauss_w(int i) {
  return N == 3 ? kGauss3[i] : N == 4 ? kGauss4[i] : N == 5 ? kGauss5[i]
       : N == 6 ? kGauss6[i] : N == 7 ? kGauss7[i] : kGauss8[i];
}

// x / b for a constant b, rounded exactly as the division rounds (to nearest), given
// rb = RN(1/b).  FP64 takes three operations instead of the division's eleven (one of
// them a quarter-rate reciprocal): q0 = x * rb lies within one ulp of x/b, the residual
// x - b*q0 is exact under fma, and one corrected step gives RN(x/b) (Markstein's theorem;
// the operands here are far from underflow and overflow).  A zero quotient may come out
// +0 where the division gives -0, which no caller can tell apart (squares and sums).
template <typename T>
__device__ __forceinline__ T div_const(T x, T b, T rb) {
  if constexpr (sizeof(T) == 8) {
    const T q0 = x * rb;
    return __builtin_fma(__builtin_fma(-q0, b, x), rb, q0);
  }
  return x / b;
}

// Derivative along one window line at position p, in the shaders' formula forms
// (ravu-lite-r3.hook:50 central; ravu-r3.hook:64 five-point; ravu-zoom-r2.hook:50
// forward/backward at the window border), in FP64 (the re-decision): the correctly rounded
// quotients, as the oracle's divisions give.  `s(k)` returns the line's k-th sample.
template <int N, bool FIVE, typename Line>
__device__ __forceinline__ double deriv(Line s, int p) {
#pragma clang fp contract(off)
  if (p == 0) return s(1) - s(0);
  if (p == N - 1) return s(N - 1) - s(N - 2);
  if (FIVE && p >= 2 && p + 2 <= N - 1) {
    const double num = -s(p + 2) + 8.0 * s(p + 1) - 8.0 * s(p - 1) + s(p - 2);
    return div_const(num, 12.0, 1.0 / 12.0);
  }
  return (s(p + 1) - s(p - 1)) / 2.0;
}

// The derivatives of the FP32 fast path without their stencil's scale, and that scale: 1 at
// the window border (forward/backward), 1/12 for the five-point form, 1/2 central.
template <int N, bool FIVE>
__device__ __host__ constexpr double deriv_scale(int p) {
  return (p == 0 || p == N - 1) ? 1.0 : (FIVE && p >= 2 && p + 2 <= N - 1) ? 1.0 / 12.0 : 0.5;
}
// The sample that a hash sees: plane 0's, or for rgb (CH = 2) the BT.709 luma in FP64.  A luma
// rounded to FP32 first would be off by 1e-7, in faint detail 1e-5 to 1e-3 of the derivative and
// outside every margin of hash_fast; the difference of FP64 lumas, rounded once, is as good as
// that of two FP32 samples.
// Bound by VALU issue: an FP64 difference and its conversion take the time of four FP32
// instructions (ordinary frames, FP32 luma -> FP64: r2-rgb 2 x 1080p 115 -> 129 us, r3-rgb 142 -> 155,
// r4-rgb 214 -> 231, zoom-ar-r2-rgb 720p -> 1440p 57.4 -> 56.0), while a re-decision reads one
// sample instead of three and no longer computes their luma (45-degree stripes 1280x720: r4-rgb
// 386 -> 116, r3-rgb 159 -> 74, zoom-r3-rgb at 1.5x 142 -> 58; large flat shapes: r4-rgb 145 -> 100).
template <int CH> struct HashSampleOf { typedef float T; };
template <> struct HashSampleOf<2> { typedef double T; };
template <int CH>
using HashSample = typename HashSampleOf<CH>::T;
// (the oracle's operations in its order)
__device__ __forceinline__ double luma709(float r, float g, float b) {
#pragma clang fp contract(off)
  return 0.2126 * static_cast<double>(r) + 0.7152 * static_cast<double>(g) + 0.0722 * static_cast<double>(b);
}
// Lumas of `count` staged samples (rounded up to pairs; n samples per plane, even; both arrays 16-byte
// aligned) by the block's NT threads.
template <int NT>
__device__ __forceinline__ void fill_luma(const float* t, double* luma, int n, int count) {
  const float2* s = reinterpret_cast<const float2*>(t);
  for (int i = threadIdx.x; 2 * i < count; i += NT) {
    const float2 r = s[i], g = s[n / 2 + i], b = s[n + i];
    reinterpret_cast<double2*>(luma)[i] = make_double2(luma709(r.x, g.x, b.x), luma709(r.y, g.y, b.y));
  }
}

__device__ __forceinline__ float difference(float a, float b) { return a - b; }
__device__ __forceinline__ float difference(double a, double b) { return static_cast<float>(a - b); }
template <int N, bool FIVE, typename Line>
__device__ __forceinline__ float deriv_unscaled(Line s, int p) {
#pragma clang fp contract(off)
  if (p == 0) return difference(s(1), s(0));
  if (p == N - 1) return difference(s(N - 1), s(N - 2));
  if (FIVE && p >= 2 && p + 2 <= N - 1)
    return fmaf(8.0f, difference(s(p + 1), s(p - 1)), difference(s(p - 2), s(p + 2)));
  return difference(s(p + 1), s(p - 1));
}

// Gradient grid of an N x N window: positions P0 .. P1 - 1 on both axes.
template <int N>
struct GradGrid {
  static constexpr int P0 = N <= 4 ? 0 : 1;
  static constexpr int P1 = N <= 4 ? N : N - 1;
  static constexpr int M = P1 - P0;
};

// abd = sum over the gradient grid of (gx*gx, gx*gy, gy*gy) * G, grid X outer, Y inner
// (ravu-lite-r3.hook:48-76), FP32 fast path, trusted only away from bucket boundaries.  get(i)
// returns window sample i = X*N + Y.  The derivatives are taken unscaled and each point's
// stencil scales folded into its Gaussian weight (compile-time constants); where gx and gy
// carry the same scale one product w'*gx serves both a and b (lite-r3 8 x 1080p 132.4 ->
// 128.4 us, zoom-r2 4 x 720p -> 1440p 117.1 -> 113.3).
// FP64 samples of a 4 x 4 window (32 derivatives of 16 samples) are first rounded relative to an
// inner one: with border derivatives in the grid no sample is far from it, and the rounding is
// at most 6.6 u of the tensor's norm, where larger windows' may be any multiple.
template <int N, bool FIVE, typename Get>
__device__ __forceinline__ void structure_tensor(Get get, float& a, float& b, float& d) {
#pragma clang fp contract(off)
  using GG = GradGrid<N>;
  if constexpr (N == 4 && sizeof(get(0)) == 8) {
    const double c = get(N + 1);
    return structure_tensor<N, FIVE>([&](int i) { return static_cast<float>(get(i) - c); }, a, b, d);
  }
  a = b = d = 0.f;
#pragma unroll
  for (int X = GG::P0; X < GG::P1; ++X) {
    // FP64 samples: one column of points at a time (7 x 7 windows one point: 100 -> 62 VGPRs, and
    // 3x-r4-rgb 1280x720 48.6 -> 47.4 us; at 6 x 6 that took zoom-r3-rgb at 1.25x from 29.5 to 34.1)
    if constexpr (sizeof(get(0)) == 8) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int Y = GG::P0; Y < GG::P1; ++Y) {
      if constexpr (sizeof(get(0)) == 8 && N == 7) __builtin_amdgcn_sched_barrier(0);
      const float gx = deriv_unscaled<N, FIVE>([&](int k) { return get(k * N + Y); }, X);
      const float gy = deriv_unscaled<N, FIVE>([&](int k) { return get(X * N + k); }, Y);
      const double cx = deriv_scale<N, FIVE>(X), cy = deriv_scale<N, FIVE>(Y);
      const double w = gauss_w<N>((X - GG::P0) * GG::M + (Y - GG::P0));
      const float u = gx * static_cast<float>(w * cx * cx);
      a = fmaf(u, gx, a);
      b = cx == cy ? fmaf(u, gy, b) : fmaf(gx * static_cast<float>(w * cx * cy), gy, b);
      d = fmaf(gy * static_cast<float>(w * cy * cy), gy, d);
    }
  }
}

// The same in FP64, in the reference's rounding steps and order, by one lane; get(i) returns the
// sample as it is stored.  LEAN (large windows): a column of points at a time, or one point for 8 x 8
// windows and FP64 samples (scheduling barriers, the partial sums pinned), so the rare re-decision
// does not hold the window in FP64 registers and set every wave's occupancy.
// Bound by the latency of its LDS reads: with one derivative at a time large flat shapes 1280x720 took
// r3 46.3 us, now 44.0, r3-yuv 58.9 -> 55.7, r4-yuv line grid 148 -> 137.  (r4 by columns: 38.2 -> 39.1 on
// ordinary frames, five waves per SIMD instead of six; zoom-r3-rgb at 1.5x 36.4 -> 37.4.)
template <int N, bool FIVE, bool LEAN, typename Get>
__device__ __forceinline__ void structure_tensor_fp64(Get get, double& a, double& b, double& d) {
#pragma clang fp contract(off)
  using GG = GradGrid<N>;
  constexpr bool POINTS = N == 8 || sizeof(get(0)) == 8;
  auto sample = [&](int i) { return static_cast<double>(get(i)); };
  a = b = d = 0.0;
#pragma unroll
  for (int X = GG::P0; X < GG::P1; ++X) {
#pragma unroll
    for (int Y = GG::P0; Y < GG::P1; ++Y) {
      const double gx = deriv<N, FIVE>([&](int k) { return sample(k * N + Y); }, X);
      const double gy = deriv<N, FIVE>([&](int k) { return sample(X * N + k); }, Y);
      const double w = gauss_w<N>((X - GG::P0) * GG::M + (Y - GG::P0));
      a = a + gx * gx * w;
      b = b + gx * gy * w;
      d = d + gy * gy * w;
      if constexpr (LEAN) {
        if (POINTS || Y == GG::P1 - 1) {
          asm volatile("" : "+v"(a), "+v"(b), "+v"(d));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
}

enum Rule : int { RULE_LITE = 0, RULE_3X = 1, RULE_LOG2 = 2 };

template <int RULE> struct RuleInfo;
template <> struct RuleInfo<RULE_LITE> { static constexpr int S = 4; };   // ravu-lite-r3.hook:86,88
template <> struct RuleInfo<RULE_3X> { static constexpr int S = 3; };     // compute/ravu-3x-r3.hook:95,97
template <> struct RuleInfo<RULE_LOG2> { static constexpr int S = 9; };   // ravu-r3.hook:117,119

struct Bucket {
  int angle, strength, coherence;
};

constexpr float kEps = 1.192092896e-7f;
constexpr double kEpsD = 1.192092896e-7;
constexpr double kPiD = 3.141592653589793;
constexpr float kPiF = 3.141592653589793f;

template <int RULE, typename T>
__device__ __forceinline__ int strength_of(T lambda) {
  if (RULE == RULE_LITE)  // ravu-lite-r3.hook:86
    return lambda >= T(0.016) ? (lambda >= T(0.05) ? 3 : 2) : (lambda >= T(0.004) ? 1 : 0);
  if (RULE == RULE_3X)    // compute/ravu-3x-r3.hook:95
    return lambda >= T(0.02) ? 2 : (lambda >= T(0.005) ? 1 : 0);
  // ravu-r3.hook:117: clamp(floor(log2(lambda*2000 + eps)), 0, 8)
  T f = floor(log2(lambda * T(2000) + T(1.192092896e-7)));
  return static_cast<int>(fmin(fmax(f, T(0)), T(8)));
}

// Eigen-analysis and bucket exactly as the reference writes it (ravu-lite-r3.hook:77-87),
// in the reference's operation order, no contraction.  Used in FP64 for re-decisions;
// mirrors the FP64 oracle operation for operation; a NaN angle or strength (windows with an
// infinity: L1 - a is inf - inf) is row 0, as there.
template <int RULE, typename T>
__device__ __forceinline__ Bucket hash_reference(T a, T b, T d) {
#pragma clang fp contract(off)
  const T eps = T(1.192092896e-7);
  const T pi = T(3.141592653589793);
  T Tr = a + d;
  T D = a * d - b * b;
  T disc = Tr * Tr / T(4) - D;
  T delta = sqrt(disc < T(0) ? T(0) : disc);  // (fmax would drop a NaN)
  T L1 = Tr / T(2) + delta;
  T L2 = Tr / T(2) - delta;
  T sqrtL1 = sqrt(L1);
  T sqrtL2 = sqrt(L2);  // NaN when L2 < 0, as in the reference
  T at = atan2(L1 - a, b) + pi;
  T theta = at - pi * floor(div_const(at, pi, T(1) / pi));  // GLSL mod
  if (fabs(b) < eps) theta = T(0);
  T ssum = sqrtL1 + sqrtL2;
  T mu = (sqrtL1 - sqrtL2) / ssum;
  if (ssum < eps) mu = T(0);
  Bucket bk;
  bk.angle = static_cast<int>(floor(div_const(theta * T(24), pi, T(1) / pi)));
  bk.strength = strength_of<RULE, T>(sqrtL1);
  bk.coherence = mu >= T(0.5) ? 2 : (mu >= T(0.25) ? 1 : 0);  // NaN -> 0
  if (theta != theta || (RULE == RULE_LOG2 && sqrtL1 != sqrtL1)) return {0, 0, 0};
  return bk;
}

// FP32 fast path.  Same quantities through cancellation-free forms (mathematically equal
// to the reference's): delta = sqrt(((a-d)/2)^2 + b^2) instead of sqrt(T^2/4 - D), and
// L1 - a = b^2 / ((a-d)/2 + delta) when d < a.  Square roots and quotients are the
// hardware's (within 1 ulp), the strength of RULE_LOG2 is the exponent of its argument
// (floor(log2 v)), and the angle atan2(L1 - a, b) in units of pi/24 is an odd degree-13
// minimax polynomial of min / max (fitted by the Remez exchange; |error| <= 2.6e-6 units
// in FP32).  Sets *near, and the caller re-decides in FP64, when a decision may differ from
// the exact one.  The tensor's own FP32 error (u = 2^-24): differences of exact samples are off by
// u each, which the five-point stencil can amplify by cancellation, but never past 1.83 u of the
// tensor's norm (the largest ratio over all 8 x 8 windows, an eigenvalue; 6 x 6: 1.69, central and
// border stencils: 1); the five-point form adds a rounding of its own.  Both count twice in a
// square, beside one rounding each of the product and the weight and one per term of a running
// sum.  That puts a and d within K u of themselves and b within K u T / 2, K = 13 for 5 x 5 windows
// (9 terms), 29 for 7 x 7 (25), 20 for 4 x 4 (16; 31 for rgb, rounded relative to an inner sample), 24
// for 6 x 6 (16), 17 and 21 for the column sums of 6 x 6 and 8 x 8 (SepTensor: two levels of four or six
// terms).  With K <= 31, sqrt(L1) lies within a relative 31 u = 1.9e-6 (margin 3.8e-6), b within
// 15.5 u T (16 u), L2 within 31 u T (99 u), mu within 42 u at 1/4 and 70 u at 1/2 (6e-6 = 100 u), the
// angle within 22 u T / (2 delta) (32 u, plus 1e-5 units for the evaluation, whose error is below
// 5e-6).  A sample that is itself rounded, like an rgb luma in FP32, has no place in this bound:
// see HashSample.  Exact cases (flat window T = 0, b = 0 exactly) are never near.
// The margin of b decides which frames of thin horizontal and vertical lines are near everywhere:
// with 24 u, a line grid 1280x720 took lite-r3 18.9 us instead of 15.7, r3 80.1 instead of 73.9,
// r4-rgb (of an FP32 luma) 339 instead of 154, zoom-r3 at 1.5x 44.0 instead of 36.6.
// Bound by VALU issue: the exactly rounded sqrtf, the library atan2f and log2f that this
// replaces took about 75 of a hash's ~150 instructions, and an angle margin of 2.4e-4 units
// sent 3-4x as many sites to FP64.  Measured: ravu-r3 1366x768 44.3 -> 37.5 us, r4-yuv
// 2 x 1080p 266 -> 248, lite-ar-r3 8 x 1080p 255.6 -> 240.9, 3x-r3 2 x 1080p 54.5 -> 51.6,
// the same bits out.
template <int RULE>
__device__ __forceinline__ Bucket hash_fast(float a, float b, float d, bool* near) {
  const float eps = 1.192092896e-7f;
  const float rel = 4e-6f, u16 = 16.0f * 5.9604645e-8f;
  const float T = a + d;
  const float h = (a - d) * 0.5f;
  const float delta = __builtin_amdgcn_sqrtf(fmaf(h, h, b * b));
  const float L1 = fmaf(T, 0.5f, delta);
  const float L2 = fmaf(T, 0.5f, -delta);
  const float y = h <= 0.f ? delta - h : b * b * __builtin_amdgcn_rcpf(h + delta);  // L1 - a >= 0
  const float sqrtL1 = __builtin_amdgcn_sqrtf(L1);
  const float sqrtL2 = __builtin_amdgcn_sqrtf(L2);  // NaN when L2 < 0, as in the reference
  // u = 24/pi * mod(atan2(y, b) + pi, pi) = 24/pi * atan2(y, b), in [0, 24], since y >= 0 (the wrap at
  // 24 is a near case); inf/inf counts as 1, a NaN takes angle 0
  const float ab = fabsf(b);
  const float r = fminf(fminf(y, ab) * __builtin_amdgcn_rcpf(fmaxf(y, ab)), 1.0f);
  const float s = r * r;
  float p = 0.05203826725482941f;
  p = fmaf(p, s, -0.256717324256897f);
  p = fmaf(p, s, 0.6082800626754761f);
  p = fmaf(p, s, -1.0109528303146362f);
  p = fmaf(p, s, 1.513205647468567f);
  p = fmaf(p, s, -2.545259475708008f);
  p = fmaf(p, s, 7.639407634735107f);
  p *= r;
  p = y > ab ? 12.0f - p : p;
  p = b < 0.f ? 24.0f - p : p;
  const bool bsmall = ab < eps;
  const float u = bsmall || __builtin_isunordered(y, b) ? 0.f : p;
  const float ssum = sqrtL1 + sqrtL2;
  float mu = (sqrtL1 - sqrtL2) * __builtin_amdgcn_rcpf(ssum);
  if (ssum < eps) mu = 0.f;
  Bucket bk;
  bk.angle = static_cast<int>(floorf(u));
  bk.coherence = mu >= 0.5f ? 2 : (mu >= 0.25f ? 1 : 0);
  bool n = fabsf(ab - eps) <= fmaf(u16, T, rel * eps);
  n |= fabsf(L2) <= (rel + 2.0f * u16) * T && !(b == 0.f && fminf(a, d) == 0.f);
  const float cond = (24.0f / kPiF) * 32.0f * 5.9604645e-8f * T * __builtin_amdgcn_rcpf(fmaxf(2.0f * delta, 1e-30f));
  n |= !bsmall && fabsf(u - rintf(u)) <= 1e-5f + cond;
  if (RULE == RULE_LOG2) {
    // floor(log2 v) clamped to 0..8; near: v within a relative 3.8e-6 (7.6e-6) below (above) 2^1 .. 2^8
    const float v = fmaf(sqrtL1, 2000.0f, eps);
    const uint32_t bits = __float_as_uint(v), up = bits + 64u;
    bk.strength = v >= 2.0f ? min(static_cast<int>(bits >> 23) - 127, 8) : 0;
    n |= (up & 0x7fffffu) < 128u && (up >> 23) - 128u < 8u;
  } else {
    bk.strength = strength_of<RULE, float>(sqrtL1);
    if (RULE == RULE_LITE)
      n |= fabsf(sqrtL1 - 0.004f) <= rel * 0.004f || fabsf(sqrtL1 - 0.016f) <= rel * 0.016f ||
           fabsf(sqrtL1 - 0.05f) <= rel * 0.05f;
    else
      n |= fabsf(sqrtL1 - 0.005f) <= rel * 0.005f || fabsf(sqrtL1 - 0.02f) <= rel * 0.02f;
  }
  n |= fminf(fabsf(mu - 0.25f), fabsf(mu - 0.5f)) <= 6e-6f;
  *near = n && T > 0.f;
  return bk;
}

// LUT row of a bucket as NEAREST + clamp-to-edge sampling hits it:
// texel row floor(((angle*S + strength)*3 + coherence + 0.5)) clamped to [0, rows-1]
// (angle can be 24 or -1 at the wrap of mod(atan(..)+pi, pi)).
template <int RULE>
__device__ __forceinline__ int bucket_row(Bucket bk, int rows) {
  int row = (bk.angle * RuleInfo<RULE>::S + bk.strength) * 3 + bk.coherence;
  return min(max(row, 0), rows - 1);
}

// hash_reference out of line: its registers (the double atan2 alone takes 56) would set the
// occupancy of every wave.
template <int RULE>
__device__ __attribute__((noinline)) Bucket hash_fp64(double a, double b, double d) {
  return hash_reference<RULE, double>(a, b, d);
}

// The structure tensor of the sites of this wave whose bit is set in `mask`, in FP64 and in
// the oracle's operation order (no contraction): the whole wave works on one site at a time, a
// grid point per lane (at most 36), and the points' terms are then added in grid order.
// `at(site)` gives an accessor (X, Y) -> sample of the window of lane `site`.  Every lane of
// the wave must be active.  a, b, d are set in the lanes of `mask`.
// Bound by the latency of the wave that takes it, which holds its block's LDS meanwhile: one
// lane's serial evaluation (up to 36 points of two five-point derivatives, for r4 rgb of a luma
// computed per sample) took 10-20 us where a wave otherwise lives about 10 (ravu-r4-rgb 640x360
// 51.6 us, 21.2 with the path switched off; with the shared one 28.7).  Small central-difference windows (lite, 3x) keep a lane's own evaluation: several
// of their lanes are near at once (lite-r2 8 x 1080p 126 us, shared 150).
template <int N, bool FIVE, typename At>
__device__ __forceinline__ void wave_tensor(uint64_t mask, At at, double& a, double& b, double& d) {
#pragma clang fp contract(off)
  using GG = GradGrid<N>;
  constexpr int POINTS = GG::M * GG::M;
  const int lane = threadIdx.x & 63;
  const int pt = min(lane, POINTS - 1);
  const int X = GG::P0 + pt / GG::M, Y = GG::P0 + pt % GG::M;
  const double w = gauss_w<N>(pt);
  // one derivative: position p of the line s, forward/backward at the border (its two samples
  // clamped into the window), central or five-point inside
  auto derivative = [](auto s, int p) {
#pragma clang fp contract(off)
    const double lo = s(max(p - 1, 0)), hi = s(min(p + 1, N - 1));
    const double diff = hi - lo;
    double r = p == 0 || p == N - 1 ? diff : diff / 2.0;
    if constexpr (FIVE && N >= 5) {
      const double num = -s(min(p + 2, N - 1)) + 8.0 * hi - 8.0 * lo + s(max(p - 2, 0));
      if (p >= 2 && p + 2 <= N - 1) r = div_const(num, 12.0, 1.0 / 12.0);
    }
    return r;
  };
  auto lane_value = [](double v, int i) {
    const uint64_t u = __double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(u), i);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(u >> 32), i);
    return __longlong_as_double(static_cast<int64_t>(static_cast<uint64_t>(hi) << 32 | lo));
  };
  while (mask) {
    const int site = __builtin_ctzll(mask);
    mask &= mask - 1;
    const auto sample = at(site);
    const double gx = derivative([&](int k) { return sample(k, Y); }, X);
    const double gy = derivative([&](int k) { return sample(X, k); }, Y);
    const double ta = gx * gx * w, tb = gx * gy * w, td = gy * gy * w;
    double sa = 0.0, sb = 0.0, sd = 0.0;
#pragma unroll 4
    for (int i = 0; i < POINTS; ++i) {
      sa = sa + lane_value(ta, i);
      sb = sb + lane_value(tb, i);
      sd = sd + lane_value(td, i);
    }
    if (lane == site) {
      a = sa;
      b = sb;
      d = sd;
    }
  }
}

// Value of lane `i` (uniform) in every lane.
__device__ __forceinline__ int from_lane(int v, int i) { return __builtin_amdgcn_readlane(v, i); }

// SITES of redecide: one turn of the wave is cheaper than a lane alone (ravu-r4 1280x720 36.5 us
// against 40.9, r4-rgb 66.7 against 70.2), two turns are not (r3, isolated dots: 37.0 with 1, 39.1 with
// 2, 39 to 41 with 4 to 16; r4-rgb, large flat shapes: 100.3 with 1, 102.6 with 2).
constexpr int kWaveSites = 1;

// The staged samples that a hash sees, as an accessor carries them into that function: an LDS
// pointer, as a generic one's reads are flat loads there (45-degree stripes 1280x720: ravu-r4
// 170 -> 133 us, r3 87 -> 82).
template <typename T>
using LdsSamples = const __attribute__((address_space(3))) T*;
template <typename T>
__device__ __forceinline__ LdsSamples<T> lds_samples(const T* p) { return (LdsSamples<T>)p; }

// One lane's own evaluation and hash, out of line: inlined, its registers (the double atan2 alone
// takes 56) would set the occupancy of every wave.  `sample(X, Y)` comes by value, and each
// kernel's accessor is a type of its own, so each has its own instance, with its caller's
// register budget (the lean tensor form keeps it from spilling).
template <int N, bool FIVE, int RULE, typename Sample>
__device__ __attribute__((noinline)) Bucket redecide_alone(Sample sample) {
  double a, b, d;
  structure_tensor_fp64<N, FIVE, true>([&](int i) { return sample(i / N, i % N); }, a, b, d);
  return hash_reference<RULE, double>(a, b, d);
}

// The FP64 re-decision of the lanes whose FP32 decision is near a boundary.  `at(o)` gives the
// accessor (X, Y) -> sample of the window at offset o, of which `o` is this lane's.
// Up to SITES near lanes are taken one after the other by the whole wave (wave_tensor, which also
// says what bounds it); more evaluate their own windows at the same time.  A wave full of near
// sites (a frame of 45-degree stripes) would take 64 turns: ravu-r4 1280x720 1512 us, against 91
// with each lane on its own.
template <int N, bool FIVE, int RULE, int SITES, typename At>
__device__ __forceinline__ void redecide(bool near, int o, At at, Bucket& bk) {
  const uint64_t mask = __ballot(near);
  if (!mask) return;
  if (__popcll(mask) <= SITES) {
    double a = 0.0, b = 0.0, d = 0.0;
    wave_tensor<N, FIVE>(mask, [&](int site) { return at(from_lane(o, site)); }, a, b, d);
    if (near) bk = hash_fp64<RULE>(a, b, d);
  } else if (near) {
    bk = redecide_alone<N, FIVE, RULE>(at(o));
  }
}

// Hash of one site: FP32, re-decided in FP64 when near a boundary.  get(i) returns window sample i
// as it is stored.  LEAN picks the FP64 tensor's form.
template <int N, bool FIVE, int RULE, bool LEAN = false, typename Get>
__device__ __forceinline__ Bucket ravu_hash(Get get) {
  float a, b, d;
  structure_tensor<N, FIVE>(get, a, b, d);
  bool near = false;
  Bucket bk = hash_fast<RULE>(a, b, d, &near);
  if (near) {
    double ad, bd, dd;
    structure_tensor_fp64<N, FIVE, LEAN>(get, ad, bd, dd);
    bk = hash_reference<RULE, double>(ad, bd, dd);
  }
  return bk;
}

// The same with the wave's shared re-decision.  o, at: see redecide.  All lanes of the wave call it together; lanes
// without a site (`valid` false) read their window too (inside the staged tile) but are never
// re-decided.
template <int N, bool FIVE, int RULE, int SITES, typename Get, typename At>
__device__ __forceinline__ Bucket ravu_hash_wave(bool valid, Get get, int o, At at) {
  float a, b, d;
  structure_tensor<N, FIVE>(get, a, b, d);
  bool near = false;
  Bucket bk = hash_fast<RULE>(a, b, d, &near);
  redecide<N, FIVE, RULE, SITES>(near && valid, o, at, bk);
  return bk;
}

}  // namespace mpx
