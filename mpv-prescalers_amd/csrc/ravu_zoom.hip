// RAVU-zoom(-ar) to an arbitrary output size, luma / yuv / rgb
// (ravu-zoom-r2.hook:15-134, ravu-zoom-ar-r2-rgb.hook:15-224, compute tiling
// compute/ravu-zoom-r3.hook:24-45).
//
// Per output pixel o: pos = (o + 1/2) * in/out (OFFSET ALIGN); subpix f = fract(pos - 1/2);
// base = pos - f.  The window is the 2r x 2r input block at offsets -(r-1)..r around base.
// The hash depends on the base pixel only, so a block first hashes every base pixel its
// output tile (32 x 8 by default) touches (into LDS), then each output pixel reads its
// base's bucket; AR variants also tabulate the per-sample powers of the anti-ringing
// weights there.
// Base and phase are computed in exact integer arithmetic:
//   pos - 1/2 = ((2o+1)*in - out) / (2*out)  ->  base = floor, f = remainder / (2*out),
// once per output column and row at plan creation (zoom_phase_kernel); the kernel reads
// them from that table.
// LUT (FILTER LINEAR): group g of 4 taps at texel x = 9g + 8f, row y = 9*bucket + 8f_y
// (LUTPOS, :21-31), bilinear between neighbouring phase texels, rows clamped to the
// texture; taps p < n^2/2 at phase f, tap n^2-1-p at phase 1-f.  AR variants use the
// separate learned ``_ar`` LUT with the same addressing (all taps), per channel, strength
// 0.8, no final clamp.  The LUTs (0.37 / 0.93 MB FP16) stay in L2.
#include "common.h"
#include "launch.h"
#include "ravu.h"
#include "internal.h"

#include <numeric>

namespace mpx {


__device__ __forceinline__ int floor_div(int64_t a, int64_t b) {  // b > 0
  int64_t q = a / b;
  if ((a % b) != 0 && (a < 0)) --q;
  return static_cast<int>(q);
}

struct Phase {
  int base;
  float f;
};
__device__ __forceinline__ Phase phase_of(int o, int in, int out) {
  const int64_t num = static_cast<int64_t>(2 * o + 1) * in - out;
  const int64_t den = 2 * static_cast<int64_t>(out);
  Phase p;
  p.base = floor_div(num, den);
  p.f = static_cast<float>(num - static_cast<int64_t>(p.base) * den) / static_cast<float>(den);
  return p;
}

// FILTER LINEAR fetch of the G texel groups of one phase: texel coordinates (9g + tx,
// 9*row + ty), tx, ty in [0, 8]; the integer row base is kept apart so the phase fraction keeps
// full FP32 precision.  Rows clamp to the texture (row can be -1 or past the last bucket).
// tx = 8 is taken as the full weight of texel 8 of the pair (7, 8).
// The table holds a texel row phase by phase (texel x * G + g), so the groups of both texels of
// a row are one run of 2 G texels (r3: 80 bytes), read 16 bytes at a time, instead of 2 G
// scattered ones, and a weight is four multiply-adds (the FP16 texel converts inside them).
// Bound by the texels' lines out of L2 (a LUT outgrows L1, neighbouring pixels rarely share a
// bucket and phase): r3 luma 1366x768 -> 1920x1080, 40 gathers and 948 VALU instructions per
// pixel, 52.0 us; with 24 and 731, 43.4 us.
// The arithmetic is spelled out (explicit fmaf, no contraction) so that every kernel that
// inlines it rounds the same way: the plan-time weight table and the per-pixel fetch agree
// bit for bit.
typedef uint32_t Texel2 __attribute__((ext_vector_type(4)));        // two FP16 RGBA texels
typedef Texel2 Texel2a __attribute__((aligned(8)));
template <int G>
struct PhaseFetch {
  const uint2 *r0, *r1;  // texels of the upper and lower row from x0 on
  float c00, c01, c10, c11;
  __device__ __forceinline__ PhaseFetch(const __half* lut, int rows, float tx, int row, float ty) {
#pragma clang fp contract(off)
    const float fx0 = fminf(floorf(tx), 7.f), fy0 = floorf(ty);
    const float ax = tx - fx0, ay = ty - fy0, bx = 1.f - ax, by = 1.f - ay;
    const int y = 9 * row + static_cast<int>(fy0);
    const int y0 = min(max(y, 0), rows - 1), y1 = min(max(y + 1, 0), rows - 1);
    const uint2* p = reinterpret_cast<const uint2*>(lut) + static_cast<int>(fx0) * G;
    r0 = p + y0 * (9 * G);
    r1 = p + y1 * (9 * G);
    c00 = bx * by;
    c01 = ax * by;
    c10 = bx * ay;
    c11 = ax * ay;
  }
  __device__ __forceinline__ float4 mix(uint2 v00, uint2 v01, uint2 v10, uint2 v11) const {
#pragma clang fp contract(off)
    auto one = [&](__half p, __half q, __half r, __half s) {
      return fmaf(__half2float(s), c11, fmaf(__half2float(r), c10, fmaf(__half2float(q), c01, __half2float(p) * c00)));
    };
    const __half2 a0 = bits_h2(v00.x), a1 = bits_h2(v00.y), b0 = bits_h2(v01.x), b1 = bits_h2(v01.y);
    const __half2 d0 = bits_h2(v10.x), d1 = bits_h2(v10.y), e0 = bits_h2(v11.x), e1 = bits_h2(v11.y);
    return make_float4(one(a0.x, b0.x, d0.x, e0.x), one(a0.y, b0.y, d0.y, e0.y), one(a1.x, b1.x, d1.x, e1.x),
                       one(a1.y, b1.y, d1.y, e1.y));
  }
  __device__ __forceinline__ float4 get(int g) const { return mix(r0[g], r0[G + g], r1[g], r1[G + g]); }
  // groups g and g + 1
  __device__ __forceinline__ void get2(int g, float4* w) const {
    const Texel2 v00 = *reinterpret_cast<const Texel2a*>(r0 + g), v01 = *reinterpret_cast<const Texel2a*>(r0 + G + g);
    const Texel2 v10 = *reinterpret_cast<const Texel2a*>(r1 + g), v11 = *reinterpret_cast<const Texel2a*>(r1 + G + g);
    w[0] = mix({v00[0], v00[1]}, {v01[0], v01[1]}, {v10[0], v10[1]}, {v11[0], v11[1]});
    w[1] = mix({v00[2], v00[3]}, {v01[2], v01[3]}, {v10[2], v10[3]}, {v11[2], v11[3]});
  }
};

// Stage the part of the PH x PW staging area that a tile's outputs read: the uh x uw
// samples per plane around its base pixels (at 2x 8 x 20 of 12 x 36), clamp-to-edge, at
// the area's row stride PW.  AR forms store each sample's anti-ringing powers beside it
// ((0.1 + l)^32, (1.1 - l)^32 and the ^33 terms, once per sample instead of once per
// output pixel that reads it).  Sample i of the dense P x uh x uw order is split with
// high-half multiply quotients: floor(i / d) = mulhi(i, floor((2^32 - 1) / d) + 1), exact
// while i * d < 2^32.
template <int P, int PH, int PW, int NT, bool AR>
__device__ __forceinline__ void stage_used(float* tile, float4* pw, const void* base, int dt, float in_max,
                                           float in_rmax, int64_t pitch, int64_t cstride, int W, int H, int ox,
                                           int oy, int uw, int uh) {
  constexpr int PN = PH * PW, E = (P * PN + NT - 1) / NT;
  static_assert(static_cast<int64_t>(P) * PN * PN < (int64_t{1} << 32), "high-half quotients exact");
  const int un = uw * uh, total = P * un;
  const uint32_t mn = 0xffffffffu / static_cast<uint32_t>(un) + 1u;
  const uint32_t mw = 0xffffffffu / static_cast<uint32_t>(uw) + 1u;
  const int lsh = dt == DT_F32 ? 2 : (dt == DT_U8 ? 0 : 1);  // log2 element bytes
  const uintptr_t b = reinterpret_cast<uintptr_t>(base);
  uint32_t v[E], sh[E];
  int li[E];
  __builtin_amdgcn_s_setprio(1);  // the loads go out ahead of other waves' arithmetic
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = static_cast<int>(threadIdx.x) + NT * e;
    li[e] = -1;
    if (i < total) {
      const int c = P == 1 ? 0 : static_cast<int>(__umulhi(static_cast<uint32_t>(i), mn));
      const int j = i - c * un;
      const int r = static_cast<int>(__umulhi(static_cast<uint32_t>(j), mw));
      const int col = j - r * uw;
      const int gx = min(max(ox + col, 0), W - 1), gy = min(max(oy + r, 0), H - 1);
      // 32-bit element offset, as the halo loaders (the host bounds the frame's span)
      const uint32_t off = static_cast<uint32_t>(c) * static_cast<uint32_t>(cstride) +
                           __umul24(static_cast<uint32_t>(gy), static_cast<uint32_t>(pitch)) + gx;
      const uintptr_t a = b + (static_cast<uintptr_t>(off) << lsh);
      v[e] = *reinterpret_cast<GlobalU32>(a & ~static_cast<uintptr_t>(3));
      sh[e] = static_cast<uint32_t>(a & 3) * 8;
      li[e] = c * PN + r * PW + col;
    }
  }
  __builtin_amdgcn_s_setprio(0);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    if (li[e] >= 0) {
      const uint32_t w = v[e] >> sh[e];
      float l;
      switch (dt) {
        case DT_F32: l = __uint_as_float(v[e]); break;
        case DT_F16: l = __half2float(__ushort_as_half(static_cast<unsigned short>(w & 0xffffu))); break;
        case DT_U8: l = unorm_quotient(static_cast<float>(w & 0xffu), in_max, in_rmax); break;
        default: l = unorm_quotient(static_cast<float>(w & 0xffffu), in_max, in_rmax); break;
      }
      tile[li[e]] = l;
      if constexpr (AR) {
        const float p0 = 0.1f + l, m0 = 1.1f - l;
        float p32 = p0, m32 = m0;
#pragma unroll
        for (int k = 0; k < 5; ++k) { p32 *= p32; m32 *= m32; }
        pw[li[e]] = make_float4(p32, m32, p32 * p0, m32 * m0);
      }
    }
  }
}

// Pre-interpolated weights.  The phase of output column o repeats with period
// out / gcd(in, out) (2 at 2x, 3 at 1.5x), so for such plans every (bucket row, phase pair)
// is interpolated once, at plan creation, by the same PhaseFetch in the same operations:
// table entry (row, py, px, g) holds the group's float4s [wf, wi (, af, ai)].  Bucket rows
// below 0 fetch the same texels as row -1 and rows past the last bucket the same as
// bucket 288 (the texel rows clamp), so rows -1..288 cover every bucket value.
constexpr int kZoomRowLo = -1, kZoomRows = 290;
constexpr int kZoomMaxPhasePairs = 64;
// float4s from one bucket row's entries to the next.  L1 serves 16 bytes per lane, four lanes per
// cycle, if the four lie in different 16-byte columns of their 64-byte halves of lines.  A lane reads
// its own row's entries at an offset that all lanes share, so with rows a multiple of 64 bytes apart
// every lane wants the same column.  An odd stride puts neighbouring rows into different ones.
// Where neighbouring lanes' column phases already differ in it (three or more phases, 160 bytes
// apart) the stride stays.  Measured at 2x, where noisy frames were bound by this path (texture data busy
// for the whole launch, 49 cycles per load): r3 4 x 720p noise 226 -> 159 us, video 113 -> 91; r3-yuv
// 235 -> 175, 129 -> 120; ar-r2 195 -> 140, 114 -> 94; r2 103 -> 77, 75 -> 71; at 1.5x ar-r2 720p 37.0 ->
// 28.9, 34.4 -> 29.8.  (r3 at 1.25x with an odd stride: 28.1 -> 30.1.)
__device__ __host__ constexpr int zoom_row_stride(int nphx, int nphy, int groups, int nt) {
  const int n = nphx * nphy * groups * nt;
  return nphx == 2 || groups * nt % 4 == 0 ? n | 1 : n;
}

template <int R, bool AR>
__global__ __launch_bounds__(256) void zoom_table_kernel(const __half* __restrict__ lut,
                                                         const __half* __restrict__ lut_ar, float4* wtab, int in_w,
                                                         int in_h, int out_w, int out_h, int nphx, int nphy) {
  constexpr int N = 2 * R;
  constexpr int GROUPS = (N * N / 2 + 3) / 4;
  constexpr int ROWS = 2592;
  constexpr int NT = AR ? 4 : 2;
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= kZoomRows * nphy * nphx * GROUPS) return;
  const int g = i % GROUPS;
  int t = i / GROUPS;
  const int px = t % nphx;
  t /= nphx;
  const int py = t % nphy;
  const int row = t / nphy + kZoomRowLo;
  const Phase phx = phase_of(px, in_w, out_w), phy = phase_of(py, in_h, out_h);
  const float txf = 8.f * phx.f, txi = 8.f * (1.f - phx.f);
  const float tyf = 8.f * phy.f, tyi = 8.f * (1.f - phy.f);
  float4* e = wtab + (row - kZoomRowLo) * zoom_row_stride(nphx, nphy, GROUPS, NT) + ((py * nphx + px) * GROUPS + g) * NT;
  e[0] = PhaseFetch<GROUPS>(lut, ROWS, txf, row, tyf).get(g);
  e[1] = PhaseFetch<GROUPS>(lut, ROWS, txi, row, tyi).get(g);
  if (AR) {
    e[2] = PhaseFetch<GROUPS>(lut_ar, ROWS, txf, row, tyf).get(g);
    e[3] = PhaseFetch<GROUPS>(lut_ar, ROWS, txi, row, tyi).get(g);
  }
}

// Phase table of a plan: entry o < out_w is output column o, entry out_w + o row o:
// {base, bits of f, o mod period, 0}.
__global__ __launch_bounds__(256) void zoom_phase_kernel(int4* tab, int in_w, int in_h, int out_w, int out_h,
                                                         int nphx, int nphy) {
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= out_w + out_h) return;
  const bool x = i < out_w;
  const int o = x ? i : i - out_w;
  const Phase ph = x ? phase_of(o, in_w, out_w) : phase_of(o, in_h, out_h);
  tab[i] = make_int4(ph.base, __float_as_int(ph.f), o % (x ? nphx : nphy), 0);
}

// Anti-ringing of one output: mix(res, clamp(res, lo, hi), 0.8), no final clamp.
__device__ __forceinline__ float zoom_ring(float v, float hi, float lo, float hi2, float lo2) {
  const float h = hi2 * __builtin_amdgcn_rcpf(hi) - 0.1f, l = 1.1f - lo2 * __builtin_amdgcn_rcpf(lo);
  const float cl = fminf(fmaxf(v, l), h);
  return v * (1.0f - 0.8f) + cl * 0.8f;
}

// The samples that the hash sees of a staged tile (n per plane): for rgb the FP64 luma, filled into
// `luma` here for `count` samples; the caller synchronises the block before and after.
template <int CH, int NT>
__device__ __forceinline__ const HashSample<CH>* zoom_luma(const float* tile, double* luma, int n, int count) {
  if constexpr (CH == 2) {
    fill_luma<NT>(tile, luma, n, count);
    return luma;
  } else {
    return tile;
  }
}

// Hash every base pixel of a tile (nbx x nby) into bucket[by * BX + bx]: the unclamped LUT row
// (bucket 9-row blocks are clamped per texel by the bilinear fetch, as the sampler does).
// r2's near lanes evaluate their own windows (16 points: a turn of the wave is no cheaper, and the
// kernel is smaller: 4 x 720p -> 1440p zoom-ar-r2-rgb 185 -> 184 us, ar-r2 94.6 -> 92.6, large flat shapes
// 207 -> 202, 100 -> 96).  TAB only
// tells the kernels apart: the out-of-line evaluation follows its caller's register budget.
template <int R, bool AR, int CH, bool TAB, int BX, int PW, int NT>
__device__ __forceinline__ void hash_bases(const HashSample<CH>* lum, int* bucket, int nbx, int nby) {
  constexpr int N = 2 * R;
  // (whole waves: the re-decision takes all lanes; those past the last base pixel repeat it)
  for (int i0 = threadIdx.x & ~63; i0 < nbx * nby; i0 += NT) {
    const int lane_i = i0 + static_cast<int>(threadIdx.x & 63), i = min(lane_i, nbx * nby - 1);
    const int by = i / nbx, bx = i - by * nbx;
    auto off = [&](int s) { return (by + s % N) * PW + bx + s / N; };
    auto sample = [&](int s) { return lum[off(s)]; };
    const Bucket bk = ravu_hash_wave<N, true, RULE_LITE, R == 2 ? 0 : kWaveSites>(
        lane_i == i, sample, by * PW + bx, [&](int o) {
          const auto t = lds_samples(lum) + o;
          return [t](int X, int Y) { return t[Y * PW + X]; };
        });
    if (lane_i == i) bucket[by * BX + bx] = (bk.angle * 4 + bk.strength) * 3 + bk.coherence;
  }
}

// One block per TX x TY output tile, one thread per output pixel (kZoomTiles).  (Kernels
// without anti-ringing: at least 6 waves per SIMD, a register budget their out-of-line
// re-decision inherits; r2 anti-ringing kernels and r3 ones on 16 x 16 tiles: 5, at most 96
// VGPRs with 16 to 80 bytes of scratch in some, measured 1-8 % faster than 4 waves; r3-rgb misses
// it at 108 and more.)  TAB: the plan has the pre-interpolated weight table; separate instances keep the per-pixel bilinear fetch's registers out of the
// table path.
template <int R, bool AR, int CH, bool TAB, int TX, int TY>
__global__ __launch_bounds__(TX * TY) __attribute__((amdgpu_waves_per_eu(AR ? ((R == 2 || TX == 16) ? 5 : 1) : 6))) void ravu_zoom_kernel(Io io, const __half* __restrict__ lut,
                                                        const __half* __restrict__ lut_ar,
                                                        const float4* __restrict__ wtab, int nphx, int nphy,
                                                        const int4* __restrict__ phase, int out_w, int out_h) {
  constexpr int P = CH == 0 ? 1 : 3;
  constexpr int N = 2 * R;
  constexpr int HALF = N * N / 2;
  constexpr int GROUPS = (HALF + 3) / 4;
  constexpr int ROWS = 2592;             // 288 buckets x 9 phases
  constexpr int BX = TX + 1, BY = TY + 1;  // base pixels a tile can touch (ratio in/out < 1)
  constexpr int PW = BX + N - 1, PH = BY + N - 1, PN = PW * PH;
  __shared__ __attribute__((aligned(16))) float tile[P * PN];
  static_assert(PN % 2 == 0, "lumas in pairs");
  __shared__ __attribute__((aligned(16))) double luma[CH == 2 ? PN : 1];
  __shared__ int bucket[BY * BX];
  // AR: per staged sample (l + 0.1)^32, (1.1 - l)^32 and the ^33 terms, computed once per
  // sample instead of once per output pixel that reads it (about 25 at 2x)
  __shared__ float4 pw[AR ? P * PN : 1];

  const BlockXYZ bk3 = block_xyz((out_w + TX - 1) / TX, (out_h + TY - 1) / TY, io.batch);
  const int f = bk3.z;
  const int ox0 = bk3.x * TX, oy0 = bk3.y * TY;
  const int4* phy_tab = phase + out_w;
  const int bx0 = phase[ox0].x;
  const int by0 = phy_tab[oy0].x;
  // base pixels this tile's (in-range) outputs touch: nbx x nby <= BX x BY (in < out)
  const int nbx = phase[min(ox0 + TX, out_w) - 1].x - bx0 + 1;
  const int nby = phy_tab[min(oy0 + TY, out_h) - 1].x - by0 + 1;
  const void* in = frame_in(io, f);
  stage_used<P, PH, PW, TX * TY, AR>(tile, pw, in, io.in_dt, io.in_max, io.in_rmax, io.in_pitch, io.in_cstride, io.W, io.H,
                            bx0 - (R - 1), by0 - (R - 1), nbx + N - 1, nby + N - 1);
  __syncthreads();
  const auto* lum = zoom_luma<CH, TX * TY>(tile, luma, PN, (nby + N - 1) * PW);
  if constexpr (CH == 2) __syncthreads();
  hash_bases<R, AR, CH, TAB, BX, PW, TX * TY>(lum, bucket, nbx, nby);
  __syncthreads();

  const int ox = ox0 + threadIdx.x % TX, oy = oy0 + threadIdx.x / TX;
  if (ox >= out_w || oy >= out_h) return;
  const int4 phx = phase[ox], phy = phy_tab[oy];
  const float fx = __int_as_float(phx.y), fy = __int_as_float(phy.y);
  const int lbx = phx.x - bx0, lby = phy.x - by0;  // in [0, nbx) x [0, nby) by construction
  const int row = bucket[lby * BX + lbx];
  if (io.buckets) io.buckets[f * io.bucket_bstride + static_cast<int64_t>(oy) * out_w + ox] = row;
  auto si = [&](int c, int i) { return c * PN + (lby + i % N) * PW + lbx + i / N; };
  const float txf = 8.f * fx, txi = 8.f * (1.f - fx);
  const float tyf = 8.f * fy, tyi = 8.f * (1.f - fy);
  // this pixel's entries of the pre-interpolated table (when the plan has one)
  constexpr int NT = AR ? 4 : 2;
  const float4* wt = nullptr;
  if constexpr (TAB) {
    const int trow = min(max(row, kZoomRowLo), kZoomRowLo + kZoomRows - 1) - kZoomRowLo;
    wt = wtab + trow * zoom_row_stride(nphx, nphy, GROUPS, NT) + (phy.z * nphx + phx.z) * (GROUPS * NT);
  }
  float res[P], mirror[P], hi[P], lo[P], hi2[P], lo2[P];  // res: taps p, mirror: taps N^2 - 1 - p
#pragma unroll
  for (int c = 0; c < P; ++c) res[c] = mirror[c] = hi[c] = lo[c] = hi2[c] = lo2[c] = 0.f;
  // weights of the table-less path: two groups' texels per load (PhaseFetch)
  constexpr int GF = TAB ? 1 : GROUPS;
  const PhaseFetch<GF> ff(lut, ROWS, txf, row, tyf), fi(lut, ROWS, txi, row, tyi);
  const PhaseFetch<GF> af_(AR ? lut_ar : lut, ROWS, txf, row, tyf), ai_(AR ? lut_ar : lut, ROWS, txi, row, tyi);
  float4 pf[2], pi[2], pa[2], pb[2];
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    // one group's operands live at a time (its sums complete before the next group)
    __builtin_amdgcn_sched_barrier(0);
    float4 wf4, wi4, a4, b4;
    if constexpr (TAB) {
      wf4 = wt[g * NT];
      wi4 = wt[g * NT + 1];
      if (AR) {
        a4 = wt[g * NT + 2];
        b4 = wt[g * NT + 3];
      }
    } else {
      if (g % 2 == 0) {
        if (g + 1 < GROUPS) {
          ff.get2(g, pf);
          fi.get2(g, pi);
          if (AR) {
            af_.get2(g, pa);
            ai_.get2(g, pb);
          }
        } else {
          pf[0] = ff.get(g);
          pi[0] = fi.get(g);
          if (AR) {
            pa[0] = af_.get(g);
            pb[0] = ai_.get(g);
          }
        }
      }
      wf4 = pf[g % 2];
      wi4 = pi[g % 2];
      if (AR) {
        a4 = pa[g % 2];
        b4 = pb[g % 2];
      }
    }
    const float wf[4] = {wf4.x, wf4.y, wf4.z, wf4.w}, wi[4] = {wi4.x, wi4.y, wi4.z, wi4.w};
    float af[4] = {0.f, 0.f, 0.f, 0.f}, ai[4] = {0.f, 0.f, 0.f, 0.f};
    if (AR) {
      af[0] = a4.x; af[1] = a4.y; af[2] = a4.z; af[3] = a4.w;
      ai[0] = b4.x; ai[1] = b4.y; ai[2] = b4.z; ai[3] = b4.w;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      // two taps' LDS reads (samples and their powers, three planes) in flight at a time
      if (AR && k == 2) __builtin_amdgcn_sched_barrier(0);
      const int p = 4 * g + k;
      if (p < HALF) {
        const int q = N * N - 1 - p;
#pragma unroll
        for (int c = 0; c < P; ++c) {
          // one fused multiply-add per tap and sum; the taps and their mirror images in sums of
          // their own, which are half as long: their rounding falls by more than four rounded
          // products per weight add over nested interpolation (r3 to an odd size 4.72e-8 rms -> 4.10e-8,
          // nested 4.66e-8; r2 at 1.5x 4.04e-8 -> 3.63e-8, nested 3.81e-8; no change of time)
          const float lp = tile[si(c, p)], lq = tile[si(c, q)];
          res[c] = fmaf(lp, wf[k], res[c]);
          mirror[c] = fmaf(lq, wi[k], mirror[c]);
          if (AR) {
            // ravu-zoom-ar-r2-rgb.hook:152-222: (0.1+l)^32, (1.1-l)^32 and the ^33 terms
            const float4 a = pw[si(c, p)], b = pw[si(c, q)];
            hi[c] = fmaf(b.x, ai[k], fmaf(a.x, af[k], hi[c]));
            lo[c] = fmaf(b.y, ai[k], fmaf(a.y, af[k], lo[c]));
            hi2[c] = fmaf(b.z, ai[k], fmaf(a.z, af[k], hi2[c]));
            lo2[c] = fmaf(b.w, ai[k], fmaf(a.w, af[k], lo2[c]));
          }
        }
      }
    }
#pragma unroll
    for (int c = 0; c < P; ++c) {
      asm volatile("" : "+v"(res[c]), "+v"(mirror[c]));
      if (AR) asm volatile("" : "+v"(hi[c]), "+v"(lo[c]), "+v"(hi2[c]), "+v"(lo2[c]));
    }
  }
  const int esz_out = elem_bytes(io.out_dt);
  char* ob = static_cast<char*>(frame_out(io, f));
#pragma unroll
  for (int c = 0; c < P; ++c) {
    float v = res[c] + mirror[c];
    if (AR) {
      v = zoom_ring(v, hi[c], lo[c], hi2[c], lo2[c]);
    } else {
      v = fminf(fmaxf(v, 0.f), 1.f);
    }
    store_elem(ob + c * io.out_cstride * esz_out, static_cast<int64_t>(oy) * io.out_pitch + ox, io.out_dt, v);
  }
}

// The same for plans that scale the width by exactly 2 (and have the weight table): outputs 2k + 1
// and 2k + 2 share base pixel k, so a thread takes both and reads the window's samples and
// powers from LDS once for the two (TX base pixels x TY output rows per block; k = -1 ..
// in_w - 1, the first and the last with one output each).  Sums run in the same order.
// One output per thread read 1.07 KB of LDS per output for AR rgb (154 of its 287 us) beside a
// VALU share that overlapped it badly; this form is bound by VALU issue.  4 x 720p -> 1440p,
// one output -> two: r2 115 -> 70 us, r2-yuv 147 -> 95, r2-rgb 150 -> 97, r3 129 -> 91, r3-yuv 173 -> 120,
// r3-rgb 207 -> 141, ar-r2 146 -> 93, ar-r2-yuv 255 -> 176, ar-r2-rgb 272 -> 184; 640 x 360 ar-r2 14.4 -> 11.9;
// 320 x 180 within 6 % either way, 160 x 90, where half as many blocks run twice as long, up to
// 0.8 us slower of 7.3.
// 256 threads per block: with FP32 lumas 512 gave 249 us for ar-r2-rgb (waits at its barriers), 128 220, 256 211.
template <int R, bool AR, int CH, int TX, int TY>
__global__ __launch_bounds__(TX * TY) void ravu_zoom_pair_kernel(Io io, const float4* __restrict__ wtab, int nphy,
                                                                 const int4* __restrict__ phase, int out_w,
                                                                 int out_h) {
  constexpr int P = CH == 0 ? 1 : 3;
  constexpr int N = 2 * R, HALF = N * N / 2, GROUPS = (HALF + 3) / 4;
  constexpr int BX = TX, BY = TY + 1;
  constexpr int PW = BX + N - 1, PH = BY + N - 1, PN = PW * PH;
  constexpr int NT = AR ? 4 : 2;
  __shared__ __attribute__((aligned(16))) float tile[P * PN];
  static_assert(PN % 2 == 0, "lumas in pairs");
  __shared__ __attribute__((aligned(16))) double luma[CH == 2 ? PN : 1];
  __shared__ int bucket[BY * BX];
  __shared__ float4 pw[AR ? P * PN : 1];

  const BlockXYZ bk3 = block_xyz((io.W + 1 + TX - 1) / TX, (out_h + TY - 1) / TY, io.batch);
  const int f = bk3.z;
  const int bx0 = bk3.x * TX - 1, oy0 = bk3.y * TY;
  const int4* phy_tab = phase + out_w;
  const int by0 = phy_tab[oy0].x;
  const int nbx = min(TX, io.W - bx0);
  const int nby = phy_tab[min(oy0 + TY, out_h) - 1].x - by0 + 1;
  stage_used<P, PH, PW, TX * TY, AR>(tile, pw, frame_in(io, f), io.in_dt, io.in_max, io.in_rmax, io.in_pitch,
                                     io.in_cstride, io.W, io.H, bx0 - (R - 1), by0 - (R - 1), nbx + N - 1,
                                     nby + N - 1);
  __syncthreads();
  const auto* lum = zoom_luma<CH, TX * TY>(tile, luma, PN, (nby + N - 1) * PW);
  if constexpr (CH == 2) __syncthreads();
  hash_bases<R, AR, CH, true, BX, PW, TX * TY>(lum, bucket, nbx, nby);
  __syncthreads();

  const int lbx = threadIdx.x % TX, oy = oy0 + threadIdx.x / TX;
  if (lbx >= nbx || oy >= out_h) return;
  const int ox = 2 * (bx0 + lbx) + 1;  // this thread's outputs: ox (phase index 1), ox + 1 (phase index 0)
  const bool first = ox >= 0, second = ox + 1 < out_w;
  const int4 phy = phy_tab[oy];
  const int lby = phy.x - by0;
  const int row = bucket[lby * BX + lbx];
  if (io.buckets) {
    int32_t* b = io.buckets + f * io.bucket_bstride + static_cast<int64_t>(oy) * out_w + ox;
    if (first) b[0] = row;
    if (second) b[1] = row;
  }
  const int trow = min(max(row, kZoomRowLo), kZoomRowLo + kZoomRows - 1) - kZoomRowLo;
  const float4* wt[2];
  wt[1] = wtab + trow * zoom_row_stride(2, nphy, GROUPS, NT) + phy.z * (2 * GROUPS * NT);
  wt[0] = wt[1] + GROUPS * NT;
  const float* tp = tile + lby * PW + lbx;
  const float4* pp = pw + lby * PW + lbx;
  float res[2][P], mirror[2][P], hi[2][P], lo[2][P], hi2[2][P], lo2[2][P];
#pragma unroll
  for (int o = 0; o < 2; ++o)
#pragma unroll
    for (int c = 0; c < P; ++c) res[o][c] = mirror[o][c] = hi[o][c] = lo[o][c] = hi2[o][c] = lo2[o][c] = 0.f;
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    __builtin_amdgcn_sched_barrier(0);  // one group's weights live at a time
    float4 w4[2][NT];
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int j = 0; j < NT; ++j) w4[o][j] = wt[o][g * NT + j];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int p = 4 * g + k;
      if (p >= HALF) continue;
      if (AR) __builtin_amdgcn_sched_barrier(0);  // one tap pair's samples and powers live at a time
      const int q = N * N - 1 - p;
      const int ip = p % N * PW + p / N, iq = q % N * PW + q / N;
#pragma unroll
      for (int c = 0; c < P; ++c) {
        const float lp = tp[c * PN + ip], lq = tp[c * PN + iq];
        float4 a, b;
        if (AR) {
          a = pp[c * PN + ip];
          b = pp[c * PN + iq];
        }
#pragma unroll
        for (int o = 0; o < 2; ++o) {
          auto w = [&](int j) { return k == 0 ? w4[o][j].x : (k == 1 ? w4[o][j].y : (k == 2 ? w4[o][j].z : w4[o][j].w)); };
          res[o][c] = fmaf(lp, w(0), res[o][c]);
          mirror[o][c] = fmaf(lq, w(1), mirror[o][c]);
          if constexpr (AR) {
            hi[o][c] = fmaf(b.x, w(3), fmaf(a.x, w(2), hi[o][c]));
            lo[o][c] = fmaf(b.y, w(3), fmaf(a.y, w(2), lo[o][c]));
            hi2[o][c] = fmaf(b.z, w(3), fmaf(a.z, w(2), hi2[o][c]));
            lo2[o][c] = fmaf(b.w, w(3), fmaf(a.w, w(2), lo2[o][c]));
          }
        }
      }
    }
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int c = 0; c < P; ++c) {
        asm volatile("" : "+v"(res[o][c]), "+v"(mirror[o][c]));
        if (AR) asm volatile("" : "+v"(hi[o][c]), "+v"(lo[o][c]), "+v"(hi2[o][c]), "+v"(lo2[o][c]));
      }
  }
  const int esz_out = elem_bytes(io.out_dt);
  char* ob = static_cast<char*>(frame_out(io, f));
#pragma unroll
  for (int c = 0; c < P; ++c) {
    float v[2];
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      const float sum = res[o][c] + mirror[o][c];
      v[o] = AR ? zoom_ring(sum, hi[o][c], lo[o][c], hi2[o][c], lo2[o][c]) : fminf(fmaxf(sum, 0.f), 1.f);
    }
    void* dst = ob + c * io.out_cstride * esz_out;
    const int64_t at = static_cast<int64_t>(oy) * io.out_pitch + ox;
    if (first && second) {
      store_pair(dst, at, io.out_dt, v[0], v[1]);
    } else {
      if (first) store_elem(dst, at, io.out_dt, v[0]);
      if (second) store_elem(dst, at + 1, io.out_dt, v[1]);
    }
  }
}

template <int T>
static hipError_t launch_zoom_tile(int r, bool ar, int channels, const Io& io, const __half* lut,
                                   const __half* lut_ar, const ZoomPlan& zp, int out_w, int out_h, hipStream_t st) {
  constexpr int TX = kZoomTiles[T].w, TY = kZoomTiles[T].h;
  const dim3 grid(((out_w + TX - 1) / TX) * ((out_h + TY - 1) / TY) * io.batch), block(TX * TY);
  const float4* wtab = reinterpret_cast<const float4*>(zp.wtab);
  // Width scaled by exactly 2 (any height whose phases fit the table): two outputs per thread,
  // faster for every variant from 640 x 360 up (the kernel's comment has the figures).
  const bool pair = zp.wtab && zp.nphx == 2 && out_w == 2 * io.W;
  const dim3 pairs(((io.W + TX) / TX) * ((out_h + TY - 1) / TY) * io.batch);
#define MPX_ZOOM(R, A, CH)                                                                                   \
  if (r == R && ar == A && channels == CH) {                                                                 \
    if (pair)                                                                                                \
      hipLaunchKernelGGL((ravu_zoom_pair_kernel<R, A, CH, TX, TY>), pairs, block, 0, st, io, wtab, zp.nphy,  \
                         zp.phase, out_w, out_h);                                                            \
    else if (zp.wtab)                                                                                        \
      hipLaunchKernelGGL((ravu_zoom_kernel<R, A, CH, true, TX, TY>), grid, block, 0, st, io, lut, lut_ar, wtab, \
                         zp.nphx, zp.nphy, zp.phase, out_w, out_h);                                          \
    else                                                                                                     \
      hipLaunchKernelGGL((ravu_zoom_kernel<R, A, CH, false, TX, TY>), grid, block, 0, st, io, lut, lut_ar,    \
                         nullptr, 0, 0, zp.phase, out_w, out_h);                                             \
    return hipGetLastError();                                                                                \
  }
  MPX_ZOOM(2, false, 0) MPX_ZOOM(2, false, 1) MPX_ZOOM(2, false, 2) MPX_ZOOM(3, false, 0) MPX_ZOOM(3, false, 1)
  MPX_ZOOM(3, false, 2) MPX_ZOOM(2, true, 0) MPX_ZOOM(2, true, 1) MPX_ZOOM(2, true, 2) MPX_ZOOM(3, true, 0)
  MPX_ZOOM(3, true, 1) MPX_ZOOM(3, true, 2)
#undef MPX_ZOOM
  return hipErrorInvalidValue;
}

hipError_t launch_ravu_zoom(int r, bool ar, int channels, const Io& io, const __half* lut, const __half* lut_ar,
                            const ZoomPlan& zp, int out_w, int out_h, int tile, hipStream_t st) {
  if (!zp.phase) return hipErrorInvalidValue;
  static_assert(kZoomTileCount == 2, "one case per tile shape");
  switch (tile) {
    case 0: return launch_zoom_tile<0>(r, ar, channels, io, lut, lut_ar, zp, out_w, out_h, st);
    case 1: return launch_zoom_tile<1>(r, ar, channels, io, lut, lut_ar, zp, out_w, out_h, st);
    default: return hipErrorInvalidValue;
  }
}

int zoom_plan_create(mpx_ctx* ctx, mpx_plan* plan, int in_w, int in_h, int out_w, int out_h) {
  ZoomPlan& zp = plan->zoom;
  zp = ZoomPlan{};
  const int nphx = out_w / std::gcd(in_w, out_w), nphy = out_h / std::gcd(in_h, out_h);
  {
    const size_t pbytes = static_cast<size_t>(out_w + out_h) * sizeof(int4);
    void* pp = nullptr;
    if (int rc = ctx->alloc(pbytes, &pp)) return rc;
    mpx_host::DeviceScope ds;
    hipError_t e = hipErrorInvalidDevice;
    if (!ds.enter(ctx->device)) {
      hipLaunchKernelGGL(zoom_phase_kernel, dim3((out_w + out_h + 255) / 256), dim3(256), 0, nullptr,
                         static_cast<int4*>(pp), in_w, in_h, out_w, out_h, nphx, nphy);
      e = hipGetLastError();
      if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
    }
    if (e != hipSuccess) {
      ctx->release(pp, pbytes);
      return mpx_host::fail(MPX_ERR_HIP, std::string("ravu-zoom phase table: ") + hipGetErrorString(e));
    }
    zp.phase = static_cast<int4*>(pp);
    zp.phase_bytes = pbytes;
  }
  if (static_cast<int64_t>(nphx) * nphy > kZoomMaxPhasePairs) return MPX_OK;  // per-pixel interpolation
  const int r = plan->v->radius;
  const bool ar = plan->v->ar != 0;
  const int groups = (2 * r * 2 * r / 2 + 3) / 4;
  const int entries = kZoomRows * nphy * nphx * groups;
  const size_t bytes = static_cast<size_t>(kZoomRows) * zoom_row_stride(nphx, nphy, groups, ar ? 4 : 2) * sizeof(float4);
  void* p = nullptr;
  if (ctx->alloc(bytes, &p)) return MPX_OK;  // over the budget: per-pixel interpolation
  mpx_host::DeviceScope ds;
  int rc;
  if ((rc = ds.enter(ctx->device))) {
    ctx->release(p, bytes);
    zoom_plan_destroy(ctx, plan);
    return rc;
  }
  const dim3 grid((entries + 255) / 256);
  float4* tab = static_cast<float4*>(p);
  if (r == 2 && !ar)
    hipLaunchKernelGGL((zoom_table_kernel<2, false>), grid, dim3(256), 0, nullptr, plan->lut, plan->lut_ar, tab, in_w,
                       in_h, out_w, out_h, nphx, nphy);
  else if (r == 2)
    hipLaunchKernelGGL((zoom_table_kernel<2, true>), grid, dim3(256), 0, nullptr, plan->lut, plan->lut_ar, tab, in_w,
                       in_h, out_w, out_h, nphx, nphy);
  else if (!ar)
    hipLaunchKernelGGL((zoom_table_kernel<3, false>), grid, dim3(256), 0, nullptr, plan->lut, plan->lut_ar, tab, in_w,
                       in_h, out_w, out_h, nphx, nphy);
  else
    hipLaunchKernelGGL((zoom_table_kernel<3, true>), grid, dim3(256), 0, nullptr, plan->lut, plan->lut_ar, tab, in_w,
                       in_h, out_w, out_h, nphx, nphy);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
  if (e != hipSuccess) {
    ctx->release(p, bytes);
    zoom_plan_destroy(ctx, plan);
    return mpx_host::fail(MPX_ERR_HIP, std::string("ravu-zoom weight table: ") + hipGetErrorString(e));
  }
  zp.wtab = static_cast<float*>(p);
  zp.wtab_bytes = bytes;
  zp.nphx = nphx;
  zp.nphy = nphy;
  return MPX_OK;
}

void zoom_plan_destroy(mpx_ctx* ctx, mpx_plan* plan) {
  ctx->release(plan->zoom.wtab, plan->zoom.wtab_bytes);
  ctx->release(plan->zoom.phase, plan->zoom.phase_bytes);
  plan->zoom = ZoomPlan{};
}

}  // namespace mpx
