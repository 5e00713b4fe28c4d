// RAVU (full, 2x with three predictions) and RAVU-3x, luma / yuv / rgb.
//
// RAVU-3x (compute/ravu-3x-r3.hook:22-163): one thread per input pixel, 3x3 output block
// (centre = input pixel), 24x3x3 buckets, two LUT texels per tap.
// RAVU (ravu-r3.hook:15-437): kernel 1 predicts int11 (x+1/2, y+1/2) from the 2r x 2r
// window into an FP32 scratch plane; kernel 2 predicts int10 (x+1/2, y) and then int01
// (x, y+1/2) on the 45-degree lattice mixing the input and int11, from one staging of
// both tiles, and writes the interleaved 2x output (the combine pass, :426-437), each
// prediction with the output row it completes.  All read LDS tiles staged with
// clamp-to-edge halos, each texture clamped on its own size as mpv's sampler does.
//
// Channel forms (ravu-r3-yuv.hook, ravu-r3-rgb.hook): the hash sees plane 0 (yuv) or
// the BT.709 luma (rgb, `dot(rgb, vec3(0.2126, 0.7152, 0.0722))`); taps apply to all
// three planes with the same weights.
#include "common.h"
#include "launch.h"
#include "ravu.h"

namespace mpx {

// Tiles: TX x TY pixels per block of TX * TY threads, one input pixel (3x) or site (full
// RAVU; two in the pair form of step 1) per thread, from the families' shape lists (k3xTiles,
// kRavuTiles).  Full RAVU's halo is up to 9 rows, so its tiles are taller than 3x's.


// Stage P planes of a frame into LDS: tile[c][r][col] = plane c at
// (clamp(ox + col), clamp(oy + r)), PH x PW per plane; all loads in flight at once.
template <int P, int PH, int PW, int NT>
__device__ __forceinline__ void stage_planes(float* tile, const void* base, int dt, float in_max, float in_rmax,
                                             int64_t pitch, int64_t cstride, int W, int H, int ox, int oy) {
  HaloTile<P, PH, PW, NT> h;
  __builtin_amdgcn_s_setprio(1);  // the loads go out ahead of other waves' arithmetic
  h.issue(base, dt, pitch, cstride, W, H, ox, oy);
  __builtin_amdgcn_s_setprio(0);
  h.commit(tile, dt, in_max, in_rmax, W, ox);
}

// Floats staged per tile sample: the P input planes and, for rgb, the FP64 BT.709 luma that the
// hash reads, in the room of two planes behind them (luma_plane).
template <int CH>
constexpr int staged_planes() { return CH == 0 ? 1 : (CH == 1 ? 3 : 5); }

// rgb: fill the luma of a staged tile (n samples per plane); the caller synchronises the block
// before and after.
template <int CH, int NT>
__device__ __forceinline__ void stage_luma(float* t, int n) {
  if constexpr (CH == 2) {
    fill_luma<NT>(t, reinterpret_cast<double*>(t + 3 * n), n, n);
  }
}

// The samples that the hash sees of a staged tile (plane stride n), at the offsets of its planes.
template <int CH>
__device__ __forceinline__ const HashSample<CH>* luma_plane(const float* t, int n) {
  if constexpr (CH == 2) return reinterpret_cast<const double*>(t + 3 * n);
  else return t;
}

// Whether full RAVU r2 re-decides a wave's near sites together (wave_tensor), as r3 and r4 do,
// or each lane its own: its 16 points are soon done, and several of its lanes are near at once
// (r2 luma together: 99.1 -> 131.9 us); only rgb, whose samples are 8 bytes, is a little faster
// together (2 x 1080p 129.4, alone 132.0).
template <int CH>
constexpr bool wave_redecide() { return CH == 2; }

// Hash of the site whose N x N window starts at staged-tile offset o (sample i at
// o + (i % N) * PW + i / N), with the FP64 re-decision out of line: it is rare, and inlined
// its registers (the double atan2 alone takes 56) would set the occupancy of every wave
// (r2 luma step1).  Its register budget follows its callers' (the kernel asks
// for 6 waves per SIMD), so it takes the lean tensor form to stay out of scratch.
template <int N, bool FIVE, int RULE, int CH, int PW, int PN>
__device__ __attribute__((noinline)) Bucket redecide_site(const float* t, int o) {
  double a, b, d;
  const auto l = lds_samples(luma_plane<CH>(t, PN)) + o;
  structure_tensor_fp64<N, FIVE, true>([&](int s) { return l[s % N * PW + s / N]; }, a, b, d);
  return hash_reference<RULE, double>(a, b, d);
}
// Hash of this lane's step-1 site; all lanes of the wave together.
template <int N, int CH, int PW, int PN>
__device__ __forceinline__ Bucket hash_site(const float* t, int o, bool valid) {
  const auto* l = luma_plane<CH>(t, PN);
  auto sample = [&](int s) { return l[o + s % N * PW + s / N]; };
  if constexpr (wave_redecide<CH>()) {
    return ravu_hash_wave<N, true, RULE_LOG2, kWaveSites>(valid, sample, o, [&](int at) {
      const auto w = lds_samples(l) + at;
      return [w](int X, int Y) { return w[Y * PW + X]; };
    });
  } else {
    float a, b, d;
    structure_tensor<N, true>(sample, a, b, d);
    bool near = false;
    const Bucket bk = hash_fast<RULE_LOG2>(a, b, d, &near);
    return near && valid ? redecide_site<N, true, RULE_LOG2, CH, PW, PN>(t, o) : bk;
  }
}

// ----------------------------------------------------------------------------- RAVU-3x

template <int R, int CH, int TX, int TY>
__global__ __launch_bounds__(TX * TY) void ravu_3x_kernel(Io io, const __half* __restrict__ lut, int total) {
  constexpr int P = CH == 0 ? 1 : 3;
  constexpr int N = 2 * R - 1;
  constexpr int HALO = R - 1;
  constexpr int PW = staged_width(TX + 2 * HALO), PH = TY + 2 * HALO, PN = PW * PH;
  constexpr int C = (N * N - 1) / 2;
  constexpr int NTEX = 2 * (C + 1);
  __shared__ __attribute__((aligned(16))) float tile[staged_planes<CH>() * PN];
  const FrameTile ft = frame_tile<TX, TY>(io, blockIdx.x, total);
  const int f = ft.f;
  const int x0 = ft.x0, y0 = ft.y0;
  const void* in = frame_in(io, f);
  stage_planes<P, PH, PW, TX * TY>(tile, in, io.in_dt, io.in_max, io.in_rmax, ft.in_pitch, ft.in_cstride, ft.W, ft.H, x0 - HALO, y0 - HALO);
  __syncthreads();
  if constexpr (CH == 2) {
    stage_luma<CH, TX * TY>(tile, PN);
    __syncthreads();
  }
  const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
  const int x = x0 + tx, y = y0 + ty;
  if (x >= ft.W || y >= ft.H) return;
  auto off = [&](int i) { return (ty + i % N) * PW + tx + i / N; };  // sample i = X*N + Y
  const auto* lum = luma_plane<CH>(tile, PN);
  const Bucket bk = ravu_hash<N, false, RULE_3X>([&](int i) { return lum[off(i)]; });
  const int row = bucket_row<RULE_3X>(bk, 216);
  if (io.buckets) io.buckets[f * io.bucket_bstride + static_cast<int64_t>(y) * ft.W + x] = row;
  const __half* lrow = lut + static_cast<int64_t>(row) * NTEX * 4;
  float r0[P][4], r1[P][4];
#pragma unroll
  for (int c = 0; c < P; ++c)
#pragma unroll
    for (int k = 0; k < 4; ++k) r0[c][k] = r1[c][k] = 0.f;
  // One step per tap pair (two LUT texels), software-pipelined: texels are fetched (as raw
  // FP16, converted inside the multiply-adds) three steps ahead, and each step's sums
  // complete before the next step's samples are read, so only one step's operands are live.
  const uint2* lraw = reinterpret_cast<const uint2*>(lrow);
  constexpr int AHEAD = 3;
  uint2 q0[AHEAD], q1[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) {
    q0[i] = lraw[2 * min(i, C)];
    q1[i] = lraw[2 * min(i, C) + 1];
  }
#pragma unroll
  for (int i = 0; i <= C; ++i) {
    __builtin_amdgcn_sched_barrier(0);
    const uint2 t0 = q0[i % AHEAD], t1 = q1[i % AHEAD];
    if (i + AHEAD <= C) {
      q0[i % AHEAD] = lraw[2 * (i + AHEAD)];
      q1[i % AHEAD] = lraw[2 * (i + AHEAD) + 1];
    }
    const __half2 h00 = bits_h2(t0.x), h01 = bits_h2(t0.y), h10 = bits_h2(t1.x), h11 = bits_h2(t1.y);
    const float a0[4] = {__low2float(h00), __high2float(h00), __low2float(h01), __high2float(h01)};
    const float a1[4] = {__low2float(h10), __high2float(h10), __low2float(h11), __high2float(h11)};
#pragma unroll
    for (int c = 0; c < P; ++c) {
      const float li = tile[c * PN + off(i)];
      if (i < C) {
        const float lj = tile[c * PN + off(N * N - 1 - i)];
        // res0 += l_i*w0 + l_j*w1.wzyx, res1 += l_i*w1 + l_j*w0.wzyx, as four fused
        // multiply-adds (the LUT operand converts inside them, v_fma_mix)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          r0[c][k] = fmaf(lj, a1[3 - k], fmaf(li, a0[k], r0[c][k]));
          r1[c][k] = fmaf(lj, a0[3 - k], fmaf(li, a1[k], r1[c][k]));
        }
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          r0[c][k] = fmaf(li, a0[k], r0[c][k]);
          r1[c][k] = fmaf(li, a1[k], r1[c][k]);
        }
      }
    }
#pragma unroll
    for (int c = 0; c < P; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) asm volatile("" : "+v"(r0[c][k]), "+v"(r1[c][k]));
  }
  const int esz_out = elem_bytes(io.out_dt);
  char* ob = static_cast<char*>(frame_out(io, f));
#pragma unroll
  for (int c = 0; c < P; ++c) {
    void* o = ob + c * ft.out_cstride * esz_out;
    const float centre = tile[c * PN + off(C)];
#pragma unroll
    for (int dy = 0; dy < 3; ++dy)
#pragma unroll
      for (int dx = 0; dx < 3; ++dx) {
        const int k = 3 * dx + dy;  // compute/ravu-3x-r3.hook:154-162
        float v = k < 4 ? r0[c][k] : (k == 4 ? centre : r1[c][k - 5]);
        if (k != 4) v = fminf(fmaxf(v, 0.f), 1.f);
        store_elem(o, static_cast<int64_t>(3 * y + dy) * ft.out_pitch + 3 * x + dx, io.out_dt, v);
      }
  }
}

template <int T>
static hipError_t launch_3x_tile(int r, int channels, Io io, const __half* lut, hipStream_t st) {
  constexpr int TX = k3xTiles[T].w, TY = k3xTiles[T].h;
  const int total = launch_tiles<TX, TY>(io);
#define MPX_3X(R, CH)                                                                                  \
  if (r == R && channels == CH) {                                                                      \
    hipLaunchKernelGGL((ravu_3x_kernel<R, CH, TX, TY>), dim3(total), dim3(TX * TY), 0, st, io, lut, total); \
    return hipGetLastError();                                                                          \
  }
  MPX_3X(2, 0) MPX_3X(2, 1) MPX_3X(2, 2) MPX_3X(3, 0) MPX_3X(3, 1) MPX_3X(3, 2) MPX_3X(4, 0) MPX_3X(4, 1) MPX_3X(4, 2)
#undef MPX_3X
  return hipErrorInvalidValue;
}

hipError_t launch_ravu_3x(int r, int channels, const Io& io, const __half* lut, int tile, hipStream_t st) {
  static_assert(k3xTileCount == 2, "one case per tile shape");
  switch (tile) {
    case 0: return launch_3x_tile<0>(r, channels, io, lut, st);
    case 1: return launch_3x_tile<1>(r, channels, io, lut, st);
    default: return hipErrorInvalidValue;
  }
}

// ----------------------------------------------------------------------------- RAVU full

// res = sum_{p < N^2/2} (s_p + s_{N^2-1-p}) * w_p, w_p = texel p/4, component p%4,
// clamped to [0,1] (ravu-r3.hook:120-146).  s(c, i) = plane c sample i.
template <int N> struct RavuLut {
  static constexpr int NTEX = (N * N / 2 + 3) / 4;  // texels per LUT row: 2 / 5 / 8 for r2 / r3 / r4
};

template <int N, int P, typename S>
__device__ __forceinline__ void ravu_taps(const __half* lrow, S s, float* res) {
#pragma unroll
  for (int c = 0; c < P; ++c) res[c] = 0.f;
#pragma unroll
  for (int t = 0; t < RavuLut<N>::NTEX; ++t) {
    // large windows (r4: 64 samples per plane): one LUT texel's taps at a time, so the
    // loads of all samples are not hoisted together (register pressure, hence occupancy;
    // small windows lose by it)
    if constexpr (N * N * P >= 64) __builtin_amdgcn_sched_barrier(0);
    const float4 w = load_lut4(lrow, t);
    const float a[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int p = 4 * t + j;
      if (p < N * N / 2) {
#pragma unroll
        for (int c = 0; c < P; ++c) res[c] += (s(c, p) + s(c, N * N - 1 - p)) * a[j];
      }
    }
    // ... and this texel's sums complete before the next texel's loads: without this the
    // multiply-adds sink below every load and all N*N*P samples are live at once (r4 yuv
    // lattice: 216 VGPRs, 2 waves per SIMD; with it 128, 4 waves)
    if constexpr (N * N * P >= 64) {
#pragma unroll
      for (int c = 0; c < P; ++c) asm volatile("" : "+v"(res[c]));
    }
  }
#pragma unroll
  for (int c = 0; c < P; ++c) res[c] = fminf(fmaxf(res[c], 0.f), 1.f);
}

// step1 for r2: int11 from the N = 2R window at offsets -(R-1)..R (ravu-r3.hook:22-146).
template <int R, int CH, int TX, int TY>
__global__ __launch_bounds__(TX * TY) __attribute__((amdgpu_waves_per_eu(6))) void ravu_step1_kernel(Io io, const __half* __restrict__ lut, float* int11,
                                                         int64_t int11_frame, int total) {
  constexpr int P = CH == 0 ? 1 : 3;
  constexpr int N = 2 * R;
  constexpr int PW = staged_width(TX + N - 1), PH = TY + N - 1, PN = PW * PH;
  __shared__ __attribute__((aligned(16))) float tile[staged_planes<CH>() * PN];
  const FrameTile ft = frame_tile<TX, TY>(io, blockIdx.x, total);
  const int f = ft.f;
  const int x0 = ft.x0, y0 = ft.y0;
  const void* in = frame_in(io, f);
  stage_planes<P, PH, PW, TX * TY>(tile, in, io.in_dt, io.in_max, io.in_rmax, ft.in_pitch, ft.in_cstride, ft.W, ft.H, x0 - (R - 1),
                  y0 - (R - 1));
  __syncthreads();
  if constexpr (CH == 2) {
    stage_luma<CH, TX * TY>(tile, PN);
    __syncthreads();
  }
  const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
  const int x = x0 + tx, y = y0 + ty;
  const bool valid = x < ft.W && y < ft.H;
  auto off = [&](int i) { return (ty + i % N) * PW + tx + i / N; };
  const Bucket bk = hash_site<N, CH, PW, PN>(tile, off(0), valid);
  if (!valid) return;
  const int row = bucket_row<RULE_LOG2>(bk, 648);
  if (io.buckets) io.buckets[f * io.bucket_bstride + static_cast<int64_t>(y) * ft.W + x] = row;
  float res[P];
  ravu_taps<N, P>(lut + static_cast<int64_t>(row) * RavuLut<N>::NTEX * 4,
                  [&](int c, int i) { return tile[c * PN + off(i)]; }, res);
  const int64_t plane = static_cast<int64_t>(ft.W) * ft.H;
  float* o = int11 + f * int11_frame + static_cast<int64_t>(y) * ft.W + x;
#pragma unroll
  for (int c = 0; c < P; ++c) o[c * plane] = io.store16 ? static_cast<float>(static_cast<_Float16>(res[c])) : res[c];
}

// Lattice position of sample (X, Y) of step 2 (int10, centre (x+1/2, y)) / step 3
// (int01, centre (x, y+1/2)): sample at centre + (X-(N-1)/2)*(1/2,-1/2) + (Y-(N-1)/2)*(1/2,1/2)
// (ravu-r3.hook:155-191, 289-325).  Returns doubled coordinates.
template <int N, int STEP>
__device__ __host__ constexpr int lat2x(int X, int Y) { return STEP == 2 ? X + Y - N + 2 : X + Y - N + 1; }
template <int N, int STEP>
__device__ __host__ constexpr int lat2y(int X, int Y) { return STEP == 2 ? Y - X : Y - X + 1; }

// FP64 samples of a step 2 / 3 window, `at` = offset of the site in the staged input (px and
// py have the same parity; the int11 tile follows the input's).  It keeps the window's lowest
// address, so the reads' offsets are non-negative immediates (otherwise the addresses are
// registers of their own).
// (`lum`: the samples that the hash sees of the input; int11's are NEXT further.)
template <int N, int STEP, int PW, int NEXT, typename T>
struct LatticeWindow {
  static constexpr int LOW = N / 2 * (PW + 1);
  LdsSamples<T> t;
  __device__ __forceinline__ LatticeWindow(const T* lum, int at) : t(lds_samples(lum) + at - LOW) {}
  __device__ __forceinline__ T operator()(int X, int Y) const {
    const int px = lat2x<N, STEP>(X, Y), py = lat2y<N, STEP>(X, Y);
    return t[LOW + (py >> 1) * PW + (px >> 1) + (px & 1) * NEXT];
  }
};

// One site's step 2 (int10, STEP = 2) or step 3 (int01, STEP = 3) on the lattice, and
// the combine for one output row: STEP 2 writes row 2y = (input, int10) pairs, STEP 3
// row 2y+1 = (int01, int11) pairs (ravu-r3.hook:426-437), so each step stores contiguous
// pairs.  hk / i11: the staged input and int11 tiles, base: the site's LDS offset.
template <int R, int CH, int STEP, int PW, int PN>
__device__ __forceinline__ void lattice_site(const Io& io, const __half* __restrict__ lut, const float* hk,
                                             const float* i11, int base, const FrameTile& ft, int x, int y,
                                             bool valid, int64_t plane) {
  constexpr int P = CH == 0 ? 1 : 3;
  constexpr int N = 2 * R;
  auto src = [&](int i) -> const float* {
    const int X = i / N, Y = i % N;
    const int px = lat2x<N, STEP>(X, Y), py = lat2y<N, STEP>(X, Y);
    return (px & 1) ? i11 + base + ((py - 1) >> 1) * PW + ((px - 1) >> 1) : hk + base + (py >> 1) * PW + (px >> 1);
  };
  auto sample = [&](int i) {
    const int px = lat2x<N, STEP>(i / N, i % N), py = lat2y<N, STEP>(i / N, i % N);
    return (px & 1) ? luma_plane<CH>(i11, PN)[base + ((py - 1) >> 1) * PW + ((px - 1) >> 1)]
                    : luma_plane<CH>(hk, PN)[base + (py >> 1) * PW + (px >> 1)];
  };
  Bucket bk;
  if constexpr (wave_redecide<CH>()) {
    bk = ravu_hash_wave<N, true, RULE_LOG2, kWaveSites>(valid, sample, base, [&](int o) {
      constexpr int NEXT = staged_planes<CH>() * PN * static_cast<int>(sizeof(float)) / static_cast<int>(sizeof(HashSample<CH>));
      return LatticeWindow<N, STEP, PW, NEXT, HashSample<CH>>(luma_plane<CH>(hk, PN), o);
    });
  } else {
    bk = ravu_hash<N, true, RULE_LOG2, true>(sample);
  }
  if (!valid) return;
  const int row = bucket_row<RULE_LOG2>(bk, 648);
  if (io.buckets)
    io.buckets[ft.f * io.bucket_bstride + (STEP - 1) * plane + static_cast<int64_t>(y) * ft.W + x] = row;
  float res[P];
  ravu_taps<N, P>(lut + static_cast<int64_t>(row) * RavuLut<N>::NTEX * 4, [&](int c, int i) { return src(i)[c * PN]; },
                  res);
  const int esz_out = elem_bytes(io.out_dt);
  char* ob = static_cast<char*>(frame_out(io, ft.f));
#pragma unroll
  for (int c = 0; c < P; ++c) {
    void* o = ob + c * ft.out_cstride * esz_out;
    if (STEP == 2)
      store_pair(o, static_cast<int64_t>(2 * y) * ft.out_pitch + 2 * x, io.out_dt, hk[c * PN + base], res[c]);
    else
      store_pair(o, static_cast<int64_t>(2 * y + 1) * ft.out_pitch + 2 * x, io.out_dt, res[c], i11[c * PN + base]);
  }
}

// Steps 2 and 3 of a tile for r2: both read the same staged input and int11 tiles (lattice
// offsets -R..R), so one kernel stages them once and runs the two steps one after the
// other per site; a scheduling barrier between them keeps one step's registers live at a
// time.
template <int R, int CH, int TX, int TY>
__global__ __launch_bounds__(TX * TY) void ravu_lattice_kernel(Io io, const __half* __restrict__ lut,
                                                           const float* __restrict__ int11, int64_t int11_frame,
                                                           int total) {
  constexpr int P = CH == 0 ? 1 : 3;
  constexpr int PW = staged_width(TX + 2 * R + 1), PH = TY + 2 * R + 1, PN = PW * PH;  // offsets -R..R
  __shared__ __attribute__((aligned(16))) float tiles[2][staged_planes<CH>() * PN];
  float *hk = tiles[0], *i11 = tiles[1];  // input (HOOKED), ravu_int11
  const FrameTile ft = frame_tile<TX, TY>(io, blockIdx.x, total);
  const int f = ft.f;
  const int x0 = ft.x0, y0 = ft.y0;
  const void* in = frame_in(io, f);
  const int64_t plane = static_cast<int64_t>(ft.W) * ft.H;
  {
    HaloTile<P, PH, PW, TX * TY> a, b;  // both tiles' loads in flight together
    __builtin_amdgcn_s_setprio(1);  // the loads go out ahead of other waves' arithmetic
    a.issue(in, io.in_dt, ft.in_pitch, ft.in_cstride, ft.W, ft.H, x0 - R, y0 - R);
    b.issue(int11 + f * int11_frame, DT_F32, ft.W, plane, ft.W, ft.H, x0 - R, y0 - R);
    __builtin_amdgcn_s_setprio(0);
    a.commit(hk, io.in_dt, io.in_max, io.in_rmax, ft.W, x0 - R);
    b.commit(i11, DT_F32, 1.f, 1.f, ft.W, x0 - R);
  }
  __syncthreads();
  if constexpr (CH == 2) {
    stage_luma<CH, TX * TY>(hk, PN);
    stage_luma<CH, TX * TY>(i11, PN);
    __syncthreads();
  }
  const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
  const int x = x0 + tx, y = y0 + ty;
  const bool valid = x < ft.W && y < ft.H;
  const int base = (ty + R) * PW + tx + R;  // LDS offset of (x, y)
  lattice_site<R, CH, 2, PW, PN>(io, lut, hk, i11, base, ft, x, y, valid, plane);
  __builtin_amdgcn_sched_barrier(0);
  lattice_site<R, CH, 3, PW, PN>(io, lut, hk, i11, base, ft, x, y, valid, plane);
}

// ----------------------------------------------------------------------------- separable tensor
//
// The structure tensor's Gaussian is a product of its two axes, and the derivative along X
// (Y) depends on a point's X (Y) index only through its stencil: central at the grid's first
// and last index, five-point between (N = 6, 8).  So the sums over Y of one window column,
//   A_t = sum_Y g(Y) gx_t^2,  B_t = sum_Y g(Y) c(Y) gx_t gy,  D = sum_Y g(Y) c(Y)^2 gy^2
// for both stencils t of gx (unscaled derivatives, c = the stencil's scale) are shared by
// the M = N - 2 windows that hold the column; a block tabulates them once in LDS and a site adds
// M table entries per sum:
//   a = sum_X g(X) c(X)^2 A_t(X),  b = sum_X g(X) c(X) B_t(X),  d = sum_X g(X) D.
// Bound by VALU issue: the M^2 points evaluated per site took 358 instructions (r4), the table
// and its sums take about 130 (with the shared tap columns: r4 4 x 1080p 292.6 -> 213.7 us, r4-yuv
// 2 x 1080p 223.7 -> 195.9, r3 4 x 1080p 178.9 -> 163.7).  r2's window has border stencils at
// every second point, so its columns would share too little: it keeps the sums per site.  The
// order of the sums is free, as every decision within its error margin is re-made in FP64.
template <int N>
struct SepTensor {
  static_assert(N == 6 || N == 8, "one inner and one outer stencil");
  static constexpr int M = N - 2;  // grid positions 1 .. N - 2 of the window
  __device__ static constexpr bool five(int i) { return i >= 1 && i + 3 <= M + 1; }  // grid index i = position i + 1
  __device__ static constexpr double c(int i) { return five(i) ? 1.0 / 12.0 : 0.5; }
  __device__ static constexpr double g(int i) {  // 1-D weight: the normalised grid's row sum
    double s = 0;
    for (int j = 0; j < M; ++j) s += gauss_w<N>(i * M + j);
    return s;
  }
  // whether some of RUN successive columns sums uses stencil `f` of gy at row r of the run
  template <int RUN>
  __device__ static constexpr bool uses(bool f, int r) {
    for (int k = 0; k < RUN; ++k)
      if (r - k >= 0 && r - k < M && five(r - k) == f) return true;
    return false;
  }

  struct Column {
    float2 c, f;  // (A, B) for the central and the five-point gx
    float d;
  };
  // Columns sums of RUN successive windows along Y: s(dx, dy) is the sample dx, dy steps from the
  // first window's first grid row.
  template <int RUN, typename S>
  __device__ __forceinline__ static void columns(S s, Column (&out)[RUN]) {
#pragma unroll
    for (int k = 0; k < RUN; ++k) out[k] = {{0.f, 0.f}, {0.f, 0.f}, 0.f};
#pragma unroll
    for (int r = 0; r < M + RUN - 1; ++r) {
      const float xc = difference(s(1, r), s(-1, r));
      const float xf = fmaf(8.0f, xc, difference(s(-2, r), s(2, r)));
      const float yc = difference(s(0, r + 1), s(0, r - 1));
      float yf = 0.f;
      if (uses<RUN>(true, r)) yf = fmaf(8.0f, yc, difference(s(0, r - 2), s(0, r + 2)));
      const float xc2 = xc * xc, xf2 = xf * xf;
      const float cc = xc * yc, fc = xf * yc, yc2 = yc * yc;
      const float cf = xc * yf, ff = xf * yf, yf2 = yf * yf;
#pragma unroll
      for (int k = 0; k < RUN; ++k) {
        const int i = r - k;
        if (i < 0 || i >= M) continue;
        const float w = static_cast<float>(g(i)), wc = static_cast<float>(g(i) * c(i));
        const float wcc = static_cast<float>(g(i) * c(i) * c(i));
        out[k].c.x = fmaf(w, xc2, out[k].c.x);
        out[k].f.x = fmaf(w, xf2, out[k].f.x);
        out[k].c.y = fmaf(wc, five(i) ? cf : cc, out[k].c.y);
        out[k].f.y = fmaf(wc, five(i) ? ff : fc, out[k].f.y);
        out[k].d = fmaf(wcc, five(i) ? yf2 : yc2, out[k].d);
      }
    }
  }
  // a, b, d of one site: ab(five, X) returns the (A, B) entry of grid index X, dd(X) its D
  template <typename AB, typename DD>
  __device__ __forceinline__ static void site(AB ab, DD dd, float& a, float& b, float& d) {
    a = b = d = 0.f;
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const float2 e = ab(five(i), i);
      a = fmaf(static_cast<float>(g(i) * c(i) * c(i)), e.x, a);
      b = fmaf(static_cast<float>(g(i) * c(i)), e.y, b);
      d = fmaf(static_cast<float>(g(i)), dd(i), d);
    }
  }
};

// Floats of the tables' LDS (tn entries of five).  rgb: the FP64 lumas (n of them) from which the sums
// are taken live there first, the tables then take their place, and a block with near sites
// fills them in again for the re-decision.  With both kept at once r3-rgb's kernels had 16 waves
// per compute unit instead of 24.
template <int CH>
constexpr int table_floats(int tn, int n) { return CH == 2 && 2 * n > 5 * tn ? 2 * n : 5 * tn; }
template <int CH>
__device__ __forceinline__ const HashSample<CH>* hash_samples(const float* tile, const float* tab) {
  if constexpr (CH == 2) return reinterpret_cast<const double*>(tab);
  else return tile;
}

// Weight p (texel p / 4, component p % 4) of a LUT row held raw.
template <int NTEX>
struct RawRow {
  uint2 t[NTEX];
  __device__ __forceinline__ explicit RawRow(const __half* row) {
    const uint2* r = reinterpret_cast<const uint2*>(row);
#pragma unroll
    for (int i = 0; i < NTEX; ++i) t[i] = r[i];
  }
  __device__ __forceinline__ float w(int p) const {
    const __half2 h = bits_h2(p % 4 < 2 ? t[p / 4].x : t[p / 4].y);
    return p % 2 ? __high2float(h) : __low2float(h);
  }
};

__device__ __forceinline__ float clamp01(float v) { return fminf(fmaxf(v, 0.f), 1.f); }

// step1 for r3 / r4, two vertically neighbouring sites per thread (TX x TY sites, TX * TY / 2
// threads): the tap windows share N of their N + 1 rows, so a pair reads N (N + 1) samples
// per plane from LDS instead of 2 N^2 (r4 yuv: LDS was busy 57 of 107 us).
template <int R, int CH, int TX, int TY>
__global__ __launch_bounds__(TX * TY / 2) __attribute__((amdgpu_waves_per_eu(4))) void ravu_step1_pair_kernel(
    Io io, const __half* __restrict__ lut, float* int11, int64_t int11_frame, int total) {
  constexpr int P = CH == 0 ? 1 : 3;
  constexpr int N = 2 * R, NT = TX * TY / 2;
  constexpr int PW = staged_width(TX + N - 1), PH = TY + N - 1, PN = PW * PH;
  using Sep = SepTensor<N>;
  constexpr int RUN = 4, NC = TX + Sep::M - 1;  // table columns: staged columns 1 .. NC
  constexpr int RUNS = NC * (TY / RUN), TN = NC * TY;
  static_assert(TY % RUN == 0 && RUNS <= NT, "whole runs, one per thread");
  __shared__ __attribute__((aligned(16))) float tile[P * PN];
  __shared__ __attribute__((aligned(16))) float tab[table_floats<CH>(TN, PN)];
  float2 *tc = reinterpret_cast<float2*>(tab), *tf = tc + TN;
  float* td = reinterpret_cast<float*>(tf + TN);
  const FrameTile ft = frame_tile<TX, TY>(io, blockIdx.x, total);
  const int f = ft.f;
  const int x0 = ft.x0, y0 = ft.y0;
  stage_planes<P, PH, PW, NT>(tile, frame_in(io, f), io.in_dt, io.in_max, io.in_rmax, ft.in_pitch, ft.in_cstride,
                              ft.W, ft.H, x0 - (R - 1), y0 - (R - 1));
  __syncthreads();
  const HashSample<CH>* lum = hash_samples<CH>(tile, tab);
  if constexpr (CH == 2) {
    fill_luma<NT>(tile, reinterpret_cast<double*>(tab), PN, PN);
    __syncthreads();
  }
  {
    const int i = threadIdx.x, q = i / NC, c = i - q * NC;
    typename Sep::Column v[RUN];
    if (i < RUNS) {
      const auto* p = lum + (q * RUN + 1) * PW + c + 1;
      Sep::template columns<RUN>([&](int dx, int dy) { return p[dy * PW + dx]; }, v);
    }
    if constexpr (CH == 2) __syncthreads();  // the tables take the lumas' place
    if (i < RUNS) {
#pragma unroll
      for (int k = 0; k < RUN; ++k) {
        const int e = (q * RUN + k) * NC + c;
        tc[e] = v[k].c;
        tf[e] = v[k].f;
        td[e] = v[k].d;
      }
    }
  }
  __syncthreads();
  const int tx = threadIdx.x % TX, ty = threadIdx.x / TX * 2;
  const int x = x0 + tx, y = y0 + ty;
  const bool valid = x < ft.W && y < ft.H, second = y + 1 < ft.H;
  const int o = ty * PW + tx;
  int row[2] = {0, 0};
  bool near[2];
  auto decide = [&](int s, Bucket& bk) {
    redecide<N, true, RULE_LOG2, kWaveSites>(near[s], o, [&](int at) {
      const auto w = lds_samples(lum) + at + s * PW;
      return [w](int X, int Y) { return w[Y * PW + X]; };
    }, bk);
    if (CH != 2 || near[s]) row[s] = bucket_row<RULE_LOG2>(bk, 648);
  };
  auto report = [&](int s) {
    if (io.buckets && valid && (s == 0 || second))
      io.buckets[f * io.bucket_bstride + static_cast<int64_t>(y + s) * ft.W + x] = row[s];
  };
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int e = (ty + s) * NC + tx;
    float a, b, d;
    Sep::site([&](bool five, int i) { return five ? tf[e + i] : tc[e + i]; }, [&](int i) { return td[e + i]; }, a, b, d);
    Bucket bk = hash_fast<RULE_LOG2>(a, b, d, &near[s]);
    near[s] = near[s] && valid && (s == 0 || second);
    if constexpr (CH == 2) {
      row[s] = bucket_row<RULE_LOG2>(bk, 648);
    } else {
      decide(s, bk);
      report(s);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (CH == 2) {
    if (__syncthreads_or(near[0] || near[1])) {
      fill_luma<NT>(tile, reinterpret_cast<double*>(tab), PN, PN);
      __syncthreads();
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        Bucket bk{};
        decide(s, bk);
      }
    }
    report(0);
    report(1);
  }
  if (!valid) return;
  constexpr int NTEX = RavuLut<N>::NTEX;
  const RawRow<NTEX> w0(lut + row[0] * (NTEX * 4)), w1(lut + row[1] * (NTEX * 4));
  const int64_t plane = static_cast<int64_t>(ft.W) * ft.H;
  float* out = int11 + f * int11_frame + static_cast<int64_t>(y) * ft.W + x;
  // res = sum over p < N^2/2 of (s_p + s_{N^2-1-p}) w_p, in order (ravu-r3.hook:120-146)
#pragma unroll
  for (int c = 0; c < P; ++c) {
    const float* p = tile + c * PN + o;
    float r0 = 0.f, r1 = 0.f;
#pragma unroll
    for (int X = 0; X < N / 2; ++X) {
      __builtin_amdgcn_sched_barrier(0);  // one column pair's samples live at a time
      float l[N + 1], h[N + 1];
#pragma unroll
      for (int Y = 0; Y <= N; ++Y) {
        l[Y] = p[Y * PW + X];
        h[Y] = p[Y * PW + N - 1 - X];
      }
#pragma unroll
      for (int Y = 0; Y < N; ++Y) {
        r0 = fmaf(l[Y] + h[N - 1 - Y], w0.w(X * N + Y), r0);
        r1 = fmaf(l[Y + 1] + h[N - Y], w1.w(X * N + Y), r1);
      }
      asm volatile("" : "+v"(r0), "+v"(r1));
    }
    r0 = clamp01(r0);
    r1 = clamp01(r1);
    out[c * plane] = io.store16 ? static_cast<float>(static_cast<_Float16>(r0)) : r0;
    if (second) out[c * plane + ft.W] = io.store16 ? static_cast<float>(static_cast<_Float16>(r1)) : r1;
  }
}

// Steps 2 and 3 for r3 / r4.  Lattice column L of pixel (x, y) holds the samples
// (x + (L + Y - N + 2) / 2, y + (Y - L) / 2), Y = 0 .. N - 1; step 2's window is columns
// 0 .. N - 1 and step 3's is columns -1 .. N - 2 (lat2x, lat2y), so the two share all but one.
// The column sums of the tensor are tabulated by the column's first grid point (Y = 1): an
// input pixel (i, j) for odd L, an int11 site (i + 1/2, j + 1/2) for even L, the next point
// along Y; one thread sums the pair.
template <int R, int CH, int TX, int TY>
__global__ __launch_bounds__(TX * TY) void ravu_lattice_pair_kernel(Io io, const __half* __restrict__ lut,
                                                                    const float* __restrict__ int11,
                                                                    int64_t int11_frame, int total) {
  constexpr int P = CH == 0 ? 1 : 3;
  constexpr int N = 2 * R, NT = TX * TY;
  constexpr int PW = staged_width(TX + 2 * R + 1), PH = TY + 2 * R + 1, PN = PW * PH;  // offsets -R..R
  using Sep = SepTensor<N>;
  constexpr int H = Sep::M / 2;
  // tables by int11 site (-H .. TX - 1, -H .. TY - 1) and input pixel (1-H .. TX - 1, 1-H .. TY - 1)
  constexpr int NC = TX + H, NR = TY + H, EC = NC - 1, ER = NR - 1, EN = EC * ER, TN = EN + NC * NR;
  __shared__ __attribute__((aligned(16))) float tiles[2][P * PN];
  float *hk = tiles[0], *i11 = tiles[1];  // input (HOOKED), ravu_int11
  __shared__ __attribute__((aligned(16))) float tab[table_floats<CH>(TN, 2 * PN)];
  float2 *tc = reinterpret_cast<float2*>(tab), *tf = tc + TN;  // input pixels' entries, then int11 sites'
  float* td = reinterpret_cast<float*>(tf + TN);
  const FrameTile ft = frame_tile<TX, TY>(io, blockIdx.x, total);
  const int f = ft.f;
  const int x0 = ft.x0, y0 = ft.y0;
  const int64_t plane = static_cast<int64_t>(ft.W) * ft.H;
  {
    HaloTile<P, PH, PW, NT> a, b;  // both tiles' loads in flight together
    __builtin_amdgcn_s_setprio(1);  // the loads go out ahead of other waves' arithmetic
    a.issue(frame_in(io, f), io.in_dt, ft.in_pitch, ft.in_cstride, ft.W, ft.H, x0 - R, y0 - R);
    b.issue(int11 + f * int11_frame, DT_F32, ft.W, plane, ft.W, ft.H, x0 - R, y0 - R);
    __builtin_amdgcn_s_setprio(0);
    a.commit(hk, io.in_dt, io.in_max, io.in_rmax, ft.W, x0 - R);
    b.commit(i11, DT_F32, 1.f, 1.f, ft.W, x0 - R);
  }
  __syncthreads();
  // the samples that the hash sees: the input's, then (NEXT further) int11's
  constexpr int NEXT = CH == 2 ? PN : P * PN;
  const HashSample<CH>* lum = hash_samples<CH>(hk, tab);
  auto lumas = [&] {
    fill_luma<NT>(hk, reinterpret_cast<double*>(tab), PN, PN);
    fill_luma<NT>(i11, reinterpret_cast<double*>(tab) + PN, PN, PN);
  };
  if constexpr (CH == 2) {
    lumas();
    __syncthreads();
  }
  {
    constexpr int E = (NC * NR + NT - 1) / NT;
    typename Sep::Column v[CH == 2 ? E : 1][2];
    auto sums = [&](int i, typename Sep::Column (&out)[2]) {
      const int q = i / NC, c = i - q * NC;
      const auto* p = lum + (q - H + R) * PW + c - H + R;  // input pixel (c - H, q - H)
      Sep::template columns<2>(
          [&](int dx, int dy) {  // lattice steps from that pixel
            const int u = dx + dy, w = dy - dx;
            return p[(u & 1) ? NEXT + ((w - 1) >> 1) * PW + ((u - 1) >> 1) : (w >> 1) * PW + (u >> 1)];
          },
          out);
    };
    auto put = [&](int i, const typename Sep::Column (&in)[2]) {
      const int q = i / NC, c = i - q * NC;
      if (q > 0 && c > 0) {
        const int e = (q - 1) * EC + c - 1;
        tc[e] = in[0].c;
        tf[e] = in[0].f;
        td[e] = in[0].d;
      }
      tc[EN + i] = in[1].c;
      tf[EN + i] = in[1].f;
      td[EN + i] = in[1].d;
    };
    if constexpr (CH == 2) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int i = static_cast<int>(threadIdx.x) + e * NT;
        if (i < NC * NR) sums(i, v[e]);
      }
      __syncthreads();  // the tables take the lumas' place
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int i = static_cast<int>(threadIdx.x) + e * NT;
        if (i < NC * NR) put(i, v[e]);
      }
    } else {
      for (int i = threadIdx.x; i < NC * NR; i += NT) {
        sums(i, v[0]);
        put(i, v[0]);
      }
    }
  }
  __syncthreads();
  const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
  const int x = x0 + tx, y = y0 + ty;
  const bool valid = x < ft.W && y < ft.H;
  const int base = (ty + R) * PW + tx + R;  // LDS offset of (x, y)
  const int ee = (ty + H - 1) * EC + tx + H - 1, oe = EN + (ty + H) * NC + tx + H;  // table entries of (x, y)
  // table entry of column L (0 .. M): input pixel (x + (L - N + 3) / 2, y + (1 - L) / 2) for odd
  // L, int11 site (x + (L - N + 2) / 2, y - L / 2) for even L
  auto entry = [&](int L) {
    return L & 1 ? ee + (L - N + 3) / 2 + (1 - L) / 2 * EC : oe + (L - N + 2) / 2 - L / 2 * NC;
  };
  auto src = [&](int L, int Y) -> const float* {
    const int px = L + Y - N + 2, py = Y - L;
    return (px & 1) ? i11 + base + ((py - 1) >> 1) * PW + ((px - 1) >> 1) : hk + base + (py >> 1) * PW + (px >> 1);
  };
  int row[2];
  bool near[2];
  auto decide = [&](int s, Bucket& bk) {
    if (s == 0)
      redecide<N, true, RULE_LOG2, kWaveSites>(
          near[s], base, [&](int o) { return LatticeWindow<N, 2, PW, NEXT, HashSample<CH>>(lum, o); }, bk);
    else
      redecide<N, true, RULE_LOG2, kWaveSites>(
          near[s], base, [&](int o) { return LatticeWindow<N, 3, PW, NEXT, HashSample<CH>>(lum, o); }, bk);
    if (CH != 2 || near[s]) row[s] = bucket_row<RULE_LOG2>(bk, 648);
  };
  auto report = [&](int s) {
    if (io.buckets && valid)
      io.buckets[f * io.bucket_bstride + (s + 1) * plane + static_cast<int64_t>(y) * ft.W + x] = row[s];
  };
#pragma unroll
  for (int s = 0; s < 2; ++s) {  // step 2, step 3: grid index i is column i + 1, i
    float a, b, d;
    Sep::site([&](bool five, int i) {
          return five ? tf[entry(i + 1 - s)] : tc[entry(i + 1 - s)];
        },
        [&](int i) { return td[entry(i + 1 - s)]; }, a, b, d);
    Bucket bk = hash_fast<RULE_LOG2>(a, b, d, &near[s]);
    near[s] = near[s] && valid;
    if constexpr (CH == 2) {
      row[s] = bucket_row<RULE_LOG2>(bk, 648);
    } else {
      decide(s, bk);
      report(s);
    }
    __builtin_amdgcn_sched_barrier(0);  // one step's registers live at a time
  }
  if constexpr (CH == 2) {
    if (__syncthreads_or(near[0] || near[1])) {
      lumas();
      __syncthreads();
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        Bucket bk{};
        decide(s, bk);
      }
    }
    report(0);
    report(1);
  }
  if (!valid) return;
  constexpr int NTEX = RavuLut<N>::NTEX;
  const RawRow<NTEX> w2(lut + row[0] * (NTEX * 4)), w3(lut + row[1] * (NTEX * 4));
  const int esz_out = elem_bytes(io.out_dt);
  char* ob = static_cast<char*>(frame_out(io, f));
#pragma unroll
  for (int c = 0; c < P; ++c) {
    // step 2 pairs columns (X, N-1-X), step 3 (X-1, N-2-X): each column is read once for both
    float r2 = 0.f, r3 = 0.f, below[N], high[N];
#pragma unroll
    for (int Y = 0; Y < N; ++Y) {
      below[Y] = src(-1, Y)[c * PN];
      high[Y] = src(N - 1, Y)[c * PN];
    }
#pragma unroll
    for (int X = 0; X < N / 2; ++X) {
      __builtin_amdgcn_sched_barrier(0);
      float low[N], next[N];
#pragma unroll
      for (int Y = 0; Y < N; ++Y) {
        low[Y] = src(X, Y)[c * PN];
        next[Y] = X + 1 < N / 2 ? src(N - 2 - X, Y)[c * PN] : low[Y];
      }
#pragma unroll
      for (int Y = 0; Y < N; ++Y) {
        r2 = fmaf(low[Y] + high[N - 1 - Y], w2.w(X * N + Y), r2);
        r3 = fmaf(below[Y] + next[N - 1 - Y], w3.w(X * N + Y), r3);
      }
      asm volatile("" : "+v"(r2), "+v"(r3));
#pragma unroll
      for (int Y = 0; Y < N; ++Y) {
        below[Y] = low[Y];
        high[Y] = next[Y];
      }
    }
    void* o = ob + c * ft.out_cstride * esz_out;
    const int64_t at = static_cast<int64_t>(2 * y) * ft.out_pitch + 2 * x;
    // the combine pass (ravu-r3.hook:426-437): rows (input, int10) and (int01, int11)
    store_pair(o, at, io.out_dt, hk[c * PN + base], clamp01(r2));
    store_pair(o, at + ft.out_pitch, io.out_dt, clamp01(r3), i11[c * PN + base]);
  }
}

template <int T>
static hipError_t launch_ravu_tile(int r, int channels, Io io, const __half* lut, float* int11, int64_t int11_frame,
                                   hipStream_t st, hipEvent_t done) {
  constexpr int TX = kRavuTiles[T].w, TY = kRavuTiles[T].h;
  const int total = launch_tiles<TX, TY>(io);
  const dim3 grid(total), block(TX * TY);
#define MPX_RAVU(R, CH)                                                                                            \
  if (r == R && channels == CH) {                                                                                  \
    if constexpr (R >= 3)                                                                                          \
      hipLaunchKernelGGL((ravu_step1_pair_kernel<R, CH, TX, TY>), grid, dim3(TX * TY / 2), 0, st, io, lut, int11,   \
                         int11_frame, total);                                                                      \
    else                                                                                                           \
      hipLaunchKernelGGL((ravu_step1_kernel<R, CH, TX, TY>), grid, block, 0, st, io, lut, int11, int11_frame, total); \
    hipError_t e = hipGetLastError();                                                                              \
    if (e != hipSuccess) return e;                                                                                 \
    if constexpr (R >= 3)                                                                                          \
      return launch_done(ravu_lattice_pair_kernel<R, CH, TX, TY>, grid, block, st, done, io, lut, int11,            \
                         int11_frame, total);                                                                      \
    else                                                                                                           \
      return launch_done(ravu_lattice_kernel<R, CH, TX, TY>, grid, block, st, done, io, lut, int11, int11_frame,    \
                         total);                                                                                   \
  }
  MPX_RAVU(2, 0) MPX_RAVU(2, 1) MPX_RAVU(2, 2) MPX_RAVU(3, 0) MPX_RAVU(3, 1) MPX_RAVU(3, 2) MPX_RAVU(4, 0)
  MPX_RAVU(4, 1) MPX_RAVU(4, 2)
#undef MPX_RAVU
  return hipErrorInvalidValue;
}

hipError_t launch_ravu(int r, int channels, const Io& io, const __half* lut, float* int11, int64_t int11_frame,
                       int tile, hipStream_t st, hipEvent_t done) {
  static_assert(kRavuTileCount == 3, "one case per tile shape");
  switch (ravu_tile_index(r, channels, tile)) {
    case 0: return launch_ravu_tile<0>(r, channels, io, lut, int11, int11_frame, st, done);
    case 1: return launch_ravu_tile<1>(r, channels, io, lut, int11, int11_frame, st, done);
    case 2: return launch_ravu_tile<2>(r, channels, io, lut, int11, int11_frame, st, done);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace mpx
