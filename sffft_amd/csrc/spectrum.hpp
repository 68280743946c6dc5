// Filter spectra in the convolution kernels' orders, in one launch up to N = 2L = 16384: a
// workgroup reads its filter rows (the zero-padded half is never stored or loaded), transforms
// them in LDS with the standalone transform's stages (transforms.hpp: fp64, complex64 between
// the stages, the same bits) and writes them in the plan's order.
//
// Padding to complex rows, transforming and gathering as three launches moved every
// spectrum over memory three times (write, read and write, read and write, of 16L bytes a
// channel); here it is written once. One row per workgroup (N/16 lanes) from N = 1024 on, so that
// a few hundred channels give every CU several rows at different stages; bound by the fp64
// stages and their barriers (VALU 20 to 42% busy, 1.4 to 1.9 TB/s). Measured, three
// launches and this kernel: spectrum_impl (api.hip).
#pragma once
#include "transforms.hpp"

namespace sffft {

// The order of a channel's N spectrum values, as pairs of consecutive values (float4 f of the
// channel's row): the frequency `s` of the first, the step `ds` to that of the second, whether the
// values are stored conjugated, or none (zero padding of the Hermitian halves). The digits are
// those of spectrum_permute_kernel and spectrum_half_kernel (api.hip), with shifts for the
// radices 2^l0, 2^l1, 2^l2.
struct SpectrumOrder {
  int mode, half;        // half: the Hermitian half of a wave plan (mode 1)
  int l0, l1, l2;
  float scale, iscale;   // of the real and imaginary parts
};
struct SpectrumPair {
  int s, ds;
  bool conj, none;
};
__host__ __device__ inline SpectrumPair spectrum_pair(const SpectrumOrder& o, int f) {
  const int r0 = 1 << o.l0;
  if (o.mode == 1 && o.half) {
    // f / pitch for the pitches 9, 17, 33 and f < 1122: the reciprocal rounded up to 16 bits is exact
    const int pitch = (8 << (o.l1 - 4)) + 1, cols = r0 / 2 + 1;
    if (f >= cols * pitch) return {0, 0, false, true};
    const int k0 = (f * ((65536 + pitch - 1) / pitch)) >> 16, rem = f - k0 * pitch;
    if (rem == pitch - 1) return {0, 0, false, true};
    const int g = rem & 3, q = (rem >> 2) & 1, kt = rem >> 3, k1 = 16 * kt + 4 * g + 2 * q;
    const bool mid = k0 == r0 / 2;
    return {k0 + r0 * (mid ? (1 << o.l1) - 1 - k1 : k1), mid ? -r0 : r0, mid, false};
  }
  if (o.mode == 0) {
    const int lane = (f >> 1) & 63, rest = f >> 7, c = lane & 15, g = lane >> 4, v = 2 * (f & 1);
    const int t1 = o.l1 - 4, t2 = o.l2 - 4;
    if (o.l2 == 0) {
      const int mt = rest & ((1 << t1) - 1);
      return {16 * (rest >> t1) + c + r0 * (16 * mt + 4 * g + v), r0, false, false};
    }
    const int mt = rest & ((1 << t2) - 1), t = (rest >> t2) & ((1 << t1) - 1), k0 = rest >> (t1 + t2);
    return {k0 + ((16 * t + c) << o.l0) + ((16 * mt + 4 * g + v) << (o.l0 + o.l1)), 1 << (o.l0 + o.l1), false, false};
  }
  // wave order (whole) of the plan, or of the row plan r1 x r2 of a multi-pass plan's row
  const int a = o.mode == 2 ? o.l1 : o.l0, b = o.mode == 2 ? o.l2 : o.l1, lrow = o.mode == 2 ? a + b : 31;
  const int row = o.mode == 2 ? (2 * f) >> lrow : 0, w = o.mode == 2 ? f & ((1 << (lrow - 1)) - 1) : f;
  const int lane = w & 63, rest = w >> 6, q = rest & 1, tile = rest >> 1, c = lane & 15, g = lane >> 4;
  const int k0 = 16 * (tile >> (b - 4)) + c, k1 = 16 * (tile & ((1 << (b - 4)) - 1)) + 4 * g + 2 * q;
  const int s = k0 + (k1 << a), up = o.mode == 2 ? o.l0 : 0;
  return {row + (s << up), 1 << (a + up), false, false};
}

// The first stage's line of a zero-padded row, x[t] = k[inner + sJ t] for t < 8 and 0 above:
// line_dft whose first radix-2 level has nothing to add, and for a real row no imaginary part. The
// rounding steps that remain are line_dft's.
template <bool CPLX>
__device__ __forceinline__ void padded_line_dft(double (&vr)[16], double (&vi)[16]) {
#pragma clang fp contract(off)
  constexpr double c16[5] = {1.0, 0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.0};
  double ar[2][8], ai[2][8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const double xr = vr[j], xi = CPLX ? vi[j] : 0.0;
    const double c = j <= 4 ? c16[j] : -c16[8 - j], sn = -(j <= 4 ? c16[4 - j] : c16[j - 4]);
    ar[0][j] = xr;
    ai[0][j] = xi;
    if (j == 0) {
      ar[1][j] = xr;
      ai[1][j] = xi;
    } else if (j == 4) {
      ar[1][j] = xi;
      ai[1][j] = -xr;
    } else if (CPLX) {
      ar[1][j] = fma(xr, c, -(xi * sn));
      ai[1][j] = fma(xr, sn, xi * c);
    } else {
      ar[1][j] = xr * c;
      ai[1][j] = xr * sn;
    }
  }
  // the remaining levels: two 8-point transforms, each in bit-reversed order
#pragma unroll
  for (int o = 0; o < 2; o++) {
    xf::line_dft<8>(ar[o], ai[o], -1);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      vr[8 * o + j] = ar[o][j];
      vi[8 * o + j] = ai[o][j];
    }
  }
}

// Lanes: one radix-16 line each, at least a wavefront.
template <int N>
struct SpectrumGeom {
  static constexpr int THREADS = N / 16 < 64 ? 64 : N / 16, G = THREADS * 16 / N, SLOTS = G * N;
};

// Spectra of the rows kr[h][0..N/2) (+ i ki[h] with CPLX) into kf, rows of N/2 float4.
template <int N, bool CPLX>
__global__ void __launch_bounds__(SpectrumGeom<N>::THREADS)
    spectrum_rows_kernel(const float* __restrict__ kr, const float* __restrict__ ki, float4* __restrict__ kf, int H,
                         SpectrumOrder o) {
  typedef SpectrumGeom<N> SG;
  constexpr int R = xf::MAX_RADIX, sJ = N / R, L = N / 2;
  static_assert(R == 16 && N >= 32, "the first stage is a padded radix-16 line");
  __shared__ float2 buf[SG::SLOTS + SG::SLOTS / 16];
  __shared__ double tc[sJ], ts[sJ];
  const int g = threadIdx.x / sJ, inner = threadIdx.x % sJ, h0 = blockIdx.x * SG::G;
  // in flight while the table is evaluated; lanes past the last row repeat it
  float xr[8], xi[8];
  const size_t first = (size_t)(h0 + g < H ? h0 + g : H - 1) * L + inner;
#pragma unroll
  for (int t = 0; t < 8; t++) {
    xr[t] = kr[first + t * sJ];
    xi[t] = CPLX ? ki[first + t * sJ] : 0.f;
  }
  __asm__ volatile("" ::: "memory");
  // one sincospi per entry of the twiddle bases, as line_kernel evaluates them
  if (threadIdx.x < sJ) {
    double sn, c;
    sincospi(2.0 * (double)threadIdx.x / (double)N, &sn, &c);
    tc[threadIdx.x] = c;
    ts[threadIdx.x] = sn;
  }
  __syncthreads();
  {
    double vr[R], vi[R];
#pragma unroll
    for (int t = 0; t < 8; t++) {
      vr[t] = (double)xr[t];
      vi[t] = (double)xi[t];
    }
    padded_line_dft<CPLX>(vr, vi);
    xf::twiddled_outputs_w<R>(vr, vi, tc[inner], -ts[inner],
                              [&](int k, float2 v) { buf[xf::lpad(g * N + inner + k * sJ)] = v; });
  }
  __syncthreads();
  xf::line_stage<N, N / R, SG::G, SG::THREADS>(buf, tc, ts, -1, 1.f);
  for (int i = threadIdx.x; i < SG::SLOTS / 2; i += SG::THREADS) {
    const int row = i / L, f = i - row * L;
    if (h0 + row >= H) break;
    const SpectrumPair p = spectrum_pair(o, f);
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (!p.none) {
      const float2 a = buf[xf::lpad(row * N + xf::line_position<N>(p.s))];
      const float2 b = buf[xf::lpad(row * N + xf::line_position<N>(p.s + p.ds))];
      v = make_float4(a.x * o.scale, (p.conj ? -a.y : a.y) * o.iscale, b.x * o.scale,
                      (p.conj ? -b.y : b.y) * o.iscale);
    }
    kf[(size_t)(h0 + row) * L + f] = v;
  }
}

constexpr int SPECTRUM_ROWS_MAX_N = xf::ONEPASS_MAX_N;

template <int N>
inline void launch_spectrum_rows(const float* kr, const float* ki, float4* kf, int H, const SpectrumOrder& o,
                                 hipStream_t s) {
  const dim3 grid((unsigned)((H + SpectrumGeom<N>::G - 1) / SpectrumGeom<N>::G)), block(SpectrumGeom<N>::THREADS);
  if (ki)
    hipLaunchKernelGGL((spectrum_rows_kernel<N, true>), grid, block, 0, s, kr, ki, kf, H, o);
  else
    hipLaunchKernelGGL((spectrum_rows_kernel<N, false>), grid, block, 0, s, kr, ki, kf, H, o);
}

// false: not a length of this kernel
inline bool run_spectrum_rows(const float* kr, const float* ki, float4* kf, int H, int N, const SpectrumOrder& o,
                              hipStream_t s) {
  switch (N) {
    case 256: launch_spectrum_rows<256>(kr, ki, kf, H, o, s); return true;
    case 512: launch_spectrum_rows<512>(kr, ki, kf, H, o, s); return true;
    case 1024: launch_spectrum_rows<1024>(kr, ki, kf, H, o, s); return true;
    case 2048: launch_spectrum_rows<2048>(kr, ki, kf, H, o, s); return true;
    case 4096: launch_spectrum_rows<4096>(kr, ki, kf, H, o, s); return true;
    case 8192: launch_spectrum_rows<8192>(kr, ki, kf, H, o, s); return true;
    case 16384: launch_spectrum_rows<16384>(kr, ki, kf, H, o, s); return true;
    default: return false;
  }
}

}  // namespace sffft
