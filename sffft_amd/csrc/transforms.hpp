// Standalone complex transforms and the 2-D circular convolution built on them.
//
// The reference lists standalone forward/inverse FFTs and 2-D convolution as not
// exposed (README.md:174); these have no counterpart there. They favour accuracy over
// speed: each stage is a radix-R DFT along one digit of the position, evaluated in fp64
// (an in-register radix-2 FFT of the R points per thread, fp64 twiddles) and stored as
// complex64 between stages (relative error ~1e-7). The fused convolution kernels, with
// fp16 MFMA operands, are separate.
//
// Algorithm: N = r[0] * r[1] * ... * r[S-1] (powers of two, 16s first). Decimation in
// frequency: stage J transforms digit J (stride s_J = r[J+1] * ... * r[S-1]) and, before
// the next stage, multiplies by w_{r[J] s_J}^(k_J * (p mod s_J)). After the last stage
// position p = sum_J k_J s_J holds frequency k = k_0 + r[0] (k_1 + r[1] (k_2 + ...)), so
// the last stage writes each value to its natural-order slot directly. Contiguous sequences
// of up to ONEPASS_MAX_N points run every stage in LDS in one launch (line_kernel); longer
// or strided ones take one launch per stage (stage_kernel), through a workspace.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace sffft {
namespace xf {

constexpr int MAX_RADIX = 16;
constexpr int MAX_STAGES = 6;
constexpr long long MAX_N = 1LL << 24;
constexpr long long MAX_ELEMS = 1LL << 31;  // sequences * N per call

constexpr bool stages_cover_max_n() {
  long long n = 1;
  for (int i = 0; i < MAX_STAGES; i++) n *= MAX_RADIX;
  return n >= MAX_N;
}
static_assert(stages_cover_max_n(), "MAX_STAGES stages of MAX_RADIX must reach MAX_N");

struct Radices {
  int S;
  int r[MAX_STAGES];
};

// N a power of two in [2, 2^24]: radix-MAX_RADIX stages, then the remainder.
inline bool split(long long N, Radices* out) {
  if (N < 2 || N > MAX_N || (N & (N - 1))) return false;
  Radices d{0, {1, 1, 1, 1, 1, 1}};
  long long rest = N;
  while (rest > MAX_RADIX) {
    if (d.S == MAX_STAGES - 1) return false;  // never write past r[MAX_STAGES - 1]
    d.r[d.S++] = MAX_RADIX;
    rest /= MAX_RADIX;
  }
  d.r[d.S++] = (int)rest;
  *out = d;
  return true;
}

// Element n of sequence s sits at (s / inner) * dist_outer + (s % inner) * dist_inner +
// n * stride (complex elements). seq_fast: consecutive threads take consecutive
// sequences (set when sequences interleave more tightly than their elements, as the
// columns of a row-major matrix do), and the stage workspace is then laid out [p][s]
// so that every stage reads and writes consecutive addresses across a wavefront.
struct Seqs {
  long long nseq, inner, dist_inner, dist_outer, stride;
  int seq_fast;
  __host__ __device__ long long base(long long s) const {
    return (s / inner) * dist_outer + (s % inner) * dist_inner;
  }
};

// x with its sign flipped where neg (0 or INT_MIN) says so
__device__ __forceinline__ double flip(double x, int neg) {
  return __hiloint2double(__double2hiint(x) ^ neg, __double2loint(x));
}

// The radix-R DFT of one line's R points, in registers, shared by all kernels below:
// radix-2 decimation in frequency over log2(R) levels, natural input order, bit-reversed
// output order, in fp64, exponents of the given sign. The 16th roots of unity are constants
// (scalar registers; from an LDS table they took 32 VGPRs and the reads), the sign goes into their
// sines on the scalar unit, and the quarter turn is a swap. About R*log2(R)/2 complex products
// instead of the R*R of the dense sum. Contraction is off and the complex products are written
// with fma, so every kernel that inlines this rounds in the same places and gets the same bits.
template <int R>
__device__ __forceinline__ void line_dft(double (&vr)[R], double (&vi)[R], int sign) {
#pragma clang fp contract(off)
  static_assert(R <= 16, "16th roots");
  constexpr double c16[5] = {1.0, 0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.0};
  const int neg = sign < 0 ? (int)0x80000000 : 0;
#pragma unroll
  for (int m = R; m >= 2; m >>= 1) {
    const int h = m >> 1, step = 16 / m;
#pragma unroll
    for (int b = 0; b < R; b += m)
#pragma unroll
      for (int j = 0; j < h; j++) {
        const int i0 = b + j, i1 = i0 + h, t = j * step;  // times w_16^t, t < 8
        const double ar = vr[i0], ai = vi[i0], dr = ar - vr[i1], di = ai - vi[i1];
        vr[i0] = ar + vr[i1];
        vi[i0] = ai + vi[i1];
        if (t == 0) {
          vr[i1] = dr;
          vi[i1] = di;
        } else if (t == 4) {
          vr[i1] = flip(-di, neg);
          vi[i1] = flip(dr, neg);
        } else {
          const double c = t < 4 ? c16[t] : -c16[8 - t], sn = flip(t < 4 ? c16[4 - t] : c16[t - 4], neg);
          vr[i1] = fma(dr, c, -(di * sn));
          vi[i1] = fma(dr, sn, di * c);
        }
      }
  }
}

template <int R>
__device__ __forceinline__ int bitrev(int k) {
  int r = 0;
#pragma unroll
  for (int b = 1; b < R; b <<= 1) r = (r << 1) | ((k & b) ? 1 : 0);
  return r;
}

// Frequency digit k of a non-last stage's line times w_Nj^(k * inner), rounded to
// complex64 once; store(k, value) for k = 0 .. R-1. The twiddles are powers of
// w_Nj^inner = w1c + i w1s, built by recurrence in fp64 (same rounding rule as line_dft).
template <int R, class Store>
__device__ __forceinline__ void twiddled_outputs_w(const double (&vr)[R], const double (&vi)[R], double w1c,
                                                   double w1s, Store store) {
#pragma clang fp contract(off)
  double wr = 1.0, wi = 0.0;
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int r = bitrev<R>(k);
    store(k, make_float2((float)fma(vr[r], wr, -(vi[r] * wi)), (float)fma(vr[r], wi, vi[r] * wr)));
    const double nr = fma(wr, w1c, -(wi * w1s));
    wi = fma(wr, w1s, wi * w1c);
    wr = nr;
  }
}

// The same with w_Nj^inner evaluated here (one fp64 sincospi of the exact angle).
template <int R, class Store>
__device__ __forceinline__ void twiddled_outputs(const double (&vr)[R], const double (&vi)[R], int inner, int Nj,
                                                 int sign, Store store) {
  double w1s, w1c;
  sincospi(2.0 * (double)inner / (double)Nj, &w1s, &w1c);
  twiddled_outputs_w<R>(vr, vi, w1c, sign * w1s, store);
}

template <int R>
__global__ void __launch_bounds__(128)
    stage_kernel(const float2* in, float2* out, float2* work, Seqs q, Radices d, int J, int N, int sign,
                 float scale) {
  const int S = d.S;
  int sJ = 1;
  for (int i = J + 1; i < S; i++) sJ *= d.r[i];
  const int lines = N / R;
  const long long gid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= q.nseq * lines) return;
  const long long s = q.seq_fast ? gid % q.nseq : gid / lines;
  const int l = (int)(q.seq_fast ? gid / q.nseq : gid % lines);
  const int inner = l % sJ, outer = l / sJ;
  const int base = outer * R * sJ + inner;
  auto widx = [&](int p) -> long long { return q.seq_fast ? (long long)p * q.nseq + s : s * N + p; };
  float2 x[R];
  if (J == 0) {
    const float2* src = in + q.base(s);
#pragma unroll
    for (int t = 0; t < R; t++) x[t] = src[(long long)(base + t * sJ) * q.stride];
  } else {
#pragma unroll
    for (int t = 0; t < R; t++) x[t] = work[widx(base + t * sJ)];
  }
  const bool last = J == S - 1;
  // natural-order frequency of this line's first output (last stage: sJ = 1, inner = 0)
  long long kbase = 0, wlast = 1;
  if (last) {
    int sj = N;
    long long w = 1;
    for (int j = 0; j < S - 1; j++) {
      sj /= d.r[j];
      kbase += (long long)((base / sj) % d.r[j]) * w;
      w *= d.r[j];
    }
    wlast = w;
  }
  float2* dst = out + q.base(s);
  const int Nj = R * sJ;
  double vr[R], vi[R];
#pragma unroll
  for (int t = 0; t < R; t++) {
    vr[t] = (double)x[t].x;
    vi[t] = (double)x[t].y;
  }
  line_dft<R>(vr, vi, sign);
  if (last) {
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int r = bitrev<R>(k);
      dst[(kbase + (long long)k * wlast) * q.stride] = make_float2((float)(vr[r] * scale), (float)(vi[r] * scale));
    }
  } else {
    // twiddle w_Nj^(k * inner) before the next stage
    twiddled_outputs<R>(vr, vi, inner, Nj, sign, [&](int k, float2 v) { work[widx(base + k * sJ)] = v; });
  }
}

// ---- one pass over short contiguous lines ------------------------------------------
// Sequences of N <= ONEPASS_MAX_N elements at unit stride are transformed in one launch: a
// workgroup loads G = max(1, ONEPASS_SLOTS / N) whole sequences into LDS, runs every stage
// there and writes the natural-order result back, so each sequence crosses HBM once
// each way instead of once per stage. The stages are those of stage_kernel (the same
// radix split, fp64 line DFTs, twiddle recurrences and complex64 rounding between
// stages), so the results are bit-identical to the staged path. One LDS slot of padding
// per 16 elements keeps the threads of the last stage (R consecutive elements each) on
// different banks.
constexpr int ONEPASS_MAX_N = 16384;  // 136 KB of LDS
constexpr int ONEPASS_SLOTS = 4096;

__device__ __forceinline__ int lpad(int p) { return p + (p >> 4); }
// with EXTRA, one more slot per EXTRA elements
template <int EXTRA>
__device__ __forceinline__ int lpadx(int p) { return lpad(p) + (EXTRA ? p / (EXTRA ? EXTRA : 1) : 0); }

template <int N>
struct LineGeom {
  static constexpr int G = N >= ONEPASS_SLOTS ? 1 : ONEPASS_SLOTS / N;  // sequences per workgroup
  static constexpr int SLOTS = G * N;
  // one thread per radix-16 line: 256 threads, 512 at N = 8192, 1024 at N = 16384
  static constexpr int THREADS = SLOTS / MAX_RADIX;
  // The last stage takes its lines in the order of their frequencies, so that its stores are
  // contiguous; those lines start N / 16 elements apart, which a slot of padding each spreads over
  // the banks (N >= 4096: the shorter strides already fall on several).
  static constexpr int EXTRA = N >= 4096 ? N / 16 : 0;
  static constexpr int LDS = SLOTS + SLOTS / 16 + (EXTRA ? 16 : 0);
  // From N = 256 the first stage loads runs of 128 bytes and more straight into registers.
  static constexpr bool DIRECT = N >= 256;
  // Sequences of 8 and 16 points leave through LDS: a lane's stores of its own sequence, 64 and 128 bytes from
  // the next lane's, took 36.2 and 38.2 us for 2^23 points and 6.95 and 7.26 for 2^14; runs across the lanes 24.0,
  // 24.2, 5.14 and 5.11 (part of it the addresses, see line_kernel). Of 2 and 4 points the direct stores, 16 and
  // 32 bytes apart, take 22.2 and 25.9 for 2^23.
  static constexpr bool STAGED = N == 8 || N == 16;
  // twiddle bases of the non-last stages: w_N^j for j < N / 16 (w_Nj^inner = w_N^(inner N/Nj))
  static constexpr int TW = N / MAX_RADIX > 1 ? N / MAX_RADIX : 1;
  // radix of the stage whose remaining product of radices is REST (16s first)
  static constexpr int radix(int rest) { return rest > MAX_RADIX ? MAX_RADIX : rest; }
  static constexpr int last() {  // of the last stage
    int r = N;
    while (r > MAX_RADIX) r /= MAX_RADIX;
    return r;
  }
};

// Orders the workgroup's LDS accesses; global accesses stay in flight.
// The memory clobbers keep LDS reads above the barrier: the compiler's sinking of instructions to
// their use does not take s_barrier for a store.
__device__ __forceinline__ void lds_sync() {
  __asm__ volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  __asm__ volatile("" ::: "memory");
}

// The stages before the last one, from the one whose remaining product of radices is REST (REST =
// N at the first stage): R = 16, sJ = REST / R its stride, each followed by a barrier.
// tc, ts: the workgroup's table of w_N^j = tc[j] + i sign ts[j], j < N/16. A line's twiddle
// base w_REST^inner is entry inner * N/REST: sincospi of 2j/N there and of 2 inner/REST in
// the staged kernel are the same exact fp64 argument, so both paths get the same bits.
// G sequences of N in buf, THREADS threads (the one-pass kernel's geometry by default).
template <int N, int REST, int G = LineGeom<N>::G, int THREADS = LineGeom<N>::THREADS, int EXTRA = 0>
__device__ __forceinline__ void line_stages(float2* buf, const double* tc, const double* ts, int sign) {
  constexpr int R = LineGeom<N>::radix(REST), sJ = REST / R, LPS = N / R;
  if constexpr (sJ > 1) {
    for (int li = threadIdx.x; li < G * LPS; li += THREADS) {
      const int g = li / LPS, l = li - g * LPS;
      const int inner = l % sJ, base = g * N + (l / sJ) * REST + inner;
      double vr[R], vi[R];
#pragma unroll
      for (int t = 0; t < R; t++) {
        const float2 x = buf[lpadx<EXTRA>(base + t * sJ)];
        vr[t] = (double)x.x;
        vi[t] = (double)x.y;
      }
      line_dft<R>(vr, vi, sign);
      const int j = inner * (N / REST);
      twiddled_outputs_w<R>(vr, vi, tc[j], sign * ts[j],
                            [&](int k, float2 v) { buf[lpadx<EXTRA>(base + k * sJ)] = v; });
    }
    lds_sync();
    line_stages<N, REST / R, G, THREADS, EXTRA>(buf, tc, ts, sign);
  }
}

// All stages from REST on, the last one in place too, scaled: element base + k of a line holds its
// frequency digit k.
template <int N, int REST, int G = LineGeom<N>::G, int THREADS = LineGeom<N>::THREADS>
__device__ __forceinline__ void line_stage(float2* buf, const double* tc, const double* ts, int sign, float scale) {
  line_stages<N, REST, G, THREADS>(buf, tc, ts, sign);
  constexpr int R = LineGeom<N>::last(), LPS = N / R;
  for (int li = threadIdx.x; li < G * LPS; li += THREADS) {
    double vr[R], vi[R];
#pragma unroll
    for (int t = 0; t < R; t++) {
      const float2 x = buf[lpad(li * R + t)];
      vr[t] = (double)x.x;
      vi[t] = (double)x.y;
    }
    line_dft<R>(vr, vi, sign);
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int r = bitrev<R>(k);
      buf[lpad(li * R + k)] = make_float2((float)(vr[r] * scale), (float)(vi[r] * scale));
    }
  }
  lds_sync();
}

// Position in the line, after the last stage, of natural-order frequency f: the digits
// of f below the last stage's (f mod W, W the product of all radices but the last) name
// the line, reversed into its base position; the last digit is the element within it.
template <int N>
__device__ __forceinline__ int line_position(int f) {
  int W = 1, rest = N;
  while (rest > MAX_RADIX) {
    W *= MAX_RADIX;
    rest /= MAX_RADIX;
  }
  int kb = f % W, base = 0, sj = N;
  for (int w = 1; w < W; w *= MAX_RADIX) {
    sj /= MAX_RADIX;
    base += ((kb / w) % MAX_RADIX) * sj;
  }
  return base + f / W;
}

// Measured (768 x 16384, 1536 x 8192, 6144 x 2048, 49152 x 256): with the sequence staged through LDS
// on the way in and out and the roots of unity in LDS 97.5, 93, 83 and 71 us; this 64, 49, 40 and
// 35 (3.2 to 5.8 TB/s of calls on three inputs in turn; a copy 5.2). At N >= 8192 one or two workgroups fill a CU and the
// round trips to memory at either end of a sequence show. Workgroups that stay and request the next
// sequence while they transform one spill (18 to 22 VGPRs at 128) and took 76 and 77 us.
template <int N>
__global__ void __launch_bounds__(LineGeom<N>::THREADS)
    line_kernel(const float2* in, float2* out, Seqs q, int sign, float scale) {
  typedef LineGeom<N> LG;
  __shared__ float2 buf[LG::LDS];
  __shared__ double tc[LG::TW], ts[LG::TW];
  constexpr int R = LG::last(), LPS = N / R;
  const long long s0 = (long long)blockIdx.x * LG::G;
  const int G = q.nseq - s0 < LG::G ? (int)(q.nseq - s0) : LG::G;
  // run_lines' sequences lie at one distance: Seqs::base's 64-bit divisions, one for each element on the way in, took
  // 2.2 us of a small call (6.9 -> 4.7 at 4096 x 4) and 2 to 4 of 2^23 points
  auto base = [&](int g) { return (s0 + g) * q.dist_inner; };
  // the first stage's line of this lane: points inner + sJ t of sequence s0 + gt, in flight while
  // the tables are evaluated
  constexpr int sJ = LG::DIRECT ? N / MAX_RADIX : 1;
  const int gt = threadIdx.x / sJ, inner = threadIdx.x % sJ;
  float2 x[MAX_RADIX];
  if constexpr (LG::DIRECT) {
    // lanes past the last sequence repeat it and store nothing: a zero instead of the load, chosen
    // per point, became a branch and a wait per point
    const float2* src = in + base(gt < G ? gt : G - 1) + inner;
#pragma unroll
    for (int t = 0; t < MAX_RADIX; t++) x[t] = src[t * sJ];
    __asm__ volatile("" ::: "memory");
  }
  // one sincospi per table entry instead of one per line and stage
  for (int j = threadIdx.x; j < LG::TW; j += LG::THREADS) {
    double sn, c;
    sincospi(2.0 * (double)j / (double)N, &sn, &c);
    tc[j] = c;
    ts[j] = sn;
  }
  if constexpr (LG::DIRECT) {
    lds_sync();
    double vr[MAX_RADIX], vi[MAX_RADIX];
#pragma unroll
    for (int t = 0; t < MAX_RADIX; t++) {
      vr[t] = (double)x[t].x;
      vi[t] = (double)x[t].y;
    }
    line_dft<MAX_RADIX>(vr, vi, sign);
    twiddled_outputs_w<MAX_RADIX>(vr, vi, tc[inner], sign * ts[inner], [&](int k, float2 v) {
      buf[lpadx<LG::EXTRA>(gt * N + inner + k * sJ)] = v;
    });
    lds_sync();
    line_stages<N, N / MAX_RADIX, LG::G, LG::THREADS, LG::EXTRA>(buf, tc, ts, sign);
  } else {
    for (int i = threadIdx.x; i < LG::SLOTS; i += LG::THREADS) {
      const int g = i / N;
      buf[lpad(i)] = g < G ? in[base(g) + (i - g * N)] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    line_stages<N, N>(buf, tc, ts, sign);
  }
  // last stage, to memory: line kb of a sequence holds its frequencies kb + LPS k
  for (int li = threadIdx.x; li < LG::G * LPS; li += LG::THREADS) {
    const int g = li / LPS, kb = li - g * LPS, at = g * N + line_position<N>(kb);
    double vr[R], vi[R];
#pragma unroll
    for (int t = 0; t < R; t++) {
      const float2 v = buf[lpadx<LG::EXTRA>(at + t)];
      vr[t] = (double)v.x;
      vi[t] = (double)v.y;
    }
    line_dft<R>(vr, vi, sign);
    if constexpr (LG::STAGED) {
#pragma unroll
      for (int k = 0; k < R; k++) {
        const int r = bitrev<R>(k);
        buf[lpad(at + k)] = make_float2((float)(vr[r] * scale), (float)(vi[r] * scale));
      }
    } else if (g < G) {
      float2* dst = out + base(g) + kb;
#pragma unroll
      for (int k = 0; k < R; k++) {
        const int r = bitrev<R>(k);
        dst[k * LPS] = make_float2((float)(vr[r] * scale), (float)(vi[r] * scale));
      }
    }
  }
  if constexpr (LG::STAGED) {
    lds_sync();
    for (int i = threadIdx.x; i < G * N; i += LG::THREADS) out[base(i / N) + i % N] = buf[lpad(i)];
  }
}

template <int N>
inline void launch_line(const float2* in, float2* out, const Seqs& q, int sign, float scale, hipStream_t st) {
  const unsigned grid = (unsigned)((q.nseq + LineGeom<N>::G - 1) / LineGeom<N>::G);
  hipLaunchKernelGGL(line_kernel<N>, dim3(grid), dim3(LineGeom<N>::THREADS), 0, st, in, out, q, sign, scale);
}

inline bool run_lines(const float2* in, float2* out, const Seqs& q, int N, int sign, float scale, hipStream_t st) {
  if (q.stride != 1 || q.seq_fast || q.inner != q.nseq) return false;
  switch (N) {
    case 2: launch_line<2>(in, out, q, sign, scale, st); return true;
    case 4: launch_line<4>(in, out, q, sign, scale, st); return true;
    case 8: launch_line<8>(in, out, q, sign, scale, st); return true;
    case 16: launch_line<16>(in, out, q, sign, scale, st); return true;
    case 32: launch_line<32>(in, out, q, sign, scale, st); return true;
    case 64: launch_line<64>(in, out, q, sign, scale, st); return true;
    case 128: launch_line<128>(in, out, q, sign, scale, st); return true;
    case 256: launch_line<256>(in, out, q, sign, scale, st); return true;
    case 512: launch_line<512>(in, out, q, sign, scale, st); return true;
    case 1024: launch_line<1024>(in, out, q, sign, scale, st); return true;
    case 2048: launch_line<2048>(in, out, q, sign, scale, st); return true;
    case 4096: launch_line<4096>(in, out, q, sign, scale, st); return true;
    case 8192: launch_line<8192>(in, out, q, sign, scale, st); return true;
    case 16384: launch_line<16384>(in, out, q, sign, scale, st); return true;
    default: return false;
  }
}

// ---- two passes over long contiguous lines ------------------------------------------
// Sequences of ONEPASS_MAX_N < N <= MAX_N points at unit stride: N = N1 * N2 with N1 = 16^k.
// The first k stages move positions only within the N1-point columns p = c + m N2 (c < N2),
// and leave N1 independent blocks of N2 contiguous positions, each of which the remaining
// stages transform as an N2-point sequence (the same twiddles, w_Nj with Nj <= N2). So:
//   pass A (col_kernel): C columns per workgroup, loaded as runs of C points from each of
//   the N1 rows, stages 0..k-1 in LDS with the stage kernel's line DFTs and twiddles (the
//   global inner index c + u N2), written back in place to the workspace;
//   pass B (row_kernel): G blocks per workgroup, the one-pass stages of an N2-point
//   sequence, and block b's frequency f written to k = rev(b) + N1 f, rev reversing b's k
//   base-16 digits; the G blocks have consecutive rev(b), so the writes are runs of G points.
// Each sequence crosses HBM twice each way instead of once per stage, with the staged
// kernels' arithmetic in the same order: the results are bit-identical to them.
constexpr int TWOPASS_MAX_N1 = 4096, TWOPASS_MAX_N2 = 4096;

template <int N1>
struct ColGeom {
  static constexpr int C = N1 >= 1024 ? 4 : 4096 / N1;  // columns per workgroup
  static constexpr int SLOTS = N1 * C;
  static constexpr int THREADS = SLOTS / MAX_RADIX;
};

template <int N2>
struct RowGeom {
  static constexpr int G = N2 >= 1024 ? 4 : 4096 / N2;  // blocks per workgroup
  static constexpr int SLOTS = G * N2;
  static constexpr int THREADS = SLOTS / MAX_RADIX;
  static constexpr int LDS = SLOTS + SLOTS / 16;
};

// Stage of pass A whose local stride is LS (N1/16 at the first stage, 1 at the last), one line per
// lane: the first one from `src`, the last one to `dst` (columns c0.., N2 points from row to row: runs of
// C points either way), through buf between them.
template <int N1, int LS>
__device__ __forceinline__ void col_stage(const float2* src, float2* dst, float2* buf, int c0, int N2, int sign) {
  constexpr int R = MAX_RADIX, C = ColGeom<N1>::C;
  static_assert((N1 / R) * C == ColGeom<N1>::THREADS, "a line per lane");
  const int j = threadIdx.x % C, l = threadIdx.x / C;  // column j (consecutive across threads), line l of it
  const int lu = l % LS, mb = (l / LS) * R * LS + lu;
  float2 x[R];
#pragma unroll
  for (int t = 0; t < R; t++) {
    if constexpr (LS == N1 / R) x[t] = src[(long long)(mb + t * LS) * N2 + j];
    else x[t] = buf[(mb + t * LS) * C + j];
  }
  double vr[R], vi[R];
#pragma unroll
  for (int t = 0; t < R; t++) {
    vr[t] = (double)x[t].x;
    vi[t] = (double)x[t].y;
  }
  line_dft<R>(vr, vi, sign);
  // the stage kernel's twiddle of this line: inner = p mod sJ, Nj = R sJ, sJ = LS N2
  twiddled_outputs<R>(vr, vi, c0 + j + lu * N2, R * LS * N2, sign, [&](int k, float2 v) {
    if constexpr (LS == 1) dst[(long long)(mb + k) * N2 + j] = v;
    else buf[(mb + k * LS) * C + j] = v;
  });
  if constexpr (LS > 1) {
    lds_sync();
    col_stage<N1, LS / R>(src, dst, buf, c0, N2, sign);
  }
}

template <int N1>
__global__ void __launch_bounds__(ColGeom<N1>::THREADS)
    col_kernel(const float2* in, float2* work, Seqs q, int N2, int sign) {
  typedef ColGeom<N1> CG;
  __shared__ float2 buf[N1 > MAX_RADIX ? CG::SLOTS : 1];
  const int per_seq = N2 / CG::C;
  const long long s = blockIdx.x / per_seq;
  const int c0 = (int)(blockIdx.x - s * per_seq) * CG::C;
  col_stage<N1, N1 / MAX_RADIX>(in + q.base(s) + c0, work + s * N1 * N2 + c0, buf, c0, N2, sign);
}

// b's k base-16 digits reversed (an involution)
__device__ __forceinline__ int digit_reverse16(int b, int k) {
  int r = 0;
  for (int i = 0; i < k; i++) {
    r = (r << 4) | (b & 15);
    b >>= 4;
  }
  return r;
}

// N2 >= 256: the first stage's lines straight from memory. The last stage's go straight to it, the
// G frequencies of one index next to each other. Measured, both passes, staged through LDS at either
// end and now: 96 x 131072 120 -> 85 us, 48 x 2^18 124 -> 98, 16 x 2^20 217 -> 185.
template <int N2>
__global__ void __launch_bounds__(RowGeom<N2>::THREADS)
    row_kernel(const float2* work, float2* out, Seqs q, int N1, int k, int sign, float scale) {
  typedef RowGeom<N2> RG;
  typedef LineGeom<N2> LG;
  __shared__ float2 buf[RG::LDS];
  __shared__ double tc[LG::TW], ts[LG::TW];
  constexpr int R = LG::last(), LPS = N2 / R, sJ = LG::DIRECT ? N2 / MAX_RADIX : 1;
  const int per_seq = N1 / RG::G;
  const long long s = blockIdx.x / per_seq;
  const int r0 = (int)(blockIdx.x - s * per_seq) * RG::G;  // rev(b) of the first block
  const long long N = (long long)N1 * N2;
  const float2* src = work + s * N;
  const int gt = threadIdx.x / sJ, inner = threadIdx.x % sJ;
  float2 x[MAX_RADIX];
  if constexpr (LG::DIRECT) {
    const float2* row = src + (long long)digit_reverse16(r0 + gt, k) * N2 + inner;
#pragma unroll
    for (int t = 0; t < MAX_RADIX; t++) x[t] = row[t * sJ];
    __asm__ volatile("" ::: "memory");
  }
  for (int j = threadIdx.x; j < LG::TW; j += RG::THREADS) {
    double sn, c;
    sincospi(2.0 * (double)j / (double)N2, &sn, &c);
    tc[j] = c;
    ts[j] = sn;
  }
  if constexpr (LG::DIRECT) {
    lds_sync();
    double vr[MAX_RADIX], vi[MAX_RADIX];
#pragma unroll
    for (int t = 0; t < MAX_RADIX; t++) {
      vr[t] = (double)x[t].x;
      vi[t] = (double)x[t].y;
    }
    line_dft<MAX_RADIX>(vr, vi, sign);
    twiddled_outputs_w<MAX_RADIX>(vr, vi, tc[inner], sign * ts[inner],
                                  [&](int kk, float2 v) { buf[lpad(gt * N2 + inner + kk * sJ)] = v; });
    lds_sync();
    line_stages<N2, N2 / MAX_RADIX, RG::G, RG::THREADS>(buf, tc, ts, sign);
  } else {
    for (int i = threadIdx.x; i < RG::SLOTS; i += RG::THREADS) {
      const int g = i / N2, e = i - g * N2;
      buf[lpad(i)] = src[(long long)digit_reverse16(r0 + g, k) * N2 + e];
    }
    __syncthreads();
    line_stages<N2, N2, RG::G, RG::THREADS>(buf, tc, ts, sign);
  }
  float2* dst = out + q.base(s) + r0;
  for (int li = threadIdx.x; li < RG::G * LPS; li += RG::THREADS) {
    const int g = li % RG::G, kb = li / RG::G, at = g * N2 + line_position<N2>(kb);
    double vr[R], vi[R];
#pragma unroll
    for (int t = 0; t < R; t++) {
      const float2 v = buf[lpad(at + t)];
      vr[t] = (double)v.x;
      vi[t] = (double)v.y;
    }
    line_dft<R>(vr, vi, sign);
#pragma unroll
    for (int t = 0; t < R; t++) {
      const int r = bitrev<R>(t);
      dst[(long long)(kb + t * LPS) * N1 + g] = make_float2((float)(vr[r] * scale), (float)(vi[r] * scale));
    }
  }
}

template <int N1>
inline void launch_cols(const float2* in, float2* work, const Seqs& q, int N2, int sign, hipStream_t st) {
  const unsigned grid = (unsigned)(q.nseq * (N2 / ColGeom<N1>::C));
  hipLaunchKernelGGL(col_kernel<N1>, dim3(grid), dim3(ColGeom<N1>::THREADS), 0, st, in, work, q, N2, sign);
}

template <int N2>
inline void launch_rows(const float2* work, float2* out, const Seqs& q, int N1, int k, int sign, float scale,
                        hipStream_t st) {
  const unsigned grid = (unsigned)(q.nseq * (N1 / RowGeom<N2>::G));
  hipLaunchKernelGGL(row_kernel<N2>, dim3(grid), dim3(RowGeom<N2>::THREADS), 0, st, work, out, q, N1, k, sign,
                     scale);
}

// The column count k (N1 = 16^k) whose passes read and write the longest runs: pass A's
// runs are C points, pass B's G points; both passes within TWOPASS_MAX_N1 / _N2. 0 if none.
inline int two_pass_k(long long N) {
  int best = 0, best_run = 0;
  for (int k = 1; k <= 3; k++) {
    const long long N1 = 1LL << (4 * k), N2 = N / N1;
    if (N1 > TWOPASS_MAX_N1 || N2 > TWOPASS_MAX_N2 || N2 < 16 || N1 * N2 != N) continue;
    const int C = N1 >= 1024 ? 4 : (int)(4096 / N1), G = N2 >= 1024 ? 4 : (int)(4096 / N2);
    if (G > N1 || C > N2) continue;
    const int run = C < G ? C : G;
    if (run > best_run) best = k, best_run = run;
  }
  return best;
}

inline bool run_two_pass(const float2* in, float2* out, float2* work, const Seqs& q, long long N, int sign,
                         float scale, hipStream_t st) {
  if (q.stride != 1 || q.seq_fast || N <= ONEPASS_MAX_N) return false;
  const int k = two_pass_k(N);
  if (!k) return false;
  const int N1 = 1 << (4 * k), N2 = (int)(N / N1);
  switch (N1) {
    case 16: launch_cols<16>(in, work, q, N2, sign, st); break;
    case 256: launch_cols<256>(in, work, q, N2, sign, st); break;
    case 4096: launch_cols<4096>(in, work, q, N2, sign, st); break;
    default: return false;
  }
  switch (N2) {
    case 16: launch_rows<16>(work, out, q, N1, k, sign, scale, st); break;
    case 32: launch_rows<32>(work, out, q, N1, k, sign, scale, st); break;
    case 64: launch_rows<64>(work, out, q, N1, k, sign, scale, st); break;
    case 128: launch_rows<128>(work, out, q, N1, k, sign, scale, st); break;
    case 256: launch_rows<256>(work, out, q, N1, k, sign, scale, st); break;
    case 512: launch_rows<512>(work, out, q, N1, k, sign, scale, st); break;
    case 1024: launch_rows<1024>(work, out, q, N1, k, sign, scale, st); break;
    case 2048: launch_rows<2048>(work, out, q, N1, k, sign, scale, st); break;
    case 4096: launch_rows<4096>(work, out, q, N1, k, sign, scale, st); break;
    default: return false;
  }
  return true;
}

// Workspace of one transform call: the stage results between the first and last stage.
inline long long work_elems(const Seqs& q, long long N) {
  Radices d;
  if (!split(N, &d)) return -1;
  return d.S > 1 ? q.nseq * N : 0;
}

// All stages of one batched 1-D transform; `work` holds work_elems(q, N) complex64.
// `in` may equal `out`: the first stage reads all of `in` before the last one writes.
inline hipError_t run(const float2* in, float2* out, float2* work, const Seqs& q, int N, int inverse, float scale,
                      hipStream_t st) {
  Radices d;
  if (!split(N, &d)) return hipErrorInvalidValue;
  const int sign = inverse ? 1 : -1;
  if (N <= ONEPASS_MAX_N && run_lines(in, out, q, N, sign, scale, st)) return hipGetLastError();
  if (run_two_pass(in, out, work, q, N, sign, scale, st)) return hipGetLastError();
  if (d.S > 1 && !work) return hipErrorInvalidValue;
  for (int J = 0; J < d.S; J++) {
    const long long threads = q.nseq * (N / d.r[J]);
    const dim3 grid((unsigned)((threads + 127) / 128)), block(128);
    const float sc = J == d.S - 1 ? scale : 1.f;
    switch (d.r[J]) {
      case 2: hipLaunchKernelGGL(stage_kernel<2>, grid, block, 0, st, in, out, work, q, d, J, N, sign, sc); break;
      case 4: hipLaunchKernelGGL(stage_kernel<4>, grid, block, 0, st, in, out, work, q, d, J, N, sign, sc); break;
      case 8: hipLaunchKernelGGL(stage_kernel<8>, grid, block, 0, st, in, out, work, q, d, J, N, sign, sc); break;
      case 16: hipLaunchKernelGGL(stage_kernel<16>, grid, block, 0, st, in, out, work, q, d, J, N, sign, sc); break;
      default: return hipErrorInvalidValue;
    }
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

// Rows then columns of nimg contiguous [N0][N1] arrays; `x` may equal `X`.
inline Seqs rows_of(long long nimg, int N0, int N1) { return Seqs{nimg * N0, nimg * N0, N1, 0, 1, 0}; }
inline Seqs cols_of(long long nimg, int N0, int N1) {
  return Seqs{nimg * N1, N1, 1, (long long)N0 * N1, N1, 1};
}

inline long long work2_elems(long long nimg, int N0, int N1) {
  const long long a = work_elems(rows_of(nimg, N0, N1), N1), b = work_elems(cols_of(nimg, N0, N1), N0);
  if (a < 0 || b < 0) return -1;
  return a > b ? a : b;
}

inline hipError_t run2(const float2* x, float2* X, float2* work, long long nimg, int N0, int N1, int inverse,
                       float scale, hipStream_t st) {
  hipError_t err = run(x, X, work, rows_of(nimg, N0, N1), N1, inverse, 1.f, st);
  if (err != hipSuccess) return err;
  return run(X, X, work, cols_of(nimg, N0, N1), N0, inverse, scale, st);
}

__global__ void widen_kernel(const float* __restrict__ u, float2* __restrict__ w, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) w[i] = make_float2(u[i], 0.f);
}

// U[b][h][p] *= scale * K[h][p]
__global__ void spectrum_product_kernel(float2* __restrict__ U, const float2* __restrict__ K, long long P, int H,
                                        long long n, float scale) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float2 a = U[i], b = K[((i / P) % H) * P + i % P];
  U[i] = make_float2((a.x * b.x - a.y * b.y) * scale, (a.x * b.y + a.y * b.x) * scale);
}

__global__ void real_part_kernel(const float2* __restrict__ w, float* __restrict__ y, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = w[i].x;
}

inline dim3 grid_for(long long n) { return dim3((unsigned)((n + 255) / 256)); }

// Workspace layout of the 2-D circular convolution (complex64 elements):
// [B*H*P spectra of u][H*P spectra of k][stage scratch of B*H images].
inline long long circconv2d_elems(long long B, long long H, int N0, int N1) {
  const long long P = (long long)N0 * N1, t = work2_elems(B * H, N0, N1);
  if (t < 0) return -1;
  return (B * H + H) * P + t;
}

inline hipError_t circconv2d(const float* u, const float* k, float* y, float2* work, long long B, int H, int N0,
                             int N1, hipStream_t st) {
  const long long P = (long long)N0 * N1, nu = B * H * P, nk = (long long)H * P;
  float2 *U = work, *K = work + nu, *T = K + nk;
  hipLaunchKernelGGL(widen_kernel, grid_for(nu), dim3(256), 0, st, u, U, nu);
  hipLaunchKernelGGL(widen_kernel, grid_for(nk), dim3(256), 0, st, k, K, nk);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  if ((err = run2(U, U, T, B * H, N0, N1, 0, 1.f, st)) != hipSuccess) return err;
  if ((err = run2(K, K, T, H, N0, N1, 0, 1.f, st)) != hipSuccess) return err;
  hipLaunchKernelGGL(spectrum_product_kernel, grid_for(nu), dim3(256), 0, st, U, (const float2*)K, P, H, nu,
                     (float)(1.0 / (double)P));
  if ((err = hipGetLastError()) != hipSuccess) return err;
  if ((err = run2(U, U, T, B * H, N0, N1, 1, 1.f, st)) != hipSuccess) return err;
  hipLaunchKernelGGL(real_part_kernel, grid_for(nu), dim3(256), 0, st, (const float2*)U, y, nu);
  return hipGetLastError();
}

}  // namespace xf
}  // namespace sffft
