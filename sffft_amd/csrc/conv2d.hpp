// 2-D circular convolution of real images in four launches (sffft_circconv2d_f32).
//
// A real row of N1 = 2M samples is transformed as M complex points (its even samples + i its odd
// ones) and untangled into the M + 1 frequencies that determine it. The first and the last are
// real and share one slot, so an image's row spectra are [N0][M] complex64, half of what the
// widened rows took. They are kept in blocks of 8 columns, [M / 8][N0][8]: a workgroup of the
// column pass reads and writes one contiguous run, and a workgroup of the row passes 64-byte
// pieces of neighbouring rows that follow each other in memory.
//
//   rows_forward   u and k rows -> row spectra
//   cols<false>    filters: transform over the rows, left in digit-reversed order
//   cols<true>     images: the same transform, times the filter's spectrum, and back, in place
//   rows_inverse   row spectra -> y
//
// Stages are radix 16 in fp64, and stay fp64 through LDS: values are rounded to complex64 only
// where they leave a launch. That more than makes up for what the half-length rows lose (a complex
// transform of real data discards half of its rounding noise with the imaginary part): 5.7e-8 from
// 64 bits at 256 x 256 against 7.3e-8 before. The
// inverse over the columns undoes the forward stages from their digit-reversed order, so nothing is
// permuted, and its first stage takes the products from the registers of the last forward one.
//
// Each image crosses memory three times each way at 4 bytes a sample; widening, three
// two-dimensional complex transforms with one launch per column stage, product and real part
// moved 8 bytes a sample 11 times each way. Two wavefronts per SIMD (the fp64 planes take the
// LDS) leave it bound by the latency between the barriers of the stages, so every launch requests
// its points before it evaluates its tables. Measured at B=8, H=16, 256 x 256: 269 us in 13
// launches -> 65 us.
#pragma once
#include "transforms.hpp"

namespace sffft {
namespace xf {
namespace c2 {

constexpr int CB = 8;  // columns per block

// What others read next has been written. The memory clobber keeps LDS reads above the barrier:
// the compiler's sinking of instructions to their use does not take s_barrier for a store.
__device__ __forceinline__ void block_sync() {
  __asm__ volatile("" ::: "memory");
  __syncthreads();
}

// A geometry G has N points per sequence, NSEQ sequences and THREADS lanes (one per radix-16
// line) in a workgroup; at(seq, p) is a point's slot in the fp64 planes, item(li, lps, ...) the
// sequence and line of work item li. tc + i ts: the twiddle bases w_N^-j, j < N / 16, every
// TSTEP-th entry of the workgroup's table.
template <int N>
struct Lines {
  static constexpr int radix(int rest) { return rest > MAX_RADIX ? MAX_RADIX : rest; }
  static constexpr int last() {
    int r = N;
    while (r > MAX_RADIX) r /= MAX_RADIX;
    return r;
  }
};

template <class G>
struct Planes {
  double re[G::SIZE], im[G::SIZE];
  double tc[G::ROOTS], ts[G::ROOTS];
  __device__ __forceinline__ void init() {
    for (int j = threadIdx.x; j < G::ROOTS; j += G::THREADS) {
      double sn, c;
      sincospi(2.0 * (double)j / (double)(G::N * G::TSTEP), &sn, &c);
      tc[j] = c;
      ts[j] = sn;
    }
  }
  __device__ __forceinline__ void put(int at, double r, double i) {
    re[at] = r;
    im[at] = i;
  }
};

// One line of a stage with REST > 16 (radix 16, twiddles; INV: positive exponents), its points
// p = base + sJ t from load(p, ...), in place at p = base + sJ k.
template <class G, int REST, bool INV, class Load>
__device__ __forceinline__ void twiddled_line(Planes<G>& sh, int seq, int l, Load load) {
  constexpr int R = MAX_RADIX, sJ = REST / R;
  const int inner = l % sJ, base = (l / sJ) * REST + inner;
  double vr[R], vi[R];
#pragma unroll
  for (int t = 0; t < R; t++) load(base + t * sJ, vr[t], vi[t]);
  line_dft<R>(vr, vi, INV ? 1 : -1);
  const int e = inner * (G::N / REST) * G::TSTEP;
  const double w1c = sh.tc[e], w1s = INV ? sh.ts[e] : -sh.ts[e];
  double wr = 1.0, wi = 0.0;
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int r = bitrev<R>(k);
    sh.put(G::at(seq, base + k * sJ), fma(vr[r], wr, -(vi[r] * wi)), fma(vr[r], wi, vi[r] * wr));
    const double nr = fma(wr, w1c, -(wi * w1s));
    wi = fma(wr, w1s, wi * w1c);
    wr = nr;
  }
}

// The stages between the first and the last one.
template <class G, int REST, bool INV>
__device__ __forceinline__ void middle_stages(Planes<G>& sh) {
  if constexpr (REST > MAX_RADIX) {
    for (int li = threadIdx.x; li < G::NSEQ * (G::N / MAX_RADIX); li += G::THREADS) {
      int seq, l;
      G::item(li, G::N / MAX_RADIX, seq, l);
      twiddled_line<G, REST, INV>(sh, seq, l, [&](int p, double& r, double& i) {
        const int at = G::at(seq, p);
        r = sh.re[at];
        i = sh.im[at];
      });
    }
    block_sync();
    middle_stages<G, REST / MAX_RADIX, INV>(sh);
  }
}

// A lane's 16 points of the first stage, src(seq, p), requested before the tables are evaluated: the
// round trip to memory and the evaluation overlap. (Up to 16 points: 16 points of any kind, which go
// to the last stage through LDS.)
template <class G, class Src>
__device__ __forceinline__ void load_first(float2 (&x)[MAX_RADIX], Src src) {
#pragma unroll
  for (int t = 0; t < MAX_RADIX; t++) {
    int seq, l;
    if constexpr (G::N > MAX_RADIX) {
      G::item(threadIdx.x, G::N / MAX_RADIX, seq, l);
      x[t] = src(seq, l + t * (G::N / MAX_RADIX));
    } else {
      G::item(threadIdx.x + t * G::THREADS, G::N, seq, l);
      x[t] = src(seq, l);
    }
  }
  __asm__ volatile("" ::: "memory");
}
template <class G>
__device__ __forceinline__ void first_stage(Planes<G>& sh, const float2 (&x)[MAX_RADIX]) {
  if constexpr (G::N > MAX_RADIX) {
    int seq, l, t = 0;
    G::item(threadIdx.x, G::N / MAX_RADIX, seq, l);
    twiddled_line<G, G::N, false>(sh, seq, l, [&](int, double& r, double& i) {
      r = (double)x[t].x;
      i = (double)x[t].y;
      t++;
    });
  } else {
#pragma unroll
    for (int t = 0; t < MAX_RADIX; t++) {
      int seq, p;
      G::item(threadIdx.x + t * G::THREADS, G::N, seq, p);
      sh.put(G::at(seq, p), (double)x[t].x, (double)x[t].y);
    }
  }
  block_sync();
  middle_stages<G, G::N / MAX_RADIX, false>(sh);
}

// Frequency at position p after the forward stages (line_position inverted).
template <int N>
__device__ __forceinline__ int freq_at(int p) {
  int f = 0, w = 1, sj = N;
  while (sj > 1) {
    const int r = sj > MAX_RADIX ? MAX_RADIX : sj;
    sj /= r;
    f += ((p / sj) % r) * w;
    w *= r;
  }
  return f;
}

// ---- rows -------------------------------------------------------------------------
// G rows of M complex points per workgroup.
template <int M>
struct Rows {
  static constexpr int N = M, SLOTS = M >= 2048 ? M : 2048, NSEQ = SLOTS / M, THREADS = SLOTS / MAX_RADIX;
  static constexpr int SIZE = SLOTS + SLOTS / 16 + NSEQ;
  static constexpr int ROOTS = M / 2 + 1, TSTEP = 2;  // roots of order 2M, which untangling needs too
  // a slot of padding per 16 points and one per row: the rows that a wavefront untangles side by
  // side start on different banks
  __device__ static __forceinline__ int at(int seq, int p) { return lpad(seq * M + p) + seq; }
  __device__ static __forceinline__ void item(int li, int lps, int& seq, int& l) {
    seq = li / lps;
    l = li % lps;
  }
};

// point (row, k) of the row spectra: block k / 8 of the row's image, images of 2^l0 rows
__device__ __forceinline__ size_t spec_at(int row, int k, int l0, int M) {
  const int img = row >> l0;
  return ((size_t)img * M << l0) + ((size_t)(k / CB) << l0) * CB + (row - (img << l0)) * CB + k % CB;
}

// Rows [0, nu) from u, [nu, nrows) from k.
template <int M>
__global__ void __launch_bounds__(Rows<M>::THREADS)
    rows_forward(const float2* __restrict__ u, const float2* __restrict__ k, float2* __restrict__ spec, int nu,
                 int nrows, int l0) {
  typedef Rows<M> G;
  constexpr int R = Lines<M>::last(), LPS = M / R;
  __shared__ Planes<G> sh;
  const int r0 = blockIdx.x * G::NSEQ;
  float2 x[MAX_RADIX];
  load_first<G>(x, [&](int seq, int p) {  // lanes past the last row repeat it
    const int row = r0 + seq < nrows ? r0 + seq : nrows - 1;
    return (row < nu ? u + (size_t)row * M : k + (size_t)(row - nu) * M)[p];
  });
  sh.init();
  __syncthreads();
  first_stage<G>(sh, x);
  // last stage, in place
  for (int li = threadIdx.x; li < G::NSEQ * LPS; li += G::THREADS) {
    int seq, l;
    G::item(li, LPS, seq, l);
    double vr[R], vi[R];
#pragma unroll
    for (int t = 0; t < R; t++) {
      const int at = G::at(seq, l * R + t);
      vr[t] = sh.re[at];
      vi[t] = sh.im[at];
    }
    line_dft<R>(vr, vi, -1);
#pragma unroll
    for (int t = 0; t < R; t++) sh.put(G::at(seq, l * R + t), vr[bitrev<R>(t)], vi[bitrev<R>(t)]);
  }
  block_sync();
  // X[f] = E + w^f O with E = (Z[f] + conj Z[M-f]) / 2, O = (Z[f] - conj Z[M-f]) / 2i; the
  // rows of a block next to each other in memory
#pragma unroll 4
  for (int i = threadIdx.x; i < G::SLOTS; i += G::THREADS) {
    const int g = (i / CB) % G::NSEQ, f = i / (CB * G::NSEQ) * CB + i % CB;
    if (r0 + g >= nrows) continue;
    const int a = G::at(g, line_position<M>(f)), z = G::at(g, line_position<M>((M - f) & (M - 1)));
    const double ar = sh.re[a], ai = sh.im[a], zr = sh.re[z], zi = sh.im[z];
    // w^(M - f) = -conj(w^f)
    const double c = f <= M / 2 ? sh.tc[f] : -sh.tc[M - f], s = -(f <= M / 2 ? sh.ts[f] : sh.ts[M - f]);
    const double er = 0.5 * (ar + zr), ei = 0.5 * (ai - zi), orr = 0.5 * (ai + zi), oi = -0.5 * (ar - zr);
    float2 x = make_float2((float)(er + (orr * c - oi * s)), (float)(ei + (orr * s + oi * c)));
    if (f == 0) x = make_float2((float)(er + orr), (float)(er - orr));  // frequencies 0 and M
    spec[spec_at(r0 + g, f, l0, M)] = x;
  }
}

template <int M>
__global__ void __launch_bounds__(Rows<M>::THREADS)
    rows_inverse(const float2* __restrict__ spec, float2* __restrict__ y, int nrows, int l0, double scale) {
  typedef Rows<M> G;
  constexpr int R = Lines<M>::last(), LPS = M / R;
  __shared__ Planes<G> sh;
  const int r0 = blockIdx.x * G::NSEQ;
  float2 xa[G::SLOTS / 2 / G::THREADS], xz[G::SLOTS / 2 / G::THREADS];  // X[f], X[M-f]; requested before the tables
#pragma unroll
  for (int v = 0; v < G::SLOTS / 2 / G::THREADS; v++) {
    const int i = threadIdx.x + v * G::THREADS, g = (i / CB) % G::NSEQ, f = i / (CB * G::NSEQ) * CB + i % CB;
    const int row = r0 + g < nrows ? r0 + g : nrows - 1;  // lanes past the last row repeat it
    xa[v] = spec[spec_at(row, f, l0, M)];
    xz[v] = spec[spec_at(row, f ? M - f : M / 2, l0, M)];
  }
  __asm__ volatile("" ::: "memory");
  sh.init();
  __syncthreads();
  // Z[f] = E + i O with E = (X[f] + conj X[M-f]) / 2, O = (X[f] - conj X[M-f]) / 2 * conj(w^f);
  // a lane takes f and M - f
#pragma unroll
  for (int v = 0; v < G::SLOTS / 2 / G::THREADS; v++) {
    const int i = threadIdx.x + v * G::THREADS, g = (i / CB) % G::NSEQ, f = i / (CB * G::NSEQ) * CB + i % CB;
    const float2 a = xa[v], z = xz[v];
    if (f == 0) {
      sh.put(G::at(g, 0), 0.5 * ((double)a.x + a.y), 0.5 * ((double)a.x - a.y));
      sh.put(G::at(g, M / 2), z.x, -z.y);  // E = Re X, O = i Im X * conj(-i)
    } else {
      const double c = sh.tc[f], s = -sh.ts[f];
      const double er = 0.5 * ((double)a.x + z.x), ei = 0.5 * ((double)a.y - z.y);
      const double dr = 0.5 * ((double)a.x - z.x), di = 0.5 * ((double)a.y + z.y);
      const double orr = dr * c + di * s, oi = di * c - dr * s;
      sh.put(G::at(g, f), er - oi, ei + orr);
      sh.put(G::at(g, M - f), er + oi, orr - ei);
    }
  }
  block_sync();
  middle_stages<G, M, true>(sh);
  // last stage, to memory: line `kb` in natural order of its first sample, which makes a wavefront's
  // stores contiguous
  for (int li = threadIdx.x; li < G::NSEQ * LPS; li += G::THREADS) {
    int seq, kb;
    G::item(li, LPS, seq, kb);
    const int l = line_position<M>(kb);  // position of sample kb: the line's first
    double vr[R], vi[R];
#pragma unroll
    for (int t = 0; t < R; t++) {
      const int at = G::at(seq, l + t);
      vr[t] = sh.re[at];
      vi[t] = sh.im[at];
    }
    line_dft<R>(vr, vi, 1);
    if (r0 + seq >= nrows) continue;
    float2* o = y + (size_t)(r0 + seq) * M + kb;
#pragma unroll
    for (int t = 0; t < R; t++)
      o[t * LPS] = make_float2((float)(vr[bitrev<R>(t)] * scale), (float)(vi[bitrev<R>(t)] * scale));
  }
}

// ---- columns ----------------------------------------------------------------------
// NB whole blocks of 8 columns of N0 points per workgroup; sequence blk * 8 + j.
template <int N0>
struct Cols {
  static constexpr int N = N0, BLOCK = N0 * CB, NB = BLOCK >= 2048 ? 1 : 2048 / BLOCK;
  static constexpr int SLOTS = NB * BLOCK, NSEQ = NB * CB, THREADS = SLOTS / MAX_RADIX;
  static constexpr int PBLOCK = (N0 + N0 / 16) * CB, SIZE = NB * PBLOCK;  // one row of 8 slots per 16 rows of padding
  static constexpr int ROOTS = N0 > MAX_RADIX ? N0 / MAX_RADIX : 1, TSTEP = 1;
  __device__ static __forceinline__ int at(int seq, int p) {
    return seq / CB * PBLOCK + lpad(p) * CB + seq % CB;
  }
  __device__ static __forceinline__ void item(int li, int lps, int& seq, int& l) {  // columns fastest
    seq = li / (CB * lps) * CB + li % CB;
    l = li / CB % lps;
  }
};
template <int N0, bool CONV>
struct ColsShared {
  Planes<Cols<N0>> s;
  double xr[CONV ? Cols<N0>::NB * N0 : 1], xi[CONV ? Cols<N0>::NB * N0 : 1];  // column 0 of each block
};

// The stages back after the first (innermost) inverse one: conjugate twiddles, inverse line, from
// REST up to N; the last one to memory.
template <int N0, int REST, class Dst>
__device__ __forceinline__ void cols_back(ColsShared<N0, true>& sh, Dst dst) {
  typedef Cols<N0> G;
  constexpr int R = MAX_RADIX, sJ = REST / R;
  for (int li = threadIdx.x; li < G::NSEQ * (N0 / R); li += G::THREADS) {
    int seq, l;
    G::item(li, N0 / R, seq, l);
    const int inner = l % sJ, base = (l / sJ) * REST + inner, e = inner * (N0 / REST);
    const double w1c = sh.s.tc[e], w1s = sh.s.ts[e];
    double vr[R], vi[R], wr = 1.0, wi = 0.0;
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int at = G::at(seq, base + k * sJ);
      const double xr = sh.s.re[at], xi = sh.s.im[at];
      vr[k] = fma(xr, wr, -(xi * wi));
      vi[k] = fma(xr, wi, xi * wr);
      const double nr = fma(wr, w1c, -(wi * w1s));
      wi = fma(wr, w1s, wi * w1c);
      wr = nr;
    }
    line_dft<R>(vr, vi, 1);
#pragma unroll
    for (int t = 0; t < R; t++) {
      if constexpr (REST == N0) dst(seq, base + t * sJ, vr[bitrev<R>(t)], vi[bitrev<R>(t)]);
      else sh.s.put(G::at(seq, base + t * sJ), vr[bitrev<R>(t)], vi[bitrev<R>(t)]);
    }
  }
  if constexpr (REST < N0) {
    block_sync();
    cols_back<N0, REST * MAX_RADIX>(sh, dst);
  }
}

// Workgroup: NB consecutive blocks of the nblocks at `spec`, in place. CONV: times the spectra of
// the filters (image i has filter i % H; `filt` as the launch without CONV left them, in position
// order) and back.
template <int N0, bool CONV>
__global__ void __launch_bounds__(Cols<N0>::THREADS)
    cols(float2* __restrict__ spec, const float2* __restrict__ filt, int nblocks, int lbpi, int H) {
  typedef Cols<N0> G;
  constexpr int R = Lines<N0>::last(), LPS = N0 / R, PER = MAX_RADIX / R;  // lines per lane in the last stage
  __shared__ ColsShared<N0, CONV> sh;
  const int b0 = blockIdx.x * G::NB;
  float2* x = spec + (size_t)b0 * G::BLOCK;
  auto live = [&](int seq) { return b0 + seq / CB < nblocks; };
  float2 x0[MAX_RADIX];
  load_first<G>(x0, [&](int seq, int p) {
    const int blk = live(seq) ? seq / CB : nblocks - 1 - b0;  // lanes past the last block repeat it
    return x[blk * G::BLOCK + p * CB + seq % CB];
  });
  sh.s.init();
  __syncthreads();
  first_stage<G>(sh.s, x0);
  // the filter's values, requested ahead of the last stage
  float2 kv[PER][R];
  if constexpr (CONV) {
#pragma unroll
    for (int m = 0; m < PER; m++) {
      int seq, l;
      G::item(threadIdx.x + m * G::THREADS, LPS, seq, l);
      const int blk = b0 + seq / CB < nblocks ? b0 + seq / CB : nblocks - 1, img = blk >> lbpi;
      const float2* K = filt + (((size_t)(img % H) << lbpi) + (blk - (img << lbpi))) * G::BLOCK;
#pragma unroll
      for (int t = 0; t < R; t++) kv[m][t] = K[(l * R + t) * CB + seq % CB];
    }
    __asm__ volatile("" ::: "memory");
  }
  double vr[PER][R], vi[PER][R];
#pragma unroll
  for (int m = 0; m < PER; m++) {
    int seq, l;
    G::item(threadIdx.x + m * G::THREADS, LPS, seq, l);
    double ar[R], ai[R];
#pragma unroll
    for (int t = 0; t < R; t++) {
      const int at = G::at(seq, l * R + t);
      ar[t] = sh.s.re[at];
      ai[t] = sh.s.im[at];
    }
    line_dft<R>(ar, ai, -1);
#pragma unroll
    for (int t = 0; t < R; t++) {
      vr[m][t] = ar[bitrev<R>(t)];
      vi[m][t] = ai[bitrev<R>(t)];
      if constexpr (!CONV) {
        if (live(seq)) x[seq / CB * G::BLOCK + (l * R + t) * CB + seq % CB] = make_float2((float)vr[m][t], (float)vi[m][t]);
      } else if (seq % CB == 0) {
        sh.xr[seq / CB * N0 + l * R + t] = vr[m][t];
        sh.xi[seq / CB * N0 + l * R + t] = vi[m][t];
      }
    }
  }
  if constexpr (CONV) {
    block_sync();
#pragma unroll
    for (int m = 0; m < PER; m++) {
      int seq, l;
      G::item(threadIdx.x + m * G::THREADS, LPS, seq, l);
      const int blk = b0 + seq / CB < nblocks ? b0 + seq / CB : nblocks - 1, img = blk >> lbpi;
      const int b = blk - (img << lbpi), j = seq % CB;
      const float2* K = filt + (((size_t)(img % H) << lbpi) + b) * G::BLOCK;
      double ar[R], ai[R];
#pragma unroll
      for (int t = 0; t < R; t++) {
        const double kr = kv[m][t].x, ki = kv[m][t].y;
        ar[t] = vr[m][t] * kr - vi[m][t] * ki;
        ai[t] = vr[m][t] * ki + vi[m][t] * kr;
      }
      if (b == 0 && j == 0) {
        // the slot of row frequencies 0 and M: two real columns c0 + i cM, whose transforms are
        // A = (Z[f] + conj Z[-f]) / 2 and B = (Z[f] - conj Z[-f]) / 2i, of image and filter;
        // their products A A' and B B' go back as A A' + i B B'
#pragma unroll
        for (int t = 0; t < R; t++) {
          const int q = line_position<N0>((N0 - freq_at<N0>(l * R + t)) & (N0 - 1));
          const float2 k = kv[m][t], k2 = K[q * CB];
          const double zr = vr[m][t], zi = vi[m][t], qr = sh.xr[seq / CB * N0 + q], qi = sh.xi[seq / CB * N0 + q];
          const double Ar = 0.5 * (zr + qr), Ai = 0.5 * (zi - qi), Br = 0.5 * (zi + qi), Bi = -0.5 * (zr - qr);
          const double Cr = 0.5 * ((double)k.x + k2.x), Ci = 0.5 * ((double)k.y - k2.y);
          const double Dr = 0.5 * ((double)k.y + k2.y), Di = -0.5 * ((double)k.x - k2.x);
          const double Pr = Ar * Cr - Ai * Ci, Pi = Ar * Ci + Ai * Cr, Qr = Br * Dr - Bi * Di, Qi = Br * Di + Bi * Dr;
          ar[t] = Pr - Qi;
          ai[t] = Pi + Qr;
        }
      }
      line_dft<R>(ar, ai, 1);
#pragma unroll
      for (int t = 0; t < R; t++) {
        if constexpr (N0 > MAX_RADIX) {
          sh.s.put(G::at(seq, l * R + t), ar[bitrev<R>(t)], ai[bitrev<R>(t)]);
        } else if (live(seq)) {
          x[seq / CB * G::BLOCK + t * CB + j] = make_float2((float)ar[bitrev<R>(t)], (float)ai[bitrev<R>(t)]);
        }
      }
    }
    if constexpr (N0 > MAX_RADIX) {
      block_sync();
      cols_back<N0, R * MAX_RADIX>(sh, [&](int seq, int p, double r, double i) {
        if (live(seq)) x[seq / CB * G::BLOCK + p * CB + seq % CB] = make_float2((float)r, (float)i);
      });
    }
  }
}

// Sizes of this path: row spectra of 16 to 2048 points (whole radix-16 lines), columns of 16 to
// 512 (LDS: 8 fp64 columns of 512 take 80 KB). Others take the complex transforms.
inline bool takes(int N0, int N1) { return N0 >= 16 && N0 <= 512 && N1 >= 32 && N1 <= 4096; }

template <int M>
inline void launch_rows_forward(const float* u, const float* k, float2* spec, int nu, int nrows, int l0,
                                hipStream_t st) {
  hipLaunchKernelGGL(rows_forward<M>, dim3((unsigned)((nrows + Rows<M>::NSEQ - 1) / Rows<M>::NSEQ)),
                     dim3(Rows<M>::THREADS), 0, st, reinterpret_cast<const float2*>(u),
                     reinterpret_cast<const float2*>(k), spec, nu, nrows, l0);
}
template <int M>
inline void launch_rows_inverse(const float2* spec, float* y, int nrows, int l0, double scale, hipStream_t st) {
  hipLaunchKernelGGL(rows_inverse<M>, dim3((unsigned)((nrows + Rows<M>::NSEQ - 1) / Rows<M>::NSEQ)),
                     dim3(Rows<M>::THREADS), 0, st, spec, reinterpret_cast<float2*>(y), nrows, l0, scale);
}
template <int N0>
inline void launch_cols(float2* spec, float2* filt, int images, int H, int lbpi, hipStream_t st) {
  typedef Cols<N0> CG;
  const int nf = H << lbpi, nu = images << lbpi;
  hipLaunchKernelGGL((cols<N0, false>), dim3((unsigned)((nf + CG::NB - 1) / CG::NB)), dim3(CG::THREADS), 0, st, filt,
                     nullptr, nf, lbpi, H);
  hipLaunchKernelGGL((cols<N0, true>), dim3((unsigned)((nu + CG::NB - 1) / CG::NB)), dim3(CG::THREADS), 0, st, spec,
                     filt, nu, lbpi, H);
}

// work: (B H + H) N0 N1 / 2 complex64, within circconv2d_elems. u, k and y are 8-byte aligned.
inline hipError_t run(const float* u, const float* k, float* y, float2* work, long long B, int H, int N0, int N1,
                      hipStream_t st) {
  auto lg = [](int n) { int e = 0; while ((1 << e) < n) e++; return e; };
  // rows and blocks of the at most 2^31 samples, of 32 at least, and of the filters: within an int
  const int M = N1 / 2, l0 = lg(N0), lbpi = lg(M / CB), images = (int)(B * H), nu = images * N0, nrows = nu + H * N0;
  float2* filt = work + (size_t)images * N0 * M;
  const double scale = 1.0 / ((double)N0 * M);
#define SFFFT_ROWS(M_) \
  case M_: launch_rows_forward<M_>(u, k, work, nu, nrows, l0, st); break;
  switch (M) {
    SFFFT_ROWS(16) SFFFT_ROWS(32) SFFFT_ROWS(64) SFFFT_ROWS(128) SFFFT_ROWS(256) SFFFT_ROWS(512) SFFFT_ROWS(1024)
    SFFFT_ROWS(2048)
    default: return hipErrorInvalidValue;
  }
#undef SFFFT_ROWS
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
#define SFFFT_COLS(N_) \
  case N_: launch_cols<N_>(work, filt, images, H, lbpi, st); break;
  switch (N0) {
    SFFFT_COLS(16) SFFFT_COLS(32) SFFFT_COLS(64) SFFFT_COLS(128) SFFFT_COLS(256) SFFFT_COLS(512)
    default: return hipErrorInvalidValue;
  }
#undef SFFFT_COLS
  if ((err = hipGetLastError()) != hipSuccess) return err;
#define SFFFT_ROWS(M_) \
  case M_: launch_rows_inverse<M_>(work, y, nu, l0, scale, st); break;
  switch (M) {
    SFFFT_ROWS(16) SFFFT_ROWS(32) SFFFT_ROWS(64) SFFFT_ROWS(128) SFFFT_ROWS(256) SFFFT_ROWS(512) SFFFT_ROWS(1024)
    SFFFT_ROWS(2048)
  }
#undef SFFFT_ROWS
  return hipGetLastError();
}

}  // namespace c2
}  // namespace xf
}  // namespace sffft
