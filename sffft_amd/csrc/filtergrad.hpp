// Filter gradient of the causal convolution, in one launch (two when its work is split):
//
//   dk[h][j] = sum_b sum_{n >= j} dy[b][h][n] u[b][h][n - j],   j < L,  L = 128..16384
//
// The sum over b commutes with the transforms, so a channel needs one inverse transform
// whatever its batch: with U_b and D_b the zero-padded 2L-point spectra of the rows,
// dk = IDFT(sum_b D_b conj(U_b)). Two batch rows travel as one complex row, z = x_b + i x_b+1:
// then Re IDFT(Z_dy conj(Z_u)) is already the sum of both rows' correlations (the cross terms
// are the imaginary part), so the pair is never taken apart.
//
// The 2L-point transform of a row whose second half is zero splits into two L-point ones,
// its even bins (the transform of x) and its odd bins (of x[n] w_2L^n), and
//   dk[j] = Re(IDFT_L(P_even)[j] + w_2L^-j IDFT_L(P_odd)[j]) / 2
// with P the summed products. The halves are independent until that last sum, which halves
// the LDS a transform needs (L = 16384 fits a CU) and doubles the independent work.
//
// A team of L/16 lanes holds a transform, 16 points per lane in registers: radix-16 stages
// (decimation in frequency, fp32), exchanged through LDS in place. The forward transforms end
// in digit-reversed order; the product is elementwise and the inverse stages undo the
// order, so nothing is ever permuted, and the lane that ends with a bin of u also ends with that bin
// of dy: spectra, products and their sum stay in registers.
//
// fp32 throughout: 3e-7 to 6e-7 from 64 bits, where fp16 operands gave 2e-4 to 3.4e-4 (the
// composition of the spectrum of every row, a convolution and a sum over b, which this
// replaced). Bound by VALU issue, about 600 fp32 instructions per lane and transform, and by
// what hides latency beside it, 2 to 3 wavefronts per SIMD. Measured, that composition before and this
// kernel now: B=8 H=768 L=1024 fp32 220 -> 20 us (2.5 TB/s of u and dy, 0.5 of a copy), B=6
// H=513 L=4096 bf16 610 -> 51, B=5 H=320 L=8192 fp32 540 -> 88.
#pragma once
#include "fftconv.hpp"

namespace sffft {
namespace fg {

struct C {
  float r, i;
};
__device__ __forceinline__ C operator+(C a, C b) { return {a.r + b.r, a.i + b.i}; }
__device__ __forceinline__ C operator-(C a, C b) { return {a.r - b.r, a.i - b.i}; }
__device__ __forceinline__ C mul(C a, C b) { return {a.r * b.r - a.i * b.i, a.r * b.i + a.i * b.r}; }
// a * b, or with CONJ a * conj(b)
template <bool CONJ>
__device__ __forceinline__ C mulc(C a, C b) {
  if constexpr (CONJ) return {a.r * b.r + a.i * b.i, a.i * b.r - a.r * b.i};
  else return mul(a, b);
}
// a * exp(-2 pi i m / 32), or its conjugate with INV; m is a constant after unrolling
template <bool INV>
__device__ __forceinline__ C rot32(C a, int m) {
  constexpr float c[9] = {1.f, 0.98078528040323043f, 0.92387953251128674f, 0.83146961230254524f, 0.70710678118654752f,
                          0.55557023301960218f, 0.38268343236508977f, 0.19509032201612825f, 0.f};
  m &= 31;
  if (INV) m = (32 - m) & 31;
  // quarter turns by -i, then the angle within the first quadrant
  const int q = m >> 3, t = m & 7;
  const C b = q == 0 ? a : q == 1 ? C{a.i, -a.r} : q == 2 ? C{-a.r, -a.i} : C{-a.i, a.r};
  if (t == 0) return b;
  if (t == 4) return {c[4] * (b.r + b.i), c[4] * (b.i - b.r)};
  return {b.r * c[t] + b.i * c[8 - t], b.i * c[t] - b.r * c[8 - t]};
}

template <bool INV>
__device__ __forceinline__ void fft4(C& a, C& b, C& c, C& d) {
  const C s = a + c, t = a - c, u = b + d, v = b - d;
  const C iv = INV ? C{-v.i, v.r} : C{v.i, -v.r};  // v times -i (forward) or i
  a = s + u;
  b = t + iv;
  c = s - u;
  d = t - iv;
}

// In place, natural order in; frequency k comes out at slot<R>(k).
template <int R>
__device__ __forceinline__ constexpr int slot(int k) {
  return R == 16 ? 4 * (k & 3) + (k >> 2) : R == 8 ? 4 * (k & 1) + (k >> 1) : k;
}
template <int R, bool INV>
__device__ __forceinline__ void fft(C* x) {
  if constexpr (R == 2) {
    const C s = x[0] + x[1], d = x[0] - x[1];
    x[0] = s;
    x[1] = d;
  } else if constexpr (R == 4) {
    fft4<INV>(x[0], x[1], x[2], x[3]);
  } else if constexpr (R == 8) {
    // radix 2 over n = j + 4m, then radix 4 over j: frequency q + 2r at 4q + r
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const C s = x[j] + x[j + 4], d = x[j] - x[j + 4];
      x[j] = s;
      x[j + 4] = rot32<INV>(d, 4 * j);
    }
    fft4<INV>(x[0], x[1], x[2], x[3]);
    fft4<INV>(x[4], x[5], x[6], x[7]);
  } else {
    static_assert(R == 16, "radix");
    // radix 4 over n = j + 4m, then radix 4 over j: frequency q + 4r at 4q + r
#pragma unroll
    for (int j = 0; j < 4; j++) {
      fft4<INV>(x[j], x[j + 4], x[j + 8], x[j + 12]);
#pragma unroll
      for (int q = 1; q < 4; q++) x[j + 4 * q] = rot32<INV>(x[j + 4 * q], 2 * j * q);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) fft4<INV>(x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]);
  }
}

// x[k] times w^k (CONJ: its conjugate), k = 0..15 in natural order or (SLOTTED) at slot<16>(k):
// as w^(k & 3) and w^(k & 12), so that six powers serve 16 points (all 15 would take 30 VGPRs
// for the same number of products).
template <bool CONJ, bool SLOTTED>
__device__ __forceinline__ void twiddle16(C* x, C w) {
  asm volatile("" : "+v"(w.r), "+v"(w.i));  // powers are rebuilt at each use: hoisted, they would stay live
  const C w2 = mul(w, w), w3 = mul(w2, w), w4 = mul(w2, w2), w8 = mul(w4, w4), w12 = mul(w8, w4);
  const C lo[4] = {{1.f, 0.f}, w, w2, w3}, hi[4] = {{1.f, 0.f}, w4, w8, w12};
#pragma unroll
  for (int k = 1; k < 16; k++) {
    C& v = x[SLOTTED ? slot<16>(k) : k];
    if (k & 3) v = mulc<CONJ>(v, lo[k & 3]);
    if (k >> 2) v = mulc<CONJ>(v, hi[k >> 2]);
  }
}

// One slot of padding per 16 points: the 16 points of a lane, and the lanes of a stage whose
// blocks are shorter than a wavefront, fall on different banks. The slot of point p = block * REST +
// inner + sJ * k (inner < sJ = REST / 16, blocks of REST points) is slot_base(t) + slot_off(k)
// with a constant offset per k, so that a stage needs one address register and not 16.
__device__ __forceinline__ constexpr int pad(int p) { return p + (p >> 4); }
template <int sJ>
__device__ __forceinline__ int slot_base(int t) {
  const int inner = t % sJ;
  return pad(t / sJ * (16 * sJ)) + inner + (sJ >= 16 ? inner >> 4 : 0);
}
template <int sJ>
__device__ __forceinline__ constexpr int slot_off(int k) { return pad(sJ * k); }

// Geometry of length L: T lanes per transform (team); a workgroup of NT lanes holds 2 halves
// (even and odd bins) x SUB subsets of the batch x CH channels when HALVES == 2, or one team
// whose half comes from the grid.
template <int L_>
struct Geom {
  static constexpr int L = L_, T = L / 16;
  static constexpr int NT = T <= 64 ? 256 : T <= 128 ? 256 : T;
  static constexpr int TEAMS = NT / T;
  static constexpr int HALVES = TEAMS >= 2 ? 2 : 1;
  static constexpr int SUB = TEAMS / HALVES > 4 ? 4 : TEAMS / HALVES;
  static constexpr int CH = TEAMS / HALVES / SUB;
  static constexpr int SLOTS = L + L / 16;  // padded points of one team
  // Wavefronts per SIMD the register allocation must allow. Three (168 VGPRs) hold the working
  // set; held to four the shorter lengths spill and take 1.2 to 1.8 times as long. At
  // L >= 8192 the LDS allows whole workgroups of 8 or 16 wavefronts only, and two of 8 (128
  // VGPRs, 22 to 43 spilled, mostly the sums during a transform) beat one: 90 against 107 us at
  // B=5, H=320, L=8192 fp32.
  static constexpr int WPE = T >= 512 ? 4 : 3;
  // a team within one wavefront exchanges without a barrier
  static constexpr bool WAVE = T <= 64;
};

// Lanes of a team (or of the whole workgroup) have written what others read next. The memory
// clobber keeps a stage's LDS reads above the barrier that ends it: the compiler's sinking of
// instructions to their use does not take s_barrier for a store, and moved reads whose values
// are used only under a condition below it.
template <class G>
__device__ __forceinline__ void team_sync() {
  if constexpr (G::WAVE) wave_lds_fence();
  else {
    __asm__ volatile("" ::: "memory");
    __syncthreads();
  }
}

// Twiddle bases of a lane: stage s of REST points has w_REST^inner; the first stage of the odd
// half carries the common factor w_2L^t of its inputs too (see forward()).
constexpr int MAXS = 4;
template <int L>
__host__ __device__ constexpr int stages() {
  int n = 1;
  for (int r = L; r > 16; r /= 16) n++;
  return n;
}

__device__ __forceinline__ C root(int num, int den) {  // exp(-2 pi i num / den), den a power of two
  float s, c;
  sincospif(2.f * (float)num / (float)den, &s, &c);
  return {c, -s};
}

// Radix-16 stages on REST-point blocks, REST > 16: butterfly, twiddle, exchange; then the last
// stage of radix REST <= 16. On entry x holds the lane's 16 points of this stage.
template <class G, int REST, int S>
__device__ __forceinline__ void forward_stage(C* x, C* buf, const C* w, int t) {
  if constexpr (REST > 16) {
    constexpr int sJ = REST / 16;
    C* at = buf + slot_base<sJ>(t);
    if constexpr (S > 0) {
#pragma unroll
      for (int j = 0; j < 16; j++) x[j] = at[slot_off<sJ>(j)];
    }
    fft<16, false>(x);
    twiddle16<false, true>(x, w[S]);
#pragma unroll
    for (int k = 0; k < 16; k++) at[slot_off<sJ>(k)] = x[slot<16>(k)];
    team_sync<G>();
    forward_stage<G, REST / 16, S + 1>(x, buf, w, t);
  } else {
    // 16 / REST blocks of REST consecutive points per lane, blocks t + T m
    const C* at = buf + pad(t * REST);
#pragma unroll
    for (int m = 0; m < 16 / REST; m++) {
#pragma unroll
      for (int r = 0; r < REST; r++) x[m * REST + r] = at[pad(G::T * REST * m) + r];
      if constexpr (REST > 1) fft<REST, false>(x + m * REST);
    }
    team_sync<G>();  // every lane has read before the next transform's first stage writes
  }
}

// The stages back, from the register order the forward transform ends in. The first
// stage's 16 points end in x in natural order of n = t + T j, at slot<16>(j).
template <class G, int REST, int S>
__device__ __forceinline__ void inverse_stage(C* x, C* buf, const C* w, int t) {
  if constexpr (REST > 16) {
    inverse_stage<G, REST / 16, S + 1>(x, buf, w, t);
    constexpr int sJ = REST / 16;
    C* at = buf + slot_base<sJ>(t);
#pragma unroll
    for (int k = 0; k < 16; k++) x[k] = at[slot_off<sJ>(k)];
    twiddle16<true, false>(x, w[S]);
    if constexpr (S > 0) {
      fft<16, true>(x);
#pragma unroll
      for (int j = 0; j < 16; j++) at[slot_off<sJ>(j)] = x[slot<16>(j)];
      team_sync<G>();
    }
  } else {
    C* at = buf + pad(t * REST);
#pragma unroll
    for (int m = 0; m < 16 / REST; m++) {
      C y[REST];
#pragma unroll
      for (int k = 0; k < REST; k++) y[k] = x[m * REST + slot<REST>(k)];
      if constexpr (REST > 1) fft<REST, true>(y);
#pragma unroll
      for (int r = 0; r < REST; r++) at[pad(G::T * REST * m) + r] = y[slot<REST>(r)];
    }
    team_sync<G>();
  }
}

// Forward transform of one half of the pair of rows xa, xb (xb null: a zero row). The odd half
// is the transform of z[n] w_2L^n at n = t + T j: w_2L^(T j) = w_32^j is a constant, and the
// lane's common factor w_2L^t goes through the first butterfly, to its outputs (w2).
template <class G, class TIO>
__device__ __forceinline__ void forward(const TIO* __restrict__ xa, const TIO* __restrict__ xb, C* x, C* buf,
                                        const C* w, C w2, bool odd, int t) {
  TIO a[16], b[16];
#pragma unroll
  for (int j = 0; j < 16; j++) a[j] = (xa + G::T * j)[(unsigned)t], b[j] = TIO(0);
  if (xb) {
#pragma unroll
    for (int j = 0; j < 16; j++) b[j] = (xb + G::T * j)[(unsigned)t];
  }
  __asm__ volatile("" ::: "memory");
#pragma unroll
  for (int j = 0; j < 16; j++) x[j] = {io_to_f32(a[j]), io_to_f32(b[j])};
  if (odd) {
#pragma unroll
    for (int j = 1; j < 16; j++) x[j] = rot32<false>(x[j], j);
#pragma unroll
    for (int j = 0; j < 16; j++) x[j] = mul(x[j], w2);
  }
  forward_stage<G, G::L, 0>(x, buf, w, t);
}

// grid: (channel groups, halves from the grid, batch splits). Partial results (one per half
// and batch split when those come from the grid) go to out + part * H * L, summed by
// fg_sum_kernel; otherwise out is dk.
template <int L, class TIO>
__global__ void __launch_bounds__(Geom<L>::NT, Geom<L>::WPE)
    filter_grad_kernel(const TIO* __restrict__ u, const TIO* __restrict__ dy, float* __restrict__ out, int B, int H,
                       int pairs_per_split) {
  typedef Geom<L> G;
  constexpr int T = G::T;
  __shared__ C lds[G::TEAMS * G::SLOTS];
  // a team of whole wavefronts is uniform across them: its row pointers are scalars, and a lane adds
  // one offset for all of its points (an address pair per few points took up to 50 VGPRs, spilled at
  // L = 2048 and 16384: 48 -> 39 us at B=8, H=768, L=2048 fp32, 200 -> 163 at B=4, H=300, L=16384)
  const int team = T >= 64 ? __builtin_amdgcn_readfirstlane(threadIdx.x / T) : (int)threadIdx.x / T;
  const int t = threadIdx.x % T;
  const int half = G::HALVES == 2 ? team & 1 : blockIdx.y;
  const int sub = G::HALVES == 2 ? (team >> 1) % G::SUB : 0;
  const int ch = G::HALVES == 2 ? (team >> 1) / G::SUB : 0;
  const int h = blockIdx.x * G::CH + ch;
  const bool live = h < H;
  C* buf = lds + team * G::SLOTS;
  const int pairs = (B + 1) / 2, p0 = blockIdx.z * pairs_per_split;
  const int np = pairs - p0 < pairs_per_split ? pairs - p0 : pairs_per_split;

  C w[MAXS];
  {
    int rest = L;
#pragma unroll
    for (int s = 0; s + 1 < stages<L>(); s++) {
      w[s] = root(t % (rest / 16), rest);
      rest /= 16;
    }
  }
  const C w2 = root(t, 2 * L);

  C acc[16];
#pragma unroll
  for (int v = 0; v < 16; v++) acc[v] = {0.f, 0.f};
  // every team runs the same number of transforms, so that the barriers match; those past
  // their subset's pairs (and past the last channel) repeat its last rows and leave the sum alone
  const int rounds = (np + G::SUB - 1) / G::SUB;
  for (int r = 0; r < rounds; r++) {
    const int p = r * G::SUB + sub;
    const bool mine = G::SUB * G::CH == 1 || (live && p < np);
    const int b = 2 * (p0 + (p < np ? p : np - 1));
    const size_t row = ((size_t)b * H + (live ? h : H - 1)) * L;
    const size_t next = b + 1 < B ? (size_t)H * L : 0;
    C xu[16], xd[16];
    forward<G, TIO>(u + row, next ? u + row + next : nullptr, xu, buf, w, w2, half != 0, t);
    forward<G, TIO>(dy + row, next ? dy + row + next : nullptr, xd, buf, w, w2, half != 0, t);
    if (mine) {
#pragma unroll
      for (int v = 0; v < 16; v++) {
        acc[v].r += xd[v].r * xu[v].r + xd[v].i * xu[v].i;
        acc[v].i += xd[v].i * xu[v].r - xd[v].r * xu[v].i;
      }
    }
  }

  if constexpr (G::SUB > 1) {
    // the subsets' sums, through their own buffers
    if (sub > 0) {
#pragma unroll
      for (int v = 0; v < 16; v++) buf[v * T + t] = acc[v];
    }
    __syncthreads();
    if (sub == 0) {
#pragma unroll
      for (int s = 1; s < G::SUB; s++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[v] = acc[v] + buf[2 * s * G::SLOTS + v * T + t];
    }
    __syncthreads();
  }
  float y[16];
  if (sub == 0) {
    inverse_stage<G, L, 0>(acc, buf, w, t);
    // acc: the first stage's inputs, twiddled; its inverse butterfly gives n = t + T j, of which
    // the odd half needs the real part of w_2L^-n z[n]: the lane's factor before the butterfly
    if (half) {
#pragma unroll
      for (int k = 0; k < 16; k++) acc[k] = mulc<true>(acc[k], w2);
    }
    fft<16, true>(acc);
#pragma unroll
    for (int j = 0; j < 16; j++) {
      const C z = acc[slot<16>(j)];
      y[j] = (half ? rot32<true>(z, j).r : z.r) * (0.5f / L);
    }
  }
  if constexpr (G::HALVES == 2) {
    float* f = reinterpret_cast<float*>(lds + team * G::SLOTS);
    __syncthreads();  // every team is done with its buffer
    if (half && sub == 0) {
#pragma unroll
      for (int j = 0; j < 16; j++) f[t + T * j] = y[j];
    }
    __syncthreads();
    if (!half && sub == 0 && live) {
      const float* o = reinterpret_cast<const float*>(lds + (team + 1) * G::SLOTS);
      float* d = out + ((size_t)blockIdx.z * H + h) * L;
#pragma unroll
      for (int j = 0; j < 16; j++) (d + T * j)[(unsigned)t] = y[j] + o[t + T * j];
    }
  } else {
    float* d = out + ((size_t)(blockIdx.z * 2 + half) * H + h) * L;
#pragma unroll
    for (int j = 0; j < 16; j++) (d + T * j)[(unsigned)t] = y[j];
  }
}

// dk = the sum of the parts, n floats each (n a multiple of 4)
__global__ void __launch_bounds__(256)
    fg_sum_kernel(const float4* __restrict__ parts, float4* __restrict__ dk, size_t n4, int count) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  float4 a = parts[i];
  for (int p = 1; p < count; p++) {
    const float4 b = parts[p * n4 + i];
    a.x += b.x;
    a.y += b.y;
    a.z += b.z;
    a.w += b.w;
  }
  dk[i] = a;
}

}  // namespace fg
}  // namespace sffft
