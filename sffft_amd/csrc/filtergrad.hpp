// Filter gradient of the causal convolution, in one launch (two when its work is split):
//
//   dk[h][j] = sum_b sum_{n >= j} dy[b][h][n] u[b][h][n - j],   j < L,  L = 128..16384
//
// The sum over b commutes with the transforms, so a channel needs one inverse transform
// whatever its batch: with U_b and D_b the zero-padded 2L-point spectra of the rows,
// dk = IDFT(sum_b D_b conj(U_b)). Two batch rows travel as one complex row, z = x_b + i x_b+1:
// then Re IDFT(Z_dy conj(Z_u)) is already the sum of both rows' correlations (the cross terms
// are the imaginary part), so the pair is never taken apart. The cross terms still round: dy of one row
// times u of the other may be far larger than either row's own product. So where they differ, row b + 1
// of u is scaled by a power of two to the size of row b, and that row of dy by its inverse
// (balance()): the sum is unchanged, and each cross term is bounded by a row's own product.
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
// fp32 throughout: 3e-7 (L = 128) to 7e-7 (L = 16384) from 64 bits, also for rows 1e12 apart in size (1e-5
// at a ratio of 100 and 0.2 at 1e6 without the balance, which costs 0 to 4% of the time), where fp16
// operands gave 2e-4 to 3.4e-4 (the composition of the spectrum of every row, a convolution and a sum over b, which this
// replaced). Bound by VALU issue, about 600 fp32 instructions per lane and transform, and by
// what hides latency beside it, 2 to 3 wavefronts per SIMD. Measured, that composition before and this
// kernel now: B=8 H=768 L=1024 fp32 220 -> 20 us (2.5 TB/s of u and dy, 0.5 of a copy), B=6
// H=513 L=4096 bf16 610 -> 53, B=5 H=320 L=8192 fp32 540 -> 88.
#pragma once
#include <type_traits>

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
  // VGPRs, 27 to 47 spilled, mostly the sums during a transform) beat one: 90 against 107 us at
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

// Radix-16 stages on REST-point blocks, REST > 16, after the first (forward()): butterfly, twiddle,
// exchange; then the last stage of radix REST <= 16.
template <class G, int REST, int S>
__device__ __forceinline__ void forward_stage(C* x, C* buf, const C* w, int t) {
  if constexpr (REST > 16) {
    constexpr int sJ = REST / 16;
    C* at = buf + slot_base<sJ>(t);
#pragma unroll
    for (int j = 0; j < 16; j++) x[j] = at[slot_off<sJ>(j)];
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

// Sum of v over groups of W consecutive lanes (2 to 64): in each of their lanes, for W = 64 as a scalar.
template <int W>
__device__ __forceinline__ float lane_sum(float v) {
  auto dpp = [](float x, auto ctrl, auto rows) {
    constexpr int c = decltype(ctrl)::value, m = decltype(rows)::value;
    const int b = __builtin_bit_cast(int, x);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, b, c, m, 0xf, false));
  };
  constexpr std::integral_constant<int, 0xf> all{};
  v += dpp(v, std::integral_constant<int, 0xb1>{}, all);                            // lane ^ 1
  if constexpr (W >= 4) v += dpp(v, std::integral_constant<int, 0x4e>{}, all);    // lane ^ 2
  if constexpr (W >= 8) v += dpp(v, std::integral_constant<int, 0x141>{}, all);   // mirrored in 8: the other four
  if constexpr (W >= 16) v += dpp(v, std::integral_constant<int, 0x140>{}, all);  // in 16: the other eight
  if constexpr (W == 32) v += __shfl_xor(v, 16);
  if constexpr (W == 64) {  // lane 15 to the next 16 lanes, lane 31 to the next 32
    v += dpp(v, std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});
    v += dpp(v, std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});
    v = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
  }
  return v;
}

// The balance of a pair: the power of two that takes the size of its second row (the imaginary
// parts) towards that of the first, as its exponent. A row's size is the root of the sum of its
// lanes' largest squares (within a factor of 4 of its norm). Pairs whose rows are within a factor of 8 of
// each other in every lane, as equal rows are, keep their scale: what they cost is lane_sizes() and a
// vote. Others are taken to within a factor of 2, by at most 2^48: beside a row of zeros too, whose dy would
// only round; fp32 keeps the inverse factor in range for dy up to 1e24.
__device__ __forceinline__ float2 lane_sizes(const C* x) {
  float a = 0.f, b = 0.f;
#pragma unroll
  for (int j = 0; j < 16; j += 2) {
    a = fmaxf(fmaxf(fabsf(x[j].r), fabsf(x[j + 1].r)), a);
    b = fmaxf(fmaxf(fabsf(x[j].i), fabsf(x[j + 1].i)), b);
  }
  return make_float2(a, b);
}
__device__ __forceinline__ bool unequal(float2 s) {  // by about a factor of 8 (bit patterns 3 exponents apart)
  const unsigned d = __builtin_bit_cast(unsigned, s.x) - __builtin_bit_cast(unsigned, s.y);
  return d + (3u << 23) > 6u << 23;
}
template <class G>
__device__ __forceinline__ int balance(float2 size2) {
  int ea = __builtin_bit_cast(int, size2.x) >> 23, eb = __builtin_bit_cast(int, size2.y) >> 23;  // not negative
  if constexpr (G::T >= 64) {
    ea = __builtin_amdgcn_readfirstlane(ea);
    eb = __builtin_amdgcn_readfirstlane(eb);
  }
  const int k = (ea - eb) / 2;
  return k < -48 ? -48 : k > 48 ? 48 : k;
}
__device__ __forceinline__ float pow2(int k) { return __builtin_bit_cast(float, (127 + k) << 23); }

// A team of several wavefronts: its wavefronts' sizes, and the latest pair with unequal rows.
template <int T>
struct Sizes {
  float2 wave[T > 64 ? T / 64 : 1];
  int vote;
};

// Forward transform of one half of the pair of rows xa, xb (xb null: a zero row). The odd half
// is the transform of z[n] w_2L^n at n = t + T j: w_2L^(T j) = w_32^j is a constant, and the
// lane's common factor w_2L^t goes through the first butterfly, to its outputs (w2).
// U: of u, which sets the pair's balance k; otherwise of dy. Teams of several wavefronts vote across
// the first stage's barrier, and the rare pair that is to be scaled runs that stage again: a barrier
// before it would keep the wavefronts whose rows have arrived from starting (5% at L = 16384).
template <class G, bool U, class TIO>
__device__ __forceinline__ void forward(const TIO* __restrict__ xa, const TIO* __restrict__ xb, C* x, C* buf,
                                        Sizes<G::T>* sizes, int pair, const C* w, C w2, bool odd, int t, int& k) {
  auto load = [&](int t) {
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
  };
  auto scale = [&](int e) {
    const float c = pow2(e);
#pragma unroll
    for (int j = 0; j < 16; j++) x[j].i *= c;
  };
  auto first_stage = [&](int t) {
    if (odd) {
#pragma unroll
      for (int j = 1; j < 16; j++) x[j] = rot32<false>(x[j], j);
#pragma unroll
      for (int j = 0; j < 16; j++) x[j] = mul(x[j], w2);
    }
    C* at = buf + slot_base<G::T>(t);
    fft<16, false>(x);
    twiddle16<false, true>(x, w[0]);
#pragma unroll
    for (int v = 0; v < 16; v++) at[slot_off<G::T>(v)] = x[slot<16>(v)];
    team_sync<G>();
  };
  constexpr int W = G::T < 64 ? G::T : 64;
  load(t);
  if constexpr (U) {
    k = 0;
    if (xb) {
      float2 s = lane_sizes(x);
      const uint64_t v = __ballot(unequal(s));
      if (v) {
        if constexpr (G::T > 64) {
          sizes->vote = pair;
        } else {
          s = make_float2(lane_sum<W>(s.x * s.x), lane_sum<W>(s.y * s.y));
          const uint64_t mine = W == 64 ? v : v >> (threadIdx.x & 63 & ~(W - 1)) & ((1ull << (W & 63)) - 1);
          k = mine ? balance<G>(s) : 0;
        }
      }
    }
  }
  if (k) scale(U ? k : -k);
  first_stage(t);
  if constexpr (U && G::T > 64) {
    if (xb && __builtin_amdgcn_readfirstlane(sizes->vote) == pair) {
      // on a lane index of its own, so that nothing of this block is made ahead of it and kept: at T = 1024,
      // where registers are shortest, all of it, below only the slots (the rest is shared with the first
      // time: 157 against 166 us at B=4, H=300, L=16384 fp32, but 92 against 88 at B=5, H=320, L=8192)
      int l = t;
      __asm__ volatile("" : "+v"(l));
      const int lane = G::T > 512 ? l : t;
      load(lane);
      float2 s = lane_sizes(x);
      s = make_float2(lane_sum<W>(s.x * s.x), lane_sum<W>(s.y * s.y));
      if ((l & 63) == 0) sizes->wave[l >> 6] = s;
      team_sync<G>();
      s = sizes->wave[l & (G::T / 64 - 1)];
      k = balance<G>(make_float2(lane_sum<G::T / 64>(s.x), lane_sum<G::T / 64>(s.y)));
      scale(k);
      first_stage(lane);
    }
  }
  forward_stage<G, G::L / 16, 1>(x, buf, w, t);
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
  __shared__ fg::Sizes<T> sizes_[T > 64 ? G::TEAMS : 1];
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
  fg::Sizes<T>* sizes = sizes_ + (T > 64 ? team : 0);
  if constexpr (T > 64) {
    if (t == 0) sizes->vote = -1;
    __syncthreads();
  }
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
    int k;
    forward<G, true>(u + row, next ? u + row + next : nullptr, xu, buf, sizes, r, w, w2, half != 0, t, k);
    forward<G, false>(dy + row, next ? dy + row + next : nullptr, xd, buf, sizes, r, w, w2, half != 0, t, k);
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
