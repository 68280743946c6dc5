// Instantiates the filter-gradient kernels (filtergrad.hpp) and their launcher and C ABI.
#include <climits>

#include "../../include/sffft.h"
#include "filtergrad.hpp"
#include "registry.hpp"

namespace sffft {
namespace {

// How a call is split: workgroups along the batch (each takes whole rounds of SUB pairs), and the
// partial results they and the two halves leave.
struct Split {
  int halves, ch, pairs_per_split, splits, parts;
};

// Lengths whose workgroup holds one half leave two parts anyway. The batch is split further only
// while the channels alone leave the chip short of wavefronts (about 12 per CU, what the kernel's
// registers allow): each split repeats the inverse transform and adds a part to the sum.
template <int L>
Split split_of(int B, int H) {
  typedef fg::Geom<L> G;
  const int pairs = (B + 1) / 2, rounds = (pairs + G::SUB - 1) / G::SUB;
  const long long waves = (long long)((H + G::CH - 1) / G::CH) * (3 - G::HALVES) * (G::NT / 64);
  long long z = 256 * 12 / waves;
  z = z < 1 ? 1 : z > rounds ? rounds : z;
  const int per = (int)((rounds + z - 1) / z) * G::SUB, splits = (pairs + per - 1) / per;
  return {3 - G::HALVES, G::CH, per, splits, splits * (3 - G::HALVES)};
}

template <int L, class TIO>
hipError_t launch(const void* u, const void* dy, float* dk, void* work, int B, int H, const Split& s, hipStream_t st) {
  typedef fg::Geom<L> G;
  float* out = s.parts > 1 ? static_cast<float*>(work) : dk;
  hipLaunchKernelGGL((fg::filter_grad_kernel<L, TIO>),
                     dim3((unsigned)((H + G::CH - 1) / G::CH), (unsigned)s.halves, (unsigned)s.splits), dim3(G::NT), 0,
                     st, static_cast<const TIO*>(u), static_cast<const TIO*>(dy), out, B, H, s.pairs_per_split);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess || s.parts == 1) return err;
  const size_t n4 = (size_t)H * L / 4;
  hipLaunchKernelGGL(fg::fg_sum_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st,
                     static_cast<const float4*>(work), reinterpret_cast<float4*>(dk), n4, s.parts);
  return hipGetLastError();
}

// f(length) for the compiled lengths
template <class F>
bool with_length(int L, F f) {
  switch (L) {
    case 128: f(std::integral_constant<int, 128>{}); return true;
    case 256: f(std::integral_constant<int, 256>{}); return true;
    case 512: f(std::integral_constant<int, 512>{}); return true;
    case 1024: f(std::integral_constant<int, 1024>{}); return true;
    case 2048: f(std::integral_constant<int, 2048>{}); return true;
    case 4096: f(std::integral_constant<int, 4096>{}); return true;
    case 8192: f(std::integral_constant<int, 8192>{}); return true;
    case 16384: f(std::integral_constant<int, 16384>{}); return true;
    default: return false;
  }
}

}  // namespace

// 0 parts: not a compiled length
int filter_grad_parts(int B, int H, int L) {
  int parts = 0;
  with_length(L, [&](auto l) { parts = split_of<decltype(l)::value>(B, H).parts; });
  return parts;
}

hipError_t filter_grad(const void* u, const void* dy, float* dk, void* work, int B, int H, int L, int io,
                       hipStream_t st) {
  hipError_t err = hipErrorInvalidValue;
  with_length(L, [&](auto l) {
    constexpr int LL = decltype(l)::value;
    const Split s = split_of<LL>(B, H);
    err = io ? launch<LL, uint16_t>(u, dy, dk, work, B, H, s, st) : launch<LL, float>(u, dy, dk, work, B, H, s, st);
  });
  return err;
}

}  // namespace sffft
