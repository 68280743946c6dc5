// PyTorch operators over the C ABI of libsffft.so, registered from C++.
//
// The reference names a library with a PyTorch binding as its next step (README.md:177),
// for the long-convolution layers of Hyena/H3/S4-style models (README.md:11):
//
//   sffft::spectrum(Tensor k, int[] plan, bool conj=False) -> Tensor
//                                    k [H, L] fp32 -> [H, 2L] complex64 (conj: its conjugate)
//   sffft::conv(Tensor u, Tensor kf, int[] plan) -> Tensor  u [B, H, L] fp32 or bf16
//   sffft::corr(Tensor u, Tensor kf, int[] plan) -> Tensor  the anti-causal correlation, conv's
//                                    adjoint in u, with conv's spectrum
//   sffft::filter_grad(Tensor u, Tensor dy) -> Tensor  the filter's gradient [H, L] fp32
//   sffft::longconv(Tensor u, Tensor k, Tensor kf, int[] plan) -> Tensor  conv(u, kf), with
//                                    gradients for u and for the filter k that kf was made from
//
// `plan` is the nine sffft_plan fields (r0, r1, r2, waves, acc, cached, seqs, mode, channels).
// Each operator launches on the current stream of its input's device, so it is ordered with
// the caller's work and captures into graphs. The GPU kernels are the library's; this file is
// host code only (no kernel of its own), built with the host compiler against torch's headers.
//
// Registering here rather than through torch.library.custom_op keeps the per-call host cost
// at the dispatcher's: the Python wrappers of custom_op (autograd, aliasing checks) took about
// 9 us per call, longer than the kernel itself at L <= 2048. The fake (meta) implementations,
// used only while tracing, stay in Python (sffft_amd/torch_ops.py).
//
// Gradients: sffft::conv is differentiable in u. The adjoint of causal convolution is the
// anti-causal correlation du[m] = sum_{n >= m} dy[n] k[n - m], which with the N = 2L zero padding
// is IDFT(DFT(dy) * conj(K))[m] for m < L: sffft::corr, the same kernels with conjugate DFT and
// twiddle tables, on the same spectrum and with no time reversal of dy or du. sffft::longconv is
// differentiable in u and in the filter. sffft::spectrum has no gradient; backpropagating through
// it raises.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/autograd.h>
#include <torch/library.h>

#include "sffft.h"

namespace {

sffft_plan to_plan(c10::IntArrayRef f) {
  TORCH_CHECK(f.size() == 9, "a plan has 9 fields (r0, r1, r2, waves, acc, cached, seqs, mode, channels), got ",
              f.size());
  return sffft_plan{(int)f[0], (int)f[1], (int)f[2], (int)f[3], (int)f[4],
                    (int)f[5], (int)f[6], (int)f[7], (int)f[8]};
}

void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

void check(int rc, const char* what) {
  TORCH_CHECK(rc == SFFFT_OK, what, " failed: ", sffft_strerror(rc), " (", rc, ") ", sffft_last_error());
}

at::Tensor spectrum_gpu(const at::Tensor& k_in, c10::IntArrayRef plan_fields, bool conj) {
  TORCH_CHECK(k_in.is_cuda() && k_in.scalar_type() == at::kFloat && k_in.dim() == 2,
              "sffft::spectrum: k must be a [H, L] float32 GPU tensor");
  // torch labels GPU tensors CUDA on this backend too; the generic guard picks the
  // backend's own device guard for that label
  const c10::DeviceGuard guard(k_in.device());
  const at::Tensor k = k_in.contiguous();
  const int64_t H = k.size(0), L = k.size(1);
  TORCH_CHECK(H <= INT32_MAX && L <= INT32_MAX, "sffft::spectrum: shape too large");
  const sffft_plan p = to_plan(plan_fields);
  at::Tensor kf = at::empty({H, 2 * L}, k.options().dtype(at::kComplexFloat));
  at::Tensor work = at::empty_like(kf);  // sffft_spectrum_bytes(H, L): scratch, clobbered
  check((conj ? sffft_spectrum_conj : sffft_spectrum)(k.data_ptr<float>(), (int)H, (int)L, &p, kf.data_ptr(),
                                                       work.data_ptr(), current_stream()),
        "sffft_spectrum");
  return kf;
}

at::Tensor run_conv(const at::Tensor& u_in, const at::Tensor& kf_in, c10::IntArrayRef plan_fields, bool corr) {
  at::Tensor kf = kf_in;
  TORCH_CHECK(u_in.is_cuda() && u_in.dim() == 3, "sffft::conv: u must be a [B, H, L] GPU tensor");
  TORCH_CHECK(u_in.scalar_type() == at::kFloat || u_in.scalar_type() == at::kBFloat16,
              "sffft::conv: u must be float32 or bfloat16");
  TORCH_CHECK(kf.is_cuda() && kf.scalar_type() == at::kComplexFloat && kf.is_contiguous(),
              "sffft::conv: kf must be a contiguous complex64 GPU tensor from sffft::spectrum");
  TORCH_CHECK(kf.device() == u_in.device(), "sffft::conv: u and kf must be on the same device");
  const c10::DeviceGuard guard(u_in.device());
  const at::Tensor u = u_in.contiguous();
  const int64_t B = u.size(0), H = u.size(1), L = u.size(2);
  TORCH_CHECK(B <= INT32_MAX && H <= INT32_MAX && L <= INT32_MAX, "sffft::conv: shape too large");
  // the kernels read H rows of 2L values from the start of kf (row h is channel h's
  // spectrum): a spectrum of fewer channels or of another length would be read past its end
  TORCH_CHECK(kf.dim() == 2 && kf.size(0) == H && kf.size(1) == 2 * L, "sffft::conv: kf must be [H, 2L] = [", H,
              ", ", 2 * L, "] for u of shape ", u.sizes(), ", got ", kf.sizes());
  const sffft_plan p = to_plan(plan_fields);
  if (corr && !p.cached) {  // in-kernel DFT fragments: no conjugate ones, so the conjugate spectrum
    kf = at::conj_physical(kf);
    corr = false;
  }
  at::Tensor y = at::empty_like(u);
  const bool bf16 = u.scalar_type() == at::kBFloat16;
  void* s = current_stream();
  if (p.mode == 2) {  // multi-pass: the workspace comes from torch's allocator
    const size_t wb = sffft_work_bytes((int)B, (int)H, (int)L, &p);
    at::Tensor work = at::empty({(int64_t)std::max<size_t>(wb, 16)}, u.options().dtype(at::kByte));
    const size_t have = (size_t)work.numel();
    const auto run16 = corr ? sffft_corr_long_bf16 : sffft_conv_long_bf16;
    const auto run32 = corr ? sffft_corr_long_f32 : sffft_conv_long_f32;
    check(bf16 ? run16(reinterpret_cast<const uint16_t*>(u.data_ptr()), kf.data_ptr(),
                       reinterpret_cast<uint16_t*>(y.data_ptr()), work.data_ptr(), have, (int)B, (int)H, (int)L, &p, s)
               : run32(u.data_ptr<float>(), kf.data_ptr(), y.data_ptr<float>(), work.data_ptr(), have, (int)B, (int)H,
                       (int)L, &p, s),
          "sffft_conv_long");
  } else {
    const auto run16 = corr ? sffft_corr_bf16 : sffft_conv_bf16;
    const auto run32 = corr ? sffft_corr_f32 : sffft_conv_f32;
    check(bf16 ? run16(reinterpret_cast<const uint16_t*>(u.data_ptr()), kf.data_ptr(),
                       reinterpret_cast<uint16_t*>(y.data_ptr()), (int)B, (int)H, (int)L, &p, s)
               : run32(u.data_ptr<float>(), kf.data_ptr(), y.data_ptr<float>(), (int)B, (int)H, (int)L, &p, s),
          "sffft_conv");
  }
  return y;
}

at::Tensor conv_gpu(const at::Tensor& u, const at::Tensor& kf, c10::IntArrayRef plan) {
  return run_conv(u, kf, plan, false);
}

at::Tensor corr_gpu(const at::Tensor& u, const at::Tensor& kf, c10::IntArrayRef plan) {
  return run_conv(u, kf, plan, true);
}

at::Tensor longconv_gpu(const at::Tensor& u, const at::Tensor& k, const at::Tensor& kf, c10::IntArrayRef plan) {
  // what the backward pass needs, refused here rather than there: the filter's gradient has k's shape and
  // type, and a kernel for these lengths only
  TORCH_CHECK(u.dim() == 3 && k.dim() == 2 && k.size(0) == u.size(1) && k.size(1) == u.size(2) &&
                  k.scalar_type() == at::kFloat && k.device() == u.device(),
              "sffft::longconv: k must be the [H, L] float32 filter of u [B, H, L] on its device, got ", k.sizes(), " ",
              k.scalar_type(), " for u of shape ", u.sizes());
  const int64_t L = u.size(2);
  TORCH_CHECK(L >= 128 && L <= 16384 && (L & (L - 1)) == 0,
              "sffft::longconv: L must be a power of two from 128 to 16384, got ", L,
              " (LongConv takes the multi-pass lengths)");
  return run_conv(u, kf, plan, false);
}

// dk[h, j] = sum_b sum_{n >= j} dy[b, h, n] u[b, h, n - j], fp32 [H, L]
at::Tensor filter_grad_gpu(const at::Tensor& u_in, const at::Tensor& dy_in) {
  TORCH_CHECK(u_in.is_cuda() && u_in.dim() == 3 && dy_in.sizes() == u_in.sizes() && dy_in.device() == u_in.device(),
              "sffft::filter_grad: u and dy must be [B, H, L] tensors of one shape on one GPU, got ", u_in.sizes(),
              " and ", dy_in.sizes());
  TORCH_CHECK((u_in.scalar_type() == at::kFloat || u_in.scalar_type() == at::kBFloat16) &&
                  dy_in.scalar_type() == u_in.scalar_type(),
              "sffft::filter_grad: u and dy must both be float32 or both bfloat16");
  const c10::DeviceGuard guard(u_in.device());
  const at::Tensor u = u_in.contiguous(), dy = dy_in.contiguous();
  const int64_t B = u.size(0), H = u.size(1), L = u.size(2);
  TORCH_CHECK(B <= INT32_MAX && H <= INT32_MAX && L <= INT32_MAX, "sffft::filter_grad: shape too large");
  at::Tensor dk = at::empty({H, L}, u.options().dtype(at::kFloat));
  const size_t wb = sffft_filter_grad_work_bytes((int)B, (int)H, (int)L);
  at::Tensor work;
  if (wb) work = at::empty({(int64_t)wb}, u.options().dtype(at::kByte));
  void* w = wb ? work.data_ptr() : nullptr;
  check(u.scalar_type() == at::kBFloat16
            ? sffft_filter_grad_bf16(reinterpret_cast<const uint16_t*>(u.data_ptr()),
                                     reinterpret_cast<const uint16_t*>(dy.data_ptr()), dk.data_ptr<float>(), w, wb,
                                     (int)B, (int)H, (int)L, current_stream())
            : sffft_filter_grad_f32(u.data_ptr<float>(), dy.data_ptr<float>(), dk.data_ptr<float>(), w, wb, (int)B,
                                    (int)H, (int)L, current_stream()),
        "sffft_filter_grad");
  return dk;
}

at::Tensor call_conv(const at::Tensor& u, const at::Tensor& kf, c10::IntArrayRef plan) {
  static const auto op = c10::Dispatcher::singleton()
                             .findSchemaOrThrow("sffft::conv", "")
                             .typed<at::Tensor(const at::Tensor&, const at::Tensor&, c10::IntArrayRef)>();
  return op.call(u, kf, plan);
}

at::Tensor call_corr(const at::Tensor& u, const at::Tensor& kf, c10::IntArrayRef plan) {
  static const auto op = c10::Dispatcher::singleton()
                             .findSchemaOrThrow("sffft::corr", "")
                             .typed<at::Tensor(const at::Tensor&, const at::Tensor&, c10::IntArrayRef)>();
  return op.call(u, kf, plan);
}

at::Tensor call_filter_grad(const at::Tensor& u, const at::Tensor& dy) {
  static const auto op = c10::Dispatcher::singleton()
                             .findSchemaOrThrow("sffft::filter_grad", "")
                             .typed<at::Tensor(const at::Tensor&, const at::Tensor&)>();
  return op.call(u, dy);
}

at::Tensor call_longconv(const at::Tensor& u, const at::Tensor& k, const at::Tensor& kf, c10::IntArrayRef plan) {
  static const auto op =
      c10::Dispatcher::singleton()
          .findSchemaOrThrow("sffft::longconv", "")
          .typed<at::Tensor(const at::Tensor&, const at::Tensor&, const at::Tensor&, c10::IntArrayRef)>();
  return op.call(u, k, kf, plan);
}

at::Tensor call_spectrum(const at::Tensor& k, c10::IntArrayRef plan, bool conj) {
  static const auto op = c10::Dispatcher::singleton()
                             .findSchemaOrThrow("sffft::spectrum", "")
                             .typed<at::Tensor(const at::Tensor&, c10::IntArrayRef, bool)>();
  return op.call(k, plan, conj);
}

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// conv and corr are each other's adjoints in u.
template <bool CORR>
class ConvFn : public torch::autograd::Function<ConvFn<CORR>> {
 public:
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& u, const at::Tensor& kf,
                            c10::IntArrayRef plan) {
    ctx->save_for_backward({kf});
    ctx->saved_data["plan"] = plan.vec();
    at::AutoDispatchBelowADInplaceOrView guard;
    return CORR ? call_corr(u, kf, plan) : call_conv(u, kf, plan);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const at::Tensor kf = ctx->get_saved_variables()[0];
    const std::vector<int64_t> plan = ctx->saved_data["plan"].toIntVector();
    at::Tensor du;
    if (ctx->needs_input_grad(0)) {
      const at::Tensor dy = grads[0].contiguous();
      du = CORR ? call_conv(dy, kf, plan) : call_corr(dy, kf, plan);
    }
    return {du, at::Tensor(), at::Tensor()};
  }
};

// The filter gradient where its own gradient is recorded (a second derivative): linear in dy, with
// the adjoint dy' = causal_conv(u, g) for g [H, L], which longconv differentiates further. u takes no
// gradient here.
class FilterGradFn : public torch::autograd::Function<FilterGradFn> {
 public:
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& u, const at::Tensor& dy, c10::IntArrayRef plan) {
    ctx->save_for_backward({u});
    ctx->saved_data["plan"] = plan.vec();
    at::AutoDispatchBelowADInplaceOrView guard;
    return call_filter_grad(u, dy);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const at::Tensor u = ctx->get_saved_variables()[0].detach();
    const std::vector<int64_t> plan = ctx->saved_data["plan"].toIntVector();
    at::Tensor ddy;
    if (ctx->needs_input_grad(1)) {
      const at::Tensor g = grads[0].contiguous();
      ddy = call_longconv(u, g, call_spectrum(g.detach(), plan, false), plan);
    }
    return {at::Tensor(), ddy, at::Tensor()};
  }
};

// y = conv(u, kf) with gradients for u and for the filter k that kf was made from (L <= 16384).
class LongConvFn : public torch::autograd::Function<LongConvFn> {
 public:
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& u, const at::Tensor& k, const at::Tensor& kf,
                            c10::IntArrayRef plan) {
    ctx->save_for_backward({u, kf});
    ctx->saved_data["plan"] = plan.vec();
    at::AutoDispatchBelowADInplaceOrView guard;
    return call_longconv(u, k, kf, plan);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const std::vector<int64_t> plan = ctx->saved_data["plan"].toIntVector();
    const at::Tensor u = saved[0];
    const at::Tensor dy = grads[0].to(u.scalar_type()).contiguous();
    at::Tensor du, dk;
    if (ctx->needs_input_grad(0)) du = call_corr(dy, saved[1], plan);
    if (ctx->needs_input_grad(1)) {
      if (at::GradMode::is_enabled() && dy.requires_grad())
        dk = FilterGradFn::apply(u.detach(), dy, plan);
      else
        dk = call_filter_grad(u.detach(), dy);
    }
    return {du, dk, at::Tensor(), at::Tensor()};
  }
};

class SpectrumFn : public torch::autograd::Function<SpectrumFn> {
 public:
  static at::Tensor forward(AutogradContext*, const at::Tensor& k, c10::IntArrayRef plan, bool conj) {
    at::AutoDispatchBelowADInplaceOrView guard;
    return call_spectrum(k, plan, conj);
  }
  static variable_list backward(AutogradContext*, variable_list) {
    TORCH_CHECK(false, "sffft::spectrum has no gradient with respect to the filter");
    return {};
  }
};

at::Tensor conv_autograd(const at::Tensor& u, const at::Tensor& kf, c10::IntArrayRef plan) {
  return ConvFn<false>::apply(u, kf, plan);
}

at::Tensor corr_autograd(const at::Tensor& u, const at::Tensor& kf, c10::IntArrayRef plan) {
  return ConvFn<true>::apply(u, kf, plan);
}

at::Tensor longconv_autograd(const at::Tensor& u, const at::Tensor& k, const at::Tensor& kf, c10::IntArrayRef plan) {
  return LongConvFn::apply(u, k, kf, plan);
}

at::Tensor spectrum_autograd(const at::Tensor& k, c10::IntArrayRef plan, bool conj) {
  return SpectrumFn::apply(k, plan, conj);
}

}  // namespace

TORCH_LIBRARY(sffft, m) {
  m.def("spectrum(Tensor k, int[] plan, bool conj=False) -> Tensor");
  m.def("conv(Tensor u, Tensor kf, int[] plan) -> Tensor");
  m.def("corr(Tensor u, Tensor kf, int[] plan) -> Tensor");
  m.def("longconv(Tensor u, Tensor k, Tensor kf, int[] plan) -> Tensor");
  m.def("filter_grad(Tensor u, Tensor dy) -> Tensor");
}

// torch names its GPU dispatch key CUDA on every backend, this one included.
TORCH_LIBRARY_IMPL(sffft, CUDA, m) {
  m.impl("spectrum", &spectrum_gpu);
  m.impl("conv", &conv_gpu);
  m.impl("corr", &corr_gpu);
  m.impl("longconv", &longconv_gpu);
  m.impl("filter_grad", &filter_grad_gpu);
}

TORCH_LIBRARY_IMPL(sffft, Autograd, m) {
  m.impl("corr", &corr_autograd);
  m.impl("longconv", &longconv_autograd);
  m.impl("spectrum", &spectrum_autograd);
  m.impl("conv", &conv_autograd);
}
