// The recurrences' autograd boundary in C++: what HipLIFFunction and
// HipALIFFunction of autograd.py do (the same entry points, outputs and saved
// tensors), without Python in either direction.  A small layer's training
// step is host work: at T=150, [37, 2051] the kernels take 57 us and the pass
// took 96 us with the Python Functions, half of the difference on the autograd
// engine's device thread, where Python code waits for the interpreter lock
// that the caller's thread holds.  With these it takes 57 us; at T=64,
// [4, 128] a pass fell from 44 to 34 us.  Passes of a few hundred us are
// bound by the kernels either way.
//
// The entry points of libmyelin_hip.so are passed in by address (bind), so
// that this module and _lib.py run the same library.

#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/Exceptions.h>
#include <torch/extension.h>

#include <string>

#include "../../include/myelin_hip.h"

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

struct Library {
  decltype(&myelin_lif_fwd_f32) lif_fwd = nullptr;
  decltype(&myelin_lif_bwd_f32) lif_bwd = nullptr;
  decltype(&myelin_alif_fwd_f32) alif_fwd = nullptr;
  decltype(&myelin_alif_bwd_f32) alif_bwd = nullptr;
  decltype(&myelin_last_error) last_error = nullptr;
  PyObject *hip_error = nullptr;  // the class of failed launches; never released
} lib;

// as _lib.call: ValueError for a rejected argument, MyelinHipError else
void check(int rc, const char *name) {
  if (rc == MYELIN_OK) return;
  const std::string message = std::string(name) + ": " + lib.last_error();
  pybind11::gil_scoped_acquire gil;
  PyErr_SetString(rc == MYELIN_EINVAL ? PyExc_ValueError : lib.hip_error, message.c_str());
  python_error error;
  error.persist();
  throw error;
}

// the stream torch launches on, read at call time (a backward may run on the
// engine's device thread)
myelin_stream_t stream_of(const Tensor &t) {
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

float *f32(const Tensor &t) { return t.defined() ? static_cast<float *>(t.data_ptr()) : nullptr; }

Tensor contiguous_f32(const Tensor &g) { return g.defined() ? g.to(torch::kFloat32).contiguous() : g; }

struct Params {
  double decay, rho, threshold, beta, reset, slope;
  int64_t rule, code, chunk;
  bool needs_grad;
};

// x [T, B, N], m0 and (ALIF) a0 [B, N], contiguous fp32.  Returns {final m,
// (final a,) spikes}; for the plain unroll (code MYELIN_SG_NONE) the spikes
// carry no gradient.
template <bool ALIF>
struct Recurrence : torch::autograd::Function<Recurrence<ALIF>> {
  static variable_list forward(AutogradContext *ctx, const Tensor &x, const Tensor &m0, const Params &p) {
    return run(ctx, x, m0, Tensor(), p);
  }
  static variable_list forward(AutogradContext *ctx, const Tensor &x, const Tensor &m0, const Tensor &a0,
                               const Params &p) {
    return run(ctx, x, m0, a0, p);
  }

  static variable_list run(AutogradContext *ctx, const Tensor &x, const Tensor &m0, const Tensor &a0,
                           const Params &p) {
    const int64_t T = x.size(0), B = x.size(1), N = x.size(2);
    Tensor m = torch::empty_like(m0), a, spikes = torch::empty_like(x), ckpt_m, ckpt_a;
    if (ALIF) a = torch::empty_like(a0);
    if (p.needs_grad) {
      ckpt_m = torch::empty({(T + p.chunk - 1) / p.chunk, B, N}, x.options());
      if (ALIF) ckpt_a = torch::empty_like(ckpt_m);
    }
    if (ALIF)
      check(lib.alif_fwd(f32(x), f32(m0), f32(a0), f32(m), f32(a), f32(spikes), nullptr, f32(ckpt_m), f32(ckpt_a), T, B,
                         N, p.decay, p.rho, p.threshold, p.beta, p.reset, p.slope, p.rule, p.chunk, stream_of(x)),
            "myelin_alif_fwd_f32");
    else
      check(lib.lif_fwd(f32(x), f32(m0), f32(m), f32(spikes), nullptr, f32(ckpt_m), T, B, N, p.decay, p.threshold,
                        p.reset, p.slope, p.rule, p.chunk, stream_of(x)),
            "myelin_lif_fwd_f32");
    ctx->set_materialize_grads(false);
    if (p.code == MYELIN_SG_NONE) ctx->mark_non_differentiable({spikes});
    if (p.needs_grad) {
      ctx->save_for_backward(ALIF ? variable_list{x, ckpt_m, ckpt_a} : variable_list{x, ckpt_m});
      ctx->saved_data["p"] = std::vector<double>{p.decay, p.rho,   p.threshold, p.beta,
                                                 p.reset, p.slope, static_cast<double>(p.code),
                                                 static_cast<double>(p.chunk)};
    }
    return ALIF ? variable_list{m, a, spikes} : variable_list{m, spikes};
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    variable_list out(ALIF ? 4 : 3);  // x, m0, (a0,) params
    const Tensor g_m = contiguous_f32(grads[0]), g_a = ALIF ? contiguous_f32(grads[1]) : Tensor(),
                 g_s = contiguous_f32(grads.back());
    if (!g_m.defined() && !g_a.defined() && !g_s.defined()) return out;
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &x = saved[0];
    const std::vector<double> p = ctx->saved_data["p"].toDoubleVector();
    const int64_t T = x.size(0), BN = x.size(1) * x.size(2), chunk = static_cast<int64_t>(p[7]);
    const int code = static_cast<int>(p[6]);
    const c10::DeviceGuard guard(x.device());
    Tensor gx = torch::empty_like(x), gm0 = torch::empty({x.size(1), x.size(2)}, x.options()), ga0;
    if (ALIF) ga0 = torch::empty_like(gm0);
    if (ALIF)
      check(lib.alif_bwd(f32(x), f32(saved[1]), f32(saved[2]), f32(g_s), f32(g_m), f32(g_a), f32(gx), f32(gm0),
                         f32(ga0), T, BN, p[0], p[1], p[2], p[3], p[4], p[5], code, chunk, stream_of(x)),
            "myelin_alif_bwd_f32");
    else
      check(lib.lif_bwd(f32(x), f32(saved[1]), f32(g_s), f32(g_m), f32(gx), f32(gm0), T, BN, p[0], p[2], p[4], p[5],
                        code, chunk, stream_of(x)),
            "myelin_lif_bwd_f32");
    if (ctx->needs_input_grad(0)) out[0] = gx;
    if (ctx->needs_input_grad(1)) out[1] = gm0;
    if (ALIF && ctx->needs_input_grad(2)) out[2] = ga0;
    return out;
  }
};

template <bool ALIF, class... States>
variable_list apply(Params p, const Tensor &x, const States &...states) {
  p.needs_grad = torch::GradMode::is_enabled() && (x.requires_grad() || ... || states.requires_grad());
  const c10::DeviceGuard guard(x.device());
  return Recurrence<ALIF>::apply(x, states..., p);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("bind", [](uintptr_t lif_fwd, uintptr_t lif_bwd, uintptr_t alif_fwd, uintptr_t alif_bwd, uintptr_t last_error,
                   const pybind11::object &hip_error) {
    lib.lif_fwd = reinterpret_cast<decltype(lib.lif_fwd)>(lif_fwd);
    lib.lif_bwd = reinterpret_cast<decltype(lib.lif_bwd)>(lif_bwd);
    lib.alif_fwd = reinterpret_cast<decltype(lib.alif_fwd)>(alif_fwd);
    lib.alif_bwd = reinterpret_cast<decltype(lib.alif_bwd)>(alif_bwd);
    lib.last_error = reinterpret_cast<decltype(lib.last_error)>(last_error);
    lib.hip_error = pybind11::object(hip_error).release().ptr();
  });
  // as ctypes does for the library's calls: other threads run meanwhile
  const auto nogil = pybind11::call_guard<pybind11::gil_scoped_release>();
  m.def("lif", [](const Tensor &x, const Tensor &m0, double decay, double threshold, double reset, double slope,
                  int64_t rule, int64_t code, int64_t chunk) {
    return apply<false>(Params{decay, 0.0, threshold, 0.0, reset, slope, rule, code, chunk, false}, x, m0);
  }, nogil);
  m.def("alif", [](const Tensor &x, const Tensor &m0, const Tensor &a0, double decay, double rho, double threshold,
                   double beta, double reset, double slope, int64_t rule, int64_t code, int64_t chunk) {
    return apply<true>(Params{decay, rho, threshold, beta, reset, slope, rule, code, chunk, false}, x, m0, a0);
  }, nogil);
}
