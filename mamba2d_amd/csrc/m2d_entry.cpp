// m2d_entry.cpp -- the scan's entry points in eager mode, issued from C++.
//
// m2dscan::entry is the projections and the scan (models/kernels/wavefront_cuda.py:315-347) as one autograd function:
// the sequence of wf_cuda_fn_proj in wavefront.py, which stays for compiled callers.  m2dscan::scan is a scan on given
// parameters that nothing will be differentiated through.  Small problems are bound by the host: forward and backward of
// one 14x14x64 bf16 grid took 160 to 225 us through a Python autograd function around four dispatched operators and take
// 106 from here (its forward alone 33 and 25, a scan alone 19 and 11).
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include "m2d_torch.h"

namespace {

using at::Tensor;
using m2dshim::dispatched;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The parameters, in the order of the operator's list: AT_log, AL_log, x_proj_w, dt_projT_w, dt_projT_b, dt_projL_w, dt_projL_b, D.
constexpr int kPar = 8;

// Contiguous and 16-byte aligned (a contiguous view into a larger buffer may start anywhere).
Tensor whole(const Tensor& t) {
  Tensor c = t.contiguous();
  return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 ? c.clone() : c;
}

std::vector<Tensor> as_f32(const std::vector<Tensor>& p) {
  bool all16 = true;
  for (const Tensor& t : p) all16 &= t.scalar_type() == at::kBFloat16 && t.is_cuda();
  std::vector<Tensor> out(kPar);
  for (int i = 0; i < kPar; ++i) out[i] = all16 ? p[i].contiguous() : whole(p[i].to(at::kFloat));
  return all16 ? m2dshim::widen(out) : out;
}

struct Forward { Tensor y, low, dT, dL, BC, ck; };

Forward forward_of(const Tensor& x, const std::vector<Tensor>& w, bool flip, bool keep, int64_t interval) {
  auto pr = m2dshim::proj_fwd(x, w[2], w[3], w[4], w[5], w[6], w[0].size(1), true, true);
  Forward f{{}, pr[0], pr[1], pr[2], pr[3], {}};
  std::tie(f.y, f.ck) = m2dshim::scan_y(x, f.dT, f.dL, w[0], w[1], f.BC, pr[4], pr[5], w[7], keep, flip, true, true, interval);
  return f;
}

struct Entry : public torch::autograd::Function<Entry> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_in, at::TensorList params, bool full, bool flip, bool keep, int64_t interval) {
    const std::vector<Tensor> raw(params.begin(), params.end());
    const Tensor x = whole(x_in);
    Forward f = forward_of(x, as_f32(raw), flip, keep, interval);
    variable_list saved = {x};
    saved.insert(saved.end(), raw.begin(), raw.end());
    if (!full) saved.insert(saved.end(), {f.low, f.dT, f.dL, f.BC, keep ? f.ck : at::empty({1}, x.options().dtype(at::kByte))});
    ctx->save_for_backward(saved);
    ctx->saved_data["flip"] = flip;
    ctx->saved_data["interval"] = interval;
    return f.y;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor& x = saved[0];
    const std::vector<Tensor> raw(saved.begin() + 1, saved.begin() + 1 + kPar);
    const std::vector<Tensor> w = as_f32(raw);
    const bool flip = ctx->saved_data["flip"].toBool(), full = saved.size() == 1 + kPar;
    const int64_t interval = ctx->saved_data["interval"].toInt();
    const Tensor dy = whole(grads[0].to(x.scalar_type()));
    Tensor low, dT, dL, BC, ck;
    const Tensor none = at::empty({0}, x.options());
    const bool graph = at::GradMode::is_enabled();
    if (full) {
      auto pr = graph ? dispatched<decltype(m2dshim::proj_fwd)>("m2dscan::proj_fwd").call(x, w[2], w[3], w[4], w[5], w[6], w[0].size(1), true, true)
                      : m2dshim::proj_fwd(x, w[2], w[3], w[4], w[5], w[6], w[0].size(1), true, true);
      low = pr[0]; dT = pr[1]; dL = pr[2]; BC = pr[3];
      ck = at::empty({1}, x.options().dtype(at::kByte));
    } else {
      low = saved[1 + kPar]; dT = saved[2 + kPar]; dL = saved[3 + kPar]; BC = saved[4 + kPar]; ck = saved[5 + kPar];
    }
    // The gradients of A_log and D come back in fp32, those of the step sizes before the softplus.  The sums over
    // channels d_BT, d_BL, d_C have one reader, the projections' backward: where its products run on the matrix cores it
    // takes the scan's per-workgroup sums as they are.
    const bool parts = x.scalar_type() == at::kBFloat16 && x.size(3) % 8 == 0;
    auto g = graph ? dispatched<decltype(m2dshim::scan_bwd)>("m2dscan::scan_bwd").call(x, dT, dL, w[0], w[1], BC, none, none, w[7], dy, ck, flip,
                                                                                       true, true, true, interval, parts)
                   : m2dshim::scan_bwd(x, dT, dL, w[0], w[1], BC, none, none, w[7], dy, ck, flip, true, true, true, interval, parts);
    // g[0] holds the scan's own gradient of x; the projections add theirs in place
    const int64_t np = parts ? g[5].size(0) : 0;
    auto q = graph ? dispatched<decltype(m2dshim::proj_bwd)>("m2dscan::proj_bwd").call(x, low, dT, dL, w[2], w[3], w[5], g[1], g[2], g[5], g[6],
                                                                                       g[7], g[0], true, true, np)
                   : m2dshim::proj_bwd(x, low, dT, dL, w[2], w[3], w[5], g[1], g[2], g[5], g[6], g[7], g[0], true, true, np);
    variable_list out = {g[0], g[3], g[4], std::get<0>(q), std::get<1>(q), std::get<2>(q), std::get<3>(q), std::get<4>(q), g[8]};
    for (int i = 0; i < kPar; ++i) out[1 + i] = out[1 + i].to(raw[i].scalar_type());
    out.resize(out.size() + 4);      // the options take none
    return out;
  }
};

Tensor entry(const Tensor& x, at::TensorList params, bool full, bool flip, bool save_ckpt, int64_t interval) {
  TORCH_CHECK(params.size() == kPar, "m2dscan: the entry point has ", kPar, " parameters, got ", params.size());
  bool record = x.requires_grad();
  for (const Tensor& t : params) record |= t.requires_grad();
  if (record && at::GradMode::is_enabled()) return Entry::apply(x, params, full, flip, save_ckpt && !full, interval);
  at::NoGradGuard no_grad;
  return forward_of(whole(x), as_f32({params.begin(), params.end()}), flip, false, interval).y;
}

Tensor scan(const Tensor& x, const Tensor& dT, const Tensor& dL, const Tensor& AT, const Tensor& AL, const Tensor& BT, const Tensor& BL,
            const Tensor& C, const Tensor& D, bool flip, int64_t interval) {
  at::NoGradGuard no_grad;
  return std::get<0>(m2dshim::scan_y(whole(x), whole(dT), whole(dL), whole(AT), whole(AL), whole(BT), whole(BL), whole(C), whole(D), false,
                                     flip, false, false, interval));
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(m2dscan, m) {
  m.def("entry(Tensor x, Tensor[] params, bool full, bool flip, bool save_ckpt, int ckpt_interval) -> Tensor");
  m.def("scan(Tensor x, Tensor deltaT, Tensor deltaL, Tensor AT, Tensor AL, Tensor BT, Tensor BL, Tensor C, Tensor D, bool flip, "
        "int ckpt_interval) -> Tensor");
}
TORCH_LIBRARY_IMPL(m2dscan, AutogradCUDA, m) { m.impl("entry", &entry); m.impl("scan", &scan); }
TORCH_LIBRARY_IMPL(m2dscan, CUDA, m) { m.impl("entry", &entry); m.impl("scan", &scan); }
