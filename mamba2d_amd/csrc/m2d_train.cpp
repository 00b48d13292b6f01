// m2d_train.cpp -- a residual block of a scan stage in bf16-mixed training as one autograd function.
//
// The block of models/mamba2d.py:191-254 with the token mixer of :157-188 and the local path and MLP of
// models/utils.py:58-118: x1 = s1 x + mixer(norm1 x), x2 = s2 x1 + MLP(norm2 x1).  Forward and backward are a fixed
// sequence of the library's kernels on one stream (9 + 11 launches beside the scan's and its projections' 2 + 5), issued
// from here: no Python between them, no cast kernels (the fp32 parameters are read as they are), activations rounded to
// bf16 where autocast rounds them.
#include <ATen/autocast_mode.h>
#include <torch/csrc/autograd/autograd.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include <algorithm>

#include "m2d_torch.h"

namespace {

using at::Tensor;
using m2dshim::check;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = c10::optional<Tensor>;

// The block's parameters, in the order of the operator's list.
enum Par { kN1W, kN1B, kInW, kInB, kATLog, kALLog, kXProj, kDtTW, kDtTB, kDtLW, kDtLB, kD, kOutW, kOutB, kRs1, kN2W, kN2B,
           kFc1W, kFc1B, kFc2W, kFc2B, kRs2, kBase,
           kLnW = kBase, kLnB, kPw1, kS1S, kS1B, kDw, kS2S, kS2B, kPw2, kAll };

struct Shape { int64_t B, H, W, C, P, R, N; bool local; };

Shape shape_of(const Tensor& x, at::TensorList p) {
  TORCH_CHECK(x.dim() == 4 && x.is_cuda() && x.is_contiguous() && x.scalar_type() == at::kFloat,
              "m2dscan: x must be a contiguous float32 (B,H,W,C) tensor on the GPU");
  TORCH_CHECK(p.size() == kBase || p.size() == kAll, "m2dscan: a block has ", (int)kBase, " parameters, or ", (int)kAll, " with a local path, got ", p.size());
  Shape s;
  s.B = x.size(0); s.H = x.size(1); s.W = x.size(2); s.C = x.size(3);
  s.P = s.B * s.H * s.W;
  s.local = p.size() == kAll;
  TORCH_CHECK(s.P > 0 && s.H > 1 && s.W > 1, "m2dscan: grid must be larger than one cell, got ", x.sizes());
  TORCH_CHECK(p[kDtTW].dim() == 2 && p[kATLog].dim() == 2, "m2dscan: dt_projT must be (C, dt_rank), AT_log (C, d_state)");
  s.R = p[kDtTW].size(1);
  s.N = p[kATLog].size(1);
  const int64_t C = s.C, M = 2 * C;
  auto want = [&](int i, at::IntArrayRef shape) {
    TORCH_CHECK(p[i].device() == x.device() && p[i].scalar_type() == at::kFloat && p[i].is_contiguous() && p[i].sizes() == shape,
                "m2dscan: parameter ", i, " of the block must be a contiguous float32 ", shape, " tensor on x's device, got ", p[i].sizes());
  };
  want(kN1W, {C}); want(kN1B, {C}); want(kInW, {C, C}); want(kInB, {C}); want(kOutW, {C, C}); want(kOutB, {C}); want(kRs1, {C});
  want(kN2W, {C}); want(kN2B, {C}); want(kFc1W, {4 * C, C}); want(kFc1B, {4 * C}); want(kFc2W, {C, 4 * C}); want(kFc2B, {C}); want(kRs2, {C});
  if (s.local) {
    want(kLnW, {C}); want(kLnB, {C}); want(kPw1, {M, C}); want(kDw, {M, 1, 3, 3}); want(kPw2, {C, M});
    for (int i : {(int)kS1S, (int)kS1B, (int)kS2S, (int)kS2B}) want(i, {1});
  }
  return s;
}

const float* f32(const Tensor& t) { return t.data_ptr<float>(); }
const float* opt(const OptTensor& t) { return t.has_value() && t->defined() ? t->data_ptr<float>() : nullptr; }

Tensor bf16_like(const Tensor& x, int64_t C) {
  return at::empty({x.size(0), x.size(1), x.size(2), C}, x.options().dtype(at::kBFloat16));
}

// bf16 autocast while it lives.
struct Autocast {
  const bool was = at::autocast::is_autocast_enabled(at::kCUDA);
  const at::ScalarType dtype = at::autocast::get_autocast_dtype(at::kCUDA);
  Autocast() {
    at::autocast::increment_nesting();
    at::autocast::set_autocast_enabled(at::kCUDA, true);
    at::autocast::set_autocast_dtype(at::kCUDA, at::kBFloat16);
  }
  ~Autocast() {
    if (at::autocast::decrement_nesting() == 0) at::autocast::clear_cache();
    at::autocast::set_autocast_enabled(at::kCUDA, was);
    at::autocast::set_autocast_dtype(at::kCUDA, dtype);
  }
};

// The block in stock operators and the entry point's, as its modules compute it under autocast: what its gradients are
// taken from where they are to be differentiated themselves.
Tensor stock_block(const Tensor& x, const std::vector<Tensor>& p, const Tensor& keep1, const Tensor& keep2, const std::vector<double>& eps,
                   bool flip, bool full, int64_t interval) {
  const Autocast on;
  const int64_t C = x.size(3);
  auto star = [](const Tensor& v, const Tensor& s, const Tensor& b) { return at::addcmul(b, s, at::relu(v).square()); };
  auto kept = [](const Tensor& v, const Tensor& keep) { return keep.defined() ? v * keep.view({-1, 1, 1, 1}) : v; };
  const Tensor n1 = at::layer_norm(x, {C}, p[kN1W], p[kN1B], eps[0]);
  Tensor local;
  if (p.size() == kAll) {
    const Tensor a = star(at::linear(at::layer_norm(n1, {C}, p[kLnW], p[kLnB], eps[2]), p[kPw1]), p[kS1S], p[kS1B]);
    const Tensor c = at::conv2d(a.permute({0, 3, 1, 2}), p[kDw], {}, 1, 1, 1, 2 * C).permute({0, 2, 3, 1});
    local = at::linear(star(c, p[kS2S], p[kS2B]), p[kPw2]);
  }
  using Entry = Tensor(const Tensor&, at::TensorList, bool, bool, bool, int64_t);
  const std::vector<Tensor> scan(p.begin() + kATLog, p.begin() + kD + 1);
  const Tensor y = m2dshim::dispatched<Entry>("m2dscan::entry").call(at::gelu(at::linear(n1, p[kInW], p[kInB])), scan, full, flip, !full, interval);
  Tensor mix = at::linear(at::gelu(y), p[kOutW], p[kOutB]);
  if (local.defined()) mix = mix + local;
  const Tensor x1 = x * p[kRs1] + kept(mix, keep1);
  const Tensor h = at::linear(at::layer_norm(x1, {C}, p[kN2W], p[kN2B], eps[1]), p[kFc1W], p[kFc1B]);
  return x1 * p[kRs2] + kept(at::linear(at::gelu(h), p[kFc2W], p[kFc2B]), keep2);
}

struct Block : public torch::autograd::Function<Block> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, at::TensorList par, const OptTensor& keep1, const OptTensor& keep2,
                        double eps1, double eps2, double eps_local, bool flip, bool full, bool save_ckpt, int64_t interval) {
    const std::vector<Tensor> p = par.vec();
    const Shape s = shape_of(x, p);
    c10::DeviceGuard guard(x.device());
    hipStream_t st = m2dshim::current_stream(x);
    const int C = (int)s.C, M = 2 * C, HD = 4 * C, rps = (int)(s.H * s.W);
    const Tensor none;
    Tensor n1 = bf16_like(x, C), nl = s.local ? bf16_like(x, C) : none;
    check(m2d_train_norm_fwd(s.P, C, rps, f32(x), nullptr, nullptr, nullptr, nullptr, nullptr, f32(p[kN1W]), f32(p[kN1B]), (float)eps1,
                             n1.data_ptr(), s.local ? f32(p[kLnW]) : nullptr, s.local ? f32(p[kLnB]) : nullptr, (float)eps_local,
                             s.local ? nl.data_ptr() : nullptr, st));
    Tensor pre, conv, loc;
    if (s.local) {
      pre = bf16_like(x, M); conv = bf16_like(x, M); loc = bf16_like(x, C);
      check(m2d_linear_fwd(s.P, C, M, M2D_F32, nl.data_ptr(), f32(p[kPw1]), nullptr, M2D_ACT_NONE, nullptr, nullptr, M2D_ACT_NONE, nullptr,
                           nullptr, pre.data_ptr(), st));
      check(m2d_starrelu_dwconv3x3_fwd((int)s.B, (int)s.H, (int)s.W, M, M2D_F32, pre.data_ptr(), f32(p[kS1S]), f32(p[kS1B]), f32(p[kDw]),
                                       conv.data_ptr(), st));
      check(m2d_linear_fwd(s.P, M, C, M2D_F32, conv.data_ptr(), f32(p[kPw2]), nullptr, M2D_ACT_STARRELU, f32(p[kS2S]), f32(p[kS2B]),
                           M2D_ACT_NONE, nullptr, nullptr, loc.data_ptr(), st));
    }
    Tensor u0 = bf16_like(x, C), u = bf16_like(x, C);
    check(m2d_linear_keep_fwd(s.P, C, C, M2D_F32, n1.data_ptr(), f32(p[kInW]), f32(p[kInB]), M2D_ACT_GELU, nullptr, nullptr, u0.data_ptr(),
                              u.data_ptr(), st));
    auto pr = m2dshim::proj_fwd(u, p[kXProj], p[kDtTW], p[kDtTB], p[kDtLW], p[kDtLB], s.N, true, true);
    auto [y, ck] = m2dshim::scan_fwd(u, pr[1], pr[2], p[kATLog], p[kALLog], pr[3], pr[4], pr[5], p[kD], save_ckpt && !full, flip, true, true,
                                     interval);
    Tensor mix = bf16_like(x, C);
    check(m2d_linear_fwd(s.P, C, C, M2D_F32, y.data_ptr(), f32(p[kOutW]), f32(p[kOutB]), M2D_ACT_GELU, nullptr, nullptr, M2D_ACT_NONE, nullptr,
                         nullptr, mix.data_ptr(), st));
    Tensor x1 = at::empty_like(x), n2 = bf16_like(x, C);
    check(m2d_train_norm_fwd(s.P, C, rps, f32(x), f32(p[kRs1]), mix.data_ptr(), s.local ? loc.data_ptr() : nullptr, opt(keep1),
                             x1.data_ptr<float>(), f32(p[kN2W]), f32(p[kN2B]), (float)eps2, n2.data_ptr(), nullptr, nullptr, 0.f, nullptr, st));
    Tensor h0 = bf16_like(x, HD), m = mix;      // (the mixer's answer has been added: its buffer takes the MLP's)
    if (C == 32 || C == 64) {      // both layers in one kernel
      check(m2d_mlp_keep_fwd(s.P, C, HD, M2D_F32, n2.data_ptr(), f32(p[kFc1W]), f32(p[kFc1B]), f32(p[kFc2W]), f32(p[kFc2B]), h0.data_ptr(),
                             m.data_ptr(), st));
    } else {
      check(m2d_linear_fwd(s.P, C, HD, M2D_F32, n2.data_ptr(), f32(p[kFc1W]), f32(p[kFc1B]), M2D_ACT_NONE, nullptr, nullptr, M2D_ACT_NONE,
                           nullptr, nullptr, h0.data_ptr(), st));
      check(m2d_linear_fwd(s.P, HD, C, M2D_F32, h0.data_ptr(), f32(p[kFc2W]), f32(p[kFc2B]), M2D_ACT_GELU, nullptr, nullptr, M2D_ACT_NONE,
                           nullptr, nullptr, m.data_ptr(), st));
    }
    Tensor x2 = at::empty_like(x);
    check(m2d_train_norm_fwd(s.P, C, rps, f32(x1), f32(p[kRs2]), m.data_ptr(), nullptr, opt(keep2), x2.data_ptr<float>(), nullptr, nullptr, 0.f,
                             nullptr, nullptr, nullptr, 0.f, nullptr, st));
    variable_list saved = {x, n1, u0, u, y, x1, n2, h0, keep1.value_or(none), keep2.value_or(none), nl, pre, conv,
                           full ? none : pr[0], full ? none : pr[1], full ? none : pr[2], full ? none : pr[3], full ? none : ck};
    saved.insert(saved.end(), p.begin(), p.end());
    ctx->save_for_backward(saved);
    ctx->saved_data["eps"] = std::vector<double>{eps1, eps2, eps_local};
    ctx->saved_data["flip"] = flip;
    ctx->saved_data["full"] = full;
    ctx->saved_data["interval"] = interval;
    return x2;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &n1 = saved[1], &u0 = saved[2], &u = saved[3], &y = saved[4], &x1 = saved[5], &n2 = saved[6], &h0 = saved[7],
                 &keep1 = saved[8], &keep2 = saved[9], &nl = saved[10], &pre = saved[11], &conv = saved[12];
    const std::vector<Tensor> p(saved.begin() + 18, saved.end());
    const Shape s = shape_of(x, p);
    c10::DeviceGuard guard(x.device());
    hipStream_t st = m2dshim::current_stream(x);
    const int C = (int)s.C, M = 2 * C, HD = 4 * C, rps = (int)(s.H * s.W);
    const auto eps = ctx->saved_data["eps"].toDoubleVector();
    const bool flip = ctx->saved_data["flip"].toBool(), full = ctx->saved_data["full"].toBool();
    const int64_t interval = ctx->saved_data["interval"].toInt();
    Tensor dy = grads[0];
    TORCH_CHECK(dy.scalar_type() == at::kFloat, "m2dscan: the gradient of a block's output must be float32, got ", dy.scalar_type());
    dy = dy.contiguous();
    if (reinterpret_cast<uintptr_t>(dy.data_ptr()) % 16) dy = dy.clone();
    if (at::GradMode::is_enabled()) return recorded(x, p, dy, keep1, keep2, eps, flip, full, interval);

    // one workspace for the workgroups' sums of all parameter gradients
    std::vector<m2d_reduce_seg> segs;
    std::vector<Tensor> out(p.size());
    int64_t at = 0;
    auto take = [&](int64_t n) { const int64_t o = at; at += (n + 63) / 64 * 64; return o; };
    const int np = m2d_train_norm_parts(s.P, C);
    const int64_t o_n2 = take((int64_t)np * 5 * C), o_n1 = take((int64_t)np * 5 * C);
    struct W { int w, b, N, K, parts; int64_t off; bool both; };      // both: input's and weight's gradient from one kernel
    std::vector<W> ws = {{kFc2W, kFc2B, C, HD, 0, 0, false}, {kFc1W, kFc1B, HD, C, 0, 0, false}, {kOutW, kOutB, C, C, 0, 0, false}, {kInW, kInB, C, C, 0, 0, false}};
    if (s.local) { ws.push_back({kPw2, -1, C, M, 0, 0, false}); ws.push_back({kPw1, -1, M, C, 0, 0, false}); }
    for (auto& w : ws) {
      w.both = m2d_train_linear_grads_parts(s.P, w.N, w.K) > 0;
      w.parts = w.both ? m2d_train_linear_grads_parts(s.P, w.N, w.K) : m2d_train_wgrad_parts(s.P, w.N, w.K);
      w.off = take((int64_t)w.parts * ((int64_t)w.N * w.K + w.N));
    }
    const int lp = !s.local ? 0 : ws[4].both ? ws[4].parts : m2d_train_linear_parts(s.P, M, C), dp = s.local ? m2d_train_dwconv_parts((int)s.B, (int)s.H, (int)s.W, M) : 0;
    TORCH_CHECK(!s.local || (lp > 0 && dp > 0), "m2dscan: block shapes outside what the training kernels are built for");
    const int64_t o_s2 = take((int64_t)lp * 2), o_dw = take((int64_t)dp * (9 * M + 2));
    Tensor part_t = at::empty({at}, x.options());
    float* part = part_t.data_ptr<float>();
    auto seg = [&](int i, int64_t off, int64_t stride, int parts) {
      out[i] = at::empty_like(p[i]);
      segs.push_back({part + off, out[i].data_ptr<float>(), stride, (int32_t)p[i].numel(), parts});
    };
    // layer i: the gradient dx of its input `in` and the sums for its weight and bias, from the gradient g of its output (before a GELU behind it, with z)
    auto layer = [&](int i, const Tensor& g, const Tensor* z, const Tensor& in, int act, const float* as, const float* ab, Tensor& dx, float* sums) {
      const W& w = ws[i];
      const int post = z ? M2D_ACT_GELU : M2D_ACT_NONE;
      const void* zp = z ? z->data_ptr() : nullptr;
      if (w.both) {
        check(m2d_train_linear_grads(s.P, w.N, w.K, g.data_ptr(), zp, post, f32(p[w.w]), in.data_ptr(), act, as, ab, w.b >= 0, dx.data_ptr(),
                                     part + w.off, sums, st));
      } else {
        check(m2d_train_linear_bwd(s.P, w.K, w.N, g.data_ptr(), zp, post, f32(p[w.w]), act != M2D_ACT_NONE ? in.data_ptr() : nullptr, act, as,
                                   dx.data_ptr(), sums, st));
        check(m2d_train_wgrad(s.P, w.N, w.K, g.data_ptr(), zp, post, in.data_ptr(), act, as, ab, w.b >= 0, part + w.off, st));
      }
      const int64_t stride = (int64_t)w.N * w.K + w.N;
      seg(w.w, w.off, stride, w.parts);
      if (w.b >= 0) seg(w.b, w.off + (int64_t)w.N * w.K, stride, w.parts);
    };

    // MLP
    Tensor dm = bf16_like(x, C), dh = bf16_like(x, HD), dn = bf16_like(x, C);
    check(m2d_train_branch(s.P * C, (int64_t)rps * C, f32(dy), keep2.defined() ? f32(keep2) : nullptr, dm.data_ptr(), st));
    layer(0, dm, nullptr, h0, M2D_ACT_GELU, nullptr, nullptr, dh, nullptr);
    layer(1, dh, nullptr, n2, M2D_ACT_NONE, nullptr, nullptr, dn, nullptr);
    // second update and norm2; dm takes the gradient of the mixer's answer
    Tensor dx1 = at::empty_like(x);
    check(m2d_train_norm_bwd(s.P, C, rps, f32(x1), dn.data_ptr(), nullptr, f32(dy), f32(p[kRs2]), keep1.defined() ? f32(keep1) : nullptr,
                             f32(p[kN2W]), f32(p[kN2B]), (float)eps[1], nullptr, 0.f, dx1.data_ptr<float>(), dm.data_ptr(), part + o_n2, st));
    seg(kN2W, o_n2, 5 * C, np); seg(kN2B, o_n2 + C, 5 * C, np); seg(kRs2, o_n2 + 4 * C, 5 * C, np);
    // local path
    Tensor dl;
    if (s.local) {
      Tensor dc = bf16_like(x, M), dpre = bf16_like(x, M);
      dl = bf16_like(x, C);
      layer(4, dm, nullptr, conv, M2D_ACT_STARRELU, f32(p[kS2S]), f32(p[kS2B]), dc, part + o_s2);
      seg(kS2S, o_s2, 2, lp); seg(kS2B, o_s2 + 1, 2, lp);
      check(m2d_train_dwconv_bwd((int)s.B, (int)s.H, (int)s.W, M, pre.data_ptr(), dc.data_ptr(), f32(p[kDw]), f32(p[kS1S]), f32(p[kS1B]),
                                 dpre.data_ptr(), part + o_dw, st));
      seg(kDw, o_dw, 9 * M + 2, dp); seg(kS1S, o_dw + 9 * M, 9 * M + 2, dp); seg(kS1B, o_dw + 9 * M + 1, 9 * M + 2, dp);
      layer(5, dpre, nullptr, nl, M2D_ACT_NONE, nullptr, nullptr, dl, nullptr);
    }
    // scan path
    Tensor dyy = dn;
    layer(2, dm, nullptr, y, M2D_ACT_GELU, nullptr, nullptr, dyy, nullptr);
    Tensor low, dT, dL, BC, ck;
    const Tensor no_bc = at::empty({0}, u.options());
    if (full) {
      auto pr = m2dshim::proj_fwd(u, p[kXProj], p[kDtTW], p[kDtTB], p[kDtLW], p[kDtLB], s.N, true, true);
      low = pr[0]; dT = pr[1]; dL = pr[2]; BC = pr[3];
      ck = at::empty({1}, u.options().dtype(at::kByte));
    } else {
      low = saved[13]; dT = saved[14]; dL = saved[15]; BC = saved[16]; ck = saved[17];
    }
    auto g = m2dshim::scan_bwd(u, dT, dL, p[kATLog], p[kALLog], BC, no_bc, no_bc, p[kD], dyy, ck, flip, true, true, true, interval, true);
    Tensor du = g[0];
    out[kATLog] = g[3]; out[kALLog] = g[4]; out[kD] = g[8];
    std::tie(out[kXProj], out[kDtTW], out[kDtTB], out[kDtLW], out[kDtLB]) =
        m2dshim::proj_bwd(u, low, dT, dL, p[kXProj], p[kDtTW], p[kDtLW], g[1], g[2], g[5], g[6], g[7], du, true, true, g[5].size(0));
    layer(3, du, &u0, n1, M2D_ACT_NONE, nullptr, nullptr, dn, nullptr);
    // first update, norm1 and the local path's norm
    Tensor dx = at::empty_like(x);
    check(m2d_train_norm_bwd(s.P, C, rps, f32(x), dn.data_ptr(), s.local ? dl.data_ptr() : nullptr, f32(dx1), f32(p[kRs1]), nullptr, f32(p[kN1W]),
                             f32(p[kN1B]), (float)eps[0], s.local ? f32(p[kLnW]) : nullptr, (float)eps[2], dx.data_ptr<float>(), nullptr,
                             part + o_n1, st));
    seg(kN1W, o_n1, 5 * C, np); seg(kN1B, o_n1 + C, 5 * C, np); seg(kRs1, o_n1 + 4 * C, 5 * C, np);
    if (s.local) { seg(kLnW, o_n1 + 2 * C, 5 * C, np); seg(kLnB, o_n1 + 3 * C, 5 * C, np); }
    check(m2d_train_reduce((int)segs.size(), segs.data(), st));

    return of_all(dx, out);
  }

  static variable_list of_all(const Tensor& dx, const std::vector<Tensor>& par) {
    variable_list all = {dx};
    all.insert(all.end(), par.begin(), par.end());
    all.resize(all.size() + 9);      // keep1, keep2 and the seven options take none
    return all;
  }

  // The gradients with a graph behind them (create_graph).  Every input goes in as a view of its own, so that a gradient
  // stops there also where one input was computed from another.
  static variable_list recorded(const Tensor& x, const std::vector<Tensor>& p, const Tensor& dy, const Tensor& keep1, const Tensor& keep2,
                                const std::vector<double>& eps, bool flip, bool full, int64_t interval) {
    std::vector<Tensor> in = {x.view_as(x)};
    for (const Tensor& t : p) in.push_back(t.view_as(t));
    const Tensor y = stock_block(in[0], {in.begin() + 1, in.end()}, keep1, keep2, eps, flip, full, interval);
    variable_list asked;
    for (const Tensor& t : in)
      if (t.requires_grad()) asked.push_back(t);
    const variable_list g = torch::autograd::grad({y}, asked, {dy}, true, true, true);
    std::vector<Tensor> out;
    size_t at = 0;
    for (const Tensor& t : in) out.push_back(t.requires_grad() ? g[at++] : Tensor());
    return of_all(out[0], {out.begin() + 1, out.end()});
  }
};

Tensor train_block(const Tensor& x, at::TensorList par, const OptTensor& keep1, const OptTensor& keep2, double eps1, double eps2,
                   double eps_local, bool flip, bool full, bool save_ckpt, int64_t interval) {
  return Block::apply(x, par, keep1, keep2, eps1, eps2, eps_local, flip, full, save_ckpt, interval);
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(m2dscan, m) {
  m.def("train_block(Tensor x, Tensor[] params, Tensor? keep1, Tensor? keep2, float eps1, float eps2, float eps_local, bool flip, "
        "bool full, bool save_ckpt, int ckpt_interval) -> Tensor");
}
TORCH_LIBRARY_IMPL(m2dscan, AutogradCUDA, m) { m.impl("train_block", &train_block); }
TORCH_LIBRARY_IMPL(m2dscan, CUDA, m) { m.impl("train_block", &train_block); }
