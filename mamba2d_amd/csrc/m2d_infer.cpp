// m2d_infer.cpp -- the blocks of a backbone stage at inference, issued from one call.
//
// A stage is a row of residual blocks (models/mamba2d.py:191-254) and the LayerNorm behind them: 8 to 11 launches a scan block (8 of a batch), 7 an
// attention block.  Issued module by module from Python they take the host 190 us a block, four times what the kernels of one
// image take; here they cost a few microseconds each.  They are the kernels that the modules run, in their order, but for the residual updates, which narrow
// blocks have inside the layers in front of them.  The matrix products of the wide
// layers stay with the stock library (at::linear, which also follows autocast), as in the modules.
#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <torch/library.h>

#include "m2d_torch.h"

namespace {

using at::Tensor;
using m2dshim::check;

// Parameters of a block, in order.  A scan block without local path ends at kBase.
enum Scan { kN1W, kN1B, kInW, kInB, kATLog, kALLog, kXProj, kDtTW, kDtTB, kDtLW, kDtLB, kD, kOutW, kOutB, kRs1, kN2W, kN2B,
            kFc1W, kFc1B, kFc2W, kFc2B, kRs2, kBase, kLnW = kBase, kLnB, kPw1, kS1S, kS1B, kDw, kS2S, kS2B, kPw2, kAll };
enum Attn { aN1W, aN1B, aQkv, aQnW, aQnB, aKnW, aKnB, aProj, aRs1, aN2W, aN2B, aFc1W, aFc1B, aFc2W, aFc2B, aRs2, aAll };
enum Kind { kScan = 0, kScanFlipped = 1, kScanLocal = 2, kScanLocalFlipped = 3, kAttention = 4 };

// Up to this many rows a wide layer runs in the library's kernel without staging (host 3 us against 19, device about the
// same up to 400 rows); beyond it the stock product's tiles win (320 -> 1280 at 784 rows: 9.6 us against 5.4), unless a
// GELU follows: that layer's own kernel writes its outputs once, where the stock product and activation write them twice.
constexpr int64_t kFewPositions = 512;
constexpr int64_t kMostPositions = 1 << 20;      // what m2d_wide_linear_fwd takes

// From this many rows the MLP of 128 channels is one kernel.  A tile of 128 rows takes it 24 us and up to 512 tiles run at once, so it takes that
// long for one tile as for 65536 rows, while the three kernels' time grows with the rows from 21 us on.  Two such blocks with everything else, three kernels and
// one, us, bf16 and fp32 weights: 2352 rows 189.7 and 201.3, 183.1 and 201.3; 6272 211.9 and 217.4, 205.5 and 211.9; 9216 266.3 and 273.2; 12544 252.1 and
// 252.4, 240.7 and 244.4; 14112 278.2 and 272.1, 269.7 and 269.1; 16384 331.7 and 320.8; 25088 342.4 and 310.2, 335.3 and 306.1; 50176 460.4 and
// 416.6.  (Of 27 sizes from 14112 rows on none is slower in one kernel, of 34 below 26 are.)
constexpr int64_t kWideMlpFrom = 14000;

struct Run {
  int64_t B, H, W, C, P;
  int wd;                 // element type of the weights
  hipStream_t st;
  at::TensorOptions opt;

  Tensor make(int64_t c) const { return at::empty({B, H, W, c}, opt); }

  Tensor norm(const Tensor& x, const Tensor& w, const Tensor& b, double eps) const {
    Tensor y = make(C);
    check(m2d_layernorm_fwd(P, (int)C, M2D_BF16, wd, x.data_ptr(), w.data_ptr(), b.data_ptr(), (float)eps, y.data_ptr(), st));
    return y;
  }
  // post(pre(x) w^T + b): the library's kernel where the layer is narrow (backbone.linear_act), the stock product otherwise
  Tensor linear(const Tensor& x, const Tensor& w, const Tensor* b, int pre, const Tensor* ps, const Tensor* pb, int post, const Tensor* qs,
                const Tensor* qb) const {
    const int64_t N = w.size(0), K = w.size(1);
    auto ptr = [](const Tensor* t) -> const void* { return t && t->defined() ? t->data_ptr() : nullptr; };
    if (K % 32 == 0 && K <= 256 && N % 16 == 0 && N <= 512) {
      Tensor y = make(N);
      check(m2d_linear_fwd(P, (int)K, (int)N, wd, x.data_ptr(), w.data_ptr(), ptr(b), pre, ptr(ps), ptr(pb), post, ptr(qs), ptr(qb),
                           y.data_ptr(), st));
      return y;
    }
    TORCH_CHECK(pre != M2D_ACT_STARRELU && post != M2D_ACT_STARRELU, "m2dscan: StarReLU next to a wide layer");
    // (fp32 weights meet bf16 activations under autocast only: without it the stock product below refuses them)
    const bool few = P <= kFewPositions && (wd == M2D_BF16 || at::autocast::is_autocast_enabled(at::kCUDA));
    const bool gelu = post == M2D_ACT_GELU && wd == M2D_BF16 && K <= 320 && N % 64 == 0 && P <= kMostPositions;
    if (pre == M2D_ACT_NONE && (few || gelu) && K % 32 == 0 && N % 32 == 0) {
      Tensor y = make(N);
      check(m2d_wide_linear_fwd(P, (int)K, (int)N, wd, x.data_ptr(), w.data_ptr(), ptr(b), post, y.data_ptr(), st));
      return y;
    }
    Tensor y = at::linear(pre == M2D_ACT_GELU ? at::gelu(x) : x, w, b && b->defined() ? c10::optional<Tensor>(*b) : c10::nullopt);
    return post == M2D_ACT_GELU ? at::gelu(y) : y;
  }
  // x s + (GELU(y) w^T + b + r2)
  Tensor linear_residual(const Tensor& y, const Tensor& w, const Tensor& b, const Tensor& x, const Tensor& s, const Tensor& r2) const {
    Tensor o = make(C);
    check(m2d_linear_residual_fwd(P, (int)C, (int)C, wd, y.data_ptr(), w.data_ptr(), b.data_ptr(), M2D_ACT_GELU, x.data_ptr(), s.data_ptr(),
                                  r2.defined() ? r2.data_ptr() : nullptr, o.data_ptr(), st));
    return o;
  }
  Tensor residual(const Tensor& x, const Tensor& s, const Tensor& r, const Tensor& r2) const {
    Tensor y = make(C);
    check(m2d_scale_residual_fwd(P, (int)C, M2D_BF16, wd, x.data_ptr(), s.data_ptr(), r.data_ptr(), r2.defined() ? r2.data_ptr() : nullptr,
                                 y.data_ptr(), st));
    return y;
  }
  Tensor residual_norm(const Tensor& x, const Tensor& s, const Tensor& r, const Tensor& r2, const Tensor& w, const Tensor& b, double eps,
                       Tensor& normed) const {
    Tensor xo = make(C);
    normed = make(C);
    check(m2d_scale_residual_layernorm_fwd(P, (int)C, M2D_BF16, wd, x.data_ptr(), s.data_ptr(), r.data_ptr(),
                                           r2.defined() ? r2.data_ptr() : nullptr, w.data_ptr(), b.data_ptr(), (float)eps, xo.data_ptr(),
                                           normed.data_ptr(), st));
    return xo;
  }
};

Tensor infer_stage(const Tensor& x_in, at::TensorList par, at::IntArrayRef kinds, at::ArrayRef<double> eps, const Tensor& cos,
                   const Tensor& sin, double att_scale) {
  TORCH_CHECK(x_in.is_cuda() && x_in.dim() == 4 && x_in.is_contiguous() && x_in.scalar_type() == at::kBFloat16 && x_in.numel() > 0,
              "m2dscan: x must be a contiguous bfloat16 (B,H,W,C) tensor on the GPU");
  int64_t want = 2;
  for (int64_t k : kinds) {
    TORCH_CHECK(k >= kScan && k <= kAttention, "m2dscan: unknown kind of block ", k);
    want += k == kAttention ? aAll : k >= kScanLocal ? kAll : kBase;
  }
  TORCH_CHECK((int64_t)par.size() == want && eps.size() == 3 * kinds.size() + 1, "m2dscan: the stage's blocks have ", want, " parameters and ",
              3 * kinds.size() + 1, " eps, got ", par.size(), " and ", eps.size());
  const auto wt = par[0].scalar_type();
  // parameters that this sequence does not take are no error: an empty answer sends the caller back to its modules
  if (wt != at::kFloat && wt != at::kBFloat16) return at::empty({0}, x_in.options());
  for (const Tensor& t : par)
    if (!t.defined() || t.device() != x_in.device() || !t.is_contiguous() || t.scalar_type() != wt || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16)
      return at::empty({0}, x_in.options());
  c10::DeviceGuard guard(x_in.device());
  Run r{x_in.size(0), x_in.size(1), x_in.size(2), x_in.size(3), 0, wt == at::kFloat ? M2D_F32 : M2D_BF16, m2dshim::current_stream(x_in), x_in.options()};
  r.P = r.B * r.H * r.W;
  const int64_t C = r.C;
  auto shaped = [&](const Tensor& t, at::IntArrayRef s) { TORCH_CHECK(t.sizes() == s, "m2dscan: a parameter of the stage has shape ", t.sizes(), ", expected ", s); };

  // the scan and its projections take fp32 parameters: bf16 ones are widened in one launch for all blocks
  std::vector<Tensor> wide;
  {
    std::vector<Tensor> narrow;
    int64_t at = 0;
    for (int64_t k : kinds) {
      if (k != kAttention)
        for (int i = kATLog; i <= kD; ++i) narrow.push_back(par[at + i]);
      at += k == kAttention ? aAll : k >= kScanLocal ? kAll : kBase;
    }
    if (!narrow.empty()) wide = m2dshim::widen(narrow);
  }

  Tensor x = x_in, normed, none;
  int64_t at = 0;
  size_t wat = 0;
  for (size_t blk = 0; blk < kinds.size(); ++blk) {
    const Tensor* p = &par[at];
    const int kind = (int)kinds[blk];
    const bool att = kind == kAttention;
    at += att ? aAll : kind >= kScanLocal ? kAll : kBase;
    const bool last = blk + 1 == kinds.size();
    const Tensor &next_w = par[at], &next_b = par[at + 1];      // norm1 of the next block, or the stage's norm
    const double next_eps = last ? eps[3 * kinds.size()] : eps[3 * (blk + 1)];
    shaped(p[kN1W], {C}); shaped(p[kN1B], {C});
    const Tensor n1 = normed.defined() ? normed : r.norm(x, p[kN1W], p[kN1B], eps[3 * blk]);
    const int64_t HD = p[att ? (int)aFc1W : (int)kFc1W].size(0);
    const bool narrow = C % 32 == 0 && C <= 128 && HD % 16 == 0 && HD <= 512;
    Tensor term, term2;
    const Tensor *rs1, *n2w, *n2b, *f1w, *f1b, *f2w, *f2b, *rs2;
    if (att) {
      const int64_t hd = p[aQnW].size(0), nh = p[aQkv].size(0) / 3 / hd, L = r.H * r.W;
      shaped(p[aQkv], {3 * nh * hd, C}); shaped(p[aProj], {C, nh * hd}); shaped(cos, {L, hd}); shaped(sin, {L, hd});
      for (int i : {(int)aQnW, (int)aQnB, (int)aKnW, (int)aKnB}) shaped(p[i], {hd});
      TORCH_CHECK(cos.is_contiguous() && sin.is_contiguous() && cos.scalar_type() == at::kBFloat16 && sin.scalar_type() == at::kBFloat16,
                  "m2dscan: cos and sin must be contiguous bfloat16 tensors");
      const Tensor qkv = r.linear(n1, p[aQkv], nullptr, M2D_ACT_NONE, nullptr, nullptr, M2D_ACT_NONE, nullptr, nullptr);
      Tensor o = at::empty({r.B, r.H, r.W, nh * hd}, r.opt);
      check(m2d_rope_attention_fwd((int)r.B, (int)L, (int)nh, (int)hd, r.wd, qkv.data_ptr(), cos.data_ptr(), sin.data_ptr(), p[aQnW].data_ptr(),
                                   p[aQnB].data_ptr(), p[aKnW].data_ptr(), p[aKnB].data_ptr(), (float)eps[3 * blk + 2], (float)att_scale,
                                   o.data_ptr(), r.st));
      term = r.linear(o, p[aProj], nullptr, M2D_ACT_NONE, nullptr, nullptr, M2D_ACT_NONE, nullptr, nullptr);
      rs1 = p + aRs1; n2w = p + aN2W; n2b = p + aN2B; f1w = p + aFc1W; f1b = p + aFc1B; f2w = p + aFc2W; f2b = p + aFc2B; rs2 = p + aRs2;
    } else {
      const bool local = kind >= kScanLocal, flip = kind & 1;
      shaped(p[kInW], {C, C}); shaped(p[kInB], {C}); shaped(p[kOutW], {C, C}); shaped(p[kOutB], {C});
      if (local) {
        const int64_t M = p[kPw1].size(0);
        shaped(p[kLnW], {C}); shaped(p[kLnB], {C});
        for (int i : {(int)kS1S, (int)kS1B, (int)kS2S, (int)kS2B}) TORCH_CHECK(p[i].numel() == 1, "m2dscan: a StarReLU's scale or bias is no single value");
        shaped(p[kPw1], {M, C}); shaped(p[kDw], {M, 1, 3, 3}); shaped(p[kPw2], {C, M});
        Tensor a;
        if (C % 32 == 0 && C <= 128 && M % 16 == 0 && M <= 512) {
          a = r.make(M);
          check(m2d_layernorm_linear_fwd(r.P, (int)C, (int)M, r.wd, n1.data_ptr(), p[kLnW].data_ptr(), p[kLnB].data_ptr(), (float)eps[3 * blk + 2],
                                         p[kPw1].data_ptr(), nullptr, M2D_ACT_STARRELU, p[kS1S].data_ptr(), p[kS1B].data_ptr(), a.data_ptr(), r.st));
        } else {
          a = r.linear(r.norm(n1, p[kLnW], p[kLnB], eps[3 * blk + 2]), p[kPw1], nullptr, M2D_ACT_NONE, nullptr, nullptr, M2D_ACT_STARRELU, p + kS1S,
                       p + kS1B);
        }
        Tensor d = r.make(M);
        check(m2d_dwconv3x3_fwd((int)r.B, (int)r.H, (int)r.W, (int)M, M2D_BF16, r.wd, a.data_ptr(), p[kDw].data_ptr(), d.data_ptr(), r.st));
        term2 = r.linear(d, p[kPw2], nullptr, M2D_ACT_STARRELU, p + kS2S, p + kS2B, M2D_ACT_NONE, nullptr, nullptr);
      }
      const Tensor u = r.linear(n1, p[kInW], p + kInB, M2D_ACT_NONE, nullptr, nullptr, M2D_ACT_GELU, nullptr, nullptr);
      const Tensor* w = &wide[wat];
      wat += kD - kATLog + 1;
      auto at_w = [&](int i) -> const Tensor& { return w[i - kATLog]; };
      const int64_t N = at_w(kATLog).size(1);
      const auto pr = m2dshim::proj_fwd(u, at_w(kXProj), at_w(kDtTW), at_w(kDtTB), at_w(kDtLW), at_w(kDtLB), N, true, true);
      const Tensor y = std::get<0>(m2dshim::scan_fwd(u, pr[1], pr[2], at_w(kATLog), at_w(kALLog), pr[3], pr[4], pr[5], at_w(kD), false, flip, true, true, 0));
      if (narrow) {      // the residual update is part of the output projection (other blocks have it with the norm behind it)
        shaped(p[kRs1], {C});
        x = r.linear_residual(y, p[kOutW], p[kOutB], x, p[kRs1], term2);
      } else {
        term = r.linear(y, p[kOutW], p + kOutB, M2D_ACT_GELU, nullptr, nullptr, M2D_ACT_NONE, nullptr, nullptr);
      }
      rs1 = p + kRs1; n2w = p + kN2W; n2b = p + kN2B; f1w = p + kFc1W; f1b = p + kFc1B; f2w = p + kFc2W; f2b = p + kFc2B; rs2 = p + kRs2;
    }
    shaped(*f1w, {HD, C}); shaped(*f2w, {C, HD}); shaped(*f1b, {HD}); shaped(*f2b, {C});
    for (const Tensor* t : {rs1, n2w, n2b, rs2, &next_w, &next_b}) shaped(*t, {C});
    Tensor branch;
    if (narrow) {      // norm2 inside the MLP's first kernel
      if (term.defined()) x = r.residual(x, *rs1, term, term2);
      // ... and the residual update and the next norm behind it too.  (At 128 channels the second layer is otherwise the stock product, which
      // refuses fp32 weights without autocast: such a call is refused at every size.)
      const bool wide = C == 128 && r.P >= kWideMlpFrom && (r.wd == M2D_BF16 || at::autocast::is_autocast_enabled(at::kCUDA));
      if ((C == 32 || C == 64 || wide) && HD == 4 * C) {
        Tensor xo = r.make(C);
        normed = r.make(C);
        check(m2d_mlp_residual_layernorm_fwd(r.P, (int)C, (int)HD, r.wd, x.data_ptr(), n2w->data_ptr(), n2b->data_ptr(), (float)eps[3 * blk + 1],
                                             f1w->data_ptr(), f1b->data_ptr(), f2w->data_ptr(), f2b->data_ptr(), rs2->data_ptr(),
                                             next_w.data_ptr(), next_b.data_ptr(), (float)next_eps, xo.data_ptr(), normed.data_ptr(), r.st));
        x = xo;
      } else {
        Tensor h = r.make(HD);
        check(m2d_layernorm_linear_fwd(r.P, (int)C, (int)HD, r.wd, x.data_ptr(), n2w->data_ptr(), n2b->data_ptr(), (float)eps[3 * blk + 1],
                                       f1w->data_ptr(), f1b->data_ptr(), M2D_ACT_GELU, nullptr, nullptr, h.data_ptr(), r.st));
        branch = r.linear(h, *f2w, f2b, M2D_ACT_NONE, nullptr, nullptr, M2D_ACT_NONE, nullptr, nullptr);
      }
    } else {
      Tensor n2;
      x = r.residual_norm(x, *rs1, term, term2, *n2w, *n2b, eps[3 * blk + 1], n2);
      branch = r.linear(r.linear(n2, *f1w, f1b, M2D_ACT_NONE, nullptr, nullptr, M2D_ACT_GELU, nullptr, nullptr), *f2w, f2b, M2D_ACT_NONE, nullptr,
                        nullptr, M2D_ACT_NONE, nullptr, nullptr);
    }
    if (branch.defined()) x = r.residual_norm(x, *rs2, branch, none, next_w, next_b, next_eps, normed);
  }
  return normed;
}

std::vector<Tensor> widen_op(at::TensorList in) { return m2dshim::widen(in); }

}  // namespace

namespace m2dshim {

// fp32 copies of bf16 tensors, in one launch; fp32 tensors pass through
std::vector<Tensor> widen(at::TensorList in) {
  std::vector<Tensor> out(in.begin(), in.end());
  std::vector<m2d_widen_seg> segs;
  for (auto& t : out) {
    if (t.scalar_type() == at::kFloat) continue;
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.is_contiguous() && t.device() == out[0].device(),
                "m2dscan: widen takes contiguous float32 or bfloat16 tensors on one GPU");
    Tensor w = at::empty(t.sizes(), t.options().dtype(at::kFloat));
    if (t.numel()) segs.push_back({t.data_ptr(), w.data_ptr<float>(), t.numel()});
    t = w;
  }
  if (!segs.empty()) {
    c10::DeviceGuard guard(out[0].device());
    check(m2d_widen((int)segs.size(), segs.data(), current_stream(out[0])));
  }
  return out;
}

}  // namespace m2dshim

TORCH_LIBRARY_FRAGMENT(m2dscan, m) {
  m.def("infer_stage(Tensor x, Tensor[] params, int[] kinds, float[] eps, Tensor cos, Tensor sin, float att_scale) -> Tensor");
  m.def("widen(Tensor[] tensors) -> Tensor[]");
}
TORCH_LIBRARY_IMPL(m2dscan, CUDA, m) {
  m.impl("infer_stage", &infer_stage);
  m.impl("widen", &widen_op);
}
