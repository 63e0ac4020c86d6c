// C++ autograd nodes of the sparse window attention and of the encoder around
// it (linear layers, projection group, LayerNorms).
//
// Sparse attention: the same operation and contract as SparseAttentionFunction in attention.py
// (the reference op is CoreAttention.sparse_attention_bias,
// NeutronGT/models/graphormer_dist_node_level.py:67-98): (q, k, v) ->
// (out, node_scores), node scores without gradient, optional detached extra
// key rows (k_ext, v_ext).  Forward and backward call the library's C ABI
// (ngt_sparse_fwd_ext / ngt_sparse_bwd_strided) through function pointers that the
// Python side hands over once from the loaded libngt_attn.so, so a layer's
// forward and backward run no Python frame, take no GIL on the autograd
// engine's device thread and convert no ctypes arguments.  Host code only:
// every kernel is in libngt_attn.so.
//
// The window is passed as two tensors: `csr` (CPU bytes of one
// ngt_window_csr) and `csr_mem` (the device allocation its pointers point
// into).  Both are kept by the node until the backward has run.
//
// q, k, v may also come as [1, n, H, d], the layout the encoders hold: the
// output is then [1, n_q, H * d] and the gradients have the inputs' shape, so
// that no view node stands between the projections, the core and the output
// projection.
//
// Linear, Projection3, LayerNorm and AddLayerNorm are _WgradLinearFn,
// _ProjectionGroupFn (of three layers), _LayerNormFn and _AddLayerNormFn of
// linear.py and layernorm.py: the same casts, library GEMMs and kernels in the
// same order, bit for bit.  Those Python nodes and the view nodes cost 10-60 us
// of host time each: forward and backward of the 3-layer GPH_Slim model (254
// launches, 1.4 ms of kernels) took 4.0 ms and take 2.9, a GPH_Large block
// over 10,007 queries 1.37 -> 0.97 ms, and the core alone over a small window
// 113 -> 91 us (74 -> 60 us on a faster host).
#include <torch/extension.h>

#include <c10/hip/HIPStream.h>

#include <map>
#include <string>

#include "ngt_attn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::tensor_list;

decltype(&ngt_sparse_fwd_ext) g_fwd = nullptr;
decltype(&ngt_sparse_bwd_strided) g_bwd = nullptr;
decltype(&ngt_last_error) g_err = nullptr;
decltype(&ngt_colsum_workspace_bytes) g_colsum_ws = nullptr;
decltype(&ngt_colsum_bf16) g_colsum = nullptr;
decltype(&ngt_chunk_sum_f32) g_chunk_sum = nullptr;
decltype(&ngt_wgrad_workspace_bytes) g_wgrad_ws = nullptr;
decltype(&ngt_wgrad_pays) g_wgrad_pays = nullptr;
decltype(&ngt_wgrad_bf16) g_wgrad = nullptr;
decltype(&ngt_layernorm_fwd) g_ln_fwd = nullptr;
decltype(&ngt_layernorm_bwd_workspace_bytes) g_ln_bwd_ws = nullptr;
decltype(&ngt_layernorm_bwd) g_ln_bwd = nullptr;
decltype(&ngt_add_layernorm_fwd) g_add_ln_fwd = nullptr;
decltype(&ngt_add_layernorm_bwd) g_add_ln_bwd = nullptr;

void check(int rc) {
  if (rc != NGT_OK) {
    const char* msg = g_err ? g_err() : nullptr;
    TORCH_CHECK(!(msg && *msg), msg);
    TORCH_CHECK(false, "libngt_attn error ", rc);
  }
}

int dtype_code(const Tensor& t) {
  if (t.scalar_type() == at::kFloat) return NGT_F32;
  if (t.scalar_type() == at::kBFloat16) return NGT_BF16;
  TORCH_CHECK(false, "unsupported dtype ", t.scalar_type(), " (float32 or bfloat16)");
  return -1;
}

void* stream_of(const Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

const ngt_window_csr* csr_of(const Tensor& bytes) {
  return reinterpret_cast<const ngt_window_csr*>(bytes.data_ptr());
}

// 16-byte aligned contiguous rows, as the library requires
Tensor rows16(const Tensor& t) {
  if (!t.is_contiguous()) return t.contiguous();
  if (reinterpret_cast<uintptr_t>(t.data_ptr()) % 16) return t.clone();
  return t;
}

// The library reads rows [n, H, d] of one dtype from 16-byte aligned,
// contiguous GPU memory on q's device; anything else is an error here rather
// than wrong reads in the kernels.
void check_rows(const char* name, const Tensor& t, const Tensor& q) {
  TORCH_CHECK(t.is_cuda(), name, " must be a GPU tensor");
  TORCH_CHECK(t.device() == q.device(), name, " is on ", t.device(), ", q on ", q.device());
  TORCH_CHECK(t.scalar_type() == q.scalar_type(), name, " has dtype ", t.scalar_type(),
              ", q has ", q.scalar_type());
  TORCH_CHECK((t.dim() == 3 || (t.dim() == 4 && t.size(0) == 1)) && t.size(-2) == q.size(-2) &&
                  t.size(-1) == q.size(-1),
              name, " must be [n, ", q.size(-2), ", ", q.size(-1), "], got ", t.sizes());
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
  TORCH_CHECK(reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, name,
              " must be 16-byte aligned");
}

Tensor workspace(int64_t bytes, const Tensor& like) {
  return at::empty({std::max<int64_t>(bytes, 1)}, like.options().dtype(at::kByte));
}

constexpr int kInputs = 15;  // forward arguments after ctx

struct SparseAttention : public torch::autograd::Function<SparseAttention> {
  static tensor_list forward(AutogradContext* ctx, Tensor q, Tensor k, Tensor v,
                             std::optional<Tensor> k_ext_opt, std::optional<Tensor> v_ext_opt,
                             Tensor csr, Tensor csr_mem, int64_t dst_end,
                             double scale, double lo, double hi, double eps, int64_t fwd_bytes,
                             int64_t bwd_bytes, bool interleave_grads) {
    TORCH_CHECK(g_fwd && g_bwd, "ngt_autograd.init() was not called");
    // an absent argument is an empty optional: autograd inputs may not be
    // undefined tensors
    const Tensor k_ext = k_ext_opt.value_or(Tensor()), v_ext = v_ext_opt.value_or(Tensor());
    const bool ext = k_ext.defined();
    TORCH_CHECK(ext == v_ext.defined(), "k_ext and v_ext must be given together");
    check_rows("q", q, q);
    check_rows("k", k, q);
    check_rows("v", v, q);
    TORCH_CHECK(k.sizes() == v.sizes(), "k and v differ in shape: ", k.sizes(), " vs ", v.sizes());
    if (ext) {
      check_rows("k_ext", k_ext, q);
      check_rows("v_ext", v_ext, q);
      TORCH_CHECK(k_ext.sizes() == v_ext.sizes(), "k_ext and v_ext differ in shape");
    }
    TORCH_CHECK(q.dim() == k.dim(), "q and k differ in dimensions");
    const int64_t n_q = q.size(-3), n_k = k.size(-3), H = q.size(-2), d = q.size(-1);
    Tensor out = q.dim() == 4 ? at::empty({1, n_q, H * d}, q.options()) : at::empty_like(q);
    const auto f32 = q.options().dtype(at::kFloat);
    Tensor rinv = at::empty({n_q, H}, f32);
    Tensor ns = at::empty({dst_end}, f32);
    Tensor ws = workspace(fwd_bytes, q);
    check(g_fwd(dtype_code(q), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                ext ? k_ext.data_ptr() : nullptr, ext ? v_ext.data_ptr() : nullptr,
                static_cast<int32_t>(n_k), csr_of(csr), static_cast<int32_t>(H),
                static_cast<int32_t>(d), static_cast<float>(scale), static_cast<float>(lo),
                static_cast<float>(hi), static_cast<float>(eps), out.data_ptr(),
                rinv.data_ptr<float>(), dst_end ? ns.data_ptr<float>() : nullptr,
                static_cast<int32_t>(dst_end), ws.data_ptr(), static_cast<size_t>(fwd_bytes),
                stream_of(q)));
    ctx->save_for_backward({q, k, v, out, rinv});
    ctx->saved_data["k_ext"] = k_ext;  // detached key rows (no gradient)
    ctx->saved_data["v_ext"] = v_ext;
    ctx->saved_data["csr"] = csr;
    ctx->saved_data["csr_mem"] = csr_mem;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["lo"] = lo;
    ctx->saved_data["hi"] = hi;
    ctx->saved_data["bwd_bytes"] = bwd_bytes;
    ctx->saved_data["interleave"] = interleave_grads && n_q == n_k;
    ctx->mark_non_differentiable({ns});
    // the node scores have no gradient: no zero tensor is made for them
    ctx->set_materialize_grads(false);
    return {out, ns};
  }

  static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
    tensor_list res(kInputs);
    if (!grads[0].defined()) return res;  // the output was not used by the loss
    const auto saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &out = saved[3], &rinv = saved[4];
    const Tensor k_ext = ctx->saved_data["k_ext"].toTensor();
    const Tensor v_ext = ctx->saved_data["v_ext"].toTensor();
    const Tensor csr = ctx->saved_data["csr"].toTensor();
    const int64_t bwd_bytes = ctx->saved_data["bwd_bytes"].toInt();
    const Tensor g = rows16(grads[0].to(q.scalar_type()));
    const int64_t n_q = q.size(-3), n_k = k.size(-3), H = q.size(-2), d = q.size(-1);
    Tensor gq, gk, gv;
    int64_t ldg = 0;
    if (ctx->saved_data["interleave"].toBool()) {
      // one [N, 3, H, d] buffer: row i holds dQ, dK, dV of row i side by side
      const Tensor buf = at::empty({n_q, 3, H, d}, q.options());
      ldg = 3 * H * d;
      const auto rows = q.dim() == 4 ? std::vector<int64_t>{n_q * ldg, ldg, d, 1}
                                     : std::vector<int64_t>{ldg, d, 1};
      gq = buf.as_strided(q.sizes(), rows, 0);
      gk = buf.as_strided(q.sizes(), rows, H * d);
      gv = buf.as_strided(q.sizes(), rows, 2 * H * d);
    } else {
      gq = at::empty_like(q);
      gk = at::empty_like(k);
      gv = at::empty_like(v);
    }
    Tensor ws = workspace(bwd_bytes, q);
    const bool ext = k_ext.defined();
    check(g_bwd(dtype_code(q), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                ext ? k_ext.data_ptr() : nullptr, ext ? v_ext.data_ptr() : nullptr,
                static_cast<int32_t>(n_k), out.data_ptr(), g.data_ptr(),
                rinv.data_ptr<float>(), csr_of(csr), static_cast<int32_t>(H),
                static_cast<int32_t>(d),
                static_cast<float>(ctx->saved_data["scale"].toDouble()),
                static_cast<float>(ctx->saved_data["lo"].toDouble()),
                static_cast<float>(ctx->saved_data["hi"].toDouble()), gq.data_ptr(),
                gk.data_ptr(), gv.data_ptr(), ldg, ws.data_ptr(), static_cast<size_t>(bwd_bytes),
                stream_of(q)));
    res[0] = gq;
    res[1] = gk;
    res[2] = gv;
    return res;
  }
};

std::tuple<Tensor, Tensor> sparse_attention(Tensor q, Tensor k, Tensor v,
                                            std::optional<Tensor> k_ext,
                                            std::optional<Tensor> v_ext, Tensor csr,
                                            Tensor csr_mem, int64_t dst_end, double scale,
                                            double lo, double hi, double eps, int64_t fwd_bytes,
                                            int64_t bwd_bytes, bool interleave_grads) {
  TORCH_CHECK(csr.device().is_cpu() && csr.scalar_type() == at::kByte &&
                  csr.numel() == static_cast<int64_t>(sizeof(ngt_window_csr)),
              "csr must hold the bytes of one ngt_window_csr (", sizeof(ngt_window_csr), ")");
  auto r = SparseAttention::apply(q, k, v, k_ext, v_ext, csr, csr_mem, dst_end, scale, lo, hi, eps,
                                  fwd_bytes, bwd_bytes, interleave_grads);
  return {r[0], r[1]};
}

// ------------------------------------------------------- the encoder's layers
// torch's casts of the operands stay off inside these nodes: their GEMMs take
// the operands as they are
struct NoAutocast {
  c10::impl::ExcludeDispatchKeyGuard guard{c10::autocast_dispatch_keyset};
};

constexpr int64_t kChunk = 2048;  // as _CHUNK and _MAX_SPLITS of linear.py
constexpr int64_t kMaxSplits = 16;

// fp32 column sums of a contiguous bf16 [K, n] matrix
Tensor colsum(const Tensor& dy) {
  const int64_t K = dy.size(0);
  const auto n = static_cast<int32_t>(dy.size(1));
  Tensor out = at::empty({n}, dy.options().dtype(at::kFloat));
  size_t bytes = 0;
  check(g_colsum_ws(K, n, &bytes));
  Tensor ws = workspace(static_cast<int64_t>(bytes), dy);
  check(g_colsum(dy.data_ptr(), K, n, out.data_ptr<float>(), ws.data_ptr(), bytes, stream_of(dy)));
  return out;
}

// dY^T X in fp32 by library GEMMs split over rows (_library_weight_grad of
// linear.py)
Tensor library_weight_grad(const Tensor& x, const Tensor& dy) {
  const int64_t K = x.size(0), n_in = x.size(1), n_out = dy.size(1);
  const int64_t most = n_out * n_in < 1500000 ? kMaxSplits : kMaxSplits / 2;
  const int64_t splits = std::max<int64_t>(1, std::min(most, K / kChunk));
  const int64_t c = K / splits, main = splits * c;
  if (splits == 1) return at::mm(dy.t(), x, at::kFloat);
  Tensor parts = at::bmm(dy.narrow(0, 0, main).view({splits, c, n_out}).transpose(1, 2),
                         x.narrow(0, 0, main).view({splits, c, n_in}), at::kFloat)
                     .contiguous();
  Tensor dw = at::empty({n_out, n_in}, parts.options());
  check(g_chunk_sum(parts.data_ptr<float>(), static_cast<int32_t>(splits), n_out * n_in,
                    dw.data_ptr<float>(), stream_of(x)));
  if (main < K) dw.add_(at::mm(dy.narrow(0, main, K - main).t(), x.narrow(0, main, K - main),
                               at::kFloat));
  return dw;
}

// dw = dY^T X and, where wanted, db = column sums of dY, in fp32 from
// contiguous bf16 rows (_grads of linear.py).  x may be undefined where dw is not
// wanted.
void linear_grads(const Tensor& x, const Tensor& dy, Tensor* dw, Tensor* db) {
  if (!dw) {
    if (db) *db = colsum(dy);
    return;
  }
  const int64_t K = x.size(0), n_in = x.size(1), n_out = dy.size(1);
  // (a vmapped backward's tensors have no storage: torch's GEMMs take them)
  if (at::GradMode::is_enabled() || !x.has_storage() || !dy.has_storage() ||
      !g_wgrad_pays(K, n_out, n_in)) {
    *dw = library_weight_grad(x, dy);
    if (db) *db = colsum(dy);
    return;
  }
  const auto opt = x.options().dtype(at::kFloat);
  *dw = at::empty({n_out, n_in}, opt);
  if (db) *db = at::empty({n_out}, opt);
  size_t bytes = 0;
  check(g_wgrad_ws(K, static_cast<int32_t>(n_out), static_cast<int32_t>(n_in), &bytes));
  Tensor ws = workspace(static_cast<int64_t>(bytes), x);
  check(g_wgrad(x.data_ptr(), dy.data_ptr(), K, static_cast<int32_t>(n_out),
                static_cast<int32_t>(n_in), dw->data_ptr<float>(),
                db ? db->data_ptr<float>() : nullptr, ws.data_ptr(), bytes, stream_of(x)));
}

Tensor bf16(const Tensor& t) { return t.to(at::kBFloat16); }

std::optional<Tensor> bf16(const std::optional<Tensor>& t) {
  return t.has_value() ? std::optional<Tensor>(bf16(*t)) : std::nullopt;
}

// y = x W^T + b in bf16; fp32 dW and db
struct Linear : public torch::autograd::Function<Linear> {
  static Tensor forward(AutogradContext* ctx, Tensor x, Tensor weight,
                        std::optional<Tensor> bias) {
    NoAutocast off;
    const Tensor x16 = bf16(x), w16 = bf16(weight);
    Tensor y = at::linear(x16, w16, bf16(bias));
    ctx->save_for_backward({x16, w16});
    ctx->saved_data["bias"] = bias.has_value();
    return y;
  }

  static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
    NoAutocast off;
    const auto saved = ctx->get_saved_variables();
    const Tensor &x16 = saved[0], &w16 = saved[1];
    const int64_t n_out = w16.size(0), n_in = w16.size(1);
    tensor_list res(3);
    const Tensor g2 = bf16(grads[0]).reshape({-1, n_out}).contiguous();
    if (ctx->needs_input_grad(0)) res[0] = at::mm(g2, w16).view(x16.sizes());
    const bool want_b = ctx->saved_data["bias"].toBool() && ctx->needs_input_grad(2);
    const bool want_w = ctx->needs_input_grad(1);
    linear_grads(want_w ? x16.reshape({-1, n_in}).contiguous() : Tensor(), g2,
                 want_w ? &res[1] : nullptr, want_b ? &res[2] : nullptr);
    return res;
  }
};

Tensor linear(Tensor x, Tensor weight, std::optional<Tensor> bias) {
  return Linear::apply(x, weight, bias);
}

// the [M, 3 * n_out] matrix whose column blocks are the gradients g, when they
// are views of one buffer laid out that way (linear.py's _joint_rows, the one
// place that knows the layout); else undefined
Tensor joint_rows(const tensor_list& g, int64_t n_out) {
  pybind11::gil_scoped_acquire gil;
  pybind11::tuple views(g.size());
  for (size_t i = 0; i < g.size(); ++i)
    views[i] = g[i].defined() ? pybind11::cast(g[i]) : pybind11::none();
  const pybind11::object r =
      pybind11::module_::import("neutrongt_amd.linear").attr("_joint_rows")(views, n_out);
  return r.is_none() ? Tensor() : r.cast<Tensor>();
}

// Three projections of one input (Q, K, V) as one node.  heads > 0: the
// outputs as [..., heads, n_out / heads].
struct Projection3 : public torch::autograd::Function<Projection3> {
  static tensor_list forward(AutogradContext* ctx, Tensor x, Tensor w0, std::optional<Tensor> b0,
                             Tensor w1, std::optional<Tensor> b1, Tensor w2,
                             std::optional<Tensor> b2, int64_t heads) {
    NoAutocast off;
    const Tensor x16 = bf16(x);
    const Tensor w[3] = {bf16(w0), bf16(w1), bf16(w2)};
    const std::optional<Tensor> b[3] = {b0, b1, b2};
    tensor_list ys;
    int64_t has_bias = 0;
    for (int i = 0; i < 3; ++i) {
      Tensor y = at::linear(x16, w[i], bf16(b[i]));
      if (heads > 0) {
        auto shape = y.sizes().vec();
        shape.back() /= heads;
        shape.insert(shape.end() - 1, heads);
        y = y.view(shape);
      }
      ys.push_back(y);
      has_bias |= int64_t(b[i].has_value()) << i;
    }
    ctx->save_for_backward({x16, w[0], w[1], w[2]});
    ctx->saved_data["bias"] = has_bias;
    ctx->set_materialize_grads(false);  // an unused output: no GEMMs, no weight gradient
    return ys;
  }

  static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
    NoAutocast off;
    const auto saved = ctx->get_saved_variables();
    const Tensor& x16 = saved[0];
    const tensor_list w(saved.begin() + 1, saved.end());
    const int64_t has_bias = ctx->saved_data["bias"].toInt();
    const int64_t n_in = x16.size(-1), n_out = w[0].size(0);
    // the node's edges are numbered over the tensors that were given
    bool want_w[3], want_b[3];
    size_t edge = 1;
    for (int i = 0; i < 3; ++i) {
      want_w[i] = ctx->needs_input_grad(edge++);
      want_b[i] = (has_bias >> i & 1) && ctx->needs_input_grad(edge++);
    }
    tensor_list res(8);
    Tensor joint;
    if (w[1].size(0) == n_out && w[2].size(0) == n_out && want_w[0] && want_w[1] && want_w[2] &&
        ((want_b[0] && want_b[1] && want_b[2]) || has_bias == 0))
      joint = joint_rows(grads, n_out);
    if (joint.defined()) {
      if (ctx->needs_input_grad(0)) res[0] = at::mm(joint, at::cat(w, 0)).view(x16.sizes());
      Tensor dw, db;
      linear_grads(x16.reshape({-1, n_in}).contiguous(), joint, &dw, has_bias ? &db : nullptr);
      for (int i = 0; i < 3; ++i) {
        res[1 + 2 * i] = dw.narrow(0, i * n_out, n_out);
        if (has_bias) res[2 + 2 * i] = db.narrow(0, i * n_out, n_out);
      }
      return res;
    }
    Tensor x2, gx;
    for (int i = 0; i < 3; ++i) {
      if (!grads[i].defined()) continue;
      const Tensor g2 = bf16(grads[i]).reshape({-1, w[i].size(0)}).contiguous();
      if (ctx->needs_input_grad(0)) {
        if (gx.defined())
          gx.addmm_(g2, w[i]);
        else
          gx = at::mm(g2, w[i]);
      }
      if (want_w[i] && !x2.defined()) x2 = x16.reshape({-1, n_in}).contiguous();
      linear_grads(x2, g2, want_w[i] ? &res[1 + 2 * i] : nullptr,
                   want_b[i] ? &res[2 + 2 * i] : nullptr);
    }
    if (gx.defined()) res[0] = gx.view(x16.sizes());
    return res;
  }
};

tensor_list project3(Tensor x, Tensor w0, std::optional<Tensor> b0, Tensor w1,
                     std::optional<Tensor> b1, Tensor w2, std::optional<Tensor> b2,
                     int64_t heads) {
  return Projection3::apply(x, w0, b0, w1, b1, w2, b2, heads);
}

// [n, n_cols] contiguous rows whose base meets the LayerNorm kernels'
// alignment: 16 bytes for fp32, 8 for bf16
Tensor ln_rows(const Tensor& t, int64_t n_cols) {
  const Tensor r = t.reshape({-1, n_cols});
  const uintptr_t align = r.scalar_type() == at::kFloat ? 16 : 8;
  if (!r.is_contiguous() || reinterpret_cast<uintptr_t>(r.data_ptr()) % align)
    return r.clone(at::MemoryFormat::Contiguous);
  return r;
}

Tensor ln_grad(const Tensor& g) {
  return g.scalar_type() == at::kFloat || g.scalar_type() == at::kBFloat16 ? g : g.to(at::kFloat);
}

Tensor f32(const Tensor& t) { return t.to(at::kFloat).contiguous(); }

struct LayerNorm : public torch::autograd::Function<LayerNorm> {
  static Tensor forward(AutogradContext* ctx, Tensor x, Tensor weight, Tensor bias, double eps,
                        bool out_bf16) {
    NoAutocast off;
    const int64_t n_cols = weight.numel();
    const Tensor x2 = ln_rows(x, n_cols), w = f32(weight), b = f32(bias);
    const int64_t n = x2.size(0);
    const auto opt = x.options().dtype(at::kFloat);
    Tensor y = at::empty(x.sizes(), out_bf16 ? x.options().dtype(at::kBFloat16) : opt,
                         at::MemoryFormat::Contiguous);
    Tensor mean = at::empty({n}, opt), rstd = at::empty({n}, opt);
    check(g_ln_fwd(dtype_code(x2), x2.data_ptr(), n, static_cast<int32_t>(n_cols),
                   w.data_ptr<float>(), b.data_ptr<float>(), static_cast<float>(eps),
                   dtype_code(y), y.data_ptr(), mean.data_ptr<float>(), rstd.data_ptr<float>(),
                   stream_of(x)));
    ctx->save_for_backward({x2, w, mean, rstd});
    ctx->saved_data["shape"] = x.sizes().vec();
    return y;
  }

  static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
    NoAutocast off;
    const auto saved = ctx->get_saved_variables();
    const Tensor &x2 = saved[0], &w = saved[1], &mean = saved[2], &rstd = saved[3];
    const int64_t n = x2.size(0), n_cols = x2.size(1);
    const Tensor g2 = ln_rows(ln_grad(grads[0]), n_cols);
    Tensor dx = at::empty_like(x2);
    Tensor dw = at::empty({n_cols}, w.options()), db = at::empty({n_cols}, w.options());
    size_t bytes = 0;
    check(g_ln_bwd_ws(n, static_cast<int32_t>(n_cols), &bytes));
    Tensor ws = workspace(static_cast<int64_t>(bytes), x2);
    check(g_ln_bwd(dtype_code(x2), x2.data_ptr(), dtype_code(g2), g2.data_ptr(), n,
                   static_cast<int32_t>(n_cols), w.data_ptr<float>(), mean.data_ptr<float>(),
                   rstd.data_ptr<float>(), dx.data_ptr(), dw.data_ptr<float>(),
                   db.data_ptr<float>(), ws.data_ptr(), bytes, stream_of(x2)));
    return {dx.view(ctx->saved_data["shape"].toIntVector()), dw, db, Tensor(), Tensor()};
  }
};

Tensor layernorm(Tensor x, Tensor weight, Tensor bias, double eps, bool out_bf16) {
  return LayerNorm::apply(x, weight, bias, eps, out_bf16);
}

// (s, LayerNorm(s)) with s = x + dropout(y)
struct AddLayerNorm : public torch::autograd::Function<AddLayerNorm> {
  static tensor_list forward(AutogradContext* ctx, Tensor x, Tensor y, Tensor weight, Tensor bias,
                             double eps, double p, std::optional<Tensor> seed_opt, bool out_bf16) {
    NoAutocast off;
    const int64_t n_cols = weight.numel();
    const Tensor x2 = ln_rows(x, n_cols), y2 = ln_rows(y, n_cols), w = f32(weight), b = f32(bias);
    TORCH_CHECK(y2.scalar_type() == x2.scalar_type() && y2.sizes() == x2.sizes(),
                "x and y differ in dtype or shape");
    const Tensor seed = seed_opt.value_or(Tensor());
    const int64_t n = x2.size(0);
    const auto opt = x.options().dtype(at::kFloat);
    Tensor s = at::empty(x.sizes(), x.options(), at::MemoryFormat::Contiguous);
    Tensor out = at::empty(x.sizes(), out_bf16 ? x.options().dtype(at::kBFloat16) : opt,
                           at::MemoryFormat::Contiguous);
    Tensor mean = at::empty({n}, opt), rstd = at::empty({n}, opt);
    check(g_add_ln_fwd(dtype_code(x2), x2.data_ptr(), y2.data_ptr(), n,
                       static_cast<int32_t>(n_cols), static_cast<float>(p), 0, seed_ptr(seed),
                       w.data_ptr<float>(), b.data_ptr<float>(), static_cast<float>(eps),
                       s.data_ptr(), dtype_code(out), out.data_ptr(), mean.data_ptr<float>(),
                       rstd.data_ptr<float>(), stream_of(x)));
    ctx->save_for_backward({s, w, mean, rstd, seed});
    ctx->saved_data["p"] = p;
    ctx->set_materialize_grads(false);  // an unused sum: no zero tensor for its gradient
    return {s, out};
  }

  static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
    NoAutocast off;
    const auto saved = ctx->get_saved_variables();
    const Tensor &s = saved[0], &w = saved[1], &mean = saved[2], &rstd = saved[3];
    const int64_t n = mean.numel(), n_cols = w.numel();
    tensor_list res(8);
    if (!grads[0].defined() && !grads[1].defined()) return res;
    const Tensor g_out =
        grads[1].defined() ? ln_rows(ln_grad(grads[1]), n_cols) : at::zeros({n, n_cols}, w.options());
    const Tensor g_s =
        grads[0].defined() ? ln_rows(grads[0].to(s.scalar_type()), n_cols) : Tensor();
    Tensor dx = at::empty_like(s), dy = at::empty_like(s);
    Tensor dw = at::empty({n_cols}, w.options()), db = at::empty({n_cols}, w.options());
    size_t bytes = 0;
    check(g_ln_bwd_ws(n, static_cast<int32_t>(n_cols), &bytes));
    Tensor ws = workspace(static_cast<int64_t>(bytes), s);
    check(g_add_ln_bwd(dtype_code(s), s.data_ptr(), dtype_code(g_out), g_out.data_ptr(),
                       g_s.defined() ? g_s.data_ptr() : nullptr, n, static_cast<int32_t>(n_cols),
                       static_cast<float>(ctx->saved_data["p"].toDouble()), 0, seed_ptr(saved[4]),
                       w.data_ptr<float>(), mean.data_ptr<float>(), rstd.data_ptr<float>(),
                       dx.data_ptr(), dy.data_ptr(), dw.data_ptr<float>(), db.data_ptr<float>(),
                       ws.data_ptr(), bytes, stream_of(s)));
    res[0] = dx;
    res[1] = dy;
    res[2] = dw;
    res[3] = db;
    return res;
  }

 private:
  static const uint64_t* seed_ptr(const Tensor& seed) {
    return seed.defined() ? static_cast<const uint64_t*>(seed.data_ptr()) : nullptr;
  }
};

std::tuple<Tensor, Tensor> add_layernorm(Tensor x, Tensor y, Tensor weight, Tensor bias, double eps,
                                         double p, std::optional<Tensor> seed, bool out_bf16) {
  auto r = AddLayerNorm::apply(x, y, weight, bias, eps, p, seed, out_bf16);
  return {r[0], r[1]};
}

template <typename F>
void entry(F*& fn, const std::map<std::string, int64_t>& addr, const char* name) {
  const auto it = addr.find(name);
  TORCH_CHECK(it != addr.end() && it->second, "ngt_autograd.init: no address of ", name);
  fn = reinterpret_cast<F*>(it->second);
}

void init(const std::map<std::string, int64_t>& addr) {
  entry(g_fwd, addr, "ngt_sparse_fwd_ext");
  entry(g_bwd, addr, "ngt_sparse_bwd_strided");
  entry(g_err, addr, "ngt_last_error");
  entry(g_colsum_ws, addr, "ngt_colsum_workspace_bytes");
  entry(g_colsum, addr, "ngt_colsum_bf16");
  entry(g_chunk_sum, addr, "ngt_chunk_sum_f32");
  entry(g_wgrad_ws, addr, "ngt_wgrad_workspace_bytes");
  entry(g_wgrad_pays, addr, "ngt_wgrad_pays");
  entry(g_wgrad, addr, "ngt_wgrad_bf16");
  entry(g_ln_fwd, addr, "ngt_layernorm_fwd");
  entry(g_ln_bwd_ws, addr, "ngt_layernorm_bwd_workspace_bytes");
  entry(g_ln_bwd, addr, "ngt_layernorm_bwd");
  entry(g_add_ln_fwd, addr, "ngt_add_layernorm_fwd");
  entry(g_add_ln_bwd, addr, "ngt_add_layernorm_bwd");
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("init", &init, "{name: address} of libngt_attn.so's entry points");
  m.def("csr_struct_bytes", []() { return static_cast<int64_t>(sizeof(ngt_window_csr)); });
  m.def("abi_version", []() { return static_cast<int64_t>(NGT_ABI_VERSION); },
        "NGT_ABI_VERSION of the header this extension was compiled against");
  m.def("sparse_attention", &sparse_attention,
        "(q, k, v, k_ext, v_ext, csr, csr_mem, dst_end, scale, lo, hi, eps, fwd_bytes, "
        "bwd_bytes, interleave_grads) -> (out, node_scores); interleave_grads: dQ, dK, dV as "
        "views of one [N, 3, H, d] buffer (when q and k have the same rows)");
  m.def("linear", &linear, "(x, weight, bias) -> y: linear.py's _WgradLinearFn");
  m.def("project3", &project3,
        "(x, w0, b0, w1, b1, w2, b2, heads) -> [y0, y1, y2]: linear.py's _ProjectionGroupFn; "
        "heads > 0: outputs [..., heads, n_out / heads]");
  m.def("layernorm", &layernorm, "(x, weight, bias, eps, out_bf16) -> y: layernorm.py's _LayerNormFn");
  m.def("add_layernorm", &add_layernorm,
        "(x, y, weight, bias, eps, p, seed tensor or None, out_bf16) -> (s, out): layernorm.py's "
        "_AddLayerNormFn");
}
