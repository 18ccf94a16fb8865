// The operator API's autograd nodes and the layer's decode step, over the C ABI
// of liblizard_hip.so (include/lizard_hip.h), for calls whose kernels take less
// time than their launches did from Python.
//
// kernels.py keeps the argument checks (and the Python nodes for calls that are
// traced or run under function transforms); what is here is the work of a call
// that passed them: casts, outputs, workspaces, launches on the tensors' current
// stream, and the graph node.  The nodes and layer_step make the launches that
// Python made on the same operands, with the same bits; layer_step_rows forms the
// projections with rows.hip's products, whose sums run in another order than the
// library's (each rounded to bf16 once, as there).  Measured for a forward and
// backward of one sequence (H = 32, L = 2048, d = 64), where the kernels take 75 and
// 35 us: gla 138 -> 87 us, swa 120 -> 75 us; a short forward (H = 4, L = 256) 17.6 ->
// 11.4 us (10.0 since its walks fold the segment records); a decode step of the layer
// (B = 4, hidden 2048) 201 -> 132 us with torch's projections, 48 us with rows.hip's.
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <cmath>
#include <stdexcept>
#include <string>
#include <tuple>

#include "../../include/lizard_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void* stream_of(const Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

void check(int rc, const char* what) {
  if (rc != 0)
    throw std::runtime_error(std::string(what) + " failed (status " + std::to_string(rc) +
                             "): " + lz_last_error());
}

template <typename T = void>
T* ptr(const Tensor& t) {
  return t.defined() && t.numel() ? static_cast<T*>(t.data_ptr()) : nullptr;
}

Tensor as(const Tensor& t, at::ScalarType dtype) {
  return (t.scalar_type() == dtype ? t : t.to(dtype)).contiguous();
}
Tensor bf16(const Tensor& t) { return as(t, at::kBFloat16); }
Tensor f32(const Tensor& t) { return as(t, at::kFloat); }

Tensor bytes(size_t n, const Tensor& like) {
  return at::empty({static_cast<int64_t>(n)}, like.options().dtype(at::kByte));
}

int i32(int64_t x) { return static_cast<int>(x); }

bool any_grad(std::initializer_list<const Tensor*> tensors) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : tensors)
    if (t->requires_grad()) return true;
  return false;
}

// gradients come back in the inputs' dtypes; the kernels write bf16 ones when
// q, k and v (fq, fk and v) are all bf16, else fp32
at::ScalarType grad_dtype(const std::vector<int64_t>& dtypes) {
  for (int i = 0; i < 3; ++i)
    if (static_cast<at::ScalarType>(dtypes[i]) != at::kBFloat16) return at::kFloat;
  return at::kBFloat16;
}

// ---------------------------------------------------------------------------
// gated linear attention
// ---------------------------------------------------------------------------

int padded(int64_t n) { return n <= 32 ? 32 : n <= 64 ? 64 : n <= 128 ? 128 : n <= 256 ? 256 : 0; }

// whether the walks take (F, D) directly (gla_fwd.hip's gla_dims_supported): the
// forward's workspace then holds segment records that the backward reuses
bool gla_native(int64_t nf, int64_t nd) {
  const int fp = padded(nf), dp = padded(nd);
  return fp && dp && dp <= 128 && (fp <= 128 || dp <= 64);
}

std::tuple<Tensor, Tensor> gla_forward(const Tensor& fq, const Tensor& fk, const Tensor& v,
                                       const Tensor& lg, bool keep_state, int64_t chunk) {
  const int64_t b = fq.size(0), h = fq.size(1), n = fq.size(2), nf = fq.size(3), nd = v.size(3);
  Tensor y = at::empty({b, h, n, nd}, v.options()), ws;
  if (y.numel()) {
    const int per_head = lg.dim() == 3 ? LZ_GATE_PER_HEAD : 0;
    const size_t need = lz_gla_fwd_workspace_bytes(i32(b), i32(h), i32(n), i32(nf), i32(nd),
                                                   per_head, i32(chunk));
    if (need) ws = bytes(need, fq);
    check(lz_gla_fwd(ptr(fq), ptr(fk), ptr(v), ptr<float>(lg), ptr(y), i32(b), i32(h),
                     i32(fk.size(1)), i32(n), i32(nf), i32(nd),
                     per_head | (keep_state ? 0 : LZ_GLA_NO_REUSE), i32(chunk), ptr(ws), need,
                     stream_of(fq)),
          "lz_gla_fwd");
  }
  return {y, keep_state && gla_native(nf, nd) ? ws : Tensor()};
}

struct Gla : torch::autograd::Function<Gla> {
  static Tensor forward(AutogradContext* ctx, const Tensor& fq_, const Tensor& fk_,
                        const Tensor& v_, const Tensor& lg_, int64_t chunk) {
    const Tensor fq = bf16(fq_), fk = bf16(fk_), v = bf16(v_), lg = f32(lg_);
    auto [y, state] = gla_forward(fq, fk, v, lg, true, chunk);
    ctx->save_for_backward({fq, fk, v, lg});
    ctx->saved_data["dtypes"] = std::vector<int64_t>{
        static_cast<int64_t>(fq_.scalar_type()), static_cast<int64_t>(fk_.scalar_type()),
        static_cast<int64_t>(v_.scalar_type()), static_cast<int64_t>(lg_.scalar_type())};
    ctx->saved_data["chunk"] = chunk;
    if (state.defined()) ctx->saved_data["state"] = state;   // the segments' state records
    return y;
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &fq = saved[0], &fk = saved[1], &v = saved[2], &lg = saved[3];
    const auto dtypes = ctx->saved_data["dtypes"].toIntVector();
    const int64_t chunk = ctx->saved_data["chunk"].toInt();
    const auto kept = ctx->saved_data.find("state");
    const Tensor state = kept == ctx->saved_data.end() ? Tensor() : kept->second.toTensor();
    const int64_t b = fq.size(0), h = fq.size(1), n = fq.size(2), nf = fq.size(3), nd = v.size(3);
    const Tensor dy = grads[0].defined() ? bf16(grads[0]) : at::zeros({b, h, n, nd}, v.options());
    const auto gdt = grad_dtype(dtypes);
    const auto opts = fq.options().dtype(gdt);
    Tensor dfq = at::empty(fq.sizes(), opts), dfk = at::empty(fq.sizes(), opts),
           dv = at::empty({b, h, n, nd}, opts), dlg = at::empty(lg.sizes(), lg.options());
    if (dy.numel()) {
      const int mode = lg.dim() == 3 ? LZ_GATE_PER_HEAD : 0;
      const size_t need = lz_gla_bwd_workspace_bytes(i32(b), i32(h), i32(n), i32(nf), i32(nd), mode,
                                                     i32(chunk));
      const Tensor ws = bytes(need ? need : 1, fq);
      check(lz_gla_bwd(ptr(fq), ptr(fk), ptr(v), ptr<float>(lg), ptr(dy), ptr(dfq), ptr(dfk),
                       ptr(dv), ptr<float>(dlg), gdt == at::kBFloat16, i32(b), i32(h),
                       i32(fk.size(1)), i32(n), i32(nf), i32(nd), mode, i32(chunk), ptr(state),
                       state.defined() ? static_cast<size_t>(state.numel()) : 0, ptr(ws),
                       static_cast<size_t>(ws.numel()), stream_of(fq)),
            "lz_gla_bwd");
    } else {
      for (Tensor* t : {&dfq, &dfk, &dv, &dlg}) t->zero_();
    }
    variable_list out{dfq, dfk, dv, dlg, Tensor()};
    for (int i = 0; i < 4; ++i) out[i] = out[i].to(static_cast<at::ScalarType>(dtypes[i]));
    return out;
  }
};

Tensor gla(const Tensor& fq, const Tensor& fk, const Tensor& v, const Tensor& lg, int64_t chunk) {
  if (any_grad({&fq, &fk, &v, &lg})) return Gla::apply(fq, fk, v, lg, chunk);
  return std::get<0>(gla_forward(bf16(fq), bf16(fk), bf16(v), f32(lg), false, chunk));
}

// ---------------------------------------------------------------------------
// sliding-window softmax with sinks
// ---------------------------------------------------------------------------

std::tuple<Tensor, Tensor> swa_forward(const Tensor& q, const Tensor& k, const Tensor& v,
                                       const Tensor& meta, int64_t window) {
  const int64_t b = q.size(0), h = q.size(1), n = q.size(2), d = q.size(3);
  Tensor y = at::empty(q.sizes(), q.options());
  Tensor lse = at::empty({b, h, n}, v.options().dtype(at::kFloat));
  if (y.numel())
    check(lz_swa_fwd(ptr(q), ptr(k), ptr(v), ptr<float>(meta), i32(meta.numel()), ptr(y),
                     ptr<float>(lse), i32(b), i32(h), i32(k.size(1)), i32(n), i32(d), i32(window),
                     static_cast<float>(1.0 / std::sqrt(static_cast<double>(d))), stream_of(q)),
          "lz_swa_fwd");
  return {y, lse};
}

struct Swa : torch::autograd::Function<Swa> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q_, const Tensor& k_, const Tensor& v_,
                        const Tensor& meta_, int64_t window) {
    const Tensor q = bf16(q_), k = bf16(k_), v = bf16(v_), meta = f32(meta_);
    auto [y, lse] = swa_forward(q, k, v, meta, window);
    ctx->save_for_backward({q, k, v, meta, lse});
    ctx->saved_data["dtypes"] = std::vector<int64_t>{
        static_cast<int64_t>(q_.scalar_type()), static_cast<int64_t>(k_.scalar_type()),
        static_cast<int64_t>(v_.scalar_type()), static_cast<int64_t>(meta_.scalar_type())};
    ctx->saved_data["window"] = window;
    return y;
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &meta = saved[3], &lse = saved[4];
    const auto dtypes = ctx->saved_data["dtypes"].toIntVector();
    const int64_t window = ctx->saved_data["window"].toInt();
    const int64_t b = q.size(0), h = q.size(1), n = q.size(2), d = q.size(3);
    const Tensor dy = grads[0].defined() ? bf16(grads[0]) : at::zeros(q.sizes(), q.options());
    const auto gdt = grad_dtype(dtypes);
    const auto opts = q.options().dtype(gdt);
    Tensor dq = at::empty(q.sizes(), opts), dk = at::empty(q.sizes(), opts),
           dv = at::empty(q.sizes(), opts), dmeta = at::empty(meta.sizes(), meta.options());
    if (dy.numel()) {
      const int sinks = i32(meta.numel());
      const size_t need = lz_swa_bwd_workspace_bytes(i32(b), i32(h), i32(n), i32(d), sinks);
      const Tensor ws = bytes(need ? need : 1, q);
      check(lz_swa_bwd(ptr(q), ptr(k), ptr(v), ptr<float>(meta), sinks, ptr<float>(lse), ptr(dy),
                       ptr(dq), ptr(dk), ptr(dv), ptr<float>(dmeta), gdt == at::kBFloat16, i32(b),
                       i32(h), i32(k.size(1)), i32(n), i32(d), i32(window),
                       static_cast<float>(1.0 / std::sqrt(static_cast<double>(d))), ptr(ws),
                       static_cast<size_t>(ws.numel()), stream_of(q)),
            "lz_swa_bwd");
    } else {
      for (Tensor* t : {&dq, &dk, &dv, &dmeta}) t->zero_();
    }
    variable_list out{dq, dk, dv, dmeta, Tensor()};
    for (int i = 0; i < 4; ++i) out[i] = out[i].to(static_cast<at::ScalarType>(dtypes[i]));
    return out;
  }
};

Tensor swa(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& meta, int64_t window) {
  if (any_grad({&q, &k, &v, &meta})) return Swa::apply(q, k, v, meta, window);
  return std::get<0>(swa_forward(bf16(q), bf16(k), bf16(v), f32(meta), window));
}

// ---------------------------------------------------------------------------
// the layer's decode step between its projections and o_proj
// ---------------------------------------------------------------------------

bool is(const Tensor& t, at::IntArrayRef sizes, const Tensor& like) {
  return t.defined() && t.sizes() == sizes && t.device() == like.device();
}

// Whether layer_step's launches, which take every size from the layer (heads, kv,
// window, hd), fit these tensors: shapes, devices, and the layout and types of the
// buffers that are written in place.  Projections that are formed later are left
// out.  A step that does not fit goes operator by operator, which casts or refuses
// what it is given.
bool step_takes(const std::vector<Tensor>& projections, const Tensor& wq, const Tensor& wk,
                const Tensor& cos, const Tensor& sin, const Tensor& meta, const Tensor& alpha,
                const Tensor& state, const Tensor& k_cache, const Tensor& v_cache, int64_t heads,
                int64_t kv, int64_t window, int64_t hd, int64_t pos) {
  if (state.dim() != 3 || wq.dim() != 2 || pos < 0) return false;
  const int64_t b = state.size(0), f = wq.size(0), nf = 2 * f;
  for (size_t i = 0; i < projections.size(); ++i)
    if (!is(projections[i], {b, 1, (i ? kv : heads) * hd}, state)) return false;
  const bool rope = cos.sizes() == sin.sizes() &&
                    (is(cos, {1, hd}, state) || is(cos, {1, 1, hd}, state) ||
                     is(cos, {b, 1, hd}, state));
  if (b <= 0 || !rope || sin.device() != state.device() || !is(wq, {f, hd}, state) ||
      !is(wk, {f, hd}, state) || !is(state, {b, heads, nf * hd + nf}, state) ||
      state.scalar_type() != at::kFloat || !state.is_contiguous() || meta.dim() != 1 ||
      meta.device() != state.device() || alpha.numel() != 1 || alpha.device() != state.device())
    return false;
  for (const Tensor* t : {&k_cache, &v_cache})
    if (!is(*t, {b, kv, window, hd}, state) || t->scalar_type() != at::kBFloat16 ||
        !t->is_contiguous())
      return false;
  return true;
}

// Whether rows_linear takes w [n, K] (any n < 1) for x's rows of K columns
bool row_weight(const Tensor& w, int64_t n, int64_t cols, const Tensor& x) {
  return w.dim() == 2 && (n < 1 || w.size(0) == n) && w.size(1) == cols &&
         w.scalar_type() == at::kBFloat16 && w.is_contiguous() && w.device() == x.device() &&
         reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0 && w.numel() < (int64_t{1} << 29);
}

// Whether layer_step_rows can form the projections of x [B, 1, hidden] by weights
// {q_proj, k_proj, v_proj, W_gamma, o_proj}: each [its outputs, its inputs]
bool rows_take(const Tensor& x, const std::vector<Tensor>& w, int64_t q_width, int64_t kv_width) {
  return x.dim() == 3 && x.size(1) == 1 && x.size(0) > 0 && x.size(0) <= LZ_ROWS_MAX &&
         x.scalar_type() == at::kBFloat16 && x.size(2) > 0 && x.size(2) % 8 == 0 &&
         reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 && w.size() == 5 &&
         row_weight(w[0], q_width, x.size(2), x) && row_weight(w[1], kv_width, x.size(2), x) &&
         row_weight(w[2], kv_width, x.size(2), x) && row_weight(w[3], 1, x.size(2), x) &&
         row_weight(w[4], 0, q_width, x);
}

// One token per sequence at position pos: the prologue on the projections' rows
// (qp [B, 1, heads hd], kp, vp [B, 1, kv hd]), the GLA step on `state` with the
// token's gate logit z [B, 1, 1] (a logit per head goes by operators), and the
// window step that puts the token's key and value into their cache slot and
// blends the two branches.  For tensors that step_takes; others raise.  Returns
// [B, 1, heads hd] (bf16 when out_bf16, else fp32).
Tensor layer_step(Tensor qp, Tensor kp, Tensor vp, const Tensor& z, Tensor wq, Tensor wk,
                  Tensor cos, Tensor sin, const Tensor& meta, const Tensor& alpha,
                  const Tensor& state, const Tensor& k_cache, const Tensor& v_cache,
                  int64_t heads_, int64_t kv_, int64_t window_, int64_t hd_, int64_t pos,
                  bool out_bf16) {
  TORCH_CHECK(step_takes({qp, kp, vp}, wq, wk, cos, sin, meta, alpha, state, k_cache, v_cache,
                         heads_, kv_, window_, hd_, pos),
              "layer_step: tensors that do not fit the layer's sizes");
  TORCH_CHECK(is(z, {qp.size(0), 1, 1}, state), "layer_step: one gate logit per token expected");
  const int b = i32(state.size(0)), heads = i32(heads_), kv = i32(kv_), window = i32(window_),
            hd = i32(hd_), f = i32(wq.size(0));
  bool all_bf16 = true;
  for (const Tensor* t : {&qp, &kp, &vp, &wq, &wk, &cos, &sin})
    all_bf16 = all_bf16 && t->scalar_type() == at::kBFloat16;
  const auto dtype = all_bf16 ? at::kBFloat16 : at::kFloat;
  for (Tensor* t : {&qp, &kp, &vp, &wq, &wk, &cos, &sin}) *t = as(*t, dtype);
  // RoPE rows [1, hd] for all sequences, or [B, 1, hd]
  const int batched = cos.numel() != hd;
  const auto opts = state.options().dtype(at::kBFloat16);
  const Tensor fq = at::empty({b, heads, 2 * f}, opts), fk = at::empty({b, kv, 2 * f}, opts),
               qr = at::empty({b, heads, hd}, opts), kr = at::empty({b, kv, hd}, opts),
               v = at::empty({b, kv, hd}, opts), yg = at::empty({b, heads, hd}, opts);
  void* stream = stream_of(state);
  check(lz_layer_prologue_fwd(ptr(qp), ptr(kp), ptr(vp), ptr(wq), ptr(wk), ptr(cos), ptr(sin),
                              batched, ptr(fq), ptr(fk), ptr(qr), ptr(kr), ptr(v), all_bf16, b, 1,
                              heads, kv, hd, f, stream),
        "lz_layer_prologue_fwd");
  const Tensor logit = f32(z);
  check(lz_gla_decode_step(ptr(fq), ptr(fk), ptr(v), ptr<float>(logit), ptr<float>(state), ptr(yg),
                           b, heads, kv, 2 * f, hd, LZ_GATE_LOGIT, stream),
        "lz_gla_decode_step");
  const bool params_bf16 =
      meta.scalar_type() == at::kBFloat16 && alpha.scalar_type() == at::kBFloat16;
  const Tensor sinks = params_bf16 ? meta.contiguous() : f32(meta);
  const Tensor blend = params_bf16 ? alpha.contiguous() : f32(alpha);
  Tensor out = at::empty({b, 1, static_cast<int64_t>(heads) * hd},
                         opts.dtype(out_bf16 ? at::kBFloat16 : at::kFloat));
  check(lz_layer_decode_swa(ptr(qr), ptr(kr), ptr(v), ptr(k_cache), ptr(v_cache), ptr(sinks),
                            i32(sinks.numel()), ptr(blend), params_bf16, ptr(yg), ptr(out),
                            out_bf16, b, heads, kv, window, hd, i32(pos),
                            static_cast<float>(1.0 / std::sqrt(static_cast<double>(hd))), stream),
        "lz_layer_decode_swa");
  return out;
}

// y_i = x w_i^T for the rows of x [.., K]; outputs [.., n_i], the ones in `wide`
// as fp32
std::vector<Tensor> rows_linear(const Tensor& x, const std::vector<Tensor>& w,
                                const std::vector<bool>& wide) {
  TORCH_CHECK(w.size() <= LZ_ROWS_MATS && w.size() == wide.size(), "rows_linear: at most ",
              LZ_ROWS_MATS, " matrices");
  TORCH_CHECK(x.dim() > 0 && x.numel() && x.scalar_type() == at::kBFloat16 && x.is_contiguous(),
              "rows_linear: x must be contiguous bf16 rows");
  const int rows = i32(x.numel() / x.size(-1)), cols = i32(x.size(-1)), mats = i32(w.size());
  const void* wp[LZ_ROWS_MATS];
  void* yp[LZ_ROWS_MATS];
  int n[LZ_ROWS_MATS], f32out[LZ_ROWS_MATS];
  for (const Tensor& m : w)
    TORCH_CHECK(row_weight(m, 0, cols, x), "rows_linear: matrices must be contiguous bf16 [n, ",
                cols, "] on x's device, 16-byte aligned");
  std::vector<Tensor> y;
  for (int i = 0; i < mats; ++i) {
    auto sizes = x.sizes().vec();
    sizes.back() = w[i].size(0);
    y.push_back(at::empty(sizes, x.options().dtype(wide[i] ? at::kFloat : at::kBFloat16)));
    wp[i] = ptr(w[i]);
    yp[i] = ptr(y[i]);
    n[i] = i32(w[i].size(0));
    f32out[i] = wide[i];
  }
  check(lz_rows_linear(ptr(x), rows, cols, mats, wp, yp, n, f32out, stream_of(x)),
        "lz_rows_linear");
  return y;
}

// The whole step of a bf16 layer whose projections are plain matrices (rows_take),
// for x [B, 1, hidden], B <= LZ_ROWS_MAX: the four projections of x in one launch
// (the gate's logit as fp32, of its bf16 value), the step, and o_proj.
Tensor layer_step_rows(const Tensor& x, const std::vector<Tensor>& w, const Tensor& wq,
                       const Tensor& wk, const Tensor& cos, const Tensor& sin, const Tensor& meta,
                       const Tensor& alpha, const Tensor& state, const Tensor& k_cache,
                       const Tensor& v_cache, int64_t heads, int64_t kv, int64_t window,
                       int64_t hd, int64_t pos) {
  TORCH_CHECK(rows_take(x, w, heads * hd, kv * hd),
              "layer_step_rows: projections that do not fit the layer's sizes");
  const auto p = rows_linear(x.contiguous(), {w[0], w[1], w[2], w[3]}, {false, false, false, true});
  const Tensor y = layer_step(p[0], p[1], p[2], p[3], wq, wk, cos, sin, meta, alpha, state, k_cache,
                             v_cache, heads, kv, window, hd, pos, true);
  return rows_linear(y, {w[4]}, {false})[0];
}

}  // namespace

PYBIND11_MODULE(lizard_torch, m) {
  const auto nogil = py::call_guard<py::gil_scoped_release>();
  m.def("gla_native", &gla_native);
  m.def("gla", &gla, nogil);
  m.def("swa", &swa, nogil);
  m.def("step_takes", &step_takes, nogil);
  m.def("rows_take", &rows_take, nogil);
  m.def("layer_step", &layer_step, nogil);
  m.def("layer_step_rows", &layer_step_rows, nogil);
  m.def("rows_linear", &rows_linear, nogil);
  m.attr("ROWS_MAX") = LZ_ROWS_MAX;
}
