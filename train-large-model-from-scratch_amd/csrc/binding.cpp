// The differentiable entry points as autograd nodes in C++: what `functional.py` calls.
//
// A small step is bound by the host (a step of 512 tokens of a narrow layer has 0.1 ms of kernels), and
// most of that host time was Python: argument handling, a dozen allocations and the node itself, in both
// directions.  The nodes below do the same with three allocations per direction besides the results, and
// the backward pass runs on the engine's thread without taking the interpreter's lock.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/extension.h>

#include <string>
#include <tuple>
#include <vector>

#include "moe_gfx950.h"
#include "router.h"

// (from internal.h and layer.hip, which only device code can include)
void moe_observe(const char* name, int after);
bool moe_router_few_ok(int64_t T, int64_t H, int64_t E, int64_t k);
int moe_router_logits(const uint16_t* x, const uint16_t* wr, int64_t T, int64_t H, int64_t E, uint16_t* logits,
                      void* stream);
int moe_cast_two(const float* a, uint16_t* to_a, int64_t na, const float* b, uint16_t* to_b, int64_t nb, void* stream);
bool moe_place_ok(int64_t T, int64_t E, int64_t k);
int64_t moe_place_bytes(int64_t T, int64_t E);
int moe_select_count(const void* logits, int logits_dtype, const float* bias, int64_t T, int64_t E, int64_t k,
                     int32_t* ids, float* gates, void* table, void* stream);
int moe_place_rows(const void* x, int x_dtype, const int32_t* ids, const void* table, int64_t T, int64_t H, int64_t E,
                   int64_t k, int32_t* counts, int32_t* offs, int32_t* pos_to_row, int32_t* row_to_pos, int32_t* bad_ids,
                   void* xp, int xp_dtype, bool counted, void* stream);
bool moe_select_place_ok(const void* logits, int64_t T, int64_t E, int64_t k);
int moe_select_place(const void* x, int x_dtype, const void* logits, int logits_dtype, const float* bias, int64_t T, int64_t H,
                     int64_t E, int64_t k, int32_t* ids, float* gates, int32_t* counts, int32_t* offs, int32_t* pos_to_row,
                     int32_t* row_to_pos, int32_t* bad_ids, void* xp, int xp_dtype, void* stream);
int moe_rmsnorm_router_count(const void* x, int x_dtype, const float* weight, float eps, const uint16_t* router_weight,
                             int64_t T, int64_t H, int64_t E, int64_t k, uint16_t* xn, float* rstd, uint16_t* logits,
                             int32_t* ids, float* gates, void* table, void* stream);
int64_t moe_forward_scratch(const moe_layer_forward_args* a);
int64_t moe_backward_scratch(const moe_layer_backward_args* a);
int moe_f32_gateup(const float* xp, const float* w1, const float* w3, const int32_t* offs, int64_t E, int64_t R, int64_t H,
                   int64_t I, float* g, float* u, float* act, void* stream);
int moe_f32_permute_bwd_router(const float* dxp, const int32_t* row_to_pos, const float* gates, const float* dgates,
                               const int32_t* ids, const float* wr, int64_t T, int64_t H, int64_t k, float* dsel, float* dx,
                               void* stream);
int64_t moe_f32_router_wgrad_floats(int64_t R, int64_t H, int64_t E);
int moe_f32_router_wgrad(const float* xp, const float* dsel, const int32_t* offs, int64_t R, int64_t H, int64_t E, float* partial,
                         float* dwr, void* stream);
int moe_f32_wgrads(const float* dg, const float* du, const float* dyp, const float* xp, const float* act, const int32_t* offs,
                   int64_t E, int64_t R, int64_t H, int64_t I, float* dw1, float* dw3, float* dw2, void* stream);

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
typedef std::optional<Tensor> OptTensor;

namespace {

PyObject* error_type = nullptr;  // lib.MoELibError

// Raised as lib.MoELibError.  (torch's own kind of exception with a Python type: the autograd engine hands those
// of a backward pass on as they are, any other becomes a plain RuntimeError.)
struct LibError : torch::PyTorchError {
  using torch::PyTorchError::PyTorchError;
  PyObject* python_type() override { return error_type ? error_type : PyExc_RuntimeError; }
};

void check(int rc, const char* name) {
  if (rc == 0) return;
  static const char* const names[] = {"MOE_ERR_NULL", "MOE_ERR_SHAPE", "MOE_ERR_LIMIT",
                                      "MOE_ERR_DTYPE", "MOE_ERR_WORKSPACE", "MOE_ERR_ALIGN"};
  const std::string what = rc < 0 && rc >= -6 ? std::string(names[-rc - 1])
                                              : (rc > 0 ? "hipError_t " : "code ") + std::to_string(rc);
  throw LibError(std::string(name) + " failed: " + what);
}

#define CALL(fn, ...)                \
  do {                               \
    moe_observe(#fn, 0);             \
    const int rc_ = fn(__VA_ARGS__); \
    moe_observe(#fn, 1);             \
    check(rc_, #fn);                 \
  } while (0)

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

int64_t dt(at::ScalarType t) {
  if (t == at::kBFloat16) return MOE_DT_BF16;
  if (t == at::kFloat) return MOE_DT_F32;
  throw torch::TypeError("unsupported dtype: the MoE kernels take bf16 or fp32");
}
int64_t dt(const Tensor& t) { return dt(t.scalar_type()); }

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

void need_gpu(const Tensor& t) {
  TORCH_CHECK(!t.defined() || t.is_cuda(), "the MoE kernels need GPU tensors (no CPU path exists)");
}

// The kernels read pointers: a tangent that forward-mode differentiation hangs on an input would be lost without a
// word, in the node (whose backward is all it has) and around it (where nothing requires a gradient).
void no_tangents(std::initializer_list<const Tensor*> inputs) {
  for (const Tensor* t : inputs)
    TORCH_CHECK_NOT_IMPLEMENTED(!t->defined() || !t->_fw_grad(/*level=*/0).defined(),
                                "the MoE kernels have no forward-mode derivative");
}

// Contiguous and 16-byte aligned, as the kernels need their buffers.
Tensor dense(const Tensor& t) {
  need_gpu(t);
  Tensor c = t.is_contiguous() ? t : t.contiguous();
  return (reinterpret_cast<uintptr_t>(c.data_ptr()) & 15) == 0 ? c : c.clone();
}

Tensor empty(at::IntArrayRef size, at::ScalarType type, const Tensor& like) {
  return at::empty(size, at::TensorOptions().dtype(type).device(like.device()));
}

Tensor cast_bf16(const Tensor& t) {
  if (t.scalar_type() == at::kBFloat16) return t;
  if (t.scalar_type() != at::kFloat) return t.to(at::kBFloat16);
  Tensor out = empty(t.sizes(), at::kBFloat16, t);
  CALL(moe_cast_f32_bf16, t.data_ptr<float>(), (uint16_t*)out.data_ptr(), t.numel(), stream_of(t));
  return out;
}

const uint16_t* bf(const Tensor& t) { return (const uint16_t*)ptr(t); }

// The bf16 product is a bf16 product whatever autocast the caller is in.
struct NoAutocast {
  c10::impl::ExcludeDispatchKeyGuard guard{c10::DispatchKey::AutocastCUDA};
};

int64_t up(int64_t n, int64_t to) { return (n + to - 1) / to * to; }

// What a forward pass leaves for the backward pass besides its inputs: the routing (int32 words, parts in
// this order: ids, gates, counts, offs, pos_to_row, row_to_pos, bad ids) and the expert-ordered rows xp
// (unless the experts read x where it is) with gu and act behind them.
struct Routing {
  enum Part { IDS, GATES, COUNTS, OFFS, POS_TO_ROW, ROW_TO_POS, BAD, PARTS };
  int64_t at[PARTS + 1];
  Routing(int64_t R, int64_t E) {
    const int64_t n[PARTS] = {R, R, E, E + 1, R, R, 1};
    at[0] = 0;
    for (int i = 0; i < PARTS; ++i) at[i + 1] = at[i] + up(n[i], 64);
  }
  int32_t* part(const Tensor& buf, Part p) const { return buf.data_ptr<int32_t>() + at[p]; }
};

struct Kept {
  int64_t gu, act, total;
  Kept(int64_t R, int64_t H, int64_t E, int64_t I, bool with_gu, bool with_xp) {
    gu = with_xp ? up(R * H * 2, 256) : 0;
    act = gu + (with_gu ? up(moe_gu_blocked_bytes(R, E, I), 256) : 0);
    total = act + up(R * I * 2, 256);
    if (total == 0) total = 256;
  }
};

struct Weights {
  Tensor w1, w3, w2;
};

Weights bf16_weights(const Tensor& w1, const Tensor& w3, const Tensor& w2, const OptTensor& s1, const OptTensor& s3,
                     const OptTensor& s2) {
  const auto one = [](const Tensor& w, const OptTensor& s) { return s && s->defined() ? *s : cast_bf16(dense(w)); };
  return {one(w1, s1), one(w3, s3), one(w2, s2)};
}

// A copy the caller made is read in place of its master: it has to be what cast_bf16(dense(master)) would be.
void check_copy(const OptTensor& s, const Tensor& w, const Tensor& x) {
  if (!s || !s->defined()) return;
  need_gpu(*s);
  TORCH_CHECK(s->device() == x.device(), "a bf16 copy of the weights is on ", s->device(), ", x on ", x.device());
  TORCH_CHECK_TYPE(s->scalar_type() == at::kBFloat16, "the copies of the weights must be bf16, got ", s->scalar_type());
  TORCH_CHECK(s->sizes() == w.sizes(), "a bf16 copy has shape ", s->sizes(), ", its weights ", w.sizes());
  TORCH_CHECK(s->is_contiguous(), "the MoE kernels need contiguous tensors: a bf16 copy of the weights is strided");
}

// Logits [tokens, E] and the fp32 constant per expert that is added to them.
void check_logits(const Tensor& logits, const Tensor& bias, const Tensor& x, int64_t E) {
  TORCH_CHECK(!logits.defined() || (logits.dim() == 2 && logits.size(0) == x.size(0) && logits.size(1) == E),
              "the logits have shape ", logits.sizes(), ", x ", x.sizes(), " and there are ", E, " experts");
  if (!bias.defined()) return;
  TORCH_CHECK_TYPE(bias.scalar_type() == at::kFloat, "the bias must be fp32, got ", bias.scalar_type());
  TORCH_CHECK(bias.numel() == E, "the bias has ", bias.numel(), " elements, there are ", E, " experts");
}

const Tensor& value(const OptTensor& t) {
  static const Tensor none;
  return t ? *t : none;
}

// Autograd counts a node's inputs without the tensors that were not given.
struct Present {
  int64_t mask = 0;
  Present() = default;
  Present(std::initializer_list<bool> given) {
    int i = 0;
    for (bool g : given) mask |= (int64_t)g << i++;
  }
  int index(int input) const { return __builtin_popcountll(mask & ((1ll << input) - 1)); }
  bool wants_gradient(AutogradContext* ctx, int input) const {
    return (mask >> input & 1) && ctx->needs_input_grad(index(input));
  }
  torch::autograd::Node* next(const torch::autograd::Node& node, int input) const {
    return node.next_edge(index(input)).function.get();
  }
};

struct Layer {  // the arguments of one call
  int64_t k = 1;
  double eps = 0;
  bool add_residual = false, fused_router = false, accumulate = false, train = false;
  OptTensor s1, s3, s2;           // bf16 copies of the weights
  Tensor* routing_out = nullptr;  // where the caller wants the routing left
};

struct Outputs {
  Tensor out, logits, routing, kept, xn, wrb, nw, rstd;
  Weights w;
  bool in_place = false;  // no rows in expert order are kept: xn is read instead
};

Outputs forward(const Layer& o, const Tensor& x_, const Tensor& norm_w, const Tensor& wr, const Tensor& logits_,
                const Tensor& w1, const Tensor& w3, const Tensor& w2, const Tensor& bias, const Tensor& ids_) {
  Outputs f;
  need_gpu(x_);
  TORCH_CHECK(x_.dim() == 2 && w1.dim() == 3, "the layer takes x [tokens, hidden] and weights [experts, ., .]");
  const int64_t T = x_.size(0), H = x_.size(1), I = w1.size(1), k = o.k, R = T * k;
  const int64_t E = wr.defined() ? wr.size(0) : logits_.defined() ? logits_.size(1) : w1.size(0);
  TORCH_CHECK(w1.size(0) == E && w3.size(0) == E && w2.size(0) == E && w1.size(2) == H && w3.size(2) == H &&
                  w3.size(1) == I && w2.size(1) == H && w2.size(2) == I,
              "the weights' shapes do not belong together");
  if (wr.defined()) {
    need_gpu(wr);
    TORCH_CHECK(wr.dim() == 2 && wr.size(1) == H, "the router weight has shape ", wr.sizes(), ", x ", x_.sizes());
    TORCH_CHECK(wr.device() == x_.device(), "the router weight is on ", wr.device(), ", x on ", x_.device());
  }
  if (norm_w.defined()) {
    need_gpu(norm_w);
    TORCH_CHECK(norm_w.numel() == H, "the norm's weight has ", norm_w.numel(), " elements, x is ", H, " wide");
    TORCH_CHECK(norm_w.device() == x_.device(), "the norm's weight is on ", norm_w.device(), ", x on ", x_.device());
  }
  check_logits(logits_, bias, x_, E);
  check_copy(o.s1, w1, x_), check_copy(o.s3, w3, x_), check_copy(o.s2, w2, x_);
  (void)dt(x_);
  const at::ScalarType x_type = x_.scalar_type();
  const c10::DeviceGuard guard(x_.device());
  const Tensor x = dense(x_);
  f.w = bf16_weights(w1, w3, w2, o.s1, o.s3, o.s2);
  void* s = stream_of(x);
  const Routing r(R, E);
  Tensor rows = x;
  Tensor logits;
  Tensor table;  // of the selection's counts, where it is done and they are wanted
  bool selected = false, inside = false;  // selection done; the forward-only call makes the logits itself
  MoeRouter router{};                     // its product is part of the layer's call where `own` says so
  bool own = false;
  const Tensor b = bias.defined() ? dense(bias) : Tensor();
  if (o.train || o.routing_out || !(wr.defined() || logits_.defined()) || norm_w.defined() || T == 0)
    f.routing = empty({r.at[Routing::PARTS]}, at::kInt, x);
  if (wr.defined()) {
    const Tensor wrd = dense(wr.detach());
    own = !norm_w.defined() && (wrd.scalar_type() == at::kFloat || wrd.scalar_type() == at::kBFloat16) &&
          moe_router_select_ok(T, H, E, k, (int)dt(wrd));
    const bool both = !own && !norm_w.defined() && x_type == at::kFloat && wrd.scalar_type() == at::kFloat && H % 8 == 0 && T > 0;
    if (own) {  // (what is to be rounded to bf16 is rounded on the way)
      const bool x_as_is = x_type == at::kBFloat16, wr_as_is = wrd.scalar_type() == at::kBFloat16;
      f.xn = x_as_is ? x : empty(x.sizes(), at::kBFloat16, x);
      f.wrb = wr_as_is || !o.train ? wrd : empty(wrd.sizes(), at::kBFloat16, x);
      logits = empty({T, E}, at::kBFloat16, x);
      router.x = x.data_ptr(), router.x_dtype = (int)dt(x), router.wr = wrd.data_ptr(), router.wr_dtype = (int)dt(wrd);
      router.xn = x_as_is ? nullptr : (uint16_t*)f.xn.data_ptr();
      router.wrb = wr_as_is || !o.train ? nullptr : (uint16_t*)f.wrb.data_ptr();
      router.bias = (const float*)ptr(b), router.logits = (uint16_t*)logits.data_ptr();
      inside = !f.routing.defined(), selected = true;
    } else if (both) {  // (a launch each took 4.7 us for the router's weight and 7.7 for 4096 tokens, 1024 wide; together 8.8)
      f.wrb = empty(wrd.sizes(), at::kBFloat16, x);
      f.xn = empty(x.sizes(), at::kBFloat16, x);
      CALL(moe_cast_two, x.data_ptr<float>(), (uint16_t*)f.xn.data_ptr(), x.numel(), wrd.data_ptr<float>(),
           (uint16_t*)f.wrb.data_ptr(), wrd.numel(), s);
    } else {
      f.wrb = dense(cast_bf16(wrd));
    }
    if (norm_w.defined()) {
      f.nw = norm_w.detach().to(at::kFloat).contiguous();
      f.xn = empty({T, H}, at::kBFloat16, x);
      f.rstd = empty({T}, at::kFloat, x);
      if (o.fused_router && !bias.defined() && T > 0 && moe_rmsnorm_router_supported(H, E, k)) {
        // norm, router product and selection in one kernel: the normalised rows are not read a second
        // time for the router, the logits are selected on before they leave the chip
        logits = empty({T, E}, at::kBFloat16, x);
        if (moe_place_ok(T, E, k)) table = empty({moe_place_bytes(T, E)}, at::kByte, x);
        const char* name = "moe_rmsnorm_router_fwd";  // (the entry that callers know; this one leaves the table too)
        moe_observe(name, 0);
        const int rc = moe_rmsnorm_router_count(x.data_ptr(), (int)dt(x), f.nw.data_ptr<float>(), (float)o.eps, bf(f.wrb), T, H, E, k,
                                                (uint16_t*)f.xn.data_ptr(), f.rstd.data_ptr<float>(), (uint16_t*)logits.data_ptr(),
                                                r.part(f.routing, Routing::IDS), (float*)r.part(f.routing, Routing::GATES),
                                                ptr(table), s);
        moe_observe(name, 1);
        check(rc, name);
        selected = true;
      } else {
        CALL(moe_rmsnorm_fwd, x.data_ptr(), (int)dt(x), f.nw.data_ptr<float>(), (float)o.eps, T, H,
             (uint16_t*)f.xn.data_ptr(), f.rstd.data_ptr<float>(), s);
      }
    } else if (!both && !own) {
      f.xn = cast_bf16(x);
    }
    rows = f.xn;
    if (!selected && moe_router_few_ok(T, H, E, k)) {
      logits = empty({T, E}, at::kBFloat16, x);
      inside = !f.routing.defined();
      if (inside) {
        router.x = f.xn.data_ptr(), router.wr = f.wrb.data_ptr(), router.x_dtype = router.wr_dtype = MOE_DT_BF16;
        router.bias = (const float*)ptr(b), router.logits = (uint16_t*)logits.data_ptr();
      } else {
        check(moe_router_logits(bf(f.xn), bf(f.wrb), T, H, E, (uint16_t*)logits.data_ptr(), s), "moe_router_few");
      }
    } else if (!selected) {
      const NoAutocast off;
      logits = at::mm(f.xn, f.wrb.t());
    }
  } else if (logits_.defined()) {
    logits = dense(logits_);
  }
  f.logits = logits;
  if (!f.routing.defined()) {  // nothing is kept and nobody asks for the routing
    f.out = empty({T, H}, x_type, x);
    const int64_t bytes = moe_forward_only_scratch(T, H, E, I, k, (int)dt(rows));
    const Tensor ws = empty({std::max<int64_t>(bytes, 256)}, at::kByte, x);
    // (it tells the observer about its launches itself, as do the two calls of a training step)
    check(moe_forward_only(inside ? &router : nullptr, rows.data_ptr(), (int)dt(rows), inside ? nullptr : logits.data_ptr(),
                           inside ? MOE_DT_BF16 : (int)dt(logits), (const float*)ptr(b), bf(f.w.w1), bf(f.w.w3), bf(f.w.w2), T, H, E, I, k,
                           f.out.data_ptr(), (int)dt(x_type), ws.data_ptr(), ws.numel(), s),
          inside ? "moe_routed_forward" : "moe_ffn_forward");
    return f;
  }
  f.out = empty({T, H}, x_type, x);
  // (only where xn is saved whatever happens: with given logits or experts the caller may change x after the call)
  f.in_place = o.train && f.xn.defined() && moe_layer_rows_from_ok(T, H, E, I, k);
  const Kept kept(R, H, E, I, o.train, !f.in_place);
  f.kept = empty({kept.total}, at::kByte, x);
  char* base = (char*)f.kept.data_ptr();
  Tensor ids = ids_;
  moe_layer_forward_args a{};
  a.T = T, a.H = H, a.E = E, a.I = I, a.k = k;
  a.x = rows.data_ptr(), a.x_dtype = dt(rows);
  a.ids = r.part(f.routing, Routing::IDS);
  a.gates = (float*)r.part(f.routing, Routing::GATES);
  if (logits.defined() && !selected) {
    a.logits = logits.data_ptr(), a.logits_dtype = dt(logits), a.bias = (const float*)ptr(b);
  } else if (!logits.defined()) {  // rows already dispatched: their experts are given
    ids = dense(ids.scalar_type() == at::kLong || ids.scalar_type() == at::kInt ? ids : ids.to(at::kInt));
    TORCH_CHECK(ids.numel() == R, "one expert id per row is needed");
    a.gates = nullptr;
    if (ids.scalar_type() == at::kLong) a.ids64 = ids.data_ptr<int64_t>();
    else a.ids = ids.data_ptr<int32_t>();
    a.bad_ids = r.part(f.routing, Routing::BAD);
  }
  a.counts = r.part(f.routing, Routing::COUNTS), a.offs = r.part(f.routing, Routing::OFFS);
  a.pos_to_row = r.part(f.routing, Routing::POS_TO_ROW), a.row_to_pos = r.part(f.routing, Routing::ROW_TO_POS);
  a.w1 = bf(f.w.w1), a.w3 = bf(f.w.w3), a.w2 = bf(f.w.w2);
  a.residual = o.add_residual ? x.data_ptr() : nullptr;
  a.out = f.out.data_ptr(), a.out_dtype = dt(x_type);
  a.xp = f.in_place ? nullptr : (uint16_t*)base;
  a.gu = o.train ? base + kept.gu : nullptr;
  a.act = (uint16_t*)(base + kept.act);
  const int64_t bytes = std::max<int64_t>(moe_forward_scratch(&a), 256);
  const Tensor scratch = empty({bytes}, at::kByte, x);
  a.scratch = scratch.data_ptr(), a.scratch_bytes = bytes;
  check(moe_selected_layer_forward(&a, own ? &router : nullptr, ptr(table), s), "moe_layer_forward");
  if (o.routing_out) *o.routing_out = f.routing;
  return f;
}

void first_order_only() {
  // Called at the top of every backward here.  The backward passes run kernels autograd cannot see
  // through, so a gradient of a gradient would silently lack their terms (grad mode is on inside a
  // backward pass only under create_graph).
  TORCH_CHECK(!at::GradMode::is_enabled(),
              "the MoE kernels' backward pass is not differentiable: call backward()/grad() without create_graph=True");
}

// Where the gradients of the three stacks go: tensors of their own that autograd receives, or (with
// `params`: the masters whose .grad the kernel may write) the existing .grad, added to, or a new one.
struct WeightGradients {
  Tensor into[3], give[3], fresh[3];
  bool add[3] = {false, false, false};
  WeightGradients(const bool (&need)[3], const std::vector<Tensor>& params, const Tensor (&w)[3], at::ScalarType type) {
    for (int i = 0; i < 3; ++i) {
      if (!need[i]) continue;
      const Tensor param = params.empty() ? Tensor() : params[i];
      const Tensor held = param.defined() ? param.grad() : Tensor();
      if (param.defined() && !held.defined()) {
        into[i] = fresh[i] = empty(w[i].sizes(), param.scalar_type(), w[i]);
      } else if (held.defined() && (held.scalar_type() == at::kFloat || held.scalar_type() == at::kBFloat16) &&
                 held.is_contiguous() && held.sizes() == w[i].sizes() && held.device() == w[i].device()) {
        into[i] = held;
        add[i] = true;
      } else {  // autograd takes the gradient (and sums it with a .grad the kernel cannot add to)
        into[i] = give[i] = empty(w[i].sizes(), type, w[i]);
      }
    }
  }
};

// dWr = dlogits^T x for dlogits [T,E], x [T,H].
Tensor router_wgrad(const Tensor& dlogits_, const Tensor& xn_, at::ScalarType type) {
  const int64_t T = xn_.size(0), H = xn_.size(1), E = dlogits_.size(1);
  if (T == 0 || E % 8 != 0 || H % 8 != 0 || !xn_.is_cuda() || xn_.scalar_type() != at::kBFloat16 ||
      dlogits_.scalar_type() != at::kBFloat16)
    return at::mm(dlogits_.t(), xn_).to(type);
  const c10::DeviceGuard guard(xn_.device());
  const Tensor dlogits = dense(dlogits_), xn = dense(xn_);
  const bool direct = type == at::kFloat || type == at::kBFloat16;
  Tensor dw = empty({E, H}, direct ? type : at::kFloat, xn);
  const int64_t bytes = moe_router_wgrad_workspace_bytes(T, H, E);
  const Tensor ws = empty({std::max<int64_t>(bytes, 16)}, at::kByte, xn);
  CALL(moe_router_wgrad, bf(dlogits), bf(xn), T, H, E, dw.data_ptr(), (int)dt(dw), ws.data_ptr(), ws.numel(),
       stream_of(xn));
  return direct ? dw : dw.to(type);
}

// Router product (or given logits, or given expert ids), routing, experts and combine as one node,
// optionally with the caller's RMSNorm in front and residual add behind.
struct LayerNode : torch::autograd::Function<LayerNode> {
  enum Input { X, NORM, WR, LOGITS, W1, W3, W2, BIAS, IDS, OPTIONS, INPUTS };

  static variable_list forward(AutogradContext* ctx, const Tensor& x, const OptTensor& norm_w_, const OptTensor& wr_,
                               const OptTensor& logits_, const Tensor& w1, const Tensor& w3, const Tensor& w2,
                               const OptTensor& bias_, const OptTensor& ids_, const Layer& o) {
    const Tensor &norm_w = value(norm_w_), &wr = value(wr_), &logits = value(logits_), &bias = value(bias_),
                 &ids = value(ids_);
    const Outputs f = ::forward(o, x, norm_w, wr, logits, w1, w3, w2, bias, ids);
    // (y is not kept: the gate gradients come out of the dgrad-down kernel)
    ctx->save_for_backward({norm_w.defined() ? dense(x) : Tensor(), f.nw, f.rstd, f.xn, f.wrb, f.kept, f.routing, f.w.w1,
                            f.w.w3, f.w.w2});
    const auto type = [](const Tensor& t) { return t.defined() ? (int64_t)t.scalar_type() : -1; };
    ctx->saved_data["i"] = std::vector<int64_t>{x.size(0), x.size(1), o.k, o.add_residual, type(x), type(norm_w),
                                                type(wr), type(logits), type(w1),
                                                Present{true, norm_w.defined(), wr.defined(), logits.defined(), true, true,
                                                        true, bias.defined(), ids.defined()}.mask, f.in_place};
    if (o.accumulate) {
      std::vector<Tensor> params;
      for (const Tensor* w : {&w1, &w3, &w2}) params.push_back(w->requires_grad() && w->is_leaf() ? *w : Tensor());
      ctx->saved_data["params"] = params;
    }
    ctx->set_materialize_grads(false);
    if (wr.defined()) return {f.out, f.logits};
    return {f.out};
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    first_order_only();
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &nw = saved[1], &rstd = saved[2], &xn = saved[3], &wrb = saved[4], &kept_buf = saved[5],
                 &routing = saved[6];
    const Tensor w[3] = {saved[7], saved[8], saved[9]};
    const std::vector<int64_t> ints = ctx->saved_data["i"].toIntVector();
    const int64_t T = ints[0], H = ints[1], k = ints[2], R = T * k, E = w[0].size(0), I = w[0].size(1);
    const bool add_residual = ints[3], has_norm = ints[5] >= 0, has_router = ints[6] >= 0, has_logits = ints[7] >= 0;
    const auto type = [&](int i) { return (at::ScalarType)ints[i]; };
    const at::ScalarType x_type = type(4);
    std::vector<Tensor> params;
    const auto held = ctx->saved_data.find("params");
    if (held != ctx->saved_data.end()) params = held->second.toTensorVector();
    const c10::DeviceGuard guard(kept_buf.device());
    Present present;
    present.mask = ints[9];
    const auto need = [&](Input i) { return present.wants_gradient(ctx, i); };

    Tensor dout = grads[0].defined() ? grads[0] : at::zeros({T, H}, kept_buf.options().dtype(x_type));
    dout = dense(dout);
    if (has_router ? dout.scalar_type() != x_type : dout.scalar_type() != at::kBFloat16 && dout.scalar_type() != at::kFloat)
      dout = dout.to(has_router ? x_type : at::kFloat);
    const Tensor ext = has_router && grads.size() > 1 ? grads[1] : Tensor();

    const bool need_w[3] = {need(W1), need(W3), need(W2)};
    const bool want_dx = need(X) || (has_norm && need(NORM)), want_bias = need(BIAS);
    const bool want_logits = has_logits && need(LOGITS), want_wr = has_router && need(WR);
    // the logits' gradient is wanted by itself (for the bias) or has a share from outside: the router's
    // side is then worked out below from the gate gradients
    const bool by_hand = want_bias || ext.defined();
    WeightGradients wg(need_w, params, w, type(8));
    Tensor dx, dxp, dwr, dlogits, dgates, dbias, dnw, d2;
    const bool rows_out = by_hand && has_router;  // the router's share joins below
    if (want_dx && !rows_out) dx = empty({T, H}, x_type, kept_buf);
    if (want_dx && rows_out) dxp = empty({R, H}, at::kBFloat16, kept_buf);
    if (by_hand) dgates = empty({R}, at::kFloat, kept_buf);
    const bool wr_direct = has_router && (type(6) == at::kFloat || type(6) == at::kBFloat16);
    if (!by_hand && want_wr) dwr = empty({E, H}, wr_direct ? type(6) : at::kFloat, kept_buf);
    if (!by_hand && want_logits) dlogits = empty({T, E}, type(7), kept_buf);

    const Routing r(R, E);
    const bool in_place = ints[10];
    const Kept kept(R, H, E, I, true, !in_place);
    const char* base = (const char*)kept_buf.data_ptr();
    void* s = stream_of(kept_buf);
    moe_layer_backward_args a{};
    a.T = T, a.H = H, a.E = E, a.I = I, a.k = k;
    a.dout = dout.data_ptr(), a.dout_dtype = dt(dout);
    const float* gates = has_router || has_logits ? (const float*)r.part(routing, Routing::GATES) : nullptr;
    const int32_t* ids = r.part(routing, Routing::IDS);
    a.gates = gates, a.ids = ids;
    a.offs = r.part(routing, Routing::OFFS);
    a.pos_to_row = r.part(routing, Routing::POS_TO_ROW), a.row_to_pos = r.part(routing, Routing::ROW_TO_POS);
    a.xp = in_place ? nullptr : (const uint16_t*)base, a.gu = base + kept.gu, a.act = (const uint16_t*)(base + kept.act);
    a.w1 = bf(w[0]), a.w3 = bf(w[1]), a.w2 = bf(w[2]);
    for (int i = 0; i < 3; ++i) {
      a.dw[i] = ptr(wg.into[i]);
      a.dw_dtype[i] = wg.into[i].defined() ? dt(wg.into[i]) : 0;
      a.dw_accumulate[i] = wg.add[i];
    }
    if (dlogits.defined()) a.dlogits = dlogits.data_ptr(), a.dlogits_dtype = dt(dlogits);
    a.dgates = (float*)ptr(dgates);
    a.wr = bf(wrb), a.xn = bf(xn);
    if (dwr.defined()) a.dwr = dwr.data_ptr(), a.dwr_dtype = dt(dwr);
    if (dx.defined()) a.dx = dx.data_ptr(), a.dx_dtype = dt(dx);
    a.dxp = (uint16_t*)ptr(dxp);
    const int64_t bytes = std::max<int64_t>(moe_backward_scratch(&a), 256);
    const Tensor scratch = empty({bytes}, at::kByte, kept_buf);
    a.scratch = scratch.data_ptr(), a.scratch_bytes = bytes;
    // (the norm's backward in the pass that adds the rows up)
    const bool norm_inside = has_norm && has_router && want_dx && !by_hand && moe_norm_rows_ok(T, H);
    if (norm_inside) {
      const int64_t nb = std::max<int64_t>(moe_rmsnorm_bwd_workspace_bytes(T, H), 16);
      const Tensor ws = empty({nb}, at::kByte, kept_buf);
      dnw = empty({H}, at::kFloat, kept_buf);
      const MoeNormBackward norm{x.data_ptr(), (int)dt(x), nw.data_ptr<float>(), rstd.data_ptr<float>(),
                                 add_residual ? dout.data_ptr() : nullptr, dnw.data_ptr<float>(), ws.data_ptr(), nb};
      check(moe_norm_layer_backward(&a, norm, s), "moe_layer_backward");
    } else {
      check(in_place ? moe_in_place_layer_backward(&a, s) : moe_layer_backward(&a, s), "moe_layer_backward");
    }
    for (int i = 0; i < 3; ++i)
      if (wg.fresh[i].defined()) params[i].mutable_grad() = wg.fresh[i];
    if (dwr.defined() && !wr_direct) dwr = dwr.to(type(6));

    if (by_hand) {
      const NoAutocast off;
      const auto logit_gradient = [&](at::ScalarType t) {
        Tensor d = empty({T, E}, t, kept_buf);
        CALL(moe_router_topk_bwd, gates, (const float*)ptr(dgates), ids, T, E, k, ptr(d), (int)dt(t), s);
        return d;
      };
      const at::ScalarType logit_type = has_logits ? type(7) : at::kBFloat16;
      if (want_bias) {
        // the bias is a per-expert constant added to the logits (in fp32): its gradient is the column
        // sum of the logits' gradient, taken before that is rounded
        Tensor d32 = logit_gradient(at::kFloat);
        if (ext.defined()) d32 = d32 + ext.to(at::kFloat);
        dbias = d32.sum(0);
        dlogits = d32.to(logit_type);
      } else {
        dlogits = logit_gradient(logit_type);
        dlogits = dlogits + ext.to(logit_type);
      }
      if (has_router) {
        if (want_wr) dwr = router_wgrad(dlogits, xn, type(6));
        if (want_dx) {
          d2 = at::mm(dlogits, wrb);
          dx = empty({T, H}, x_type, kept_buf);
          // (with the norm, the router's share joins inside the norm's backward kernel)
          if (has_norm || T == 0)
            CALL(moe_permute_bwd, bf(dxp), r.part(routing, Routing::ROW_TO_POS), nullptr, T, H, k, ptr(dx), (int)dt(dx), s);
          else
            CALL(moe_permute_bwd_addend, bf(dxp), r.part(routing, Routing::ROW_TO_POS), d2.data_ptr(), (int)dt(d2), T, H, k,
                 ptr(dx), (int)dt(dx), s);
        }
      }
      if (!want_logits) dlogits = Tensor();
    }
    if (norm_inside) {
      dnw = need(NORM) ? dnw.to(type(5)) : Tensor();
    } else if (want_dx && has_norm) {
      const int64_t nb = std::max<int64_t>(moe_rmsnorm_bwd_workspace_bytes(T, H), 16);
      const Tensor ws = empty({nb}, at::kByte, kept_buf);
      const Tensor d1 = dx;
      dx = empty({T, H}, x_type, kept_buf);
      dnw = empty({H}, at::kFloat, kept_buf);
      CALL(moe_rmsnorm_bwd, x.data_ptr(), (int)dt(x), nw.data_ptr<float>(), rstd.data_ptr<float>(), d1.data_ptr(),
           (int)dt(d1), bf(d2), add_residual ? dout.data_ptr() : nullptr, T, H, dx.data_ptr(), dnw.data_ptr<float>(),
           ws.data_ptr(), nb, s);
      dnw = need(NORM) ? dnw.to(type(5)) : Tensor();
    } else if (want_dx && add_residual) {
      dx = dx + dout;
    }
    if (!need(X)) dx = Tensor();
    variable_list out(INPUTS);
    out[X] = dx, out[NORM] = dnw, out[WR] = dwr, out[LOGITS] = dlogits, out[BIAS] = dbias;
    out[W1] = wg.give[0], out[W3] = wg.give[1], out[W2] = wg.give[2];
    return out;
  }
};

// The router product alone: bf16 x [T,H] and wr [E,H] -> bf16 logits, the bits the layer selects on.
Tensor router_logits(const Tensor& x, const Tensor& wr) {
  const at::NoGradGuard off;
  const NoAutocast no_autocast;
  const int64_t T = x.size(0), H = x.size(1), E = wr.size(0);
  if (!x.is_cuda() || x.scalar_type() != at::kBFloat16 || wr.scalar_type() != at::kBFloat16 || H % 8 != 0 ||
      !moe_router_few_ok(T, H, E, 1) || x.dim() != 2 || wr.dim() != 2 || wr.size(1) != H || wr.device() != x.device())
    return at::mm(x, wr.t());  // (which also refuses what does not belong together)
  const c10::DeviceGuard guard(x.device());
  const Tensor xd = dense(x), wd = dense(wr);
  Tensor logits = empty({T, E}, at::kBFloat16, x);
  check(moe_router_logits(bf(xd), bf(wd), T, H, E, (uint16_t*)logits.data_ptr(), stream_of(x)), "moe_router_few");
  return logits;
}

// -> (out, logits if the router product is inside, routing words if asked for)
std::tuple<Tensor, OptTensor, OptTensor> layer(const Tensor& x, const OptTensor& norm_w, const OptTensor& wr,
                                               const OptTensor& logits, const OptTensor& ids, const Tensor& w1,
                                               const Tensor& w3, const Tensor& w2, const OptTensor& bias,
                                               const OptTensor& s1, const OptTensor& s3, const OptTensor& s2, int64_t k,
                                               double eps, bool add_residual, bool fused_router, bool accumulate,
                                               bool want_routing) {
  const Tensor &n = value(norm_w), &r = value(wr), &l = value(logits), &b = value(bias), &i = value(ids);
  no_tangents({&x, &n, &r, &l, &w1, &w3, &w2, &b});
  Layer o;
  o.k = k, o.eps = eps, o.add_residual = add_residual, o.fused_router = fused_router, o.accumulate = accumulate;
  o.s1 = s1, o.s3 = s3, o.s2 = s2;
  Tensor routing;
  if (want_routing) o.routing_out = &routing;
  if (at::GradMode::is_enabled())
    for (const Tensor* p : {&x, &n, &r, &l, &w1, &w3, &w2, &b}) o.train = o.train || (p->defined() && p->requires_grad());
  Tensor out, lg;
  if (o.train) {
    const variable_list v = LayerNode::apply(x, norm_w, wr, logits, w1, w3, w2, bias, ids, o);
    out = v[0];
    if (v.size() > 1) lg = v[1];
  } else {
    const at::NoGradGuard off;
    const Outputs f = forward(o, x, n, r, l, w1, w3, w2, b, i);
    out = f.out;
    if (r.defined()) lg = f.logits;
  }
  return {out, lg.defined() ? OptTensor(lg) : std::nullopt, want_routing ? OptTensor(routing) : std::nullopt};
}


// ---- the layer in fp32 (model/modules/mlp.py:101-167 with fp32 operands and no autocast) --------------

// Kept for the backward pass: xp [R,H], g, u, act [R,I], y [R,H] (y with logits only: the gate gradient
// reads it), all fp32.
struct KeptF32 {
  int64_t g, u, act, y, total;
  KeptF32(int64_t R, int64_t H, int64_t I) {
    const int64_t rh = up(R * H, 64), ri = up(R * I, 64);
    g = rh, u = g + ri, act = u + ri, y = act + ri, total = y + rh;
    if (total == 0) total = 64;
  }
};

struct OutputsF32 {
  Tensor out, routing, kept, w[3];
};

OutputsF32 forward_f32(const Layer& o, const Tensor& x_, const Tensor& logits_, const Tensor& w1, const Tensor& w3,
                       const Tensor& w2, const Tensor& bias, const Tensor& ids_) {
  OutputsF32 f;
  need_gpu(x_);
  TORCH_CHECK(x_.dim() == 2 && w1.dim() == 3, "the layer takes x [tokens, hidden] and weights [experts, ., .]");
  const int64_t T = x_.size(0), H = x_.size(1), E = w1.size(0), I = w1.size(1), k = o.k, R = T * k;
  TORCH_CHECK(w3.size(0) == E && w2.size(0) == E && w1.size(2) == H && w3.size(2) == H && w3.size(1) == I &&
                  w2.size(1) == H && w2.size(2) == I,
              "the weights' shapes do not belong together");
  check_logits(logits_, bias, x_, E);
  const c10::DeviceGuard guard(x_.device());
  const Tensor x = dense(x_);
  f.w[0] = dense(w1), f.w[1] = dense(w3), f.w[2] = dense(w2);
  void* s = stream_of(x);
  const Routing r(R, E);
  f.routing = empty({r.at[Routing::PARTS]}, at::kInt, x);
  f.out = empty({T, H}, at::kFloat, x);
  const KeptF32 kept(R, H, I);
  f.kept = empty({kept.total}, at::kFloat, x);
  float* base = f.kept.data_ptr<float>();
  float *xp = base, *g = base + kept.g, *u = base + kept.u, *act = base + kept.act, *y = base + kept.y;
  float* gates = nullptr;
  const bool place = logits_.defined() && H % 8 == 0 && moe_place_ok(T, E, k);
  const int64_t wsb = std::max<int64_t>(place ? moe_place_bytes(T, E) : moe_dispatch_workspace_bytes(R, E), 16);
  const Tensor ws = empty({wsb}, at::kByte, x);
  int32_t* counts = r.part(f.routing, Routing::COUNTS);
  int32_t* offs = r.part(f.routing, Routing::OFFS);
  int32_t* p2r = r.part(f.routing, Routing::POS_TO_ROW);
  int32_t* r2p = r.part(f.routing, Routing::ROW_TO_POS);
  int32_t* ids = r.part(f.routing, Routing::IDS);
  Tensor logits, b;
  if (logits_.defined()) {
    logits = dense(logits_);
    if (bias.defined()) b = dense(bias);
    gates = (float*)r.part(f.routing, Routing::GATES);
  }
  if (place && moe_select_place_ok(logits.data_ptr(), T, E, k)) {
    CALL(moe_select_place, x.data_ptr<float>(), MOE_DT_F32, logits.data_ptr(), (int)dt(logits), (const float*)ptr(b), T, H, E, k, ids,
         gates, counts, offs, p2r, r2p, nullptr, xp, MOE_DT_F32, s);
  } else if (place) {
    CALL(moe_select_count, logits.data_ptr(), (int)dt(logits), (const float*)ptr(b), T, E, k, ids, gates, ws.data_ptr(), s);
    CALL(moe_place_rows, x.data_ptr<float>(), MOE_DT_F32, ids, ws.data_ptr(), T, H, E, k, counts, offs, p2r, r2p,
         nullptr, xp, MOE_DT_F32, false, s);
  } else {
    int32_t* bad = nullptr;
    Tensor given;
    const int32_t* sorted = ids;
    if (logits.defined()) {
      CALL(moe_router_topk_fwd, logits.data_ptr(), (int)dt(logits), (const float*)ptr(b), T, E, k, ids, gates, s);
    } else {
      given = dense(ids_.to(at::kInt));
      TORCH_CHECK(given.numel() == R, "one expert id per row is needed");
      sorted = given.data_ptr<int32_t>();
      bad = r.part(f.routing, Routing::BAD);
    }
    CALL(moe_histogram_scan_checked, sorted, R, E, counts, offs, p2r, r2p, bad, ws.data_ptr(), wsb, s);
    CALL(moe_f32_gather_rows, x.data_ptr<float>(), p2r, T, R, H, k, xp, s);
  }
  CALL(moe_f32_gateup, xp, f.w[0].data_ptr<float>(), f.w[1].data_ptr<float>(), offs, E, R, H, I,
       o.train ? g : nullptr, o.train ? u : nullptr, act, s);
  CALL(moe_f32_gemm_rows, act, f.w[2].data_ptr<float>(), offs, E, R, H, I, 1, y, 0, s);
  CALL(moe_f32_combine_fwd, y, gates, r2p, T, H, k, f.out.data_ptr<float>(), s);
  if (o.routing_out) *o.routing_out = f.routing;
  return f;
}

// Whether anything but the router's input and weight is there to see or to change the gradient that comes to `logits`, the
// product of the two: a hook on it or on one of the nodes from it to the product, or a gradient asked for right there.
bool logits_observed(torch::autograd::Node* node) {
  const auto* info = torch::autograd::get_current_graph_task_exec_info();
  for (; node; node = node->num_outputs() ? node->next_edge(0).function.get() : nullptr) {
    if (!node->tensor_pre_hooks().empty() || !node->retains_grad_hooks().empty() || !node->pre_hooks().empty() ||
        !node->post_hooks().empty())
      return true;
    if (info) {
      const auto at = info->find(node);
      if (at != info->end() && at->second.captures_) return true;
    }
    if (node->num_outputs() == 2) return false;  // the product
  }
  return true;
}

// The logits of the layer's own product, whose leading dimensions are x's, as a matrix; those that a caller brings as they are.
Tensor flat(const Tensor& logits, const Tensor& wr) { return wr.defined() && logits.dim() != 2 ? logits.flatten(0, -2) : logits; }

// Given the router weight too, `logits` are the fp32 product of x with it, made by the library in a graph of its own: the
// layer hands their gradient on to it only where somebody observes it, and else works out what it comes to in x and in the
// weight along with its own.
struct LayerF32Node : torch::autograd::Function<LayerF32Node> {
  enum Input { X, WR, LOGITS, W1, W3, W2, BIAS, IDS, OPTIONS, INPUTS };

  static variable_list forward(AutogradContext* ctx, const Tensor& x, const OptTensor& wr_, const OptTensor& logits_,
                               const Tensor& w1, const Tensor& w3, const Tensor& w2, const OptTensor& bias_,
                               const OptTensor& ids_, const Layer& o) {
    const Tensor &wr = value(wr_), &logits = value(logits_), &bias = value(bias_), &ids = value(ids_);
    const OutputsF32 f = forward_f32(o, x, flat(logits, wr), w1, w3, w2, bias, ids);
    ctx->save_for_backward({f.kept, f.routing, f.w[0], f.w[1], f.w[2], wr});
    ctx->saved_data["i"] = std::vector<int64_t>{x.size(0), o.k, logits.defined(),
                                                Present{true, wr.defined(), logits.defined(), true, true, true,
                                                        bias.defined(), ids.defined()}.mask};
    ctx->saved_data["shape"] = logits.defined() ? logits.sizes().vec() : std::vector<int64_t>();
    ctx->set_materialize_grads(false);
    return {f.out};
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    first_order_only();
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &kept_buf = saved[0], &routing = saved[1], &w1 = saved[2], &w3 = saved[3], &w2 = saved[4], &wr = saved[5];
    const std::vector<int64_t> ints = ctx->saved_data["i"].toIntVector();
    const int64_t T = ints[0], k = ints[1], R = T * k, E = w1.size(0), I = w1.size(1), H = w1.size(2);
    const bool routed = ints[2];
    const c10::DeviceGuard guard(kept_buf.device());
    Present present;
    present.mask = ints[3];
    const auto need = [&](Input i) { return present.wants_gradient(ctx, i); };
    const auto node = torch::autograd::get_current_node();
    const bool inside = wr.defined() && need(LOGITS) && node && !logits_observed(present.next(*node, LOGITS));
    const bool by_hand = (need(LOGITS) && !inside) || need(BIAS);
    const bool want_gates = routed && (by_hand || inside);
    const Tensor dout = grads[0].defined() ? dense(grads[0].to(at::kFloat)) : at::zeros({T, H}, kept_buf.options());
    const Routing r(R, E);
    const KeptF32 kept(R, H, I);
    const float* base = kept_buf.data_ptr<float>();
    const float *xp = base, *g = base + kept.g, *u = base + kept.u, *act = base + kept.act, *y = base + kept.y;
    const float* gates = routed ? (const float*)r.part(routing, Routing::GATES) : nullptr;
    const int32_t* offs = r.part(routing, Routing::OFFS);
    const int32_t* p2r = r.part(routing, Routing::POS_TO_ROW);
    const int32_t* r2p = r.part(routing, Routing::ROW_TO_POS);
    void* s = stream_of(kept_buf);
    const int64_t rh = up(R * H, 64), ri = up(R * I, 64);
    const int64_t partial = inside && need(WR) ? moe_f32_router_wgrad_floats(R, H, E) : 0;
    const Tensor scratch = empty({2 * rh + 2 * ri + 2 * up(R, 64) + partial + 64}, at::kFloat, kept_buf);
    float* dyp = scratch.data_ptr<float>();
    float *dxp = dyp + rh, *dg = dxp + rh, *du = dg + ri, *dgates = du + ri, *dsel = dgates + up(R, 64), *part = dsel + up(R, 64);
    CALL(moe_f32_combine_bwd, dout.data_ptr<float>(), want_gates ? y : nullptr, gates, p2r, T, R, H, k, dyp,
         want_gates ? dgates : nullptr, s);
    CALL(moe_f32_gemm_down_swiglu_bwd, dyp, w2.data_ptr<float>(), g, u, offs, E, R, H, I, dg, du, s);
    Tensor dx, dwr, dw1, dw3, dw2, dlogits, dbias;
    const int32_t* ids = r.part(routing, Routing::IDS);
    if (need(X)) {
      dx = empty({T, H}, at::kFloat, kept_buf);
      CALL(moe_f32_gemm_gateup_bwd, dg, du, w1.data_ptr<float>(), w3.data_ptr<float>(), offs, E, R, H, I, dxp, s);
    }
    if (inside) {
      const Tensor wrd = dense(wr);
      CALL(moe_f32_permute_bwd_router, dxp, r2p, gates, dgates, ids, wrd.data_ptr<float>(), T, H, k, dsel, (float*)ptr(dx), s);
      if (need(WR)) {
        dwr = empty({E, H}, at::kFloat, kept_buf);
        CALL(moe_f32_router_wgrad, xp, dsel, offs, R, H, E, part, dwr.data_ptr<float>(), s);
      }
    } else if (need(X)) {
      CALL(moe_f32_permute_bwd, dxp, r2p, T, H, k, dx.data_ptr<float>(), s);
    }
    if (need(W1)) dw1 = empty({E, I, H}, at::kFloat, kept_buf);
    if (need(W3)) dw3 = empty({E, I, H}, at::kFloat, kept_buf);
    if (need(W2)) dw2 = empty({E, H, I}, at::kFloat, kept_buf);
    CALL(moe_f32_wgrads, dg, du, dyp, xp, act, offs, E, R, H, I, (float*)ptr(dw1), (float*)ptr(dw3),
         (float*)ptr(dw2), s);
    if (by_hand) {
      dlogits = empty({T, E}, at::kFloat, kept_buf);
      CALL(moe_router_topk_bwd, gates, dgates, ids, T, E, k, dlogits.data_ptr(), MOE_DT_F32, s);
      if (need(BIAS)) dbias = dlogits.sum(0);
      dlogits = need(LOGITS) ? dlogits.view(ctx->saved_data["shape"].toIntVector()) : Tensor();
    }
    variable_list out(INPUTS);
    out[X] = dx, out[WR] = dwr, out[LOGITS] = dlogits, out[W1] = dw1, out[W3] = dw3, out[W2] = dw2, out[BIAS] = dbias;
    return out;
  }
};

// -> (out [tokens, hidden], logits if the router weight is given, routing words if asked for); x: any number of leading
// dimensions with a router weight, whose logits have them too.
std::tuple<Tensor, OptTensor, OptTensor> layer_f32(const Tensor& x_, const OptTensor& wr, const OptTensor& logits,
                                                   const OptTensor& ids, const Tensor& w1, const Tensor& w3, const Tensor& w2,
                                                   const OptTensor& bias, int64_t k, bool want_routing) {
  const Tensor &r = value(wr), &b = value(bias), &i = value(ids);
  Tensor x = x_, l = value(logits);
  no_tangents({&x, &r, &l, &w1, &w3, &w2, &b});
  Layer o;
  o.k = k;
  Tensor routing;
  if (want_routing) o.routing_out = &routing;
  if (r.defined()) {
    need_gpu(x);
    need_gpu(r);
    TORCH_CHECK(x.dim() >= 2 && w1.dim() == 3 && r.dim() == 2 && r.size(0) == w1.size(0) && r.size(1) == x.size(-1),
                "the router weight has shape ", r.sizes(), ", x ", x.sizes(), " and the experts' ", w1.sizes());
    TORCH_CHECK(r.device() == x.device(), "the router weight is on ", r.device(), ", x on ", x.device());
    TORCH_CHECK_TYPE(r.scalar_type() == at::kFloat && x.scalar_type() == at::kFloat, "x and the router weight must be fp32");
    const NoAutocast off;
    l = at::linear(x, r);
    if (x.dim() != 2) x = x.flatten(0, -2);
  }
  if (at::GradMode::is_enabled())
    for (const Tensor* p : std::initializer_list<const Tensor*>{&x, &r, &l, &w1, &w3, &w2, &b}) o.train = o.train || (p->defined() && p->requires_grad());
  Tensor out;
  if (o.train) {
    out = LayerF32Node::apply(x, wr, l.defined() ? OptTensor(l) : std::nullopt, w1, w3, w2, bias, ids, o)[0];
  } else {
    const at::NoGradGuard off;
    out = forward_f32(o, x, flat(l, r), w1, w3, w2, b, i).out;
  }
  return {out, r.defined() ? OptTensor(l) : std::nullopt, want_routing ? OptTensor(routing) : std::nullopt};
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("set_error_type", [](py::object t) { error_type = t.release().ptr(); });  // (as long as the process)
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (torch::PyTorchError& e) {
      PyErr_SetString(e.python_type(), e.what());
    }
  });
  m.def("layer", &layer, py::call_guard<py::gil_scoped_release>());
  m.def("router_logits", &router_logits, py::call_guard<py::gil_scoped_release>());
  m.def("router_wgrad",
        [](const Tensor& dlogits, const Tensor& xn, py::object type) {
          const at::ScalarType t = torch::python::detail::py_object_to_dtype(type);
          const py::gil_scoped_release off;
          return router_wgrad(dlogits, xn, t);
        });
  m.def("layer_f32", &layer_f32, py::call_guard<py::gil_scoped_release>());
}
