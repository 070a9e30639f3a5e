// PyTorch binding of the eager operators: one call from Python per forward, and a backward that runs
// without Python at all.
//
// What a call of a few workgroups costs is host work, not device work.  Measured on `sb_attn` of
// 1 x 4 heads x 512 tokens x d = 64, forward + backward: 205 us per step with the autograd function and
// the launchers in Python (ctypes), 55 us of it on the GPU; the backward alone took 150 us of host time
// because its Python ran on the autograd thread and handed the interpreter lock back and forth with
// the caller's.  Here the autograd node is C++, calls the C ABI of include/sba.h directly and
// holds no interpreter lock.
//
// Upstream counterpart: the autograd functions of stickbreaking_attention/sb_varlen/__init__.py:24-68
// and sb_attn/__init__.py:16-54 with their launchers.  Tracing, graph capture and the table-rebuilding
// backward stay in Python (_ops.py), which decides what comes here.
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_cpp_function.h>

#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <utility>

#include "sba.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

constexpr int64_t kWorkWords = 64;   // counter words at the end of every carry table (see sba_table_bytes)

// Everything of a call that is not q, k, v.
struct Call {
  Tensor cu, sched;          // cu_seqlens without the leading zero (undefined: fixed length); schedule workspace
  bool build;                // the schedule still has to be written
  int64_t table_floats;      // size of one carry table
  int64_t max_doc_len;
  double inv_temp;
  uint32_t flags;
  bool fixed;
  bool need_table;           // a backward will follow
};

void check(int code, const char* what) {
  if (code == 0) return;
  const char* msg = sba_error_string(code);
  if (code < 0) TORCH_CHECK_VALUE(false, what, ": ", msg, " (SBA error ", code, ")");
  TORCH_CHECK(false, what, ": HIP error ", code, ": ", msg);
}

void* current_stream(const Tensor& t) {
  return reinterpret_cast<void*>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}

bool capturing(void* stream) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(reinterpret_cast<hipStream_t>(stream), &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

sba_view view(const Tensor& t, bool fixed) {
  sba_view v{nullptr, 0, 0, 0};
  if (!t.defined() || t.numel() == 0) return v;
  v.ptr = t.data_ptr();
  const auto s = t.strides();
  if (fixed) v.stride_b = s[0];
  v.stride_h = s[fixed ? 1 : 0];
  v.stride_t = s[fixed ? 2 : 1];
  return v;
}

sba_problem problem(const Tensor& q, const Call& c) {
  sba_problem p{};
  const auto z = q.sizes();
  p.dtype = q.scalar_type() == at::kHalf ? SBA_F16 : SBA_BF16;
  p.head_dim = (int32_t)z.back();
  p.heads = (int32_t)z[c.fixed ? 1 : 0];
  p.batch = c.fixed ? (int32_t)z[0] : 1;
  p.tokens = (int32_t)z[c.fixed ? 2 : 1];
  p.n_docs = c.fixed ? 0 : (int32_t)c.cu.numel();
  p.max_doc_len = (int32_t)(c.fixed ? p.tokens : c.max_doc_len);
  p.flags = c.flags | (c.fixed ? SBA_FIXED_LENGTH : 0u);
  p.inv_temp = (float)c.inv_temp;
  p.cu_seqlens = c.fixed || c.cu.numel() == 0 ? nullptr : c.cu.data_ptr();
  return p;
}

// Element type `dt`, head_dim padded with zeros to `dpad` (the next multiple of 8), unit inner stride, other strides multiples of
// 8 elements, 16-byte aligned rows.
Tensor prepared(Tensor t, int64_t dpad, at::ScalarType dt) {
  if (t.scalar_type() != dt) t = t.to(dt);
  const int64_t d = t.size(-1);
  if (d != dpad) t = at::constant_pad_nd(t, {0, dpad - d}, 0);
  bool ok = t.stride(-1) == 1;
  for (int64_t i = 0; i + 1 < t.dim(); ++i) ok = ok && t.stride(i) % 8 == 0;
  if (!ok) t = t.contiguous();
  if (reinterpret_cast<uintptr_t>(t.data_ptr()) % 16) t = t.clone(at::MemoryFormat::Contiguous);
  return t;
}

int64_t padded_dim(int64_t d) {
  TORCH_CHECK_VALUE(d <= 256, "head_dim ", d, " is not supported (maximum 256)");
  return (d + 7) & ~int64_t(7);   // (rows of 16-byte chunks; the kernels take every multiple of 8)
}

at::ScalarType compute_type(at::ScalarType t) { return t == at::kHalf ? at::kHalf : at::kBFloat16; }

Tensor as_caller(const Tensor& t, int64_t d, at::ScalarType dt) {
  Tensor r = t.size(-1) == d ? t : t.narrow(-1, 0, d);
  return r.scalar_type() == dt ? r : r.to(dt);
}

// Tensors of a float32 caller that need nothing but rounding (dense, head_dim and addresses fit the kernels): all of them
// in one launch of sba_round_floats.  False: nothing was done, every tensor goes its own way.
bool rounded(std::initializer_list<const Tensor*> from, std::initializer_list<Tensor*> to, int64_t d, at::ScalarType ct, void* stream) {
  if (d % 8) return false;
  for (const Tensor* t : from) {
    bool ok = t->scalar_type() == at::kFloat && t->is_non_overlapping_and_dense() && reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0 && t->stride(-1) == 1;
    for (int64_t i = 0; i + 1 < t->dim(); ++i) ok = ok && t->stride(i) % 8 == 0;
    if (!ok) return false;
  }
  const void* src[3];
  void* dst[3];
  int64_t counts[3];
  int n = 0;
  auto out = to.begin();
  for (const Tensor* t : from) {
    **out = at::empty_like(*t, t->options().dtype(ct));
    src[n] = t->data_ptr();
    dst[n] = (*out)->data_ptr();
    counts[n++] = t->numel();
    ++out;
  }
  check(sba_round_floats(ct == at::kHalf ? SBA_F16 : SBA_BF16, n, src, dst, counts, stream), "sba_round_floats");
  return true;
}

// float32 outputs straight from the kernels: where no column has to be cut off and 32-bit offsets reach every row.
bool writes_f32(const Tensor& like, int64_t d, bool fixed) {
  return like.size(-1) == d && (like.size(fixed ? 2 : 1) + 1024) * like.stride(fixed ? 2 : 1) * 4 < (int64_t(1) << 31);
}

// The scratch of a backward (gradient table, or the one-pass form's; not p and dz of head_dim 129 .. 256): one grow-only buffer per (device, stream), shared by every layer (the dk/dv pass
// of one backward has read it before the next backward on that stream writes it).  Packed documents change
// the size with every batch; growth goes to the next eighth of a power of two, and by at least a quarter.
// The lock is held while a backward's kernels are enqueued: two threads on one stream must not interleave theirs.
struct GradTables {
  std::mutex mutex;
  std::map<std::pair<int, void*>, Tensor> tables;
  static int64_t size_class(int64_t n) {
    if (n <= 1 << 16) return 1 << 16;
    int bits = 64 - __builtin_clzll((unsigned long long)n);
    const int64_t step = int64_t(1) << (bits > 4 ? bits - 4 : 0);
    return (n + step - 1) / step * step;
  }
  Tensor get(int64_t n, const Tensor& like, void* stream) {   // (mutex held)
    Tensor& t = tables[{(int)like.device().index(), stream}];
    if (!t.defined() || t.numel() < n) {
      const int64_t grown = t.defined() ? t.numel() * 5 / 4 : 0;
      t = Tensor();            // back to the allocator before the larger one is asked for
      t = at::empty({size_class(std::max(n, grown))}, like.options().dtype(at::kFloat));
    }
    return t;
  }
};
GradTables& grad_tables() {
  static GradTables* g = new GradTables;   // (never destroyed: its tensors must not outlive the allocator at exit)
  return *g;
}

struct Attention : public torch::autograd::Function<Attention> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Call& c) {
    ctx->set_materialize_grads(false);   // a gradient nobody asked for arrives undefined, not as zeros
    const c10::DeviceGuard guard(q.device());
    const int64_t d = q.size(-1), dpad = padded_dim(d);
    const at::ScalarType dt = q.scalar_type(), ct = compute_type(dt);
    void* const stream = current_stream(q);
    Tensor qp, kp, vp;
    if (dt != at::kFloat || !rounded({&q, &k, &v}, {&qp, &kp, &vp}, d, ct, stream)) {
      qp = prepared(q, dpad, ct);
      kp = prepared(k, dpad, ct);
      vp = prepared(v, dpad, ct);
    }
    const bool f32 = dt == at::kFloat && writes_f32(qp, d, c.fixed);
    const auto out = qp.options().dtype(f32 ? at::kFloat : ct);
    Tensor o = at::empty_like(qp, out), rem = at::empty_like(qp.select(-1, 0), out);
    const Tensor table = c.need_table ? at::empty({c.table_floats}, qp.options().dtype(at::kFloat)) : Tensor();
    sba_problem p = problem(qp, c);
    if (f32) p.flags |= SBA_F32_OUT;
    void* const sched = c.sched.data_ptr();
    const size_t sched_bytes = (size_t)c.sched.numel();
    if (c.build) check(sba_build_schedule(&p, sched, sched_bytes, stream), "sba_build_schedule");
    const sba_view vq = view(qp, c.fixed), vk = view(kp, c.fixed), vv = view(vp, c.fixed), vo = view(o, c.fixed), vr = view(rem, c.fixed);
    check((c.fixed ? sba_attn_fwd : sba_varlen_fwd)(&p, sched, sched_bytes, &vq, &vk, &vv, &vo, &vr,
                                                    c.need_table ? table.data_ptr<float>() : nullptr,
                                                    c.need_table ? (size_t)c.table_floats * 4 : 0, stream),
          c.fixed ? "sba_attn_fwd" : "sba_varlen_fwd");
    if (c.need_table) {
      ctx->save_for_backward({qp, kp, vp, table, c.sched, c.cu});
      ctx->saved_data["d"] = d;
      ctx->saved_data["max_doc_len"] = c.max_doc_len;
      ctx->saved_data["inv_temp"] = c.inv_temp;
      ctx->saved_data["flags"] = (int64_t)c.flags;
      ctx->saved_data["fixed"] = c.fixed;
      ctx->saved_data["types"] = ((int64_t)q.scalar_type() << 16) | ((int64_t)k.scalar_type() << 8) | (int64_t)v.scalar_type();
    }
    o = as_caller(o, d, dt);
    if (rem.scalar_type() != dt) rem = rem.to(dt);
    if (c.flags & SBA_FUSE_REMAINDER) return {o};
    return {o, rem};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &qp = saved[0], &kp = saved[1], &vp = saved[2], &table = saved[3];
    const c10::DeviceGuard guard(qp.device());
    Call c;
    c.sched = saved[4];
    c.cu = saved[5];
    c.max_doc_len = ctx->saved_data["max_doc_len"].toInt();
    c.inv_temp = ctx->saved_data["inv_temp"].toDouble();
    c.flags = (uint32_t)ctx->saved_data["flags"].toInt();
    c.fixed = ctx->saved_data["fixed"].toBool();
    const int64_t d = ctx->saved_data["d"].toInt(), types = ctx->saved_data["types"].toInt(), dpad = qp.size(-1);
    const at::ScalarType ct = qp.scalar_type();
    void* const stream = current_stream(qp);
    Tensor go;
    if (!grads[0].defined()) go = at::zeros_like(qp);   // (only rem was used)
    else if (!rounded({&grads[0]}, {&go}, dpad, ct, stream)) go = prepared(grads[0], dpad, ct);
    Tensor gr = grads.size() > 1 ? grads[1] : Tensor();
    if (gr.defined() && gr.scalar_type() != ct) gr = gr.to(ct);
    constexpr int64_t kAllFloat = ((int64_t)at::kFloat << 16) | ((int64_t)at::kFloat << 8) | (int64_t)at::kFloat;
    const bool f32 = types == kAllFloat && writes_f32(qp, d, c.fixed) && writes_f32(kp, d, c.fixed) && writes_f32(vp, d, c.fixed);
    const auto out = qp.options().dtype(f32 ? at::kFloat : ct);
    Tensor dq = at::empty_like(qp, out), dk = at::empty_like(kp, out), dv = at::empty_like(vp, out);
    sba_problem p = problem(qp, c);
    if (f32) p.flags |= SBA_F32_OUT;
    const sba_view vq = view(qp, c.fixed), vk = view(kp, c.fixed), vv = view(vp, c.fixed), vg = view(go, c.fixed), vr = view(gr, c.fixed);
    const sba_view wq = view(dq, c.fixed), wk = view(dk, c.fixed), wv = view(dv, c.fixed);
    size_t chain_bytes = sba_bwd_scratch_bytes(&p, (size_t)table.numel() * 4);   // 0: the two-pass form
    // p and dz of head_dim 129 .. 256 are 32 times a gradient table, up to 3.75 GiB: they are asked for and given back by every call, so that
    // between two of them the memory is the allocator's for anything else, and where it is not to be had the scores are formed twice.
    Tensor handed_on;
    if (chain_bytes && p.head_dim > 128) {
      try {
        handed_on = at::empty({(int64_t)(chain_bytes / 4)}, table.options());
      } catch (const c10::OutOfMemoryError&) {
        chain_bytes = 0;
      }
    }
    const int64_t scratch_floats = chain_bytes ? (int64_t)(chain_bytes / 4) : table.numel();
    auto launch = [&](const Tensor& scratch) {
      if (chain_bytes) {
        check((c.fixed ? sba_attn_bwd_chained : sba_varlen_bwd_chained)(&p, c.sched.data_ptr(), (size_t)c.sched.numel(), &vq, &vk, &vv, &vg, &vr,
                                                                        table.data_ptr<float>(), (size_t)table.numel() * 4,
                                                                        scratch.data_ptr(), chain_bytes, &wq, &wk, &wv, stream),
              c.fixed ? "sba_attn_bwd_chained" : "sba_varlen_bwd_chained");
        return;
      }
      check((c.fixed ? sba_attn_bwd : sba_varlen_bwd)(&p, c.sched.data_ptr(), (size_t)c.sched.numel(), &vq, &vk, &vv, &vg, &vr,
                                                      table.data_ptr<float>(), scratch.data_ptr<float>(), (size_t)table.numel() * 4,
                                                      &wq, &wk, &wv, stream),
            c.fixed ? "sba_attn_bwd" : "sba_varlen_bwd");
    };
    if (handed_on.defined()) {
      launch(handed_on);
    } else if (capturing(stream)) {   // a graph's replays must not depend on a buffer that may be replaced
      launch(at::empty({scratch_floats}, table.options()));
    } else {
      GradTables& g = grad_tables();
      const std::lock_guard<std::mutex> lock(g.mutex);
      launch(g.get(scratch_floats, table, stream));
    }
    return {as_caller(dq, d, (at::ScalarType)(types >> 16)), as_caller(dk, d, (at::ScalarType)((types >> 8) & 255)),
            as_caller(dv, d, (at::ScalarType)(types & 255)), Tensor()};
  }
};

// (o, rem), or (o,) with SBA_FUSE_REMAINDER.
std::vector<Tensor> attention(const Tensor& q, const Tensor& k, const Tensor& v, const std::optional<Tensor>& cu, const Tensor& sched,
                              bool build, int64_t table_floats, int64_t max_doc_len, double inv_temp, int64_t flags) {
  Call c;
  c.fixed = !cu.has_value();
  if (!c.fixed) {
    c.cu = cu->contiguous();
    if (c.cu.scalar_type() == at::kLong) flags |= SBA_CU_INT64;
  }
  TORCH_CHECK_VALUE(q.dim() == (c.fixed ? 4 : 3), "expected a ", c.fixed ? 4 : 3, "-d tensor, got shape ", q.sizes());
  TORCH_CHECK_VALUE(k.sizes() == q.sizes() && v.sizes() == q.sizes(), "q, k and v differ in shape: ", q.sizes(), ", ", k.sizes(), ", ", v.sizes());
  TORCH_CHECK(k.is_cuda() && v.is_cuda() && k.device() == q.device() && v.device() == q.device(), "q, k and v are on different devices");
  c.sched = sched;
  c.build = build;
  c.table_floats = table_floats;
  c.max_doc_len = max_doc_len;
  c.inv_temp = inv_temp;
  c.flags = (uint32_t)flags;
  c.need_table = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
  return Attention::apply(q, k, v, c);
}

void release() {
  std::map<std::pair<int, void*>, Tensor> old;
  {
    GradTables& g = grad_tables();
    const std::lock_guard<std::mutex> lock(g.mutex);
    old.swap(g.tables);
  }
}

// `grad_fn.saved_tensors`, as a Python autograd function has it: what the forward keeps for the backward.
PyObject* saved_tensors(PyObject* self, void*) {
  HANDLE_TH_ERRORS
  auto* node = reinterpret_cast<torch::autograd::THPCppFunction*>(self)->cdata.get();
  py::list out;
  for (const Tensor& t : static_cast<torch::autograd::CppNode<Attention>*>(node)->ctx_.get_saved_variables())
    if (t.defined()) out.append(t);
  return py::tuple(out).release().ptr();
  END_HANDLE_TH_ERRORS
}

void register_grad_fn_type() {
  using namespace torch::autograd;
  static PyGetSetDef properties[] = {THP_FUNCTION_DEFAULT_PROPERTIES,
                                     {(char*)"saved_tensors", saved_tensors, nullptr, nullptr, nullptr},
                                     {nullptr, nullptr, nullptr, nullptr, nullptr}};
  static PyTypeObject type;
  registerCppFunction(typeid(CppNode<Attention>), _initFunctionPyTypeObject(type, "StickBreakingAttentionBackward", properties, nullptr));
}

}  // namespace

PYBIND11_MODULE(_sba_torch, m) {
  m.doc() = "Eager stick-breaking attention operators on libsba.so";
  register_grad_fn_type();
  m.def("attention", &attention, py::call_guard<py::gil_scoped_release>());
  m.def("release", &release, py::call_guard<py::gil_scoped_release>());
  m.def("version", &sba_version);
}
