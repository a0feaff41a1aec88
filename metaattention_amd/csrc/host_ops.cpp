// The operators' calls in native code: what stands between a Python call of an operator and its kernel launches.
//
// A call through the Python binding (hip_backend) costs 18 - 29 us of interpreter time (argument checks, some sixty ctypes
// field stores, three allocations, the launch) and a forward + backward pair 160 us, more than the kernels themselves take
// for short prompts and single-token decode; here the same work is a few microseconds, and the backward pass runs on
// autograd's thread without the interpreter.  A plan holds what an operator fixes at construction; a call checks that the
// tensors are the ordinary case, allocates the outputs, fills the C ABI's parameter block and launches.
//
// Anything out of the ordinary (another argument count, views the kernels cannot read in place, another device than the
// current one, an argument set the C ABI refuses) makes a call return None without having launched anything: the caller
// then takes the Python binding, which serves it or raises with the reason.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../include/metaattention_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ------------------------------------------------------------------------------------------------------------- helpers
// A plain tensor of torch's own types (Tensor, Parameter).  Subclasses, functorch's wrappers (whose Python type is Tensor), any
// tensor under a dispatch mode and dual tensors, whose tangents only the binding's autograd functions account for (they refuse
// forward mode), take the Python binding.
inline const Tensor* tensor_of(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  return at::isTensorSubclassLike(t) || t._fw_grad(0).defined() ? nullptr : &t;
}

// torch.jit.trace records the binding's autograd functions, but nothing that happens here (the output would be a constant).
inline bool traced() { return torch::jit::tracer::isTracing(); }

inline bool on(const Tensor& t, int device) { return t.is_cuda() && t.device().index() == device; }

// rows of 16-byte aligned, 16-byte multiples with a contiguous last dimension: what the kernels read in place
inline bool kernel_readable(const Tensor& t) {
  const int n = (int)t.dim();
  if (n == 0 || t.stride(n - 1) != 1 || ((uintptr_t)t.data_ptr() & 15) != 0) return false;
  for (int i = 0; i + 1 < n; i++)
    if (t.stride(i) % 8 != 0) return false;
  return true;
}
inline Tensor kernel_view(const Tensor& t) { return kernel_readable(t) ? t : t.contiguous(); }

inline int dtype_code(const Tensor& t) {
  return t.scalar_type() == at::kBFloat16 ? MA_BF16 : t.scalar_type() == at::kHalf ? MA_FP16 : -1;
}

inline Tensor empty(at::IntArrayRef size, at::ScalarType dt, const c10::Device& dev) {
  return at::detail::empty_cuda(size, dt, dev, std::nullopt);
}

inline c10::DataPtr scratch(size_t bytes) {
  return bytes ? c10::hip::HIPCachingAllocator::get()->allocate(bytes) : c10::DataPtr();
}

// The launches themselves run without the interpreter lock (a launch waits when the device's queue is full).
struct NoGil {
  PyThreadState* s = PyGILState_Check() ? PyEval_SaveThread() : nullptr;
  ~NoGil() {
    if (s) PyEval_RestoreThread(s);
  }
};

inline ma_stream_t stream_of(int device) { return (ma_stream_t)c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

// ------------------------------------------------------------------------------------------- parallel attention, decode
// Dense masks of one shape, as the engine builds them (AttentionEngine._dense_mask): the keep mask and its tile mask, and
// the transposed pair for the backward (undefined until the engine has built it).
struct Masks {
  int64_t B, H, Sq, Skv;
  Tensor elem, blocks, elem_t, blocks_t;
};

struct AttnPlan {
  int family;
  bool causal, masked;      // masked: any other mask_mod, through `masks`
  float scale, bias;
  at::ScalarType dtype;
  std::shared_ptr<const Masks> masks;   // (replaced as a whole, under the interpreter lock)
};

#define MA_SET_TENSOR(P, NAME, PRE, T)       \
  (P).NAME = (decltype((P).NAME))(T).data_ptr(); \
  (P).PRE##_stride_b = (T).stride(0);        \
  (P).PRE##_stride_s = (T).stride(1);        \
  (P).PRE##_stride_h = (T).stride(2)

inline int64_t mask_stride(const Tensor& t, int dim) { return t.size(dim) > 1 ? t.stride(dim) : 0; }

// k [B,Skv,Hkv,Dqk] and v [B,Skv,Hkv,Dv] beside q [B,Sq,H,Dqk], all of them as the kernels take them
bool attn_ordinary(const AttnPlan& pl, const Tensor& q, const Tensor& k, const Tensor& v, int dev) {
  if (!on(q, dev) || !on(k, dev) || !on(v, dev) || q.dim() != 4 || k.dim() != 4 || v.dim() != 4) return false;
  if (q.scalar_type() != pl.dtype || k.scalar_type() != pl.dtype || v.scalar_type() != pl.dtype) return false;
  const int64_t B = q.size(0), H = q.size(2), Skv = k.size(1), Hkv = k.size(2);
  if (k.size(0) != B || k.size(3) != q.size(3) || v.size(0) != B || v.size(1) != Skv || v.size(2) != Hkv) return false;
  if (q.numel() == 0 || k.numel() == 0 || v.numel() == 0 || H % Hkv != 0) return false;
  const int64_t most = std::numeric_limits<int32_t>::max();
  if (B > most || H > most || q.size(1) > most || Skv > most || q.size(3) > most || v.size(3) > most) return false;
  return kernel_readable(q) && kernel_readable(k) && kernel_readable(v);
}

// Forward of the ordinary call.  Returns false (nothing launched) when the library refuses it; `row_scale` stays undefined
// for the families without one.
bool attn_forward(const AttnPlan& pl, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor* mult, bool mult_is_gamma,
                  const Masks* masks, int dev, Tensor& out, Tensor& row_scale) {
  const int64_t B = q.size(0), Sq = q.size(1), H = q.size(2), Hkv = k.size(2), Dv = v.size(3), grp = H / Hkv;
  out = empty({B, Sq, H, Dv}, pl.dtype, q.device());
  const bool has_rs = pl.family == MA_ATTN_SOFTMAX || pl.family == MA_ATTN_RETENTION;
  if (has_rs) row_scale = empty({B, H, Sq}, at::kFloat, q.device());
  ma_attn_params p{};
  p.family = pl.family; p.dtype = dtype_code(q); p.mask = pl.causal ? MA_MASK_CAUSAL : MA_MASK_NONE;
  p.batch = (int)B; p.heads = (int)H; p.seqlen_q = (int)Sq; p.seqlen_kv = (int)k.size(1); p.dim_qk = (int)q.size(3); p.dim_v = (int)Dv;
  p.heads_kv = (int)Hkv;
  MA_SET_TENSOR(p, q, q, q); MA_SET_TENSOR(p, k, k, k); MA_SET_TENSOR(p, v, v, v); MA_SET_TENSOR(p, o, o, out);
  if (Sq == 1 && grp > 1 && !pl.causal && !masks && pl.family != MA_ATTN_RETENTION) {
    // one query token, grouped-query: the query heads of a kv head become the rows of that head (the decode kernels of the
    // reference pack them the same way, attn_gqa_decode_tl.py:81-84); only strides change
    p.heads = (int)Hkv; p.seqlen_q = (int)grp;
    p.q_stride_s = q.stride(2); p.q_stride_h = grp * q.stride(2);
    p.o_stride_s = out.stride(2); p.o_stride_h = grp * out.stride(2);
  }
  p.row_scale = has_rs ? (float*)row_scale.data_ptr() : nullptr;
  p.scale = pl.scale; p.bias = pl.bias;
  if (mult && mult_is_gamma) p.decay_gamma = (const float*)mult->data_ptr();
  if (mult && !mult_is_gamma) {
    p.score_mask = mult->data_ptr();
    p.sm_stride_b = mask_stride(*mult, 0); p.sm_stride_h = mult->stride(1); p.sm_stride_q = mult->stride(2);
  }
  if (masks) {
    p.elem_mask = (const uint8_t*)masks->elem.data_ptr();
    p.em_stride_b = mask_stride(masks->elem, 0); p.em_stride_h = mask_stride(masks->elem, 1); p.em_stride_q = masks->elem.stride(2);
    p.kv_block_mask = (const uint8_t*)masks->blocks.data_ptr(); p.kv_block_size = 32; p.kbm_per_query_head = 1;
    p.kbm_stride_b = mask_stride(masks->blocks, 0); p.kbm_stride_h = mask_stride(masks->blocks, 1); p.kbm_stride_q = masks->blocks.stride(2);
  }
  const size_t need = ma_attn_workspace_bytes(&p);
  const c10::DataPtr ws = scratch(need);
  p.workspace = ws.get(); p.workspace_bytes = need;
  const ma_stream_t st = stream_of(dev);
  NoGil release;
  return ma_attn_fwd(&p, st) == MA_OK;
}

// The softmax, sigmoid and relu operators with gradients.  forward: what has been computed is put on the graph; backward: (dq, dk,
// dv) from what it saved, as _attention.backward (tl_template/attn/attn_tl.py:669-692).  (A torch::autograd::Function, not a
// Node of this file's own: it refuses forward mode and works under compiled autograd.)
struct AttentionFunction : torch::autograd::Function<AttentionFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor* out, const Tensor* row_scale,
                        const AttnPlan* pl, const Masks* masks) {
    // (the output without its history: a saved-tensor hook that raises, as checkpointing's does to stop a recomputation, leaves what
    // was to be saved in the node, and with a history that would be a cycle that keeps the whole graph)
    ctx->save_for_backward({q, k, v, out->tensor_data(), *row_scale});
    auto& d = ctx->saved_data;
    d["plan"] = std::vector<double>{(double)pl->family, pl->causal ? 1. : 0., pl->scale, pl->bias};
    if (masks) {   // (the operator's, not this call's: no business of saved-tensor hooks)
      d["elem"] = masks->elem; d["elem_t"] = masks->elem_t; d["blocks"] = masks->blocks; d["blocks_t"] = masks->blocks_t;
    }
    return *out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &o = saved[3], &rs = saved[4];
    auto& d = ctx->saved_data;
    const std::vector<double> plan = d["plan"].toDoubleVector();
    at::AutoDispatchBelowADInplaceOrView no_autograd;
    const Tensor dout = kernel_view(grads[0]);
    const Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    ma_attn_bwd_params p{};
    p.family = (int)plan[0]; p.dtype = dtype_code(q); p.mask = plan[1] != 0 ? MA_MASK_CAUSAL : MA_MASK_NONE;
    p.batch = (int)q.size(0); p.heads = (int)q.size(2); p.heads_kv = (int)k.size(2); p.seqlen_q = (int)q.size(1); p.seqlen_kv = (int)k.size(1);
    p.dim_qk = (int)q.size(3); p.dim_v = (int)v.size(3);
    MA_SET_TENSOR(p, q, q, q); MA_SET_TENSOR(p, k, k, k); MA_SET_TENSOR(p, v, v, v); MA_SET_TENSOR(p, o, o, o);
    MA_SET_TENSOR(p, dout, do, dout); MA_SET_TENSOR(p, dq, dq, dq); MA_SET_TENSOR(p, dk, dk, dk); MA_SET_TENSOR(p, dv, dv, dv);
    if (rs.defined()) p.lse = (const float*)rs.data_ptr();
    p.scale = (float)plan[2]; p.bias = (float)plan[3];
    if (d.count("elem")) {
      const Tensor elem = d["elem"].toTensor(), elem_t = d["elem_t"].toTensor(), blocks = d["blocks"].toTensor(), blocks_t = d["blocks_t"].toTensor();
      p.elem_mask = (const uint8_t*)elem.data_ptr();
      p.em_stride_b = mask_stride(elem, 0); p.em_stride_h = mask_stride(elem, 1); p.em_stride_q = elem.stride(2);
      p.elem_mask_t = (const uint8_t*)elem_t.data_ptr();
      p.emt_stride_b = mask_stride(elem_t, 0); p.emt_stride_h = mask_stride(elem_t, 1); p.emt_stride_k = elem_t.stride(2);
      p.kv_block_mask = (const uint8_t*)blocks.data_ptr();
      p.kbm_stride_b = mask_stride(blocks, 0); p.kbm_stride_h = mask_stride(blocks, 1); p.kbm_stride_q = blocks.stride(2);
      p.q_block_mask = (const uint8_t*)blocks_t.data_ptr();
      p.qbm_stride_b = mask_stride(blocks_t, 0); p.qbm_stride_h = mask_stride(blocks_t, 1); p.qbm_stride_k = blocks_t.stride(2);
    }
    const size_t need = ma_attn_bwd_workspace_bytes(&p);
    const c10::DataPtr ws = scratch(need);
    p.workspace = ws.get(); p.workspace_bytes = need;
    {
      NoGil release;
      TORCH_CHECK(ma_attn_bwd(&p, stream_of(q.device().index())) == MA_OK, ma_last_error());
    }
    return {dq, dk, dv, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

constexpr const char* kAttnPlan = "metaattention.AttnPlan";

PyObject* none() { Py_RETURN_NONE; }

// attention(q, k, v[, multiplier]) -> (out, row scale or None), or None: see the head of the file.  The multiplier of the
// retention family is its mask tensor [1|B,H,Sq,Skv] or, fp32 [H], the decay of the mask it stands for.
PyObject* attention_call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const AttnPlan& pl = *(const AttnPlan*)PyCapsule_GetPointer(self, kAttnPlan);
  const bool retention = pl.family == MA_ATTN_RETENTION;
  if (n != (retention ? 4 : 3) || traced()) return none();
  const Tensor *qp = tensor_of(args[0]), *kp = tensor_of(args[1]), *vp = tensor_of(args[2]), *mult = retention ? tensor_of(args[3]) : nullptr;
  if (!qp || !kp || !vp || (retention && !mult)) return none();
  const Tensor &q = *qp, &k = *kp, &v = *vp;
  if (!q.is_cuda()) return none();
  const int dev = c10::hip::current_device();
  if (!attn_ordinary(pl, q, k, v, dev)) return none();
  const bool grad = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
  bool gamma = false;
  if (retention) {
    if (grad || !on(*mult, dev)) return none();
    gamma = mult->dim() == 1;
    if (gamma) {
      if (mult->scalar_type() != at::kFloat || mult->size(0) != q.size(2) || mult->stride(0) != 1) return none();
    } else if (mult->dim() != 4 || mult->scalar_type() != pl.dtype || mult->stride(3) != 1 || (mult->size(0) != 1 && mult->size(0) != q.size(0)) ||
               mult->size(1) != q.size(2) || mult->size(2) != q.size(1) || mult->size(3) != k.size(1)) {
      return none();
    }
  }
  std::shared_ptr<const Masks> masks;
  if (pl.masked) {
    masks = pl.masks;
    if (!masks || masks->B != q.size(0) || masks->H != q.size(2) || masks->Sq != q.size(1) || masks->Skv != k.size(1) ||
        !on(masks->elem, dev) || (grad && !masks->elem_t.defined()))
      return none();
  }
  Tensor out, rs;
  if (!attn_forward(pl, q, k, v, mult, gamma, masks.get(), dev, out, rs)) return none();
  if (grad) out = AttentionFunction::apply(q, k, v, &out, &rs, &pl, masks.get());
  PyObject* r = PyTuple_New(2);
  if (!r) return nullptr;
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(out));
  if (rs.defined()) {
    PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(rs));
  } else {
    Py_INCREF(Py_None);
    PyTuple_SET_ITEM(r, 1, Py_None);
  }
  return r;
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------------------ MLA decode
struct MlaPlan {
  float scale;
  at::ScalarType dtype;
};
constexpr const char* kMlaPlan = "metaattention.MlaPlan";

bool mla_launch(ma_mla_params& p, int dev) {
  const size_t need = ma_mla_workspace_bytes(&p);
  const c10::DataPtr ws = scratch(need);
  p.workspace = ws.get(); p.workspace_bytes = need;
  const ma_stream_t st = stream_of(dev);
  NoGil release;
  return ma_mla_decode(&p, st) == MA_OK;
}

// mla(q [B,1,Hq,D], q_pe [B,1,Hq,Dpe], kv [B,Skv,1,D], k_pe [B,Skv,1,Dpe]) -> out [B,1,Hq,D], or None
PyObject* mla_call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const MlaPlan& pl = *(const MlaPlan*)PyCapsule_GetPointer(self, kMlaPlan);
  if (n != 4 || traced()) return none();
  const Tensor* t[4];
  for (int i = 0; i < 4; i++)
    if (!(t[i] = tensor_of(args[i])) || !t[i]->is_cuda()) return none();
  const int dev = c10::hip::current_device();
  for (int i = 0; i < 4; i++)
    if (!on(*t[i], dev) || t[i]->dim() != 4 || t[i]->scalar_type() != pl.dtype || t[i]->numel() == 0 || !kernel_readable(*t[i])) return none();
  const Tensor &q = *t[0], &q_pe = *t[1], &kv = *t[2], &k_pe = *t[3];
  const int64_t B = q.size(0), Hq = q.size(2), D = q.size(3), Skv = kv.size(1), Dpe = q_pe.size(3);
  if (q.size(1) != 1 || q_pe.size(0) != B || q_pe.size(1) != 1 || q_pe.size(2) != Hq || kv.size(0) != B || kv.size(2) != 1 || kv.size(3) != D ||
      k_pe.size(0) != B || k_pe.size(1) != Skv || k_pe.size(2) != 1 || k_pe.size(3) != Dpe || B > 65535 || Hq > (1 << 20) || Skv > (1 << 30))
    return none();
  Tensor out = empty({B, 1, Hq, D}, pl.dtype, q.device());
  ma_mla_params p{};
  p.dtype = dtype_code(q);
  p.batch = (int)B; p.heads_q = (int)Hq; p.seqlen_kv = (int)Skv; p.dim = (int)D; p.dim_pe = (int)Dpe;
  p.q = q.data_ptr(); p.q_stride_b = q.stride(0); p.q_stride_h = q.stride(2);
  p.q_pe = q_pe.data_ptr(); p.qpe_stride_b = q_pe.stride(0); p.qpe_stride_h = q_pe.stride(2);
  p.kv = kv.data_ptr(); p.kv_stride_b = kv.stride(0); p.kv_stride_s = kv.stride(1);
  p.k_pe = k_pe.data_ptr(); p.kpe_stride_b = k_pe.stride(0); p.kpe_stride_s = k_pe.stride(1);
  p.o = out.data_ptr(); p.o_stride_b = out.stride(0); p.o_stride_h = out.stride(2);
  p.scale = pl.scale;
  return mla_launch(p, dev) ? THPVariable_Wrap(out) : none();
  END_HANDLE_TH_ERRORS
}

// mla_paged(q [B,1,Hq,D+Dpe], k_cache [pages, page, 1, D+Dpe], block_table, cache_seqlens, D, scale, metadata | None,
// num_splits | None) -> (out [B,1,Hq,D], lse [B,Hq,1]), or None.  The paged interface of flash_mla_with_kvcache.
PyObject* mla_paged_call(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8 || traced()) return none();
  const Tensor *q = tensor_of(args[0]), *kc = tensor_of(args[1]), *bt = tensor_of(args[2]), *sl = tensor_of(args[3]);
  if (!q || !kc || !bt || !sl || !q->is_cuda()) return none();
  const int dev = c10::hip::current_device();
  const int64_t D = PyLong_AsLongLong(args[4]);
  const double scale = PyFloat_AsDouble(args[5]);
  if (PyErr_Occurred()) return nullptr;
  if (!on(*q, dev) || !on(*kc, dev) || !on(*bt, dev) || !on(*sl, dev)) return none();
  if (q->dim() != 4 || kc->dim() != 4 || bt->dim() != 2 || sl->dim() != 1 || dtype_code(*q) < 0 || kc->scalar_type() != q->scalar_type()) return none();
  const int64_t B = q->size(0), Hq = q->size(2), full = q->size(3), page = kc->size(1), Dpe = full - D;
  if (q->size(1) != 1 || kc->size(2) != 1 || kc->size(3) != full || D <= 0 || Dpe <= 0 || B == 0 || B > 65535 || Hq == 0 || Hq > (1 << 20) || page == 0 ||
      bt->size(1) * page > (1 << 30) || bt->size(1) == 0)
    return none();
  if (!kernel_readable(*q) || !kc->is_contiguous() || bt->scalar_type() != at::kInt || bt->size(0) != B || bt->stride(1) != 1 ||
      sl->scalar_type() != at::kInt || sl->size(0) != B || !sl->is_contiguous())
    return none();
  const Tensor *meta = nullptr, *splits = nullptr;
  if (args[6] != Py_None) {
    meta = tensor_of(args[6]);
    splits = tensor_of(args[7]);
    if (!meta || !splits || !on(*meta, dev) || !on(*splits, dev) || meta->dim() != 2 || meta->size(1) != 8 || meta->size(0) > 65535 ||
        meta->scalar_type() != at::kInt || !meta->is_contiguous() || splits->dim() != 1 || splits->size(0) != B + 1 ||
        splits->scalar_type() != at::kInt || !splits->is_contiguous())
      return none();
  }
  Tensor out = empty({B, 1, Hq, D}, q->scalar_type(), q->device()), lse = empty({B, Hq, 1}, at::kFloat, q->device());
  ma_mla_params p{};
  p.dtype = dtype_code(*q);
  p.batch = (int)B; p.heads_q = (int)Hq; p.seqlen_kv = (int)(bt->size(1) * page); p.dim = (int)D; p.dim_pe = (int)Dpe;
  const int64_t esz = 2;
  p.q = q->data_ptr(); p.q_stride_b = q->stride(0); p.q_stride_h = q->stride(2);
  p.q_pe = (const char*)q->data_ptr() + D * esz; p.qpe_stride_b = q->stride(0); p.qpe_stride_h = q->stride(2);
  p.kv = kc->data_ptr(); p.kv_stride_s = full;
  p.k_pe = (const char*)kc->data_ptr() + D * esz; p.kpe_stride_s = full;
  p.o = out.data_ptr(); p.o_stride_b = out.stride(0); p.o_stride_h = out.stride(2);
  p.lse = (float*)lse.data_ptr();
  p.scale = (float)scale;
  p.kv_seqlens = (const int32_t*)sl->data_ptr();
  p.block_table = (const int32_t*)bt->data_ptr(); p.block_table_stride = bt->stride(0); p.page_size = (int)page;
  if (meta) {
    p.tile_scheduler_metadata = (const int32_t*)meta->data_ptr(); p.num_splits = (const int32_t*)splits->data_ptr();
    p.num_sm_parts = (int)meta->size(0);
  }
  if (!mla_launch(p, dev)) return none();
  PyObject* r = PyTuple_New(2);
  if (!r) return nullptr;
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(out));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(lse));
  return r;
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------ chunked linear attention
enum DecayKind { DECAY_AS_IS = 0, DECAY_LOG = 1, DECAY_MUL_HEAD = 2 };
struct LinearPlan {
  int decay_kind;
  int decay_head_arg, v_scale_arg;   // which custom tensor multiplies the decay / the values (-1: none)
  int n_custom;
  float q_scale;
};
constexpr const char* kLinearPlan = "metaattention.LinearPlan";

void linear_sizes(const Tensor& q, const Tensor& k, const Tensor& v, int32_t& B, int32_t& H, int32_t& Hq, int32_t& Hk, int32_t& T, int32_t& Dk, int32_t& Dv) {
  B = (int)v.size(0); H = (int)v.size(1); Hq = (int)q.size(1); Hk = (int)k.size(1); T = (int)v.size(2); Dk = (int)q.size(3); Dv = (int)v.size(3);
}

// fp32, contiguous, the heads and tokens as they are: what the kernels take per-token factors as
Tensor per_token(const Tensor& t) { return t.to(at::kFloat).contiguous().resolve_neg(); }

// g: the log decay, or what the kernel makes it from (decay_kind); vs: fp32 or bf16
bool linear_forward(const LinearPlan& pl, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g, const Tensor& vs, int dev, Tensor& out,
                    int decay_kind = DECAY_AS_IS, const float* decay_head = nullptr) {
  out = empty(v.sizes(), v.scalar_type(), v.device());
  ma_linear_params p{};
  p.dtype = MA_BF16;
  linear_sizes(q, k, v, p.batch, p.heads, p.heads_q, p.heads_k, p.seqlen, p.dim_k, p.dim_v);
  p.q = q.data_ptr(); p.k = k.data_ptr(); p.v = v.data_ptr(); p.o = out.data_ptr();
  p.log_decay = (const float*)g.data_ptr();
  p.v_scale = vs.defined() ? (const float*)vs.data_ptr() : nullptr;
  const int32_t vs_dtype = vs.defined() && vs.scalar_type() == at::kBFloat16 ? MA_BF16 : MA_LINEAR_FP32;
  p.q_scale = pl.q_scale;
  const size_t need = ma_linear_workspace_bytes(&p);
  const c10::DataPtr ws = scratch(need);
  p.workspace = ws.get(); p.workspace_bytes = need;
  const ma_stream_t st = stream_of(dev);
  NoGil release;
  return ma_linear_fwd_factors(&p, decay_kind == DECAY_LOG, decay_head, vs_dtype, st) == MA_OK;
}

// The chunked operator with gradients for q, k, v, the log decay and the value scale (if any), as LinearAttention.backward
// (tl_template/linear/linear_tl.py:1268-1340); see AttentionFunction.
struct LinearFunction : torch::autograd::Function<LinearFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g, const std::optional<Tensor>& vs, const Tensor* out,
                        double q_scale) {
    ctx->save_for_backward(vs ? variable_list{q, k, v, g, *vs} : variable_list{q, k, v, g});
    ctx->saved_data["q_scale"] = q_scale;
    return *out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const bool has_vs = saved.size() > 4;
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2];
    at::AutoDispatchBelowADInplaceOrView no_autograd;
    const Tensor g = per_token(saved[3]), vs = has_vs ? per_token(saved[4]) : Tensor();
    const Tensor dout = grads[0].to(v.scalar_type()).contiguous();
    const Tensor dq = empty(q.sizes(), q.scalar_type(), q.device()), dk = empty(k.sizes(), k.scalar_type(), k.device()),
                 dv = empty(v.sizes(), v.scalar_type(), v.device());
    // (nobody asks for the decay's gradient or the value scale's: a call that leaves them out)
    const bool with_decay = ctx->needs_input_grad(3) || (has_vs && ctx->needs_input_grad(4));
    Tensor dg, dvs;
    if (with_decay) dg = empty(g.sizes(), at::kFloat, v.device());
    if (with_decay && has_vs) dvs = empty(vs.sizes(), at::kFloat, v.device());
    ma_linear_bwd_params p{};
    p.dtype = MA_BF16;
    linear_sizes(q, k, v, p.batch, p.heads, p.heads_q, p.heads_k, p.seqlen, p.dim_k, p.dim_v);
    p.q = q.data_ptr(); p.k = k.data_ptr(); p.v = v.data_ptr(); p.dout = dout.data_ptr();
    p.log_decay = (const float*)g.data_ptr();
    p.v_scale = has_vs ? (const float*)vs.data_ptr() : nullptr;
    p.q_scale = (float)ctx->saved_data["q_scale"].toDouble();
    p.dq = dq.data_ptr(); p.dk = dk.data_ptr(); p.dv = dv.data_ptr(); p.dlog_decay = dg.defined() ? (float*)dg.data_ptr() : nullptr;
    p.dv_scale = dvs.defined() ? (float*)dvs.data_ptr() : nullptr;
    const size_t need = ma_linear_bwd_call_workspace_bytes(&p, with_decay);
    const c10::DataPtr ws = scratch(need);
    p.workspace = ws.get(); p.workspace_bytes = need;
    {
      NoGil release;
      TORCH_CHECK((with_decay ? ma_linear_bwd : ma_linear_bwd_qkv)(&p, stream_of(v.device().index())) == MA_OK, ma_last_error());
    }
    if (dg.defined()) dg = dg.to(saved[3].scalar_type());
    if (dvs.defined()) dvs = dvs.to(saved[4].scalar_type());
    return {dq, dk, dv, dg, dvs, Tensor(), Tensor()};
  }
};

// linear(q [B,Hq,T,Dk], k [B,Hk,T,Dk], v [B,H,T,Dv], decay [B,H,T], *custom) -> out [B,H,T,Dv], or None
PyObject* linear_call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const LinearPlan& pl = *(const LinearPlan*)PyCapsule_GetPointer(self, kLinearPlan);
  if (n != 4 + pl.n_custom || n > 12 || traced()) return none();
  const Tensor* t[12];
  for (int i = 0; i < n; i++)
    if (!(t[i] = tensor_of(args[i])) || !t[i]->is_cuda()) return none();
  const int dev = c10::hip::current_device();
  const Tensor &q = *t[0], &k = *t[1], &v = *t[2], &decay = *t[3];
  for (int i = 0; i < n; i++)
    if (!on(*t[i], dev)) return none();
  for (int i = 0; i < 3; i++)
    if (t[i]->dim() != 4 || t[i]->scalar_type() != at::kBFloat16 || t[i]->numel() == 0 || !t[i]->is_contiguous() || ((uintptr_t)t[i]->data_ptr() & 15))
      return none();
  const int64_t B = v.size(0), H = v.size(1), T = v.size(2);
  if (q.size(0) != B || k.size(0) != B || q.size(2) != T || k.size(2) != T || q.size(3) != k.size(3) || B > (1 << 30) || H > (1 << 30) || T > (1 << 30)) return none();
  if (decay.dim() != 3 || decay.size(0) != B || decay.size(1) != H || decay.size(2) != T) return none();
  Tensor vs;
  if (pl.v_scale_arg >= 0) {
    vs = *t[4 + pl.v_scale_arg];
    if (vs.dim() != 3 || vs.size(0) != B || vs.size(1) != H || vs.size(2) != T) return none();
  }
  // Without gradients the kernel takes the decay, a head's factor and a bf16 value scale as they are (a launch less each)
  bool wanted = false;
  for (int i = 0; i < n; i++) wanted = wanted || t[i]->requires_grad();
  if (!(wanted && at::GradMode::is_enabled())) {
    const Tensor* head = pl.decay_kind == DECAY_MUL_HEAD ? t[4 + pl.decay_head_arg] : nullptr;
    // (its values as they stand in memory: a tensor whose negation is a bit of its own goes the other way)
    auto as_it_is = [](const Tensor& x) { return x.layout() == at::kStrided && x.is_contiguous() && !x.is_neg(); };
    const bool plain = (q.size(3) == 128 || q.size(3) == 256) && decay.scalar_type() == at::kFloat && as_it_is(decay) &&
                       (!vs.defined() || ((vs.scalar_type() == at::kFloat || vs.scalar_type() == at::kBFloat16) && as_it_is(vs))) &&
                       (!head || (head->scalar_type() == at::kFloat && as_it_is(*head) && head->numel() == H));
    if (plain) {
      Tensor out;
      at::AutoDispatchBelowADInplaceOrView no_autograd;
      if (!linear_forward(pl, q, k, v, decay, vs, dev, out, pl.decay_kind, head ? (const float*)head->data_ptr() : nullptr)) return none();
      return THPVariable_Wrap(out);
    }
  }
  Tensor g = decay.to(at::kFloat);
  if (pl.decay_kind == DECAY_LOG) {
    g = g.log();
  } else if (pl.decay_kind == DECAY_MUL_HEAD) {
    g = g * t[4 + pl.decay_head_arg]->to(at::kFloat).reshape({1, -1, 1});
    if (g.dim() != 3 || g.size(0) != B || g.size(1) != H || g.size(2) != T) return none();
  }
  const bool grad = at::GradMode::is_enabled() &&
                    (q.requires_grad() || k.requires_grad() || v.requires_grad() || g.requires_grad() || (vs.defined() && vs.requires_grad()));
  Tensor out;
  {
    at::AutoDispatchBelowADInplaceOrView no_autograd;
    if (!linear_forward(pl, q, k, v, per_token(g), vs.defined() ? per_token(vs) : vs, dev, out)) return none();
  }
  if (grad) out = LinearFunction::apply(q, k, v, g, vs.defined() ? std::optional<Tensor>(vs) : std::nullopt, &out, (double)pl.q_scale);
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------------------------------------------------------- module
template <typename P>
void delete_plan(PyObject* capsule) {
  delete (P*)PyCapsule_GetPointer(capsule, PyCapsule_GetName(capsule));
}

// the callable of a plan: a built-in function whose self is the capsule that owns the plan
template <typename P>
PyObject* callable_of(P* plan, const char* name, PyMethodDef* def) {
  PyObject* capsule = PyCapsule_New(plan, name, delete_plan<P>);
  if (!capsule) {
    delete plan;
    return nullptr;
  }
  PyObject* f = PyCFunction_New(def, capsule);
  Py_DECREF(capsule);
  return f;
}

PyMethodDef kAttnDef = {"attention", (PyCFunction)(void (*)(void))attention_call, METH_FASTCALL, nullptr};
PyMethodDef kMlaDef = {"mla", (PyCFunction)(void (*)(void))mla_call, METH_FASTCALL, nullptr};
PyMethodDef kLinearDef = {"linear", (PyCFunction)(void (*)(void))linear_call, METH_FASTCALL, nullptr};

at::ScalarType scalar_type(int code) { return code == MA_BF16 ? at::kBFloat16 : at::kHalf; }

// attention_plan(family, dtype, causal, masked, scale, bias)
PyObject* attention_plan(PyObject*, PyObject* args) {
  int family, dtype, causal, masked;
  float scale, bias;
  if (!PyArg_ParseTuple(args, "iippff", &family, &dtype, &causal, &masked, &scale, &bias)) return nullptr;
  return callable_of(new AttnPlan{family, causal != 0, masked != 0, scale, bias, scalar_type(dtype), nullptr}, kAttnPlan, &kAttnDef);
}

// attention_masks(plan's callable, B, H, Sq, Skv, elem, blocks, elem_t | None, blocks_t | None)
PyObject* attention_masks(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *f, *t[4];
  long long B, H, Sq, Skv;
  if (!PyArg_ParseTuple(args, "OLLLLOOOO", &f, &B, &H, &Sq, &Skv, &t[0], &t[1], &t[2], &t[3])) return nullptr;
  auto* pl = (AttnPlan*)PyCapsule_GetPointer(PyCFunction_Check(f) ? PyCFunction_GetSelf(f) : nullptr, kAttnPlan);
  if (!pl) return nullptr;
  auto m = std::make_shared<Masks>(Masks{B, H, Sq, Skv, {}, {}, {}, {}});
  Tensor* to[4] = {&m->elem, &m->blocks, &m->elem_t, &m->blocks_t};
  for (int i = 0; i < 4; i++)
    if (t[i] != Py_None) {
      TORCH_CHECK(THPVariable_Check(t[i]), "attention_masks: tensors expected");
      *to[i] = THPVariable_Unpack(t[i]);
    }
  TORCH_CHECK(m->elem.defined() && m->blocks.defined(), "attention_masks: the keep mask and its tile mask are needed");
  pl->masks = std::move(m);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// mla_plan(dtype, scale)
PyObject* mla_plan(PyObject*, PyObject* args) {
  int dtype;
  float scale;
  if (!PyArg_ParseTuple(args, "if", &dtype, &scale)) return nullptr;
  return callable_of(new MlaPlan{scale, scalar_type(dtype)}, kMlaPlan, &kMlaDef);
}

// linear_plan(decay kind, index of the tensor multiplying the decay | -1, of the one multiplying the values | -1, number of custom tensors, q_scale)
PyObject* linear_plan(PyObject*, PyObject* args) {
  LinearPlan p{};
  if (!PyArg_ParseTuple(args, "iiiif", &p.decay_kind, &p.decay_head_arg, &p.v_scale_arg, &p.n_custom, &p.q_scale)) return nullptr;
  return callable_of(new LinearPlan(p), kLinearPlan, &kLinearDef);
}

PyMethodDef kMethods[] = {
    {"attention_plan", attention_plan, METH_VARARGS, "callable of a parallel attention operator"},
    {"attention_masks", attention_masks, METH_VARARGS, "the dense masks of one shape for a parallel attention operator"},
    {"mla_plan", mla_plan, METH_VARARGS, "callable of an MLA decode operator"},
    {"linear_plan", linear_plan, METH_VARARGS, "callable of a chunked linear attention operator"},
    {"mla_paged", (PyCFunction)(void (*)(void))mla_paged_call, METH_FASTCALL, "paged MLA decode"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "ma_host", "native calls of the attention operators", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_ma_host(void) { return PyModule_Create(&kModule); }
