// Native call path of the operators a generation calls per layer and step
// (attention, the QKV producer, the slab pack): the Python extension
// heatkv_amd._op_call.
//
// A small launch runs 6-8 us on the device, but checking eight tensors, reading
// the knobs and marshalling about thirty arguments cost the Python operator
// 15-16 us per call, so calls on early scales ran at the host's pace.  Here the
// same checks read the tensors in C++ (nothing is remembered from one call for
// the next), the outputs are allocated and the library is called: 16.4 -> 6.1 us
// per call of 16 tokens (B=2, 16 heads), back to back; a whole layer's ten small
// scales at B=1 966 -> 837 us.
//
// Only calls that the Python operator would take as they are: every function
// returns None, having launched nothing, when anything asks for more (an
// error to raise, an input to convert, a knob that is set, a HIP graph being
// captured, a tensor subclass, a torch mode or transform, the stream's first
// call, which makes its workspace), and the caller runs the operator's Python
// body, which stays the one place that defines what is refused and why.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <type_traits>

#include "heatkv.h"

namespace {

constexpr int64_t kD = 128;

// The library's entry points (addresses from the handle that _lib.load()
// opened) and the Python dicts that hold the environment, the per-stream
// workspaces and the checked devices.
struct State {
  decltype(&hkv_segmented_attention) attention = nullptr;
  decltype(&hkv_segmented_attention_split) attention_split = nullptr;
  decltype(&hkv_segmented_attention_split_bytes) split_bytes = nullptr;
  decltype(&hkv_segmented_attention_item_shape) item_shape = nullptr;
  decltype(&hkv_qkv_produce) produce = nullptr;
  decltype(&hkv_pack_segments) pack = nullptr;
  PyObject* env = nullptr;
  PyObject* knobs = nullptr;  // tuple of the environment keys that change a launch
  PyObject* workspaces = nullptr;
  PyObject* devices = nullptr;
  PyObject* plan_queries = nullptr;  // attribute names of a work plan
  PyObject* plan_shape = nullptr;
  bool ready = false;
} g;

struct Ref {  // a new reference
  PyObject* p;
  explicit Ref(PyObject* o) : p(o) {}
  ~Ref() { Py_XDECREF(p); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
};

int32_t code_of(at::ScalarType t) {
  switch (t) {
    case at::kHalf: return HKV_DTYPE_F16;
    case at::kBFloat16: return HKV_DTYPE_BF16;
    case at::kFloat: return HKV_DTYPE_F32;
    default: return 0;
  }
}

// A plain strided tensor of the GPU: a torch.Tensor or Parameter that no
// subclass, transform, conjugate / negative view or fake mode stands behind.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  const c10::DispatchKeySet rest =
      t.key_set() - c10::autograd_dispatch_keyset_with_ADInplaceOrView - c10::autocast_dispatch_keyset;
  return rest == c10::DispatchKeySet(c10::DispatchKey::CUDA) ? &t : nullptr;
}

bool dense(const at::Tensor& t, int64_t dim) { return t.dim() == dim && t.is_contiguous(); }
bool aligned(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

// No mode or transform that would see the operator's torch calls.
bool no_modes() {
  if (at::impl::torch_function_mode_enabled()) return false;
  const c10::DispatchKeySet usual =
      c10::DispatchKeySet({c10::DispatchKey::BackendSelect, c10::DispatchKey::ADInplaceOrView});
  return (c10::impl::tls_local_dispatch_key_set().included_ - usual).empty();
}

// The current device, gfx950 as already checked, with its current stream not
// under capture; -1 otherwise.
int current_device(void** stream) {
  const c10::DeviceIndex dev = c10::hip::current_device();
  Ref index(PyLong_FromLong(dev));
  if (PyDict_GetItem(g.devices, index.p) != Py_True) return -1;
  if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return -1;
  *stream = c10::hip::getCurrentHIPStream(dev).stream();
  return dev;
}

bool knobs_set() {
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(g.knobs); ++i)
    if (PyDict_GetItem(g.env, PyTuple_GET_ITEM(g.knobs, i)) != nullptr) return true;
  return false;
}

bool flag(PyObject* o, bool* v) {
  *v = o == Py_True;
  return o == Py_True || o == Py_False;
}

bool number(PyObject* o, double* v) {
  if (!PyFloat_CheckExact(o)) return false;
  *v = PyFloat_AS_DOUBLE(o);
  return true;
}

bool whole(PyObject* o, int64_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}

// Whether `plan` (None: no plan) is what segmented_attention_plan made for
// items of `queries`, batch B and length L on `dev`; its tensor in *out.
bool plan_fits(PyObject* plan, int32_t queries, int64_t B, int64_t L, int dev, const at::Tensor** out) {
  *out = nullptr;
  if (plan == Py_None) return true;
  const at::Tensor* t = plain(plan);
  if (t == nullptr || t->scalar_type() != at::kInt || !dense(*t, 2) || t->size(1) != 8 || t->size(0) == 0 ||
      t->get_device() != dev)
    return false;
  Ref have(PyObject_GetAttr(plan, g.plan_queries)), shape(PyObject_GetAttr(plan, g.plan_shape));
  int64_t q = 0, b = 0, l = 0;
  if (have.p == nullptr || shape.p == nullptr) {
    PyErr_Clear();
    return false;
  }
  *out = t;
  return whole(have.p, &q) && q == queries && PyTuple_CheckExact(shape.p) && PyTuple_GET_SIZE(shape.p) == 2 &&
         whole(PyTuple_GET_ITEM(shape.p, 0), &b) && whole(PyTuple_GET_ITEM(shape.p, 1), &l) && b == B && l == L;
}

// Where an all-fp32 call is better split (_split_values_pays in
// real_pruning_fused_attention.py, which holds the figures; `split_from` and
// `split_slab` are its two limits).
bool split_values_pays(int64_t B, int64_t H, int64_t L, int64_t cap, int64_t split_from, int64_t split_slab, int dev) {
  const int64_t pairs = B * H, rows = pairs * L;
  int64_t limit = split_slab;
  if (rows >= split_from) limit = std::max((L > 256 ? 8 : 4) * rows, split_slab / 4);
  if (B * cap > limit) return false;
  if (rows < 8192 || pairs <= 64) return true;
  int32_t cus = 0;  // the staged kernel's resident workgroups
  if (g.item_shape(HKV_DTYPE_F32, HKV_DTYPE_F32, HKV_DTYPE_F32, 1, 0, 0, dev, &cus) < 0) return false;
  return pairs * ((L + 127) / 128) > cus;
}

// attention(q, persisted_k, persisted_v, segment_starts, segment_ends,
// segment_counts, current_k, current_v, softmax_scale, softmax_mode,
// return_lse, out_dtype, work_plan, k_split_rows, split_values_rows,
// split_values_slab_rows)
PyObject* attention_call(PyObject* const* args, Py_ssize_t n) {
  if (!g.ready || n != 16 || !no_modes() || knobs_set()) Py_RETURN_NONE;
  const at::Tensor* t[8];
  for (int i = 0; i < 8; ++i)
    if ((t[i] = plain(args[i])) == nullptr) Py_RETURN_NONE;
  const at::Tensor &q = *t[0], &pk = *t[1], &pv = *t[2], &st = *t[3], &en = *t[4], &ct = *t[5], &ck = *t[6],
                   &cv = *t[7];
  double scale = 0;
  int64_t split_from = 0, split_slab = 0;
  bool with_lse = false, k_split = false;
  if (!number(args[8], &scale) || !flag(args[10], &with_lse) || !flag(args[13], &k_split) ||
      !whole(args[14], &split_from) || !whole(args[15], &split_slab))
    Py_RETURN_NONE;
  const char* mode = PyUnicode_CheckExact(args[9]) ? PyUnicode_AsUTF8(args[9]) : nullptr;
  if (mode == nullptr || (std::strcmp(mode, "exp") != 0 && std::strcmp(mode, "exp2") != 0)) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  at::ScalarType out_type = q.scalar_type();
  if (args[11] != Py_None) {
    if (!THPDtype_Check(args[11])) Py_RETURN_NONE;
    out_type = reinterpret_cast<THPDtype*>(args[11])->scalar_type;
  }
  void* stream = nullptr;
  const int dev = current_device(&stream);
  if (dev < 0) Py_RETURN_NONE;
  for (const at::Tensor* x : t)
    if (x->get_device() != dev) Py_RETURN_NONE;

  if (!dense(q, 4) || !dense(ck, 4) || !dense(cv, 4) || !dense(pk, 3) || !dense(pv, 3) || !dense(st, 2) ||
      !dense(en, 2) || !dense(ct, 1))
    Py_RETURN_NONE;
  const int64_t B = q.size(0), H = q.size(1), L = q.size(2), cap = pk.size(1), S = st.size(1);
  if (ck.sizes() != q.sizes() || cv.sizes() != q.sizes() || q.size(3) != kD || L <= 0 || B <= 0 || H <= 0 ||
      pk.sizes() != pv.sizes() || pk.size(0) != B || pk.size(2) != kD || st.sizes() != en.sizes() ||
      st.size(0) != H || ct.size(0) != H || B > 0x7fffffff || H > 0x7fffffff || L > 0x7fffffff || S > 0x7fffffff)
    Py_RETURN_NONE;
  const int32_t qc = code_of(q.scalar_type()), kc = code_of(ck.scalar_type()), vc = code_of(cv.scalar_type()),
                oc = code_of(out_type);
  if (qc == 0 || kc != qc || vc == 0 || oc == 0 || pk.scalar_type() != ck.scalar_type() ||
      pv.scalar_type() != cv.scalar_type() || st.scalar_type() != at::kInt || en.scalar_type() != at::kInt ||
      ct.scalar_type() != at::kInt)
    Py_RETURN_NONE;
  // fp32 q and k at the default dot modes: K (and V) as split rows, made by the
  // call itself unless the caller has them
  const bool rows32 = qc == HKV_DTYPE_F32 && vc != HKV_DTYPE_F32;
  if (k_split && !rows32) Py_RETURN_NONE;
  const bool split_v =
      qc == HKV_DTYPE_F32 && vc == HKV_DTYPE_F32 && split_values_pays(B, H, L, cap, split_from, split_slab, dev);
  const bool splits = (rows32 && !k_split) || split_v;
  if (splits && (!aligned(ck) || !aligned(pk) || (split_v && (!aligned(cv) || !aligned(pv))))) Py_RETURN_NONE;
  const int32_t queries = rows32 ? g.item_shape(qc, HKV_DTYPE_SPLIT_ROWS, vc, 1, 0, 0, 0, nullptr) : 128;
  const at::Tensor* plan = nullptr;
  if (!plan_fits(args[12], queries, B, L, dev, &plan)) Py_RETURN_NONE;

  Ref index(PyLong_FromLong(dev)), handle(PyLong_FromVoidPtr(stream));
  Ref key(PyTuple_Pack(2, index.p, handle.p));
  PyObject* const ws_obj = key.p != nullptr ? PyDict_GetItem(g.workspaces, key.p) : nullptr;
  if (ws_obj == nullptr || !THPVariable_Check(ws_obj)) Py_RETURN_NONE;
  const at::Tensor ws = THPVariable_Unpack(ws_obj);

  const auto options = q.options().requires_grad(false);
  int64_t need = 0;
  if (splits && (need = g.split_bytes(static_cast<int32_t>(B), static_cast<int32_t>(H), static_cast<int32_t>(L), cap,
                                      vc)) < 0)
    Py_RETURN_NONE;
  at::Tensor out = at::empty({B, L, H * kD}, options.dtype(out_type));
  at::Tensor lse, scratch;
  if (with_lse) lse = at::empty({B, H, L}, options.dtype(at::kFloat));
  if (splits) scratch = at::empty({need}, options.dtype(at::kByte));
  const int32_t* const plan_p = plan != nullptr ? static_cast<const int32_t*>(plan->data_ptr()) : nullptr;
  const int32_t units = plan != nullptr ? static_cast<int32_t>(plan->size(0)) : 0;
  float* const lse_p = with_lse ? static_cast<float*>(lse.data_ptr()) : nullptr;
  const int32_t k_code = k_split ? HKV_DTYPE_SPLIT_ROWS : kc, exp2 = mode[3] != 0 ? 1 : 0;
  const int32_t b = static_cast<int32_t>(B), h = static_cast<int32_t>(H), l = static_cast<int32_t>(L),
                s = static_cast<int32_t>(S), d = static_cast<int32_t>(kD);
  const int32_t *sp = static_cast<const int32_t*>(st.data_ptr()), *ep = static_cast<const int32_t*>(en.data_ptr()),
                *cp = static_cast<const int32_t*>(ct.data_ptr());
  const float fscale = static_cast<float>(scale);
  int32_t code;
  Py_BEGIN_ALLOW_THREADS
  if (splits)
    code = g.attention_split(q.data_ptr(), pk.data_ptr(), pv.data_ptr(), sp, ep, cp, ck.data_ptr(), cv.data_ptr(),
                             out.data_ptr(), lse_p, b, h, l, cap, s, d, qc, k_code, vc, oc, fscale, exp2, 0, 0,
                             plan_p, units, ws.data_ptr(), ws.numel(), nullptr, nullptr, nullptr, 0, nullptr,
                             scratch.data_ptr(), need, stream);
  else
    code = g.attention(q.data_ptr(), pk.data_ptr(), pv.data_ptr(), sp, ep, cp, ck.data_ptr(), cv.data_ptr(),
                       out.data_ptr(), lse_p, b, h, l, cap, s, d, qc, k_code, vc, oc, fscale, exp2, 0, 0, plan_p,
                       units, ws.data_ptr(), ws.numel(), stream);
  Py_END_ALLOW_THREADS
  if (code != HKV_OK) Py_RETURN_NONE;  // refused: the Python body repeats the call and raises
  if (!with_lse) return THPVariable_Wrap(std::move(out));
  Ref o(THPVariable_Wrap(std::move(out))), e(THPVariable_Wrap(std::move(lse)));
  return o.p != nullptr && e.p != nullptr ? PyTuple_Pack(2, o.p, e.p) : nullptr;
}

// produce(qkv, num_heads, scale_mul, rope_table, rope_start_row, normalize,
// eps, qk_dtype, append, k_split_rows)
PyObject* produce_call(PyObject* const* args, Py_ssize_t n) {
  if (!g.ready || n != 10 || !no_modes()) Py_RETURN_NONE;
  const at::Tensor* qkv = plain(args[0]);
  int64_t H = 0, start = 0;
  bool normalize = false, k_split = false;
  double eps = 0;
  if (qkv == nullptr || !whole(args[1], &H) || !whole(args[4], &start) || !flag(args[5], &normalize) ||
      !number(args[6], &eps) || !THPDtype_Check(args[7]) || !flag(args[9], &k_split))
    Py_RETURN_NONE;
  void* stream = nullptr;
  const int dev = current_device(&stream);
  if (dev < 0 || qkv->get_device() != dev || !qkv->is_contiguous()) Py_RETURN_NONE;
  if (H <= 0 || H > 0x7fffffff) Py_RETURN_NONE;
  const bool whole_rows = qkv->dim() == 3 && qkv->size(2) == 3 * H * kD;
  const bool parts = qkv->dim() == 5 && qkv->size(2) == 3 && qkv->size(3) == H && qkv->size(4) == kD;
  if (!whole_rows && !parts) Py_RETURN_NONE;
  const int64_t B = qkv->size(0), L = qkv->size(1);
  const at::ScalarType qk = reinterpret_cast<THPDtype*>(args[7])->scalar_type;
  const int32_t ic = code_of(qkv->scalar_type()), oc = code_of(qk);
  if (B <= 0 || L <= 0 || B > 0x7fffffff || L > 0x7fffffff || ic == 0 || oc == 0 ||
      (k_split && oc != HKV_DTYPE_F32))
    Py_RETURN_NONE;
  const float *sm = nullptr, *rope = nullptr;
  int64_t rope_rows = 0;
  if (args[2] != Py_None) {
    const at::Tensor* t = plain(args[2]);
    if (t == nullptr || t->get_device() != dev || t->scalar_type() != at::kFloat || !t->is_contiguous() ||
        t->numel() != H)
      Py_RETURN_NONE;
    sm = static_cast<const float*>(t->data_ptr());
  }
  if (args[3] != Py_None) {
    const at::Tensor* t = plain(args[3]);
    if (t == nullptr || t->get_device() != dev || t->scalar_type() != at::kFloat || !dense(*t, 3) ||
        t->size(0) != 2 || t->size(2) != kD / 2)
      Py_RETURN_NONE;
    rope = static_cast<const float*>(t->data_ptr());
    rope_rows = t->size(1);
  }
  const at::Tensor *slab_k = nullptr, *slab_v = nullptr, *offsets = nullptr;
  if (args[8] != Py_None) {
    if (!PyTuple_CheckExact(args[8]) || PyTuple_GET_SIZE(args[8]) != 3) Py_RETURN_NONE;
    slab_k = plain(PyTuple_GET_ITEM(args[8], 0));
    slab_v = plain(PyTuple_GET_ITEM(args[8], 1));
    offsets = plain(PyTuple_GET_ITEM(args[8], 2));
    if (slab_k == nullptr || slab_v == nullptr || offsets == nullptr || slab_k->get_device() != dev ||
        slab_v->get_device() != dev || offsets->get_device() != dev || !dense(*slab_k, 3) || !dense(*slab_v, 3) ||
        slab_k->sizes() != slab_v->sizes() || slab_k->size(0) != B || slab_k->size(2) != kD ||
        slab_k->scalar_type() != qk || slab_v->scalar_type() != qkv->scalar_type() ||
        offsets->scalar_type() != at::kInt || !offsets->is_contiguous() || offsets->numel() != H)
      Py_RETURN_NONE;
  }
  const auto options = qkv->options().requires_grad(false);
  at::Tensor q = at::empty({B, H, L, kD}, options.dtype(qk)), k = at::empty({B, H, L, kD}, options.dtype(qk)),
             v = at::empty({B, H, L, kD}, options);
  int32_t code;
  Py_BEGIN_ALLOW_THREADS
  code = g.produce(qkv->data_ptr(), 3 * H * kD, nullptr, nullptr, sm, rope, rope_rows, start, q.data_ptr(),
                   k.data_ptr(), v.data_ptr(), slab_k != nullptr ? slab_k->data_ptr() : nullptr,
                   slab_v != nullptr ? slab_v->data_ptr() : nullptr,
                   offsets != nullptr ? static_cast<const int32_t*>(offsets->data_ptr()) : nullptr,
                   slab_k != nullptr ? slab_k->size(1) : 0, static_cast<int32_t>(B), static_cast<int32_t>(H),
                   static_cast<int32_t>(L), static_cast<int32_t>(kD), ic, oc, k_split ? HKV_DTYPE_SPLIT_ROWS : oc,
                   ic, normalize ? 1 : 0, static_cast<float>(eps), stream);
  Py_END_ALLOW_THREADS
  if (code != HKV_OK) Py_RETURN_NONE;
  Ref a(THPVariable_Wrap(std::move(q))), b(THPVariable_Wrap(std::move(k))), c(THPVariable_Wrap(std::move(v)));
  return a.p != nullptr && b.p != nullptr && c.p != nullptr ? PyTuple_Pack(3, a.p, b.p, c.p) : nullptr;
}

// pack(dst_k, dst_v, src_k, src_v, dst_starts, src_starts, lengths, max_length,
// block_t): True when the copy was launched
PyObject* pack_call(PyObject* const* args, Py_ssize_t n) {
  int64_t longest = 0, block = 0;
  if (!g.ready || n != 9 || !no_modes() || !whole(args[7], &longest) || !whole(args[8], &block)) Py_RETURN_NONE;
  const at::Tensor* t[7];
  for (int i = 0; i < 7; ++i)
    if ((t[i] = plain(args[i])) == nullptr) Py_RETURN_NONE;
  const at::Tensor &dk = *t[0], &dv = *t[1], &sk = *t[2], &sv = *t[3], &ds = *t[4], &ss = *t[5], &ln = *t[6];
  void* stream = nullptr;
  const int dev = current_device(&stream);
  if (dev < 0) Py_RETURN_NONE;
  for (const at::Tensor* x : t)
    if (x->get_device() != dev) Py_RETURN_NONE;
  if (!dense(dk, 3) || !dense(dv, 3) || !dense(sk, 3) || !dense(sv, 3) || dk.sizes() != dv.sizes() ||
      sk.sizes() != sv.sizes() || dk.size(0) != sk.size(0) || dk.size(2) != sk.size(2) || dk.size(2) > kD ||
      dk.numel() == 0 || sk.numel() == 0 || sk.scalar_type() != dk.scalar_type() ||
      sv.scalar_type() != dv.scalar_type() || dk.size(0) > 0x7fffffff)
    Py_RETURN_NONE;
  const int64_t items = ln.numel();
  for (const at::Tensor* x : {&ds, &ss, &ln})
    if (x->scalar_type() != at::kLong || !x->is_contiguous() || x->numel() != items) Py_RETURN_NONE;
  if (items <= 0 || items > 0x7fffffff || longest <= 0 || longest > 0x7fffffff || block <= 0 || block > 0x7fffffff)
    Py_RETURN_NONE;
  const int64_t limit = (longest + block - 1) / block * block;
  int32_t code;
  Py_BEGIN_ALLOW_THREADS
  code = g.pack(sk.data_ptr(), sv.data_ptr(), dk.data_ptr(), dv.data_ptr(), sk.stride(0), dk.stride(0), sk.size(1),
                dk.size(1), static_cast<int32_t>(dk.size(0)), static_cast<int32_t>(dk.size(2)),
                static_cast<int32_t>(dk.element_size()), static_cast<int32_t>(dv.element_size()),
                static_cast<const int64_t*>(ds.data_ptr()), static_cast<const int64_t*>(ss.data_ptr()),
                static_cast<const int64_t*>(ln.data_ptr()), static_cast<int32_t>(items),
                static_cast<int32_t>(limit < 0x7fffffff ? limit : 0x7fffffff), stream);
  Py_END_ALLOW_THREADS
  if (code != HKV_OK) Py_RETURN_NONE;
  Py_RETURN_TRUE;
}

// torch's exceptions (out of memory among them) end at this boundary: the
// Python body then runs and meets them itself.
template <PyObject* (*F)(PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject*, PyObject* const* args, Py_ssize_t n) {
  try {
    return F(args, n);
  } catch (const std::exception&) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

// A prototype as compiled here: return and argument types, i int32, l int64,
// f float, p pointer.
template <typename T>
constexpr char type_code() {
  if (std::is_pointer<T>::value) return 'p';
  if (std::is_same<T, float>::value) return 'f';
  return sizeof(T) == 8 ? 'l' : 'i';
}
template <typename R, typename... A>
std::string prototype(R (*)(A...)) {
  return {type_code<R>(), type_code<A>()...};
}

// prototypes(): those of init's entry points, in its order.
PyObject* prototypes(PyObject*, PyObject*) {
  const std::string p[6] = {prototype(g.attention), prototype(g.attention_split), prototype(g.split_bytes),
                            prototype(g.item_shape), prototype(g.produce), prototype(g.pack)};
  return Py_BuildValue("(ssssss)", p[0].c_str(), p[1].c_str(), p[2].c_str(), p[3].c_str(), p[4].c_str(),
                       p[5].c_str());
}

// init(addresses, env, knobs, workspaces, devices)
PyObject* init(PyObject*, PyObject* args) {
  unsigned long long a[6];
  PyObject *env, *knobs, *workspaces, *devices;
  if (!PyArg_ParseTuple(args, "(KKKKKK)O!O!O!O!", a, a + 1, a + 2, a + 3, a + 4, a + 5, &PyDict_Type, &env,
                        &PyTuple_Type, &knobs, &PyDict_Type, &workspaces, &PyDict_Type, &devices))
    return nullptr;
  if (!g.ready) {
    g.attention = reinterpret_cast<decltype(g.attention)>(a[0]);
    g.attention_split = reinterpret_cast<decltype(g.attention_split)>(a[1]);
    g.split_bytes = reinterpret_cast<decltype(g.split_bytes)>(a[2]);
    g.item_shape = reinterpret_cast<decltype(g.item_shape)>(a[3]);
    g.produce = reinterpret_cast<decltype(g.produce)>(a[4]);
    g.pack = reinterpret_cast<decltype(g.pack)>(a[5]);
    for (PyObject* o : {env, knobs, workspaces, devices}) Py_INCREF(o);
    g.env = env;
    g.knobs = knobs;
    g.workspaces = workspaces;
    g.devices = devices;
    g.plan_queries = PyUnicode_InternFromString("hkv_queries_per_item");
    g.plan_shape = PyUnicode_InternFromString("hkv_plan_shape");
    g.ready = g.plan_queries != nullptr && g.plan_shape != nullptr;
  }
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"attention", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<attention_call>)),
     METH_FASTCALL, "The attention operator's launch, or None"},
    {"produce", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<produce_call>)), METH_FASTCALL,
     "The QKV producer's launch, or None"},
    {"pack", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<pack_call>)), METH_FASTCALL,
     "The slab pack's launch, or None"},
    {"prototypes", prototypes, METH_NOARGS, "The entry points' prototypes as compiled, in init's order"},
    {"init", init, METH_VARARGS, "init(addresses, env, knobs, workspaces, devices)"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_op_call", "Native call path of the operators", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__op_call() { return PyModule_Create(&module); }
