// The C-ABI entry points as Python callables and as torch operators, in
// native code (module idempotent_llm_amd._native).
//
// What bounds a call of these entry points from Python at small sizes is the
// host: a ctypes call converts its 10 to 50 arguments one by one in Python
// (8 to 15 us), and an operator registered from Python adds its dispatch
// through the interpreter (20 us and more), against 5 us of kernel. Here an
// entry's argument list is converted by a thunk generated from the function
// type that include/detllm_hip.h declares, and the detllm_rocm:: operators'
// CUDA (HIP) kernels allocate their outputs and launch without returning to
// the interpreter. Measured per call: the 12-argument fused
// product 9.3 -> 5.2 us (its kernel alone 4.9), an MLP block of 8 rows (three
// operators, two products, two copies) 84 -> 40, decode attention 18 -> 12,
// the prefill of 200 tokens 3.42 -> 2.73 ms.
//
// The operators' schemas, fakes and documentation stay in torch_ops.py (the
// pattern of src/detllm/ops/int_prims.py:96-136); each kernel below makes the
// same outputs and passes the same arguments as its docstring there states.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/library.h>

#include <string>
#include <tuple>
#include <utility>

#include "../../include/detllm_hip.h"

namespace {

// ------------------------------------------------- entries from Python

// The current torch stream of the current device, as the entries take it.
hipStream_t current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

// One Python argument as an entry's parameter type. Pointers: a tensor's
// data, None, or an address; integers as int(x) gives them, truncated to the
// parameter's width as ctypes does. False: a Python exception is set.
bool as_int(PyObject* o, long long* v) {
  if (PyLong_CheckExact(o)) {
    *v = (long long)PyLong_AsUnsignedLongLongMask(o);
    return !PyErr_Occurred();
  }
  PyObject* n = PyNumber_Long(o);
  if (!n) return false;
  *v = (long long)PyLong_AsUnsignedLongLongMask(n);
  Py_DECREF(n);
  return !PyErr_Occurred();
}
template <class T>
bool convert(PyObject* o, T* out) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) {
      *out = nullptr;
      return true;
    }
    if (THPVariable_Check(o)) {
      *out = reinterpret_cast<T>(THPVariable_Unpack(o).data_ptr());
      return true;
    }
    long long v;
    if (!as_int(o, &v)) return false;
    *out = reinterpret_cast<T>((uintptr_t)v);
    return true;
  } else {
    long long v;
    if (!as_int(o, &v)) return false;
    *out = static_cast<T>(v);
    return true;
  }
}

// Runs entry f on `args` (every parameter but a trailing stream, which is
// `stream`): the entry's return code, or -1 with a Python exception set.
template <class... A, size_t... I>
bool run(int (*f)(A...), PyObject* const* args, hipStream_t stream, std::index_sequence<I...>,
         int* rc) {
  std::tuple<A...> v;
  constexpr size_t N = sizeof...(A);
  auto one = [&](auto idx) {
    constexpr size_t k = decltype(idx)::value;
    using T = std::tuple_element_t<k, std::tuple<A...>>;
    if constexpr (k == N - 1 && std::is_same_v<T, hipStream_t>) {
      std::get<k>(v) = stream;
      return true;
    } else {
      return convert<T>(args[k], &std::get<k>(v));
    }
  };
  if (!(one(std::integral_constant<size_t, I>{}) && ...)) return false;
  Py_BEGIN_ALLOW_THREADS
  *rc = f(std::get<I>(v)...);
  Py_END_ALLOW_THREADS
  return true;
}

struct Entry {
  const char* name;
  int nargs;        // Python arguments: the parameters but a trailing stream
  bool has_stream;
  bool (*call)(PyObject* const*, hipStream_t, int*);
};

template <auto F>
struct Bind;
template <class... A, int (*F)(A...)>
struct Bind<F> {
  static constexpr bool has_stream =
      std::is_same_v<std::tuple_element_t<sizeof...(A) - 1, std::tuple<A...>>, hipStream_t>;
  static bool call(PyObject* const* args, hipStream_t s, int* rc) {
    return run(F, args, s, std::index_sequence_for<A...>{}, rc);
  }
  static constexpr Entry entry(const char* name) {
    return Entry{name, (int)sizeof...(A) - (has_stream ? 1 : 0), has_stream, &call};
  }
};

#define DI_ENTRY(NAME) Bind<&NAME>::entry(#NAME)
const Entry ENTRIES[] = {
    DI_ENTRY(detllm_igemm_nt), DI_ENTRY(detllm_igemv_nt), DI_ENTRY(detllm_igemv_nt_pf),
    DI_ENTRY(detllm_igemv_plan), DI_ENTRY(detllm_attn_split_plan), DI_ENTRY(detllm_transpose_i8), DI_ENTRY(detllm_pack_nt),
    DI_ENTRY(detllm_greedy_pick), DI_ENTRY(detllm_greedy_pick_noalloc),
    DI_ENTRY(detllm_logits_digest), DI_ENTRY(detllm_embed_normq), DI_ENTRY(detllm_residual_normq),
    DI_ENTRY(detllm_norm_quant), DI_ENTRY(detllm_attn_decode_split), DI_ENTRY(detllm_attn_decode_split_sum),
    DI_ENTRY(detllm_igemv_resnormq), DI_ENTRY(detllm_igemv_merge),
    DI_ENTRY(detllm_igemv_merge_ext), DI_ENTRY(detllm_swiglu_quant),
    DI_ENTRY(detllm_igemv_swiglu), DI_ENTRY(detllm_merge_rowcol), DI_ENTRY(detllm_merge_ext),
    DI_ENTRY(detllm_qkv_epilogue), DI_ENTRY(detllm_kq_est), DI_ENTRY(detllm_requant_static_cols),
    DI_ENTRY(detllm_igemv_requant_static), DI_ENTRY(detllm_attn_prefill),
    DI_ENTRY(detllm_attn_decode), DI_ENTRY(detllm_qkv_attn_decode),
    DI_ENTRY(detllm_qkv_attn_decode_ext), DI_ENTRY(detllm_decode_prologue),
    DI_ENTRY(detllm_op_quant_i8_pertoken), DI_ENTRY(detllm_op_requant_i32_common),
    DI_ENTRY(detllm_op_requant_i8_rowcol), DI_ENTRY(detllm_op_requant_i8_static),
    DI_ENTRY(detllm_op_residual), DI_ENTRY(detllm_op_rmsnorm), DI_ENTRY(detllm_op_softmax),
    DI_ENTRY(detllm_op_di_exp), DI_ENTRY(detllm_op_swiglu), DI_ENTRY(detllm_op_rope),
    DI_ENTRY(detllm_op_scalar),
};
#undef DI_ENTRY

// entry(stream, *args): stream None (torch's current one) or a handle.
// Raises TypeError for another argument count and RuntimeError for a nonzero
// return code.
PyObject* call_entry(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  const Entry* e = static_cast<const Entry*>(PyCapsule_GetPointer(self, "detllm entry"));
  if (!e) return nullptr;
  if (n != e->nargs + 1) {
    PyErr_Format(PyExc_TypeError, "%s: expected %d arguments, got %zd", e->name, e->nargs, n - 1);
    return nullptr;
  }
  int rc = 0;
  try {
    hipStream_t s = nullptr;
    if (e->has_stream) {
      long long v;
      if (args[0] == Py_None) s = current_stream();
      else if (as_int(args[0], &v)) s = reinterpret_cast<hipStream_t>((uintptr_t)v);
      else return nullptr;
    }
    if (!e->call(args + 1, s, &rc)) return nullptr;
  } catch (const std::exception& ex) {
    PyErr_SetString(PyExc_RuntimeError, ex.what());
    return nullptr;
  }
  if (rc != 0) {
    PyErr_Format(PyExc_RuntimeError, "%s failed (code %d)", e->name, rc);
    return nullptr;
  }
  Py_RETURN_NONE;
}

PyMethodDef ENTRY_DEF = {"entry", (PyCFunction)(void (*)(void))call_entry, METH_FASTCALL, nullptr};

// {name: callable} of every entry point
PyObject* make_entries(PyObject*, PyObject*) {
  PyObject* d = PyDict_New();
  if (!d) return nullptr;
  for (const Entry& e : ENTRIES) {
    PyObject* cap = PyCapsule_New((void*)&e, "detllm entry", nullptr);
    PyObject* fn = cap ? PyCFunction_New(&ENTRY_DEF, cap) : nullptr;
    Py_XDECREF(cap);
    if (!fn || PyDict_SetItemString(d, e.name, fn) != 0) {
      Py_XDECREF(fn);
      Py_DECREF(d);
      return nullptr;
    }
    Py_DECREF(fn);
  }
  return d;
}

PyMethodDef METHODS[] = {
    {"entries", make_entries, METH_NOARGS, "{name: entry(stream, *args)} of the C ABI"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef MODULE = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, METHODS,
                      nullptr, nullptr, nullptr, nullptr};

// --------------------------------------------------------- torch operators

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using T2 = std::tuple<Tensor, Tensor>;
using T3 = std::tuple<Tensor, Tensor, Tensor>;

void check(int rc, const char* name) {
  if (rc != 0) throw std::runtime_error(std::string(name) + " failed (code " + std::to_string(rc) + ")");
}
#define DI_RUN(F, ...) check(F(__VA_ARGS__, current_stream()), #F)

template <class T>
T* ptr(const Tensor& t) {
  return static_cast<T*>(t.data_ptr());
}
template <class T>
T* ptr(const OptTensor& t) {
  return t && t->defined() ? static_cast<T*>(t->data_ptr()) : nullptr;
}
const int64_t* i64(const Tensor& t) { return ptr<int64_t>(t); }
const int64_t* i64(const OptTensor& t) { return ptr<int64_t>(t); }

Tensor empty(at::IntArrayRef shape, at::ScalarType dt, const Tensor& like) {
  return at::empty(shape, at::TensorOptions().dtype(dt).device(like.device()));
}
// An operand written in place: its version moves on, as for any mutated input
void mutated(const Tensor& t) {
  if (!t.is_inference()) t.unsafeGetTensorImpl()->bump_version();
}
// Operands of another rank are refused, as unpacking their shape did.
void rank(const Tensor& t, int64_t n, const char* op) {
  TORCH_CHECK_VALUE(t.dim() == n, op, ": expected ", n, " dimensions, got ", t.dim());
}
T3 rows_out(int64_t R, int64_t C, const Tensor& like) {
  return {empty({R, C}, at::kChar, like), empty({R}, at::kLong, like), empty({R}, at::kLong, like)};
}

// What the packing and product kernels index by a's shape alone: one-byte
// elements, one K, b's matrices one for all or one each, one device.
void check_int_gemm(const Tensor& a, const Tensor& b) {
  TORCH_CHECK_VALUE(a.element_size() == 1 && b.element_size() == 1,
                    "int_gemm: expected int8 operands, got ", a.scalar_type(), " and ",
                    b.scalar_type());
  TORCH_CHECK_VALUE(a.dim() >= 2 && b.dim() >= 2 && a.size(-1) == b.size(-2) &&
                        (b.dim() == 2 || a.sizes().slice(0, a.dim() - 2) ==
                                             b.sizes().slice(0, b.dim() - 2)),
                    "int_gemm: expected [*, M, K] and [K, N] or [*, K, N], got ", a.sizes(),
                    " and ", b.sizes());
  TORCH_CHECK_VALUE(a.device() == b.device(), "int_gemm: operands on ", a.device(), " and ",
                    b.device());
}

Tensor op_int_gemm(const Tensor& a, const Tensor& b) {
  check_int_gemm(a, b);
  if (b.dim() == 2 && a.dim() > 2) {
    auto lead = a.sizes().vec();
    lead.back() = b.size(-1);
    return op_int_gemm(a.reshape({-1, a.size(-1)}), b).reshape(lead);
  }
  const int64_t M = a.size(-2), K = a.size(-1), N = b.size(-1);
  auto shape = a.sizes().vec();
  shape.back() = N;
  if (M == 0 || N == 0) return at::zeros(shape, a.options().dtype(at::kInt));
  // few rows of one matrix take the skinny kernels (K in steps of 16), the
  // rest the tiled one, at its best in whole 128-byte slices of K (unless
  // those pass the largest K of an int32 sum, 131071)
  const bool skinny = a.dim() == 2 && M <= 64;
  const int64_t step = skinny || (K + 127) / 128 * 128 > 131071 ? 16 : 128;
  const int64_t Kp = std::max(step, (K + step - 1) / step * step);
  int64_t batch = 1;
  for (int64_t i = 0; i < a.dim() - 2; ++i) batch *= a.size(i);
  const Tensor ac = a.contiguous(), bc = b.contiguous();
  // (the products load 16 bytes at a time)
  const bool as_is = K == Kp && (reinterpret_cast<uintptr_t>(ac.data_ptr()) & 15) == 0;
  const Tensor bt = empty({batch, N, Kp}, at::kChar, a);
  const Tensor ap = as_is ? ac : empty({batch, M, Kp}, at::kChar, a);
  DI_RUN(detllm_pack_nt, ptr<int8_t>(ac), as_is ? nullptr : ptr<int8_t>(ap), ptr<int8_t>(bc),
         ptr<int8_t>(bt), (int)M, (int)N, (int)K, (int)Kp, (int)batch);
  Tensor out = empty(shape, at::kInt, a);
  if (skinny)
    DI_RUN(detllm_igemv_nt, ptr<int8_t>(ap), ptr<int8_t>(bt), ptr<int32_t>(out), (int)M, (int)N,
           (int)Kp, 1, M * N);
  else
    DI_RUN(detllm_igemm_nt, ptr<int8_t>(ap), ptr<int8_t>(bt), ptr<int32_t>(out), (int)M, (int)N,
           (int)Kp, (int)batch, M * Kp, N * Kp, M * N);
  return out;
}

Tensor scalar_op(int op, const Tensor& a) {
  const Tensor x = a.to(at::kLong).contiguous();
  Tensor out = empty(a.sizes(), at::kLong, a);
  DI_RUN(detllm_op_scalar, op, i64(x), nullptr, nullptr, x.numel(), ptr<int64_t>(out), nullptr);
  return out;
}
Tensor op_isqrt(const Tensor& a) { return scalar_op(0, a); }
Tensor op_ilog2(const Tensor& a) { return scalar_op(1, a); }

Tensor op_greedy_pick(const Tensor& logits, const Tensor& head_m) {
  rank(logits, 2, "greedy_pick");
  constexpr int64_t chunk = 2048;
  const int64_t R = logits.size(0), V = logits.size(1), nch = (V + chunk - 1) / chunk;
  Tensor pv = empty({R, nch}, at::kLong, logits), pi = empty({R, nch}, at::kLong, logits);
  Tensor out = empty({R}, at::kLong, logits);
  const Tensor lg = logits.contiguous(), hm = head_m.contiguous();
  DI_RUN(detllm_greedy_pick, ptr<int32_t>(lg), i64(hm), (int)R, (int)V, (int)chunk,
         ptr<int64_t>(pv), ptr<int64_t>(pi), ptr<int64_t>(out));
  return out;
}

std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> op_embed_normq(
    const Tensor& ids, const Tensor& e8, const Tensor& em, const Tensor& ek, const OptTensor& sm_m,
    int64_t sm_k, const Tensor& err) {
  const int64_t R = ids.numel(), H = e8.size(1);
  Tensor h = empty({R, H}, at::kInt, ids), k_res = empty({R}, at::kLong, ids);
  auto [x8, xm, xk] = rows_out(R, H, ids);
  const Tensor idc = ids.contiguous();
  DI_RUN(detllm_embed_normq, i64(idc), (int)R, (int)H, e8.size(0), ptr<int8_t>(e8), i64(em), i64(ek),
         ptr<int32_t>(h), ptr<int64_t>(k_res), i64(sm_m), sm_k, ptr<int8_t>(x8), ptr<int64_t>(xm),
         ptr<int64_t>(xk), ptr<int32_t>(err));
  mutated(err);
  return {h, k_res, x8, xm, xk};
}

T3 op_norm_quant(const Tensor& h, const OptTensor& sm_m, int64_t sm_k) {
  rank(h, 2, "norm_quant");
  const int64_t R = h.size(0), C = h.size(1);
  auto [x8, xm, xk] = rows_out(R, C, h);
  const Tensor hc = h.contiguous();
  DI_RUN(detllm_norm_quant, ptr<int32_t>(hc), (int)R, (int)C, i64(sm_m), sm_k, ptr<int8_t>(x8),
         ptr<int64_t>(xm), ptr<int64_t>(xk));
  return {x8, xm, xk};
}

T3 op_residual_normq(const Tensor& P, const Tensor& row_m, const Tensor& row_k,
                     const Tensor& col_m, int64_t col_k, int64_t tb, const Tensor& h,
                     const Tensor& k_res, const OptTensor& sm_m, int64_t sm_k) {
  rank(P, 3, "residual_normq");
  const int64_t ns = P.size(0), R = P.size(1), C = P.size(2);
  auto [x8, xm, xk] = rows_out(R, C, P);
  const Tensor Pc = P.contiguous();
  DI_RUN(detllm_residual_normq, ptr<int32_t>(Pc), (int)ns, R * C, (int)R, (int)C, i64(row_m),
         i64(row_k), i64(col_m), col_k, (int)tb, ptr<int32_t>(h), ptr<int64_t>(k_res), i64(sm_m),
         sm_k, ptr<int8_t>(x8), ptr<int64_t>(xm), ptr<int64_t>(xk), nullptr, 0, 0, 0, 0);
  mutated(h);
  mutated(k_res);
  return {x8, xm, xk};
}

T3 op_swiglu_quant(const Tensor& P, const Tensor& xm, const Tensor& xk, const Tensor& gate_m,
                   int64_t gate_k, const Tensor& up_m, int64_t up_k, const Tensor& ds_m,
                   int64_t ds_k) {
  rank(P, 3, "swiglu_quant");
  const int64_t ns = P.size(0), R = P.size(1), C2 = P.size(2), I = C2 / 2;
  auto [y8, ym, yk] = rows_out(R, I, P);
  const Tensor Pc = P.contiguous();
  DI_RUN(detllm_swiglu_quant, ptr<int32_t>(Pc), (int)ns, R * C2, (int)R, (int)I, i64(xm), i64(xk),
         i64(gate_m), gate_k, i64(up_m), up_k, i64(ds_m), ds_k, ptr<int8_t>(y8), ptr<int64_t>(ym),
         ptr<int64_t>(yk), nullptr, 0, 0, 0, 0);
  return {y8, ym, yk};
}

T3 op_merge_rowcol(const Tensor& attn, const Tensor& os_m, int64_t os_k, const Tensor& col_m,
                   int64_t col_k) {
  rank(attn, 2, "merge_rowcol");
  const int64_t R = attn.size(0), C = attn.size(1);
  auto [a8, am, ak] = rows_out(R, C, attn);
  const Tensor ac = attn.contiguous();
  DI_RUN(detllm_merge_rowcol, i64(ac), 1, 0, (int)R, (int)C, i64(os_m), os_k, i64(col_m), col_k,
         ptr<int8_t>(a8), ptr<int64_t>(am), ptr<int64_t>(ak), nullptr, 0, 0, 0, 0);
  return {a8, am, ak};
}

T2 op_qkv_epilogue(const Tensor& P, int64_t B, int64_t T, int64_t n_q, int64_t n_kv,
                   const Tensor& xm, const Tensor& xk, const Tensor& positions, const Tensor& q_m,
                   int64_t q_k, const Tensor& k_m, int64_t k_k, const Tensor& v_m, int64_t v_k,
                   const Tensor& q_norm_m, int64_t q_norm_k, const Tensor& k_norm_m,
                   int64_t k_norm_k, const Tensor& qs_m, int64_t qs_k, const Tensor& kq_m,
                   const Tensor& kq_k, const Tensor& ks_m, const Tensor& ks_k, const Tensor& vq_m,
                   const Tensor& vq_k, const Tensor& cos_t, const Tensor& sin_t,
                   const Tensor& kpool, const Tensor& vpool, const Tensor& table,
                   int64_t slot_base, const Tensor& err) {
  rank(P, 3, "qkv_epilogue");
  const int64_t ns = P.size(0), R = P.size(1);
  Tensor q8 = empty({B, n_q, T, 128}, at::kChar, P), tpos = empty({B, n_q, T}, at::kLong, P);
  const Tensor Pc = P.contiguous(), pos = positions.contiguous();
  DI_RUN(detllm_qkv_epilogue, ptr<int32_t>(Pc), (int)ns, R * P.size(2), (int)B, (int)T, (int)n_q,
         (int)n_kv, i64(xm), i64(xk), i64(pos), i64(q_m), q_k, i64(k_m), k_k, i64(v_m), v_k,
         i64(q_norm_m), q_norm_k, i64(k_norm_m), k_norm_k, i64(qs_m), qs_k, i64(kq_m), i64(kq_k),
         i64(ks_m), i64(ks_k), i64(vq_m), i64(vq_k), ptr<int16_t>(cos_t), ptr<int16_t>(sin_t),
         cos_t.size(0), ptr<int8_t>(q8), ptr<int64_t>(tpos), nullptr, ptr<int8_t>(kpool),
         ptr<int8_t>(vpool), ptr<int32_t>(table), (int)table.size(1), nullptr, slot_base, nullptr,
         ptr<int32_t>(err));
  mutated(kpool);
  mutated(vpool);
  mutated(err);
  return {q8, tpos};
}

Tensor op_attn_prefill(const Tensor& q8, const Tensor& tpos, const Tensor& kpool,
                       const Tensor& vpool, const Tensor& table, const Tensor& valid,
                       int64_t S_past) {
  rank(q8, 4, "attn_prefill");
  const int64_t B = q8.size(0), n_q = q8.size(1), T = q8.size(2), n_kv = kpool.size(1);
  Tensor out = empty({B, T, n_q * 128}, at::kLong, q8);
  const Tensor qc = q8.contiguous(), tc = tpos.contiguous(), v = valid.view(at::kByte);
  DI_RUN(detllm_attn_prefill, ptr<int8_t>(qc), i64(tc), ptr<int8_t>(kpool), ptr<int8_t>(vpool),
         ptr<int32_t>(table), (int)table.size(1), ptr<uint8_t>(v), valid.size(1), (int)B, (int)T,
         (int)S_past, (int)n_q, (int)n_kv, ptr<int64_t>(out));
  return out;
}

// Slots from which attn_decode cuts a row into chunks, G query heads per kv
// head. A block per (row, kv head) leaves CUs idle when pairs are few; a chunk
// block sums its row's whole denominator for each of its heads, so more heads
// need longer rows, and more pairs (whose blocks fill the chip) longer ones
// still. us per call, one block / chunks:
//   pairs <= 64, G = 2: 768 slots 13.5 / 12.3, 1024 16.5 / 12.4, 4096 56 / 24;
//     G = 4: 768 16.0 / 17.3, 896 18.2 / 17.7, 1024 19.1 / 17.7
//   65 to 128 pairs, G = 2: 768 13.5 / 14.5, 1024 16.4 / 16.6, 1152 19 / 18.5,
//     1280 20.4 / 18.2; G = 4: 1152 22 / 25, 1408 27 / 27, 1536 28 / 28
//   G = 8: 768 19 / 27, 1536 30 / 31; from 1537 slots on the one block's scores
//     (32 bytes a slot) are past its 48 KiB of LDS: 40 / 33
// More than 128 pairs take one block at any length. At G = 2 that is the better
// form to about 2048 slots only: 192 pairs 1024 slots 18.8 / 21.9, 2048 32 / 30,
// 4096 58 / 42; 256 pairs 19.2 / 23.2, 32.5 / 32.5, 60 / 54.
int64_t split_from(int64_t G, int64_t pairs) {
  if (pairs > 128) return INT64_MAX;
  if (G > 4) return 1537;
  if (G > 2) return pairs <= 64 ? 896 : 1536;
  return pairs <= 64 ? 768 : 1152;
}

Tensor op_attn_decode(const Tensor& q8, const Tensor& tpos, const Tensor& kpool,
                      const Tensor& vpool, const Tensor& table, const Tensor& valid, int64_t S,
                      const Tensor& err) {
  const int64_t B = q8.size(0), n_q = q8.size(1), n_kv = kpool.size(1);
  TORCH_CHECK_VALUE(n_kv > 0, "attn_decode: no kv heads");
  const int64_t G = n_q / n_kv;
  Tensor out = empty({B, n_q * 128}, at::kLong, q8);
  const Tensor qc = q8.contiguous(), tc = tpos.contiguous(), v = valid.view(at::kByte);
  if (B > 0 && S >= split_from(G, B * n_kv)) {
    int chunk = 0, ns = 0;
    check(detllm_attn_split_plan((int)B, (int)S, (int)n_q, (int)n_kv, &chunk, &ns),
          "detllm_attn_split_plan");
    const Tensor scores = empty({B, n_q, (int64_t)ns * chunk}, at::kInt, q8);
    const Tensor cmax = empty({B, n_q, ns}, at::kInt, q8);
    DI_RUN(detllm_attn_decode_split_sum, ptr<int8_t>(qc), i64(tc), ptr<int8_t>(kpool),
           ptr<int8_t>(vpool), ptr<int32_t>(table), (int)table.size(1), ptr<uint8_t>(v),
           valid.size(1), (int)B, (int)S, (int)n_q, (int)n_kv, nullptr, chunk,
           ptr<int32_t>(scores), ptr<int32_t>(cmax), ptr<int64_t>(out), ptr<int32_t>(err));
    mutated(err);
    return out;
  }
  const int64_t Spad = (S + 15) / 16 * 16;
  OptTensor scratch;
  if (G * Spad * 4 > 48 * 1024) scratch = empty({B, n_q, Spad}, at::kInt, q8);
  DI_RUN(detllm_attn_decode, ptr<int8_t>(qc), i64(tc), ptr<int8_t>(kpool), ptr<int8_t>(vpool),
         ptr<int32_t>(table), (int)table.size(1), ptr<uint8_t>(v), valid.size(1), (int)B, (int)S,
         (int)n_q, (int)n_kv, nullptr, ptr<int32_t>(scratch), ptr<int64_t>(out), ptr<int32_t>(err));
  mutated(err);
  return out;
}

}  // namespace

TORCH_LIBRARY_IMPL(detllm_rocm, CUDA, m) {
  m.impl("int_gemm", &op_int_gemm);
  m.impl("isqrt_i64", &op_isqrt);
  m.impl("ilog2_i64", &op_ilog2);
  m.impl("greedy_pick", &op_greedy_pick);
  m.impl("embed_normq", &op_embed_normq);
  m.impl("norm_quant", &op_norm_quant);
  m.impl("residual_normq", &op_residual_normq);
  m.impl("swiglu_quant", &op_swiglu_quant);
  m.impl("merge_rowcol", &op_merge_rowcol);
  m.impl("qkv_epilogue", &op_qkv_epilogue);
  m.impl("attn_prefill", &op_attn_prefill);
  m.impl("attn_decode", &op_attn_decode);
}

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&MODULE); }
