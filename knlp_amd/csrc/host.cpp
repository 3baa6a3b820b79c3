// CPython extension knlp_amd._host: the host side of the hot operators.
//
// A decode call of a small batch runs about 9 us on the GPU; checking two
// planes, filling their structs, planning, sizing the workspace and
// marshalling 27 arguments through ctypes took 23 us of Python per call.
// This module does the same from the tensors themselves: the operators of
// knlp_amd.ops pass their tensors and flags, and it validates them (the
// messages are those of ops), allocates the workspace and the output with
// torch's allocator and calls the C ABI (include/knlp_int4kv.h) on the current
// stream.  The GIL is released around allocation and launches, as ctypes does.
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <optional>
#include <string>

#include "../../include/knlp_int4kv.h"

namespace {

using OptTensor = std::optional<at::Tensor>;

at::Tensor tensor(PyObject* o, const char* what) {
  TORCH_CHECK_TYPE(THPVariable_Check(o), what, " must be a tensor");
  return THPVariable_Unpack(o);
}

OptTensor opt_tensor(PyObject* o, const char* what) {
  if (o == Py_None) return std::nullopt;
  return tensor(o, what);
}

int64_t integer(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}

double real(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw python_error();
  return v;
}

void require_device(const OptTensor& t) {
  TORCH_CHECK_VALUE(!t || t->is_cuda(),
                    "knlp_amd ops need device tensors (the HIP path has no CPU fallback)");
}

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

// A negative status as the Python exception the reference raises for the same
// misuse (ValueError for shapes, dtypes and arguments).
void check_status(int64_t status, const char* what) {
  if (status >= 0) return;
  const char* msg = knlp_status_string(static_cast<int>(status));
  TORCH_CHECK(status != KNLP_ERR_LAUNCH, what, ": ", msg);
  TORCH_CHECK_VALUE(false, what, ": ", msg, " (status ", status, ")");
}

// One side's cache with what the C ABI's struct does not carry (the tensors
// and their shapes).
struct Plane {
  at::Tensor data;
  OptTensor scales, zeros;
  knlp_kv_plane p{};
};

std::string shape_of(const at::Tensor& t) {
  std::string s = "[";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + "]";
}

Plane make_plane(PyObject* const* a, bool on_device) {
  Plane r;
  r.data = tensor(a[0], "cache");
  r.scales = opt_tensor(a[1], "scales");
  r.zeros = opt_tensor(a[2], "zeros");
  const int64_t fmt = integer(a[3]);
  TORCH_CHECK_VALUE(fmt >= KNLP_KV_INT4_SYM && fmt <= KNLP_KV_FP16, "unknown cache format");
  const at::ScalarType want = fmt == KNLP_KV_FP16 ? at::kHalf
                              : fmt == KNLP_KV_INT8_SYM ? at::kChar : at::kByte;
  if (on_device) {
    require_device(r.data);
    require_device(r.scales);
    if (fmt == KNLP_KV_INT4_ASYM) require_device(r.zeros);
  }
  TORCH_CHECK_VALUE(r.data.scalar_type() == want, "cache dtype ", r.data.scalar_type(),
                    " does not match format (want ", want, ")");
  TORCH_CHECK_VALUE(r.data.dim() == 4 && r.data.stride(3) == 1,
                    "cache must be [num_blocks, block_size, num_heads, packed_dim] "
                    "with a contiguous last axis");
  r.p.data = r.data.data_ptr();
  r.p.stride_block = r.data.stride(0);
  r.p.stride_page = r.data.stride(1);
  r.p.stride_head = r.data.stride(2);
  r.p.format = static_cast<int32_t>(fmt);
  r.p.group_size = static_cast<int32_t>(integer(a[4]));
  if (fmt != KNLP_KV_FP16) {
    TORCH_CHECK_VALUE(r.scales && r.scales->scalar_type() == at::kHalf && r.scales->dim() == 4 &&
                          r.scales->stride(3) == 1,
                      "scales must be fp16 [num_blocks, block_size, num_heads, num_groups]");
    r.p.scales = r.scales->data_ptr();
    r.p.s_stride_block = r.scales->stride(0);
    r.p.s_stride_page = r.scales->stride(1);
    r.p.s_stride_head = r.scales->stride(2);
  } else {
    r.scales.reset();
  }
  if (fmt == KNLP_KV_INT4_ASYM) {
    TORCH_CHECK_VALUE(r.zeros && r.zeros->scalar_type() == at::kHalf && r.zeros->dim() == 4 &&
                          r.zeros->stride(3) == 1,
                      "asymmetric mode needs fp16 zero-points shaped like the scales");
    r.p.zeros = r.zeros->data_ptr();
    r.p.z_stride_block = r.zeros->stride(0);
    r.p.z_stride_page = r.zeros->stride(1);
    r.p.z_stride_head = r.zeros->stride(2);
  } else {
    r.zeros.reset();
  }
  return r;
}

// ValueError unless the cache holds `heads` heads of `d` elements and its
// scales / zero-points cover every (block, slot, head, group) of it: the
// kernels index these tensors through their strides without bounds checks.
void check_plane(const Plane& r, const char* name, int64_t heads, int64_t d) {
  const bool int4 = r.p.format == KNLP_KV_INT4_SYM || r.p.format == KNLP_KV_INT4_ASYM;
  const int64_t packed = int4 ? d / 2 : d;
  TORCH_CHECK_VALUE(r.data.size(2) >= heads && r.data.size(3) >= packed, name, " cache ",
                    shape_of(r.data), " holds fewer than ", heads, " heads of ", packed, " ",
                    r.p.format != KNLP_KV_FP16 ? "bytes" : "halves");
  if (r.p.format == KNLP_KV_FP16) return;
  const int64_t ng = r.p.group_size > 0 ? d / r.p.group_size : 0;
  const auto covers = [&](const OptTensor& t, const char* what) {
    if (!t) return;
    TORCH_CHECK_VALUE(t->size(0) >= r.data.size(0) && t->size(1) >= r.data.size(1) &&
                          t->size(2) >= heads && t->size(3) >= ng,
                      name, " ", what, " ", shape_of(*t), " do not cover a cache of ",
                      shape_of(r.data), " with ", ng, " groups per head");
  };
  covers(r.scales, "scales");
  covers(r.zeros, "zeros");
}

int32_t src_dtype(const at::Tensor& t) {
  const auto s = t.scalar_type();
  TORCH_CHECK_VALUE(s == at::kHalf || s == at::kBFloat16, "key/value dtype ", s,
                    " not supported (fp16 or bf16)");
  TORCH_CHECK_VALUE(t.dim() == 3 && t.stride(2) == 1,
                    "key/value must be [num_tokens, num_heads, head_size], last axis contiguous");
  return s == at::kHalf ? KNLP_DT_F16 : KNLP_DT_BF16;
}

int32_t slot_dtype(const at::Tensor& t) {
  const auto s = t.scalar_type();
  TORCH_CHECK_VALUE(s == at::kLong || s == at::kInt, "slot_mapping must be int32 or int64");
  return s == at::kLong ? KNLP_DT_I64 : KNLP_DT_I32;
}

const void* ptr(const OptTensor& t) { return t ? t->data_ptr() : nullptr; }
int64_t stride(const OptTensor& t, int64_t i) { return t ? t->stride(i) : 0; }

void want_args(Py_ssize_t got, Py_ssize_t want, const char* what) {
  TORCH_CHECK_TYPE(got == want, what, " takes ", want, " arguments, got ", got);
}

// plane(data, scales, zeros, format, group_size, address): validate the tensors
// and fill the knlp_kv_plane at `address`.
PyObject* py_plane(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 6, "plane");
  const Plane r = make_plane(a, false);
  *reinterpret_cast<knlp_kv_plane*>(static_cast<uintptr_t>(integer(a[5]))) = r.p;
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// check_plane(data, scales, zeros, format, group_size, name, heads, head_size)
PyObject* py_check_plane(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 8, "check_plane");
  const char* name = PyUnicode_AsUTF8(a[5]);
  if (name == nullptr) throw python_error();
  check_plane(make_plane(a, false), name, integer(a[6]), integer(a[7]));
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// append(key, value, *key plane (5), *value plane (5), slot_mapping, clip_ratio,
// block_size); a side whose rows are None has no plane (its five are ignored).
PyObject* py_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 15, "append");
  const OptTensor key = opt_tensor(a[0], "key"), value = opt_tensor(a[1], "value");
  at::Tensor slots = tensor(a[12], "slot_mapping");
  require_device(key);
  require_device(value);
  require_device(slots);
  TORCH_CHECK_VALUE(key || value, "append needs key or value");
  Plane kp, vp;
  if (key) kp = make_plane(a + 2, true);
  if (value) vp = make_plane(a + 7, true);
  const at::Tensor& src = key ? *key : *value;
  const int32_t dt = src_dtype(src);
  if (key && value) {
    src_dtype(*value);                     // its own layout checks too
    TORCH_CHECK_VALUE(key->scalar_type() == value->scalar_type(),
                      "key and value must share a dtype");
    TORCH_CHECK_VALUE(key->sizes() == value->sizes(),
                      "key and value must have the same shape");
  }
  slots = slots.contiguous();
  const int64_t tokens = src.size(0), heads = src.size(1), d = src.size(2);
  TORCH_CHECK_VALUE(slots.numel() >= tokens, "slot_mapping shorter than num_tokens");
  if (key) check_plane(kp, "key", heads, d);
  if (value) check_plane(vp, "value", heads, d);
  TORCH_CHECK_VALUE(!key || !value || kp.data.size(1) == vp.data.size(1),
                    "key and value caches have different block sizes");
  const int32_t sdt = slot_dtype(slots);
  const float clip = static_cast<float>(real(a[13]));
  const int32_t block_size = static_cast<int32_t>(integer(a[14]));
  int st;
  {
    pybind11::gil_scoped_release nogil;
    st = knlp_kv_append(ptr(key), ptr(value), dt, tokens, static_cast<int32_t>(heads),
                        static_cast<int32_t>(d), stride(key, 0), stride(key, 1), stride(value, 0),
                        stride(value, 1), key ? &kp.p : nullptr, value ? &vp.p : nullptr,
                        slots.data_ptr(), sdt, block_size, clip, stream());
  }
  check_status(st, "knlp_kv_append");
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// decode(query, *key plane (5), *value plane (5), block_size, block_table,
// seq_lens, num_kv_heads, head_size, scale or None, split_tokens (-1: the
// library's schedule), total_context, key, value, slot_mapping or None,
// clip_ratio) -> output
PyObject* py_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 23, "decode");
  const at::Tensor query = tensor(a[0], "query");
  const Plane kp = make_plane(a + 1, true), vp = make_plane(a + 6, true);
  const int32_t block_size = static_cast<int32_t>(integer(a[11]));
  at::Tensor table = tensor(a[12], "block_table"), lens = tensor(a[13], "seq_lens");
  const int64_t hkv = integer(a[14]), d = integer(a[15]);
  const int64_t total = integer(a[18]);
  int64_t split = integer(a[17]);
  const OptTensor key = opt_tensor(a[19], "key"), value = opt_tensor(a[20], "value");
  OptTensor slots = opt_tensor(a[21], "slot_mapping");
  for (const OptTensor& t : {OptTensor(query), OptTensor(table), OptTensor(lens), key, value, slots})
    require_device(t);
  const auto qs = query.scalar_type();
  TORCH_CHECK_VALUE(qs == at::kHalf || qs == at::kBFloat16, "query dtype ", qs,
                    " not supported (fp16 or bf16)");
  TORCH_CHECK_VALUE(query.dim() == 3 && query.stride(2) == 1 && query.size(2) == d,
                    "query must be [num_seqs, num_heads, head_size], last axis contiguous");
  const int64_t seqs = query.size(0), hq = query.size(1);
  TORCH_CHECK_VALUE(hkv > 0 && hq % hkv == 0, "num_heads must be a multiple of num_kv_heads");
  if (seqs == 0) return THPVariable_Wrap(at::empty_like(query));
  TORCH_CHECK_VALUE(table.dim() == 2, "block_table must be [num_seqs, max_blocks]");
  if (table.scalar_type() != at::kInt) table = table.to(at::kInt);
  if (table.stride(1) != 1) table = table.contiguous();
  if (lens.scalar_type() != at::kInt || !lens.is_contiguous())
    lens = lens.to(at::kInt).contiguous();
  check_plane(kp, "key", hkv, d);
  check_plane(vp, "value", hkv, d);
  TORCH_CHECK_VALUE(kp.data.size(1) == vp.data.size(1),
                    "key and value caches have different block sizes");
  const int64_t max_context = table.size(1) * block_size;
  if (split < 0) {
    split = knlp_kv_decode_schedule_planes(
        static_cast<int32_t>(seqs), static_cast<int32_t>(hkv), static_cast<int32_t>(hq),
        static_cast<int32_t>(d), static_cast<int32_t>(max_context), total, &kp.p, &vp.p,
        block_size);
    check_status(split, "knlp_kv_decode_schedule_planes");
  }
  const int64_t ws_bytes = knlp_kv_decode_workspace_bytes(
      static_cast<int32_t>(seqs), static_cast<int32_t>(hq), static_cast<int32_t>(d),
      static_cast<int32_t>(max_context), static_cast<int32_t>(split));
  check_status(ws_bytes, "knlp_kv_decode_workspace_bytes");
  const float scale = a[16] == Py_None ? static_cast<float>(1.0 / std::sqrt(static_cast<double>(d)))
                                       : static_cast<float>(real(a[16]));
  const int32_t dt = qs == at::kHalf ? KNLP_DT_F16 : KNLP_DT_BF16;
  TORCH_CHECK_VALUE(slots || (!key && !value), "key and value need a slot_mapping");
  int32_t src = 0, sdt = 0;
  const float clip = static_cast<float>(real(a[22]));
  if (slots) {
    TORCH_CHECK_VALUE(key || value, "append needs key or value");
    for (const OptTensor& t : {key, value})
      TORCH_CHECK_VALUE(!t || (t->dim() == 3 && t->size(0) >= seqs && t->stride(2) == 1 &&
                               t->size(1) == hkv && t->size(2) == d),
                        "key/value must be [num_seqs, num_kv_heads, head_size], "
                        "last axis contiguous");
    TORCH_CHECK_VALUE(!key || !value || key->scalar_type() == value->scalar_type(),
                      "key and value must share a dtype");
    slots = slots->contiguous();
    TORCH_CHECK_VALUE(slots->numel() >= seqs, "slot_mapping shorter than num_seqs");
    src = src_dtype(key ? *key : *value);
    sdt = slot_dtype(*slots);
  }
  at::Tensor out;
  int st;
  {
    pybind11::gil_scoped_release nogil;
    const at::Tensor ws = at::empty({(ws_bytes + 3) / 4}, query.options().dtype(at::kFloat));
    out = at::empty_like(query);
    if (slots)
      st = knlp_kv_append_decode(
          query.data_ptr(), dt, query.stride(0), query.stride(1), static_cast<int32_t>(seqs),
          static_cast<int32_t>(hq), static_cast<int32_t>(hkv), static_cast<int32_t>(d), ptr(key),
          ptr(value), src, stride(key, 0), stride(key, 1), stride(value, 0), stride(value, 1),
          slots->data_ptr(), sdt, clip, &kp.p, &vp.p, table.data_ptr<int32_t>(), table.stride(0),
          lens.data_ptr<int32_t>(), block_size, static_cast<int32_t>(max_context), scale,
          static_cast<int32_t>(split), ws.data_ptr(), ws_bytes, out.data_ptr(), dt, out.stride(0),
          out.stride(1), stream());
    else
      st = knlp_kv_decode(
          query.data_ptr(), dt, query.stride(0), query.stride(1), static_cast<int32_t>(seqs),
          static_cast<int32_t>(hq), static_cast<int32_t>(hkv), static_cast<int32_t>(d), &kp.p,
          &vp.p, table.data_ptr<int32_t>(), table.stride(0), lens.data_ptr<int32_t>(), block_size,
          static_cast<int32_t>(max_context), scale, static_cast<int32_t>(split), ws.data_ptr(),
          ws_bytes, out.data_ptr(), dt, out.stride(0), out.stride(1), stream());
  }
  check_status(st, slots ? "knlp_kv_append_decode" : "knlp_kv_decode");
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"plane", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_plane)), METH_FASTCALL, nullptr},
    {"check_plane", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_check_plane)),
     METH_FASTCALL, nullptr},
    {"append", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_append)), METH_FASTCALL,
     nullptr},
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_decode)), METH_FASTCALL,
     nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }
