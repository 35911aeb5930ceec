// Descriptor building for kvx_amd/paged.py: write() and gather() fill the
// kvx_abi.h structs of a call from torch tensors and call the library's entry
// point.  Filling them field by field through ctypes bound every small call:
// on the MI355X host a gather of eight short sequences took 19.3 us, 4.8 us
// through this module (of which the launch is about 3).
//
// Both return the kvx_status_t, or None for anything that the ctypes helpers
// must decide (an argument that is not a plain tensor, a dtype outside the
// ABI's, more than five axes, sizes past 32 bits): the caller then takes
// those helpers, which raise what they always raised.  The entry points are
// passed as addresses, so that the module calls whichever libkvx_amd.so the
// process has loaded.  A plain CPython module rather than a torch operator:
// the calls stay outside torch's dispatcher, as ctypes calls are.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/autograd/python_variable.h>

#include "kvx_ext.h"
#include "kvx_paged_kv.h"

namespace {

kvx_dtype_t dtype_of(at::ScalarType t) {
  switch (t) {
    case at::ScalarType::Half: return KVX_DTYPE_F16;
    case at::ScalarType::BFloat16: return KVX_DTYPE_BF16;
    case at::ScalarType::Float: return KVX_DTYPE_F32;
    case at::ScalarType::Float8_e4m3fn: return KVX_DTYPE_F8_E4M3;
    case at::ScalarType::Float8_e5m2: return KVX_DTYPE_F8_E5M2;
    case at::ScalarType::Int: return KVX_DTYPE_S32;
    case at::ScalarType::Long: return KVX_DTYPE_S64;
    default: return KVX_DTYPE_INVALID;
  }
}

// The argument's tensor, or null: exactly torch.Tensor (or Parameter), with
// storage of its own, so that no subclass override is passed by.
const at::Tensor *plain(PyObject *o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  if (!t.defined() || t.layout() != at::kStrided || !t.has_storage() || t.is_neg() || t.is_conj())
    return nullptr;
  return &t;
}

bool fits32(int64_t v) { return v >= 0 && v <= 0xFFFFFFFFll; }

// paged.tensor_desc
bool describe(kvx_tensor_desc_t *d, const at::Tensor &t, int layout) {
  const kvx_dtype_t dt = dtype_of(t.scalar_type());
  if (dt == KVX_DTYPE_INVALID || t.dim() > KVX_MAX_TENSOR_DIMS) return false;
  d->size = sizeof(kvx_tensor_desc_t);
  d->dtype = dt;
  d->layout = static_cast<kvx_layout_t>(layout);
  d->memory = t.is_cuda() ? KVX_MEMORY_DEVICE : KVX_MEMORY_HOST;
  d->ndim = static_cast<uint32_t>(t.dim());
  const auto sizes = t.sizes();
  const auto strides = t.strides();
  for (size_t i = 0; i < sizes.size(); ++i) {
    d->shape[i] = sizes[i];
    d->stride[i] = strides[i];
  }
  d->data = t.data_ptr();
  return true;
}

// paged.scale_desc_of: granularity -1 for a tensor that is a per-tensor scale.
bool describe_scale(kvx_scale_desc_t *d, const at::Tensor &t, int granularity) {
  d->size = sizeof(kvx_scale_desc_t);
  d->dtype = KVX_DTYPE_F32;
  d->granularity = granularity < 0 ? KVX_SCALE_PER_TENSOR
                                   : static_cast<kvx_scale_granularity_t>(granularity);
  d->ndim = 1;
  d->shape[0] = 1;
  d->stride[0] = 1;
  if (granularity >= 0 && t.dim() > 0) {
    if (t.dim() > KVX_MAX_TENSOR_DIMS) return false;
    d->ndim = static_cast<uint32_t>(t.dim());
    for (int64_t i = 0; i < t.dim(); ++i) {
      d->shape[i] = t.size(i);
      d->stride[i] = t.stride(i);
    }
  }
  d->data = t.data_ptr();
  return true;
}

// Arguments in order, each a plain tensor or number; `ok` turns false at the
// first that is not.
struct Args {
  PyObject *const *v;
  Py_ssize_t n;
  Py_ssize_t at = 0;
  bool ok = true;

  PyObject *next() {
    if (at >= n) {
      ok = false;
      return Py_None;
    }
    return v[at++];
  }
  const at::Tensor *tensor() {
    const at::Tensor *t = plain(next());
    if (t == nullptr) ok = false;
    return t;
  }
  const at::Tensor *tensor_or_none() {
    PyObject *o = next();
    if (o == Py_None) return nullptr;
    const at::Tensor *t = plain(o);
    if (t == nullptr) ok = false;
    return t;
  }
  int64_t number() {
    PyObject *o = next();
    if (!ok || !PyLong_Check(o)) {
      ok = false;
      return 0;
    }
    const int64_t x = PyLong_AsLongLong(o);
    if (x == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      ok = false;
    }
    return x;
  }
  uint32_t number32() {
    const int64_t x = number();
    if (!fits32(x)) ok = false;
    return static_cast<uint32_t>(x);
  }
  template <class F>
  F function() {
    PyObject *o = next();
    void *p = ok && PyLong_Check(o) ? PyLong_AsVoidPtr(o) : nullptr;
    if (p == nullptr) {
      PyErr_Clear();
      ok = false;
    }
    return reinterpret_cast<F>(p);
  }
};

// (key_cache, value_cache, k_layout, v_layout, num_blocks, block_size, heads,
// head_dim) of a PagedCache.
bool cache_of(Args &a, kvx_cache_desc_t *c) {
  const at::Tensor *k = a.tensor();
  const at::Tensor *v = a.tensor();
  const int64_t kl = a.number();
  const int64_t vl = a.number();
  c->size = sizeof(kvx_cache_desc_t);
  c->num_blocks = a.number32();
  c->block_size = a.number32();
  c->num_kv_heads = a.number32();
  c->head_dim = a.number32();
  return a.ok && describe(&c->k, *k, static_cast<int>(kl)) &&
         describe(&c->v, *v, static_cast<int>(vl));
}

// The stream argument: a handle, or None for torch's current stream.
void *stream_of(Args &a) {
  PyObject *o = a.next();
  if (o == Py_None)
    return reinterpret_cast<void *>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream());
  void *p = PyLong_Check(o) ? PyLong_AsVoidPtr(o) : nullptr;
  if (p == nullptr && PyErr_Occurred()) {
    PyErr_Clear();
    a.ok = false;
  }
  if (!PyLong_Check(o)) a.ok = false;
  return p;
}

template <class F>
PyObject *status_of(F &&call) {
  kvx_status_t st;
  Py_BEGIN_ALLOW_THREADS
  st = call();
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(static_cast<long>(st));
}

typedef kvx_status_t (*WriteFn)(const kvx_cache_desc_t *, const kvx_write_desc_t *, void *);
typedef kvx_status_t (*PrefillFn)(const kvx_cache_desc_t *, const kvx_write_desc_t *, int32_t,
                                  void *);
typedef kvx_status_t (*GatherFn)(const kvx_cache_desc_t *, const kvx_gather_desc_t *, void *);
typedef kvx_status_t (*DequantFn)(const kvx_cache_desc_t *, const kvx_gather_desc_t *,
                                  const kvx_scale_desc_t *, const kvx_scale_desc_t *, void *);

// write(fn, tokens_per_seq (None: fn takes none), stream, cache..., key, value,
//       slots, k_scale, k_granularity, v_scale, v_granularity)
PyObject *host_write(Args a) {
  void *fn = a.function<void *>();
  const bool prefill = a.at < a.n && a.v[a.at] != Py_None;
  int64_t per_seq = 0;
  if (prefill) per_seq = a.number();
  else a.next();
  void *stream = stream_of(a);
  kvx_cache_desc_t c{};
  if (!a.ok || !cache_of(a, &c)) Py_RETURN_NONE;
  kvx_write_desc_t w{};
  const at::Tensor *key = a.tensor();
  const at::Tensor *value = a.tensor();
  const at::Tensor *slots = a.tensor();
  const at::Tensor *ks = a.tensor_or_none();
  const int64_t kg = a.number();
  const at::Tensor *vs = a.tensor_or_none();
  const int64_t vg = a.number();
  if (!a.ok || a.at != a.n || key->dim() != 3 || !fits32(key->size(0)) ||
      !fits32(key->size(1)) || !fits32(key->size(2)) || !fits32(slots->numel()) ||
      per_seq > 0x7FFFFFFF || per_seq < -0x80000000ll)
    Py_RETURN_NONE;
  w.size = sizeof(kvx_write_desc_t);
  w.io.size = sizeof(kvx_kv_io_desc_t);
  const kvx_dtype_t sdt = dtype_of(slots->scalar_type());
  if (!describe(&w.io.key, *key, KVX_LAYOUT_BLOCK_CUSTOM) ||
      !describe(&w.io.value, *value, KVX_LAYOUT_BLOCK_CUSTOM) || sdt == KVX_DTYPE_INVALID)
    Py_RETURN_NONE;
  w.io.num_tokens = static_cast<uint32_t>(key->size(0));
  w.io.num_kv_heads = static_cast<uint32_t>(key->size(1));
  w.io.head_dim = static_cast<uint32_t>(key->size(2));
  w.slots.size = sizeof(kvx_slot_mapping_t);
  w.slots.dtype = sdt;
  w.slots.token_count = static_cast<uint32_t>(slots->numel());
  w.slots.invalid_slot = -1;
  w.slots.slots = slots->data_ptr();
  if (ks && !describe_scale(&w.k_scale_desc, *ks, static_cast<int>(kg))) Py_RETURN_NONE;
  if (vs && !describe_scale(&w.v_scale_desc, *vs, static_cast<int>(vg))) Py_RETURN_NONE;
  if (prefill)
    return status_of([&] {
      return reinterpret_cast<PrefillFn>(fn)(&c, &w, static_cast<int32_t>(per_seq), stream);
    });
  return status_of([&] { return reinterpret_cast<WriteFn>(fn)(&c, &w, stream); });
}

// gather(fn, stream, cache..., key_out, value_out, table, indptr, primary,
//        secondary, bytes_per_block, lens, max_seq_len, k_scale,
//        k_granularity, v_scale, v_granularity): indptr set for a RAGGED
//        table (`table` its indices), primary for a KV_OFFSETS one (`table`
//        its offsets); with scales fn is the dequantizing gather.
PyObject *host_gather(Args a) {
  void *fn = a.function<void *>();
  void *stream = stream_of(a);
  kvx_cache_desc_t c{};
  if (!a.ok || !cache_of(a, &c)) Py_RETURN_NONE;
  const at::Tensor *ko = a.tensor();
  const at::Tensor *vo = a.tensor();
  const at::Tensor *table = a.tensor();
  const at::Tensor *indptr = a.tensor_or_none();
  const at::Tensor *primary = a.tensor_or_none();
  const at::Tensor *secondary = a.tensor_or_none();
  const uint32_t bytes_per_block = a.number32();
  const at::Tensor *lens = a.tensor();
  const uint32_t width = a.number32();
  const at::Tensor *ks = a.tensor_or_none();
  const int64_t kg = a.number();
  const at::Tensor *vs = a.tensor_or_none();
  const int64_t vg = a.number();
  if (!a.ok || a.at != a.n || (ks == nullptr) != (vs == nullptr) || ko->dim() != 4 ||
      !fits32(ko->size(2)) || !fits32(ko->size(3)) || !fits32(lens->numel()))
    Py_RETURN_NONE;
  kvx_gather_desc_t g{};
  g.size = sizeof(kvx_gather_desc_t);
  g.io.size = sizeof(kvx_kv_io_desc_t);
  const kvx_dtype_t tdt = dtype_of(table->scalar_type());
  const kvx_dtype_t ldt = dtype_of(lens->scalar_type());
  if (!describe(&g.io.key, *ko, KVX_LAYOUT_BLOCK_CUSTOM) ||
      !describe(&g.io.value, *vo, KVX_LAYOUT_BLOCK_CUSTOM) || tdt == KVX_DTYPE_INVALID ||
      ldt == KVX_DTYPE_INVALID)
    Py_RETURN_NONE;
  kvx_block_table_t &t = g.block_table;
  t.size = sizeof(kvx_block_table_t);
  t.index_dtype = tdt;
  t.beam_width = 1;
  t.indices = table->data_ptr();
  if (indptr != nullptr) {
    const kvx_dtype_t pdt = dtype_of(indptr->scalar_type());
    if (pdt == KVX_DTYPE_INVALID || indptr->numel() < 1 || !fits32(indptr->numel()) ||
        !fits32(table->numel()))
      Py_RETURN_NONE;
    t.format = KVX_BLOCK_TABLE_RAGGED;
    t.indptr_dtype = pdt;
    t.seq_count = static_cast<uint32_t>(indptr->numel() - 1);
    t.max_blocks_per_seq = 1;
    t.indptr = indptr->data_ptr();
    t.indices_count = static_cast<uint32_t>(table->numel());
    t.indptr_count = static_cast<uint32_t>(indptr->numel());
  } else if (primary != nullptr) {
    if (table->dim() != 4 || table->size(2) != 2 || tdt != KVX_DTYPE_S32 ||
        !fits32(table->size(0)) || !fits32(table->size(1)) || !fits32(table->size(3)) ||
        !fits32(table->numel()))
      Py_RETURN_NONE;
    t.format = KVX_BLOCK_TABLE_KV_OFFSETS;
    t.seq_count = static_cast<uint32_t>(table->size(0));
    t.beam_width = static_cast<uint32_t>(table->size(1));
    t.max_blocks_per_seq = static_cast<uint32_t>(table->size(3));
    t.indices_count = static_cast<uint32_t>(table->numel());
    t.flags = KVX_BLOCK_TABLE_FLAG_KVCACHEINDEX;
    c.pool.size = sizeof(kvx_pool_desc_t);
    c.pool.memory = primary->is_cuda() ? KVX_MEMORY_DEVICE : KVX_MEMORY_HOST;
    c.pool.bytes_per_block = bytes_per_block;
    c.pool.primary = primary->data_ptr();
    c.pool.secondary = secondary ? secondary->data_ptr() : nullptr;
  } else {
    if (table->dim() != 2 || !fits32(table->size(0)) || !fits32(table->size(1)) ||
        !fits32(table->numel()))
      Py_RETURN_NONE;
    t.format = KVX_BLOCK_TABLE_PACKED;
    t.seq_count = static_cast<uint32_t>(table->size(0));
    t.max_blocks_per_seq = static_cast<uint32_t>(table->size(1));
    t.indices_count = static_cast<uint32_t>(table->numel());
  }
  if ((uint64_t)t.seq_count * width > 0xFFFFFFFFull) Py_RETURN_NONE;
  g.io.num_tokens = t.seq_count * width;
  g.io.num_kv_heads = static_cast<uint32_t>(ko->size(2));
  g.io.head_dim = static_cast<uint32_t>(ko->size(3));
  g.seq_lens.size = sizeof(kvx_seq_lens_t);
  g.seq_lens.dtype = ldt;
  g.seq_lens.seq_count = static_cast<uint32_t>(lens->numel());
  g.seq_lens.lengths = lens->data_ptr();
  g.max_seq_len = width;
  if (ks == nullptr)
    return status_of([&] { return reinterpret_cast<GatherFn>(fn)(&c, &g, stream); });
  kvx_scale_desc_t ksd{}, vsd{};
  if (!describe_scale(&ksd, *ks, static_cast<int>(kg)) ||
      !describe_scale(&vsd, *vs, static_cast<int>(vg)))
    Py_RETURN_NONE;
  return status_of([&] { return reinterpret_cast<DequantFn>(fn)(&c, &g, &ksd, &vsd, stream); });
}

template <PyObject *(*F)(Args)>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
  try {
    return F(Args{args, n});
  } catch (...) {
    // torch refuses a tensor (no data to point at, say): the ctypes helpers
    // raise for it
    Py_RETURN_NONE;
  }
}

PyMethodDef kMethods[] = {
    {"write", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<host_write>)),
     METH_FASTCALL, nullptr},
    {"gather", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<host_gather>)),
     METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_paged_host", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__paged_host(void) { return PyModule_Create(&kModule); }
