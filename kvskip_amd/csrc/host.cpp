// The operators' host side in native code (module kvskip_amd._host): argument checks, output
// allocation, the C ABI's argument blocks and the launches of kvskip_amd/ext.py, whose functions pass
// their arguments through and document them. Same checks, messages and results as the Python code this
// replaced; what bounds a small call is this path and not its kernels. Measured (eager calls one after
// another, us a call; before: checks in Python, ctypes blocks, torch.empty, the split rule scanned in
// Python): a decode of 200 tokens, whose kernel takes 6 us, 20.1 -> 7.9; B 1 at 32k 67.9 -> 25.7 (the
// kernels' time); single-pass V-skip at 64k 87.6 -> 41.5; four layers x 12 planner steps at 32k
// 6800 -> 1830.
// Nothing is kept from one call to the next but what bind() was given: the entry points' addresses and
// torch's function of the current stream.
#include <Python.h>

#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstring>
#include <stdexcept>
#include <string>
#include <vector>

#include "kvskip_amd.h"

namespace {

constexpr int64_t TILE = KVSKIP_BLOCK;

// ---- the library's entry points (addresses from the library that ext.py loaded)
struct Api {
  int (*decode)(const kvskip_attn_args*, int, int, void*);
  int (*decode_splits)(const kvskip_attn_args*, int, int, void*);
  int (*merge_splits)(const kvskip_attn_args*, int, int, void*);
  int (*pv)(const kvskip_attn_args*, void*);
  int (*vskip1)(const kvskip_attn_args*, void*);
  int (*pv_select)(const kvskip_attn_args*, const kvskip_select_args*, void*);
  int (*select)(const kvskip_select_args*, void*);
  int (*plan)(const kvskip_plan_args*, void*);
  int (*plan_scores)(const kvskip_plan_args*, void*);
  int (*update)(const kvskip_update_args*, void*);
  int (*merge_update)(const kvskip_attn_args*, const kvskip_update_args*, void*);
  int (*decode_splits_update)(const kvskip_attn_args*, const kvskip_update_args*, void*);
  int (*decode_splits_planned)(const kvskip_attn_args*, const kvskip_plan_args*, const kvskip_update_args*, void*);
  int64_t (*plan_part_floats)(int32_t, int32_t, int32_t, int32_t);
  const char* (*last_error)();
};
constexpr int N_API = sizeof(Api) / sizeof(void*);
Api api;
PyObject* raw_stream = nullptr;  // torch's function of a device index: its current stream's handle

// ---- arguments
[[noreturn]] void fail(const std::string& msg) { throw std::runtime_error(msg); }
inline void require(bool cond, const char* msg) {
  if (!cond) fail(msg);
}
struct PyErr {};  // a Python exception is set

const at::Tensor& tensor(PyObject* o, const char* name) {
  if (!THPVariable_Check(o)) fail(std::string(name) + " must be a tensor");
  return THPVariable_Unpack(o);
}
const at::Tensor* opt_tensor(PyObject* o, const char* name) { return o == Py_None ? nullptr : &tensor(o, name); }
int64_t integer(PyObject* o) {
  if (PyLong_Check(o)) {
    const int64_t v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw PyErr{};
    return v;
  }
  PyObject* n = PyNumber_Long(o);
  if (n == nullptr) throw PyErr{};
  const int64_t v = PyLong_AsLongLong(n);
  Py_DECREF(n);
  if (v == -1 && PyErr_Occurred()) throw PyErr{};
  return v;
}
int32_t int32(PyObject* o) {
  const int64_t v = integer(o);
  if (v < INT32_MIN || v > INT32_MAX) fail("integer argument out of range");
  return static_cast<int32_t>(v);
}
double real(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PyErr{};
  return v;
}
bool truth(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw PyErr{};
  return v != 0;
}
PyObject* item(PyObject* dict, const char* key) {
  PyObject* o = PyDict_GetItemString(dict, key);
  if (o == nullptr) {
    PyErr_SetString(PyExc_KeyError, key);
    throw PyErr{};
  }
  return o;
}
template <class S>
S* block(PyObject* o) {  // the address of a ctypes argument block
  return reinterpret_cast<S*>(static_cast<uintptr_t>(integer(o)));
}
void* ptr(const at::Tensor* t) { return t == nullptr ? nullptr : t->data_ptr(); }
PyObject* wrap(const at::Tensor& t) {
  if (t.defined()) return THPVariable_Wrap(t);
  Py_RETURN_NONE;
}
PyObject* list_of(std::initializer_list<at::Tensor> ts) {
  PyObject* l = PyList_New(static_cast<Py_ssize_t>(ts.size()));
  if (l == nullptr) throw PyErr{};
  Py_ssize_t i = 0;
  for (const at::Tensor& t : ts) PyList_SET_ITEM(l, i++, wrap(t));
  return l;
}

// Device guard and current stream of a launch; the launch itself runs without the interpreter lock.
template <class F>
void launch(const at::Device& dev, F&& f) {
  TORCH_CHECK_VALUE(dev.is_cuda(), "Expected a cuda device, but got: ", dev.str());
  c10::DeviceGuard guard(dev);
  PyObject* i = PyLong_FromLong(dev.index());
  PyObject* s = i != nullptr ? PyObject_CallOneArg(raw_stream, i) : nullptr;
  Py_XDECREF(i);
  if (s == nullptr) throw PyErr{};
  void* stream = PyLong_AsVoidPtr(s);
  Py_DECREF(s);
  if (stream == nullptr && PyErr_Occurred()) throw PyErr{};
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f(stream);
  Py_END_ALLOW_THREADS
  if (rc != 0) {
    const char* m = api.last_error();
    fail(m != nullptr && m[0] != '\0' ? std::string(m) : "kvskip_amd: error " + std::to_string(rc));
  }
}

bool is_bf16_cuda(const at::Tensor& t) { return t.is_cuda() && t.scalar_type() == at::kBFloat16; }
bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0; }
bool is(const at::Tensor& t, at::ScalarType ty) { return t.scalar_type() == ty && t.is_contiguous(); }
int64_t tiles(int64_t T) { return (T + TILE - 1) / TILE; }

void check_kv(const at::Tensor& t, const std::string& n) {
  if (!is_bf16_cuda(t)) fail(n + " must be a CUDA bf16 tensor");
  if (t.dim() != 4) fail(n + " must be [B, Hkv, T, D]");
  if (t.stride(3) != 1) fail(n + " must have a contiguous last dim");
  if (t.stride(2) % 8 != 0 || t.stride(1) % 8 != 0 || t.stride(0) % 8 != 0)
    fail(n + " strides must be multiples of 8 elements (16-byte rows)");
  if (!aligned16(t)) fail(n + " must be 16-byte aligned");
  if ((t.size(2) - 1) * t.stride(2) + t.size(3) >= (int64_t(1) << 30)) fail(n + ": one head's rows must span < 2 GiB");
}
void check_q(const at::Tensor& q) {
  require(is_bf16_cuda(q) && q.dim() == 3, "q must be CUDA bf16 [B, Hq, D]");
  require(q.stride(2) == 1 && q.stride(1) % 8 == 0 && q.stride(0) % 8 == 0 && aligned16(q),
          "q rows must be 16-byte aligned");
}
void check_f32(const at::Tensor& t, const char* n) {
  if (!(t.is_cuda() && is(t, at::kFloat))) fail(std::string(n) + " must be contiguous CUDA fp32");
}

struct Dims {
  int64_t B, Hq, D, Hkv, T, nb;
};

int64_t pool_tokens(const at::Tensor& k, const at::Tensor& v, int64_t B, int64_t Hkv, int64_t D, const at::Tensor& bt,
                    PyObject* T_) {
  require(T_ != Py_None, "paged cache: T (tokens per sequence, or the capacity) is required");
  const int64_t T = integer(T_);
  require(T >= 1, "paged cache: T (tokens per sequence, or the capacity) is required");
  for (const at::Tensor* x : {&k, &v})
    require(x->dim() == 4 && x->size(1) == Hkv && x->size(2) == TILE && x->size(3) == D && x->size(0) == k.size(0),
            "paged cache: k, v must be page pools [num_pages, Hkv, 64, D]");
  require(bt.is_cuda() && bt.scalar_type() == at::kInt && bt.dim() == 2 && bt.size(0) == B && bt.stride(1) == 1 &&
              bt.size(1) >= tiles(T),
          "block_table: int32 [B, >= ceil(T / 64)] on the device, rows contiguous");
  return T;
}

Dims kv_dims(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor* bt, PyObject* T_) {
  require(q.dim() == 3, "q must be CUDA bf16 [B, Hq, D]");
  Dims d{q.size(0), q.size(1), q.size(2), 0, 0, 0};
  require(k.dim() == 4 && v.dim() == 4, "shape mismatch between q, k, v");
  d.Hkv = k.size(1);
  if (bt == nullptr) {
    // every kernel reads v (and k) as [B, Hkv, T, D] of k's sizes: a shorter or narrower view would be
    // read past its end
    require(k.size(0) == d.B && k.size(3) == d.D && v.sizes() == k.sizes(), "shape mismatch between q, k, v");
    d.T = k.size(2);
  } else {
    d.T = pool_tokens(k, v, d.B, d.Hkv, d.D, *bt, T_);
  }
  d.nb = tiles(d.T);
  return d;
}

void set_base(kvskip_attn_args& a, const at::Tensor* q, const at::Tensor* k, const at::Tensor* v, double scale,
              const Dims& d) {
  std::memset(&a, 0, sizeof(a));
  if (q != nullptr) {
    a.q = q->data_ptr();
    a.q_sb = q->stride(0), a.q_sh = q->stride(1);
  }
  if (k != nullptr) {
    a.k = k->data_ptr();
    a.k_sb = k->stride(0), a.k_sh = k->stride(1), a.k_st = k->stride(2);
  }
  if (v != nullptr) {
    a.v = v->data_ptr();
    a.v_sb = v->stride(0), a.v_sh = v->stride(1), a.v_st = v->stride(2);
  }
  a.B = static_cast<int32_t>(d.B), a.Hq = static_cast<int32_t>(d.Hq), a.Hkv = static_cast<int32_t>(d.Hkv);
  a.T = static_cast<int32_t>(d.T), a.D = static_cast<int32_t>(d.D);
  a.scale = static_cast<float>(scale);
}

void set_pages(kvskip_attn_args& a, const at::Tensor* bt, const at::Tensor& pool) {
  if (bt == nullptr) return;  // page pools: the dim-0 strides of k / v are the page strides
  a.block_table = static_cast<const int32_t*>(bt->data_ptr());
  a.bt_stride = bt->stride(0);
  a.num_pages = static_cast<int32_t>(pool.size(0));
}

const int32_t* lens_ptr(const at::Tensor* l, int64_t B) {
  if (l == nullptr) return nullptr;
  require(l->is_cuda() && is(*l, at::kInt) && l->numel() == B, "seq_lens: contiguous CUDA int32 [B]");
  return static_cast<const int32_t*>(l->data_ptr());
}

void set_lists(kvskip_attn_args& a, const at::Tensor* bi, const at::Tensor* bc, const Dims& d) {
  if (bi == nullptr) return;
  require(bc != nullptr, "block_cnt is required with block_idx");
  require(bi->is_cuda() && bi->dim() == 3 && is(*bi, at::kInt) && bi->size(0) == d.B && bi->size(1) == d.Hkv,
          "block_idx must be contiguous int32 [B, Hkv, max_blocks]");
  require(bc->is_cuda() && is(*bc, at::kInt) && bc->numel() == d.B * d.Hkv, "block_cnt must be contiguous int32 [B, Hkv]");
  a.block_idx = static_cast<const int32_t*>(bi->data_ptr());
  a.block_cnt = static_cast<const int32_t*>(bc->data_ptr());
  a.max_blocks = static_cast<int32_t>(bi->size(2));
}

// The argument block of a decode call's pointers (ext._decode_args).
struct Outs {
  void *out = nullptr, *lse = nullptr, *bmax = nullptr, *bsum = nullptr, *out32 = nullptr, *p = nullptr,
       *part_acc = nullptr, *part_ml = nullptr;
};
Dims set_decode(kvskip_attn_args& a, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, double scale,
                const at::Tensor* bi, const at::Tensor* bc, int64_t S, const Outs& o, const at::Tensor* lens,
                const at::Tensor* bt, PyObject* T_, int list_partition) {
  const Dims d = kv_dims(q, k, v, bt, T_);
  set_base(a, &q, &k, &v, scale, d);
  set_pages(a, bt, k);
  a.seq_lens = lens_ptr(lens, d.B);
  set_lists(a, bi, bc, d);
  a.num_splits = static_cast<int32_t>(S);
  a.part_acc = static_cast<float*>(o.part_acc), a.part_ml = static_cast<float*>(o.part_ml);
  a.out = o.out, a.out_f32 = static_cast<float*>(o.out32), a.lse = static_cast<float*>(o.lse);
  a.blk_max = static_cast<float*>(o.bmax), a.blk_sum = static_cast<float*>(o.bsum);
  a.p_out = o.p;
  a.list_partition = list_partition;
  return d;
}

at::Tensor empty(at::IntArrayRef sizes, at::ScalarType ty, const at::Device& dev) {
  return at::empty(sizes, at::TensorOptions().dtype(ty).device(dev));
}

// A call's split partials in one allocation: acc [B, Hq, S, D] (with_acc), then ml [B, Hq, S, 2].
at::Tensor partials(Outs& o, const Dims& d, int64_t S, bool with_acc, const at::Device& dev) {
  const int64_t rows = d.B * d.Hq * S, n_acc = with_acc ? rows * d.D : 0;
  at::Tensor t = empty({n_acc + rows * 2}, at::kFloat, dev);
  float* f = static_cast<float*>(t.data_ptr());
  if (with_acc) o.part_acc = f;
  o.part_ml = f + n_acc;
  return t;
}

// ---- operators (argument order as in ext.py)
// decode(q, k, v, scale, block_idx, block_cnt, stats, load_v, num_splits, stages, want_f32, write_p, seq_lens,
//        block_table, T, merge, list_partition)
PyObject* decode(PyObject* const* a) {
  const at::Tensor &q = tensor(a[0], "q"), &k = tensor(a[1], "k"), &v = tensor(a[2], "v");
  check_q(q);
  check_kv(k, "k");
  check_kv(v, "v");
  const at::Tensor *bi = opt_tensor(a[4], "block_idx"), *bc = opt_tensor(a[5], "block_cnt"),
                   *lens = opt_tensor(a[12], "seq_lens"), *bt = opt_tensor(a[13], "block_table");
  const Dims d = kv_dims(q, k, v, bt, a[14]);
  require(d.Hkv > 0 && d.Hq % d.Hkv == 0, "Hq must be a multiple of Hkv");
  const bool stats = truth(a[6]), load_v = truth(a[7]), want_f32 = truth(a[10]), write_p = truth(a[11]),
             merge = truth(a[15]);
  const int64_t S = integer(a[8]), stages = integer(a[9]);
  require(1 <= S && S <= 256, "num_splits in 1..256");
  require(load_v || stats, "load_v=false only makes sense with stats=true");
  require(!write_p || stats, "write_p needs stats=true");
  require(merge || !load_v, "merge=False needs load_v=False");
  require(stages == 2 || stages == 3, "kvskip: unsupported head dim / stages");
  const at::Device dev = q.device();
  at::Tensor out, out32, bmax, bsum, p, part;
  Outs o;
  if (load_v) o.out = (out = empty({d.B, d.Hq, d.D}, at::kBFloat16, dev)).data_ptr();
  if (load_v && want_f32) o.out32 = (out32 = empty({d.B, d.Hq, d.D}, at::kFloat, dev)).data_ptr();
  at::Tensor lse = empty({d.B, d.Hq}, at::kFloat, dev);
  o.lse = lse.data_ptr();
  if (stats) {  // every block is written (-inf / 0 where a list skips it)
    o.bmax = (bmax = empty({d.B, d.Hq, d.nb}, at::kFloat, dev)).data_ptr();
    o.bsum = (bsum = empty({d.B, d.Hq, d.nb}, at::kFloat, dev)).data_ptr();
  }
  if (write_p) o.p = (p = empty({d.B, d.Hq, d.nb * TILE}, at::kHalf, dev)).data_ptr();
  if (S > 1) part = partials(o, d, S, load_v, dev);
  const bool split_only = !merge && S > 1;
  kvskip_attn_args args;
  set_decode(args, q, k, v, real(a[3]), bi, bc, S, o, lens, bt, a[14], int32(a[16]));
  launch(dev, [&](void* s) { return (split_only ? api.decode_splits : api.decode)(&args, stats, load_v, s); });
  return list_of({out, split_only ? at::Tensor() : lse, bmax, bsum, out32, p});
}

// The statistics and partial buffers of a pass into caller-owned buffers.
void pass_bufs(Outs& o, PyObject* bufs, bool stats, int64_t S, const Dims& d, bool typed) {
  if (stats) {
    const at::Tensor &m = tensor(item(bufs, "blk_max"), "blk_max"), &s = tensor(item(bufs, "blk_sum"), "blk_sum");
    for (const at::Tensor* t : {&m, &s}) require(is(*t, at::kFloat) && t->numel() >= d.B * d.Hq * d.nb, "bufs: stats");
    o.bmax = m.data_ptr(), o.bsum = s.data_ptr();
  }
  if (S > 1) {
    const at::Tensor &c = tensor(item(bufs, "part_acc"), "part_acc"), &m = tensor(item(bufs, "part_ml"), "part_ml");
    const int64_t rows = d.B * d.Hq * S;
    if (typed) {
      require(is(c, at::kFloat) && c.numel() >= rows * d.D, "bufs: part_acc");
      require(is(m, at::kFloat) && m.numel() >= rows * 2, "bufs: part_ml");
    } else {
      require(c.numel() >= rows * d.D && m.numel() >= rows * 2, "bufs: split partials");
    }
    o.part_acc = c.data_ptr(), o.part_ml = m.data_ptr();
  }
}

// decode_into(q, k, v, scale, bufs, block_idx, block_cnt, stats, num_splits, seq_lens, phase, block_table, T,
//             list_partition, key_sums)
PyObject* decode_into(PyObject* const* a) {
  const at::Tensor &q = tensor(a[0], "q"), &k = tensor(a[1], "k"), &v = tensor(a[2], "v");
  check_q(q);
  check_kv(k, "k");
  check_kv(v, "v");
  const at::Tensor* bt = opt_tensor(a[11], "block_table");
  const Dims d = kv_dims(q, k, v, bt, a[12]);
  const int64_t S = integer(a[8]), phase = integer(a[10]);
  require(1 <= S && S <= 256, "num_splits in 1..256");
  const bool stats = truth(a[7]);
  const at::Tensor &out = tensor(item(a[4], "out"), "out"), &lse = tensor(item(a[4], "lse"), "lse");
  require(is(out, at::kBFloat16) && out.numel() >= d.B * d.Hq * d.D, "bufs: out");
  require(is(lse, at::kFloat) && lse.numel() >= d.B * d.Hq, "bufs: lse");
  Outs o;
  o.out = out.data_ptr(), o.lse = lse.data_ptr();
  pass_bufs(o, a[4], stats, S, d, true);
  kvskip_attn_args args;
  set_decode(args, q, k, v, real(a[3]), opt_tensor(a[5], "block_idx"), opt_tensor(a[6], "block_cnt"), S, o,
             opt_tensor(a[9], "seq_lens"), bt, a[12], int32(a[13]));
  if (const at::Tensor* t = opt_tensor(a[14], "key_sums")) {
    check_f32(*t, "key_sums");
    require(t->dim() == 4 && t->size(0) == d.B && t->size(1) == d.Hkv && t->size(2) >= d.nb && t->size(3) == d.D,
            "key_sums: [B, Hkv, >= ceil(T / 64), D]");
    args.key_sums = static_cast<float*>(t->data_ptr()), args.sums_cap = static_cast<int32_t>(t->size(2));
  }
  auto* fn = phase == 3 ? api.decode : phase == 1 ? api.decode_splits : phase == 2 ? api.merge_splits : nullptr;
  require(fn != nullptr, "phase in {1, 2, 3}");
  launch(q.device(), [&](void* s) { return fn(&args, stats, 1, s); });
  Py_RETURN_NONE;
}

// The masked + statistics split pass into a planner's buffers, its arguments in a[0..6] = q, k, v, scale, bufs,
// block_idx, block_cnt and a[7] num_splits, seq_lens, block_table, T, list_partition.
void pass_args(kvskip_attn_args& args, PyObject* const* a, PyObject* S_, PyObject* lens, PyObject* bt_, PyObject* T_,
               PyObject* lp) {
  const at::Tensor &q = tensor(a[0], "q"), &k = tensor(a[1], "k"), &v = tensor(a[2], "v");
  check_q(q);
  check_kv(k, "k");
  check_kv(v, "v");
  const at::Tensor* bt = opt_tensor(bt_, "block_table");
  const Dims d = kv_dims(q, k, v, bt, T_);
  const int64_t S = integer(S_);
  require(1 <= S && S <= 256, "num_splits in 1..256");
  Outs o;
  pass_bufs(o, a[4], true, S, d, false);
  o.out = tensor(item(a[4], "out"), "out").data_ptr();
  o.lse = tensor(item(a[4], "lse"), "lse").data_ptr();
  set_decode(args, q, k, v, real(a[3]), opt_tensor(a[5], "block_idx"), opt_tensor(a[6], "block_cnt"), S, o,
             opt_tensor(lens, "seq_lens"), bt, T_, int32(lp));
}

// splits_planned(q, k, v, scale, bufs, None, None, plan block, num_splits, update block or None, seq_lens, block_table,
//                T, 0)
PyObject* splits_planned(PyObject* const* a) {
  kvskip_attn_args args;
  pass_args(args, a, a[8], a[10], a[11], a[12], a[13]);
  const auto* p = block<const kvskip_plan_args>(a[7]);
  const auto* u = a[9] == Py_None ? nullptr : block<const kvskip_update_args>(a[9]);
  launch(tensor(a[0], "q").device(), [&](void* s) { return api.decode_splits_planned(&args, p, u, s); });
  Py_RETURN_NONE;
}

// splits_update(q, k, v, scale, bufs, block_idx, block_cnt, num_splits, update block, seq_lens, block_table, T,
//               list_partition)
PyObject* splits_update(PyObject* const* a) {
  kvskip_attn_args args;
  pass_args(args, a, a[7], a[9], a[10], a[11], a[12]);
  const auto* u = block<const kvskip_update_args>(a[8]);
  launch(tensor(a[0], "q").device(), [&](void* s) { return api.decode_splits_update(&args, u, s); });
  Py_RETURN_NONE;
}

// attn_block(attn block, q, k, v, scale, block_idx, block_cnt, num_splits, out, lse, blk_max, blk_sum, out_f32, P,
//            part_acc, part_ml, seq_lens, block_table, T, list_partition)
PyObject* attn_block(PyObject* const* a) {
  Outs o;
  o.out = ptr(opt_tensor(a[8], "out")), o.lse = tensor(a[9], "lse").data_ptr();
  o.bmax = ptr(opt_tensor(a[10], "blk_max")), o.bsum = ptr(opt_tensor(a[11], "blk_sum"));
  o.out32 = ptr(opt_tensor(a[12], "out_f32")), o.p = ptr(opt_tensor(a[13], "P"));
  o.part_acc = ptr(opt_tensor(a[14], "part_acc")), o.part_ml = ptr(opt_tensor(a[15], "part_ml"));
  set_decode(*block<kvskip_attn_args>(a[0]), tensor(a[1], "q"), tensor(a[2], "k"), tensor(a[3], "v"), real(a[4]),
             opt_tensor(a[5], "block_idx"), opt_tensor(a[6], "block_cnt"), integer(a[7]), o,
             opt_tensor(a[16], "seq_lens"), opt_tensor(a[17], "block_table"), a[18], int32(a[19]));
  Py_RETURN_NONE;
}

// vskip1(q, k, v, scale, tau, local, num_splits, want_f32, count, lse_prev, block_table, T, v_keep)
PyObject* vskip1(PyObject* const* a) {
  const at::Tensor &q = tensor(a[0], "q"), &k = tensor(a[1], "k"), &v = tensor(a[2], "v");
  check_q(q);
  check_kv(k, "k");
  check_kv(v, "v");
  const double tau = real(a[4]);
  const int32_t local = int32(a[5]);
  const int64_t S = integer(a[6]);
  require(tau > 0.0 && local >= 0 && S >= 1, "tau > 0, local >= 0, num_splits >= 1");
  const at::Tensor* bt = opt_tensor(a[10], "block_table");
  const Dims d = kv_dims(q, k, v, bt, a[11]);
  require(d.Hkv > 0 && d.Hq % d.Hkv == 0, "Hq must be a multiple of Hkv");
  const bool want_f32 = truth(a[7]), count = truth(a[8]);
  const at::Device dev = q.device();
  Outs o;
  at::Tensor out = empty({d.B, d.Hq, d.D}, at::kBFloat16, dev), out32, vcount, part;
  if (want_f32) out32 = empty({d.B, d.Hq, d.D}, at::kFloat, dev);
  at::Tensor lse = empty({d.B, d.Hq}, at::kFloat, dev);
  if (count) vcount = at::zeros({d.B, d.Hkv}, at::TensorOptions().dtype(at::kInt).device(dev));
  if (S > 1) part = partials(o, d, S, true, dev);
  kvskip_attn_args args;
  set_base(args, &q, &k, &v, real(a[3]), d);
  args.num_splits = static_cast<int32_t>(std::min<int64_t>(S, INT32_MAX));
  args.part_acc = static_cast<float*>(o.part_acc), args.part_ml = static_cast<float*>(o.part_ml);
  args.out = out.data_ptr(), args.lse = static_cast<float*>(lse.data_ptr());
  args.out_f32 = want_f32 ? static_cast<float*>(out32.data_ptr()) : nullptr;
  args.tau = static_cast<float>(tau), args.local = local;
  args.vcount = count ? static_cast<int32_t*>(vcount.data_ptr()) : nullptr;
  if (const at::Tensor* lp = opt_tensor(a[9], "lse_prev")) {
    require(lp->is_cuda() && is(*lp, at::kFloat) && lp->numel() == d.B * d.Hq, "lse_prev: contiguous fp32 [B, Hq]");
    args.lse_prev = static_cast<const float*>(lp->data_ptr());
  }
  if (const at::Tensor* vk = opt_tensor(a[12], "v_keep")) {
    require(vk->is_cuda() && is(*vk, at::kByte) && vk->sizes() == at::IntArrayRef({d.B, d.Hkv, d.nb}),
            "v_keep: contiguous uint8 [B, Hkv, nb]");
    args.v_keep = static_cast<uint8_t*>(vk->data_ptr());
  }
  set_pages(args, bt, k);
  launch(dev, [&](void* s) { return api.vskip1(&args, s); });
  return list_of({out, lse, out32, vcount});
}

// The selection's argument block (ext._select_args): a = blk_max, blk_sum, Hkv, rule, value, local, keep, block_idx,
// block_cnt, blk_scale.
void select_args(kvskip_select_args& s, PyObject* const* a) {
  const char* rule = PyUnicode_Check(a[3]) ? PyUnicode_AsUTF8(a[3]) : nullptr;
  const bool topp = rule != nullptr && std::strcmp(rule, "topp") == 0;
  require(topp || (rule != nullptr && std::strcmp(rule, "tau") == 0), "rule must be tau or topp");
  const at::Tensor &m = tensor(a[0], "blk_max"), &sm = tensor(a[1], "blk_sum");
  check_f32(m, "blk_max");
  check_f32(sm, "blk_sum");
  require(m.dim() == 3 && sm.sizes() == m.sizes(), "blk_max / blk_sum: [B, Hq, nb]");
  const int64_t B = m.size(0), Hq = m.size(1), nb = m.size(2), Hkv = integer(a[2]);
  require(Hkv > 0 && Hq % Hkv == 0, "Hq must be a multiple of Hkv");
  std::memset(&s, 0, sizeof(s));
  s.blk_max = static_cast<const float*>(m.data_ptr()), s.blk_sum = static_cast<const float*>(sm.data_ptr());
  s.B = static_cast<int32_t>(B), s.Hq = static_cast<int32_t>(Hq), s.Hkv = static_cast<int32_t>(Hkv);
  s.nb = static_cast<int32_t>(nb);
  s.rule = topp ? 1 : 0, s.value = static_cast<float>(real(a[4])), s.local = int32(a[5]);
  auto out = [&](PyObject* o, std::vector<int64_t> shape, at::ScalarType ty, const char* tyname,
                 const char* name) -> void* {
    const at::Tensor* t = opt_tensor(o, name);
    if (t == nullptr) return nullptr;
    if (!(t->is_cuda() && is(*t, ty) && t->sizes() == at::IntArrayRef(shape))) {
      std::string l;
      for (int64_t x : shape) l += (l.empty() ? "" : ", ") + std::to_string(x);
      fail(std::string(name) + ": contiguous torch." + tyname + " [" + l + "] on the device");
    }
    return t->data_ptr();
  };
  s.keep = static_cast<uint8_t*>(out(a[6], {B, Hkv, nb}, at::kByte, "uint8", "keep"));
  s.block_idx = static_cast<int32_t*>(out(a[7], {B, Hkv, nb}, at::kInt, "int32", "block_idx"));
  s.block_cnt = static_cast<int32_t*>(out(a[8], {B, Hkv}, at::kInt, "int32", "block_cnt"));
  s.blk_scale = static_cast<float*>(out(a[9], {B, Hkv, nb, Hq / Hkv}, at::kFloat, "float32", "blk_scale"));
  require(s.block_idx == nullptr || s.block_cnt != nullptr, "block_cnt is required with block_idx");
}

// select(blk_max, blk_sum, Hkv, rule, value, local, keep, block_idx, block_cnt, blk_scale)
PyObject* select(PyObject* const* a) {
  kvskip_select_args s;
  select_args(s, a);
  launch(tensor(a[0], "blk_max").device(), [&](void* st) { return api.select(&s, st); });
  Py_RETURN_NONE;
}

// The outputs and partials of pass 2 into args; keeps the tensors.
struct PvOut {
  at::Tensor out, out32, part;
  PvOut(kvskip_attn_args& args, const at::Tensor& v, const Dims& d, int64_t S, bool want_f32) {
    const at::Device dev = v.device();
    Outs o;
    out = empty({d.B, d.Hq, d.D}, at::kBFloat16, dev);
    if (want_f32) out32 = empty({d.B, d.Hq, d.D}, at::kFloat, dev);
    if (S > 1) part = partials(o, d, S, true, dev);
    set_base(args, nullptr, nullptr, &v, 1.0, d);
    args.num_splits = static_cast<int32_t>(std::min<int64_t>(S, INT32_MAX));
    args.part_acc = static_cast<float*>(o.part_acc), args.part_ml = static_cast<float*>(o.part_ml);
    args.out = out.data_ptr(), args.out_f32 = want_f32 ? static_cast<float*>(out32.data_ptr()) : nullptr;
  }
};

// pv(P, v, blk_scale, block_idx, block_cnt, num_splits, want_f32, block_table, T)
PyObject* pv(PyObject* const* a) {
  const at::Tensor &P = tensor(a[0], "P"), &v = tensor(a[1], "v"), &sc = tensor(a[2], "blk_scale"),
                   &bi = tensor(a[3], "block_idx"), &bc = tensor(a[4], "block_cnt");
  check_kv(v, "v");
  require(P.is_cuda() && P.dim() == 3 && is(P, at::kHalf), "P: fp16 [B, Hq, t_pad]");
  require(sc.is_cuda() && sc.dim() == 4 && is(sc, at::kFloat), "blk_scale: contiguous fp32 [B, Hkv, nb, G]");
  const at::Tensor* bt = opt_tensor(a[7], "block_table");
  Dims d{bt == nullptr ? v.size(0) : P.size(0), P.size(1), v.size(3), v.size(1), v.size(2), 0};
  if (bt != nullptr) d.T = pool_tokens(v, v, d.B, d.Hkv, d.D, *bt, a[8]);
  d.nb = tiles(d.T);
  require(d.Hkv > 0 && d.Hq % d.Hkv == 0, "Hq must be a multiple of Hkv");
  require(P.size(0) == d.B && P.size(2) == d.nb * TILE, "P shape");
  require(sc.sizes() == at::IntArrayRef({d.B, d.Hkv, d.nb, d.Hq / d.Hkv}), "blk_scale shape");
  require(is(bi, at::kInt) && bi.dim() == 3 && bi.size(0) == d.B && bi.size(1) == d.Hkv, "block_idx");
  require(is(bc, at::kInt) && bc.numel() == d.B * d.Hkv, "block_cnt");
  const int64_t S = integer(a[5]);
  require(S >= 1, "num_splits >= 1");
  kvskip_attn_args args;
  const bool want_f32 = truth(a[6]);
  PvOut o(args, v, d, S, want_f32);
  args.block_idx = static_cast<const int32_t*>(bi.data_ptr()), args.block_cnt = static_cast<const int32_t*>(bc.data_ptr());
  args.max_blocks = static_cast<int32_t>(bi.size(2));
  args.p_in = P.data_ptr(), args.blk_scale = static_cast<const float*>(sc.data_ptr());
  set_pages(args, bt, v);
  launch(v.device(), [&](void* s) { return api.pv(&args, s); });
  return list_of({o.out, o.out32});
}

// pv_select(P, v, blk_max, blk_sum, rule, value, local, num_splits, want_f32, keep, block_idx, block_cnt, blk_scale)
PyObject* pv_select(PyObject* const* a) {
  const at::Tensor &P = tensor(a[0], "P"), &v = tensor(a[1], "v"), &m = tensor(a[2], "blk_max");
  check_kv(v, "v");
  require(P.is_cuda() && P.dim() == 3 && is(P, at::kHalf), "P: fp16 [B, Hq, t_pad]");
  const Dims d{v.size(0), P.size(1), v.size(3), v.size(1), v.size(2), tiles(v.size(2))};
  require(P.size(0) == d.B && P.size(2) == d.nb * TILE, "P shape");
  require(m.sizes() == at::IntArrayRef({d.B, d.Hq, d.nb}), "blk_max: [B, Hq, nb] of the pass's cache");
  const int64_t S = integer(a[7]);
  require(S >= 1, "num_splits >= 1");
  PyObject* hkv = PyLong_FromLongLong(d.Hkv);
  if (hkv == nullptr) throw PyErr{};
  PyObject* sel[10] = {a[2], a[3], hkv, a[4], a[5], a[6], a[9], a[10], a[11], a[12]};
  kvskip_select_args sa;
  try {
    select_args(sa, sel);
  } catch (...) {
    Py_DECREF(hkv);
    throw;
  }
  Py_DECREF(hkv);
  kvskip_attn_args args;
  PvOut o(args, v, d, S, truth(a[8]));
  args.p_in = P.data_ptr();
  launch(v.device(), [&](void* s) { return api.pv_select(&args, &sa, s); });
  return list_of({o.out, o.out32});
}

// plan_block(plan block, q, k, csum, lse_ref, cs_ref, keep, lse_att, age, flags, cs_now, trig, block_idx, block_cnt,
//            scale, delta, max_age, local, add_token, idx, calib, est, calib_on, calib_kind, aix, part, seq_lens,
//            seq_lens_out, ids, idx_out, block_table, T, ticket): ext._plan_args
PyObject* plan_block(PyObject* const* a) {
  kvskip_plan_args& p = *block<kvskip_plan_args>(a[0]);
  const at::Tensor &q = tensor(a[1], "q"), &k = tensor(a[2], "k");
  require(is_bf16_cuda(q) && q.dim() == 3 && q.stride(2) == 1, "q: CUDA bf16 [B, Hq, D]");
  check_kv(k, "k");
  const at::Tensor* bt = opt_tensor(a[30], "block_table");
  const Dims d = kv_dims(q, k, k, bt, a[31]);
  const at::Tensor &csum = tensor(a[3], "csum"), &lref = tensor(a[4], "lse_ref"), &cref = tensor(a[5], "cs_ref"),
                   &keep = tensor(a[6], "keep"), &latt = tensor(a[7], "lse_att"), &age = tensor(a[8], "age"),
                   &flags = tensor(a[9], "flags"), &cnow = tensor(a[10], "cs_now"), &trig = tensor(a[11], "trig"),
                   &bi = tensor(a[12], "block_idx"), &bc = tensor(a[13], "block_cnt");
  check_f32(csum, "csum");
  check_f32(lref, "lse_ref");
  check_f32(cref, "cs_ref");
  check_f32(latt, "lse_att");
  check_f32(cnow, "cs_now");
  require(keep.dim() == 3, "keep: contiguous uint8 [B, Hkv, NBC]");
  const int64_t NBC = keep.size(2), BH = d.B * d.Hkv;
  require(d.nb <= NBC, "block capacity exceeded");
  require(csum.dim() > 2 && lref.dim() > 2 && cref.dim() > 2 && cnow.dim() > 2 && bi.dim() > 2 && csum.size(2) == NBC &&
              lref.size(2) == NBC && cref.size(2) == NBC && cnow.size(2) == NBC && bi.size(2) == NBC,
          "capacity mismatch");
  require(is(age, at::kInt) && age.numel() == BH, "age: int32 [B, Hkv]");
  require(flags.scalar_type() == at::kInt && flags.numel() == d.Hkv, "flags: int32 [Hkv]");
  require(is(keep, at::kByte), "keep: contiguous uint8 [B, Hkv, NBC]");
  require(trig.scalar_type() == at::kByte && bi.scalar_type() == at::kInt && bc.scalar_type() == at::kInt,
          "trig uint8, block_idx / block_cnt int32");
  std::memset(&p, 0, sizeof(p));
  auto f = [](const at::Tensor& t) { return static_cast<float*>(t.data_ptr()); };
  auto u8 = [](const at::Tensor& t) { return static_cast<uint8_t*>(t.data_ptr()); };
  auto i32 = [](const at::Tensor& t) { return static_cast<int32_t*>(t.data_ptr()); };
  p.q = q.data_ptr(), p.q_sb = q.stride(0), p.q_sh = q.stride(1);
  p.k = k.data_ptr(), p.k_sb = k.stride(0), p.k_sh = k.stride(1), p.k_st = k.stride(2);
  p.csum = f(csum), p.lse_ref = f(lref), p.cs_ref = f(cref), p.keep = u8(keep);
  p.lse_att = f(latt), p.age = i32(age), p.flags = i32(flags);
  const at::Tensor *idx = opt_tensor(a[19], "idx"), *ids = opt_tensor(a[28], "ids"), *part = opt_tensor(a[25], "part");
  if (idx != nullptr) {
    require(idx->is_cuda() && idx->dim() == 2 && is(*idx, at::kByte) && idx->size(0) == d.B && idx->size(1) == NBC,
            "idx: contiguous uint8 [B, NBC]");
    p.idx = u8(*idx);
  }
  if (const at::Tensor* t = opt_tensor(a[20], "calib")) {
    check_f32(*t, "calib");
    require(t->numel() == BH, "calib: [B, Hkv]");
    p.calib = f(*t);
  }
  if (const at::Tensor* t = opt_tensor(a[21], "est")) {
    check_f32(*t, "est");
    require(t->numel() == BH, "est: [B, Hkv]");
    p.est = f(*t);
  }
  p.calib_on = truth(a[22]), p.calib_kind = int32(a[23]);
  if (const at::Tensor* t = opt_tensor(a[24], "aix")) {
    require(t->is_cuda() && is(*t, at::kByte) && t->numel() == BH, "aix: contiguous uint8 [B, Hkv]");
    require(idx != nullptr || ids != nullptr, "aix needs idx");
    p.aix = u8(*t);
  }
  p.cs_now = f(cnow), p.trig = u8(trig), p.block_idx = i32(bi), p.block_cnt = i32(bc);
  p.B = static_cast<int32_t>(d.B), p.Hq = static_cast<int32_t>(d.Hq), p.Hkv = static_cast<int32_t>(d.Hkv);
  p.T = static_cast<int32_t>(d.T), p.D = static_cast<int32_t>(d.D), p.NBC = static_cast<int32_t>(NBC);
  p.local = int32(a[17]), p.max_age = int32(a[16]), p.add_token = truth(a[18]);
  p.scale = static_cast<float>(real(a[14])), p.delta = static_cast<float>(real(a[15]));
  if (part != nullptr) {
    check_f32(*part, "part");
    require(part->numel() >= api.plan_part_floats(p.B, p.Hq, p.Hkv, p.NBC), "part: too small");
    p.part = f(*part);
  }
  p.seq_lens = lens_ptr(opt_tensor(a[26], "seq_lens"), d.B);
  if (bt != nullptr) {
    p.block_table = i32(*bt), p.bt_stride = bt->stride(0);
    p.num_pages = static_cast<int32_t>(k.size(0));
  }
  if (const at::Tensor* t = opt_tensor(a[27], "seq_lens_out")) {
    require(t->is_cuda() && is(*t, at::kInt) && t->numel() == d.B, "seq_lens_out: contiguous int32 [B] on the device");
    p.seq_lens_out = i32(*t);
  }
  if (ids != nullptr) {
    const at::Tensor* io = opt_tensor(a[29], "idx_out");
    require(part != nullptr && idx == nullptr && io != nullptr, "plan: ids needs part and idx_out, and no idx");
    require(ids->is_cuda() && ids->scalar_type() == at::kInt && ids->dim() == 2 && ids->stride(1) == 1 &&
                ids->size(0) == d.B && ids->size(1) >= d.T,
            "ids: CUDA int32 [B, >= T]");
    require(is(*io, at::kByte) && io->sizes() == at::IntArrayRef({d.B, NBC}), "idx_out: uint8 [B, NBC]");
    p.ids = i32(*ids), p.ids_sb = ids->stride(0), p.idx_out = u8(*io);
  }
  if (const at::Tensor* t = opt_tensor(a[32], "ticket")) {
    require(part != nullptr, "plan: ticket needs part");
    require(t->is_cuda() && is(*t, at::kInt) && t->numel() == BH, "ticket: contiguous int32 [B * Hkv] on the device");
    p.ticket = i32(*t);
  }
  Py_RETURN_NONE;
}

// update_block(update block, blk_max, blk_sum, trig, cs_now, keep, lse_ref, cs_ref, lse_att, T, level, local, flags,
//              idx, est, calib, calib_rate, calib_free, calib_kind, aix, aix_thr, list_stats, seq_lens, age):
// ext._update_args
PyObject* update_block(PyObject* const* a) {
  kvskip_update_args& p = *block<kvskip_update_args>(a[0]);
  const at::Tensor &m = tensor(a[1], "blk_max"), &s = tensor(a[2], "blk_sum"), &keep = tensor(a[5], "keep"),
                   &latt = tensor(a[8], "lse_att");
  check_f32(m, "blk_max");
  check_f32(s, "blk_sum");
  require(keep.dim() == 3, "keep: contiguous uint8 [B, Hkv, NBC]");
  require(latt.dim() > 1, "lse_att: [B, Hq]");
  const int64_t B = keep.size(0), Hkv = keep.size(1), NBC = keep.size(2), T = integer(a[9]);
  require(m.dim() > 2 && m.size(2) == tiles(T), "stats length mismatch");
  require(is(keep, at::kByte), "keep: contiguous uint8 [B, Hkv, NBC]");
  std::memset(&p, 0, sizeof(p));
  auto f = [](const at::Tensor& t) { return static_cast<float*>(t.data_ptr()); };
  auto u8 = [](const at::Tensor& t) { return static_cast<uint8_t*>(t.data_ptr()); };
  auto i32 = [](const at::Tensor& t) { return static_cast<int32_t*>(t.data_ptr()); };
  p.blk_max = f(m), p.blk_sum = f(s);
  p.trig = static_cast<uint8_t*>(tensor(a[3], "trig").data_ptr());
  p.cs_now = static_cast<float*>(tensor(a[4], "cs_now").data_ptr());
  p.keep = u8(keep);
  p.lse_ref = static_cast<float*>(tensor(a[6], "lse_ref").data_ptr());
  p.cs_ref = static_cast<float*>(tensor(a[7], "cs_ref").data_ptr());
  p.lse_att = static_cast<float*>(latt.data_ptr());
  p.B = static_cast<int32_t>(B), p.Hq = static_cast<int32_t>(latt.size(1)), p.Hkv = static_cast<int32_t>(Hkv);
  p.T = static_cast<int32_t>(T), p.NBC = static_cast<int32_t>(NBC), p.local = int32(a[11]);
  p.level = static_cast<float>(real(a[10]));
  const at::Tensor *flags = opt_tensor(a[12], "flags"), *idx = opt_tensor(a[13], "idx"), *est = opt_tensor(a[14], "est"),
                   *calib = opt_tensor(a[15], "calib"), *aix = opt_tensor(a[19], "aix");
  auto set_flags_idx = [&] {
    require(flags->is_cuda() && flags->scalar_type() == at::kInt && flags->numel() == Hkv, "flags: int32 [Hkv]");
    p.flags = i32(*flags);
    if (idx != nullptr) {
      require(idx->is_cuda() && idx->dim() == 2 && is(*idx, at::kByte) && idx->size(0) == B && idx->size(1) == NBC,
              "idx: contiguous uint8 [B, NBC]");
      p.idx = u8(*idx);
    }
  };
  if (calib != nullptr) {
    require(flags != nullptr && est != nullptr, "calibration needs flags and est");
    require(flags->is_cuda() && flags->scalar_type() == at::kInt && flags->numel() == Hkv, "flags: int32 [Hkv]");
    check_f32(*est, "est");
    check_f32(*calib, "calib");
    require(est->numel() == B * Hkv && calib->numel() == B * Hkv, "est / calib: [B, Hkv]");
    p.est = f(*est), p.calib = f(*calib);
    p.calib_rate = static_cast<float>(real(a[16])), p.calib_free = truth(a[17]), p.calib_kind = int32(a[18]);
    if (aix != nullptr) {
      require(aix->is_cuda() && is(*aix, at::kByte) && aix->numel() == B * Hkv, "aix: contiguous uint8 [B, Hkv]");
      require(idx != nullptr, "aix needs idx");
      p.aix = u8(*aix), p.aix_thr = static_cast<float>(real(a[20]));
    }
    set_flags_idx();
  }
  if (truth(a[21])) {
    require(flags != nullptr, "list_stats needs flags");
    set_flags_idx();
    p.list_stats = 1;
  }
  p.seq_lens = lens_ptr(opt_tensor(a[22], "seq_lens"), B);
  if (const at::Tensor* t = opt_tensor(a[23], "age")) {
    require(t->is_cuda() && is(*t, at::kInt) && t->numel() == B * Hkv, "age: contiguous int32 [B, Hkv]");
    p.age = i32(*t);
  }
  Py_RETURN_NONE;
}

// Launches of a filled block on the device of a tensor: plan / plan_scores / update (block, tensor) and
// merge_update(attn block, update block, tensor).
PyObject* plan(PyObject* const* a) {
  launch(tensor(a[1], "tensor").device(), [p = block<const kvskip_plan_args>(a[0])](void* s) { return api.plan(p, s); });
  Py_RETURN_NONE;
}
PyObject* merge_update(PyObject* const* a) {
  const auto* p = block<const kvskip_attn_args>(a[0]);
  const auto* u = block<const kvskip_update_args>(a[1]);
  launch(tensor(a[2], "tensor").device(), [&](void* s) { return api.merge_update(p, u, s); });
  Py_RETURN_NONE;
}
// plan_scores(plan block, device index) / update(update block, device index); -1: the current device.
PyObject* plan_scores(PyObject* const* a) {
  launch(at::Device(at::kCUDA, static_cast<c10::DeviceIndex>(integer(a[1]))),
         [p = block<const kvskip_plan_args>(a[0])](void* s) { return api.plan_scores(p, s); });
  Py_RETURN_NONE;
}
PyObject* update(PyObject* const* a) {
  launch(at::Device(at::kCUDA, static_cast<c10::DeviceIndex>(integer(a[1]))),
         [p = block<const kvskip_update_args>(a[0])](void* s) { return api.update(p, s); });
  Py_RETURN_NONE;
}

// num_splits(bh, n_tiles, slots, max_splits, min_tiles): kvskip.num_splits_for's rule over `slots`
// resident workgroups, count by count in the same double arithmetic. In Python the scan took 45 us of a
// decode call at 32k (63.8 us a call, 27 of them kernels) and 80 us of a planner layer-step.
PyObject* num_splits(PyObject* const* a) {
  const int64_t bh = integer(a[0]), n = integer(a[1]), slots = integer(a[2]), cap = integer(a[3]), least = integer(a[4]);
  require(bh > 0 && slots > 0, "num_splits_for: bh >= 1 and at least one workgroup slot");
  auto score = [&](int64_t s) {
    const double waves = static_cast<double>(bh * s) / static_cast<double>(slots);
    return waves / std::ceil(waves) - 0.002 * static_cast<double>(s);
  };
  int64_t most = 1;  // ceil(n / s) only falls as s grows
  while (most < cap && std::ceil(static_cast<double>(n) / static_cast<double>(most + 1)) >= static_cast<double>(least))
    ++most;
  int64_t best = 1;
  double best_score = score(1);
  for (int64_t s = 2; s <= most; ++s) {
    const double x = score(s);
    if (x > best_score + 1e-9) best = s, best_score = x;
  }
  return PyLong_FromLongLong(best);
}

// zeroed(dtype-named shapes, tensor): tensors of zeros on the tensor's device, carved from one zeroed
// allocation (each 256-byte aligned): names = (("f4" | "i4" | "u1", shape), ...) -> list.
PyObject* zeroed(PyObject* const* a) {
  const at::Device dev = tensor(a[1], "tensor").device();
  struct Part {
    at::ScalarType ty;
    std::vector<int64_t> shape;
    int64_t at, bytes;
  };
  std::vector<Part> parts;
  int64_t total = 0;
  const Py_ssize_t n = PyTuple_Size(a[0]);
  if (n < 0) throw PyErr{};
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* e = PyTuple_GET_ITEM(a[0], i);
    const char* ty = PyTuple_Check(e) && PyTuple_Size(e) == 2 ? PyUnicode_AsUTF8(PyTuple_GET_ITEM(e, 0)) : nullptr;
    require(ty != nullptr, "zeroed: (type, shape) pairs");
    Part p{ty[0] == 'f' ? at::kFloat : ty[0] == 'i' ? at::kInt : at::kByte, {}, total, ty[0] == 'u' ? 1 : 4};
    PyObject* sh = PyTuple_GET_ITEM(e, 1);
    const Py_ssize_t dims = PyTuple_Size(sh);
    if (dims < 0) throw PyErr{};
    for (Py_ssize_t j = 0; j < dims; ++j) {
      p.shape.push_back(integer(PyTuple_GET_ITEM(sh, j)));
      p.bytes *= p.shape.back();
    }
    total += (p.bytes + 255) / 256 * 256;
    parts.push_back(std::move(p));
  }
  at::Tensor base = at::zeros({total}, at::TensorOptions().dtype(at::kByte).device(dev));
  PyObject* l = PyList_New(n);
  if (l == nullptr) throw PyErr{};
  for (Py_ssize_t i = 0; i < n; ++i) {
    const Part& p = parts[static_cast<size_t>(i)];
    PyList_SET_ITEM(l, i, THPVariable_Wrap(base.narrow(0, p.at, p.bytes).view(p.ty).view(p.shape)));
  }
  return l;
}

template <PyObject* (*F)(PyObject* const*), int N>
PyObject* call(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "kvskip_amd._host: %d arguments, got %zd", N, n);
    return nullptr;
  }
  if (raw_stream == nullptr) fail("kvskip_amd._host: bind() first");
  try {
    return F(a);
  } catch (const PyErr&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

// bind(addresses of Api's entry points in order, torch._C._cuda_getCurrentRawStream)
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !PyTuple_Check(a[0]) || PyTuple_Size(a[0]) != N_API) fail("bind: the entry points' addresses and torch's stream function");
  void* fn[N_API];
  for (int i = 0; i < N_API; ++i) {
    fn[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(a[0], i));
    if (fn[i] == nullptr) return nullptr;
  }
  std::memcpy(&api, fn, sizeof(api));
  Py_INCREF(a[1]);
  Py_XDECREF(raw_stream);
  raw_stream = a[1];
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

#define KVS_FN(f, n) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(call<f, n>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(bind)), METH_FASTCALL, nullptr},
    KVS_FN(decode, 17), KVS_FN(decode_into, 15), KVS_FN(splits_planned, 14), KVS_FN(splits_update, 13),
    KVS_FN(attn_block, 20), KVS_FN(vskip1, 13), KVS_FN(select, 10), KVS_FN(pv, 9), KVS_FN(pv_select, 13),
    KVS_FN(plan_block, 33), KVS_FN(update_block, 24), KVS_FN(plan, 2), KVS_FN(merge_update, 3), KVS_FN(plan_scores, 2),
    KVS_FN(update, 2), KVS_FN(num_splits, 5), KVS_FN(zeroed, 2),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
