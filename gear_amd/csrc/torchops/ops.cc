// Native module `_hostops`: the host side of gear_amd.ops and of a loader step -- checks, outputs,
// scratch, the call into libgearhip.so -- without Python between them.
//
// A step of a small batch is bound by the host: its kernels take 10 to 25 us, and the same work
// from Python (ctypes marshalling, a torch.empty per output, four to six attribute calls per
// tensor) took 35 to 60 us, of which the launches themselves are 2.6 us apiece.  Here a tensor
// costs an unpack and an output an allocation of the caching allocator (0.5 us).  The module links
// libtorch for that; it computes nothing on tensors.  Allocations and calls into the library run without
// the GIL: a launch that waits for room in its queue, or an allocation that waits for the driver, stops
// no other Python thread.
#include <ATen/ATen.h>
#include <ATen/hip/HIPGeneratorImpl.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <optional>
#include <string>
#include <tuple>
#include <unordered_map>
#include <vector>

#include "gear_hip.h"

namespace py = pybind11;

namespace {

// ---- arguments -----------------------------------------------------------------------------------
const char *dtype_text(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return "torch.float32";
    case at::kDouble: return "torch.float64";
    case at::kLong: return "torch.int64";
    case at::kByte: return "torch.uint8";
    default: return c10::toString(t);
  }
}

const at::Tensor &any_tensor(py::handle h, const char *name) {
  if (!THPVariable_Check(h.ptr())) throw py::type_error(std::string(name) + " must be a torch.Tensor");
  return THPVariable_Unpack(h.ptr());
}

const at::Tensor &need(py::handle h, at::ScalarType dtype, const char *name) {
  const at::Tensor &t = any_tensor(h, name);
  if (t.scalar_type() != dtype)
    throw py::type_error(std::string(name) + " must have dtype " + dtype_text(dtype) + ", got " +
                         std::string(py::str(h.attr("dtype"))));
  if (!t.is_contiguous()) throw py::value_error(std::string(name) + " must be contiguous");
  if (!t.is_cuda()) throw py::value_error(std::string(name) + " must live on the GPU");
  return t;
}

template <typename T>
T *ptr(const at::Tensor &t) {
  return static_cast<T *>(t.data_ptr());
}
// an optional output: the tensor, or null
template <typename T>
T *ptr_or_null(py::handle h, const char *name) {
  return h.is_none() ? nullptr : static_cast<T *>(any_tensor(h, name).data_ptr());
}

// (where the GIL is held)
at::Tensor empty(int64_t n, at::ScalarType dtype, const at::Device &device) {
  py::gil_scoped_release nogil;
  return at::empty({n}, at::TensorOptions().dtype(dtype).device(device));
}

py::object wrap(const at::Tensor &t) { return py::reinterpret_steal<py::object>(THPVariable_Wrap(t)); }

void *current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

// (with or without the GIL)
void check(const char *fn, int code) {
  if (code == 0) return;
  py::gil_scoped_acquire gil;
  py::module_::import("gear_amd._cabi").attr("check")(fn, code);  // raises
}

// ---- scratch -------------------------------------------------------------------------------------
// Scratch tensors per (purpose, device, stream), grown on demand and reused: no allocation in
// steady state, and calls enqueued on different streams never share a workspace.  Python sees
// get(); an instance whose get() was replaced is asked through it.
class Workspace {
 public:
  struct Entry {
    at::Tensor buf;
    std::mutex order;  // held while a call enqueues its launches on the buffer's stream
  };
  // (the GIL is held)
  std::shared_ptr<Entry> entry(const char *tag, const at::Device &device) {
    const c10::DeviceIndex index = device.has_index() ? device.index() : c10::hip::current_device();
    std::shared_ptr<Entry> &slot = entries_[Key{tag, index, c10::hip::getCurrentHIPStream(index).stream()}];
    if (!slot) slot = std::make_shared<Entry>();
    return slot;
  }
  static at::Tensor buffer(Entry &e, size_t bytes, const at::Device &device) {
    if (!e.buf.defined() || (size_t)e.buf.numel() < bytes) {
      at::Tensor grown = empty((int64_t)std::max<size_t>(bytes, 256), at::kByte, device);
      // (another thread may have been here meanwhile)
      if (!e.buf.defined() || e.buf.numel() < grown.numel()) e.buf = grown;
    }
    return e.buf;
  }

 private:
  struct Key {
    std::string tag;
    c10::DeviceIndex device;
    void *stream;
    bool operator==(const Key &o) const { return stream == o.stream && device == o.device && tag == o.tag; }
  };
  struct Hash {
    size_t operator()(const Key &k) const {
      return std::hash<std::string>()(k.tag) ^ (std::hash<void *>()(k.stream) * 31 + (size_t)k.device);
    }
  };
  std::unordered_map<Key, std::shared_ptr<Entry>, Hash> entries_;
};

struct Scratch {
  void *ptr = nullptr;
  size_t bytes = 0;
  at::Tensor keep;
  std::shared_ptr<Workspace::Entry> entry;
  Scratch() = default;  // none
  Scratch(py::handle ws, const char *tag, size_t want, const at::Device &device) {
    entry = ws.cast<Workspace &>().entry(tag, device);
    PyObject **dict = _PyObject_GetDictPtr(ws.ptr());
    if (dict != nullptr && *dict != nullptr && PyDict_GET_SIZE(*dict) != 0)
      keep = THPVariable_Unpack(
          ws.attr("get")(tag, want, py::reinterpret_steal<py::object>(THPDevice_New(device))).ptr());
    else
      keep = Workspace::buffer(*entry, want, device);
    ptr = keep.data_ptr();
    bytes = (size_t)keep.numel();
  }
};

// f(args) without the GIL.  Two threads that enqueue on one stream share its scratch: the launches of
// one call follow each other, so that no other call's lie between them.
template <typename F>
int launches(const Scratch &s, const F &f) {
  if (!s.entry) return f();
  std::lock_guard<std::mutex> order(s.entry->order);
  return f();
}
template <typename F, typename... A>
void call(const char *name, const Scratch &s, const F &f, A... args) {
  int code;
  {
    py::gil_scoped_release nogil;
    code = launches(s, [&] { return f(args...); });
  }
  check(name, code);
}

// ---- prefix sums -----------------------------------------------------------------------------------
template <typename Launch>
py::object prefix(py::handle in, py::object out, py::handle ws, at::ScalarType from, at::ScalarType to,
                  const char *name, const char *fn, const Launch &launch) {
  const at::Tensor &p = need(in, from, name);
  const int64_t n = p.numel();
  if (out.is_none()) {
    out = wrap(empty(n, to, p.device()));
  } else if (need(out, to, "out").numel() < n) {
    throw py::value_error("out is too small");
  }
  Scratch s(ws, "scan", gear_hip_scan_workspace_bytes(n), p.device());
  call(fn, s, launch, p.data_ptr(), THPVariable_Unpack(out.ptr()).data_ptr(), n, s.ptr, s.bytes,
       current_stream());
  return out;
}

py::object prefix_sum(py::handle in, py::object out, py::handle ws) {
  return prefix(in, std::move(out), ws, at::kFloat, at::kDouble, "priorities", "gear_hip_scan_f32_f64",
                [](void *i, void *o, int64_t n, void *w, size_t b, void *st) {
                  return gear_hip_scan_f32_f64(static_cast<float *>(i), static_cast<double *>(o), n, w, b, st);
                });
}

py::object prefix_sum_i64(py::handle in, py::object out, py::handle ws) {
  return prefix(in, std::move(out), ws, at::kLong, at::kLong, "weights", "gear_hip_scan_i64",
                [](void *i, void *o, int64_t n, void *w, size_t b, void *st) {
                  return gear_hip_scan_i64(static_cast<int64_t *>(i), static_cast<int64_t *>(o), n, w, b, st);
                });
}

// first_changed <= 0: full scan
void rescan(const at::Tensor &in, const at::Tensor &out, int64_t first_changed, const at::Tensor &ws) {
  if (first_changed <= 0)
    call("gear_hip_scan_f32_f64", Scratch(), gear_hip_scan_f32_f64, ptr<float>(in), ptr<double>(out),
         in.numel(), ws.data_ptr(), (size_t)ws.numel(), current_stream());
  else
    call("gear_hip_rescan_f32_f64", Scratch(), gear_hip_rescan_f32_f64, ptr<float>(in),
         ptr<double>(out), in.numel(), first_changed, ws.data_ptr(), (size_t)ws.numel(),
         current_stream());
}

// ---- draws -----------------------------------------------------------------------------------------
py::object upper_bound(py::handle prefix_, py::handle u_, bool unit, py::object idx_out, py::handle pri,
                       double beta, py::object weights_out, py::handle ws) {
  const at::Tensor &prefix = need(prefix_, at::kDouble, "prefix"), &u = need(u_, at::kFloat, "u");
  const int64_t num = u.numel(), n = prefix.numel();
  if (idx_out.is_none())
    idx_out = wrap(empty(num, at::kLong, u.device()));
  else
    need(idx_out, at::kLong, "idx_out");
  int64_t *idx = ptr<int64_t>(THPVariable_Unpack(idx_out.ptr()));
  if (pri.is_none()) {
    call("gear_hip_upper_bound_f64", Scratch(), gear_hip_upper_bound_f64, ptr<double>(prefix), n,
         ptr<float>(u), num, unit, idx, nullptr, beta, nullptr, nullptr, 0, current_stream());
    return idx_out;
  }
  const at::Tensor &p = need(pri, at::kFloat, "priorities");
  if (p.numel() != n) throw py::value_error("priorities and prefix differ in length");
  if (weights_out.is_none()) weights_out = wrap(empty(num, at::kFloat, u.device()));
  Scratch s(ws, "search", gear_hip_search_workspace_bytes(num), u.device());
  call("gear_hip_upper_bound_f64", s, gear_hip_upper_bound_f64, ptr<double>(prefix), n, ptr<float>(u),
       num, unit, idx, ptr<float>(p), beta, ptr_or_null<float>(weights_out, "weights_out"), s.ptr,
       s.bytes, current_stream());
  return py::make_tuple(std::move(idx_out), std::move(weights_out));
}

py::object upper_bound_i64(py::handle prefix_, py::handle u_, bool unit, py::object idx_out) {
  const at::Tensor &prefix = need(prefix_, at::kLong, "prefix");
  const at::Tensor &u = need(u_, unit ? at::kDouble : at::kLong, "u");
  if (idx_out.is_none()) idx_out = wrap(empty(u.numel(), at::kLong, u.device()));
  call("gear_hip_upper_bound_i64", Scratch(), gear_hip_upper_bound_i64, ptr<int64_t>(prefix),
       prefix.numel(), u.data_ptr(), u.numel(), unit, ptr_or_null<int64_t>(idx_out, "idx_out"),
       current_stream());
  return idx_out;
}

py::object sample_sorted(py::handle prefix_, py::handle u_, bool unit, py::object sorted_out,
                         int64_t trajectory_length, int64_t modulo, py::object idxs, py::object tss,
                         py::object lens, py::handle ws) {
  const at::Tensor &prefix = need(prefix_, at::kDouble, "prefix"), &u = need(u_, at::kFloat, "u");
  const int64_t num = u.numel();
  auto output = [&](py::object &o) {
    if (o.is_none()) o = wrap(empty(num, at::kLong, u.device()));
  };
  output(sorted_out);
  if (trajectory_length > 0) {
    output(idxs);
    output(tss);
    output(lens);
  }
  Scratch s(ws, "sample", gear_hip_sample_workspace_bytes(num), u.device());
  call("gear_hip_sample_sorted_f64", s, gear_hip_sample_sorted_f64, ptr<double>(prefix),
       prefix.numel(), ptr<float>(u), num, unit, ptr_or_null<int64_t>(sorted_out, "sorted_out"),
       trajectory_length, modulo, ptr_or_null<int64_t>(idxs, "idxs"), ptr_or_null<int64_t>(tss, "tss"),
       ptr_or_null<int64_t>(lens, "lens"), s.ptr, s.bytes, current_stream());
  if (trajectory_length > 0)
    return py::make_tuple(std::move(sorted_out), std::move(idxs), std::move(tss), std::move(lens));
  return sorted_out;
}

// The tables and outputs that the look-up calls share.
struct LookupArgs {
  const int64_t *index_table = nullptr, *lengths_table = nullptr;
  int64_t index_n = 0, lengths_n = 0;
  py::object sampled, local, lens;
  LookupArgs(int64_t num, const at::Device &device, py::handle index_table_, py::handle lengths_table_,
             py::object sampled_, py::object local_, py::object lens_)
      : sampled(std::move(sampled_)), local(std::move(local_)), lens(std::move(lens_)) {
    if (!index_table_.is_none()) {
      const at::Tensor &t = need(index_table_, at::kLong, "index_table");
      index_table = ptr<int64_t>(t);
      index_n = t.numel();
    }
    if (!lengths_table_.is_none()) {
      const at::Tensor &t = need(lengths_table_, at::kLong, "lengths_table");
      lengths_table = ptr<int64_t>(t);
      lengths_n = t.numel();
    }
    if (sampled.is_none()) sampled = wrap(empty(num, at::kLong, device));
    if (local.is_none()) local = wrap(empty(num, at::kLong, device));
    if (lens.is_none() && lengths_table) lens = wrap(empty(num, at::kLong, device));
  }
  int64_t *sampled_ptr() const { return ptr_or_null<int64_t>(sampled, "sampled_out"); }
  int64_t *local_ptr() const { return ptr_or_null<int64_t>(local, "local_out"); }
  int64_t *lens_ptr() const { return ptr_or_null<int64_t>(lens, "lens_out"); }
};

py::object sample_lookup(py::handle prefix_, py::handle u_, bool unit, py::handle index_table,
                         int64_t index_offset, py::handle lengths_table, py::object sampled_out,
                         py::object local_out, py::object lens_out, py::handle start_uniforms,
                         int64_t window, py::object starts_out, py::handle ws) {
  const bool i64 = any_tensor(prefix_, "prefix").scalar_type() == at::kLong;
  if (!start_uniforms.is_none() && !i64)
    throw py::value_error("window starts come with an int64 prefix only");
  const at::Tensor &prefix = need(prefix_, i64 ? at::kLong : at::kDouble, "prefix");
  const at::Tensor &u = need(u_, i64 ? (unit ? at::kDouble : at::kLong) : at::kFloat, "u");
  const int64_t num = u.numel();
  LookupArgs a(num, u.device(), index_table, lengths_table, std::move(sampled_out),
               std::move(local_out), std::move(lens_out));
  if (a.index_table && a.index_n != prefix.numel())
    throw py::value_error("index_table and prefix differ in length");
  Scratch s(ws, "sample", gear_hip_sample_workspace_bytes(num), u.device());
  if (!i64) {
    call("gear_hip_sample_lookup_f64", s, gear_hip_sample_lookup_f64, ptr<double>(prefix),
         prefix.numel(), ptr<float>(u), num, unit, a.index_table, index_offset, a.lengths_table,
         a.lengths_n, a.sampled_ptr(), a.local_ptr(), a.lens_ptr(), s.ptr, s.bytes, current_stream());
    return py::make_tuple(a.sampled, a.local, a.lens);
  }
  const double *v = nullptr;
  int64_t *starts = nullptr;
  if (!start_uniforms.is_none()) {
    const at::Tensor &t = need(start_uniforms, at::kDouble, "start_uniforms");
    if (t.numel() != num || !a.lengths_table || window < 1)
      throw py::value_error("window starts need a uniform per draw, lengths_table and window >= 1");
    v = ptr<double>(t);
    if (starts_out.is_none()) starts_out = wrap(empty(num, at::kLong, u.device()));
    starts = ptr_or_null<int64_t>(starts_out, "starts_out");
  }
  call("gear_hip_sample_lookup_i64", s, gear_hip_sample_lookup_i64, ptr<int64_t>(prefix),
       prefix.numel(), u.data_ptr(), num, unit, a.index_table, index_offset, a.lengths_table,
       a.lengths_n, a.sampled_ptr(), a.local_ptr(), a.lens_ptr(), v, window, starts, s.ptr, s.bytes,
       current_stream());
  if (starts) return py::make_tuple(a.sampled, a.local, a.lens, starts_out);
  return py::make_tuple(a.sampled, a.local, a.lens);
}

py::object sort_lookup(py::handle positions_, int64_t bound, py::handle index_table,
                       int64_t index_offset, py::handle lengths_table, py::object sampled_out,
                       py::object local_out, py::object lens_out, py::handle ws) {
  const at::Tensor &positions = need(positions_, at::kLong, "positions");
  const int64_t num = positions.numel();
  LookupArgs a(num, positions.device(), index_table, lengths_table, std::move(sampled_out),
               std::move(local_out), std::move(lens_out));
  Scratch s(ws, "sample", gear_hip_sample_workspace_bytes(num), positions.device());
  call("gear_hip_sort_lookup_i64", s, gear_hip_sort_lookup_i64, ptr<int64_t>(positions), num, bound,
       a.index_table, a.index_n, index_offset, a.lengths_table, a.lengths_n, a.sampled_ptr(),
       a.local_ptr(), a.lens_ptr(), s.ptr, s.bytes, current_stream());
  return py::make_tuple(a.sampled, a.local, a.lens);
}

py::object lookup(py::handle positions_, py::handle index_table, int64_t index_offset,
                  py::handle lengths_table, py::object sampled_out, py::object local_out,
                  py::object lens_out) {
  const at::Tensor &positions = need(positions_, at::kLong, "positions");
  const int64_t num = positions.numel();
  LookupArgs a(num, positions.device(), index_table, lengths_table, std::move(sampled_out),
               std::move(local_out), std::move(lens_out));
  call("gear_hip_lookup_i64", Scratch(), gear_hip_lookup_i64, ptr<int64_t>(positions), num,
       a.index_table, a.index_n, index_offset, a.lengths_table, a.lengths_n, a.sampled_ptr(),
       a.local_ptr(), a.lens_ptr(), current_stream());
  return py::make_tuple(a.sampled, a.local, a.lens);
}

py::object take_i64(py::handle table_, py::handle idx_, int64_t add, py::object out) {
  const at::Tensor &table = need(table_, at::kLong, "table"), &idx = need(idx_, at::kLong, "idx");
  if (out.is_none()) out = wrap(empty(idx.numel(), at::kLong, idx.device()));
  call("gear_hip_take_i64", Scratch(), gear_hip_take_i64, ptr<int64_t>(table), table.numel(),
       ptr<int64_t>(idx), idx.numel(), add, ptr_or_null<int64_t>(out, "out"), current_stream());
  return out;
}

py::object take_sorted(py::handle table_, py::handle idx_, py::handle ws) {
  const at::Tensor &table = need(table_, at::kLong, "table"), &idx = need(idx_, at::kLong, "idx");
  const int64_t num = idx.numel();
  py::object out = wrap(empty(num, at::kLong, idx.device()));
  Scratch s(ws, "take_sorted", gear_hip_take_sorted_workspace_bytes(num), idx.device());
  call("gear_hip_take_sorted_i64", s, gear_hip_take_sorted_i64, ptr<int64_t>(table), table.numel(),
       ptr<int64_t>(idx), num, ptr<int64_t>(THPVariable_Unpack(out.ptr())), s.ptr, s.bytes, current_stream());
  return out;
}

// ---- sort, top-k, updates --------------------------------------------------------------------------
py::object sort_i64(py::handle keys_, py::handle vals_, int64_t key_bits, py::handle ws) {
  const at::Tensor &keys = need(keys_, at::kLong, "keys");
  const int64_t num = keys.numel();
  auto like = [](const at::Tensor &t) {
    py::gil_scoped_release nogil;
    return at::empty_like(t);
  };
  py::object keys_out = wrap(like(keys)), vals_out = py::none();
  const int64_t *vals = nullptr;
  if (!vals_.is_none()) {
    const at::Tensor &v = need(vals_, at::kLong, "vals");
    vals = ptr<int64_t>(v);
    vals_out = wrap(like(v));
  }
  Scratch s(ws, "sort", gear_hip_sort_workspace_bytes(num), keys.device());
  call("gear_hip_sort_i64", s, gear_hip_sort_i64, ptr<int64_t>(keys), ptr_or_null<int64_t>(keys_out,
       "keys_out"), vals, ptr_or_null<int64_t>(vals_out, "vals_out"), num, (int)key_bits, s.ptr,
       s.bytes, current_stream());
  if (vals) return py::make_tuple(std::move(keys_out), std::move(vals_out));
  return keys_out;
}

py::object topk(py::handle priorities, int64_t k, bool by_value, bool want_values, bool warm,
                py::handle workspace, py::handle ws) {
  const at::Tensor &p = need(priorities, at::kFloat, "priorities");
  const int64_t n = p.numel();
  py::object vals = py::none();
  if (want_values) vals = wrap(empty(k, at::kFloat, p.device()));
  py::object idx = wrap(empty(k, at::kLong, p.device()));
  const size_t want = gear_hip_topk_workspace_bytes(n, k);
  const Scratch s = workspace.is_none() ? Scratch(ws, "topk", want, p.device()) : Scratch();
  const at::Tensor &buf = workspace.is_none() ? s.keep : any_tensor(workspace, "workspace");
  if ((size_t)buf.numel() < want)
    throw py::value_error("top-k workspace holds " + std::to_string(buf.numel()) + " bytes, " +
                          std::to_string(want) + " needed");
  const auto fn = warm ? gear_hip_topk_f32_warm : gear_hip_topk_f32;
  call(warm ? "gear_hip_topk_f32_warm" : "gear_hip_topk_f32", s, fn, ptr<float>(p), n, k, by_value,
       ptr_or_null<float>(vals, "values"), ptr_or_null<int64_t>(idx, "indices"), buf.data_ptr(),
       (size_t)buf.numel(), current_stream());
  return py::make_tuple(std::move(vals), std::move(idx));
}

py::object scatter(py::object weights_, py::handle idx_, py::handle values_, bool unique, py::handle ws) {
  const at::ScalarType dtype = any_tensor(weights_, "weights").scalar_type();
  if (dtype != at::kFloat && dtype != at::kLong)
    throw py::type_error("scatter works on float32 or int64 tables");
  const at::Tensor &weights = need(weights_, dtype, "weights"), &idx = need(idx_, at::kLong, "idx"),
                   &values = need(values_, dtype, "values");
  const int64_t num = idx.numel();
  if (values.numel() != num) throw py::value_error("idx and values differ in length");
  const Scratch s = unique ? Scratch()
                           : Scratch(ws, "scatter", gear_hip_scatter_workspace_bytes(num), weights.device());
  if (dtype == at::kFloat)
    call("gear_hip_scatter_f32", s, gear_hip_scatter_f32, ptr<float>(weights), weights.numel(),
         ptr<int64_t>(idx), ptr<float>(values), num, unique, s.ptr, s.bytes, current_stream());
  else
    call("gear_hip_scatter_i64", s, gear_hip_scatter_i64, ptr<int64_t>(weights), weights.numel(),
         ptr<int64_t>(idx), ptr<int64_t>(values), num, unique, s.ptr, s.bytes, current_stream());
  return weights_;
}

// ---- gathers ---------------------------------------------------------------------------------------
// Column descriptors of gear_hip_subcopy_multi_checked made once; run() takes the three index
// tensors of a step.
struct Gather {
  uintptr_t src;
  int64_t traj_stride, num, capacity, trajectory_length;
  std::vector<gear_hip_column_desc> descs;

  Gather(uintptr_t src, int64_t traj_stride, int64_t num, int64_t capacity, int64_t trajectory_length,
         const std::vector<std::tuple<uintptr_t, uintptr_t, int64_t, int64_t, int64_t, int64_t, int64_t,
                                      bool, bool>> &columns)
      : src(src), traj_stride(traj_stride), num(num), capacity(capacity),
        trajectory_length(trajectory_length) {
    for (const auto &c : columns) {
      gear_hip_column_desc d;
      d.dst = reinterpret_cast<void *>(std::get<0>(c));
      d.mask_out = reinterpret_cast<uint8_t *>(std::get<1>(c));
      d.ofst = std::get<2>(c);
      d.span = std::get<3>(c);
      d.step_bytes = std::get<4>(c);
      d.col_base = std::get<5>(c);
      d.dst_stride = std::get<6>(c);
      d.pad_head = std::get<7>(c) ? 1 : 0;
      d.zero_fill = std::get<8>(c) ? 1 : 0;
      descs.push_back(d);
    }
  }

  void run(py::handle idxs_, py::handle tss_, py::handle lens_) const {
    const at::Tensor &idxs = any_tensor(idxs_, "idxs"), &tss = any_tensor(tss_, "tss"),
                     &lens = any_tensor(lens_, "lens");
    if (idxs.numel() != num || tss.numel() != num || lens.numel() != num)
      throw py::value_error("the plan was made for " + std::to_string(num) + " windows");
    if (idxs.scalar_type() != at::kLong || tss.scalar_type() != at::kLong ||
        lens.scalar_type() != at::kLong)
      throw py::type_error("idxs, tss and lens must be int64 tensors");
    const c10::DeviceIndex dev = idxs.is_cuda() ? idxs.get_device() : c10::hip::current_device();
    call("gear_hip_subcopy_multi_checked", Scratch(), gear_hip_subcopy_multi_checked,
         reinterpret_cast<const void *>(src), num, ptr<int64_t>(idxs), ptr<int64_t>(tss),
         ptr<int64_t>(lens), traj_stride, capacity, trajectory_length, descs.data(), (int)descs.size(),
         c10::hip::getCurrentHIPStream(dev).stream());
  }
};

// ---- a loader step ---------------------------------------------------------------------------------
// What a loader's step does after the draws: the batch is selected and looked up, its tensors are
// allocated and all subscribed columns gathered, with the offline convention timestep == length
// (gear/loader/offline_loader.py:155-204).  Holds what does not change from step to step; the
// table's address is asked for at each step.
void hip(const char *what, hipError_t e) {
  if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

// Pinned memory for lengths on their way to the host.  Memory that a kernel may still write (an error
// between its launch and the end of the wait) is waited for, or never given back where not even that
// works: the next pinned tensor would be written over.
struct Staging {
  at::Tensor buf;
  hipStream_t pending = nullptr;  // the stream of a kernel that may write buf
  bool is_pending = false;
  Staging() = default;
  Staging(const Staging &) = delete;
  Staging &operator=(const Staging &) = delete;
  void swap(Staging &o) {
    std::swap(buf, o.buf);
    std::swap(pending, o.pending);
    std::swap(is_pending, o.is_pending);
  }
  ~Staging() {
    if (is_pending && hipStreamSynchronize(pending) != hipSuccess) (void)buf.unsafeReleaseIntrusivePtr().release();
  }

  // Lengths that a kernel stores in buf one by one are there when none of them is the mark that was put
  // there before; an event between the two costs the host 5.7 us to record and the wait 6 us more
  // (after one kernel 7.8 instead of 13.5, after four 17.5 instead of 22.9).  A wait that gets long -- work
  // of the caller's ahead of the kernel, more lengths than are worth looking at, a length that is the
  // mark -- ends with the stream's.
  static constexpr int64_t kMark = INT64_MIN, kMostMarked = 8192;
  static constexpr int kSpins = 100000;  // reads of memory; a tenth of a millisecond and more
  void mark(int64_t num) {
    if (num <= kMostMarked) std::fill_n(ptr<int64_t>(buf), num, kMark);
  }
  void wait(int64_t num) {
    bool arrived = num <= kMostMarked;
    const volatile int64_t *at = ptr<int64_t>(buf);
    for (int64_t i = 0, spins = 0; arrived && i < num; ++i)
      while (at[i] == kMark)
        if (++spins > kSpins) {
          arrived = false;
          break;
        }
    if (!arrived) hip("stream wait", hipStreamSynchronize(pending));
    std::atomic_thread_fence(std::memory_order_acquire);
    is_pending = false;
  }
};

// ---- draws -----------------------------------------------------------------------------------------
// A batch of random numbers from a torch generator costs a call of torch's, 6 us of the host and a launch of
// 2.2 us, for numbers that a few instructions give where they are used (philox.hpp).  Only where a call
// of torch's would take one block of the generator's stream a draw, and not while the stream is captured,
// when the generator's state is not the host's to read.
bool draws_here(const at::Generator &gen, bool weighted, int64_t range, int64_t num, const at::Device &device) {
  if (!gen.defined() || gen.device().type() != at::kCUDA || num < 1 || num > gear_hip_draw_max()) return false;
  if (gen.device().index() != (device.has_index() ? device.index() : c10::hip::current_device())) return false;
  if (!weighted && (range < 1 || range > gear_hip_draw_max_bound())) return false;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(static_cast<hipStream_t>(current_stream()), &capture) == hipSuccess &&
         capture == hipStreamCaptureStatusNone;
}
py::object torch_draws(const at::Generator &gen, bool weighted, int64_t range, int64_t num,
                       const at::Device &device) {
  at::Tensor t;
  {
    py::gil_scoped_release nogil;
    const auto options = at::TensorOptions().device(device);
    t = weighted ? at::rand({num}, gen, options.dtype(at::kFloat))
                 : at::randint(range, {num}, gen, options.dtype(at::kLong));
  }
  return wrap(t);
}
// the seed and the offset of the next call's numbers, which are taken from the generator
std::pair<uint64_t, uint64_t> next_block(at::Generator &gen) {
  std::lock_guard<std::mutex> lock(gen.mutex());
  const auto state = at::check_generator<at::CUDAGeneratorImpl>(gen)->philox_cuda_state(4);
  return {state.seed_.val, state.offset_.val};
}

class LoaderStep {
 public:
  struct Column {
    at::ScalarType dtype;
    std::vector<int64_t> shape;  // of one window: [length, ...]
    int64_t ofst, span, step_bytes, col_base;
    bool pad_head;
  };

  LoaderStep(py::object table, int64_t traj_stride, int64_t capacity, int64_t trajectory_length,
             const py::list &columns, bool with_mask, const at::Device &device)
      : table_(std::move(table)), traj_stride_(traj_stride), capacity_(capacity),
        trajectory_length_(trajectory_length), with_mask_(with_mask), device_(device) {
    for (py::handle h : columns) {
      py::tuple c = py::reinterpret_borrow<py::tuple>(h);
      if (!THPDtype_Check(c[0].ptr())) throw py::type_error("a column's dtype must be a torch.dtype");
      columns_.push_back(Column{reinterpret_cast<THPDtype *>(c[0].ptr())->scalar_type,
                                c[1].cast<std::vector<int64_t>>(), c[2].cast<int64_t>(),
                                c[3].cast<int64_t>(), c[4].cast<int64_t>(), c[5].cast<int64_t>(),
                                c[6].cast<bool>()});
    }
    if (columns_.size() > GEAR_HIP_MAX_COLUMNS)
      throw std::runtime_error("more than 16 columns: one launch gathers 16 at most");
  }

  // kind, draws, prefix: as WeightedSampler / UniformSampler / TopKSampler.prepare() return them; or the
  // generator to draw from and how many draws there are: the same draws, worked out where they are used.
  // Returns (sampled, timesteps, [batch tensors], [masks] or None); the timesteps on the host when
  // host_timesteps is set.
  py::tuple run(const std::string &kind, py::object draws_, py::handle prefix_, py::handle indices_,
                int64_t index_offset, py::handle timesteps_, bool host_timesteps, py::handle ws, int64_t to_draw) {
    const at::Tensor &indices = need(indices_, at::kLong, "indices"),
                     &timesteps = need(timesteps_, at::kLong, "timesteps");
    const bool weighted = kind == "weighted";
    const bool uniform = kind == "uniform";
    if (!weighted && !uniform && kind != "positions")
      throw std::invalid_argument("kind must be 'weighted', 'uniform' or 'positions'");
    std::optional<at::Generator> generator;
    if (to_draw >= 0) {
      generator = draws_.cast<at::Generator>();
      if (!draws_here(*generator, weighted, indices.numel(), to_draw, device_)) {
        draws_ = torch_draws(*generator, weighted, indices.numel(), to_draw, device_);
        generator.reset();
      }
    }
    const at::Tensor none;
    const at::Tensor &draws = generator ? none : need(draws_, weighted ? at::kFloat : at::kLong, "draws");
    const int64_t num = generator ? to_draw : draws.numel();
    const uintptr_t base = table_.attr("device_address").cast<uintptr_t>();
    if (base == 0)
      throw std::runtime_error(
          "table memory is not visible to the GPU: connect() it, with placement 'pinned' or 'device'");
    const double *prefix = nullptr;
    if (weighted) {
      const at::Tensor &p = need(prefix_, at::kDouble, "prefix");
      if (p.numel() != indices.numel()) throw std::runtime_error("prefix and indices differ in length");
      prefix = ptr<double>(p);
    }
    Scratch w;
    if (weighted || uniform) w = Scratch(ws, "sample", gear_hip_sample_workspace_bytes(num), device_);
    void *st = current_stream();
    at::Tensor sampled, lens, host;
    std::vector<at::Tensor> batch(columns_.size()), masks(with_mask_ ? columns_.size() : 0);
    Staging staged;
    if (host_timesteps) staged.swap(staging_);
    {
      py::gil_scoped_release nogil;
      const auto on_gpu = at::TensorOptions().device(device_);
      sampled = at::empty({num}, on_gpu.dtype(at::kLong));
      lens = at::empty({num}, on_gpu.dtype(at::kLong));
      const at::Tensor local = at::empty({num}, on_gpu.dtype(at::kLong));
      if (host_timesteps) host = at::empty({num}, at::TensorOptions().dtype(at::kLong));
      std::vector<gear_hip_column_desc> descs(columns_.size());
      std::vector<int64_t> shape;
      for (size_t k = 0; k < columns_.size(); ++k) {
        const Column &c = columns_[k];
        shape.assign(1, num);
        shape.insert(shape.end(), c.shape.begin(), c.shape.end());
        batch[k] = at::empty(shape, on_gpu.dtype(c.dtype));
        if (with_mask_) masks[k] = at::empty({num, c.span}, on_gpu.dtype(at::kByte));
        gear_hip_column_desc &d = descs[k];
        d.dst = batch[k].data_ptr();
        d.mask_out = with_mask_ ? ptr<uint8_t>(masks[k]) : nullptr;
        d.ofst = c.ofst;
        d.span = c.span;
        d.step_bytes = c.step_bytes;
        d.col_base = c.col_base;
        d.dst_stride = c.span * c.step_bytes;
        d.pad_head = c.pad_head ? 1 : 0;
        d.zero_fill = 1;
      }
      const int64_t *table = ptr<int64_t>(indices), *lengths = ptr<int64_t>(timesteps);
      int64_t *s = ptr<int64_t>(sampled), *l = ptr<int64_t>(local), *len = ptr<int64_t>(lens);
      const int64_t count = indices.numel();
      uint64_t seed = 0, offset = 0;
      if (generator) std::tie(seed, offset) = next_block(*generator);
      if (generator && weighted)
        check("gear_hip_draw_lookup_f64", launches(w, [&] {
                return gear_hip_draw_lookup_f64(prefix, count, seed, offset, num, table, index_offset, lengths,
                                                timesteps.numel(), s, l, len, w.ptr, w.bytes, st);
              }));
      else if (generator)
        check("gear_hip_draw_sort_lookup_i64", launches(w, [&] {
                return gear_hip_draw_sort_lookup_i64(seed, offset, num, count, table, count, index_offset,
                                                     lengths, timesteps.numel(), s, l, len, w.ptr, w.bytes, st);
              }));
      else if (weighted)
        check("gear_hip_sample_lookup_f64", launches(w, [&] {
                return gear_hip_sample_lookup_f64(prefix, indices.numel(), ptr<float>(draws), num, 1, table,
                                                  index_offset, lengths, timesteps.numel(), s, l, len, w.ptr,
                                                  w.bytes, st);
              }));
      else if (uniform)
        check("gear_hip_sort_lookup_i64", launches(w, [&] {
                return gear_hip_sort_lookup_i64(ptr<int64_t>(draws), num, std::max<int64_t>(indices.numel(), 1),
                                                table, indices.numel(), index_offset, lengths,
                                                timesteps.numel(), s, l, len, w.ptr, w.bytes, st);
              }));
      else
        check("gear_hip_lookup_i64",
              gear_hip_lookup_i64(ptr<int64_t>(draws), num, table, indices.numel(), index_offset, lengths,
                                  timesteps.numel(), s, l, len, st));
      if (num > 0)
        check("gear_hip_subcopy_multi_checked",
              gear_hip_subcopy_multi_checked(reinterpret_cast<const void *>(base), num, l, len, len,
                                             traj_stride_, capacity_, trajectory_length_, descs.data(),
                                             (int)descs.size(), st));
      // The lengths on the host.  The call returns when the gather has ended, as one that copied the
      // lengths behind it: a table in host memory may be written again, and the batch read on any stream.
      // (The staging buffer leaves the object for the time of the call: another thread that comes
      // in meanwhile makes one of its own.)
      if (host_timesteps && num > 0) {
        if (!staged.buf.defined() || staged.buf.numel() < num)
          staged.buf = at::empty({num}, at::TensorOptions().dtype(at::kLong).pinned_memory(true));
        staged.mark(num);
        staged.pending = static_cast<hipStream_t>(st);
        staged.is_pending = true;
        check("gear_hip_take_i64", gear_hip_take_i64(lengths, timesteps.numel(), l, num, 0,
                                                     ptr<int64_t>(staged.buf), st));
        staged.wait(num);
        std::memcpy(host.data_ptr(), staged.buf.data_ptr(), (size_t)num * 8);
      }
    }
    if (host_timesteps) staged.swap(staging_);
    py::list batch_list(columns_.size());
    py::object mask_list = py::none();
    if (with_mask_) mask_list = py::list(columns_.size());
    for (size_t k = 0; k < columns_.size(); ++k) {
      PyList_SET_ITEM(batch_list.ptr(), (Py_ssize_t)k, THPVariable_Wrap(batch[k]));
      if (with_mask_) PyList_SET_ITEM(mask_list.ptr(), (Py_ssize_t)k, THPVariable_Wrap(masks[k]));
    }
    return py::make_tuple(wrap(sampled), wrap(host_timesteps ? host : lens), batch_list, mask_list);
  }

 private:
  py::object table_;
  int64_t traj_stride_, capacity_, trajectory_length_;
  bool with_mask_;
  at::Device device_;
  std::vector<Column> columns_;
  Staging staging_;
};

}  // namespace

PYBIND11_MODULE(_hostops, m) {
  py::class_<Workspace>(m, "Workspace", py::dynamic_attr())
      .def(py::init<>())
      .def("get", [](Workspace &w, const std::string &tag, size_t bytes, const at::Device &device) {
        const std::shared_ptr<Workspace::Entry> e = w.entry(tag.c_str(), device);
        return wrap(Workspace::buffer(*e, bytes, device));
      });
  m.def("prefix_sum", &prefix_sum);
  m.def("prefix_sum_i64", &prefix_sum_i64);
  m.def("rescan", [](py::handle in, py::handle out, int64_t first_changed, py::handle ws) {
    rescan(any_tensor(in, "priorities"), any_tensor(out, "out"), first_changed,
           any_tensor(ws, "workspace"));
  });
  m.def("upper_bound", &upper_bound);
  m.def("upper_bound_i64", &upper_bound_i64);
  m.def("sample_sorted", &sample_sorted);
  m.def("sample_lookup", &sample_lookup);
  m.def("sort_lookup", &sort_lookup);
  m.def("lookup", &lookup);
  m.def("take_i64", &take_i64);
  m.def("take_sorted", &take_sorted);
  m.def("sort_i64", &sort_i64);
  m.def("topk", &topk);
  m.def("scatter", &scatter);
  py::class_<Gather>(m, "Gather")
      .def(py::init<uintptr_t, int64_t, int64_t, int64_t, int64_t,
                    const std::vector<std::tuple<uintptr_t, uintptr_t, int64_t, int64_t, int64_t, int64_t,
                                                 int64_t, bool, bool>> &>())
      .def("run", &Gather::run);
  py::class_<LoaderStep>(m, "LoaderStep")
      .def(py::init<py::object, int64_t, int64_t, int64_t, const py::list &, bool, const at::Device &>())
      .def("run", &LoaderStep::run, py::arg("kind"), py::arg("draws"), py::arg("prefix"), py::arg("indices"),
           py::arg("index_offset"), py::arg("timesteps"), py::arg("host_timesteps"), py::arg("ws"),
           py::arg("to_draw") = -1);
}
