"""Tensor-level entry points over the C ABI (include/gear_hip.h).

torch tensors are used for what they are here: handles to device memory plus the current HIP
stream.  All arithmetic happens in libgearhip.so; nothing in this module computes on tensors and
nothing falls back to torch or to the CPU.
"""
import ctypes
import functools

import torch

from . import _cabi
from ._cabi import ColumnDesc, call, load

try:
    from . import _hostops  # checks, outputs, scratch and calls of the functions below, natively
except ImportError as _e:  # pragma: no cover - only without a build
    raise ImportError(
        "gear_amd.ops: the native module _hostops is not built; run "
        "`python -c 'import __graft_entry__ as g; g.build()'` in the repository root") from _e


# torch's C accessor for the raw current stream (a fraction of the cost of
# torch.cuda.current_stream(), which builds a Stream object through several Python layers)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_cur_device = getattr(torch._C, "_cuda_getDevice", None)


def _stream_value(device=None):
    if _raw_stream is not None and _cur_device is not None:
        index = device.index if (device is not None and device.index is not None) \
            else _cur_device()
        return _raw_stream(index)
    return torch.cuda.current_stream(device).cuda_stream


def _stream():
    # (plain integers: ctypes converts them for the void* parameters itself, and building a
    # c_void_p object per argument is a measurable part of a small step)
    return _stream_value()


def _ptr(t):
    if t is None:
        return None
    return t.data_ptr()


def _need(t, dtype, name, device=True):
    if not isinstance(t, torch.Tensor):
        raise TypeError("%s must be a torch.Tensor" % name)
    if t.dtype != dtype:
        raise TypeError("%s must have dtype %s, got %s" % (name, dtype, t.dtype))
    if not t.is_contiguous():
        raise ValueError("%s must be contiguous" % name)
    if device and not t.is_cuda:
        raise ValueError("%s must live on the GPU" % name)
    return t


def _src_ptr(src):
    """Table base: an int address (MemoryPtr-style), or a tensor (device, or pinned host)."""
    if isinstance(src, int):
        return src
    if isinstance(src, torch.Tensor):
        return src.data_ptr()
    if hasattr(src, "address"):
        return int(src.address)
    raise TypeError("unsupported table source %r" % type(src))


@functools.lru_cache(maxsize=512)
def _ws_bytes(query, *sizes):
    """Result of a *_workspace_bytes query of the library (a pure function of the sizes)."""
    return getattr(load(), query)(*[int(v) for v in sizes])


# Scratch tensors per (purpose, device, stream), grown on demand and reused: no allocation in steady
# state, and calls enqueued on different streams never share a workspace.
_ws = _hostops.Workspace()


def set_device(device_id):
    call("gear_hip_set_device", int(device_id))


def subcopy(src, dst, idxs, tss, lens, *, pad_head, ofst, span, traj_stride, step_bytes,
            col_base, zero_fill=True, mask_out=None, dst_stride=None):
    """One column of windows -> dst[num, span, ...]; see gear_hip_subcopy."""
    _need(idxs, torch.int64, "idxs")
    _need(tss, torch.int64, "tss")
    _need(lens, torch.int64, "lens")
    num = idxs.numel()
    if tss.numel() != num or lens.numel() != num:
        raise ValueError("idxs, tss and lens must have the same number of elements")
    if not dst.is_cuda or not dst.is_contiguous():
        raise ValueError("dst must be a contiguous GPU tensor")
    if dst_stride is None:
        dst_stride = span * step_bytes
    if dst.numel() * dst.element_size() < num * dst_stride:
        raise ValueError("dst is smaller than num * dst_stride bytes")
    if mask_out is not None:
        _need(mask_out, torch.uint8, "mask_out")
        if mask_out.numel() < num * span:
            raise ValueError("mask_out is smaller than num * span")
    call("gear_hip_subcopy", _src_ptr(src), _ptr(dst), num, _ptr(idxs), _ptr(tss), _ptr(lens),
         int(bool(pad_head)), int(ofst), int(span), int(traj_stride), int(step_bytes),
         int(col_base), int(dst_stride), int(bool(zero_fill)), _ptr(mask_out), _stream())
    return dst


def subcopy_multi(src, idxs, tss, lens, traj_stride, columns, capacity=0, trajectory_length=0):
    """All columns of one batch in one launch.

    columns: list of dicts with keys dst, ofst, span, step_bytes, col_base, pad_head and
    optionally zero_fill (default True), mask_out, dst_stride.
    capacity / trajectory_length > 0: the kernel checks every window against the table (an index
    outside [0, capacity) gathers nothing, lens are clamped to trajectory_length).
    """
    _need(idxs, torch.int64, "idxs")
    _need(tss, torch.int64, "tss")
    _need(lens, torch.int64, "lens")
    num = idxs.numel()
    n = len(columns)
    if n > _cabi.MAX_COLUMNS:
        raise ValueError("at most %d columns per launch" % _cabi.MAX_COLUMNS)
    descs = (ColumnDesc * max(n, 1))()
    for i, c in enumerate(columns):
        dst = c["dst"]
        stride = c.get("dst_stride", c["span"] * c["step_bytes"])
        if not dst.is_cuda or not dst.is_contiguous():
            raise ValueError("column %d: dst must be a contiguous GPU tensor" % i)
        if dst.numel() * dst.element_size() < num * stride:
            raise ValueError("column %d: dst is smaller than num * dst_stride bytes" % i)
        m = c.get("mask_out")
        if m is not None and m.numel() < num * c["span"]:
            raise ValueError("column %d: mask_out is smaller than num * span" % i)
        descs[i].dst = dst.data_ptr()
        descs[i].mask_out = m.data_ptr() if m is not None else None
        descs[i].ofst = int(c["ofst"])
        descs[i].span = int(c["span"])
        descs[i].step_bytes = int(c["step_bytes"])
        descs[i].col_base = int(c["col_base"])
        descs[i].dst_stride = int(stride)
        descs[i].pad_head = int(bool(c["pad_head"]))
        descs[i].zero_fill = int(bool(c.get("zero_fill", True)))
    call("gear_hip_subcopy_multi_checked", _src_ptr(src), num, _ptr(idxs), _ptr(tss), _ptr(lens),
         int(traj_stride), int(capacity), int(trajectory_length), descs, n, _stream())


class GatherPlan:
    """subcopy_multi for a loop that gathers into the same batch tensors every step: the column
    descriptors and every argument that does not change are marshalled once, run() is one call
    into the library with the three index tensors of the step."""

    def __init__(self, src, traj_stride, columns, num, capacity=0, trajectory_length=0):
        n = len(columns)
        if n > _cabi.MAX_COLUMNS:
            raise ValueError("at most %d columns per launch" % _cabi.MAX_COLUMNS)
        self._descs = (ColumnDesc * max(n, 1))()
        self._keep = []
        for i, c in enumerate(columns):
            dst = c["dst"]
            stride = c.get("dst_stride", c["span"] * c["step_bytes"])
            if not dst.is_cuda or not dst.is_contiguous():
                raise ValueError("column %d: dst must be a contiguous GPU tensor" % i)
            if dst.numel() * dst.element_size() < num * stride:
                raise ValueError("column %d: dst is smaller than num * dst_stride bytes" % i)
            m = c.get("mask_out")
            if m is not None and m.numel() < num * c["span"]:
                raise ValueError("column %d: mask_out is smaller than num * span" % i)
            d = self._descs[i]
            d.dst = dst.data_ptr()
            d.mask_out = m.data_ptr() if m is not None else None
            d.ofst, d.span = int(c["ofst"]), int(c["span"])
            d.step_bytes, d.col_base, d.dst_stride = int(c["step_bytes"]), int(c["col_base"]), int(stride)
            d.pad_head = int(bool(c["pad_head"]))
            d.zero_fill = int(bool(c.get("zero_fill", True)))
            self._keep.append((dst, m))
        self._keep.append(src)
        self._gather = _hostops.Gather(
            _src_ptr(src), int(traj_stride), int(num), int(capacity), int(trajectory_length),
            [(d.dst or 0, d.mask_out or 0, d.ofst, d.span, d.step_bytes, d.col_base, d.dst_stride,
              bool(d.pad_head), bool(d.zero_fill)) for d in self._descs[:n]])

    def run(self, idxs, tss, lens):
        self._gather.run(idxs, tss, lens)


def vcopy(src, dst, src_offsets, dst_offsets, strides, max_stride):
    _need(src_offsets, torch.int64, "src_offsets")
    _need(dst_offsets, torch.int64, "dst_offsets")
    _need(strides, torch.int64, "strides")
    num = min(src_offsets.numel(), dst_offsets.numel(), strides.numel())
    call("gear_hip_vcopy", _src_ptr(src), _ptr(dst), num, _ptr(src_offsets), _ptr(dst_offsets),
         _ptr(strides), int(max_stride), _stream())
    return dst


def copy(src, dst, src_offsets, dst_offsets, stride):
    _need(src_offsets, torch.int64, "src_offsets")
    _need(dst_offsets, torch.int64, "dst_offsets")
    num = min(src_offsets.numel(), dst_offsets.numel())
    call("gear_hip_copy", _src_ptr(src), _ptr(dst), num, _ptr(src_offsets), _ptr(dst_offsets),
         int(stride), _stream())
    return dst


def sub(idxs, tss, lens, *, pad_head, ofst, span, traj_stride, step_bytes, col_base,
        src_offsets=None, dst_offsets=None, copy_lens=None):
    _need(idxs, torch.int64, "idxs")
    _need(tss, torch.int64, "tss")
    _need(lens, torch.int64, "lens")
    num = idxs.numel()
    outs = []
    for t in (src_offsets, dst_offsets, copy_lens):
        outs.append(t if t is not None else torch.empty(num, dtype=torch.int64,
                                                        device=idxs.device))
    call("gear_hip_sub", num, _ptr(idxs), _ptr(tss), _ptr(lens), int(bool(pad_head)), int(ofst),
         int(span), int(traj_stride), int(step_bytes), int(col_base), _ptr(outs[0]),
         _ptr(outs[1]), _ptr(outs[2]), _stream())
    return outs[0], outs[1], outs[2], span * step_bytes


def split_step_index(flat, trajectory_length, modulo=0, idxs=None, tss=None, lens=None):
    """flat step indices -> (trajectory, timestep, length = timestep + 1) on the device."""
    _need(flat, torch.int64, "flat")
    num = flat.numel()
    outs = [t if t is not None else torch.empty(num, dtype=torch.int64, device=flat.device)
            for t in (idxs, tss, lens)]
    call("gear_hip_split_step_index", _ptr(flat), num, int(trajectory_length), int(modulo),
         _ptr(outs[0]), _ptr(outs[1]), _ptr(outs[2]), _stream())
    return outs[0], outs[1], outs[2]


def take_i64(table, idx, add=0, out=None):
    """out[j] = table[idx[j]] + add (int64, device)."""
    return _hostops.take_i64(table, idx, int(add), out)


def take_sorted_i64(table, idx):
    """sort(table[idx]) (int64, device), for entries that are mostly in order already."""
    return _hostops.take_sorted(table, idx, _ws)


def prefix_sum(priorities, out=None):
    """fp32[n] -> inclusive fp64 prefix[n] (gear_hip_scan_f32_f64)."""
    return _hostops.prefix_sum(priorities, out, _ws)


def prefix_sum_static(priorities, out):
    """fp32[n] -> fp64 prefix[n] into the caller's `out` with no allocation anywhere: the range
    sums live in the library's static device array (gear_hip_scan_f32_f64_static).  Calls that
    overlap on one GPU share that array and race."""
    _need(priorities, torch.float32, "priorities")
    _need(out, torch.float64, "out")
    n = priorities.numel()
    if out.numel() < n:
        raise ValueError("out is too small")
    call("gear_hip_scan_f32_f64_static", _ptr(priorities), _ptr(out), n, _stream())
    return out


class PrefixState:
    """The fp64 prefix of ONE priority array together with a workspace of its own, so that the
    range sums of the last scan survive other scans and a rescan can start at the first changed
    priority (gear_hip_rescan_f32_f64).  All calls must be enqueued on the same stream."""

    def __init__(self):
        self.out = None
        self._ws = None
        self._n = -1
        self._src = None
        self._valid = False

    def scan(self, priorities, first_changed=0):
        """first_changed = 0: full scan; k > 0: only priorities[k:] changed since the last call;
        k >= n: nothing changed (no launch).  Returns the fp64 prefix (the same tensor each call)."""
        _need(priorities, torch.float32, "priorities")
        n = priorities.numel()
        if self.out is None or self._n != n or self.out.device != priorities.device:
            self.out = torch.empty(n, dtype=torch.float64, device=priorities.device)
            nbytes = _ws_bytes("gear_hip_scan_workspace_bytes", n)
            self._ws = torch.empty(max(int(nbytes), 256), dtype=torch.uint8,
                                   device=priorities.device)
            self._n = n
            self._valid = False
        if self._src != priorities.data_ptr():
            self._valid = False
        _hostops.rescan(priorities, self.out, int(first_changed) if self._valid else 0, self._ws)
        self._src = priorities.data_ptr()
        self._valid = True
        return self.out


def prefix_sum_i64(weights, out=None):
    return _hostops.prefix_sum_i64(weights, out, _ws)


def sum_f32(values, out=None, out_f64=None):
    _need(values, torch.float32, "values")
    n = values.numel()
    if out is None:
        out = torch.empty(1, dtype=torch.float32, device=values.device)
    nbytes = _ws_bytes("gear_hip_sum_workspace_bytes", n)
    ws = _ws.get("sum", nbytes, values.device)
    call("gear_hip_sum_f32", _ptr(values), n, _ptr(out), _ptr(out_f64), _ptr(ws), ws.numel(),
         _stream())
    return out


def upper_bound(prefix, u, *, unit_uniforms=False, idx_out=None, priorities=None, beta=0.4,
                weights_out=None):
    """Batched search of draws in an fp64 prefix array; optionally importance weights."""
    return _hostops.upper_bound(prefix, u, bool(unit_uniforms), idx_out, priorities, float(beta),
                                weights_out, _ws)


def sample_sorted(prefix, u, *, unit_uniforms=True, sorted_out=None, trajectory_length=0,
                  modulo=0, idxs=None, tss=None, lens=None):
    """Search + ascending sort (+ split into window arguments) of one batch of draws."""
    return _hostops.sample_sorted(prefix, u, bool(unit_uniforms), sorted_out, int(trajectory_length),
                                  int(modulo), idxs, tss, lens, _ws)


def sample_lookup(prefix, u, *, unit_uniforms=True, index_table=None, index_offset=0,
                  lengths_table=None, sampled_out=None, local_out=None, lens_out=None,
                  start_uniforms=None, window=0, starts_out=None):
    """Weighted draws, sorted, with the loader's look-ups in the same call: positions of the
    draws in the prefix, ascending -> (sampled = index_table[position], local = sampled -
    index_offset, lens = lengths_table[local]).  An fp64 prefix takes float32 draws
    (gear_hip_sample_lookup_f64), an int64 prefix -- a sampler over lengths -- float64 uniforms
    or int64 targets (gear_hip_sample_lookup_i64); there, `start_uniforms` (float64 in [0, 1), one
    per draw) and `window` add a fourth result: starts = floor(start_uniforms * (lens - window + 1)),
    where a window of that many steps begins inside each drawn entry."""
    return _hostops.sample_lookup(prefix, u, bool(unit_uniforms), index_table, int(index_offset),
                                  lengths_table, sampled_out, local_out, lens_out, start_uniforms,
                                  int(window), starts_out, _ws)


def sort_lookup(positions, bound, *, index_table=None, index_offset=0, lengths_table=None,
                sampled_out=None, local_out=None, lens_out=None):
    """Given positions (each in [0, bound)): ascending sort, then the same look-ups
    (gear_hip_sort_lookup_i64)."""
    return _hostops.sort_lookup(positions, int(bound), index_table, int(index_offset), lengths_table,
                                sampled_out, local_out, lens_out, _ws)


def lookup(positions, *, index_table=None, index_offset=0, lengths_table=None, sampled_out=None,
           local_out=None, lens_out=None):
    """The look-ups alone, for positions that are already in the wanted order
    (gear_hip_lookup_i64)."""
    return _hostops.lookup(positions, index_table, int(index_offset), lengths_table, sampled_out,
                           local_out, lens_out)


def upper_bound_i64(prefix, u, *, unit_uniforms=True, idx_out=None):
    return _hostops.upper_bound_i64(prefix, u, bool(unit_uniforms), idx_out)


def sort_i64(keys, vals=None, key_bits=63):
    return _hostops.sort_i64(keys, vals, int(key_bits), _ws)


def topk(priorities, k, *, sorted_by_value=True, want_values=True, warm=False, workspace=None):
    """Top-k of fp32 priorities (values, indices), by value descending or by index ascending.
    warm=True: the call may start from the bound that the last call on `workspace` (same n, k and
    order) left there instead of sampling the array; the result is the same either way."""
    return _hostops.topk(priorities, k, bool(sorted_by_value), bool(want_values), bool(warm),
                         workspace, _ws)


class TopKState:
    """A top-k selection that is repeated on one slowly changing priority array (the priority
    maintenance of a replay buffer): owns the workspace, so that every call after the first can
    take up the bound the call before it left (gear_hip_topk_f32_warm)."""

    def __init__(self):
        self._ws = None
        self._shape = None

    def select(self, priorities, k, *, sorted_by_value=True, want_values=True):
        n = priorities.numel()
        shape = (n, int(k), bool(sorted_by_value), priorities.device)
        nbytes = _ws_bytes("gear_hip_topk_workspace_bytes", n, k)
        warm = self._shape == shape
        if self._ws is None or self._ws.numel() < nbytes or self._ws.device != priorities.device:
            self._ws = torch.empty(max(int(nbytes), 256), dtype=torch.uint8,
                                   device=priorities.device)
            warm = False
        self._shape = shape
        return topk(priorities, k, sorted_by_value=sorted_by_value, want_values=want_values,
                    warm=warm, workspace=self._ws)


def scatter(weights, idx, values, *, unique_indices=False):
    """weights[idx[j]] = values[j]; duplicates: last one wins.  fp32 or int64 tables."""
    return _hostops.scatter(weights, idx, values, bool(unique_indices), _ws)
