"""Performance cases of the replay-sampling path, each called as a training program calls it.

A case names its `kind` (which public entry points a pass goes through) and its sizes:

  loader     next(OfflineLoader): draw, look-ups and the gather of all columns; with `update` the
             priorities of the sampled batch are written back after the step (prioritized replay)
  sampler    WeightedSampler / UniformSampler.sync_sample: a sorted batch of indices, no gather
  draws      prefix sum of fp32 priorities, unsorted draws and their importance weights
  lengths    int64 prefix over trajectory lengths, draws, window starts, gather with a mask
  steps      per-step priorities: prefix sum, sorted draws split into windows, gather
  maintain   new priorities scattered, top-k of them, prefix sum, sorted draws
  topk       one selection out of an array that was not selected from before
  scan       one prefix sum

Inputs follow the benchmark configurations: priorities are lognormal(0, 1) ** 0.6, float columns
N(0, 1), images uniform bytes, trajectory lengths uniform.
"""
import itertools
import math
import os

import torch

from gear_amd import _cabi, ops
from gear_amd.dataset import SharedDataset
from gear_amd.loader import OfflineLoader
from gear_amd.mpu import ModelParallelismUnit
from gear_amd.sampler import UniformSampler, WeightedSampler
from gear_amd.specs import TableSpec

SCHEMAS = {
    "locomotion": [("obs", (17,), torch.float32), ("action", (6,), torch.float32),
                   ("reward", (), torch.float32), ("done", (), torch.uint8)],
    "returns": [("obs", (17,), torch.float32), ("action", (6,), torch.float32),
                ("reward", (), torch.float32), ("rtg", (), torch.float32),
                ("timestep", (), torch.int32)],
    "frames": [("obs", (4, 84, 84), torch.uint8), ("action", (), torch.int32),
               ("reward", (), torch.float32), ("done", (), torch.uint8)],
}
_keys = itertools.count(1)


def listed():
    return [
        # a batch of whole short trajectories, the smallest call: launches and host work
        dict(name="loader_uniform", kind="loader", method="Uniform", schema="locomotion", cap=4096,
             T=64, shortest=64, span=64, batch=256, pad="tail", mask=False, update=False,
             on_device=True, placement="device"),
        # sequence-model windows with masks out of long trajectories of unequal length, the
        # timesteps handed to the host as the loader does by default
        dict(name="loader_weighted", kind="loader", method="Weighted", schema="returns", cap=100000,
             T=1000, shortest=200, span=20, batch=1024, pad="head", mask=True, update=False,
             on_device=False, placement="device"),
        # prioritized replay: draw, gather, write the batch's new priorities back
        dict(name="loader_update", kind="loader", method="Weighted", schema="locomotion", cap=1000000,
             T=16, shortest=4, span=8, batch=512, pad="tail", mask=False, update=True,
             on_device=True, placement="device"),
        # the highest-priority trajectories of a shard
        dict(name="loader_topk", kind="loader", method="TopK", schema="locomotion", cap=300007,
             T=40, shortest=8, span=20, batch=1000, pad="head", mask=False, update=False,
             on_device=True, placement="device"),
        # a table in pinned host memory (the loader's default placement) read in place
        dict(name="loader_host_table", kind="loader", method="Weighted", schema="frames", cap=24,
             T=500, shortest=100, span=30, batch=64, pad="head", mask=False, update=False,
             on_device=True, placement="pinned"),
        # indices of a large batch, sorted, without a gather
        dict(name="sampler_sync", kind="sampler", method="Weighted", n=1000003, batch=20000),
        # prioritized sampling with importance weights
        dict(name="draws", kind="draws", n=1000000, batch=4096),
        # length-weighted windows with an attention mask
        dict(name="lengths", kind="lengths", cap=100000, T=1000, shortest=200, span=20, batch=1024),
        # frame windows drawn by per-step priorities: the largest gather
        dict(name="steps_frames", kind="steps", schema="frames", cap=1000, T=1000, span=30,
             batch=2048),
        # priority maintenance of a large replay buffer
        dict(name="maintain", kind="maintain", n=10000000, changed=65536, k=65536, batch=2048,
             unique=False),
        # a first selection, largest first
        dict(name="topk", kind="topk", n=3000001, k=20000, by_value=True),
        # a prefix sum whose arrays leave the caches
        dict(name="scan", kind="scan", n=100000000, dtype="float32"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["loader"] * 4 + ["sampler", "draws", "lengths", "steps", "maintain", "topk",
                                        "scan"])
    if kind == "loader":
        schema = rng.choice(["locomotion", "returns", "frames"])
        placement = "pinned" if rng.random() < 0.2 else "device"
        most = (400 << 20) if placement == "pinned" else (10 << 30)
        T = _log_int(rng, 16, 1000)
        fit = max(2, most // (T * sum(_step_bytes(schema))))
        cap = _log_int(rng, min(64, fit), min(1000000, fit))
        span = _log_int(rng, 1, min(T, 100))
        most = (60 << 20) if placement == "pinned" else (1 << 30)
        fit = max(8, min(4096, most // (span * sum(_step_bytes(schema)))))
        method = rng.choice(["Uniform", "Weighted", "Weighted", "TopK"])
        batch = _log_int(rng, 8, fit)
        return dict(kind=kind, method=method, schema=schema, cap=cap, T=T,
                    shortest=rng.choice([T, max(1, T // 5)]), span=span,
                    batch=min(batch, cap) if method == "TopK" else batch,
                    pad=rng.choice(["head", "tail"]), mask=rng.random() < 0.3,
                    update=method == "Weighted" and rng.random() < 0.5,
                    on_device=rng.random() < 0.7, placement=placement)
    if kind == "sampler":
        return dict(kind=kind, method=rng.choice(["Weighted", "Uniform"]),
                    n=_log_int(rng, 1000, 10000000), batch=_log_int(rng, 32, 100000))
    if kind == "draws":
        return dict(kind=kind, n=_log_int(rng, 1000, 10000000), batch=_log_int(rng, 32, 100000))
    if kind == "lengths":
        T = _log_int(rng, 50, 1000)
        return dict(kind=kind, cap=_log_int(rng, 100, 100000), T=T, shortest=max(1, T // 5),
                    span=_log_int(rng, 1, max(1, T // 5)), batch=_log_int(rng, 32, 8192))
    if kind == "steps":
        schema = rng.choice(["locomotion", "returns", "frames"])
        T = _log_int(rng, 50, 1000)
        fit = max(2, (10 << 30) // (T * sum(_step_bytes(schema))))
        span = _log_int(rng, 1, min(T, 64))
        fit_batch = max(16, min(8192, (1 << 30) // (span * sum(_step_bytes(schema)))))
        return dict(kind=kind, schema=schema, cap=_log_int(rng, 2, min(20000, fit)), T=T, span=span,
                    batch=_log_int(rng, 16, fit_batch))
    if kind == "maintain":
        n = _log_int(rng, 10000, 20000000)
        return dict(kind=kind, n=n, changed=_log_int(rng, 64, min(n // 8, 131072)),
                    k=_log_int(rng, 64, min(n // 8, 131072)), batch=_log_int(rng, 64, 8192),
                    unique=rng.random() < 0.4)
    if kind == "topk":
        n = _log_int(rng, 10000, 60000000)
        return dict(kind=kind, n=n, k=_log_int(rng, 16, min(n // 4, 200000)),
                    by_value=rng.random() < 0.6)
    return dict(kind="scan", n=_log_int(rng, 1000, 130000000),
                dtype=rng.choice(["float32", "float32", "int64"]))


def _step_bytes(schema):
    return [torch.empty(0, dtype=dt).element_size() * math.prod(shape)
            for _, shape, dt in SCHEMAS[schema]]


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _priorities(n, g):
    return torch.randn(n, device="cuda", generator=g).mul_(0.6).exp_()


def _lengths(case, g):
    return torch.randint(case["shortest"], case["T"] + 1, (case["cap"],), device="cuda", generator=g)


def _column(dtype, steps, width, g):
    if dtype is torch.float32:
        return torch.randn(steps, width, device="cuda", generator=g)
    if dtype is torch.int32:
        return torch.randint(0, 1000, (steps, width), dtype=dtype, device="cuda", generator=g)
    if width == 1:  # the done flag
        return (torch.rand(steps, 1, device="cuda", generator=g) < 0.001).to(torch.uint8)
    words = torch.empty(steps, width // 8, dtype=torch.int64, device="cuda")
    return words.random_(generator=g).view(torch.uint8)


def _fill(schema, T, cap, g, put):
    """Trajectory bytes in the table's layout ([T] steps of one column after the other), handed
    to put(byte offset, bytes) a few trajectories at a time."""
    stride = T * sum(_step_bytes(schema))
    many = max(1, min(cap, (512 << 20) // stride))
    block = torch.empty(many, stride, dtype=torch.uint8, device="cuda")
    for first in range(0, cap, many):
        rows, at = min(many, cap - first), 0
        for (_, shape, dtype), size in zip(SCHEMAS[schema], _step_bytes(schema)):
            col = _column(dtype, rows * T, math.prod(shape), g)
            block[:rows, at:at + T * size] = col.view(torch.uint8).view(rows, T * size)
            at += T * size
        put(first * stride, block[:rows])


def _plain_table(schema, T, cap, g):
    """A table in HBM and what a gather plan has to know of it."""
    sizes = _step_bytes(schema)
    table = torch.empty(cap * T * sum(sizes), dtype=torch.uint8, device="cuda")

    def put(at, rows):
        table[at:at + rows.numel()] = rows.view(-1)

    _fill(schema, T, cap, g, put)
    bases = [T * sum(sizes[:c]) for c in range(len(sizes))]
    return table, T * sum(sizes), sizes, bases


def _dataset(case, g):
    spec = TableSpec.create(trajectory_length=case["T"], capacity=case["cap"], column_specs=[
        dict(shape=list(shape), dtype=dtype, name=name)
        for name, shape, dtype in SCHEMAS[case["schema"]]])
    data = SharedDataset.create(spec, key=(os.getpid() << 20) + next(_keys),
                                placement=case["placement"])
    base = data._table.device_address

    def put(at, rows):
        torch.cuda.synchronize()
        _cabi.call("gear_hip_memcpy", base + at, rows.data_ptr(), rows.numel())

    _fill(case["schema"], case["T"], case["cap"], g, put)
    data.weights[:] = _priorities(case["cap"], g).cpu()
    data.timesteps[:] = _lengths(case, g).cpu()
    return data


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    state = {"case": case}
    if kind == "loader":
        patterns = [dict(name=name, offset=-case["span"], length=case["span"], pad=case["pad"])
                    for name, _, _ in SCHEMAS[case["schema"]]]
        state["loader"] = OfflineLoader(
            _dataset(case, g), case["batch"], ModelParallelismUnit(), case["method"], patterns,
            timesteps_on_device=case["on_device"], with_mask=case["mask"])
        # what the training step would return for the batch
        state["errors"] = _priorities(case["batch"], g)
    elif kind == "sampler":
        cls = {"Weighted": WeightedSampler, "Uniform": UniformSampler}[case["method"]]
        state["sampler"] = cls(ModelParallelismUnit(), seed=seed & 0x7fffffff)
        state["indices"] = torch.arange(case["n"], device="cuda") + 3 * case["n"]
        state["weights"] = _priorities(case["n"], g)
    elif kind == "draws":
        state["weights"] = _priorities(case["n"], g)
        state["u"] = torch.rand(case["batch"], device="cuda", generator=g)
    elif kind == "lengths":
        schema, span, batch = "returns", case["span"], case["batch"]
        table, stride, sizes, bases = _plain_table(schema, case["T"], case["cap"], g)
        state["lengths"] = _lengths(case, g)
        state["u"], state["v"] = torch.rand(2, batch, dtype=torch.float64, device="cuda", generator=g)
        state["mask"] = torch.empty(batch, span, dtype=torch.uint8, device="cuda")
        state["dsts"] = [torch.empty(batch, span * s, dtype=torch.uint8, device="cuda")
                         for s in sizes]
        state["plan"] = ops.GatherPlan(table, stride, [
            dict(dst=state["dsts"][c], ofst=0, span=span, step_bytes=sizes[c], col_base=bases[c],
                 pad_head=False, mask_out=state["mask"] if c == 0 else None)
            for c in range(len(sizes))], batch)
    elif kind == "steps":
        T, cap, span, batch = case["T"], case["cap"], case["span"], case["batch"]
        table, stride, sizes, bases = _plain_table(case["schema"], T, cap, g)
        state["weights"] = _priorities(T * cap, g)
        state["u"] = torch.rand(batch, device="cuda", generator=g)
        state["dsts"] = [torch.empty(batch, span * s, dtype=torch.uint8, device="cuda")
                         for s in sizes]
        state["plan"] = ops.GatherPlan(table, stride, [
            dict(dst=state["dsts"][c], ofst=1 - span, span=span, step_bytes=sizes[c],
                 col_base=bases[c], pad_head=True) for c in range(len(sizes))], batch)
    elif kind == "maintain":
        n, changed = case["n"], case["changed"]
        state["weights"] = _priorities(n, g)
        # four rounds of updates, taken in turn
        state["updates"] = []
        for _ in range(4):
            if case["unique"]:
                at = torch.randperm(n, device="cuda", generator=g)[:changed].contiguous()
            else:
                at = torch.randint(0, n, (changed,), device="cuda", generator=g)
            state["updates"].append((at, _priorities(changed, g)))
        state["round"] = 0
        state["top"] = ops.TopKState()
        state["prefix"] = ops.PrefixState()
        state["u"] = torch.rand(case["batch"], device="cuda", generator=g)
    elif kind == "topk":
        state["weights"] = _priorities(case["n"], g)
    elif case["dtype"] == "float32":
        state["weights"] = _priorities(case["n"], g)
    else:
        state["weights"] = torch.randint(200, 1001, (case["n"],), device="cuda", generator=g)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "loader":
        loader = state["loader"]
        timesteps, batch = next(loader)
        out = {"timesteps": timesteps, "batch": batch, "sampled": loader.last_sampled}
        if case["mask"]:
            out["masks"] = loader.last_masks
        if case["update"]:
            loader.update_priorities(loader.last_sampled, state["errors"])
        return out
    if kind == "sampler":
        return state["sampler"].sync_sample(state["indices"], state["weights"], case["batch"])
    if kind == "draws":
        prefix = ops.prefix_sum(state["weights"])
        index, importance = ops.upper_bound(prefix, state["u"], unit_uniforms=True,
                                            priorities=state["weights"], beta=0.4)
        return {"prefix": prefix, "index": index, "importance": importance}
    if kind == "lengths":
        prefix = ops.prefix_sum_i64(state["lengths"])
        sampled, local, lens, starts = ops.sample_lookup(
            prefix, state["u"], lengths_table=state["lengths"], start_uniforms=state["v"],
            window=case["span"])
        state["plan"].run(local, starts, lens)
        return {"prefix": prefix, "sampled": sampled, "lens": lens, "starts": starts,
                "batch": state["dsts"], "mask": state["mask"]}
    if kind == "steps":
        prefix = ops.prefix_sum(state["weights"])
        flat, idxs, tss, lens = ops.sample_sorted(prefix, state["u"], unit_uniforms=True,
                                                  trajectory_length=case["T"])
        state["plan"].run(idxs, tss, lens)
        return {"prefix": prefix, "flat": flat, "idxs": idxs, "tss": tss, "lens": lens,
                "batch": state["dsts"]}
    if kind == "maintain":
        at, values = state["updates"][state["round"] % 4]
        state["round"] += 1
        weights = ops.scatter(state["weights"], at, values, unique_indices=case["unique"])
        top, index = state["top"].select(weights, case["k"], sorted_by_value=True)
        prefix = state["prefix"].scan(weights)
        drawn = ops.sample_sorted(prefix, state["u"], unit_uniforms=True)
        return {"weights": weights, "top": top, "index": index, "prefix": prefix, "drawn": drawn}
    if kind == "topk":
        top, index = ops.topk(state["weights"], case["k"], sorted_by_value=case["by_value"])
        return {"top": top, "index": index}
    if case["dtype"] == "float32":
        return ops.prefix_sum(state["weights"])
    return ops.prefix_sum_i64(state["weights"])


def work(case):
    kind = case["kind"]
    if kind == "loader":
        row = sum(_step_bytes(case["schema"]))
        lo, hi, span, batch = case["shortest"], case["T"], case["span"], case["batch"]
        kept = sum(min(v, span) for v in range(lo, hi + 1)) / (hi - lo + 1)
        bytes_ = batch * row * (span + kept) + 24 * batch
        if case["mask"]:
            bytes_ += batch * span * len(SCHEMAS[case["schema"]])
        # priorities are read where they may have changed since the last batch
        if case["method"] == "TopK" or case["update"]:
            bytes_ += 4 * case["cap"]
        return {"bytes": bytes_, "flops": 0}
    batch = case.get("batch", 0)
    if kind == "sampler":
        return {"bytes": 16 * batch + (4 * case["n"] if case["method"] == "Weighted" else 0),
                "flops": 0}
    if kind == "draws":
        return {"bytes": 12 * case["n"] + 20 * batch, "flops": 0}
    if kind == "lengths":
        return {"bytes": 16 * case["cap"] + batch * case["span"] * (
            2 * sum(_step_bytes("returns")) + 1) + 48 * batch, "flops": 0}
    if kind == "steps":
        T, span = case["T"], case["span"]
        kept = sum(min(t + 1, span) for t in range(T)) / T
        return {"bytes": 12 * T * case["cap"] + 36 * batch +
                batch * sum(_step_bytes(case["schema"])) * (span + kept), "flops": 0}
    if kind == "maintain":
        return {"bytes": 12 * case["n"] + 16 * case["changed"] + 12 * case["k"] + 12 * batch,
                "flops": 0}
    if kind == "topk":
        return {"bytes": 4 * case["n"] + 12 * case["k"], "flops": 0}
    return {"bytes": (12 if case["dtype"] == "float32" else 16) * case["n"], "flops": 0}


def tolerance(case):
    # Indices, lengths, masks, gathered bytes and selected priorities are copies and counts: exact.
    # fp64 sums of 1e8 such priorities in another order differ by 1.1e-16 (2-norm) and 8.6e-16 (the
    # largest); importance weights, rounded to fp32 once, are within 2.5e-8 and 5.9e-8 of the same
    # in fp64.  Four times that.
    if case["kind"] in ("steps", "maintain") or (case["kind"] == "scan" and
                                                 case["dtype"] == "float32"):
        return {"rel": 5e-16, "max": 4e-15}
    if case["kind"] == "draws":
        return {"rel": 1e-7, "max": 2.4e-7}
    return "exact"
