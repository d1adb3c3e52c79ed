"""What a loader's step promises around its batch: when it is complete, what a failure leaves behind,
what another thread may do meanwhile."""
import ctypes
import os

import numpy as np
import pytest

from conftest import announce

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

T, CAP, WIDTH = 64, 64, 8192


def _loader(placement, key, batch=CAP, method="Uniform", **kw):
    """One fp32 column of WIDTH values a step, each trajectory filled with its number + 1."""
    from gear_amd.dataset import SharedDataset
    from gear_amd.loader import OfflineLoader
    from gear_amd.mpu import ModelParallelismUnit
    from gear_amd.specs import TableSpec
    spec = TableSpec.create(trajectory_length=T, capacity=CAP, column_specs=[
        dict(shape=[WIDTH], dtype=torch.float32, name="x")])
    data = SharedDataset.create(spec, key=(os.getpid() << 8) + key, placement=placement)
    for i in range(CAP):
        data[i] = (1.0, 1 + i % T, [torch.full((T, WIDTH), float(i + 1))])
    patterns = [dict(name="x", offset=-T, length=T, pad="tail")]
    return OfflineLoader(data, batch, ModelParallelismUnit(device=torch.device("cuda:0")), method,
                         patterns, **kw)


def _check(loader, timesteps, batch):
    at = loader.last_sampled.cpu()
    assert torch.equal(timesteps.cpu(), 1 + at % T)
    got = batch[0].cpu()
    for j, (i, n) in enumerate(zip(at.tolist(), timesteps.tolist())):
        assert bool((got[j, :n] == float(i + 1)).all()) and not bool(got[j, n:].any())


def test_a_host_table_may_be_written_after_the_step():
    """The gather reads the table in host memory: it has ended when next() returns the timesteps on the
    host, so that what is written then does not reach the batch."""
    loader = _loader("pinned", 1)
    address, nbytes = int(loader._table.get_address().address), 4 * WIDTH * T * CAP
    saved = ctypes.string_at(address, nbytes)
    announce("host table written after next()")
    for _ in range(3):
        timesteps, batch = next(loader)
        ctypes.memset(address, 0x41, nbytes)
        _check(loader, timesteps, batch)
        ctypes.memmove(address, saved, nbytes)


def test_the_batch_may_be_read_on_another_stream():
    loader = _loader("device", 2)
    side = torch.cuda.Stream()
    announce("batch read on another stream")
    for _ in range(5):
        torch.cuda.synchronize()
        timesteps, batch = next(loader)
        with torch.cuda.stream(side):
            early = batch[0].clone()
        torch.cuda.synchronize()
        assert torch.equal(early, batch[0])
        _check(loader, timesteps, batch)


def test_a_step_that_runs_out_of_memory_leaves_nothing_behind():
    """The batch does not fit: the step raises, nothing on the GPU still writes the pinned memory the
    lengths would have gone through, and the loader goes on."""
    loader = _loader("device", 3, batch=16384)      # a batch of 32 GiB
    small = _loader("device", 4, batch=1024)
    timesteps, batch = next(small)                  # (what the step keeps is in the caches)
    del batch
    torch.cuda.empty_cache()
    announce("out of memory in a loader's step")
    torch.cuda.set_per_process_memory_fraction(0.05)
    try:
        for _ in range(2):
            torch.cuda._sleep(50_000_000)           # what the step enqueues runs late
            with pytest.raises(RuntimeError, match="out of memory"):
                next(loader)
            pinned = [torch.full((n,), -7, dtype=torch.int64).pin_memory() for n in (16384, 16384, 16000)]
            torch.cuda.synchronize()
            assert all(bool((p == -7).all()) for p in pinned)
            del pinned
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    timesteps, batch = next(small)
    at = small.last_sampled.cpu()
    assert torch.equal(timesteps, 1 + at % T) and torch.equal(batch[0][:, 0, 0].cpu(), at + 1.0)


def test_two_threads_in_one_loader():
    """A thread that comes in while another waits for its lengths has memory of its own for them."""
    import threading
    loader = _loader("device", 5, batch=32)
    next(loader)
    step, errors = loader._step, []
    tables = [torch.randint(1, T + 1, (CAP,), device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    announce("two threads in one loader's step")

    def work(lengths):
        try:
            host = lengths.cpu()
            with torch.cuda.stream(torch.cuda.Stream()):
                draws = torch.randint(0, CAP, (32,), device="cuda")
                for _ in range(200):
                    sampled, ts, _, _ = step.run("uniform", draws, None, loader._indices, 0, lengths, True,
                                                 _ops()._ws)
                    if not torch.equal(ts, host[sampled.cpu()]):
                        errors.append("lengths of another thread's step")
                        return
        except Exception as e:  # noqa: BLE001 (reported by the test's own thread)
            errors.append(repr(e))

    threads = [threading.Thread(target=work, args=(t,)) for t in tables]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors


@pytest.mark.parametrize("method", ["Uniform", "Weighted", "TopK"])
@pytest.mark.parametrize("placement", ["pinned", "device"])
def test_the_handlers_step_is_the_loaders(method, placement):
    """CpuTrajectoryStorageHandler.select_subcopy into a caller's tensors gives what the loader's step
    gives in fresh ones."""
    loader = _loader(placement, {"Uniform": 10, "Weighted": 11, "TopK": 12}[method] + 3 * (placement == "device"),
                     batch=24, method=method, with_mask=True)
    loader._device_weights.copy_(torch.rand(CAP, device="cuda") + 0.1)
    announce("handler.select_subcopy %s %s" % (method, placement))
    kind, picks, prefix = loader._sampler.prepare(
        loader._indices, loader._device_weights, loader._sampler.draw(CAP, 24), dirty_from=None)
    want = loader._step.run(kind, picks, prefix, loader._indices, loader._iset.index_offset,
                            loader._device_timesteps, False, _ops()._ws)
    dst = torch.full((24, T, WIDTH), -1.0, device="cuda")
    mask = torch.full((24, T), 9, dtype=torch.uint8, device="cuda")
    looked = torch.full((3, 24), -1, dtype=torch.int64, device="cuda")
    loader._handler.select_subcopy(kind, picks, prefix, loader._indices, loader._iset.index_offset,
                                   loader._device_timesteps, loader._sub_cols, [dst], True, [mask],
                                   looked[0], looked[1], looked[2])
    assert torch.equal(looked[0], want[0]) and torch.equal(looked[2], want[1])
    assert torch.equal(looked[1], want[0] - loader._iset.index_offset)
    assert torch.equal(dst, want[2][0]) and torch.equal(mask, want[3][0])
    _check(type("L", (), {"last_sampled": want[0]}), want[1], want[2])


def test_more_columns_than_one_launch_gathers():
    """A loader of 17 columns can be made; the fused step refuses it, the step column by column does not."""
    from gear_amd.dataset import SharedDataset
    from gear_amd.loader import OfflineLoader
    from gear_amd.mpu import ModelParallelismUnit
    from gear_amd.specs import TableSpec
    names = ["c%02d" % c for c in range(17)]
    spec = TableSpec.create(trajectory_length=4, capacity=6, column_specs=[
        dict(shape=[c + 1], dtype=torch.float32, name=n) for c, n in enumerate(names)])
    data = SharedDataset.create(spec, key=(os.getpid() << 8) + 6, placement="pinned")
    for i in range(6):
        data[i] = (1.0, 4, [torch.full((4, c + 1), 10.0 * i + c) for c in range(17)])
    loader = OfflineLoader(data, 3, ModelParallelismUnit(device=torch.device("cuda:0")), "Uniform",
                           [dict(name=n, offset=-4, length=4, pad="tail") for n in names])
    announce("a loader of 17 columns")
    with pytest.raises(RuntimeError, match="more than 16 columns"):
        next(loader)
    _, batch = loader.exposed_low_level_controlled_iterate(torch.tensor([4, 0, 5]))
    for c in range(17):
        for j, i in enumerate([4, 0, 5]):
            assert bool((batch[c][j].cpu() == 10.0 * i + c).all())
    timesteps, batch = loader.low_level_controlled_iterate()
    assert timesteps.tolist() == [4, 4, 4] and len(batch) == 17


def _ops():
    from gear_amd import ops
    return ops
