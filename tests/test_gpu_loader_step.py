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
