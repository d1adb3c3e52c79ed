"""A loader's step that draws its batch itself gives what torch's rand or randint of the same generator would have
given it, and leaves the generator where that call leaves it: at the sizes where the draws move from the
selection to a launch of their own and from there to torch, and for ranges of one entry to just beyond 2^28, from
where torch draws."""
import os

import pytest

from conftest import announce

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _ops():
    from gear_amd import ops
    return ops


def _loader(key, batch, method="Uniform", **kw):
    """One value a step, windows of one step."""
    from gear_amd.dataset import SharedDataset
    from gear_amd.loader import OfflineLoader
    from gear_amd.mpu import ModelParallelismUnit
    from gear_amd.specs import TableSpec
    spec = TableSpec.create(trajectory_length=4, capacity=64, column_specs=[
        dict(shape=[1], dtype=torch.float32, name="x")])
    data = SharedDataset.create(spec, key=(os.getpid() << 8) + key, placement="device")
    data.weights[:] = torch.rand(64) + 0.1
    data.timesteps[:] = torch.randint(1, 5, (64,))
    return OfflineLoader(data, batch, ModelParallelismUnit(device=torch.device("cuda:0")), method,
                         [dict(name="x", offset=-1, length=1, pad="tail")], **kw)


def _tables(n):
    table = torch.arange(n, device="cuda") + 5
    lengths = torch.zeros(n + 5, dtype=torch.int64, device="cuda")
    return table, lengths


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("num", [1, 2, 255, 257, 1024, 1025, 4096, 4097, 20_000, 33_000])
def test_draws(weighted, num):
    step = _loader(40, batch=8)._step
    g = torch.Generator("cuda")
    for seed, skip, n in ((1, 0, 1), (42, 3, 64), ((1 << 40) + 7, 1 << 33, 100_003)):
        g.manual_seed(seed)
        if skip:
            g.set_offset(4 * skip)
        table, lengths = _tables(n)
        prefix = _ops().prefix_sum(torch.rand(n, device="cuda") + 0.01) if weighted else None
        state = g.get_state()
        announce("draws num=%d n=%d weighted=%d" % (num, n, weighted))
        kind = "weighted" if weighted else "uniform"
        got = step.run(kind, g, prefix, table, 5, lengths, False, _ops()._ws, num)
        offset = g.get_offset()
        g.set_state(state)
        draws = torch.rand(num, generator=g, device="cuda") if weighted else \
            torch.randint(0, n, (num,), generator=g, device="cuda")
        assert g.get_offset() == offset
        want = step.run(kind, draws, prefix, table, 5, lengths, False, _ops()._ws)
        assert torch.equal(got[0], want[0])
        if not weighted:
            assert torch.equal(got[0], draws.sort().values + 5)


@pytest.mark.parametrize("n", [(1 << 28) - 1, 1 << 28, (1 << 28) + 1])
def test_ranges_beyond_one_word_a_draw(n):
    """From 2^28 on torch's randint takes two words a draw."""
    step = _loader(46, batch=8)._step
    g = torch.Generator("cuda")
    table, lengths = torch.arange(n, device="cuda") + 5, torch.zeros(1, dtype=torch.int64, device="cuda")
    for num in (48, 5000):
        g.manual_seed(num)
        announce("draws num=%d n=%d" % (num, n))
        got = step.run("uniform", g, None, table, 5, lengths, False, _ops()._ws, num)
        offset = g.get_offset()
        g.manual_seed(num)
        want = torch.randint(0, n, (num,), generator=g, device="cuda")
        assert torch.equal(got[0], want.sort().values + 5)
        assert g.get_offset() == offset


@pytest.mark.parametrize("weighted", [False, True])
def test_more_draws_than_the_gpu_holds_threads(weighted):
    from gear_amd import _cabi
    props = torch.cuda.get_device_properties(0)
    most = _cabi.load().gear_hip_draw_max()
    assert most == props.multi_processor_count * (props.max_threads_per_multi_processor // 256) * 256
    step = _loader(48 + weighted, batch=8)._step
    g = torch.Generator("cuda")
    table, lengths = _tables(1000)
    prefix = _ops().prefix_sum(torch.rand(1000, device="cuda") + 0.01) if weighted else None
    kind = "weighted" if weighted else "uniform"
    for num in (most, most + 1):
        g.manual_seed(num)
        announce("%s draws num=%d" % (kind, num))
        got = step.run(kind, g, prefix, table, 5, lengths, False, _ops()._ws, num)
        offset = g.get_offset()
        g.manual_seed(num)
        draws = torch.rand(num, generator=g, device="cuda") if weighted else \
            torch.randint(0, 1000, (num,), generator=g, device="cuda")
        assert g.get_offset() == offset
        want = step.run(kind, draws, prefix, table, 5, lengths, False, _ops()._ws)
        assert torch.equal(got[0], want[0])


def test_uniforms_bit_for_bit():
    """The draws themselves: searched in a prefix whose entries are the draws of a call."""
    step = _loader(41, batch=8)._step
    g = torch.Generator("cuda")
    g.manual_seed(3)
    state = g.get_state()
    u = torch.rand(524_288, generator=g, device="cuda")
    prefix = torch.cat([u.double().unique(), torch.ones(1, dtype=torch.float64, device="cuda")])
    table, lengths = _tables(prefix.numel())
    announce("524288 uniforms")
    for num in (1000, 524_288):
        g.set_state(state)
        u = torch.rand(num, generator=g, device="cuda")
        g.set_state(state)
        got = step.run("weighted", g, prefix, table, 5, lengths, False, _ops()._ws, num)[0] - 5
        assert torch.equal(got, torch.searchsorted(prefix, u.double(), right=True).sort().values)


@pytest.mark.parametrize("weighted", [False, True])
def test_a_captured_step_draws_with_torch(weighted):
    """The generator's state is not the host's to read then: every replay has the next numbers of it."""
    ops, num, n = _ops(), 300, 10_000
    step = _loader(50 + weighted, batch=8)._step
    table, lengths = _tables(n)
    prefix = ops.prefix_sum(torch.rand(n, device="cuda") + 0.01) if weighted else None
    kind = "weighted" if weighted else "uniform"
    g, twin = torch.Generator("cuda"), torch.Generator("cuda")
    g.manual_seed(9)
    twin.manual_seed(9)
    announce("%s step captured" % kind)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):  # (what is allocated by the first call is allocated)
        step.run(kind, twin, prefix, table, 5, lengths, False, ops._ws, num)
    stream.synchronize()
    twin.manual_seed(9)
    graph = torch.cuda.CUDAGraph()
    graph.register_generator_state(g)
    with torch.cuda.graph(graph, stream=stream):
        got = step.run(kind, g, prefix, table, 5, lengths, False, ops._ws, num)[0]
    for _ in range(4):
        graph.replay()
        torch.cuda.synchronize()
        want = step.run(kind, twin, prefix, table, 5, lengths, False, ops._ws, num)[0]
        assert torch.equal(got, want)


def test_a_sampler_with_a_draw_of_its_own():
    loader = _loader(42, batch=16)
    mine = torch.arange(16, device="cuda")
    announce("a sampler whose draw() was replaced")
    loader._sampler.draw = lambda n, batch: mine.clone()
    next(loader)
    assert torch.equal(loader.last_sampled, mine + loader._iset.index_offset)


@pytest.mark.parametrize("method", ["Uniform", "Weighted"])
def test_a_loaders_batches_are_those_of_its_generator(method):
    loader = _loader(43 + (method == "Weighted"), batch=48, method=method, timesteps_on_device=True)
    g = torch.Generator("cuda")
    g.manual_seed(42)
    announce("batches of a %s loader" % method)
    for _ in range(3):
        next(loader)
        n = loader._indices.numel()
        if method == "Uniform":
            want = torch.randint(0, n, (48,), generator=g, device="cuda").sort().values
        else:
            prefix = _ops().prefix_sum(loader._device_weights)
            want = _ops().sample_sorted(prefix, torch.rand(48, generator=g, device="cuda"))
        assert torch.equal(loader.last_sampled, want + loader._iset.index_offset)
