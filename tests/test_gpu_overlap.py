"""Outputs that lie on top of the inputs of the same call: what has to be read is read before it is
written over, at the batch sizes of every form of the calls (one launch or several)."""
import numpy as np
import pytest

from conftest import announce

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

SIZES = [1, 16, 17, 500, 4096, 4097, 20_000, 32_768, 32_769]


@pytest.mark.parametrize("num", SIZES)
def test_batch_outputs_on_top_of_integer_draws_or_prefix(num):
    from gear_amd import ops
    rng = np.random.default_rng(num)
    n = 40_009
    lengths = rng.integers(1, 30, size=n)
    prefix = np.cumsum(lengths)
    t = rng.integers(0, prefix[-1], size=num)
    at = np.sort(np.searchsorted(prefix, t, side="right"))
    lens_dev, pre_dev = torch.from_numpy(lengths).cuda(), torch.from_numpy(prefix).cuda()
    v = rng.random(num)
    starts = np.where(lengths[at] >= 3, np.floor(v * (lengths[at] - 2.0)), 0).astype(np.int64)
    for name in ("sampled_out", "local_out", "lens_out", "starts_out"):
        announce("integer draws num=%d %s on the draws" % (num, name))
        u = torch.from_numpy(t).cuda()
        got = ops.sample_lookup(pre_dev, u, unit_uniforms=False, lengths_table=lens_dev,
                                start_uniforms=torch.from_numpy(v).cuda(), window=3, **{name: u})
        for g, want in zip(got, (at, at, lengths[at], starts)):
            assert np.array_equal(g.cpu().numpy(), want), name
    announce("integer draws num=%d on the prefix" % num)
    p = pre_dev.clone()
    got = ops.sample_lookup(p, torch.from_numpy(t).cuda(), unit_uniforms=False,
                            lengths_table=lens_dev, local_out=p[n - num:])
    assert np.array_equal(got[0].cpu().numpy(), at) and np.array_equal(got[1].cpu().numpy(), at)


@pytest.mark.parametrize("num", SIZES)
def test_batch_outputs_on_top_of_float_draws_or_prefix(num):
    from gear_amd import ops
    rng = np.random.default_rng(num)
    n, T = 40_009, 7
    prefix = np.cumsum(rng.integers(0, 9, size=n).astype(np.float64))
    u = rng.random(num, dtype=np.float32)
    at = np.sort(np.minimum(np.searchsorted(prefix, u.astype(np.float64) * prefix[-1], side="right"), n - 1))
    for name in ("sorted_out", "idxs", "tss", "lens"):
        for where in ("draws", "prefix"):
            announce("float draws num=%d %s on the %s" % (num, name, where))
            p = torch.from_numpy(prefix).cuda()
            if where == "draws":      # the draws are the first half of the output's memory
                out = torch.empty(num, dtype=torch.int64, device="cuda")
                d = out.view(torch.float32)[:num]
                d.copy_(torch.from_numpy(u))
            else:
                out, d = p.view(torch.int64)[:num], torch.from_numpy(u).cuda()
            got = ops.sample_sorted(p, d, trajectory_length=T, **{name: out})
            for g, want in zip(got, (at, at // T, at % T, at % T + 1)):
                assert np.array_equal(g.cpu().numpy(), want), (name, where)
    p = torch.from_numpy(prefix).cuda()
    got = ops.sample_lookup(p, torch.from_numpy(u).cuda(), sampled_out=p.view(torch.int64)[:num])
    assert np.array_equal(got[0].cpu().numpy(), at) and np.array_equal(got[1].cpu().numpy(), at)


@pytest.mark.parametrize("num", SIZES)
@pytest.mark.parametrize("bound", [30_011, 1 << 40])
def test_look_ups_on_top_of_the_positions(num, bound):
    from gear_amd import ops
    rng = np.random.default_rng(num)
    pos = rng.integers(0, bound, size=num)
    for name in ("sampled_out", "local_out"):
        announce("positions num=%d bound=%d %s" % (num, bound, name))
        x = torch.from_numpy(pos).cuda()
        got = ops.sort_lookup(x, bound, index_offset=5, **{name: x})
        assert np.array_equal(got[0].cpu().numpy(), np.sort(pos)), name
        assert np.array_equal(got[1].cpu().numpy(), np.sort(pos) - 5), name


@pytest.mark.parametrize("num", [100, 4096, 4097, 50_000])
def test_updates_of_a_table_that_holds_their_indices(num):
    """The indices are read before the table, whose first entries they are, is written over."""
    from gear_amd import ops
    rng = np.random.default_rng(num)
    n = 70_001
    table = rng.integers(0, n, size=n)
    val = rng.integers(-5, 0, size=num)
    want = table.copy()
    for i, v in zip(table[:num], val):
        want[i] = v
    announce("updates num=%d by indices in the table" % num)
    got = torch.from_numpy(table).cuda()
    ops.scatter(got, got[:num], torch.from_numpy(val).cuda())
    assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("num", [4097, 20_000, 32_768])
def test_sorted_keys_on_top_of_a_part_of_the_payload(num):
    """Outputs that overlap inputs other than themselves, through the C ABI (the sort refuses outputs that
    are its inputs)."""
    import ctypes
    from gear_amd import _cabi
    lib = _cabi.load()
    rng = np.random.default_rng(num)
    keys = rng.integers(0, 1 << 16, size=num)      # two digits: the payload is read by the first launches
    order = np.argsort(keys, kind="stable")
    announce("sort num=%d with the keys stored over half of the payload" % num)
    block = torch.empty(num + num // 2, dtype=torch.int64, device="cuda")
    vin, kout = block[:num], block[num // 2:]
    vin.copy_(torch.arange(num, device="cuda"))
    kin, vout = torch.from_numpy(keys).cuda(), torch.empty(num, dtype=torch.int64, device="cuda")
    ws = torch.empty(int(lib.gear_hip_sort_workspace_bytes(num)), dtype=torch.uint8, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    code = lib.gear_hip_sort_i64(p(kin), p(kout), p(vin), p(vout), num, 16, p(ws), ws.numel(),
                                 ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert code == 0
    assert np.array_equal(vout.cpu().numpy(), order)
    assert np.array_equal(kout.cpu().numpy(), keys[order])
