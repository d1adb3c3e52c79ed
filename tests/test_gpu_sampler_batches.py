"""Batches of draws at the sizes where the search and the one-launch sorted batch change shape:
numbers of draws around a workgroup's share and around the limits of the lanes per draw, prefixes
of a few entries, runs of zero priorities, draws that repeat, leave [0, sum) or are not numbers."""
import numpy as np
import pytest

from conftest import announce

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _found(prefix, targets):
    """upper_bound of the targets, clipped; a target that is not a number finds entry 0."""
    at = np.searchsorted(prefix, np.where(np.isnan(targets), -np.inf, targets), side="right")
    return np.minimum(at, len(prefix) - 1)


@pytest.mark.parametrize("n", [1, 2, 7, 8, 15, 16, 17, 255, 4097, 1_000_003])
@pytest.mark.parametrize("num", [1, 15, 16, 17, 511, 1024, 4095, 4096, 4097, 32_768, 32_769])
def test_draws_in_a_float_prefix(n, num):
    from gear_amd import ops
    rng = np.random.default_rng(1000 * num + n)
    announce("draws n=%d num=%d" % (n, num))
    pri = rng.integers(0, 9, size=n).astype(np.float32)      # exact sums, a ninth of them zeros
    pri[rng.integers(0, n)] = 5.0
    prefix = np.cumsum(pri.astype(np.float64))
    dev = torch.from_numpy(prefix).cuda()
    for unit in (True, False):
        u = rng.random(num, dtype=np.float32)
        if not unit:
            u = np.floor(u * np.float32(prefix[-1]))         # targets that hit entries exactly
        u[rng.integers(0, num, size=num // 3)] = u[0]
        odd = np.array([np.nan, -0.0, 0.0, 1.0, -1.0, 3e38, np.inf, -np.inf], np.float32)
        u[rng.integers(0, num, size=min(num // 2, 8))] = odd[:min(num // 2, 8)]
        with np.errstate(invalid="ignore"):
            want = _found(prefix, u.astype(np.float64) * (prefix[-1] if unit else 1.0))
        draws = torch.from_numpy(u).cuda()
        got = ops.upper_bound(dev, draws, unit_uniforms=unit).cpu().numpy()
        assert np.array_equal(got, want)
        flat, idxs, tss, lens = [t.cpu().numpy() for t in ops.sample_sorted(
            dev, draws, unit_uniforms=unit, trajectory_length=7, modulo=n)]
        assert np.array_equal(flat, np.sort(want))
        assert np.array_equal(idxs, flat // 7) and np.array_equal(tss, flat % 7)
        assert np.array_equal(lens, tss + 1)


@pytest.mark.parametrize("num", [1, 16, 17, 1000, 4096, 4097])
def test_draws_in_an_integer_prefix_and_given_positions(num):
    from gear_amd import ops
    n = 5003
    rng = np.random.default_rng(num)
    announce("integer draws num=%d" % num)
    lengths = rng.integers(0, 50, size=n)
    lengths[-1] = 1 << 40                                     # a total beyond 32 bits
    prefix = np.cumsum(lengths)
    table = torch.from_numpy(rng.integers(0, 1 << 40, size=n)).cuda()
    t = rng.integers(-5, prefix[-2] + 5, size=num)
    t[num // 2:] = t[0]
    got = ops.sample_lookup(torch.from_numpy(prefix).cuda(), torch.from_numpy(t).cuda(),
                            unit_uniforms=False, index_table=table,
                            index_offset=3)
    want = np.sort(np.minimum(np.searchsorted(prefix, t, side="right"), n - 1))
    assert np.array_equal(got[0].cpu().numpy(), table.cpu().numpy()[want])
    assert np.array_equal(got[1].cpu().numpy(), table.cpu().numpy()[want] - 3)
    pos = rng.integers(0, n, size=num)
    got = ops.sort_lookup(torch.from_numpy(pos).cuda(), n, index_table=table,
                          lengths_table=torch.from_numpy(lengths).cuda())
    want = np.sort(pos)
    assert np.array_equal(got[0].cpu().numpy(), table.cpu().numpy()[want])


@pytest.mark.parametrize("num", [17, 4096, 4097, 20_481, 32_768, 32_769])
@pytest.mark.parametrize("total", [0.0, np.inf, -np.inf, np.nan])
def test_batches_ascend_whatever_the_total_is(num, total):
    """Unit draws times a total of 0, an infinity or no number: some targets are not numbers, which find
    entry 0, wherever the draw lies among the others."""
    from gear_amd import ops
    rng = np.random.default_rng(num)
    n = 1000
    prefix = np.zeros(n) if total == 0.0 else np.arange(1.0, n + 1.0)
    prefix[-3:] = total
    u = rng.random(num, dtype=np.float32)
    odd = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1.0, -1.0], np.float32)
    u[rng.integers(0, num, size=num // 2)] = odd[rng.integers(0, len(odd), size=num // 2)]
    announce("batch of %d draws, total %r" % (num, total))
    dev, draws = torch.from_numpy(prefix).cuda(), torch.from_numpy(u).cuda()
    got = ops.sample_sorted(dev, draws, unit_uniforms=True).cpu().numpy()
    assert np.all(got[:-1] <= got[1:])
    found = ops.upper_bound(dev, draws, unit_uniforms=True).cpu().numpy()
    if total in (0.0, np.inf):       # (the prefix ascends: what is found does not depend on the probes)
        assert np.array_equal(got, np.sort(found))


@pytest.mark.parametrize("num", [4096, 4097, 8192, 8193, 20_480, 20_481, 32_768, 32_769])
def test_batches_ascend_in_a_prefix_with_dips(num):
    """A prefix of rounded sums can dip by a unit in the last place behind zero priorities."""
    from gear_amd import ops
    rng = np.random.default_rng(num)
    n = 20_011
    prefix = np.cumsum(rng.random(n) * (rng.random(n) < 0.3))
    dips = rng.integers(1, n - 1, size=n // 4)
    prefix[dips] = np.nextafter(prefix[dips], 0.0)
    u = (prefix[rng.integers(0, n, size=num)] / prefix[-1]).astype(np.float32)   # draws at the entries
    announce("batch of %d draws, prefix with dips" % num)
    dev = torch.from_numpy(prefix).cuda()
    got = ops.sample_sorted(dev, torch.from_numpy(u).cuda(), unit_uniforms=True).cpu().numpy()
    assert np.all(got[:-1] <= got[1:])
    t = prefix[rng.integers(0, n, size=num)].astype(np.float32)
    got = ops.sample_lookup(dev, torch.from_numpy(t).cuda(), unit_uniforms=False)[0].cpu().numpy()
    assert np.all(got[:-1] <= got[1:])


@pytest.mark.parametrize("num", [1, 17, 4096, 4097, 24_576, 24_577, 32_768, 32_769, 49_152, 49_153])
def test_importance_weights_at_the_limits_of_the_search(num):
    """Weights against the same in float64, rounded once: two roundings of float32 apart at most."""
    from gear_amd import ops
    rng = np.random.default_rng(num)
    n = 30_011
    pri = rng.lognormal(size=n).astype(np.float32)
    prefix = np.cumsum(pri.astype(np.float64))
    u = rng.random(num, dtype=np.float32)
    announce("importance weights num=%d" % num)
    at, w = ops.upper_bound(torch.from_numpy(prefix).cuda(), torch.from_numpy(u).cuda(),
                            unit_uniforms=True, priorities=torch.from_numpy(pri).cuda(), beta=0.4)
    want = np.minimum(np.searchsorted(prefix, u.astype(np.float64) * prefix[-1], side="right"), n - 1)
    assert np.array_equal(at.cpu().numpy(), want)
    raw = (n * pri[want].astype(np.float64) / prefix[-1]) ** -0.4
    assert np.max(np.abs(w.cpu().numpy() / (raw / raw.max()) - 1)) < 2.0 ** -23
