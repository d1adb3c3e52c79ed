"""Prefix sums of more than 6656 ranges, whose sums are handed on by groups of 64: sizes around whole groups and
the last one that a single pass takes, and the bounded waits of ranges and groups running out.  Integer-valued
inputs, so every sum is exact."""
import pytest

from conftest import announce

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

R32, R64 = 16 * 256 * 4, 16 * 256 * 2     # elements of a range of 16 granules a thread


def _weights(n, dtype):
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    return torch.randint(0, 8, (n,), device="cuda", generator=g).to(dtype)


@pytest.mark.parametrize("n", [6656 * R32, 6656 * R32 + 1, 6720 * R32 - 1, 6720 * R32, 6720 * R32 + 1, 6783 * R32 + 5,
                               16384 * R32, 16384 * R32 + 1])
def test_float_prefix(n, monkeypatch):
    from gear_amd import ops
    w = _weights(n, torch.float32)
    want = torch.cumsum(w, 0, dtype=torch.float64)
    announce("grouped scan f32 n=%d" % n)
    assert torch.equal(ops.prefix_sum(w), want)
    monkeypatch.setenv("GEAR_HIP_SCAN_SINGLE_PASS", "0")
    announce("... in two launches")
    assert torch.equal(ops.prefix_sum(w), want)


@pytest.mark.parametrize("n", [6720 * R64 + 1, 16384 * R64, 16384 * R64 + 1])
def test_integer_prefix(n):
    from gear_amd import ops
    announce("grouped scan i64 n=%d" % n)
    w = _weights(n, torch.int64)
    assert torch.equal(ops.prefix_sum_i64(w), torch.cumsum(w, 0))


@pytest.mark.parametrize("limit", [0, 3])
def test_waits_that_run_out(limit, monkeypatch):
    from gear_amd import ops
    n = 6721 * R32 + 9
    w = _weights(n, torch.float32)
    want = torch.cumsum(w, 0, dtype=torch.float64)
    monkeypatch.setenv("GEAR_HIP_SCAN_SPIN_LIMIT", str(limit))
    announce("grouped scan, %d polls" % limit)
    state = ops.PrefixState()
    assert torch.equal(state.scan(w), want)
    for first in (64 * R32 * 3 + 1, n - 70 * R32, n - 1):
        w[first] += 2.0
        announce("grouped rescan from %d, %d polls" % (first, limit))
        assert torch.equal(state.scan(w, first), torch.cumsum(w, 0, dtype=torch.float64))
