"""Prefix sums at the sizes where the number of ranges changes the kernel: around 4096 and 8192
ranges of 16 granules per thread.  The inputs are small integers, so every sum is exact."""
import pytest

from conftest import announce

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

R32, R64 = 16 * 256 * 4, 16 * 256 * 2     # elements of such a range


@pytest.mark.parametrize("n", [4096 * R32, 4096 * R32 + 1, 8192 * R32 - 3, 8192 * R32, 8192 * R32 + 1])
def test_float_prefix(n):
    from gear_amd import ops
    announce("scan f32 n=%d" % n)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    w = torch.randint(0, 8, (n,), device="cuda", generator=g).float()
    state = ops.PrefixState()
    out = state.scan(w)
    assert torch.equal(out, torch.cumsum(w, 0, dtype=torch.float64))
    w[n // 2 + 5] += 3.0
    assert torch.equal(state.scan(w, n // 2 + 5), torch.cumsum(w, 0, dtype=torch.float64))


@pytest.mark.parametrize("n", [4096 * R64 + 1, 8192 * R64, 8192 * R64 + 1])
def test_integer_prefix(n):
    from gear_amd import ops
    announce("scan i64 n=%d" % n)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    w = torch.randint(0, 1 << 30, (n,), device="cuda", generator=g)
    assert torch.equal(ops.prefix_sum_i64(w), torch.cumsum(w, 0))


@pytest.mark.parametrize("n", [4096 * R32 // 2 + 1, 4096 * R32 + 77])
def test_rescans_of_wide_ranges_are_the_full_scan(n, monkeypatch):
    """Sums that round: the rescan of a suffix, chained or in two launches, has the full scan's bits."""
    from gear_amd import ops
    announce("rescan of wide ranges n=%d" % n)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    w = torch.rand(n, device="cuda", generator=g)
    for first in (1, R32 - 1, R32, n // 3, n - R32 // 2, n - 1):
        state = ops.PrefixState()
        state.scan(w)
        w[first:].mul_(1.5)
        want = ops.prefix_sum(w)
        got = state.scan(w, first).clone()
        assert torch.equal(got, want), first
        monkeypatch.setenv("GEAR_HIP_SCAN_SINGLE_PASS", "0")
        state.out[first:] = 0
        assert torch.equal(state.scan(w, first), want), first
        monkeypatch.delenv("GEAR_HIP_SCAN_SINGLE_PASS")


@pytest.mark.parametrize("n", [4096 * R64 // 2, 4096 * R64 // 2 + 1, 8192 * R64, 8192 * R64 + 1])
def test_captured_integer_prefix(n):
    from gear_amd import ops
    announce("captured i64 n=%d" % n)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    w = torch.randint(0, 1 << 30, (n,), device="cuda", generator=g)
    out = torch.empty_like(w)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        ops.prefix_sum_i64(w, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        ops.prefix_sum_i64(w, out=out)
    for _ in range(3):
        w.add_(1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, torch.cumsum(w, 0))
