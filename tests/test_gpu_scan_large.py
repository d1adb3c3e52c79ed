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
