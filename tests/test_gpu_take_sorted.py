"""table[idx] in ascending order: entries that come in order (the sort ends at once) and entries that do not,
at the edges of the look-up's workgroups and of the sorts behind it."""
import numpy as np
import pytest

from conftest import announce

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("num", [1, 2, 255, 256, 257, 512, 513, 4095, 4096, 4097, 20_000, 32_768, 32_769, 70_001])
def test_take_sorted(num):
    from gear_amd import ops
    rng = np.random.default_rng(num)
    n = 100_003
    ascending = np.sort(rng.integers(0, 1 << 62, size=n))
    idx = np.sort(rng.integers(0, n, size=num))
    tables = {"ascending": ascending, "shuffled": rng.permutation(ascending), "constant": np.full(n, 7)}
    swapped = ascending.copy()  # one pair out of order, across a workgroup's edge where there is one
    at = min(255, num - 2) if num > 1 else 0
    swapped[idx[at]], swapped[idx[min(at + 1, num - 1)]] = ascending[-1], ascending[0]
    tables["one pair swapped"] = swapped
    outside = idx.copy()
    outside[num // 2] = n  # reads as 0
    for name, table in tables.items():
        for what, i in (("in range", idx), ("one outside", outside)):
            announce("take_sorted %s, %s, num=%d" % (name, what, num))
            got = ops.take_sorted_i64(torch.from_numpy(table).cuda(), torch.from_numpy(i).cuda())
            padded = np.append(table, 0)
            assert np.array_equal(got.cpu().numpy(), np.sort(padded[i])), name
