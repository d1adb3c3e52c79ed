"""Priority updates with repeated indices, last one wins: batches at the limits of the one-launch
form and of the hash table, indices that repeat in runs, in turn and everywhere, indices outside
the table, and a table with more entries than 32 bits count."""
import numpy as np
import pytest

from conftest import announce

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _indices(kind, n, num, rng):
    if kind == "random":
        return rng.integers(-2, n + 2, size=num)       # some outside the table: ignored
    if kind == "runs":
        return np.sort(rng.integers(0, max(1, n // 7), size=num))
    if kind == "turns":
        return np.arange(num) % 3 * ((n - 1) // 3)
    if kind == "equal":
        return np.full(num, n - 1)
    return np.arange(num)[::-1] * 64 % n               # a stride


@pytest.mark.parametrize("dtype", ["float32", "int64"])
@pytest.mark.parametrize("num", [1, 2, 63, 64, 65, 1023, 4095, 4096, 4097, 65_536, 200_001])
def test_last_update_wins(oracle, num, dtype):
    from gear_amd import ops
    rng = np.random.default_rng(num)
    for n in (1, 5, 1000, 300_007):
        for kind in ("random", "runs", "turns", "equal", "stride"):
            announce("scatter %s num=%d n=%d %s" % (dtype, num, n, kind))
            idx = _indices(kind, n, num, rng)
            val = np.arange(1, num + 1).astype(dtype)
            want = np.zeros(n, dtype)
            inside = (idx >= 0) & (idx < n)
            last = np.full(n, -1)
            np.maximum.at(last, idx[inside], np.nonzero(inside)[0])
            want[last >= 0] = val[last[last >= 0]]
            got = torch.zeros(n, dtype=getattr(torch, dtype), device="cuda")
            ops.scatter(got, torch.from_numpy(idx).cuda(), torch.from_numpy(val).cuda(),
                        unique_indices=False)
            assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("num", [1000, 20_000])
def test_more_entries_than_32_bits_count(num):
    from gear_amd import ops
    announce("scatter beyond 2**32 entries num=%d" % num)
    n = (1 << 32) + 77
    table = torch.empty(n, device="cuda")
    rng = np.random.default_rng(num)
    idx = rng.integers(0, n, size=num)
    idx[::3] = idx[0] + (1 << 32) * (idx[0] < 77)          # repeats
    idx[1::3] = (1 << 32) + rng.integers(0, 77, size=len(idx[1::3]))
    val = np.arange(num, dtype=np.float32)
    dev = torch.from_numpy(idx).cuda()
    ops.scatter(table, dev, torch.from_numpy(val).cuda(), unique_indices=False)
    last = {i: v for i, v in zip(idx.tolist(), val.tolist())}
    assert table[dev].cpu().numpy().tolist() == [last[i] for i in idx.tolist()]
