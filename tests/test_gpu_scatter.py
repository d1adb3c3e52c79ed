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


def _expected(n, idx, val):
    want = np.zeros(n, val.dtype)
    last = np.full(n, -1)
    inside = (idx >= 0) & (idx < n)
    np.maximum.at(last, idx[inside], np.nonzero(inside)[0])
    want[last >= 0] = val[last[last >= 0]]
    return want


@pytest.mark.parametrize("num", [40_960, 40_961, 131_071, 131_072, 131_073])
@pytest.mark.parametrize("n", [255, 256, 70_000])
def test_limits_of_the_one_launch_form(num, n):
    from gear_amd import ops
    rng = np.random.default_rng(num + n)
    for kind in ("random", "turns"):
        announce("scatter limits num=%d n=%d %s" % (num, n, kind))
        idx = _indices(kind, n, num, rng)
        val = np.arange(1, num + 1)
        got = torch.zeros(n, dtype=torch.int64, device="cuda")
        ops.scatter(got, torch.from_numpy(idx).cuda(), torch.from_numpy(val).cuda())
        assert np.array_equal(got.cpu().numpy(), _expected(n, idx, val))


@pytest.mark.parametrize("distinct,num", [(1500, 4096), (2048, 2048), (2049, 2049), (3000, 9000),
                                          (20_000, 50_000), (100_000, 131_072)])
def test_indices_that_crowd_in_one_class(distinct, num):
    """Indices that all belong to one workgroup's hash table of 2048 slots, so that it takes them in 2, 4,
    ... 64 parts (the class of an index as scatter.hip computes it)."""
    from gear_amd import ops
    n = 1 << 25
    x = np.arange(n, dtype=np.uint64)
    own = (((x ^ (x >> np.uint64(15))) & np.uint64(0xffffff)) * np.uint64(0x9E3779) & np.uint64(0xffffffff)) \
        >> np.uint64(24)
    rng = np.random.default_rng(distinct)
    some = rng.permutation(np.nonzero(own == 77)[0])[:distinct]
    assert len(some) == distinct
    idx = np.concatenate([some, some[rng.integers(0, distinct, size=num - distinct)]]).astype(np.int64)
    rng.shuffle(idx)
    val = np.arange(1, num + 1).astype(np.float32)
    announce("scatter one class distinct=%d num=%d" % (distinct, num))
    got = torch.zeros(n, device="cuda")
    ops.scatter(got, torch.from_numpy(idx).cuda(), torch.from_numpy(val).cuda())
    want = _expected(n, idx, val)
    assert np.array_equal(got[torch.from_numpy(some).cuda()].cpu().numpy(), want[some])
    assert int((got != 0).sum()) == distinct


def test_a_short_table_takes_no_longer_than_a_long_one():
    """131072 updates of 5 entries: one digit to sort (14 us against 23 for a long table); each workgroup
    that looked through them for the few of its class took 32."""
    from gear_amd import ops
    num = 131_072
    announce("time of updates of a short table")

    def ms(n):
        w, v = torch.zeros(n, device="cuda"), torch.ones(num, device="cuda")
        at = torch.randint(0, n, (num,), device="cuda")
        best = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                ops.scatter(w, at, v)
            b.record()
            b.synchronize()
            best.append(a.elapsed_time(b))
        return min(best)

    ms(5)
    assert ms(5) < 1.1 * ms(10_000_000)
