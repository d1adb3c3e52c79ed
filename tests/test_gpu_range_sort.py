"""The one-launch sort of batches between the ranking sort and the radix sort: batch sizes at its
limits, keys spread evenly, crowded into a corner of their range, repeated more often than a
workgroup's list holds, in order already, and 64 bits wide; with and without a payload."""
import numpy as np
import pytest

from conftest import announce

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _keys(kind, num, bits, rng):
    top = (1 << bits) - 1
    if kind == "even":
        k = rng.integers(0, top, size=num, endpoint=True, dtype=np.uint64)
    elif kind == "few":                       # each key many times over
        k = rng.integers(0, 7, size=num).astype(np.uint64) * np.uint64(top // 7)
    elif kind == "crowded":                   # one far key, the others next to each other
        k = rng.integers(0, 3 * num, size=num).astype(np.uint64) & np.uint64(top)
        k[num // 2] = top
    elif kind == "repeats":                   # half of the batch is one key, inside a crowd
        k = rng.integers(0, 2000, size=num).astype(np.uint64)
        k[rng.permutation(num)[:num // 2]] = 1234
        k[0] = top
    elif kind == "equal":
        k = np.full(num, top, np.uint64)
    elif kind == "log":                       # every binary order of magnitude
        k = rng.integers(0, top, size=num, endpoint=True, dtype=np.uint64) >> \
            rng.integers(0, bits, size=num).astype(np.uint64)
    else:                                     # in order
        k = np.sort(rng.integers(0, top, size=num, endpoint=True, dtype=np.uint64))
        if kind == "nearly":
            k[num - 1] = k[0]
    return k


@pytest.mark.parametrize("num", [4097, 8192, 8193, 20_480, 20_481, 32_768, 32_769, 65_536, 65_537])
@pytest.mark.parametrize("bits", [13, 20, 32, 33, 63, 64])
def test_sort_is_the_stable_sort(num, bits):
    from gear_amd import ops
    rng = np.random.default_rng(num + bits)
    for kind in ("even", "few", "crowded", "repeats", "equal", "log", "ordered", "nearly"):
        announce("sort num=%d bits=%d %s" % (num, bits, kind))
        k = _keys(kind, num, bits, rng).view(np.int64)
        keys = torch.from_numpy(k).cuda()
        vals = torch.arange(num, device="cuda") * 3
        order = np.argsort(k.view(np.uint64), kind="stable")
        ko, vo = ops.sort_i64(keys, vals, key_bits=bits)
        assert np.array_equal(ko.cpu().numpy(), k[order]), kind
        assert np.array_equal(vo.cpu().numpy(), 3 * order), kind
        assert np.array_equal(ops.sort_i64(keys, key_bits=bits).cpu().numpy(), k[order]), kind


@pytest.mark.parametrize("num", [5000, 20_481, 40_000])
def test_only_the_low_bits_count(num):
    """Keys beyond key_bits are sorted by their low bits, in input order where those are equal."""
    from gear_amd import ops
    rng = np.random.default_rng(num)
    announce("sort low bits num=%d" % num)
    k = rng.integers(-(1 << 62), 1 << 62, size=num)
    for bits in (4, 20, 40):
        order = np.argsort(k & ((1 << bits) - 1), kind="stable")
        got = ops.sort_i64(torch.from_numpy(k).cuda(), key_bits=bits).cpu().numpy()
        assert np.array_equal(got, k[order])


@pytest.mark.parametrize("num", [4097, 20_000, 32_768, 32_769, 65_536, 65_537, 100_000])
@pytest.mark.parametrize("crowd", ["even", "narrow", "equal"])
def test_batches_of_draws(num, crowd):
    """Draws, integer draws with window starts and given positions beyond the ranking sort."""
    from gear_amd import ops
    rng = np.random.default_rng(num)
    n = 50_021
    announce("batch num=%d %s" % (num, crowd))
    u = rng.random(num)
    if crowd == "narrow":
        u = 0.25 + u * 1e-3
    elif crowd == "equal":
        u[num // 3:] = u[0]
    lengths = rng.integers(1, 40, size=n)
    prefix = np.cumsum(lengths)
    look = dict(index_table=torch.arange(n, device="cuda") * 5 + 7, index_offset=2,
                lengths_table=torch.from_numpy(lengths).cuda())

    def check(at, got):
        at = np.sort(at)
        local = at * 5 + 5
        lens = np.where(local < n, lengths[np.minimum(local, n - 1)], 0)
        assert np.array_equal(got[0].cpu().numpy(), at * 5 + 7)
        assert np.array_equal(got[1].cpu().numpy(), local)
        assert np.array_equal(got[2].cpu().numpy(), lens)
        return lens

    u32 = u.astype(np.float32)
    f64 = torch.from_numpy(prefix.astype(np.float64)).cuda()
    at = np.minimum(np.searchsorted(prefix, u32.astype(np.float64) * prefix[-1], side="right"), n - 1)
    check(at, ops.sample_lookup(f64, torch.from_numpy(u32).cuda(), **look))
    assert np.array_equal(ops.sample_sorted(f64, torch.from_numpy(u32).cuda(),
                                            unit_uniforms=True).cpu().numpy(), np.sort(at))
    v = rng.random(num)
    at = np.searchsorted(prefix, np.floor(u * prefix[-1]).astype(np.int64), side="right")
    got = ops.sample_lookup(torch.from_numpy(prefix).cuda(), torch.from_numpy(u).cuda(),
                            start_uniforms=torch.from_numpy(v).cuda(), window=4, **look)
    lens = check(at, got)
    starts = np.where(lens >= 4, np.floor(v * (lens - 3.0)), 0).astype(np.int64)
    assert np.array_equal(got[3].cpu().numpy(), starts)
    pos = np.floor(u * n).astype(np.int64)
    check(pos, ops.sort_lookup(torch.from_numpy(pos).cuda(), n, **look))


@pytest.mark.parametrize("num", [4097, 8193, 20_480, 20_481, 32_767, 32_768])
@pytest.mark.parametrize("bits", [17, 24, 32, 63])
def test_runs_of_equal_keys(num, bits):
    """Keys repeated about as often as a list may hold beside a share (448 times), or far more often;
    spaced evenly (one bank of the counts), far apart, and next to a key that is far from them all."""
    from gear_amd import ops
    rng = np.random.default_rng(num + bits)
    top = (1 << bits) - 1
    for run in (63, 127, 128, 129, 447, 448, 449, 450, 1000, num // 3, num // 2 + 1):
        for step in (1, 64, max(top // (num // run + 1), 1)):
            announce("runs num=%d bits=%d run=%d step=%d" % (num, bits, run, step))
            k = np.minimum(np.arange(num) // run * step, top)
            k[:3] = top
            k = rng.permutation(k)
            order = np.argsort(k, kind="stable")
            ko, vo = ops.sort_i64(torch.from_numpy(k).cuda(), torch.arange(num, device="cuda"),
                                  key_bits=bits)
            assert np.array_equal(vo.cpu().numpy(), order)
            assert np.array_equal(ko.cpu().numpy(), k[order])


@pytest.mark.parametrize("num", [4097, 12_288, 12_289, 20_481, 32_768])
@pytest.mark.parametrize("n", [1, 2, 5, 255, 256, 257])
def test_batches_from_a_few_entries(num, n):
    """Many positions or draws among few entries: the forms of both sides of the rules."""
    from gear_amd import ops
    rng = np.random.default_rng(num + n)
    announce("few entries num=%d n=%d" % (num, n))
    pos = rng.integers(0, n, size=num)
    got = ops.sort_lookup(torch.from_numpy(pos).cuda(), n, index_offset=1)
    assert np.array_equal(got[0].cpu().numpy(), np.sort(pos))
    assert np.array_equal(got[1].cpu().numpy(), np.sort(pos) - 1)
    prefix = np.cumsum(rng.integers(1, 4, size=n))
    u = rng.random(num)
    at = np.searchsorted(prefix, np.floor(u * prefix[-1]).astype(np.int64), side="right")
    got = ops.sample_lookup(torch.from_numpy(prefix).cuda(), torch.from_numpy(u).cuda())
    assert np.array_equal(got[0].cpu().numpy(), np.sort(at))
    u[: num // 2] = u[0]
    u = u.astype(np.float32)
    at = np.searchsorted(prefix, u.astype(np.float64) * prefix[-1], side="right")
    got = ops.sample_sorted(torch.from_numpy(prefix.astype(np.float64)).cuda(), torch.from_numpy(u).cuda())
    assert np.array_equal(got.cpu().numpy(), np.sort(np.minimum(at, n - 1)))


@pytest.mark.parametrize("bits", [20, 63])
def test_a_few_keys_take_no_multiple_of_the_time(bits):
    """A batch of two keys takes about 1.6 times a batch of distinct ones; it took 6 to 12 times when
    one workgroup stored a run by itself and the counts of one key followed each other."""
    from gear_amd import ops
    num = 32_768
    announce("time of a few keys, %d bits" % bits)
    g = torch.Generator(device="cuda")
    g.manual_seed(bits)
    distinct = torch.randint(0, 1 << bits if bits < 63 else 1 << 62, (num,), device="cuda", generator=g)
    two = torch.randint(0, 2, (num,), device="cuda", generator=g) * (1 << (bits - 2))

    def ms(x):
        best = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                ops.sort_i64(x, key_bits=bits)
            b.record()
            b.synchronize()
            best.append(a.elapsed_time(b))
        return min(best)

    ms(distinct)
    assert ms(two) < 3.0 * ms(distinct)
