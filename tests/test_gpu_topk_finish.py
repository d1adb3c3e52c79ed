"""Top-k finished by its first level: a workgroup orders the few bins that concern it, fetched from every
workgroup's binned list.  Edges: bins that hold nearly, exactly and more than a workgroup orders (4096, less its
share of the output; by index 8192), a slot of equal keys, the zeros, the first and the last place; and what is left to the
launch behind it, whose phases hand over inside it, with several of them on the GPU at once."""
import numpy as np
import pytest

from conftest import announce

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _values(n, seed):
    return (np.random.default_rng(seed).lognormal(0, 1, size=n) ** 0.6).astype(np.float32)


def _check(oracle, w, k, label):
    from gear_amd import ops
    dw = torch.from_numpy(w).cuda()
    for by_value in (True, False):
        announce("topk %s n=%d k=%d by_value=%d" % (label, len(w), k, by_value))
        _, expected = oracle.topk_f32(w, k, by_value)
        state = ops.TopKState()
        for _ in range(2):  # from a sample, from the bound of the call before
            values, index = state.select(dw, k, sorted_by_value=by_value)
            torch.cuda.synchronize()
            assert np.array_equal(index.cpu().numpy(), expected), (label, by_value)
            assert np.array_equal(values.cpu().numpy().view(np.uint32), w[expected].view(np.uint32))
        none, index = ops.topk(dw, k, sorted_by_value=by_value, want_values=False)
        assert none is None and np.array_equal(index.cpu().numpy(), expected)


def _finished(state):
    """Whether level 1 of the state's last selection wrote the result (`done` of the workspace's header)."""
    return bool(state._ws[:256].view(torch.int32)[26].item())


@pytest.mark.parametrize("ties,at,finished", [(100, 5_000, True), (6_000, 10_000, True)])
def test_what_level_1_finishes_by_index(oracle, ties, at, finished):
    """A bin that holds too many entries is in the way only where the selection ends: not at the 2k-th key, the
    next call's bound."""
    from gear_amd import ops
    n, k = 600_001, 5_000
    w = _values(n, 3)
    order = np.argsort(-w, kind="stable")
    w[order[at:at + ties]] = w[order[at]]
    state = ops.TopKState()
    dw = torch.from_numpy(w).cuda()
    for _ in range(2):
        announce("topk by index, %d ties at the %d-th" % (ties, at))
        _, index = state.select(dw, k, sorted_by_value=False)
        assert np.array_equal(index.cpu().numpy(), oracle.topk_f32(w, k, False)[1])
        assert _finished(state) == finished


@pytest.mark.parametrize("n,k", [(262_144, 1), (262_145, 64), (262_207, 32_768), (1_048_577, 131_072),
                                 (1_500_001, 255), (1_500_001, 65_537), (5_000_011, 100_000), (10_000_000, 7_000)])
def test_sizes(oracle, n, k):
    _check(oracle, _values(n, n + k), k, "lognormal")


@pytest.mark.parametrize("ties", [64, 65, 2_000, 3_800, 4_094, 4_097, 30_000])
def test_equal_priorities_inside_the_selection(oracle, ties):
    n, k = 600_001, 20_000
    w = _values(n, ties)
    at = np.random.default_rng(ties).permutation(n)[:ties]
    order = np.sort(w)
    for where, value in (("at the top", order[-1]), ("at the threshold", order[-k]),
                         ("in the middle", order[-k // 2])):
        v = w.copy()
        v[at] = value
        _check(oracle, v, k, "%d ties %s" % (ties, where))


def test_zeros_and_infinities(oracle):
    n, k = 400_003, 30_000
    w = np.full(n, -1.0, np.float32) - _values(n, 5)
    rng = np.random.default_rng(6)
    at = rng.permutation(n)[:k + 500]
    w[at] = rng.random(k + 500, dtype=np.float32)
    w[at[:900]] = np.where(rng.random(900) < 0.5, np.float32(0.0), np.float32(-0.0))
    w[at[900:1000]] = np.inf
    _check(oracle, w, k, "both zeros around the threshold")


def _crowds(n, kind, rng):
    w = _values(n, n)
    top = np.float32(2) * w.max()
    if kind == "equal":
        w[:] = 1.0
    elif kind == "equal and negative":
        w[:] = -3.5
    elif kind == "both zeros":
        w = np.where(rng.random(n) < 0.5, np.float32(0.0), np.float32(-0.0))
    elif kind == "infinite":
        w[rng.random(n) < 0.4] = np.inf
    elif kind == "most at the top":
        w[rng.random(n) < 0.9] = top
    elif kind == "the last tenth at the top":
        w[-(n // 10):] = top
    elif kind == "ten values":
        w = rng.integers(0, 10, size=n).astype(np.float32)
    elif kind == "many values":  # bins of some 4500 entries each
        w = rng.integers(0, n // 4500 + 1, size=n).astype(np.float32)
    elif kind == "a mass below the best":
        w[rng.random(n) < 0.05] = top
        w[rng.permutation(n)[:300]] = top + np.arange(300, dtype=np.float32)
    return w


# n: one wave's ranges as long as its list (up to 1048576) and longer ones, whose lists a mass overflows
@pytest.mark.parametrize("kind", ["equal", "equal and negative", "both zeros", "infinite", "most at the top",
                                  "the last tenth at the top", "ten values", "many values",
                                  "a mass below the best"])
@pytest.mark.parametrize("n", [20_000, 262_145, 1_048_576, 1_048_577, 3_000_017])
def test_masses_of_equal_priorities_are_finished(oracle, n, kind):
    """A bin that holds more entries than a workgroup orders, all of the same priority."""
    from gear_amd import ops
    rng = np.random.default_rng(n)
    w = _crowds(n, kind, rng)
    ks = {1, 255, 5_000, min(n // 4, 131_072), min(n // 8 + 1, 100_001)}
    first = int((w == w.max()).sum())  # the largest priority's last place, and its neighbours
    ks |= {v for v in (first - 1, first, first + 1) if 0 < v <= min(n // 4, 131_072)}
    dw = torch.from_numpy(w).cuda()
    for k in sorted(ks):
        for by_value in (False, True):
            announce("topk %s n=%d k=%d by_value=%d" % (kind, n, k, by_value))
            _, expected = oracle.topk_f32(w, k, by_value)
            state = ops.TopKState()
            for _ in range(2):
                values, index = state.select(dw, k, sorted_by_value=by_value)
                assert np.array_equal(index.cpu().numpy(), expected), (kind, k, by_value)
                assert np.array_equal(values.cpu().numpy().view(np.uint32), w[expected].view(np.uint32))
            # (where lists overflow only crowds are left to place)
            if n <= 1_048_576 or kind in ("equal", "equal and negative", "both zeros") or \
                    kind == "most at the top" and k <= first:
                assert _finished(state), (kind, k, by_value)


def test_a_mass_with_neighbours_in_its_bin(oracle):
    n, k = 1_000_003, 40_000
    w = _values(n, 11)
    rng = np.random.default_rng(12)
    at = rng.permutation(n)[:k + 7_000]
    w[at] = np.float32(100.0)
    w[at[:50]] = np.nextafter(np.float32(100.0), np.float32(200.0))
    _check(oracle, w, k, "47000 ties, 50 an ulp above")
    w[at[50:90]] = np.nextafter(np.float32(100.0), np.float32(0.0))
    _check(oracle, w, k, "and 40 an ulp below")


def test_what_level_1_leaves_on_two_streams(oracle):
    """Selections that level 1 cannot finish, of two streams at once: neither launch has the GPU to itself."""
    n, k = 1_000_003, 50_000
    w = np.random.default_rng(8).integers(0, 50, size=n).astype(np.float32)
    _on_two_streams(oracle, w, k)


def test_bins_of_two_keys_on_two_streams(oracle):
    n, k = 1_000_003, 50_000
    rng = np.random.default_rng(9)
    w = rng.integers(0, 50, size=n).astype(np.float32)
    w[rng.permutation(n)[:2000]] += np.float32(1e-5)
    _on_two_streams(oracle, w, k)


@pytest.mark.parametrize("looks", ["0", "1", "8"])
def test_what_level_1_leaves_whatever_says_that_it_is_complete(oracle, monkeypatch, looks):
    """Level 2's histogram that adds up, or the flags of the workgroups; after a sample that misleads too."""
    monkeypatch.setenv("GEAR_HIP_TOPK_LOOKS", looks)
    rng = np.random.default_rng(10)
    n, k = 1_500_007, 20_000
    w = _values(n, 13)
    w[rng.random(n) < 0.04] = np.float32(7.0)
    w[rng.permutation(n)[:500]] = np.nextafter(np.float32(7.0), np.float32(8.0))
    _check(oracle, w, k, "two keys a bin, %s looks" % looks)
    s = np.arange(2048, dtype=np.uint64)
    stride = np.uint64(n // 2048)
    at = s * stride + (((s * np.uint64(2654435761)) & np.uint64(0xffffffff)) * stride >> np.uint64(32))
    w = _values(n, 14)
    w[at.astype(np.int64)] = 1000.0 + np.arange(2048, dtype=np.float32)
    _check(oracle, w, k, "a sample of the largest, %s looks" % looks)


def _on_two_streams(oracle, w, k):
    from gear_amd import ops
    dw = torch.from_numpy(w).cuda()
    expected = [torch.from_numpy(oracle.topk_f32(w, k, bool(v))[1]).cuda() for v in (0, 1)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    announce("topk of ties on two streams")
    torch.cuda.synchronize()
    got = []
    for turn in range(20):
        for s, stream in enumerate(streams):
            with torch.cuda.stream(stream):
                by_value = (turn + s) % 2
                got.append((by_value, ops.topk(dw, k, sorted_by_value=bool(by_value))[1]))
    torch.cuda.synchronize()
    for by_value, index in got:
        assert torch.equal(index, expected[by_value])


@pytest.mark.parametrize("n,k", [(2_048, 1), (2_049, 512), (4_097, 1_024), (10_007, 2_501), (32_768, 8_192),
                                 (131_073, 32_768), (1_048_576, 131_072), (1_048_576, 250_000)])
def test_small_inputs_and_large_shares(oracle, n, k):
    w = _values(n, n + k)
    _check(oracle, w, k, "lognormal")
    _check(oracle, np.full(n, 1.0, np.float32), k, "all equal")


@pytest.mark.parametrize("n,k", [(5_000, 600), (60_000, 3_000), (1_000_000, 50_000)])
def test_neighbours_in_the_input_that_are_neighbours_in_value(oracle, n, k):
    """A workgroup's entries lie in one other's list: dealt out to its threads."""
    w = np.sort(_values(n, k))
    _check(oracle, w, k, "ascending")
    _check(oracle, w[::-1].copy(), k, "descending")
    _check(oracle, np.arange(n, dtype=np.float32), k, "0 to n - 1")


@pytest.mark.parametrize("crowd", ["stretch", "two values", "neighbours", "two stretches", "close", "two clusters"])
@pytest.mark.parametrize("ties", [65, 1_025, 3_000])
def test_a_crowded_slot(oracle, crowd, ties):
    n, k = 300_007, 2_500
    w = _values(n, ties)
    rng = np.random.default_rng(ties)
    top = np.float32(2) * w.max()
    at = rng.permutation(n)[:ties]
    if crowd == "stretch":
        w[100_000:100_000 + ties] = top
    elif crowd == "two values":
        w[at] = np.where(rng.random(ties) < 0.5, top, np.float32(1.5) * top)
    elif crowd == "neighbours":  # a few ulps apart
        w[at] = (np.full(ties, top).view(np.uint32) + rng.integers(0, 5, ties).astype(np.uint32)).view(np.float32)
    elif crowd == "close":  # several crowded slots
        w[at] = top * (1 + rng.random(ties, dtype=np.float32) * np.float32(4e-4))
    elif crowd == "two clusters":
        w[at] = (np.full(ties, top).view(np.uint32) + rng.integers(0, 26, ties).astype(np.uint32)).view(np.float32)
        w[at[:ties // 3]] *= np.float32(1.002)
    else:
        w[5:5 + ties // 2] = top
        w[n - ties // 2:] = top
    _check(oracle, w, k, "%d %s" % (ties, crowd))


@pytest.mark.parametrize("together", [4_096, 4_097, 8_192, 8_193])
def test_the_most_entries_that_level_1_looks_through_by_index(oracle, together):
    """Of a bin that is not one key."""
    from gear_amd import ops
    n, k = 300_007, 2_500
    w = _values(n, 7)
    rng = np.random.default_rng(together)
    top = np.float32(2) * w.max()
    w[rng.permutation(n)[:together]] = (np.full(together, top).view(np.uint32) +
                                        rng.integers(0, 5, together).astype(np.uint32)).view(np.float32)
    _check(oracle, w, k, "%d together" % together)
    state = ops.TopKState()
    announce("topk by index, %d together" % together)
    state.select(torch.from_numpy(w).cuda(), k, sorted_by_value=False)
    assert _finished(state) == (together <= 8_192)
