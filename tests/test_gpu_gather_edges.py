"""Windows of a few bytes and windows that end inside a 16-byte vector, for every step size at which
their edges fall between words, between bytes, or leave a vector with nothing to copy."""
import numpy as np
import pytest

from conftest import announce

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("span", [1, 2, 3, 4, 5, 8, 17, 63])
@pytest.mark.parametrize("pad_head,zero_fill", [(False, True), (True, True), (True, False)])
def test_short_windows_of_every_step_size(oracle, span, pad_head, zero_fill):
    from gear_amd import ops
    T, cap, num = 70, 37, 101
    sizes = [1, 2, 3, 4, 6, 8, 12, 17, 20, 68, 100]
    rng = np.random.default_rng(span)
    announce("short windows span=%d head=%s fill=%s" % (span, pad_head, zero_fill))
    stride = T * sum(sizes)
    table = rng.integers(0, 256, size=cap * stride, dtype=np.uint8)
    idxs = rng.integers(0, cap, size=num)
    lens = rng.integers(0, T + 1, size=num)
    tss = np.maximum(lens + rng.integers(-3, 2, size=num), 0)   # windows past the end copy nothing
    ofst = -(span // 2)
    dsts = [torch.full((num, span * sb), 7, dtype=torch.uint8, device="cuda") for sb in sizes]
    bases = [T * sum(sizes[:c]) for c in range(len(sizes))]
    ops.subcopy_multi(torch.from_numpy(table).cuda(), *[torch.from_numpy(a).cuda() for a in
                                                       (idxs, tss, lens)], stride,
                      [dict(dst=dsts[c], ofst=ofst, span=span, step_bytes=sizes[c], col_base=bases[c],
                            pad_head=pad_head, zero_fill=zero_fill) for c in range(len(sizes))],
                      capacity=cap, trajectory_length=T)
    for c, sb in enumerate(sizes):
        exp = np.full((num, span * sb), 0 if zero_fill else 7, np.uint8)
        for w in range(num):
            first = max(tss[w] + ofst, 0)
            steps = max(min(first + span, lens[w]) - first, 0)
            at = (span - steps) * sb if pad_head else 0
            src = idxs[w] * stride + bases[c] + first * sb
            exp[w, at:at + steps * sb] = table[src:src + steps * sb]
        assert np.array_equal(dsts[c].cpu().numpy(), exp), (sb, c)
