"""The lengths of a step on the host, which are waited for one by one: more of them than are looked at, a length
that is the mark of one still under way, and work of the caller's that makes the wait a long one."""
import pytest

from conftest import announce
from test_gpu_loader_step import CAP, _loader, _ops

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("num", [1, 33, 8192, 8193])
def test_lengths_on_the_host(num):
    loader = _loader("device", 20 + num % 7, batch=16)
    lengths = torch.randint(0, 1 << 40, (CAP,), device="cuda")
    lengths[3] = -(1 << 63)
    draws = torch.randint(0, CAP, (num,), device="cuda")
    draws[0] = 3
    host, errors = lengths.cpu(), []
    announce("lengths of %d windows" % num)
    for busy in (False, True, False):
        if busy:
            torch.cuda._sleep(20_000_000)
        sampled, timesteps, _, _ = loader._step.run("uniform", draws, None, loader._indices, 0, lengths, True,
                                                    _ops()._ws)
        if not torch.equal(timesteps, host[sampled.cpu()]):
            errors.append(busy)
    assert not errors
