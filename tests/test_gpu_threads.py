"""Python threads around the native calls: a call that has to wait for the GPU's queue lets others run,
and calls of two threads on one stream, which share scratch, do not mix."""
import threading
import time

import pytest

from conftest import announce

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def test_a_call_that_waits_for_its_queue_stops_no_other_thread():
    from gear_amd import ops
    table = torch.arange(64, device="cuda")
    idx = torch.arange(64, device="cuda")
    out = torch.empty_like(idx)
    ops.take_i64(table, idx, out=out)
    torch.cuda.synchronize()
    longest, done = [0.0], threading.Event()

    def watch():
        last = time.perf_counter()
        while not done.is_set():
            time.sleep(0.001)
            now = time.perf_counter()
            longest[0] = max(longest[0], now - last)
            last = now

    announce("more launches than the queue holds, behind a kernel of about a second")
    thread = threading.Thread(target=watch)
    thread.start()
    t0 = time.perf_counter()
    torch.cuda._sleep(2_000_000_000)
    slowest = 0.0
    for _ in range(20_000):
        t1 = time.perf_counter()
        ops.take_i64(table, idx, out=out)
        slowest = max(slowest, time.perf_counter() - t1)
    torch.cuda.synchronize()
    done.set()
    thread.join()
    print("slowest call %.3f s, longest pause of the other thread %.3f s, all %.3f s" % (
        slowest, longest[0], time.perf_counter() - t0), flush=True)
    assert longest[0] < 0.5 * max(slowest, 0.4)
    assert torch.equal(out, table)


@pytest.mark.parametrize("replaced", [False, True])
def test_two_threads_on_one_stream(replaced, monkeypatch):
    from gear_amd import ops
    if replaced:    # scratch handed out by somebody else's get(), one buffer a purpose as well
        monkeypatch.setattr(ops._ws, "get", ops._ws.get)
    n, k = 300_000, 5_000
    errors = []
    inputs = []
    for seed in range(2):
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        w = torch.randn(n, device="cuda", generator=g)
        keys = torch.randint(0, 1 << 40, (50_000,), device="cuda", generator=g)
        inputs.append((w, torch.topk(w, k).values, keys, keys.sort()[0]))
    torch.cuda.synchronize()
    announce("two threads on one stream")

    def work(w, top, keys, ordered):
        try:
            for _ in range(60):
                if not torch.equal(ops.topk(w, k)[0], top):
                    errors.append("top-k")
                if not torch.equal(ops.sort_i64(keys), ordered):
                    errors.append("sort")
        except Exception as e:  # noqa: BLE001 (reported by the test's own thread)
            errors.append(repr(e))

    threads = [threading.Thread(target=work, args=i) for i in inputs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors


def test_out_of_memory_is_torchs_own_error():
    from gear_amd import ops
    announce("an output larger than the GPU's memory")
    with pytest.raises(torch.OutOfMemoryError):
        ops.topk(torch.zeros(8, device="cuda"), 1 << 42)
