"""Counts of filters and compactions called from several threads, each on a
stream of its own (GPU).  An exception in a thread fails the test, and every
thread has to end its calls.  The bindings hold the interpreter lock through a
call, so the threads interleave between calls, not inside one."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_counts_of_threads(ops, dev):
    errors, done = [], []

    def run(seed):
        try:
            g = torch.Generator(device=dev).manual_seed(seed)
            with torch.cuda.stream(torch.cuda.Stream()):
                for i in range(30):
                    x = torch.randn(70_000 * (i % 3) + 501 * seed + 37 * i + 1, generator=g, device=dev)
                    m = (x > 0.1 * seed).to(torch.int8)
                    assert torch.equal(ops.run_filter_greater_eq(x, 0.25 * seed, 128), x[x >= 0.25 * seed]), i
                    assert torch.equal(ops.run_compress(x, m, 128), x[m.bool()]), i
                    assert torch.equal(ops.run_where(x, 0.25 * seed, 128).long(),
                                       torch.nonzero(x >= 0.25 * seed).flatten()), i
            done.append(seed)
        except BaseException as e:  # noqa: BLE001 - reported below
            errors.append((seed, repr(e)))

    threads = [threading.Thread(target=run, args=(s,)) for s in range(1, 5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors and sorted(done) == [1, 2, 3, 4]
