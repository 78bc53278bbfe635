"""The pipelined plain scan through its look-back fallback (poll limit 0) at
its default tiles and each default window: above the short scan's sizes (64
predecessors a step), above 2^23 (16) and above 2^26 elements (6) (GPU)."""
import pytest
import torch

import oracle
from _util import assert_exact, gen, to_np, uniform_pm1

pytestmark = pytest.mark.gpu


@pytest.fixture
def fallback(ops, dev):
    like = torch.empty(1, device=dev)
    ops._set_lookback_poll_limit(like, 0)
    torch.cuda.synchronize()
    yield
    ops._set_lookback_poll_limit(like, -1)
    torch.cuda.synchronize()


@pytest.mark.parametrize("n", [(3 << 20) + 333, (1 << 23) + 333, (1 << 26) + 333])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32, torch.int8], ids=str)
def test_pipelined_scan_fallback(ops, dev, fallback, n, dtype):
    x = (torch.randint(-4, 5, (n,), generator=gen(n), dtype=torch.int8) if dtype == torch.int8
         else uniform_pm1(n, dtype, n))
    y = ops.run_scan_single_core(x.to(dev), 128, 0.0)
    assert_exact(to_np(y), oracle.scan(to_np(x)), f"{dtype} n={n}")
