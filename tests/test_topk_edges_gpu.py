"""Top-k at the sizes where its way changes (GPU), against torch's stable
sort: the sort's two limits (2^21 and 6 * 2^20 keys of one and two bytes, 2^18
and 3 * 2^20 of four), sub-chunks of one and of four vectors, and sizes just
above a multiple of the number of groups, with winners from a third of the
groups on either side."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SMALL = [(1 << 21), (1 << 21) + 1, 6 << 20, (6 << 20) + 1, 8_388_609, 9_000_001]
WIDE = [(1 << 18), (1 << 18) + 1, 3 << 20, (3 << 20) + 1, 4_194_305, 4_300_001, (1 << 25) + 1]


@pytest.mark.parametrize("dtype", [torch.float16, torch.int16, torch.int8, torch.float32, torch.int32], ids=str)
def test_topk_limits(ops, dev, dtype):
    b = torch.empty(0, dtype=dtype).element_size()
    for n in SMALL if b <= 2 else WIDE:
        g = torch.Generator(device=dev).manual_seed(n)
        x = torch.randn(n, generator=g, device=dev) if dtype.is_floating_point else torch.randint(
            torch.iinfo(dtype).min, torch.iinfo(dtype).max, (n,), generator=g, device=dev, dtype=dtype)
        x = x.to(dtype)
        ref = torch.sort(x, descending=True, stable=True)
        third = min(-(-n // (64 * 16 // b)), 16384) // 3
        for k in sorted({1, 300, 3000, min(third, 4096), min(third + 1, 4096), 4096, 4097, 20_000}):
            v, i = ops.run_topk(x, k, True)
            assert torch.equal(v, ref.values[:k]) and torch.equal(i.long(), ref.indices[:k]), (n, k)


@pytest.mark.parametrize("dtype,n", [(torch.float16, (1 << 29) + 2049), (torch.int32, (1 << 28) + 1025)], ids=str)
def test_topk_large_with_few_winners(ops, dev, dtype, n):
    """Sizes whose groups of 4096 would take more than 64 sub-chunks."""
    g = torch.Generator(device=dev).manual_seed(5)
    x = torch.empty(n, dtype=dtype, device=dev)
    for a in range(0, n, 1 << 27):
        m = min(1 << 27, n - a)
        x[a:a + m] = (torch.randn(m, generator=g, device=dev).to(dtype) if dtype == torch.float16 else
                      torch.randint(-2**30, 2**30, (m,), generator=g, device=dev, dtype=dtype))
    at = torch.tensor([0, n // 3, n - 2, n - 1], device=dev)
    top = torch.tensor([50, 60, 70, 60], dtype=torch.float64) * (1 if dtype == torch.float16 else 2**23)
    x[at] = top.to(dtype).to(dev) if dtype == torch.float16 else (top + 2**30).to(dtype).to(dev)
    for k in (1, 3, 1000):
        v, i = ops.run_topk(x, k, True)
        exp = torch.topk(x, k).values
        assert torch.equal(v, exp) and torch.equal(x[i.long()], v)
        want = [n - 2, n // 3, n - 1][:k]  # the two 60s in input order
        assert i[:3].tolist() == want
