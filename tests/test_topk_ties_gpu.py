"""Top-k where the winners lie together or repeat (GPU), against torch's
stable sort: ordered keys, a region of large ones, few values."""
import pytest
import torch

pytestmark = pytest.mark.gpu

KINDS = ["ordered", "reversed", "region", "four_values", "two_values_at_the_end"]


def _keys(kind, n, dtype, dev):
    g = torch.Generator(device=dev).manual_seed(n)
    x = torch.randn(n, generator=g, device=dev)
    if kind == "ordered":
        x = x.sort().values
    elif kind == "reversed":
        x = x.sort(descending=True).values
    elif kind == "region":
        a = n // 3
        x[a:a + 30_000] += 20
    elif kind == "four_values":
        x = torch.randint(0, 4, (n,), generator=g, device=dev).float()
    else:
        x = (torch.arange(n, device=dev) >= n - 50_000).float()
    return (x * 4).to(dtype) if dtype == torch.int8 else x.to(dtype)


@pytest.mark.parametrize("dtype,n", [(torch.float16, (1 << 21) + 1), (torch.float16, (1 << 26) + 8193),
                                     (torch.float32, (1 << 18) + 1), (torch.float32, (1 << 25) + 77),
                                     (torch.int8, (1 << 22) + 5)], ids=str)
@pytest.mark.parametrize("kind", KINDS)
def test_topk_winners_together(ops, dev, kind, dtype, n):
    x = _keys(kind, n, dtype, dev)
    for largest in (True, False):
        ref = torch.sort(x, descending=largest, stable=True)
        for k in (1, 300, 4096):
            v, i = ops.run_topk(x, k, largest)
            assert torch.equal(v, ref.values[:k]) and torch.equal(i.long(), ref.indices[:k]), (largest, k)
