"""int8 seg-sums whose tiles reach more rows than a workgroup has threads
(GPU): nearly all rows empty, at the ends, in the middle or everywhere, against
prefix differences."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [511, 512, 513, 1024, 2047, 2048, 2049, 6000, 300_001])
@pytest.mark.parametrize("place", ["front", "back", "middle", "spread", "one_value_rows"])
@pytest.mark.parametrize("idx", [torch.int32, torch.int64], ids=str)
def test_many_rows_a_tile(ops, dev, rows, place, idx):
    g = torch.Generator(device=dev).manual_seed(rows)
    nnz = 40_007
    if place == "front":
        p = torch.zeros(rows + 1, dtype=torch.int64, device=dev)
    elif place == "back":
        p = torch.full((rows + 1,), nnz, device=dev)
    elif place == "middle":
        p = torch.full((rows + 1,), nnz // 3, device=dev)
    elif place == "spread":
        p = torch.randint(0, 40, (rows + 1,), generator=g, device=dev).sort().values * 1000
    else:
        p = torch.arange(rows + 1, device=dev).clamp(max=nnz)
    p[0], p[-1] = 0, nnz
    x = torch.randint(-128, 128, (nnz,), generator=g, device=dev, dtype=torch.int8)
    c = torch.cat([torch.zeros(1, dtype=torch.int64, device=dev), x.long().cumsum(0)])
    y = ops.run_seg_sum_multi_core(x, p.to(idx), 128)
    assert torch.equal(y.long(), c[p[1:]] - c[p[:-1]])
