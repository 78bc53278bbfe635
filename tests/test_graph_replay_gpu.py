"""Top-k, searchsorted and int8 seg-sums in one captured graph (GPU): replays on
inputs that take each of their ways (the select behind the maxima and not,
tiles of one slice and not) equal the calls made eagerly, with eager calls
between the replays."""
import pytest
import torch

pytestmark = pytest.mark.gpu

LO, HI = -2**31, 2**31 - 1


def test_replays_equal_eager_calls(ops, dev):
    g = torch.Generator(device=dev).manual_seed(3)

    def ints(n):
        return torch.randint(LO, HI, (n,), generator=g, device=dev, dtype=torch.int32)

    hay = ints(1 << 21).sort().values
    v = ints((1 << 20) + 16385)
    x = torch.randn((1 << 22) + 5, generator=g, device=dev).half()
    w = ints((1 << 20) + 3)
    x8 = torch.randint(-128, 128, (1 << 20,), generator=g, device=dev, dtype=torch.int8)
    p = torch.arange(0, (1 << 20) + 1, 64, device=dev, dtype=torch.int32)

    def calls():
        return [ops.run_searchsorted(hay, v), *ops.run_topk(x, 300, True), *ops.run_topk(w, 2048, False),
                ops.run_seg_sum_multi_core(x8, p, 128)]

    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        for _ in range(2):
            calls()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        outs = calls()
    for turn in range(5):
        nv, nx, nw = ints(v.numel()), torch.randn(x.numel(), generator=g, device=dev).half(), ints(w.numel())
        if turn == 1:  # in order
            nv, nx, nw = nv.sort().values, nx.sort().values, nw.sort().values
        elif turn == 3:  # one value
            nv, nx, nw = torch.full_like(nv, 7), torch.full_like(nx, 1.5), torch.full_like(nw, -3)
        v.copy_(nv)
        x.copy_(nx)
        w.copy_(nw)
        p[1:-1] = torch.randint(0, 1 << 20, (p.numel() - 2,), generator=g, device=dev).sort().values.int()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for i, (a, b) in enumerate(zip(outs, calls())):
            assert torch.equal(a, b), (turn, i)
        assert torch.equal(outs[0], torch.searchsorted(hay, v, out_int32=True)), turn
        assert torch.equal(outs[1], torch.sort(x, descending=True, stable=True).values[:300]), turn
