"""searchsorted at the ends of what its arguments allow (GPU): the longest
haystacks, and haystacks that are not sorted, whose results are unspecified
but stay in range."""
import ctypes
import os

import pytest
import torch

pytestmark = pytest.mark.gpu

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(REPO, "pytorch-tcuscan_amd", "libtcuscan_hip.so")
I32_MIN, I32_MAX = -2**31, 2**31 - 1


@pytest.fixture(scope="module")
def lib():
    lib = ctypes.CDLL(LIB)
    lib.tcs_searchsorted_indexed.argtypes = [ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p, ctypes.c_void_p,
                                             ctypes.c_int64, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p]
    for f in (lib.tcs_searchsorted_workspace_bytes, lib.tcs_searchsorted_preferred_bytes):
        f.restype = ctypes.c_size_t
    lib.tcs_searchsorted_workspace_bytes.argtypes = [ctypes.c_int64]
    lib.tcs_searchsorted_preferred_bytes.argtypes = [ctypes.c_int64, ctypes.c_int64]
    return lib


def _indexed(lib, hay, needles, wsb):
    """The lower bounds by tcs_searchsorted_indexed with wsb bytes of stale
    workspace; nothing written past it."""
    ws = torch.full((wsb // 4 + 8,), -1, dtype=torch.int32, device=hay.device)
    out = torch.full_like(needles, -7)
    assert lib.tcs_searchsorted_indexed(hay.data_ptr(), hay.numel(), needles.data_ptr(), out.data_ptr(),
                                        needles.numel(), ws.data_ptr(), wsb,
                                        torch.cuda.current_stream().cuda_stream) == 0
    assert bool((ws[wsb // 4:] == -1).all())
    return out


@pytest.mark.parametrize("n", [2**31 - 512, 2**31 - 1])
def test_longest_haystacks(lib, ops, dev, n):
    """n elements -2^30, -2^30 + 1, ...: from n = 2^31 - 511 on the table
    build's elements per workgroup, rounded up, pass int32."""
    hay = torch.arange(-2**30, n - 2**30, dtype=torch.int32, device=dev)
    g = torch.Generator(device=dev).manual_seed(31)
    v = torch.randint(I32_MIN, I32_MAX, ((1 << 23) + 5,), generator=g, device=dev, dtype=torch.int32)
    v[:4] = torch.tensor([I32_MIN, I32_MAX, -2**30, n - 2**30 - 1], dtype=torch.int32)
    exp = (v.long() + 2**30).clamp(0, n).int()
    for m in (70_000, v.numel()):
        assert torch.equal(ops.run_searchsorted(hay, v[:m].contiguous()), exp[:m])
        assert torch.equal(_indexed(lib, hay, v[:m].contiguous(), lib.tcs_searchsorted_workspace_bytes(n)), exp[:m])


@pytest.mark.parametrize("n", [70_001, (1 << 20) + 3, (1 << 22) + 5])
@pytest.mark.parametrize("order", ["descending", "shuffled", "zigzag", "beyond_ends", "sorted"])
def test_unsorted_haystacks_stay_in_range(lib, ops, dev, n, order):
    """Every answer lies in [0, n] and nothing outside the workspace and the
    outputs is written, whatever the order of the haystack: by sixteen lanes
    a needle, by the table (of the least workspace and the preferred one) and
    by slices; a later search of a sorted haystack is right."""
    g = torch.Generator(device=dev).manual_seed(n)
    hay = torch.randint(I32_MIN, I32_MAX, (n,), generator=g, device=dev, dtype=torch.int32).sort().values
    good = hay.clone()
    if order == "descending":
        hay = hay.flip(0).contiguous()
    elif order == "shuffled":
        hay = hay[torch.randperm(n, generator=g, device=dev)]
    elif order == "zigzag":  # falls and rises across the whole table
        hay[0::2], hay[1::2] = good[: (n + 1) // 2], good[(n + 1) // 2:].flip(0)
    elif order == "beyond_ends":  # keys outside the first and last element
        hay[n // 3], hay[n // 2], hay[0], hay[-1] = I32_MIN, I32_MAX, -1000, 1000
    for m in (1000, 70_000, 600_001, (3 << 20) + 5):
        v = torch.randint(I32_MIN, I32_MAX, (m,), generator=g, device=dev, dtype=torch.int32)
        for out in (ops.run_searchsorted(hay, v), _indexed(lib, hay, v, lib.tcs_searchsorted_workspace_bytes(n)),
                    _indexed(lib, hay, v, lib.tcs_searchsorted_preferred_bytes(n, m))):
            assert int(out.min()) >= 0 and int(out.max()) <= n
            if order == "sorted":
                assert torch.equal(out, torch.searchsorted(hay, v, out_int32=True))
        assert torch.equal(ops.run_searchsorted(good, v), torch.searchsorted(good, v, out_int32=True))


@pytest.mark.parametrize("n", [1, 2, 100, 16384, 16385, 65536])
@pytest.mark.parametrize("m", [(1 << 16) + 1, 1 << 18, (1 << 18) + 1])
def test_one_needle_a_thread(ops, dev, n, m):
    """The sampled search with one needle a thread, up to 2^18 of them, and
    with four above."""
    g = torch.Generator(device=dev).manual_seed(n)
    hay = torch.randint(I32_MIN, I32_MAX, (n,), generator=g, device=dev, dtype=torch.int32).sort().values
    v = torch.randint(I32_MIN, I32_MAX, (m,), generator=g, device=dev, dtype=torch.int32)
    v[: m // 2] = hay[torch.randint(0, n, (m // 2,), generator=g, device=dev)]
    assert torch.equal(ops.run_searchsorted(hay, v), torch.searchsorted(hay, v, out_int32=True))


@pytest.mark.parametrize("n", [1 << 22, (1 << 22) - 1, (1 << 24) + 1, (1 << 25) + 5])
@pytest.mark.parametrize("kind", ["uniform", "clustered", "two_runs"])
def test_least_workspace_of_long_haystacks(lib, dev, n, kind):
    """The table in the least workspace: wide buckets, searched by samples and
    table together from 2^22 elements on, without the counts above 2^24."""
    g = torch.Generator(device=dev).manual_seed(n)
    hay = torch.randint(I32_MIN, I32_MAX, (n,), generator=g, device=dev, dtype=torch.int32)
    if kind == "clustered":
        hay = (hay.double() / 2**31).pow(9).mul(2**31).int()
    elif kind == "two_runs":
        hay = torch.where(hay < 0, -5, 2**30).int()
        hay[:3] = torch.tensor([I32_MIN, 7, I32_MAX], dtype=torch.int32)
    hay = hay.sort().values
    v = torch.randint(I32_MIN, I32_MAX, (300_001,), generator=g, device=dev, dtype=torch.int32)
    v[:100_000] = hay[torch.randint(0, n, (100_000,), generator=g, device=dev)]
    v[-6:] = torch.tensor([I32_MIN, I32_MAX, -5, -4, 2**30, 2**30 + 1], dtype=torch.int32)
    got = _indexed(lib, hay, v, lib.tcs_searchsorted_workspace_bytes(n))
    assert torch.equal(got, torch.searchsorted(hay, v, out_int32=True))


@pytest.mark.parametrize("n,m", [((1 << 16) + 1, (6 << 20) + 1), ((7 << 14) + 1, (3 << 20) + 1), ((7 << 14) + 16384, (1 << 24) + 16385),
                                 ((1 << 22) + 3, (1 << 20) + 16383), ((1 << 25) + 16386, 700_001)])
@pytest.mark.parametrize("needles", ["ordered", "one", "one_but_a_few", "above", "below", "two_halves"])
def test_tiles_of_one_slice(ops, dev, n, m, needles):
    """Tiles whose needles all lie in one slice, which are answered without the
    sweep, beside tiles that are not, and a last tile of one needle and of
    one less than a tile; in place too."""
    g = torch.Generator(device=dev).manual_seed(n + m)
    hay = torch.randint(I32_MIN, I32_MAX, (n,), generator=g, device=dev, dtype=torch.int32).sort().values
    v = torch.randint(I32_MIN, I32_MAX, (m,), generator=g, device=dev, dtype=torch.int32)
    if needles == "ordered":
        v = v.sort().values
    elif needles in ("one", "one_but_a_few"):
        v[:] = hay[n // 2]
        if needles == "one_but_a_few":
            v[::100_003] = hay[n // 5]
    elif needles == "above":
        hay, v = hay // 2, torch.full_like(v, I32_MAX)
    elif needles == "below":
        hay, v = hay // 2, torch.full_like(v, I32_MIN)
    else:
        v[: m // 2] = hay[n // 3]
    exp = torch.searchsorted(hay, v, out_int32=True)
    assert torch.equal(ops.run_searchsorted(hay, v), exp)
