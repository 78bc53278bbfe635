"""Scratch sized for the largest call serves every smaller one: the C ABI's
size queries do not fall as sizes grow (host only), or what they return for
a larger size is taken for a smaller one (GPU)."""
import ctypes
import os

import pytest
import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(REPO, "pytorch-tcuscan_amd", "libtcuscan_hip.so")


@pytest.fixture(scope="module")
def lib():
    lib = ctypes.CDLL(LIB)
    for f in (lib.tcs_sort_scratch_bytes, lib.tcs_topk_scratch_bytes, lib.tcs_topk_workspace_bytes,
              lib.tcs_sort_workspace_bytes):
        f.restype = ctypes.c_size_t
    lib.tcs_sort_scratch_bytes.argtypes = lib.tcs_sort_workspace_bytes.argtypes = [ctypes.c_int64, ctypes.c_int]
    lib.tcs_topk_scratch_bytes.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    lib.tcs_topk_workspace_bytes.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    return lib


def test_sort_scratch_does_not_fall(lib):
    """At the sizes where the chunks, their rounding or the tiles change."""
    sizes = sorted({max(0, b + d) for b in (8192, 2048 * 49, 1 << 17, 1 << 19, 2048 * 512, 3 << 20, 6 << 20, 1 << 23,
                                            1 << 24, 1 << 28, 1 << 30) for d in (-513, -1, 0, 1, 2, 513, 4097, 70_000)})
    for code in range(7):
        got = [lib.tcs_sort_scratch_bytes(n, code) for n in sizes]
        assert got == sorted(got), code


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.int32], ids=str)
def test_sort_in_the_scratch_of_a_larger_one(lib, dev, dtype):
    """2^20 + 1 keys take fewer chunks than 2^20: their scratch serves both."""
    code = {torch.float16: 0, torch.int32: 5}[dtype]
    top = (1 << 20) + 1
    scratch = torch.empty(lib.tcs_sort_scratch_bytes(top, code), dtype=torch.uint8, device=dev)
    ws = torch.zeros(lib.tcs_sort_workspace_bytes(top, code), dtype=torch.uint8, device=dev)
    g = torch.Generator(device=dev).manual_seed(1)
    for n in (top, 1 << 20, 300_001, 9000):
        x = torch.randint(-30000, 30000, (n,), generator=g, device=dev).to(dtype)
        y, idx = torch.empty_like(x), torch.empty(n, dtype=torch.int32, device=dev)
        assert lib.tcs_sort(ctypes.c_void_p(x.data_ptr()), code, None, ctypes.c_void_p(y.data_ptr()),
                            ctypes.c_void_p(idx.data_ptr()), ctypes.c_int64(n), 0, ctypes.c_void_p(ws.data_ptr()),
                            ctypes.c_size_t(ws.numel()), ctypes.c_void_p(scratch.data_ptr()),
                            ctypes.c_size_t(scratch.numel()),
                            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        ref = torch.sort(x, stable=True)
        assert torch.equal(y, ref.values) and torch.equal(idx.long(), ref.indices)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.int8, torch.int32], ids=str)
def test_topk_in_the_scratch_of_a_larger_one(lib, dev, dtype):
    """The scratch and workspace of the largest of several calls serve them
    all, whichever way each size takes by itself."""
    code = {torch.float16: 0, torch.int8: 3, torch.int32: 5}[dtype]
    top, kmax = (1 << 23) + 5, 3000
    scratch = torch.full((lib.tcs_topk_scratch_bytes(top, kmax, code),), -1, dtype=torch.int8, device=dev)
    ns = (top, 4_300_001, 1 << 21, 1 << 18, 5000)
    ws = torch.zeros(max(lib.tcs_topk_workspace_bytes(n, kmax, code) for n in ns), dtype=torch.uint8, device=dev)
    g = torch.Generator(device=dev).manual_seed(2)
    for n in ns:
        x = torch.randint(-128 if code == 3 else -30000, 128 if code == 3 else 30000, (n,), generator=g,
                          device=dev).to(dtype)
        ref = torch.sort(x, descending=True, stable=True)
        for k in (1, 300, kmax):
            y, idx = torch.empty(k, dtype=dtype, device=dev), torch.empty(k, dtype=torch.int32, device=dev)
            assert lib.tcs_topk(ctypes.c_void_p(x.data_ptr()), code, ctypes.c_int64(n), ctypes.c_int64(k), 1,
                                ctypes.c_void_p(y.data_ptr()), ctypes.c_void_p(idx.data_ptr()),
                                ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(ws.numel()),
                                ctypes.c_void_p(scratch.data_ptr()), ctypes.c_size_t(scratch.numel()),
                                ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
            assert torch.equal(y, ref.values[:k]) and torch.equal(idx.long(), ref.indices[:k]), (n, k)
