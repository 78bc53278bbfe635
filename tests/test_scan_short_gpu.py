"""Which plain scans run as one 4096-element tile per workgroup (GPU): told by
the descriptors that a scan leaves in a zeroed workspace, one per tile."""
import ctypes
import os

import pytest
import torch

import oracle
from _util import assert_exact, to_np, uniform_pm1

pytestmark = pytest.mark.gpu

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(REPO, "pytorch-tcuscan_amd", "libtcuscan_hip.so")
HEADER_BYTES = 18 * 256
SHORT_TILE, SHORT_MAX = 4096, 3 << 20


@pytest.fixture(scope="module")
def lib():
    lib = ctypes.CDLL(LIB)
    lib.tcs_scan_workspace_bytes.restype = ctypes.c_size_t
    lib.tcs_scan_workspace_bytes.argtypes = [ctypes.c_int64, ctypes.c_int, ctypes.c_int]
    lib.tcs_scan_method.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_int64, ctypes.c_int,
                                    ctypes.c_int, ctypes.c_double, ctypes.c_int, ctypes.c_int, ctypes.c_void_p,
                                    ctypes.c_size_t, ctypes.c_void_p]
    return lib


def _scan_tiles(lib, x, nbytes, method=0):
    """Scans x (fp16) in a zeroed workspace of nbytes; the number of tiles
    that published a descriptor (16 bytes each)."""
    ws = torch.zeros(nbytes // 8, dtype=torch.int64, device=x.device)
    y = torch.empty(x.numel(), device=x.device)
    assert lib.tcs_scan_method(x.data_ptr(), 0, y.data_ptr(), x.numel(), 128, 0, 0.0, method, 0, ws.data_ptr(),
                               nbytes, torch.cuda.current_stream().cuda_stream) == 0
    assert_exact(to_np(y), oracle.scan(to_np(x)))
    return int((ws[HEADER_BYTES // 8:].view(-1, 2) != 0).any(1).sum())


@pytest.mark.parametrize("n", [4097, 65536, 65537, 1 << 20, SHORT_MAX])
def test_short_scan_with_the_queried_workspace(lib, dev, n):
    x = uniform_pm1(n, torch.float16, n).to(dev)
    need = lib.tcs_scan_workspace_bytes(n, 128, 0)
    assert _scan_tiles(lib, x, need) == -(-n // SHORT_TILE)


@pytest.mark.parametrize("n", [SHORT_MAX + 1, SHORT_MAX + 70_001])
def test_larger_scans_keep_their_tiles(lib, dev, n):
    x = uniform_pm1(n, torch.float16, n).to(dev)
    need = lib.tcs_scan_workspace_bytes(n, 128, 0)
    assert need >= lib.tcs_scan_workspace_bytes(SHORT_MAX, 128, 0)
    assert _scan_tiles(lib, x, need) < -(-n // SHORT_TILE)


@pytest.mark.parametrize("n", [65_537, 1 << 20])
def test_a_named_method_is_not_the_short_scan(lib, dev, n):
    """TCS_METHOD_DPP (1) and TCS_METHOD_MFMA (2) run the pipelined scan with
    that local scan, whatever the workspace holds."""
    x = uniform_pm1(n, torch.float16, n).to(dev)
    need = lib.tcs_scan_workspace_bytes(n, 128, 0)
    for method in (1, 2):
        assert _scan_tiles(lib, x, need, method) < -(-n // SHORT_TILE)
