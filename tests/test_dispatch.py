"""MX_KERNEL_AUTO never picks a kernel whose launch refuses the operands: few rows of A with weights whose rows overlap (a
broadcast or a sliding window) or with scale rows that span 2 GiB.  On the host: where there is no device a dispatched
launch ends in MX_ERR_LAUNCH, a refusal in MX_ERR_LAYOUT."""
import ctypes

import pytest
import torch

import cutile_amd
from cutile_amd import _lib as L
from test_cabi import _desc

# the descriptors name host memory, or extents that are not there
pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="would launch kernels on host pointers")

WIDE = 1 << 26   # 32 rows of this pitch are 2 GiB


def _gemm(M, N, K, fmt, b_pitch=None, as_pitch=None, bs_pitch=None, kernel=L.MX_KERNEL_AUTO):
    lib = cutile_amd.lib()
    buf = torch.zeros(1 << 22, dtype=torch.uint8)
    p = (buf.data_ptr() + 255) // 256 * 256
    packed = fmt == L.MX_E2M1
    row = K // 2 if packed else K
    A = _desc(p, L.MX_E4M3, (M, K), (K, 1))
    As = _desc(p, L.MX_E8M0, (M, K // 32), (K // 32 if as_pitch is None else as_pitch, 1))
    B = _desc(p, fmt, (K, N), (1, row if b_pitch is None else b_pitch), 0 if packed else -1)
    Bs = _desc(p, L.MX_E8M0, (K // 32, N), (1, K // 32 if bs_pitch is None else bs_pitch))
    C = _desc(p, L.MX_F32, (M, N), (N, 1))
    o = L.MxGemmOpts(struct_size=32, kernel=kernel, block_size=32)
    rc = lib.mx_gemm(*(ctypes.byref(t) for t in (A, As, B, Bs, C)), ctypes.byref(o), p, 1 << 21, None)
    return rc, L.last_error()


@pytest.mark.parametrize("fmt", [L.MX_E4M3, L.MX_E2M1])
@pytest.mark.parametrize("M", [1, 8, 33, 64, 65])
@pytest.mark.parametrize("K", [512, 640, 8704])
def test_auto_launches_something(fmt, M, K):
    for kw in ({}, {"b_pitch": 0}, {"b_pitch": 16}, {"b_pitch": 0, "bs_pitch": 0}, {"as_pitch": WIDE}, {"as_pitch": 1 << 31},
               {"as_pitch": WIDE + 4, "b_pitch": 16}):
        rc, message = _gemm(M, 256, K, fmt, **kw)
        assert rc == L.MX_ERR_LAUNCH, (kw, rc, message)
    # the scale rows of FP4 weights for the decode kernel are held to 2 GiB, other kernels re-lay them
    if not (fmt == L.MX_E2M1 and M <= 32 and K == 512):
        rc, message = _gemm(M, 256, K, fmt, bs_pitch=WIDE)
        assert rc == L.MX_ERR_LAUNCH, (rc, message)


def test_a_forced_streaming_kernel_says_what_it_cannot_take():
    rc, message = _gemm(8, 256, 512, L.MX_E4M3, bs_pitch=WIDE, kernel=9)
    assert rc == L.MX_ERR_LAYOUT and "B_scale spans 2 GiB" in message
    rc, message = _gemm(8, 256, 512, L.MX_E4M3, b_pitch=520, kernel=9)
    assert rc == L.MX_ERR_LAYOUT and "16-byte aligned rows" in message
