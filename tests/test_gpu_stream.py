"""GPU parity of the weight-streaming kernel (MX_KERNEL_STREAM) at the edges of its splits: row counts around its row
tiles, column counts that end inside a tile or a 64-row group, K ranges that leave waves with unequal shares or a partial
K-quad, plain and packed weight scales."""
import pytest
import torch

from mxutil import oracle_matmul, randn_operand, raw_operand
from oracle import mx_oracle as O
from test_gpu_edges import _check_guarded, _guarded

pytestmark = pytest.mark.gpu
PAIRS = [(O.E4M3, O.E2M1), (O.E4M3, O.E4M3), (O.E5M2, O.E5M2), (O.E5M2, O.E2M1)]


def _scales(ct, b, packed):
    return ct.pack_scales(b.scale_t, operand="b") if packed else b.scale_t.T


@pytest.mark.parametrize("packed", [False, True], ids=["plain", "packed"])
@pytest.mark.parametrize("fa,fb", PAIRS, ids=str)
@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (16, 63, 384), (17, 64, 512), (32, 65, 640), (33, 130, 1024),
                                   (64, 1000, 2176), (65, 259, 1536), (130, 72, 4096), (5, 4096, 2048),
                                   (3, 16448, 512), (33, 8192, 640), (64, 8200, 1024)])
def test_stream_kernel(ct, dev, packed, fa, fb, M, N, K):
    a = randn_operand(M, K, fa, 7000 + M, dev)
    b = raw_operand(N, K, fb, 7100 + N, dev)
    ref = oracle_matmul(a, b)
    for out_dtype, pitch in ((torch.float32, N), (torch.bfloat16, N + 3)):
        c, buf = _guarded(M, N, pitch, out_dtype, dev)
        ct.block_scaled_matmul(a.storage, a.scale_t, b.storage.T, _scales(ct, b, packed), C=c, a_format=a.fmt_kw,
                               b_format=b.fmt_kw, kernel="stream")
        _check_guarded(c, buf, ref)
    c = torch.full((M, N), 3.0, device=dev)
    ct.block_scaled_matmul(a.storage, a.scale_t, b.storage.T, _scales(ct, b, packed), C=c, a_format=a.fmt_kw,
                           b_format=b.fmt_kw, kernel="stream", accumulate=True)
    assert O.rel_fro(c.cpu(), ref + 3.0) <= 1e-3


def test_stream_kernel_ignores_scales_beyond_k(ct, dev):
    """K that ends inside a K-quad: the scale bytes behind it belong to the next row and may be NaN."""
    M, N, K = 4, 64, 640
    a, b = randn_operand(M, K, O.E4M3, 1, dev), randn_operand(N, K, O.E2M1, 2, dev)
    ref = oracle_matmul(a, b)
    pad = torch.full((N + M, 32), 0xFF, dtype=torch.uint8, device=dev)
    pad[:N, :K // 32] = b.scale_t.view(torch.uint8)
    pad[N:, :K // 32] = a.scale_t.view(torch.uint8)
    s = pad.view(torch.float8_e8m0fnu)
    c = ct.block_scaled_matmul(a.storage, s[N:, :K // 32], b.storage.T, s[:N, :K // 32].T, b_format="e2m1", kernel="stream")
    assert O.rel_fro(c.cpu(), ref) <= 1e-3
