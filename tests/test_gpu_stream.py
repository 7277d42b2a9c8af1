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


def _spread(rows, pitch, dev):
    """`rows` at `pitch` bytes from one another, in a buffer of their own."""
    n, k = rows.shape
    buf = torch.empty((n - 1) * pitch + k, dtype=torch.uint8, device=dev)
    out = buf.as_strided((n, k), (pitch, 1))
    out.copy_(rows.view(torch.uint8))
    return out.view(rows.dtype)


@pytest.mark.parametrize("M", [8, 64, 65])
@pytest.mark.parametrize("fb,pitch", [(O.E4M3, 0), (O.E4M3, 16), (O.E2M1, 0), (O.E2M1, 16)])
def test_rows_of_the_weights_may_overlap(ct, dev, M, fb, pitch):
    """B as one broadcast row, or as windows that slide over one buffer, and its scales broadcast."""
    N, K = 200, 1152
    row = K // 2 if fb == O.E2M1 else K
    flat = raw_operand(1, K + 32 * N, fb, 11, dev)   # (a source of valid element bytes)
    a, s = randn_operand(M, K, O.E4M3, 12, dev), raw_operand(1, K, fb, 13, dev).scale_t
    w = flat.storage.view(-1).as_strided((N, row), (pitch, 1))
    codes = torch.from_numpy(flat.storage_np).view(-1).as_strided((N, row), (pitch, 1)).contiguous().numpy()
    if fb == O.E2M1:
        codes = O.unpack_fp4(codes)
    scales = s.view(torch.uint8).cpu().expand(N, K // 32).contiguous().numpy()
    ref = O.reference_matmul(a.codes, a.scales, codes.T.copy(), scales.T.copy(), O.E4M3, fb, 32)
    for bs in (s.expand(N, K // 32).T, s.expand(N, K // 32).contiguous().T):
        c = ct.block_scaled_matmul(a.storage, a.scale_t, w.T, bs, b_format="e2m1" if fb == O.E2M1 else None,
                                   out_dtype=torch.float32)
        assert O.rel_fro(c.cpu(), ref) <= 1e-3


@pytest.mark.parametrize("M,K,fb,side", [(8, 640, O.E4M3, "b"), (33, 640, O.E2M1, "b"), (64, 1024, O.E4M3, "a"),
                                         (8, 8704, O.E2M1, "a")])
def test_scale_rows_that_span_2_gib(ct, dev, M, K, fb, side):
    """Beyond the streaming kernel's 32-bit offsets: another kernel takes the problem."""
    N = 256
    a, b = randn_operand(M, K, O.E4M3, 21, dev), randn_operand(N, K, fb, 22, dev)
    sa, sb = a.scale_t, b.scale_t
    if side == "a":
        sa = _spread(sa, (1 << 31) // M // 16 * 16 + 16, dev)
    else:
        sb = _spread(sb, (1 << 31) // N // 16 * 16 + 16, dev)
    c = ct.block_scaled_matmul(a.storage, sa, b.storage.T, sb.T, b_format=b.fmt_kw, out_dtype=torch.float32)
    assert O.rel_fro(c.cpu(), oracle_matmul(a, b)) <= 1e-3
