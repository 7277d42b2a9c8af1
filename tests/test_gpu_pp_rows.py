"""Ping-pong kernel on tiles of 192 rows: shapes for which its rounds are the better filled ones, against the same kernel on
tiles of 256 rows.  Every output is the same sum in the same order, so the bits are the same."""
import pytest
import torch

from mxutil import raw_operand
from oracle import mx_oracle as O
from test_gpu_edges import _guarded

pytestmark = pytest.mark.gpu


# whole tiles; one row and one column more and less; walks of several tiles; K inside a stage, inside a K-quad, one stage
@pytest.mark.parametrize("M,N,K", [(3072, 4096, 512), (1531, 14336, 512), (1537, 14300, 1024), (1343, 14085, 512), (1900, 5000, 992),
                                   (1921, 4999, 1280), (3071, 4090, 128), (3000, 4096, 96)])
@pytest.mark.parametrize("fa,fb", [(O.E4M3, O.E4M3), (O.E5M2, O.E5M2), (O.E2M1, O.E2M1), (O.E4M3, O.E2M1)], ids=str)
def test_192_row_tiles(ct, dev, fa, fb, M, N, K):
    a, b = raw_operand(M, K, fa, M, dev), raw_operand(N, K, fb, N, dev)
    run = lambda **kw: ct.block_scaled_matmul(a.storage, a.scale_t, b.storage.T, b.scale_t.T, a_format=a.fmt_kw, b_format=b.fmt_kw, **kw)
    for dt in (torch.float32, torch.bfloat16):
        assert torch.equal(run(out_dtype=dt), run(out_dtype=dt, kernel="pingpong"))
    # rows of C that are not 16-byte aligned, inside a guarded buffer; then accumulated into
    outs = []
    for kernel in ("auto", "pingpong"):
        c, buf = _guarded(M, N, N + 3, torch.float32, dev)
        run(C=c, kernel=kernel)
        run(C=c, kernel=kernel, accumulate=True)
        outs.append(buf)
    assert torch.equal(outs[0].view(torch.int32), outs[1].view(torch.int32))
