"""GPU parity at the sizes where a tile, a K range or a store can go wrong: every remainder of the output stores,
nothing written beside C."""
import pytest
import torch

from mxutil import oracle_matmul, randn_operand
from oracle import mx_oracle as O

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-3, torch.bfloat16: 8e-3}


def _guarded(rows, cols, pitch, dtype, dev, fill=7.0):
    """(C, buffer): C is a rows x cols window of the buffer with one guard row above and below and pitch - cols
    guard columns behind every row."""
    buf = torch.full((rows + 2, pitch), fill, dtype=dtype, device=dev)
    return buf[1:rows + 1, :cols], buf


def _check_guarded(c, buf, ref, fill=7.0):
    err = O.rel_fro(c.float().cpu(), ref)
    assert err <= TOL[c.dtype], err
    guard = buf.clone()
    guard[1:c.shape[0] + 1, :c.shape[1]] = fill
    assert (guard == fill).all(), "written beside C"


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("kernel", ["pingpong", "mfma128"])
@pytest.mark.parametrize("tail", range(9))
def test_output_column_remainders(ct, dev, kernel, out_dtype, tail):
    """Column counts of every remainder modulo 8, rows that end inside a tile, output pitches of every alignment, plain
    and accumulating."""
    M, N, K = 259, 256 + tail, 256
    a, b = randn_operand(M, K, O.E4M3, 1000 + tail, dev), randn_operand(N, K, O.E4M3, 1100 + tail, dev)
    ref = oracle_matmul(a, b)
    for pitch in (N, N + 1, (N + 7) // 8 * 8 + 8):
        c, buf = _guarded(M, N, pitch, out_dtype, dev)
        ct.block_scaled_matmul(a.storage, a.scale_t, b.storage.T, b.scale_t.T, C=c, kernel=kernel)
        _check_guarded(c, buf, ref)
        c.fill_(2.0)
        ct.block_scaled_matmul(a.storage, a.scale_t, b.storage.T, b.scale_t.T, C=c, kernel=kernel, accumulate=True)
        _check_guarded(c, buf, ref + 2.0)
