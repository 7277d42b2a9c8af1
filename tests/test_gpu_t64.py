"""The 128 x 128 kernel's 64 x 64 tiles: either side of the numbers of workgroups at which the tile and the depth of its
pipeline change, ragged edges, every place of a wave's rows in a 64-row scale group, addends, and splits along K."""
import pytest
import torch

from mxutil import oracle_matmul, raw_operand
from oracle import mx_oracle as O
from test_gpu_edges import _check_guarded, _guarded

pytestmark = pytest.mark.gpu
PAIRS = [(O.E4M3, O.E4M3), (O.E5M2, O.E5M2), (O.E2M1, O.E2M1), (O.E4M3, O.E2M1)]
TOL = 1e-3   # of the norm: 128 products of a K-step, each cut at most 2^-17 below the largest


def _run(ct, a, b, layout, **kw):
    sa = ct.pack_scales(a.scale_t, operand="a") if layout == "packed" else a.scale_t
    sb = ct.pack_scales(b.scale_t, operand="b") if layout in ("packed", "b packed") else b.scale_t.T
    return ct.block_scaled_matmul(a.storage, sa, b.storage.T, sb, a_format=a.fmt_kw, b_format=b.fmt_kw, kernel="mfma128", **kw)


# 64-tiles: 1, 4 (one row and column over), 15, 256, 272, 506; then 529 (128 x 128 tiles, one per CU); K of one block, inside
# a stage, of more stages than are in flight
@pytest.mark.parametrize("M,N,K", [(64, 64, 32), (65, 65, 640), (130, 316, 1184), (1024, 1024, 256), (1000, 1088, 96), (1400, 1472, 384),
                                   (1472, 1472, 640)])
@pytest.mark.parametrize("fa,fb", PAIRS, ids=str)
@pytest.mark.parametrize("layout", ["plain", "b packed", "packed"])
def test_tiles(ct, dev, layout, fa, fb, M, N, K):
    a, b = raw_operand(M, K, fa, 2100 + M, dev), raw_operand(N, K, fb, 2200 + N, dev)
    ref = oracle_matmul(a, b)
    c, buf = _guarded(M, N, N + 4, torch.float32, dev)
    _run(ct, a, b, layout, C=c)
    assert O.rel_fro(c.cpu(), ref) <= TOL
    _run(ct, a, b, layout, C=c, accumulate=True)
    assert O.rel_fro(c.cpu(), 2 * ref) <= TOL
    buf[1:M + 1, :N] = 7
    assert (buf == 7).all(), "written beside C"
    c, buf = _guarded(M, N, N + 3, torch.bfloat16, dev)
    _run(ct, a, b, layout, C=c)
    _check_guarded(c, buf, ref)


@pytest.mark.parametrize("fa,fb", PAIRS, ids=str)
@pytest.mark.parametrize("M,N,K,split_k", [(300, 300, 8192, 0), (70, 1024, 4096, 0), (100, 2048, 6144 + 32, 0), (64, 64, 1024, 2), (520, 512, 2048, 4)])
def test_splits(ct, dev, fa, fb, M, N, K, split_k):
    a, b = raw_operand(M, K, fa, 2300 + M, dev), raw_operand(N, K, fb, 2400 + N, dev)
    out = _run(ct, a, b, "plain", out_dtype=torch.float32, split_k=split_k)
    assert O.rel_fro(out.cpu(), oracle_matmul(a, b)) <= TOL


@pytest.mark.parametrize("fmt", [O.E4M3, O.E5M2, O.E2M1])
@pytest.mark.parametrize("n,M,N,K", [(6, 200, 328, 992), (3, 17, 33, 128), (5, 64, 130, 256), (40, 200, 200, 160)])
def test_batches_with_an_addend(ct, dev, fmt, n, M, N, K):
    xs, ys = [raw_operand(M, K, fmt, 70 + i, dev) for i in range(n)], [raw_operand(N, K, fmt, 180 + i, dev) for i in range(n)]
    stack = lambda v: torch.stack([t.view(torch.uint8) for t in v]).view(v[0].dtype)
    z = torch.randn((n, M, N), generator=torch.Generator().manual_seed(3)).to(dev)
    keep = z.clone()
    out = ct.mma_scaled(stack([x.storage for x in xs]), stack([x.scale_t for x in xs]), stack([y.storage for y in ys]).transpose(1, 2),
                        stack([y.scale_t for y in ys]).transpose(1, 2), z, x_format=xs[0].fmt_kw, y_format=ys[0].fmt_kw)
    assert torch.equal(z, keep)
    for i in range(n):
        assert O.rel_fro((out[i] - z[i]).cpu(), oracle_matmul(xs[i], ys[i])) <= TOL
