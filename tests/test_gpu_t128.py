"""GPU parity of the pipelined 128 x 128 kernel at the edges of its dispatch: grids either side of one workgroup per CU
(its two pipeline depths), K that ends inside a stage or a K-quad, scales read in place or from the native layout, K
split over the workgroups, and a whole batch in one launch with an addend."""
import pytest
import torch

from mxutil import oracle_matmul, randn_operand, raw_operand
from oracle import mx_oracle as O
from test_gpu_edges import _check_guarded, _guarded

pytestmark = pytest.mark.gpu
PAIRS = [(O.E4M3, O.E4M3), (O.E5M2, O.E5M2), (O.E2M1, O.E2M1), (O.E4M3, O.E2M1)]
# The matrix instruction aligns the 128 products of a K-step to the largest of them and drops what falls below its
# accumulator, at most 2^-17 of the largest for each E4M3 product of these operands (raw codes, scales over 15 binades):
# 128 * 2^-17 = 1e-3 of the norm.  A scale, row or K-step taken from the wrong place is an error of the order of 1.
TOL = 1e-3


def _run(ct, a, b, layout, **kw):
    sa = ct.pack_scales(a.scale_t, operand="a") if layout == "packed" else a.scale_t
    sb = ct.pack_scales(b.scale_t, operand="b") if layout in ("packed", "b packed") else b.scale_t.T
    return ct.block_scaled_matmul(a.storage, sa, b.storage.T, sb, a_format=a.fmt_kw, b_format=b.fmt_kw,
                                  kernel="mfma128", **kw)


@pytest.mark.parametrize("layout", ["plain", "b packed", "packed"])
@pytest.mark.parametrize("fa,fb", PAIRS, ids=str)
@pytest.mark.parametrize("M,N,K", [(1, 1, 32), (128, 128, 128), (129, 127, 384), (64, 200, 640), (300, 260, 1184),
                                   (130, 136, 256), (2048, 2176, 256), (2177, 1930, 160)])
def test_t128_kernel(ct, dev, layout, fa, fb, M, N, K):
    a, b = raw_operand(M, K, fa, 100 + M, dev), raw_operand(N, K, fb, 200 + N, dev)
    ref = oracle_matmul(a, b)
    out = _run(ct, a, b, layout, out_dtype=torch.float32)
    assert O.rel_fro(out.cpu(), ref) <= TOL
    c, buf = _guarded(M, N, N + 3, torch.bfloat16, dev)
    _run(ct, a, b, layout, C=c)
    _check_guarded(c, buf, ref)


@pytest.mark.parametrize("fa,fb", PAIRS, ids=str)
@pytest.mark.parametrize("layout", ["plain", "packed"])
@pytest.mark.parametrize("M,N,K", [(70, 130, 2048), (256, 128, 4096 + 128), (33, 65, 6144 + 32)])
def test_t128_splits_k(ct, dev, layout, fa, fb, M, N, K):
    a, b = raw_operand(M, K, fa, 300 + M, dev), raw_operand(N, K, fb, 400 + N, dev)
    out = _run(ct, a, b, layout, out_dtype=torch.float32)
    assert O.rel_fro(out.cpu(), oracle_matmul(a, b)) <= TOL


@pytest.mark.parametrize("fa,fb", [(O.E4M3, O.E4M3), (O.E2M1, O.E2M1)], ids=str)
@pytest.mark.parametrize("bx,by", [(3, 3), (1, 4), (4, 1)])
@pytest.mark.parametrize("M,N,K", [(16, 16, 64), (128, 256, 512), (130, 70, 1056), (40, 24, 4096)])
def test_batch_in_one_launch(ct, dev, fa, fb, bx, by, M, N, K):
    xs = [randn_operand(M, K, fa, 500 + i, dev) for i in range(bx)]
    ys = [randn_operand(N, K, fb, 600 + i, dev) for i in range(by)]
    z = torch.randn((max(bx, by), M, N), generator=torch.Generator().manual_seed(7)).to(dev)
    keep = z.clone()
    stack = lambda v: torch.stack([t.view(torch.uint8) for t in v]).view(v[0].dtype)
    out = ct.mma_scaled(stack([x.storage for x in xs]), stack([x.scale_t for x in xs]),
                        stack([y.storage for y in ys]).transpose(1, 2), stack([y.scale_t for y in ys]).transpose(1, 2),
                        z, x_format=xs[0].fmt_kw, y_format=ys[0].fmt_kw)
    for i in range(max(bx, by)):
        ref = oracle_matmul(xs[i % bx], ys[i % by], z[i].cpu())
        assert O.rel_fro(out[i].cpu(), ref) <= TOL
    assert torch.equal(z, keep)


@pytest.mark.parametrize("split_k", [0, 2])
def test_unpromised_split_without_workspace_runs_whole(ct, dev, split_k):
    """Packed scales and no workspace at all: the bits of the unsplit product, as one call and as a list of one."""
    from cutile_amd import _lib as L
    M, N, K = 130, 200, 8192
    a, b = randn_operand(M, K, O.E4M3, 31, dev), randn_operand(N, K, O.E4M3, 32, dev)
    sa, sb = ct.pack_scales(a.scale_t, operand="a"), ct.pack_scales(b.scale_t, operand="b")
    want = ct.block_scaled_matmul(a.storage, sa, b.storage.T, sb, split_k=1, out_dtype=torch.float32)
    assert O.rel_fro(want.cpu(), oracle_matmul(a, b)) <= TOL
    o = L.MxGemmOpts(struct_size=32, block_size=32, split_k=split_k, a_scale_layout=2, b_scale_layout=2)
    for call in (ct.lib().mx_gemm, lambda *t: ct.lib().mx_gemm_list(1, *t)):
        c = torch.zeros((M, N), device=dev)
        t = (L.desc(a.storage, L.MX_E4M3), L.desc(a.scale_t, L.MX_E8M0), L.desc(b.storage.T, L.MX_E4M3),
             L.desc(b.scale_t.T, L.MX_E8M0), L.desc(c, L.MX_F32))
        t[1].ptr, t[3].ptr = sa.data.data_ptr(), sb.data.data_ptr()
        assert call(*t, o, None, 0, L.stream_ptr(dev)) == 0, L.last_error()
        assert torch.equal(c, want)
