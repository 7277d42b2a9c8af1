"""Scales that the 128 x 128 kernel reads where they are although their rows start at any byte: the same bits as with the
re-laid ones, and nothing of the bytes between, before and behind the rows (they hold NaN scales) in the result."""
import pytest
import torch

from mxutil import oracle_matmul, raw_operand
from oracle import mx_oracle as O

pytestmark = pytest.mark.gpu
PAIRS = [(O.E4M3, O.E4M3), (O.E5M2, O.E5M2), (O.E2M1, O.E2M1), (O.E4M3, O.E2M1)]
TOL = 1e-3   # of the norm: 128 products of a K-step, each cut at most 2^-17 below the largest


def _placed(scale, offset, pad):
    """`scale` as a view whose rows lie `pad` bytes apart, the first `offset` bytes into a buffer of NaN scales."""
    rows, kb = scale.shape
    buf = torch.full((offset + rows * (kb + pad) + 7,), 0xFF, dtype=torch.uint8, device=scale.device)
    v = buf[offset:offset + rows * (kb + pad)].view(rows, kb + pad)[:, :kb]
    v.copy_(scale.view(torch.uint8))
    return v.view(scale.dtype) if pad == 0 else torch.as_strided(buf.view(scale.dtype), (rows, kb), (kb + pad, 1), offset)


@pytest.mark.parametrize("fa,fb", PAIRS, ids=str)
# K inside one K-step, inside a K-quad, one block beyond a quad, many quads; both pipeline depths; K split
@pytest.mark.parametrize("M,N,K", [(1, 1, 32), (130, 70, 96), (129, 257, 544), (200, 328, 992), (64, 136, 2080), (2177, 1930, 160)])
@pytest.mark.parametrize("oa,pa,ob,pb", [(0, 0, 0, 0), (1, 0, 3, 5), (2, 3, 1, 1), (0, 4, 2, 0)])
def test_rows_at_any_byte(ct, dev, fa, fb, M, N, K, oa, pa, ob, pb):
    a, b = raw_operand(M, K, fa, 1100 + M, dev), raw_operand(N, K, fb, 1200 + N, dev)
    run = lambda sa, sb, **kw: ct.block_scaled_matmul(a.storage, sa, b.storage.T, sb, a_format=a.fmt_kw, b_format=b.fmt_kw,
                                                      kernel="mfma128", out_dtype=torch.float32, **kw)
    sa, sb = _placed(a.scale_t, oa, pa), _placed(b.scale_t, ob, pb)
    out = run(sa, sb.T)
    want = run(ct.pack_scales(a.scale_t, operand="a"), ct.pack_scales(b.scale_t, operand="b"))
    assert torch.equal(out, want) or O.rel_fro(out.cpu(), want.cpu()) <= 1e-6   # (K split elsewhere: another order of sums)
    assert O.rel_fro(out.cpu(), oracle_matmul(a, b)) <= TOL


@pytest.mark.parametrize("fa,fb", PAIRS, ids=str)
@pytest.mark.parametrize("K", [4000, 4384])   # the last that is read in place, the first that is re-laid (288 tiles)
def test_either_side_of_the_line(ct, dev, fa, fb, K):
    M, N = 2177, 1930
    a, b = raw_operand(M, K, fa, 1300 + K, dev), raw_operand(N, K, fb, 1400 + K, dev)
    run = lambda sa, sb: ct.block_scaled_matmul(a.storage, sa, b.storage.T, sb, a_format=a.fmt_kw, b_format=b.fmt_kw,
                                                kernel="mfma128", out_dtype=torch.float32)
    out = run(_placed(a.scale_t, 1, 0), _placed(b.scale_t, 3, 5).T)
    assert torch.equal(out, run(ct.pack_scales(a.scale_t, operand="a"), ct.pack_scales(b.scale_t, operand="b")))


@pytest.mark.parametrize("fa,fb", PAIRS, ids=str)
@pytest.mark.parametrize("K", [4096, 4128, 5120, 5152])   # the last whose requests are spread over a stage, the first whose are not
def test_either_side_of_long_k_on_64_x_64_tiles(ct, dev, fa, fb, K):
    M, N = 130, 70
    a, b = raw_operand(M, K, fa, 1500 + K, dev), raw_operand(N, K, fb, 1600 + K, dev)
    run = lambda sa, sb: ct.block_scaled_matmul(a.storage, sa, b.storage.T, sb, a_format=a.fmt_kw, b_format=b.fmt_kw,
                                                kernel="mfma128", out_dtype=torch.float32, split_k=1)
    out = run(_placed(a.scale_t, 1, 0), _placed(b.scale_t, 3, 5).T)
    assert torch.equal(out, run(ct.pack_scales(a.scale_t, operand="a"), ct.pack_scales(b.scale_t, operand="b")))
    assert O.rel_fro(out.cpu(), oracle_matmul(a, b)) <= TOL


@pytest.mark.parametrize("fmt", [O.E4M3, O.E2M1])
def test_in_lists_and_batches(ct, dev, fmt):
    shapes = [(96, 200, 96), (128, 128, 512), (300, 64, 1056), (33, 130, 32), (257, 129, 992)]
    ops = [(raw_operand(M, K, fmt, 10 + i, dev), raw_operand(N, K, fmt, 50 + i, dev)) for i, (M, N, K) in enumerate(shapes)]
    view = (lambda t: t.view(torch.float4_e2m1fn_x2)) if fmt == O.E2M1 else (lambda t: t)
    out = ct.grouped_block_scaled_matmul([view(a.storage) for a, _ in ops], [_placed(a.scale_t, 1, 0) for a, _ in ops],
                                         [view(b.storage).T for _, b in ops], [_placed(b.scale_t, 3, 2).T for _, b in ops],
                                         out_dtype=torch.float32)
    for o, (a, b) in zip(out, ops):
        assert O.rel_fro(o.cpu(), oracle_matmul(a, b)) <= TOL
    M, N, K, n = 70, 136, 992, 3
    xs, ys = [raw_operand(M, K, fmt, 70 + i, dev) for i in range(n)], [raw_operand(N, K, fmt, 80 + i, dev) for i in range(n)]
    stack = lambda v: torch.stack([t.view(torch.uint8) for t in v]).view(v[0].dtype)
    z = torch.zeros((n, M, N), device=dev)
    # the scales of a batch entry start 31 M (31 N) bytes behind the last one's
    out = ct.mma_scaled(stack([x.storage for x in xs]), stack([x.scale_t for x in xs]), stack([y.storage for y in ys]).transpose(1, 2),
                        stack([y.scale_t for y in ys]).transpose(1, 2), z, x_format=xs[0].fmt_kw, y_format=ys[0].fmt_kw)
    for i in range(n):
        assert O.rel_fro(out[i].cpu(), oracle_matmul(xs[i], ys[i])) <= TOL
