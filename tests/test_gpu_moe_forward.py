"""GPU parity of the whole mixture-of-experts layer (cutile_moe_scaled -> mx_moe_forward) where its splits can go wrong:
one row, rows around the row tiles, experts with no row and with more rows than a pass takes, routed ids outside the
experts, column counts that leave a workgroup partly idle, plain and packed scales, both id widths, and the sizes on
either side of the switch to grouped GEMMs."""
import numpy as np
import pytest
import torch

from oracle import mx_oracle as O
from test_gpu_stream import _spread

pytestmark = pytest.mark.gpu


def _elems(codes, fmt, dev):
    return torch.from_numpy(O.pack_fp4(codes)).to(dev) if fmt == O.E2M1 else torch.from_numpy(codes).to(dev).view(torch.float8_e4m3fn)


def _scale(sc, dev):
    return torch.from_numpy(sc).to(dev).view(torch.float8_e8m0fnu)


# T, H, F, E, topk, skew: share of the copies that go to expert 0
CASES = [(1, 128, 128, 4, 2, 0.0), (17, 256, 128, 8, 1, 0.0), (48, 512, 256, 4, 2, 0.0), (40, 640, 384, 3, 1, 1.0),
         (33, 1024, 256, 16, 4, 0.7), (64, 128, 640, 8, 2, 0.5), (150, 256, 128, 2, 2, 0.9), (700, 256, 256, 16, 4, 0.3),
         # grouped GEMMs on the slots in use, the last round of the second one split along K
         (300, 128, 6144, 3, 2, 0.4)]


@pytest.mark.parametrize("packed", [False, True], ids=["plain", "packed"])
@pytest.mark.parametrize("w_fmt", [O.E4M3, O.E2M1], ids=str)
@pytest.mark.parametrize("T,H,F,E,topk,skew", CASES)
def test_moe_forward(ct, dev, T, H, F, E, topk, skew, w_fmt, packed):
    rng = np.random.default_rng(T * 7 + F)
    H_out = H + 72                       # not a multiple of a tile
    hq, hs = O.block_quantize(rng.standard_normal((T, H)).astype(np.float32), 32, O.E4M3, "floor")
    w1q, w1s = O.block_quantize((rng.standard_normal((E, 2 * F, H)) * 0.2).astype(np.float32), 32, w_fmt, "floor")
    w2q, w2s = O.block_quantize((rng.standard_normal((E, H_out, F)) * 0.2).astype(np.float32), 32, w_fmt, "floor")
    ids = rng.integers(0, E, (T, topk))
    ids[rng.random((T, topk)) < skew] = 0
    lost = rng.random((T, topk)) < 0.1   # copies that no expert claims
    wts = rng.random((T, topk)).astype(np.float32)
    want = O.moe_forward(hq, hs, w1q, w1s, w2q, w2s, np.where(lost, 0, wts), ids, w_fmt=w_fmt)
    ids = np.where(lost, np.where(rng.random((T, topk)) < 0.5, -1, E + 3), ids)
    s1, s2 = _scale(w1s, dev), _scale(w2s, dev)
    if packed:
        s1, s2 = ct.pack_scales(s1, operand="b"), ct.pack_scales(s2, operand="b")
    for out_dtype, id_dtype in ((torch.float32, torch.int64), (torch.bfloat16, torch.int32)):
        got = ct.cutile_moe_scaled(_elems(hq, O.E4M3, dev), _scale(hs, dev), _elems(w1q, w_fmt, dev), s1,
                                   _elems(w2q, w_fmt, dev), s2, torch.from_numpy(wts).to(dev),
                                   torch.from_numpy(ids).to(dev, id_dtype), out_dtype=out_dtype,
                                   w_format="e2m1" if w_fmt == O.E2M1 else None)
        assert got.shape == (T, H_out) and got.dtype == out_dtype
        # the activation is rounded to bf16 and re-quantised on both sides: a last-bit difference of the first product
        # can move an element by one E4M3 step, as in test_moe_pipeline_matches_oracle
        err = O.rel_fro(got.float().cpu(), want)
        print(f"{T} {H} {F} {E} {topk} {w_fmt} packed={packed} {out_dtype}: {err:.2e}", flush=True)
        assert err < 2e-2


def test_moe_forward_scale_rows_that_span_2_gib(ct, dev):
    T, E, topk, H, F = 9, 4, 2, 256, 128
    rng = np.random.default_rng(1)
    q = lambda *shape: ct.block_quantize(torch.from_numpy(rng.standard_normal(shape).astype(np.float32)).to(dev), 32)
    (x, xs), (w1, s1), (w2, s2) = q(T, H), q(E, 2 * F, H), q(E, H, F)
    wide = _spread(xs, (1 << 32) // (T - 1) // 16 * 16, dev)
    wt, ids = torch.rand((T, topk), device=dev), torch.from_numpy(rng.integers(0, E, (T, topk))).to(dev)
    got, want = (ct.cutile_moe_scaled(x, s, w1, s1, w2, s2, wt, ids, out_dtype=torch.float32) for s in (wide, xs))
    # the same products, added up in another order, then rounded to bf16 and E4M3 on the way (tolerance as above)
    assert ((got - want).norm() / want.norm()).item() < 2e-2


@pytest.mark.parametrize("tile_m", [16, 128, 384, 512])
@pytest.mark.parametrize("T,E,topk,skew", [(150, 2, 2, 0.9), (300, 5, 1, 0.2), (1100, 16, 2, 0.0)])
def test_moe_forward_tile_m(ct, dev, T, E, topk, skew, tile_m):
    """Slot tiles other than the default one, beyond the sizes that stream: 128-row kernel, 256-row kernel with wider slots, and
    the single operators where no tiled kernel takes them."""
    H, F = 256, 128
    rng = np.random.default_rng(T)
    hq, hs = O.block_quantize(rng.standard_normal((T, H)).astype(np.float32), 32, O.E4M3, "floor")
    w1q, w1s = O.block_quantize((rng.standard_normal((E, 2 * F, H)) * 0.2).astype(np.float32), 32, O.E4M3, "floor")
    w2q, w2s = O.block_quantize((rng.standard_normal((E, H, F)) * 0.2).astype(np.float32), 32, O.E4M3, "floor")
    ids = rng.integers(0, E, (T, topk))
    ids[rng.random((T, topk)) < skew] = 0
    wts = rng.random((T, topk)).astype(np.float32)
    want = O.moe_forward(hq, hs, w1q, w1s, w2q, w2s, wts, ids)
    got = ct.cutile_moe_scaled(_elems(hq, O.E4M3, dev), _scale(hs, dev), _elems(w1q, O.E4M3, dev), _scale(w1s, dev),
                               _elems(w2q, O.E4M3, dev), _scale(w2s, dev), torch.from_numpy(wts).to(dev),
                               torch.from_numpy(ids).to(dev), tile_m, out_dtype=torch.float32)
    # (tolerance as above)
    assert O.rel_fro(got.cpu(), want) < 2e-2


@pytest.mark.parametrize("T,topk,H_out", [(9, 3, 1027), (5, 5, 2052), (7, 1, 1100), (40, 3, 1284),
                                          # several tokens per workgroup (the last one not full), of one wave, two, and 17 parts
                                          (2049, 1, 260), (2050, 3, 136), (1025, 2, 516), (127, 1, 4100), (122, 2, 4100)])
def test_sum_of_copies(ct, dev, T, topk, H_out):
    """The sum over a token's copies where it is taken apart: an odd number of copies, columns in several parts (more than 1024),
    parts that leave lanes idle, rows that are not whole 16-byte pieces; one copy of every token is dropped, or the only copy of
    every second one."""
    H, F, E = 128, 256, 6
    rng = np.random.default_rng(T + H_out)
    hq, hs = O.block_quantize(rng.standard_normal((T, H)).astype(np.float32), 32, O.E4M3, "floor")
    w1q, w1s = O.block_quantize((rng.standard_normal((E, 2 * F, H)) * 0.2).astype(np.float32), 32, O.E4M3, "floor")
    w2q, w2s = O.block_quantize((rng.standard_normal((E, H_out, F)) * 0.2).astype(np.float32), 32, O.E4M3, "floor")
    ids = np.stack([rng.permutation(E)[:topk] for _ in range(T)])
    wts = rng.random((T, topk)).astype(np.float32)
    lost = np.zeros((T, topk), bool)
    lost[np.arange(T)[:: 2 if topk == 1 else 1], rng.integers(0, topk, T)[:: 2 if topk == 1 else 1]] = True
    want = O.moe_forward(hq, hs, w1q, w1s, w2q, w2s, np.where(lost, 0, wts), ids, w_fmt=O.E4M3)
    for out_dtype in (torch.float32, torch.bfloat16):
        got = ct.cutile_moe_scaled(_elems(hq, O.E4M3, dev), _scale(hs, dev), _elems(w1q, O.E4M3, dev), _scale(w1s, dev),
                                   _elems(w2q, O.E4M3, dev), _scale(w2s, dev), torch.from_numpy(wts).to(dev),
                                   torch.from_numpy(np.where(lost, -1, ids)).to(dev), out_dtype=out_dtype)
        # (the bound of test_moe_forward: the activation is rounded to bf16 and re-quantised on both sides)
        assert O.rel_fro(got.float().cpu(), want) < 2e-2
        if topk == 1:
            assert not got[::2].any()
