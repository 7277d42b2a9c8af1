"""GPU parity of the mixture-of-experts layer at medium sizes (row tiles, mx_moe_tile.hip): rows around the tiles of 64 and 128,
experts with no row and with several tiles, ids outside the experts, odd K-steps and column counts, K in several ranges,
non-temporal weights, and replays of a captured call."""
import ctypes

import numpy as np
import pytest
import torch

from cutile_amd import _lib as L
from oracle import mx_oracle as O
from test_gpu_moe_forward import _elems, _scale

pytestmark = pytest.mark.gpu

# T, H, F, E, topk, skew: share of the copies that go to expert 0.  Packed scales and rows per expert on average that leave streaming, but
# for the ones that it still takes
STREAMED = [(25, 128, 128, 2, 2, 0.0), (32, 128, 128, 2, 2, 0.0)]
CASES = [(33, 128, 128, 2, 2, 0.0), (54, 256, 128, 4, 2, 0.2), (64, 256, 128, 1, 1, 0.0), (65, 384, 256, 1, 1, 0.0), (128, 128, 640, 1, 1, 0.0),
         (129, 640, 128, 1, 1, 0.0), (100, 256, 384, 4, 2, 0.9), (210, 1152, 128, 16, 4, 0.2),
         # K of the second product in several ranges, the last of them not a whole K-quad
         (60, 128, 5248, 2, 2, 0.4),
         # FP4: tiles of 128 rows (long rows of W, more than 64 rows per expert): one of them, full; two of an expert
         (70, 2176, 128, 1, 1, 0.0), (128, 2176, 256, 1, 1, 0.0), (120, 2304, 128, 2, 2, 0.6),
         # ... three of one expert, none of another, K of the second product in two ranges
         (160, 2176, 2176, 4, 2, 0.95)]
GROUPED = [(129, 2304, 128, 2, 2, 0.6)]   # the first that 256-row tiles take


@pytest.mark.parametrize("w_fmt", [O.E4M3, O.E2M1], ids=str)
@pytest.mark.parametrize("T,H,F,E,topk,skew", STREAMED + CASES + GROUPED)
def test_moe_row_tiles(ct, dev, T, H, F, E, topk, skew, w_fmt):
    rng = np.random.default_rng(T * 7 + F)
    H_out = H + 72                       # not a multiple of a tile
    hq, hs = O.block_quantize(rng.standard_normal((T, H)).astype(np.float32), 32, O.E4M3, "floor")
    w1q, w1s = O.block_quantize((rng.standard_normal((E, 2 * F, H)) * 0.2).astype(np.float32), 32, w_fmt, "floor")
    w2q, w2s = O.block_quantize((rng.standard_normal((E, H_out, F)) * 0.2).astype(np.float32), 32, w_fmt, "floor")
    ids = rng.integers(0, E, (T, topk))
    ids[rng.random((T, topk)) < skew] = 0
    if F == 2176:
        ids[ids == 2] = 3
    lost = rng.random((T, topk)) < (0.1 if E > 1 else 0.0)   # copies that no expert claims
    wts = rng.random((T, topk)).astype(np.float32)
    want = O.moe_forward(hq, hs, w1q, w1s, w2q, w2s, np.where(lost, 0, wts), ids, w_fmt=w_fmt)
    ids = np.where(lost, np.where(rng.random((T, topk)) < 0.5, -1, E + 3), ids)
    s1, s2 = (ct.pack_scales(_scale(s, dev), operand="b") for s in (w1s, w2s))
    for out_dtype, id_dtype in ((torch.float32, torch.int64), (torch.bfloat16, torch.int32)):
        got = ct.cutile_moe_scaled(_elems(hq, O.E4M3, dev), _scale(hs, dev), _elems(w1q, w_fmt, dev), s1,
                                   _elems(w2q, w_fmt, dev), s2, torch.from_numpy(wts).to(dev),
                                   torch.from_numpy(ids).to(dev, id_dtype), out_dtype=out_dtype,
                                   w_format="e2m1" if w_fmt == O.E2M1 else None)
        assert got.shape == (T, H_out) and got.dtype == out_dtype
        # the activation is rounded to bf16 and re-quantised on both sides: a last-bit difference of the first product
        # can move an element by one E4M3 step, as in test_moe_pipeline_matches_oracle
        err = O.rel_fro(got.float().cpu(), want)
        print(f"{T} {H} {F} {E} {topk} {w_fmt} {out_dtype}: {err:.2e}", flush=True)
        assert err < 2e-2


def _random_layer(ct, dev, T, H, F, E, H_out, w_format, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    q = lambda rows, K, fmt: ct.block_quantize(torch.randn((rows, K), generator=g, device=dev) * 0.05, 32, fmt, scale_mode="floor")
    x, xs = q(T, H, torch.float8_e4m3fn)
    fmt = "e2m1" if w_format else torch.float8_e4m3fn
    (w1, s1), (w2, s2) = q(E * 2 * F, H, fmt), q(E * H_out, F, fmt)
    return (x, xs, w1.view(E, 2 * F, -1), s1.view(E, 2 * F, -1), w2.view(E, H_out, -1), s2.view(E, H_out, -1),
            torch.rand((T, 2), generator=g, device=dev), torch.randint(0, E, (T, 2), generator=g, device=dev))


# 96 MB of W and more, rows of whole lines, at most 48 rows per expert: T, H, F, E, H_out.  Both products of each layer; K of the second in
# ranges; even numbers of K-steps, and odd ones (FP4 stages hold two), where FP4 rows have whole lines by their pitch only
ONCE = {None: [(40, 3968, 6528, 2, 7808), (90, 2048, 6656, 4, 4096)],
        "e2m1": [(40, 4096, 12288, 2, 8192), (40, 3968, 12928, 2, 7808), (90, 2048, 12544, 4, 4104)]}
once_pitch = lambda K, w_format: (K // 2 if w_format else K) + 127 & -128   # bytes


def _pitched(w, w_format):
    """The same rows, of whole lines each, with NaN bytes between them."""
    v = w.view(torch.uint8)
    E, rows, row = v.shape
    pitch = once_pitch(2 * row if w_format else row, w_format)
    buf = torch.full((E, rows, pitch), 0xFF, dtype=torch.uint8, device=v.device)
    buf[..., :row] = v
    return buf.view(w.dtype)[..., :row]


@pytest.mark.parametrize("w_format,T,H,F,E,H_out", [(f, *s) for f, layers in ONCE.items() for s in layers])
def test_moe_row_tiles_non_temporal(ct, dev, w_format, T, H, F, E, H_out):
    """Non-temporal weights of both products, and a token whose scales are NaN: it stays alone."""
    x, xs, w1, s1, w2, s2, wt, ids = _random_layer(ct, dev, T, H, F, E, H_out, w_format, 3)
    w1, w2 = _pitched(w1, w_format), _pitched(w2, w_format)
    p1, p2 = ct.pack_scales(s1, operand="b"), ct.pack_scales(s2, operand="b")
    run = lambda scales, a, b: ct.cutile_moe_scaled(x, scales, w1, a, w2, b, wt, ids, out_dtype=torch.float32, w_format=w_format)
    got, plain = run(xs, p1, p2), run(xs, s1, s2)
    # plain scales run another form: the same products in another order (tolerance as above)
    assert ((got - plain).norm() / plain.norm()).item() < 2e-2
    bad = xs.view(torch.uint8).clone()
    bad[7] = 0xFF
    lone = run(bad.view(xs.dtype), p1, p2)
    others = [t for t in range(T) if t != 7]
    assert torch.equal(lone[others], got[others]) and not torch.isfinite(lone[7]).any()


@pytest.mark.parametrize("w_format", [None, "e2m1"])
def test_moe_row_tiles_in_less_room(ct, dev, w_format):
    """A workspace that leaves room for fewer ranges of K than the layer would take, down to one: the same sums in another order."""
    T, H, F, E, H_out, topk = 60, 128, 5248, 2, 200, 2
    x, xs, w1, s1, w2, s2, wt, ids = _random_layer(ct, dev, T, H, F, E, H_out, w_format, 7)
    p1, p2 = ct.pack_scales(s1, operand="b"), ct.pack_scales(s2, operand="b")
    want = ct.cutile_moe_scaled(x, xs, w1, p1, w2, p2, wt, ids, out_dtype=torch.float32, w_format=w_format)
    lib, out = ct.lib(), torch.empty((T, H_out), device=dev)
    o = L.MxGemmOpts(struct_size=32, block_size=32, a_scale_layout=L.MX_SCALE_NATIVE, b_scale_layout=L.MX_SCALE_NATIVE)
    wd = lambda w: L.desc(w.view(torch.uint8), L.MX_E2M1 if w_format else L.MX_E4M3, 2 if w_format else -1)
    packed = [L.MxTensor(ptr=p.data.data_ptr(), dtype=L.MX_E8M0, ndim=3, shape=(E, 1, 1, 0), stride=(1, 1, 1, 0), packed_dim=-1) for p in (p1, p2)]
    args = [L.desc(x.view(torch.uint8), L.MX_E4M3), L.desc(xs.view(torch.uint8), L.MX_E8M0), wd(w1), packed[0], wd(w2), packed[1]]
    ref = [ctypes.byref(a) for a in args]
    need = lib.mx_moe_forward_workspace_bytes(T, topk, ref[2], ref[4], ctypes.byref(o))
    one = T * topk * H_out * 4
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    done = 0
    for ranges_less in range(8):
        out.fill_(float("nan"))
        rc = lib.mx_moe_forward(*ref, wt.data_ptr(), ids.data_ptr(), 1, topk, ctypes.byref(L.desc(out, L.MX_F32)), 1, ctypes.byref(o),
                                ws.data_ptr(), need - ranges_less * one, L.stream_ptr(dev))
        if rc == L.MX_ERR_WORKSPACE:
            break
        assert rc == L.MX_OK, L.last_error()
        # (fp32 sums of 5248 products in another order, 2^-24 for each of their some 16 roundings)
        assert ((out - want).norm() / want.norm()).item() < 1e-6
        done += 1
    assert done > 2


def test_moe_row_tiles_replayed(ct, dev):
    T, H, F, E, H_out = 90, 512, 1024, 4, 520
    x, xs, w1, s1, w2, s2, wt, ids = _random_layer(ct, dev, T, H, F, E, H_out, None, 5)
    p1, p2 = ct.pack_scales(s1, operand="b"), ct.pack_scales(s2, operand="b")
    run = lambda: ct.cutile_moe_scaled(x, xs, w1, p1, w2, p2, wt, ids, out_dtype=torch.float32)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run()
    for i in range(3):
        ids.copy_(torch.randint(-1, E + 1, ids.shape, device=dev))
        want = run()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
