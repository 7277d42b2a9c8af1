"""Weights of 96 MB and more, which the streaming, decode and mixture-of-experts kernels read non-temporally.  The loads' policy
is all that differs from the instances that the other tests compare with the oracle, so the bits are those of the same weights
at an address or a pitch that keeps to the plain policy; sampled outputs are compared with float64 as well."""
import pytest
import torch

from oracle import mx_oracle as O

pytestmark = pytest.mark.gpu

STREAM_K, STREAM_N = 7936, {"e4m3": 12687, "e5m2": 12687, "e2m1": 25371}   # K-quads and 64-row groups that are not whole
DECODE_NK = [(24592, 8192), (49168, 4096)]                                 # both lengths of a K-slice
MOE_H, MOE_F, MOE_OUT, MOE_TOPK, MOE_T, MOE_E = 1536, 2048, 3080, 2, (60, 150), {"e4m3": 16, "e2m1": 32}
ELEM = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
FP4 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _bytes(shape, fmt, seed, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    b = torch.randint(0, 256, shape, dtype=torch.uint8, device=dev, generator=g)
    if fmt == "e4m3":
        b[(b & 0x7F) == 0x7F] = 0x3C
    elif fmt == "e5m2":
        b[(b & 0x7C) == 0x7C] = 0x3C
    return b


def _scales(shape, seed, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.randint(115, 130, shape, dtype=torch.uint8, device=dev, generator=g).view(torch.float8_e8m0fnu)


def _elem(b, fmt):
    return b if fmt == "e2m1" else b.view(ELEM[fmt])


def _moved(b, offset=0, pad=0):
    """The rows of b at `offset` bytes into a buffer of their own, `pad` bytes between them."""
    rows, row = b.numel() // b.shape[-1], b.shape[-1]
    buf = torch.empty(rows * (row + pad) + offset, dtype=torch.uint8, device=b.device)
    out = buf[offset:].as_strided(b.shape, (*(s // row * (row + pad) for s in b.stride()[:-1]), 1), buf.storage_offset() + offset)
    return out.copy_(b)


def _float(b, s, fmt):
    """float64 values of rows of codes and their scales"""
    if fmt == "e2m1":
        lut = torch.tensor(FP4 + [-v for v in FP4], dtype=torch.float64, device=b.device)
        v = torch.stack((lut[(b & 15).long()], lut[(b >> 4).long()]), -1).flatten(-2)
    else:
        v = b.view(ELEM[fmt]).double()
    return v * torch.exp2(s.view(torch.uint8).double() - 127).repeat_interleave(32, -1)


@pytest.mark.parametrize("packed", [False, True], ids=["plain", "packed"])
@pytest.mark.parametrize("M", [7, 32, 50])   # one row tile of 16, 32 and 64 rows
@pytest.mark.parametrize("fx,fw", [("e4m3", "e4m3"), ("e4m3", "e2m1"), ("e5m2", "e5m2"), ("e5m2", "e2m1")])
def test_streamed_weights(ct, dev, fx, fw, M, packed):
    N, K = STREAM_N[fw], STREAM_K
    x, xs = _bytes((M, K), fx, 1, dev), _scales((M, K // 32), 2, dev)
    w, ws = _bytes((N, K // 2 if fw == "e2m1" else K), fw, 3, dev), _scales((N, K // 32), 4, dev)
    scales = ct.pack_scales(ws, operand="b") if packed else ws.T
    run = lambda b: ct.block_scaled_matmul(_elem(x, fx), xs, _elem(b, fw).T, scales, a_format=fx, b_format=fw, kernel="stream",
                                           out_dtype=torch.float32)
    c = run(w)
    assert w.data_ptr() % 128 == 0 and torch.equal(c.view(torch.int32), run(_moved(w, 16)).view(torch.int32))
    cols = torch.cat((torch.arange(0, N, 997, device=dev), torch.arange(N - 70, N, device=dev)))
    assert O.rel_fro(c[:, cols].double().cpu(), (_float(x, xs, fx) @ _float(w[cols], ws[cols], fw).T).cpu()) <= 1e-3


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("M", [32, 40])      # one slab of rows and two
@pytest.mark.parametrize("N,K", DECODE_NK)
def test_decode_kernel(ct, dev, N, K, M, out_dtype):
    x, xs = _bytes((M, K), "e4m3", 1, dev), _scales((M, K // 32), 2, dev)
    w, ws = _bytes((N, K // 2), "e2m1", 3, dev), _scales((N, K // 32), 4, dev)
    run = lambda b: ct.block_scaled_matmul(_elem(x, "e4m3"), xs, b.T, ws.T, b_format="e2m1", kernel="decode", out_dtype=out_dtype)
    c = run(w)
    assert torch.equal(c.view(torch.uint8), run(_moved(w, 0, 16)).view(torch.uint8))
    cols = torch.cat((torch.arange(0, N, 997, device=dev), torch.arange(N - 16, N, device=dev)))
    err = O.rel_fro(c[:, cols].double().cpu(), (_float(x, xs, "e4m3") @ _float(w[cols], ws[cols], "e2m1").T).cpu())
    assert err <= (1e-3 if out_dtype == torch.float32 else 8e-3)


@pytest.mark.parametrize("packed", [False, True], ids=["plain", "packed"])
@pytest.mark.parametrize("T", MOE_T)         # passes of 16 and of 32 rows
@pytest.mark.parametrize("fw", ["e4m3", "e2m1"])
def test_moe_layer(ct, dev, fw, T, packed):
    E, k = MOE_E[fw], (lambda n: n // 2 if fw == "e2m1" else n)
    g = torch.Generator(device=dev).manual_seed(T)
    x, xs = ct.block_quantize(torch.randn((T, MOE_H), device=dev, generator=g), 32, scale_mode="floor")
    w1, w2 = _bytes((E, 2 * MOE_F, k(MOE_H)), fw, 3, dev), _bytes((E, MOE_OUT, k(MOE_F)), fw, 4, dev)
    s = [(_scales((E, n, K // 32), 5, dev).view(torch.uint8) - 8).view(torch.float8_e8m0fnu)
         for n, K in ((2 * MOE_F, MOE_H), (MOE_OUT, MOE_F))]
    if packed:
        s = [ct.pack_scales(t, operand="b") for t in s]
    ids = torch.randint(0, E, (T, MOE_TOPK), device=dev, generator=g)
    ids[:40, 0] = 1                          # more rows than a pass takes
    wt = torch.rand((T, MOE_TOPK), device=dev, generator=g)
    run = lambda a, b: ct.cutile_moe_scaled(x, xs, _elem(a, fw), s[0], _elem(b, fw), s[1], wt, ids, out_dtype=torch.float32, w_format=fw)
    c = run(w1, w2)
    assert c.shape == (T, MOE_OUT) and bool(torch.isfinite(c).all()) and int((c != 0).sum()) > 0.9 * c.numel()
    assert torch.equal(c.view(torch.int32), run(_moved(w1, 16), _moved(w2, 16)).view(torch.int32))
