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


def test_cached_scales_follow_a_tensor_whose_data_was_replaced(ct, dev):
    """`tensor.data = other` keeps the object and its version: the cached re-layout of the old bytes must not be used."""
    ct.clear_scale_cache()
    a, b = randn_operand(256, 512, O.E4M3, 5, dev), randn_operand(384, 512, O.E4M3, 6, dev)
    run = lambda: ct.block_scaled_matmul(a.storage, s, b.storage.T, bs, cache_scales=True)
    s, bs = a.scale_t.clone(), b.scale_t.T
    first = [run() for _ in range(3)][-1]
    s.data = (a.scale_t.view(torch.uint8) + 1).view(torch.float8_e8m0fnu)
    assert torch.equal(run(), first * 2)
    ct.clear_scale_cache()


@pytest.mark.parametrize("K", [3584, 4000])
@pytest.mark.parametrize("packed", [False, True])
def test_split_that_never_applied_and_static_scratch_run_whole(ct, dev, K, packed):
    """A forced split of a K (or scale layout) that is not split runs whole instead of failing, and the static scratch
    takes the problems whose automatic split alone would not fit into it."""
    a, b = randn_operand(600, K, O.E4M3, 7, dev), randn_operand(1500, K, O.E4M3, 8, dev)
    As = ct.pack_scales(a.scale_t, operand="a") if packed else a.scale_t
    Bs = ct.pack_scales(b.scale_t, operand="b") if packed else b.scale_t.T
    whole = ct.block_scaled_matmul(a.storage, As, b.storage.T, Bs, split_k=1)
    if packed or K % 512:
        forced = ct.block_scaled_matmul(a.storage, As, b.storage.T, Bs, split_k=3)
        assert O.rel_fro(forced.cpu(), whole.cpu()) <= 1e-5   # (fp32 sums, order of the K steps at most)
    c = ct.block_scaled_matmul(a.storage, As, b.storage.T, Bs, static_scratch=True)
    assert O.rel_fro(c.cpu(), whole.cpu()) <= 1e-5


@pytest.mark.parametrize("fmt,K", [(O.E4M3, 2560), (O.E5M2, 4608), (O.E2M1, 4096), (O.E4M3, 14336)])
@pytest.mark.parametrize("M,N", [(300, 260), (1000, 1030), (2800, 6200), (4097, 4096), (1000, 8000), (2500, 3300), (4000, 6400)])
@pytest.mark.parametrize("out_dtype,accumulate", [(torch.float32, True), (torch.bfloat16, False)], ids=str)
def test_pingpong_last_round_split_along_k(ct, dev, fmt, K, M, N, out_dtype, accumulate):
    """Tile counts that leave the last (or only) round partly filled: one to 16 tiles per XCD beyond whole rounds (and
    XCDs whose share leaves nothing to split beside XCDs that split), split two to eight ways into slices of unequal
    length, ragged edges, accumulation; nothing written beside C.  The sums differ from the unsplit kernel's by the order
    of fp32 additions."""
    def raw(rows, seed):
        g = torch.Generator(device=dev).manual_seed(seed)
        q, s = ct.block_quantize(torch.randn((rows, K), generator=g, device=dev), 32, {O.E4M3: torch.float8_e4m3fn,
                                 O.E5M2: torch.float8_e5m2, O.E2M1: "e2m1"}[fmt], scale_mode="floor")
        return q, s
    (a, sa), (b, sb) = raw(M, 1), raw(N, 2)
    kw = dict(a_format="e2m1", b_format="e2m1") if fmt == O.E2M1 else {}
    pitch = N + 24
    bufs = [torch.full((M + 2, pitch), 7.0, dtype=out_dtype, device=dev) for _ in range(2)]
    for buf, kernel in zip(bufs, ("pingpong", "mfma128")):
        c = buf[1:M + 1, :N]
        ct.block_scaled_matmul(a, sa, b.T, sb.T, C=c, accumulate=accumulate, kernel=kernel, split_k=0 if kernel == "pingpong" else 1, **kw)
    if not accumulate:   # split_k = 1 forbids this split too
        whole = ct.block_scaled_matmul(a, sa, b.T, sb.T, out_dtype=out_dtype, kernel="pingpong", split_k=1, **kw)
        assert torch.equal(whole, bufs[1][1:M + 1, :N])
    got, ref = bufs[0].float(), bufs[1].float()
    rel = ((got - ref).norm() / ref[1:M + 1, :N].norm()).item()
    assert rel <= (1e-5 if out_dtype == torch.float32 else 4e-3), rel   # (guards are equal on both sides)
    assert (bufs[0][0] == 7).all() and (bufs[0][-1] == 7).all() and (bufs[0][:, N:] == 7).all()


@pytest.mark.parametrize("kernel", ["mfma128", "mfma256", "mfma256w4", "pingpong", "pingpong32", "w4p", "generic"])
@pytest.mark.parametrize("side", ["a", "b"])
@pytest.mark.parametrize("fmt,K", [(O.E4M3, 1152), (O.E2M1, 2304), (O.E4M3, 2048)])
def test_rows_may_overlap(ct, dev, kernel, side, fmt, K):
    """One operand as a broadcast row, or as windows that slide over one buffer: every kernel reads its last rows to their
    end.  (K = 2048 also split along K.)"""
    if fmt == O.E2M1 and kernel in ("pingpong32", "w4p"):
        pytest.skip("8-bit element formats only")
    M, N = 300, 272
    a, b = randn_operand(M, K, fmt, 41, dev), randn_operand(N, K, fmt, 42, dev)
    rows, row = (M, N)[side == "b"], (K // 2 if fmt == O.E2M1 else K)
    flat = randn_operand(1, K + 32 * max(M, N), fmt, 43, dev)
    for pitch in (0, 16):
        t = flat.storage.view(-1).as_strided((rows, row), (pitch, 1))
        codes = torch.from_numpy(flat.storage_np).view(-1).as_strided((rows, row), (pitch, 1)).contiguous().numpy()
        op = a if side == "a" else b
        op.storage, op.codes = t, O.unpack_fp4(codes) if fmt == O.E2M1 else codes
        ref = oracle_matmul(a, b)
        for split_k in (0, 2) if K == 2048 and kernel.startswith("mfma") else (0,):
            c = ct.block_scaled_matmul(a.storage, a.scale_t, b.storage.T, b.scale_t.T, a_format=a.fmt_kw, b_format=b.fmt_kw,
                                       kernel=kernel, split_k=split_k, out_dtype=torch.float32)
            assert O.rel_fro(c.cpu(), ref) <= TOL[torch.float32], (pitch, split_k)
