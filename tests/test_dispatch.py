"""MX_KERNEL_AUTO never picks a kernel whose launch refuses the operands: few rows of A with weights whose rows overlap (a
broadcast or a sliding window) or with scale rows that span 2 GiB.  What a split along K needs is asked for only where the
split is a contract; a mixture-of-experts layer keeps to the caller's tile_m; no rows, no launch.  On the host: where there is no device a dispatched launch ends in MX_ERR_LAUNCH, a refusal in
MX_ERR_LAYOUT or MX_ERR_WORKSPACE."""
import ctypes

import pytest
import torch

import cutile_amd
from cutile_amd import _lib as L
from test_cabi import _desc

# the descriptors name host memory, or extents that are not there
pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="would launch kernels on host pointers")

WIDE = 1 << 26   # 32 rows of this pitch are 2 GiB


def _gemm(M, N, K, fmt, b_pitch=None, as_pitch=None, bs_pitch=None, kernel=L.MX_KERNEL_AUTO):
    lib = cutile_amd.lib()
    buf = torch.zeros(1 << 22, dtype=torch.uint8)
    p = (buf.data_ptr() + 255) // 256 * 256
    packed = fmt == L.MX_E2M1
    row = K // 2 if packed else K
    A = _desc(p, L.MX_E4M3, (M, K), (K, 1))
    As = _desc(p, L.MX_E8M0, (M, K // 32), (K // 32 if as_pitch is None else as_pitch, 1))
    B = _desc(p, fmt, (K, N), (1, row if b_pitch is None else b_pitch), 0 if packed else -1)
    Bs = _desc(p, L.MX_E8M0, (K // 32, N), (1, K // 32 if bs_pitch is None else bs_pitch))
    C = _desc(p, L.MX_F32, (M, N), (N, 1))
    o = L.MxGemmOpts(struct_size=32, kernel=kernel, block_size=32)
    rc = lib.mx_gemm(*(ctypes.byref(t) for t in (A, As, B, Bs, C)), ctypes.byref(o), p, 1 << 21, None)
    return rc, L.last_error()


@pytest.mark.parametrize("fmt", [L.MX_E4M3, L.MX_E2M1])
@pytest.mark.parametrize("M", [1, 8, 33, 64, 65])
@pytest.mark.parametrize("K", [512, 640, 8704])
def test_auto_launches_something(fmt, M, K):
    for kw in ({}, {"b_pitch": 0}, {"b_pitch": 16}, {"b_pitch": 0, "bs_pitch": 0}, {"as_pitch": WIDE}, {"as_pitch": 1 << 31},
               {"as_pitch": WIDE + 4, "b_pitch": 16}):
        rc, message = _gemm(M, 256, K, fmt, **kw)
        assert rc == L.MX_ERR_LAUNCH, (kw, rc, message)
    # the scale rows of FP4 weights for the decode kernel are held to 2 GiB, other kernels re-lay them
    if not (fmt == L.MX_E2M1 and M <= 32 and K == 512):
        rc, message = _gemm(M, 256, K, fmt, bs_pitch=WIDE)
        assert rc == L.MX_ERR_LAUNCH, (rc, message)


def test_a_forced_streaming_kernel_says_what_it_cannot_take():
    rc, message = _gemm(8, 256, 512, L.MX_E4M3, bs_pitch=WIDE, kernel=9)
    assert rc == L.MX_ERR_LAYOUT and "B_scale spans 2 GiB" in message
    rc, message = _gemm(8, 256, 512, L.MX_E4M3, b_pitch=520, kernel=9)
    assert rc == L.MX_ERR_LAYOUT and "16-byte aligned rows" in message


def _split_problem(M, N, K, layouts, split_k):
    p = (torch.zeros(1 << 16, dtype=torch.uint8).data_ptr() + 255) // 256 * 256
    t = (_desc(p, L.MX_E4M3, (M, K), (K, 1)), _desc(p, L.MX_E8M0, (M, K // 32), (K // 32, 1)),
         _desc(p, L.MX_E4M3, (K, N), (1, K)), _desc(p, L.MX_E8M0, (K // 32, N), (1, K // 32)),
         _desc(p, L.MX_F32, (M, N), (N, 1)))
    o = L.MxGemmOpts(struct_size=32, block_size=32, split_k=split_k, a_scale_layout=layouts[0], b_scale_layout=layouts[1])
    return p, [ctypes.byref(x) for x in t], o


@pytest.mark.parametrize("split_k", [0, 2])
@pytest.mark.parametrize("K,layouts", [(8192, (2, 2)), (8192, (0, 2)), (8000, (0, 0))])
def test_an_unpromised_split_needs_no_workspace(K, layouts, split_k):
    """Packed scales, or a K that is not whole slices of 512: with room for the scales alone the product runs whole, as one
    call, as an entry of a list and in the static scratch."""
    lib, (M, N) = cutile_amd.lib(), (300, 200)
    p, t, o = _split_problem(M, N, K, layouts, split_k)
    scales = sum(lib.mx_packed_scale_bytes(rows, K) for rows, layout in ((M, layouts[0]), (N, layouts[1])) if layout == 0)
    assert split_k == 2 and K == 8000 or lib.mx_gemm_workspace_bytes(M, N, K, ctypes.byref(o)) > scales
    for have in (scales, scales + 256):
        ws = p if have else None
        assert lib.mx_gemm(*t, ctypes.byref(o), ws, have, None) == L.MX_ERR_LAUNCH, L.last_error()
        assert lib.mx_gemm_list(1, *t, ctypes.byref(o), ws, have, None) == L.MX_ERR_LAUNCH, L.last_error()
    if scales:
        assert lib.mx_gemm(*t, ctypes.byref(o), p, scales - 256, None) == L.MX_ERR_WORKSPACE
        assert lib.mx_gemm_list(1, *t, ctypes.byref(o), p, scales - 256, None) == L.MX_ERR_WORKSPACE
    p, t, o = _split_problem(1000, 2000, K, layouts, 2 if K == 8192 else 0)
    if layouts != (0, 0):   # two slices of 8 MB: more than the static scratch holds
        assert lib.mx_gemm_static(*t, ctypes.byref(o), None) == L.MX_ERR_DEVICE, L.last_error()


@pytest.mark.parametrize("split_k", [0, 2])
def test_a_promised_split_is_held_to_its_workspace(split_k):
    """Plain scales and equal slices of 512: less than the partial sums need is refused."""
    lib, (M, N, K) = cutile_amd.lib(), (300, 200, 8192)
    p, t, o = _split_problem(M, N, K, (0, 0), split_k)
    need = lib.mx_gemm_workspace_bytes(M, N, K, ctypes.byref(o))
    assert lib.mx_gemm(*t, ctypes.byref(o), p, need, None) == L.MX_ERR_LAUNCH
    assert lib.mx_gemm(*t, ctypes.byref(o), p, need - 256, None) == L.MX_ERR_WORKSPACE
    assert lib.mx_gemm_list(1, *t, ctypes.byref(o), p, need - 256, None) == L.MX_ERR_WORKSPACE


@pytest.mark.parametrize("M,N,K", [(6319, 3444, 9216), (1554, 13416, 10240), (759, 26481, 7680), (9970, 7006, 4096)])
@pytest.mark.parametrize("layouts", [(0, 0), (0, 2), (2, 2)])
def test_no_room_is_asked_for_a_split_that_192_row_tiles_do_not_make(M, N, K, layouts):
    """MX_KERNEL_AUTO takes 192-row tiles here, with room for the split last round of 256-row tiles and without; the forced kernel,
    which keeps to 256 rows, is given the room as before."""
    lib = cutile_amd.lib()
    scales = sum(lib.mx_packed_scale_bytes(rows, K) for rows, layout in ((M, layouts[0]), (N, layouts[1])) if layout == 0)
    need = lambda **kw: lib.mx_gemm_workspace_bytes(M, N, K, ctypes.byref(
        L.MxGemmOpts(struct_size=32, block_size=32, a_scale_layout=layouts[0], b_scale_layout=layouts[1], **kw)))
    assert need() == need(split_k=1) == scales
    assert need(kernel=L.MX_KERNEL_MFMA_PINGPONG) > scales


def test_moe_slots_follow_tile_m(monkeypatch):
    """The grouped form of the layer aligns to the caller's tile_m (its workspace shrinks with the padding), refuses what the
    tiled kernels cannot take, and the operator hands its tile_m over; streamed layers have no slots."""
    lib, E, H, F = cutile_amd.lib(), 16, 512, 256
    p = (torch.zeros(1 << 16, dtype=torch.uint8).data_ptr() + 255) // 256 * 256
    W1, W2 = _desc(p, 0, (E, 2 * F, H), (2 * F * H, H, 1)), _desc(p, 0, (E, H, F), (H * F, F, 1))

    def need(T, tile_m):
        o = L.MxGemmOpts(struct_size=32, block_size=32, tile_m=tile_m)
        return lib.mx_moe_forward_workspace_bytes(T, 2, ctypes.byref(W1), ctypes.byref(W2), ctypes.byref(o))
    assert need(2000, 128) < need(2000, 256) < need(2000, 512)
    assert need(2000, 0) == need(2000, 256)
    assert need(64, 128) == need(64, 256) == need(64, 16)   # streamed

    def forward(T, tile_m, xs_pitch=H // 32):
        o = L.MxGemmOpts(struct_size=32, block_size=32, tile_m=tile_m)
        X, Xs = _desc(p, 0, (T, H), (H, 1)), _desc(p, L.MX_E8M0, (T, H // 32), (xs_pitch, 1))
        W1s = _desc(p, L.MX_E8M0, (E, 2 * F, H // 32), (2 * F * H // 32, H // 32, 1))
        W2s = _desc(p, L.MX_E8M0, (E, H, F // 32), (H * F // 32, F // 32, 1))
        out = _desc(p, L.MX_F32, (T, H), (H, 1))
        return lib.mx_moe_forward(*(ctypes.byref(t) for t in (X, Xs, W1, W1s, W2, W2s)), p, p, 0, 2, ctypes.byref(out), 1,
                                  ctypes.byref(o), p, 1 << 40, None)
    assert [forward(2000, t) for t in (0, 128, 384, 512)] == [L.MX_ERR_LAUNCH] * 4
    assert forward(2000, 64) == L.MX_ERR_LAYOUT and "tile_m" in L.last_error()
    assert forward(64, 64) == L.MX_ERR_LAUNCH
    # scale rows that lane offsets do not reach go to the single operators, streamed or not
    for T in (64, 2000):
        assert forward(T, 0, ((1 << 31) - 1) // T // 4 * 4) == L.MX_ERR_LAUNCH
        assert forward(T, 0, ((1 << 31) - 1) // T // 4 * 4 + 4) == L.MX_ERR_LAYOUT and "X_scale" in L.last_error()

    class Host:
        def moe(self, *args):
            self.args = args
            return torch.zeros(0)
    monkeypatch.setattr(L, "_host", Host())
    cutile_amd.cutile_moe_scaled(*[None] * 8, 128)
    assert L._host.args[-1] == 128


@pytest.mark.parametrize("kernel,tile_m", [(0, 128), (0, 256), (2, 128), (2, 256), (3, 256), (4, 256), (6, 256)])
def test_grouped_product_of_no_rows_launches_nothing(kernel, tile_m):
    """Slots that are all padding over an A without rows, whose row pitch is wider than a row: a descriptor that ended behind
    its last row would wrap around."""
    lib, E, N, K = cutile_amd.lib(), 2, 256, 512
    p = (torch.zeros(1 << 16, dtype=torch.uint8).data_ptr() + 255) // 256 * 256
    W, Ws = _desc(p, 0, (E, N, K), (N * K, K, 1)), _desc(p, L.MX_E8M0, (E, N, K // 32), (N * K // 32, K // 32, 1))
    o = L.MxGemmOpts(struct_size=32, block_size=32, kernel=kernel)
    for T, want in ((0, L.MX_OK), (3, L.MX_ERR_LAUNCH)):
        A, As = _desc(p, 0, (T, K), (K + 16, 1)), _desc(p, L.MX_E8M0, (T, K // 32), (K // 32, 1))
        C = _desc(p, L.MX_F32, (T, N), (N, 1))
        rc = lib.mx_gemm_grouped(*(ctypes.byref(t) for t in (A, As, W, Ws, C)), None, p, tile_m, p, tile_m, 1, T,
                                 ctypes.byref(o), p, 1 << 30, None)
        assert rc == want, L.last_error()
