"""Which form a mixture-of-experts layer takes (csrc/mx_api.hip, moe_plan), on the host: each form's workspace has a size of its own."""
import ctypes
import pathlib
import subprocess

import pytest
import torch

import cutile_amd
from cutile_amd import _lib as L
from test_load_once import evaluate as load_once  # noqa: F401

E4M3, E2M1 = L.MX_E4M3, L.MX_E2M1


def form(rows, E, H, F, w, H_out=None, tile_m=0, packed=True, topk=2):
    """"streamed", "grouped" or (row tiles of the library's own) their height and the ranges of K of the second product, for `rows` rows
    per expert on average."""
    lib, H_out, T = cutile_amd.lib(), H_out or H, int(rows * E) // topk
    weight = lambda n, k: L.MxTensor(ptr=4096, dtype=w, ndim=3, shape=(E, n, k, 0), stride=(n * k, k, 1, 0), packed_dim=2 if w == E2M1 else -1)
    layout = L.MX_SCALE_NATIVE if packed else L.MX_SCALE_2D
    o = L.MxGemmOpts(struct_size=32, block_size=32, tile_m=tile_m, a_scale_layout=layout, b_scale_layout=layout)
    W1, W2 = weight(2 * F, H), weight(H_out, F)
    need = lib.mx_moe_forward_workspace_bytes(T, topk, ctypes.byref(W1), ctypes.byref(W2), ctypes.byref(o))
    up, n = lambda b: (b + 255) // 256 * 256, T * topk
    activation, out = up(n * F) + up(n * (F // 32)), n * H_out * 4
    if need == activation + up(out):
        return "streamed"
    for height in (64, 128):
        tiles = (n + min(E, n) * (height - 1)) // height
        for splits in range(1, 9):
            if need == activation + up(out * splits) + up(tiles * 16) + up(tiles * height * 4):
                return height, splits
    assert need > activation + up(out) + n * F * 4   # the bf16 activation of both halves
    return "grouped"


def test_gpu_tests_reach_the_row_tiles_that_they_are_about(load_once):
    import test_gpu_moe_tiles as g
    at = lambda w, T, H, F, E, topk, _=0.0: form(T * topk / E, E, H, F, w, H + 72, topk=topk)
    assert [at(E4M3, *c)[0] for c in g.CASES] == [64] * len(g.CASES)
    # (the two cases of one expert before the last two need as much room with either height)
    assert all(tiled(T * topk / E, E, H, F, E2M1, H + 72, topk=topk) for T, H, F, E, topk, _ in g.CASES)
    assert [at(E2M1, *c)[0] for c in g.CASES[-2:]] == [128] * 2 and at(E2M1, *g.CASES[-1])[1] == 2
    assert all(at(w, *c) == "grouped" for w in (E4M3, E2M1) for c in g.GROUPED)
    assert all(at(w, *c) == "streamed" for w in (E4M3, E2M1) for c in g.STREAMED)
    # both products of the layers with non-temporal weights; some of the second ones in ranges of K
    ranges = [form(2 * T / E, E, H, F, E2M1 if f else E4M3, H_out) for f, layers in g.ONCE.items() for T, H, F, E, H_out in layers]
    assert all(height == 64 for height, _ in ranges) and any(n > 1 for _, n in ranges[:2]) and any(n > 1 for _, n in ranges[2:])
    row = lambda K, f: K // 2 if f else K
    assert load_once(*[f"stream_loads_once({min(2 * T, E) * n}LL, {row(K, f)}, {g.once_pitch(K, f)}, 0, 1)" for f, layers in g.ONCE.items()
                       for T, H, F, E, H_out in layers for n, K in ((2 * F, H), (H_out, F))]) == [1] * 10
    assert all(2 * T <= 48 * E for layers in g.ONCE.values() for T, _, _, E, _ in layers)


def tiled(*a, **kw):
    return form(*a, **kw) not in ("streamed", "grouped")


@pytest.mark.parametrize("w", [E4M3, E2M1])
def test_forms_by_rows_per_expert(w):
    for E, H, F in ((8, 2048, 7168), (8, 4096, 14336), (64, 1024, 1024)):
        assert form(24, E, H, F, w) == "streamed"
        assert all(tiled(r, E, H, F, w) for r in (25.5, 32, 64, 96))
        assert form(161, E, H, F, w) == "grouped"
    assert form(64, 8, 2048, 7168, w, packed=False) == "grouped" and form(32, 8, 2048, 7168, w, packed=False) == "streamed"


def test_streaming_ends_where_random_routing_gives_an_expert_more_than_32_rows():
    for w in (E4M3, E2M1):
        at = lambda E, topk: next(T * topk / E for T in range(1, 1000) if form(T * topk / E, E, 2048, 4096, w, topk=topk) != "streamed")
        assert [at(E, E) for E in (1, 2, 4, 8)] == [33] * 4            # every expert has the same
        assert [at(2, 1), at(4, 2), at(4, 1), at(8, 4), at(8, 2), at(8, 1)] == [27, 27, 25.5, 27, 25.5, 25]
        assert at(16, 2) == 24.125 and at(64, 2) == 24.03125


def test_padding_that_the_caller_asks_for():
    """An explicit tile_m is kept to where there are slots; 0 leaves the form to the library."""
    for w in (E4M3, E2M1):
        assert tiled(64, 8, 2048, 7168, w, tile_m=0)
        assert [form(64, 8, 2048, 7168, w, tile_m=t) for t in (128, 256, 512)] == ["grouped"] * 3


def test_row_tiles_of_three_per_expert():
    """Beyond 128 rows only where the 256-row tiles are not ahead."""
    ahead = [(8, 2048, 7168), (8, 2048, 8192), (8, 1536, 7168), (4, 2048, 14336), (16, 2048, 4096), (64, 2048, 1024), (8, 1024, 14336), (32, 1024, 2048)]
    behind = [(8, 2048, 14336), (8, 1536, 14336), (16, 1280, 8192), (32, 1536, 2048), (32, 2048, 2048), (64, 1536, 1024)]
    for w in (E4M3, E2M1):
        assert all(tiled(128, *s, w) for s in ahead + behind)
        assert [tiled(r, *s, w) for r in (129, 160) for s in ahead + behind] == ([True] * len(ahead) + [False] * len(behind)) * 2


@pytest.mark.parametrize("E,H,F,w", [(8, 1024, 14336, E4M3), (8, 2048, 7168, E2M1), (16, 2048, 4096, E4M3), (2, 4096, 14336, E2M1), (1, 1024, 14336, E4M3),
                                     (64, 1024, 1024, E2M1)])
def test_room_for_many_tokens_is_enough_for_fewer(E, H, F, w):
    """A row-tiled layer asks for more ranges of K, and more room for their sums, with fewer rows; it makes do with fewer of them."""
    if torch.cuda.is_available():
        pytest.skip("these pointers are the host's")
    lib, packed, topk = cutile_amd.lib(), 2 if w == E2M1 else -1, 1 if E == 1 else 2
    p = (torch.zeros(1 << 16, dtype=torch.uint8).data_ptr() + 255) // 256 * 256
    desc = lambda dtype, shape, strides, packed_dim=-1: L.MxTensor(ptr=p, dtype=dtype, ndim=len(shape), shape=shape + (0,) * (4 - len(shape)),
                                                                   stride=strides + (0,) * (4 - len(strides)), packed_dim=packed_dim)
    W = [desc(w, (E, n, k), (n * k, k, 1), packed) for n, k in ((2 * F, H), (H, F))]
    o = L.MxGemmOpts(struct_size=32, block_size=32, a_scale_layout=L.MX_SCALE_NATIVE, b_scale_layout=L.MX_SCALE_NATIVE)
    Ws = desc(L.MX_E8M0, (E, 1, 1), (1, 1, 1))
    need = lambda T: lib.mx_moe_forward_workspace_bytes(T, topk, *(ctypes.byref(t) for t in W), ctypes.byref(o))

    def forward(T, room):
        X, Xs = desc(E4M3, (T, H), (H, 1)), desc(L.MX_E8M0, (T, H // 32), (H // 32, 1))
        return lib.mx_moe_forward(*(ctypes.byref(t) for t in (X, Xs, W[0], Ws, W[1], Ws)), p, p, 0, topk,
                                  ctypes.byref(desc(L.MX_F32, (T, H), (H, 1))), 1, ctypes.byref(o), p, room, None)
    tokens = [t for t in range(1, 180 * E // topk, max(1, E // 2))]
    for i, T in enumerate(tokens):
        assert forward(T, min(need(t) for t in tokens[i:])) == L.MX_ERR_LAUNCH   # (no GPU here: everything before was in order)
        f = form(T * topk / E, E, H, F, w, topk=topk)
        ranges = 1 if isinstance(f, str) else f[1]
        assert forward(T, need(T) - (ranges - 1) * T * topk * H * 4 - 1) == L.MX_ERR_WORKSPACE


@pytest.mark.parametrize("E,H,F,limits", [
    (8, 4096, 7168, (128, 128)), (8, 4096, 14336, (96, 128)), (16, 3072, 8192, (96, 120)), (16, 4096, 8192, (64, 120)), (12, 3584, 14336, (64, 128)),
    (16, 4096, 4096, (120, 120)), (32, 4096, 2048, (128, 128)), (64, 4096, 1024, (128, 128)),      # long rows
    (32, 1536, 8192, (72, 72)), (64, 2048, 4096, (72, 72)), (64, 1024, 4096, (96, 96)),            # short ones, large layers
    (32, 1536, 4096, (120, 120)), (128, 1536, 1024, (120, 120)), (16, 2048, 8192, (128, 128)), (12, 1536, 14336, (128, 128)),
    (16, 1024, 8192, (160, 160)), (32, 1024, 4096, (128, 128)), (64, 1024, 2048, (128, 128)), (32, 1024, 2048, (160, 160))])
def test_rows_up_to_which_a_layer_has_row_tiles(E, H, F, limits):
    for w, limit in zip((E4M3, E2M1), limits):
        assert tiled(limit, E, H, F, w) and form(limit + 1, E, H, F, w) == "grouped"


def test_routing_by_one_workgroup_where_it_is_the_faster_one(tmp_path):
    cases = [(1, 1), (12288, 256), (12288, 257), (14336, 64), (12289, 65), (16384, 16), (16384, 17), (14337, 64), (16385, 1), (0, 8)]
    src = pathlib.Path(__file__).resolve().parent.parent / "cutile-python_amd" / "csrc"
    body = "".join(f'std::printf("%d\\n", (int)mx::moe_align_in_one_workgroup({n}, {e}));' for n, e in cases)
    (tmp_path / "p.cpp").write_text('#include <cstdio>\n#include "mx_moe_rules.h"\nint main() { %s }\n' % body)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{src}", "-o", str(tmp_path / "p"), str(tmp_path / "p.cpp")], check=True)
    got = subprocess.run([str(tmp_path / "p")], check=True, capture_output=True, text=True).stdout.split()
    assert got == ["1", "1", "0", "1", "0", "1", "0", "0", "0", "0"]
