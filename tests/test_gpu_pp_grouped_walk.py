"""Grouped products on 256-row tiles: the order in which the tiles are walked, and the ids requested ahead of each tile.

Every tile of every expert is computed once, whatever the experts' numbers of tile rows (groups of up to 5 rows that don't
cross experts and are cut where 64 tile rows end), and the ids are there with one stage of K per tile or many, with sentinels
among the rows."""
import pytest
import torch

from mxutil import raw_operand
from oracle import mx_oracle as O

pytestmark = pytest.mark.gpu
# of the norm: 128 products of a K-step, each cut at most 2^-17 below the largest; half a unit of bf16 (2^-9 of each value)
TOL = {torch.float32: 1e-3, torch.bfloat16: 1e-3 + 2 ** -9}


# tile rows of the experts: every size of a group, experts with none, groups cut at 64 tile rows, one expert over several of these
TILES = [(1, 2, 3, 4, 5, 6, 7), (0, 9, 0, 11, 1, 1), (40, 30, 3), (131,)]


@pytest.mark.parametrize("K", [96, 256, 416, 544, 1024, 1536])
@pytest.mark.parametrize("tiles", TILES, ids=str)
@pytest.mark.parametrize("fa,fb", [(O.E4M3, O.E4M3), (O.E2M1, O.E2M1), (O.E4M3, O.E2M1)], ids=str)
def test_grouped_walk(ct, dev, fa, fb, tiles, K):
    E, N, tokens, slots = len(tiles), 1288, 300, 256 * sum(tiles)
    g = torch.Generator(device=dev).manual_seed(slots + K)
    w, x = raw_operand(E * N, K, fb, K, dev), raw_operand(tokens, K, fa, K + 1, dev)
    W, Ws = w.storage.view(E, N, -1), w.scale_t.view(E, N, -1)
    # every routed slot once, in any order; a third of the rows are sentinels
    valid = slots * 2 // 3
    ids = torch.randperm(slots, generator=g, device=dev).clamp(max=valid).to(torch.int32)
    eids = torch.repeat_interleave(torch.arange(E, device=dev), torch.tensor(tiles, device=dev)).to(torch.int32)
    replicas = -(-valid // tokens)
    weights = torch.rand(valid, generator=g, device=dev)
    deq = lambda o: torch.as_tensor(O.dequantize(o.codes, o.scales, o.fmt)).to(dev, torch.float64)
    wd, xd = deq(w).view(E, N, K), deq(x)
    want = torch.empty((valid, N), dtype=torch.float64, device=dev)
    for e, rows in enumerate(ids.view(-1, 256)):
        rows = rows[rows < valid].long()
        want[rows] = xd[rows // replicas] @ wd[int(eids[e])].T
    for dt, routed in ((torch.float32, False), (torch.bfloat16, True)):
        out = torch.full((valid, N), float("nan"), device=dev, dtype=dt)
        ct.invoke_fused_moe_scaled(x.storage, x.scale_t, W, ct.pack_scales(Ws, operand="b"), out, weights, ids, eids, routed, replicas,
                                   256, a_format=x.fmt_kw, b_format=w.fmt_kw, kernel="pingpong")
        err = O.rel_fro(out.double(), want * weights[:, None] if routed else want)
        print(f"{fa} {fb} {tiles} K={K} {dt}: {float(err):.2e}", flush=True)
        assert err < TOL[dt]
