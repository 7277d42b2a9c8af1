"""The quantiser of aligned rows at the sizes where its launch changes form (loads, units per thread): bit-exact."""
import numpy as np
import pytest
import torch

from oracle import mx_oracle as O

pytestmark = pytest.mark.gpu
DT = {O.E4M3: torch.float8_e4m3fn, O.E5M2: torch.float8_e5m2, O.E2M1: "e2m1"}


# 2^20 units of 8 elements and 48 Mi elements are the lines; a row more, a row less, and the last thread's units partly beyond the end
@pytest.mark.parametrize("rows", [4095, 4096, 4099, 24577])
@pytest.mark.parametrize("fmt", [O.E4M3, O.E2M1])
def test_quantize_at_the_lines(ct, dev, rows, fmt):
    _check(ct, dev, rows, fmt, torch.bfloat16)


# the line of the non-temporal loads lies at a number of elements, whatever the input's type
@pytest.mark.parametrize("rows", [24575, 24576])
@pytest.mark.parametrize("src,fmt", [(torch.float32, O.E4M3), (torch.float32, O.E2M1), (torch.float16, O.E5M2)], ids=str)
def test_quantize_other_inputs_at_the_line(ct, dev, rows, src, fmt):
    _check(ct, dev, rows, fmt, src)


def _check(ct, dev, rows, fmt, src):
    K, period = 2048, 61
    g = torch.Generator().manual_seed(rows)
    base = (torch.randn((period, K), generator=g) * torch.logspace(-6, 3, period)[:, None]).to(src)
    base[5, 64:96] = 0          # blocks that the hardware conversion does not serve
    base[6, 32] = float("inf")  # (the ceiling rule says what becomes of such a block; the floor rule does not)
    x = base.repeat((rows + period - 1) // period, 1)[:rows].to(dev)
    q, sc = ct.block_quantize(x, 32, DT[fmt], scale_mode="ceil")
    codes, sb = O.block_quantize(base.float().numpy(), 32, fmt, "ceil")
    want = torch.from_numpy(O.pack_fp4(codes) if fmt == O.E2M1 else codes).to(dev)
    idx = torch.arange(rows, device=dev) % period
    assert torch.equal(q.view(torch.uint8), want[idx])
    assert torch.equal(sc.view(torch.uint8), torch.from_numpy(sb).to(dev)[idx])
