"""The prefill GEMM's tile heights and edges against the oracle.

The height follows from the batch and the shape, so each case names one that
the rule picks on 256 CUs. Gate as in ``test_fused_gpu.py``: max abs/rel 2e-2
and relative L2 < 0.005 (the prefill path multiplies the reference's exact
weights, so what differs is the order of fp32 sums).
"""

import numpy as np
import pytest
import torch

from loraforge_amd.ops import nf4_lora_linear
from tests import _cases
from tests.test_fused_gpu import bits, close, to_device, workspace_clean

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "m,n,k,slices,bounds,ranks",
    [
        # One token past a tile of 64; N past the last 256-column tile by 64; K = one, two and three 64-k blocks.
        (65, 320, 64, 1, None, (16, 5)),
        (129, 64, 128, 1, None, (64, 1)),
        (193, 576, 192, 3, [0, 250, 383, 576], (33, 8, 0)),  # slice bounds inside a wave's columns
        (320, 256, 320, 2, [0, 128, 256], (4, 16, 48)),  # an odd number of 128-k stages plus a block
        (161, 1024, 896, 1, None, tuple([8, 16, 32, 64] * 12)),  # an odd number of stages, 48 slots
    ],
)
def test_small_heights_and_edges(m, n, k, slices, bounds, ranks, device):
    case = _cases.fused_case(m, n, k, ranks=ranks, slices=slices, bounds=bounds, bias=bool(m & 1), seed=m + n)
    x, q, st, lora, bias = to_device(case, device)
    y = nf4_lora_linear(x, q, st, lora=lora, bias=bias, plan="prefill")
    torch.cuda.synchronize()
    close(bits(y), _cases.fused_expected(case))
    workspace_clean(device)


@pytest.mark.parametrize(
    "m,n",
    [
        (300, 16384),  # 160 tokens a tile (128 tiles; 96-token tiles would need 256)
        (380, 24576),  # 192: 2 x 96 tiles
        (520, 16320),  # 128 or 192 with a last column tile of 192 columns
        (2000, 8192),  # 256: 8 x 32 tiles fill the chip once, z in a launch of its own
    ],
)
def test_tall_tiles_against_torch(m, n, device):
    """Every element against fp64 products of the dequantised weight in PyTorch."""
    k = 256
    g = torch.Generator(device=device).manual_seed(m + n)
    from loraforge_amd.ops import LoraBatch, dequantize_nf4, quantize_nf4

    q, st = quantize_nf4((torch.randn(n, k, generator=g, device=device) * 0.02).bfloat16())
    x = torch.randn(m, k, generator=g, device=device).bfloat16()
    r, slots = 16, 5
    a = (torch.randn(slots, r, k, generator=g, device=device) * 0.02).bfloat16()
    b = (torch.randn(slots, n, r, generator=g, device=device) * 0.02).bfloat16()
    routes = torch.repeat_interleave(torch.arange(-1, slots), -(-m // (slots + 1)))[:m].int()
    i64, i32 = dict(dtype=torch.int64, device=device), dict(dtype=torch.int32, device=device)
    lora = LoraBatch(a.reshape(-1), torch.arange(slots, **i64) * (r * k), b.reshape(-1), torch.arange(slots, **i64) * (n * r),
                     torch.full((slots,), r, **i32), torch.full((slots,), r, **i32), torch.full((slots,), 2.0, device=device),
                     routes.to(device), torch.tensor([0, n], **i32), max_rank=r)
    y = nf4_lora_linear(x, q, st, lora=lora, plan="prefill")
    w = dequantize_nf4(q, st.absmax, st.code, (n, k)).double()
    want = (x.double() @ w.t()).bfloat16().double()
    for s in range(slots):
        rows = (routes == s).to(device)
        z = (x[rows].double() @ a[s].double().t()).bfloat16().double()
        want[rows] = (want[rows] + (2.0 * (z @ b[s].double().t())).bfloat16().double()).bfloat16().double()
    torch.cuda.synchronize()
    # A bf16 result whose fp32 sums run in another order: one rounding of y and one of z and of the delta.
    err = (y.double() - want).abs()
    assert (err.norm() / want.norm()).item() < 0.005
    assert bool((err <= 2e-2 + 2e-2 * want.abs()).all())
