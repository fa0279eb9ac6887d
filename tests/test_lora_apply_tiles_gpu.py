"""``lora_apply`` above 64 tokens (shrink and expand as two launches) against the oracle.

Gate as in ``test_lora_apply_gpu.py``: max abs/rel 2e-2, relative L2 < 0.005,
rows without an adapter keep their bits.
"""

import ctypes

import numpy as np
import pytest
import torch

from loraforge_amd import _lib
from loraforge_amd.ops import lora_apply
from loraforge_amd.ops.fused import workspace_bytes
from tests import _cases
from tests.test_fused_gpu import bits
from tests.test_lora_apply_gpu import check, make_case, on_device

pytestmark = pytest.mark.gpu


def two_launches(m, n, k, slices, ranks):
    two = ctypes.c_int32()
    _lib.check(_lib.library().lf_lora_apply_plan(m, n, k, slices, max(ranks), len(ranks), ctypes.byref(two)))
    return bool(two.value)


@pytest.mark.parametrize(
    "m,n,k,slices,bounds,ranks,two",
    [
        (128, 64, 64, 1, None, (16,), False),  # the most tokens of the smallest N and K that take launches per 64 tokens,
        (129, 64, 64, 1, None, (16,), True),  # and the fewest that take the two launches
        (257, 320, 192, 3, [0, 190, 257, 320], (64, 7, 0, 16), True),  # slice bounds inside fragments, a wave past N; a second z tile of one token
        (330, 576, 320, 2, [0, 300, 576], (2, 4, 8, 17, 48), True),  # a last tile of ten tokens
        (700, 1024, 1024, 1, None, tuple([4, 8, 16, 32] * 4), True),  # 16 slots: the most that take the two launches
        (300, 1024, 256, 1, None, tuple([4, 8, 16, 32] * 16), False),  # 64 slots: launches per 64 tokens
    ],
)
def test_tiles(m, n, k, slices, bounds, ranks, two, device):
    assert two_launches(m, n, k, slices, ranks) == two
    case = make_case(m, n, k, ranks, slices=slices, bounds=bounds, seed=m + k)
    x, y, batch = on_device(case, device)
    assert lora_apply(x, y, batch) is y
    check(case, y)
    # An output whose rows are not 8-byte aligned (element-wise updates) gives the same bits.
    wide = torch.zeros(m, n + 3, dtype=torch.bfloat16, device=device)
    odd = wide[:, 1 : n + 1]
    odd.copy_(torch.from_numpy(case["y"].view(np.int16)).view(torch.bfloat16))
    lora_apply(x, odd, batch)
    torch.cuda.synchronize()
    assert torch.equal(odd, y) and not wide[:, 0].any() and not wide[:, n + 1 :].any()


def test_routes_in_segments_and_a_workspace_of_few_tokens(device):
    """Contiguous prompts; a workspace that holds 256 tokens' z rows takes two rounds of launches
    (same bits), one that holds fewer than 128 the launches per 64 tokens (the oracle's gate)."""
    m, n, k = 500, 512, 256
    routes = np.repeat(np.array([2, 0, -1, 1], np.int32), [130, 200, 50, 120])
    assert two_launches(m, n, k, 1, (32, 16, 8))
    case = make_case(m, n, k, (32, 16, 8), seed=77, routes=routes)
    x, y, batch = on_device(case, device)
    lora_apply(x, y, batch)
    check(case, y)
    flags, header = 262144, 262144 + 16384  # the prefill flags' region ahead of the z rows stays untouched
    for rows, same in ((300, True), (100, False)):
        ws = torch.zeros(max(header + rows * 128, workspace_bytes(64, n, k, max_rank=32)), dtype=torch.uint8, device=device)
        _, again, _ = on_device(case, device)
        lora_apply(x, again, batch, workspace=ws)
        check(case, again)
        assert not same or np.array_equal(bits(again), bits(y))
        assert not ws[flags:header].any()


@pytest.mark.parametrize(
    "m,n,k,slices,bounds,ranks",
    [
        (200, 512, 2112, 1, None, (16, 3)),  # 16.5 stages of 128 k: one wave with three, the last of half a stage
        (333, 256, 3136, 2, [0, 64, 256], (64, 5, 33)),  # 24.5 stages; units of several passes
        (65, 1024, 4096, 1, None, (1,)),  # four stages a wave; one A row; a unit of one token
    ],
)
def test_z_stages(m, n, k, slices, bounds, ranks, device):
    """K where the waves of a z unit have different numbers of stages, and reuse their slots."""
    assert two_launches(m, n, k, slices, ranks)
    routes = np.arange(m, dtype=np.int32) % (len(ranks) + 1) - 1 if len(ranks) > 1 else np.zeros(m, np.int32)
    case = make_case(m, n, k, ranks, slices=slices, bounds=bounds, seed=m + k, routes=routes)
    x, y, batch = on_device(case, device)
    lora_apply(x, y, batch)
    check(case, y)
