"""The prefill GEMM's tile heights and edges against the oracle.

The height follows from the batch and the shape; each case asserts the one that
it is meant to run (``lf_nf4_lora_plan``). Gate as in ``test_fused_gpu.py``: max
abs/rel 2e-2 and relative L2 < 0.005 (the prefill path multiplies the reference's
exact weights, so what differs is the order of fp32 sums).
"""

import ctypes

import numpy as np
import pytest
import torch

from loraforge_amd import _lib
from loraforge_amd.ops import LoraBatch, dequantize_nf4, nf4_lora_linear, quantize_nf4
from loraforge_amd.ops.fused import _lora_struct, _weight_struct, workspace_bytes
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


def plan_of(m, n, k, lora=None, swiglu=False):
    plan = _lib.Plan()
    adapters = (lora.num_slices, lora.max_rank, lora.ranks.numel()) if lora is not None else (0, 1, 0)
    flags = _lib.LF_PLAN_PREFILL | (_lib.LF_SWIGLU_OUTPUT if swiglu else 0)
    _lib.check(_lib.library().lf_nf4_lora_plan(m, n, k, *adapters, flags, ctypes.byref(plan)))
    assert plan.kernel == _lib.LF_KERNEL_PREFILL
    return plan


class Problem:
    """A linear with ``slots`` adapters of rank ``r`` and its result in fp32 products in PyTorch."""

    def __init__(self, m, n, k, device, *, r=16, slots=5, slices=1, routes="together", seed=0):
        g = torch.Generator(device=device).manual_seed(m + n + k + seed)
        rand = lambda *shape, std=0.02: (torch.randn(*shape, generator=g, device=device) * std).bfloat16()
        self.m, self.n, self.k, self.r, self.slots, self.slices = m, n, k, r, slots, slices
        self.q, self.st = quantize_nf4(rand(n, k))
        self.x = rand(m, k, std=1.0)
        self.a, self.b = rand(slots, slices * r, k), rand(slots, n, r)
        if routes == "together":
            at = torch.repeat_interleave(torch.arange(-1, slots), -(-m // (slots + 1)))[:m]
        else:
            at = torch.arange(m) % (slots + 1) - 1
        self.routes = at.int().to(device)
        i64, i32 = dict(dtype=torch.int64, device=device), dict(dtype=torch.int32, device=device)
        self.bounds = [n * s // slices for s in range(slices + 1)]
        stride = 1 << (r - 1).bit_length()
        padded = torch.zeros(slots, n, stride, dtype=torch.bfloat16, device=device)
        padded[:, :, :r] = self.b
        self.lora = LoraBatch(
            a_store=self.a.reshape(-1), a_offsets=torch.arange(slots, **i64) * (slices * r * k),
            b_store=padded.reshape(-1), b_offsets=torch.arange(slots, **i64) * (n * stride),
            b_strides=torch.full((slots,), stride, **i32), ranks=torch.full((slots,), r, **i32),
            scales=torch.linspace(1.0, 2.0, slots, device=device), token_slots=self.routes,
            slice_offsets=torch.tensor(self.bounds, **i32), max_rank=r)

    def expected(self, lora=True, swiglu=False):
        rnd = lambda t: t.bfloat16().float()
        w = dequantize_nf4(self.q, self.st.absmax, self.st.code, (self.n, self.k)).float()
        y = rnd(self.x.float() @ w.t())
        if lora:
            for g in range(self.slots):
                rows = self.routes == g
                z = rnd(self.x[rows].float() @ self.a[g].float().t())
                scale = self.lora.scales[g].float()
                for s in range(self.slices):
                    lo, hi = self.bounds[s], self.bounds[s + 1]
                    delta = rnd(scale * (z[:, s * self.r : (s + 1) * self.r] @ self.b[g, lo:hi].float().t()))
                    y[rows, lo:hi] = rnd(y[rows, lo:hi] + delta)
        if swiglu:
            gate, up = y.chunk(2, 1)
            y = rnd(rnd(gate * torch.sigmoid(gate)) * up)
        return y


def near(y, want):
    """A bf16 result whose fp32 sums run in another order: one rounding of y and one of z and of the delta."""
    err = (y.float() - want).abs()
    assert (err.norm() / want.norm()).item() < 0.005
    assert bool((err <= 2e-2 + 2e-2 * want.abs()).all())


@pytest.mark.parametrize(
    "m,n,rows",
    [
        (300, 16384, 128),
        (380, 24576, 192),  # 2 x 96 tiles
        (520, 16320, 192),  # a last column tile of 192 columns
        (2000, 8192, 256),  # z in a launch of its own
    ],
)
def test_tall_tiles_against_torch(m, n, rows, device):
    p = Problem(m, n, 256, device)
    assert plan_of(m, n, 256, p.lora).tile_rows == rows
    near(nf4_lora_linear(p.x, p.q, p.st, lora=p.lora, plan="prefill"), p.expected())


WIDE_N = 16320  # 63.75 column tiles: three or four row tiles of one height fill the chip once
STAGES = {192: "1.5", 320: "2.5", 896: "7", 1088: "8.5"}  # of 128 k: odd counts, a 64-k tail, rings that wrap


@pytest.mark.parametrize("k", STAGES)
@pytest.mark.parametrize("rows,m", [(64, 250), (96, 380), (128, 450), (160, 600), (192, 700), (256, 1000)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_every_height(swiglu, rows, m, k, device):
    """Every tile height without adapters, with a ragged last row of tiles and last column tile."""
    n = WIDE_N + 64 if swiglu else WIDE_N
    p = Problem(m, n, k, device, slots=1)
    assert plan_of(m, n, k, None, swiglu).tile_rows == rows
    near(nf4_lora_linear(p.x, p.q, p.st, swiglu=swiglu, plan="prefill"), p.expected(False, swiglu))


@pytest.mark.parametrize("k", STAGES)
@pytest.mark.parametrize("rows", [64, 96, 128, 160, 192, 256])
@pytest.mark.parametrize("swiglu", [False, True])
def test_every_height_with_adapters(swiglu, rows, k, device):
    n, m = WIDE_N + 64 if swiglu else WIDE_N, 3 * rows - 10
    p = Problem(m, n, k, device, slots=1, slices=2 if swiglu else 1)
    assert plan_of(m, n, k, p.lora, swiglu).tile_rows == rows
    near(nf4_lora_linear(p.x, p.q, p.st, lora=p.lora, swiglu=swiglu, plan="prefill"), p.expected(True, swiglu))


@pytest.mark.parametrize("m,k,rows,slots", [(182, 320, 64, 12), (278, 192, 96, 12), (374, 896, 128, 12), (470, 1088, 160, 3)])
@pytest.mark.parametrize("r,slices", [(3, 1), (33, 3), (16, 3)])
def test_slots_in_turn(m, k, rows, slots, r, slices, device):
    """Slots in turn among the tokens, slice bounds inside a wave's columns."""
    n = WIDE_N
    p = Problem(m, n, k, device, r=r, slots=slots, slices=slices, routes="in turn")
    p.bounds = [0, n] if slices == 1 else [0, n // 3 + 5, n - 70, n]
    p.lora.slice_offsets = torch.tensor(p.bounds, dtype=torch.int32, device=device)
    assert plan_of(m, n, k, p.lora).tile_rows == rows
    near(nf4_lora_linear(p.x, p.q, p.st, lora=p.lora, plan="prefill"), p.expected())


@pytest.mark.parametrize("m,rows", [(182, 64), (278, 96), (374, 128), (470, 160)])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), -3.0e38])
def test_an_infinite_b_reaches_its_own_slot_only(m, rows, value, device):
    """Slots that share an expand pass multiply each other's B with zeros."""
    n, k = WIDE_N, 320
    p = Problem(m, n, k, device, slots=9, routes="in turn")
    assert plan_of(m, n, k, p.lora).tile_rows == rows
    good = nf4_lora_linear(p.x, p.q, p.st, lora=p.lora, plan="prefill")
    bad = p.lora.b_store.clone().reshape(9, n, 16)
    bad[4, 100:300, 7] = value
    p.lora.b_store = bad.reshape(-1)
    y = nf4_lora_linear(p.x, p.q, p.st, lora=p.lora, plan="prefill")
    own = p.routes == 4
    assert torch.equal(y[~own], good[~own])
    assert torch.equal(y[own][:, :100], good[own][:, :100]) and torch.equal(y[own][:, 300:], good[own][:, 300:])
    changed = y[own][:, 100:300].float()
    assert not torch.isfinite(changed).any() if value != -3.0e38 else bool((changed.abs() > 1e30).all())


@pytest.mark.parametrize("m,n,k,r", [(2048, 8192, 1024, 16), (1024, 16384, 512, 16), (1024, 16384, 1024, 16)])
def test_producers_in_a_launch_of_their_own(m, n, k, r, device):
    """z from its own launch (another summation order than in the GEMM launch)."""
    p = Problem(m, n, k, device, r=r)
    assert plan_of(m, n, k, p.lora).z_launch == 1
    near(nf4_lora_linear(p.x, p.q, p.st, lora=p.lora, plan="prefill"), p.expected())
    workspace_clean(device)


# Producers in a launch of their own; and in the GEMM launch, fewer than a tile has units of 16 tokens, so of 32.
WITHHELD = [(1024, 16384, 256, 1, 16, True), (1024, 16384, 256, 3, 16, True), (700, 5120, 1088, 1, 16, False),
            (1350, 4096, 576, 3, 33, False), (2048, 5120, 320, 2, 33, False)]


@pytest.mark.parametrize("routes", ["together", "in turn"])
@pytest.mark.parametrize("m,n,k,slices,r,launch", WITHHELD)
def test_producers_and_their_recomputation(m, n, k, slices, r, launch, routes, device):
    """Without flags the GEMM launch's bounded waits run out and its tiles recompute every z row: the same
    bits where the producers are in that launch."""
    p = Problem(m, n, k, device, slices=slices, r=r, routes=routes)
    plan = plan_of(m, n, k, p.lora)
    assert plan.z_launch == launch and (launch or plan.z_parts < plan.tile_rows // 16)
    weight, keep = _weight_struct(p.q, p.st, None, n, k, device, m)
    lora = _lora_struct(p.lora, m, k, n, device)
    need = workspace_bytes(m, n, k, num_slices=slices, max_rank=r)
    ws = torch.zeros(need, dtype=torch.uint8, device=device)
    lib, stream = _lib.library(), _lib.stream_of(device)
    out = []
    for withhold in (0, _lib.LF_TEST_WITHHOLD_PARTIALS):
        y = torch.zeros(m, n, dtype=torch.bfloat16, device=device)
        _lib.check(lib.lf_nf4_lora_linear(p.x.data_ptr(), m, k, weight, None, lora, y.data_ptr(), n, ws.data_ptr(), need,
                                          _lib.LF_PLAN_PREFILL | withhold, stream))
        status = ctypes.c_int32(-1)
        _lib.check(lib.lf_nf4_lora_status(ws.data_ptr(), stream, ctypes.byref(status)))
        assert status.value == (1 if withhold else 0)
        near(y, p.expected())
        out.append(y)
    assert launch or torch.equal(*out)
    del keep
