"""The kernel and tiles that a fused linear takes (``lf_nf4_lora_plan``: host arithmetic, CPU only)."""

import ctypes
import math
import random

import pytest

from loraforge_amd import _lib


def plan_of(m, n, k, slices=0, rank=1, slots=0, flags=0):
    plan = _lib.Plan()
    _lib.check(_lib.library().lf_nf4_lora_plan(m, n, k, slices, rank, slots, flags, ctypes.byref(plan)))
    return plan


@pytest.mark.parametrize("m", [1024, 1500, 2048, 4096])
@pytest.mark.parametrize("n,k", [(4096, 4096), (11008, 4096), (4096, 11008), (5120, 8192), (24576, 4096)])
@pytest.mark.parametrize("slices,rank", [(1, 8), (1, 16), (1, 32), (1, 64), (2, 16), (2, 32), (2, 64), (3, 16), (3, 64)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_z_producers_keep_up_with_the_tiles(m, n, k, slices, rank, swiglu):
    """What z producers inside the GEMM launch take beyond the first round's k-loop, which their tiles
    wait for, is at most a fifth of all rounds' (nine tenths above 64 A rows a slot; eight prompts of
    equal length)."""
    if swiglu and slices != 2:
        pytest.skip("a SwiGLU output has two slices")
    plan = plan_of(m, n, k, slices, rank, 8, _lib.LF_PLAN_PREFILL | (_lib.LF_SWIGLU_OUTPUT if swiglu else 0))
    if plan.z_launch:
        return
    size = 16
    units = math.ceil(plan.tile_rows / size + 0.5 * (1 + 8 * plan.tile_rows / m))
    if units > plan.z_parts:  # then they are of 32 tokens
        size = 32
        units = math.ceil(plan.tile_rows / size + 0.5 * (1 + 8 * plan.tile_rows / m))
    row_tiles = math.ceil(slices * rank / 16)
    # A unit takes 3.7 us per 4096 of K for each 16 A rows and, in each pass of 64 of them, for each 16 tokens, the
    # k-loop 10 us per 32 tokens (and no less than 47 us, for the decode of the weights).
    z_us = math.ceil(units / plan.z_parts) * 3.7 * (math.ceil(row_tiles / 4) * size / 16 + row_tiles)
    loop_us = max(47.0, 10.0 * plan.tile_rows / 32)
    tiles = math.ceil(m / plan.tile_rows) * math.ceil(n / 256)
    share = 0.2 if row_tiles <= 4 else 0.9
    assert z_us - loop_us <= share * loop_us * math.ceil(tiles / 256), (plan.tile_rows, plan.z_parts)


def test_refusals():
    for bad in (dict(m=0), dict(n=100), dict(k=0), dict(slices=4), dict(slices=1, rank=65)):
        with pytest.raises(ValueError):
            plan_of(**{**dict(m=128, n=256, k=256), **bad})


# Without adapters, and with: calls whose K is short against their tiles' fixed time.
SHORT = [(2048, 18944, 64, 0), (4096, 24576, 64, 0), (512, 24576, 128, 0), (2048, 8192, 256, 0), (430, 13312, 384, 1), (1024, 24576, 192, 1)]


@pytest.mark.parametrize("m,n,k,slices", SHORT)
def test_short_k_stays_on_the_prefill_gemm(m, n, k, slices):
    """Its exact weights, and up to twelve times its speed: rounds of decode workgroups have a fixed part."""
    assert plan_of(m, n, k, slices, 16, 8 * slices).kernel == _lib.LF_KERNEL_PREFILL


def _exact_before(m, n, k, slices, rank):
    """Calls above 64 tokens that are too many, or too long, for the decode kernels by the bound on where
    they may take a default call: 256 x 192 tiles at 85 us a round per 4096 of K."""
    rounds = math.ceil(math.ceil(m / 256) * math.ceil(n / 192) / 256)
    tiles_us = rounds * 85.0 * k / 4096
    decode_rounds = math.ceil(math.ceil(n / 32 / 8) * 8 * math.ceil(m / 32) / 256)
    chunks_us = math.ceil(m / 64) * ((6.0 if slices else 0.0) + n * k * 0.5625 / 0.8e6)
    return decode_rounds * 4.0 * k / 4096 >= tiles_us and chunks_us >= tiles_us + (20.0 if slices else 0.0)


def test_no_default_call_leaves_the_exact_weights():
    rng = random.Random(5)
    for _ in range(20000):
        log = lambda lo, hi: math.exp(rng.uniform(math.log(lo), math.log(hi)))
        m, n, k = int(log(65, 8192)), 64 * max(1, round(log(256, 40000) / 64)), 64 * max(1, round(log(64, 16384) / 64))
        slices, rank, slots = rng.choice((0, 1, 2, 3)), rng.choice((4, 16, 64)), rng.choice((0, 1, 8, 32, 128))
        if _exact_before(m, n, k, slices, rank):
            assert plan_of(m, n, k, slices, rank, slots).kernel == _lib.LF_KERNEL_PREFILL, (m, n, k, slices, rank, slots)


def two_launches(m, n, k, slices, rank, slots):
    two = ctypes.c_int32()
    _lib.check(_lib.library().lf_lora_apply_plan(m, n, k, slices, rank, slots, ctypes.byref(two)))
    return bool(two.value)


# Launches of the decode kernel that run in one round of workgroups: faster than the two launches over all tokens up to
# these sizes, by tokens in turn and by the mean of tokens in turn and in runs.
@pytest.mark.parametrize(
    "m,n,k,slices,rank,slots,two",
    [
        (65, 4096, 4096, 1, 16, 1, True), (65, 4096, 4096, 1, 16, 4, False), (65, 2048, 8192, 1, 16, 4, False),
        (128, 4096, 4096, 1, 16, 4, False), (128, 2048, 8192, 1, 16, 4, False), (128, 4096, 4096, 1, 64, 4, True),
        (192, 4096, 4096, 1, 16, 4, True), (192, 4096, 4096, 1, 16, 8, False), (192, 2048, 8192, 1, 16, 8, False),
        (192, 4096, 4096, 1, 64, 8, True), (256, 4096, 4096, 1, 16, 8, True), (500, 5120, 4096, 3, 16, 4, True),
        (64, 4096, 4096, 1, 16, 4, False), (500, 4096, 4096, 1, 16, 17, False),
    ],
)
def test_lora_apply_launches(m, n, k, slices, rank, slots, two):
    assert two_launches(m, n, k, slices, rank, slots) == two


def test_lora_apply_plan_refusals():
    for bad in (dict(m=0), dict(n=100), dict(k=0), dict(slices=0), dict(slices=4), dict(rank=65)):
        with pytest.raises(ValueError):
            two_launches(**{**dict(m=128, n=256, k=256, slices=1, rank=16, slots=4), **bad})
