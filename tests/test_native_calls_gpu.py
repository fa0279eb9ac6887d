"""The operators' native call path (``csrc/host/binding.cpp``) against their Python path.

Every form the native path takes must give the Python path's bits, and every
call it declines must be served, or refused with the same error, as before:
the second call of a shape runs natively, a call with ``workspace=`` or with
the native path switched off runs in Python.
"""

import contextlib
import ctypes
import dataclasses
import threading
import types

import pytest
import torch

from loraforge_amd import _lib
from loraforge_amd.ops import (
    LoraBatch,
    dequantize_nf4,
    dequantize_nf4_nested,
    lora_apply,
    nf4_lora_linear,
    quantize_nf4,
    row_expand,
    row_shrink,
)
from tests import _cases
from tests.test_fused_gpu import to_device

pytestmark = pytest.mark.gpu


class _Declines:
    """Stands in for the binding: every call goes the Python way."""

    def __getattr__(self, name):
        return lambda *args: None


class _Noting:
    """The binding, noting which calls it took."""

    def __init__(self, module):
        self.module, self.took = module, []

    def __getattr__(self, name):
        def call(*args):
            answer = getattr(self.module, name)(*args)
            self.took.append(answer is not None)
            return answer

        return call


@contextlib.contextmanager
def standing_in(**replaced):
    """The native call path with other entry points (addresses by name)."""
    _lib.bind(_lib.binding(), **replaced)
    try:
        yield
    finally:
        _lib.bind(_lib.binding())


def both(monkeypatch, call, native=True):
    """``call``'s result on the native path (which has to take it, or with native=False to decline) and in Python."""
    call()  # warms the device flags and the workspace
    with monkeypatch.context() as patch:
        noting = _Noting(_lib.binding())
        patch.setattr(_lib, "_binding_module", noting)
        taken = call()
    assert noting.took and set(noting.took) == {native}
    with monkeypatch.context() as patch:
        patch.setattr(_lib, "_binding_module", _Declines())
        python = call()
    torch.cuda.synchronize()
    return taken, python


@pytest.mark.parametrize("dq", [False, True])
@pytest.mark.parametrize("m,lead,swiglu,bias", [(1, None, False, True), (6, (2, 3), False, False), (9, None, True, False),
                                                (80, None, True, False), (96, (3, 32), False, True)])
def test_linear_forms(m, lead, swiglu, bias, dq, device, monkeypatch):
    bounds = [0, 256, 512] if swiglu else None
    case = _cases.fused_case(m, 512, 320, ranks=(16, 8, 4), slices=2 if swiglu else 1, bounds=bounds, double_quant=dq,
                             bias=bias, seed=400 + m)
    x, q, st, lora, b = to_device(case, device)
    x = x if lead is None else x.reshape(*lead, -1)
    wide = torch.zeros(m, x.shape[-1] + 64, dtype=torch.bfloat16, device=device)
    forms = [dict(lora=lora), dict(lora=None), dict(lora=lora, exact=True), dict(lora=lora, plan="decode")]
    if dq:
        forms.append(dict(lora=lora, scales="nested"))
    for kw in forms:
        taken, python = both(monkeypatch, lambda: nf4_lora_linear(x, q, st, bias=b, swiglu=swiglu, **kw))
        assert taken.shape == python.shape and torch.equal(taken, python), kw
    if lead is None:
        strided = wide[:, : x.shape[-1]].copy_(x)
        taken, python = both(monkeypatch, lambda: nf4_lora_linear(strided, q, st, bias=b, swiglu=swiglu, lora=lora))
        assert torch.equal(taken, python)
        out = torch.empty(m, 520, dtype=torch.bfloat16, device=device)[:, : 256 if swiglu else 512]
        taken, python = both(monkeypatch, lambda: nf4_lora_linear(x, q, st, bias=b, swiglu=swiglu, lora=lora, out=out).clone(),
                             native=not (swiglu and m > 64))  # (such an output has alignment rules of its own)
        assert torch.equal(taken, python)


def test_prepared_scales_follow_an_update(device, monkeypatch):
    """A nested state whose tensors change in place is prepared again, not served from the cached scales."""
    case = _cases.fused_case(4, 256, 512, ranks=(8,), double_quant=True, seed=431)
    x, q, st, lora, _ = to_device(case, device)
    before, _ = both(monkeypatch, lambda: nf4_lora_linear(x, q, st, lora=lora))
    st.state2.absmax.mul_(2.0)
    after, python = both(monkeypatch, lambda: nf4_lora_linear(x, q, st, lora=lora))
    assert torch.equal(after, python) and not torch.equal(after, before)


def test_row_operators_and_dequant(device, monkeypatch):
    c = _cases.c2_case(seed=441, tokens=24, k=512, n=256, adapters=4)
    t = lambda a: torch.from_numpy(a.view("int16") if a.dtype == "uint16" else a).to(device)
    bf = lambda a: t(a).view(torch.bfloat16)
    x, a, b = bf(c["x"]), bf(c["a"]), bf(c["b"])
    routes = t(c["routes"])
    meta = {k: t(v) for k, v in c["meta"].items()}

    def rows():
        z, y = bf(c["z"]).clone(), bf(c["y"]).clone()
        row_shrink(x, a, z, routes, meta["ranks"], max_rank=16)
        row_expand(z, b, y, **meta)
        return torch.cat([z.reshape(-1), y.reshape(-1)])

    taken, python = both(monkeypatch, rows)
    assert torch.equal(taken, python)
    case = _cases.fused_case(24, 256, 512, ranks=(16, 8), seed=442)
    xl, q, st, lora, _ = to_device(case, device)
    base = torch.randn(24, 256, device=device).bfloat16()
    taken, python = both(monkeypatch, lambda: lora_apply(xl, base.clone(), lora))
    assert torch.equal(taken, python)
    taken, python = both(monkeypatch, lambda: dequantize_nf4(q, st.absmax, st.code, (256, 512)))
    assert torch.equal(taken, python)


@pytest.mark.parametrize("n,k", [(64, 64), (192, 320), (4096, 8192)])
def test_nested_dequant_checks_the_codebook(n, k, device, monkeypatch):
    """Below and at the four-step size (32 M elements): bits of the Python path; a codebook with one other
    value is refused, and so is the next call with it."""
    g = torch.Generator(device=device).manual_seed(n + k)
    q, st = quantize_nf4((torch.randn(n, k, generator=g, device=device) * 0.02).bfloat16(), compress_statistics=True)
    taken, python = both(monkeypatch, lambda: dequantize_nf4_nested(q, st))
    assert torch.equal(taken, python)
    wrong = dataclasses.replace(st, code=st.code.clone())
    wrong.code[11] += 1e-6
    for _ in range(2):
        with pytest.raises(ValueError, match="canonical"):
            dequantize_nf4_nested(q, wrong)
    assert torch.equal(dequantize_nf4_nested(q, st), python)


def test_refusals_are_the_python_path_s(device):
    """What the operators refuse they refuse after native calls too, with their own messages."""
    case = _cases.fused_case(4, 256, 512, ranks=(8, 4), seed=451)
    x, q, st, lora, _ = to_device(case, device)
    for _ in range(2):
        good = nf4_lora_linear(x, q, st, lora=lora)
    with pytest.raises(ValueError, match="inference-only"):
        nf4_lora_linear(x.clone().requires_grad_(), q, st, lora=lora)
    with pytest.raises(ValueError, match="unit column stride"):
        nf4_lora_linear(x[:, ::2], q, st, lora=lora)
    with pytest.raises(ValueError, match="share storage"):
        nf4_lora_linear(x, q, st, out=x[:, :256])
    with pytest.raises(ValueError, match="token_slots"):
        nf4_lora_linear(x, q, st, lora=lora.with_tokens(lora.token_slots[:2]))
    with pytest.raises(ValueError, match="nested"):
        nf4_lora_linear(x, q, st, scales="nested")
    with pytest.raises(ValueError, match="16-entry"):
        dequantize_nf4(q, st.absmax, st.code[:8], (256, 512))
    assert torch.equal(nf4_lora_linear(x, q, st, lora=lora), good)


def operators(device):
    """Each operator with a native path, as a function that says whether that path took the call."""
    case = _cases.fused_case(4, 256, 512, ranks=(8, 4), seed=461)
    x, q, st, lora, _ = to_device(case, device)
    y = torch.zeros(4, 256, dtype=torch.bfloat16, device=device)
    nested = _cases.fused_case(4, 256, 512, ranks=(8,), double_quant=True, seed=462)
    _, q2, st2, _, _ = to_device(nested, device)
    c = _cases.c2_case(seed=463, tokens=24, k=512, n=256, adapters=4)
    t = lambda a: torch.from_numpy(a.view("int16") if a.dtype == "uint16" else a).to(device)
    bf = lambda a: t(a).view(torch.bfloat16)
    rx, a, b, z, ry, routes = bf(c["x"]), bf(c["a"]), bf(c["b"]), bf(c["z"]), bf(c["y"]), t(c["routes"])
    meta = {k: t(v) for k, v in c["meta"].items()}
    order = ("b_offsets", "b_strides", "ranks", "scales", "segment_indptr", "segment_slots", "token_indices", "slice_offsets",
             "segment_count")
    # A first call of each through its Python path: device flags, workspaces.
    nf4_lora_linear(x, q, st, lora=lora)
    lora_apply(x, y, lora)
    row_shrink(rx, a, z, routes, meta["ranks"], max_rank=16)
    row_expand(z, b, ry, **meta)
    dequantize_nf4(q, st.absmax, st.code, (256, 512))
    dequantize_nf4_nested(q2, st2)
    native = _lib.binding()
    return {
        "lf_nf4_lora_linear": lambda: native.linear(x, q, st, None, None, lora, None, False, False, 0),
        "lf_lora_apply": lambda: native.apply(x, y, lora),
        "lf_row_shrink": lambda: native.shrink(rx, a, z, routes, meta["ranks"], 1, 16),
        "lf_row_expand": lambda: native.expand(z, b, ry, *(meta[k] for k in order), None, 256),
        "lf_nf4_dequant": lambda: native.dequant(q, st.absmax, st.code, (256, 512)),
        "lf_nf4_dequant_dq_checked": lambda: native.dequant_nested(q2, st2),
    }


def test_library_calls_run_without_the_gil(device):
    """In the library's place stands PyGILState_Check, whose answer reads as a status: 0 (no GIL held)
    is LF_OK, 1 LF_EINVAL, on which the native path declines. (The checked dequantisation then finds
    its unset answer not canonical and declines too.)"""
    check = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    for name, call in operators(device).items():
        assert call() is not None, name
        with standing_in(**{name: check}):
            assert (call() is not None) or name == "lf_nf4_dequant_dq_checked", name


def test_threads_on_one_stream_share_its_workspace(device):
    """Calls of several launches that hand z rows over in the cached workspace, from threads on one
    stream: each keeps its launches together."""
    cases = [_cases.fused_case(m, 512, 2048, ranks=(16, 8, 4), seed=470 + m) for m in (200, 270, 330)]
    jobs = []
    for case in cases:
        x, q, st, lora, _ = to_device(case, device)
        base = torch.randn(case["m"], 512, device=device).bfloat16()
        want = lora_apply(x, base.clone(), lora)
        jobs.append((x, base, lora, want))
    torch.cuda.synchronize()
    wrong = []

    def work(x, base, lora, want):
        for _ in range(100):
            if not torch.equal(lora_apply(x, base.clone(), lora), want):
                wrong.append(x.shape)

    threads = [threading.Thread(target=work, args=job) for job in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_hip_errors_carry_the_library_s_text(device):
    """A library call that fails with a HIP error raises lf_last_error()'s text, as the Python path does."""
    status = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: _lib.LF_EHIP)
    words = ctypes.create_string_buffer(b"hipLaunchKernel failed: out of memory")
    text = ctypes.CFUNCTYPE(ctypes.c_void_p)(lambda: ctypes.addressof(words))
    address = lambda fn: ctypes.cast(fn, ctypes.c_void_p).value
    for name, call in operators(device).items():
        with standing_in(**{name: address(status), "lf_last_error": address(text)}):
            with pytest.raises(RuntimeError, match="hipLaunchKernel failed: out of memory"):
                call()


def test_other_batches_go_the_python_way(device):
    """The native path reads LoraBatch itself; an object with a num_slices of its own, or without one, is
    served or refused by the Python path."""

    class Disagreeing(LoraBatch):
        num_slices = 2

    case = _cases.fused_case(4, 256, 512, ranks=(8, 4), seed=465)
    x, q, st, lora, _ = to_device(case, device)
    want = nf4_lora_linear(x, q, st, lora=lora)
    fields = {f.name: getattr(lora, f.name) for f in dataclasses.fields(lora)}
    same = type("Same", (LoraBatch,), {})(**fields)
    assert torch.equal(nf4_lora_linear(x, q, st, lora=same), want)
    for _ in range(2):
        with pytest.raises(ValueError, match="slice_offsets length disagrees"):
            nf4_lora_linear(x, q, st, lora=Disagreeing(**fields))
        with pytest.raises(ValueError, match="slice_offsets length disagrees"):
            lora_apply(x, torch.zeros(4, 256, dtype=torch.bfloat16, device=device), Disagreeing(**fields))
        with pytest.raises(AttributeError, match="num_slices"):
            nf4_lora_linear(x, q, st, lora=types.SimpleNamespace(**fields))
    assert torch.equal(nf4_lora_linear(x, q, st, lora=lora), want)
