"""Checked nested dequantisation: calls of several threads and streams in flight at a time."""

import threading
import time

import pytest
import torch

from loraforge_amd.ops import dequantize_nf4_nested, quantize_nf4

pytestmark = pytest.mark.gpu


def test_a_waiting_call_keeps_its_answer(device):
    """One call waits behind a stream's long work (and has more of it behind itself) while another
    thread makes several times 256 calls on another stream."""
    g = torch.Generator(device=device).manual_seed(7)
    q, st = quantize_nf4((torch.randn(256, 512, generator=g, device=device) * 0.02).bfloat16(), compress_statistics=True)
    want = dequantize_nf4_nested(q, st)
    side = torch.cuda.Stream()
    # About 30 ms of waiting, by the clock that the sleep kernel counts.
    start, stop = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    start.record()
    torch.cuda._sleep(1_000_000)
    stop.record()
    torch.cuda.synchronize()
    cycles = int(1_000_000 * 30.0 / start.elapsed_time(stop))
    for _ in range(3):
        result = []

        def waiting():
            with torch.cuda.stream(side):
                try:
                    result.append(dequantize_nf4_nested(q, st))
                except RuntimeError as error:
                    result.append(error)

        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            torch.cuda._sleep(cycles)
        thread = threading.Thread(target=waiting)
        thread.start()
        time.sleep(0.0003)
        with torch.cuda.stream(side):
            torch.cuda._sleep(2 * cycles)
        until = time.monotonic() + 0.08
        while time.monotonic() < until:
            assert torch.equal(dequantize_nf4_nested(q, st), want)
        thread.join()
        torch.cuda.synchronize()
        assert torch.is_tensor(result[0]) and torch.equal(result[0], want), result[0]
