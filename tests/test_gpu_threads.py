"""The native host module runs its calls without the interpreter's lock (csrc/host_path.cpp): a launch may wait for room in
its stream's queue, and the program's other Python threads (data loading, logging) go on meanwhile.  With a switch
interval of minutes the lock changes hands only where its holder gives it up, so another thread counts during a loop of
calls only if the calls release it (their results are kept: freeing a tensor releases it too)."""
import sys
import threading
import time

import pytest
import torch

import _native
import mxfp8

pytestmark = pytest.mark.gpu


def _calls(gpu):
    h, T, K = _native.host(), 16, 128
    x = torch.randn(T, K, device=gpu).to(torch.bfloat16)
    w = torch.randn(16, K, device=gpu).to(torch.bfloat16)
    q, s = mxfp8.mx_quant_tiled(x)
    qw, sw = mxfp8.mx_quant_tiled(torch.randn(128, K, device=gpu).to(torch.bfloat16))
    st = _native.stream_of(x)
    return {"quant_rows": lambda: h.quant_rows(x, st), "quant_tiled": lambda: h.quant_tiled(x, st),
            "quant_lora": lambda: h.quant_lora(x, w, 1.0, True, st),
            "gemm": lambda: h.gemm(q, s, qw, sw, None, None, None, 1.0, 3, T, st)}


@pytest.mark.parametrize("name", ["quant_rows", "quant_tiled", "quant_lora", "gemm"])
def test_other_threads_run_during_native_calls(name, gpu):
    call = _calls(gpu)[name]
    call()
    torch.cuda.synchronize()
    count, stop, ready = [0], [False], threading.Event()

    def other():
        ready.set()
        while not stop[0]:
            count[0] += 1
            time.sleep(0)  # gives the lock back at once

    before = sys.getswitchinterval()
    t = threading.Thread(target=other)
    sys.setswitchinterval(300.0)
    try:
        t.start()
        ready.wait()
        first, kept = count[0], []
        while count[0] < first + 3 and len(kept) < 5000:
            kept.append(call())
        seen = count[0] - first
    finally:
        stop[0] = True
        sys.setswitchinterval(before)
        t.join()
        torch.cuda.synchronize()
    assert seen >= 3
