"""Memory that the fused MLP holds at its peak: the native calls (csrc/host_path.cpp) against the same launches from
Python with one tensor for every temporary, dropped after its last reader."""
import pytest
import torch

import fused_linear
import fused_mlp
import mxfp8
import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,N,r", [(4096, 1024, 3584, 16), (4096, 1024, 3584, 32), (3000, 2048, 2048, 16),
                                     (1000, 2048, 6144, 32)])
@pytest.mark.parametrize("need_out,need_x", [(True, True), (False, True), (True, False)])
def test_peak_of_a_pass(T, K, N, r, need_out, need_x, gpu, monkeypatch):
    monkeypatch.setitem(workloads.CONFIGS, 63, dict(name="m", T=T, K=K, N=N, r=r, alpha=32, backward=True, layers=1))
    model, inps = workloads.build_model(63, T=T, device=gpu)
    mxfp8.enable_mxfp8(model)
    mod = model.layers[0].mlp
    x, dy = inps[0]["x"].to(gpu), inps[0]["dy"].to(gpu)

    def peak_of(call):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        base = torch.cuda.memory_stats()
        out = call()
        # the bytes asked for (a block handed out may be up to 1 MB larger, by what the allocator has at hand)
        return out, torch.cuda.memory_stats()["requested_bytes.all.peak"] - base["requested_bytes.all.current"]

    def peaks():
        fused_linear.new_step()
        for p in model.parameters():
            p.grad = None
        xi = x.clone().requires_grad_(need_x)
        y, fwd = peak_of(lambda: fused_mlp.mlp(mod, xi, need_out=need_out))
        return fwd, peak_of(lambda: y.backward(dy))[1]

    peaks()  # what is kept from call to call
    native = peaks()
    monkeypatch.setattr(fused_mlp, "_fwd_in_one_call", lambda *a: False)
    monkeypatch.setattr(fused_mlp, "_bwd_in_one_call", lambda *a: False)
    peaks()
    python = peaks()
    slack = 256 * 32  # pieces of one allocation start at multiples of 256 bytes
    assert native[0] <= python[0] + slack and native[1] <= python[1] + slack, (native, python)
