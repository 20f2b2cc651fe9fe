"""The fused MLP's native calls (csrc/host_path.cpp) against the same launches issued one by one from Python, at ranks 16
and 32, with and without the output and dx: every result bit for bit."""
import pytest
import torch

import fused_linear
import fused_mlp
import mxfp8
import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r", [16, 32])
@pytest.mark.parametrize("T,K,N", [(1, 256, 384), (300, 512, 768), (1000, 512, 1536)])
@pytest.mark.parametrize("need_out,need_x", [(True, True), (False, True), (True, False)])
def test_native_calls_give_the_same_bits(T, K, N, r, need_out, need_x, gpu, monkeypatch):
    monkeypatch.setitem(workloads.CONFIGS, 63, dict(name="n", T=T, K=K, N=N, r=r, alpha=32, backward=True, layers=1))
    model, inps = workloads.build_model(63, T=T, device=gpu)
    mxfp8.enable_mxfp8(model)
    mod = model.layers[0].mlp
    x, dy = inps[0]["x"].to(gpu), inps[0]["dy"].to(gpu)
    taken = []

    def step():
        fused_linear.new_step()
        for p in model.parameters():
            p.grad = None
        xi = x.clone().requires_grad_(need_x)
        y = fused_mlp.mlp(mod, xi, need_out=need_out)
        y.backward(dy)
        out = [p.grad for n in ("gate_proj", "up_proj", "down_proj") for p in getattr(mod, n).parameters() if p.requires_grad]
        return out + [y.detach()] * need_out + [xi.grad] * need_x

    for name in ("_fwd_in_one_call", "_bwd_in_one_call"):
        real = getattr(fused_mlp, name)
        monkeypatch.setattr(fused_mlp, name, lambda *a, real=real, name=name: taken.append((name, real(*a))) or real(*a))
    native = step()
    assert taken == [("_fwd_in_one_call", True), ("_bwd_in_one_call", True)]
    monkeypatch.setattr(fused_mlp, "_fwd_in_one_call", lambda *a: False)
    monkeypatch.setattr(fused_mlp, "_bwd_in_one_call", lambda *a: False)
    python = step()
    assert len(native) == len(python) == 6 + need_out + need_x
    for k, (a, b) in enumerate(zip(native, python)):
        assert a.dtype == b.dtype and torch.equal(a, b), k
