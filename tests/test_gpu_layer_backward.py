"""The per-layer backward of a group without a concatenated Wᵀ (fused_linear._native_backward: lora_bwd, MX GEMMs with
dS·S in the last one's epilogue, the token reduction) against _plain_backward, the same sums as torch products.  Both
round every result to bf16 or better from the same bf16 operands; the torch path also rounds dB and d(xa) to bf16 before
their scale: at most two roundings of 2^-9 on either side, so 2^-7 normwise."""
import pytest
import torch

import fused_linear
import mxfp8
import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r,T,names", [(16, 300, ("gate_proj", "up_proj")), (32, 129, ("gate_proj", "up_proj")),
                                       (16, 1000, ("down_proj",)), (32, 31, ("down_proj",))])
@pytest.mark.parametrize("need_x", [True, False])
def test_matches_the_torch_products(r, T, names, need_x, gpu, monkeypatch):
    monkeypatch.setitem(workloads.CONFIGS, 63, dict(name="u", T=T, K=512, N=768, r=r, alpha=32, backward=True, layers=1))
    model, _ = workloads.build_model(63, T=T, device=gpu)
    monkeypatch.setattr(mxfp8, "FUSE_GU", False)
    mxfp8.enable_mxfp8(model)
    mods = [getattr(model.layers[0].mlp, n) for n in names]
    g = torch.Generator(device=gpu).manual_seed(T)
    x = torch.randn(T, mods[0].base_layer.in_features, device=gpu, generator=g).to(torch.bfloat16)
    dys = [(torch.randn(T, m.base_layer.out_features, device=gpu, generator=g) * 1e-2).to(torch.bfloat16) for m in mods]

    def run():
        fused_linear.new_step()
        for p in model.parameters():
            p.grad = None
        xi = x.clone().requires_grad_(need_x)
        torch.autograd.backward(list(fused_linear.group_linear(xi, mods)), dys)
        return [p for m in mods for p in (m.lora_A["default"].weight.grad, m.lora_B["default"].weight.grad)] + [
            xi.grad] * need_x

    calls, real = [], fused_linear._native_backward
    monkeypatch.setattr(fused_linear, "_native_backward", lambda *a: calls.append(1) or real(*a))
    got = run()
    assert calls
    monkeypatch.setattr(fused_linear, "_native_per_layer", lambda *a: None)
    want = run()
    for k, (a, b) in enumerate(zip(got, want)):
        assert a.dtype == b.dtype and ((a.double() - b.double()).norm() <= 2.0 ** -7 * b.double().norm()), k
