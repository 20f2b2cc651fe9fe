"""The backward of a group without a concatenated Wᵀ (gate|up and down outside the fused MLP: fused_linear._plain_backward)
bit for bit against the operations it stands for (fused_linear.py:128-196): every layer's MX
dgrad added in bf16, then dS·S onto that sum; d(xa) and dB as bf16 products, scaled in bf16.  The order matters in the
last bits: with dS·S added to the last layer's product before the sum over the layers, dx is 3e-3 off (normwise), and a
dB that is not rounded to bf16 1.7e-3."""
import pytest
import torch

import fused_linear
import mxfp8
import workloads

pytestmark = pytest.mark.gpu


def _transposed(t):
    """t with its storage transposed."""
    return t.t().contiguous().t()


def _expected(mods, x, dys, b_t):
    """dx and [dA, dB] of every layer from torch products and single MX GEMMs (xS as the forward makes it, beside the
    codes of x)."""
    parts = [fused_linear._part(m) for m in mods]
    bf = torch.bfloat16
    S = torch.cat([A.detach().to(bf) for _, A, _, _ in parts])
    xS = mxfp8.mx_quant_lora(x, S)[2]
    dx, dS, grads, col = None, [], [], 0
    for (base, A, B, s), dy in zip(parts, dys):
        g = mxfp8.mx_mm(*mxfp8.mx_quant(dy), *mxfp8.mx_wt(base))
        dx = g if dx is None else dx + g
        dB, dxa = dy.t() @ xS[:, col:col + A.shape[0]], dy @ (_transposed(B.detach().to(bf)) if b_t else B.detach().to(bf))
        dS.append(dxa * s if s != 1 else dxa)
        grads.append([None, dB * s if s != 1 else dB])
        col += A.shape[0]
    dS = torch.cat(dS, 1) if len(dS) > 1 else dS[0]
    dx.addmm_(dS, S)
    dA, col = dS.t() @ x, 0
    for (_, A, _, _), g in zip(parts, grads):
        g[0] = dA[col:col + A.shape[0]]
        col += A.shape[0]
    return dx, [t for g in grads for t in g]


# b_t: a saved-tensor hook gives the saved B back with the storage [r, N]
@pytest.mark.parametrize("r,T,names,b_t", [
    (16, 300, ("gate_proj", "up_proj"), False), (32, 129, ("gate_proj", "up_proj"), False),
    (16, 1000, ("down_proj",), False), (32, 31, ("down_proj",), False), (16, 300, ("gate_proj", "up_proj"), True)])
@pytest.mark.parametrize("need_x", [True, False])
def test_bits_of_the_torch_products(r, T, names, b_t, need_x, gpu, monkeypatch):
    monkeypatch.setitem(workloads.CONFIGS, 63, dict(name="u", T=T, K=512, N=768, r=r, alpha=1.5 * r, backward=True, layers=1))
    model, _ = workloads.build_model(63, T=T, device=gpu)
    monkeypatch.setattr(mxfp8, "FUSE_GU", False)
    mxfp8.enable_mxfp8(model)
    mods = [getattr(model.layers[0].mlp, n) for n in names]
    g = torch.Generator(device=gpu).manual_seed(T)
    x = torch.randn(T, mods[0].base_layer.in_features, device=gpu, generator=g).to(torch.bfloat16)
    dys = [(torch.randn(T, m.base_layer.out_features, device=gpu, generator=g) * 1e-2).to(torch.bfloat16) for m in mods]
    xi = x.clone().requires_grad_(need_x)
    fused_linear.new_step()
    b_shapes = [m.lora_B["default"].weight.shape for m in mods] * b_t
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: _transposed(t) if t.shape in b_shapes else t):
        outs = fused_linear.group_linear(xi, mods)
    torch.autograd.backward(list(outs), dys)
    dx, want = _expected(mods, x, dys, b_t)
    got = [p for m in mods for p in (m.lora_A["default"].weight.grad, m.lora_B["default"].weight.grad)]
    for k, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b.to(a.dtype)), k
    if need_x:
        assert torch.equal(xi.grad.view(torch.int16), dx.view(torch.int16))
