"""Which per-layer backward a group takes (fused_linear._native_per_layer): the library's kernels index each B as a
contiguous bf16 [N, r], so a B with other strides (the cast of a transposed fp64 or fp16 parameter keeps them, and a
saved-tensor hook may return them) stays with the torch products, as does one of another dtype."""
import types

import pytest
import torch

import fused_linear


def _slots(B, monkeypatch, T=40, N=256, r=16):
    monkeypatch.setattr(fused_linear, "_native_ok", lambda x2, dt, n: True)  # the sizes and device, met on a GPU
    slot = types.SimpleNamespace(width=r, col=0, cols=slice(0, r), index=0, layer=0, scale=2.0)
    spec = types.SimpleNamespace(thin=[], plain=[], mx=[0], adapters=[slot], _adapter={0: slot}, width=r)
    e = lambda *s: torch.zeros(s, dtype=torch.bfloat16)  # noqa: E731
    return fused_linear._native_per_layer(spec, e(T, 128), e(T, r), [B], [e(T, N)], torch.bfloat16)


def test_contiguous_b_runs_on_the_kernels(monkeypatch):
    assert _slots(torch.zeros(256, 16, dtype=torch.bfloat16), monkeypatch) is not None


@pytest.mark.parametrize("B", [torch.zeros(16, 256, dtype=torch.float64).t().to(torch.bfloat16),
                               torch.zeros(256, 32, dtype=torch.bfloat16)[:, :16], torch.zeros(256, 16)])
def test_other_b_stays_with_the_torch_products(B, monkeypatch):
    assert _slots(B, monkeypatch) is None
