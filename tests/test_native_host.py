"""Argument checks of the native host module (csrc/host_path.cpp) that come before its first launch."""
import pytest
import torch

import _native

T, K, N, R = 64, 256, 384, 16


def _bf(*shape):
    return torch.zeros(shape, dtype=torch.bfloat16)


def _codes(*shape):
    return torch.zeros(shape, dtype=torch.uint8).view(torch.float8_e4m3fn)


def _forward(wf, wd):
    s = torch.zeros(8, dtype=torch.uint8)
    return _native.host().mlp_forward(_bf(T, K), _bf(2 * R, K), _bf(N, R), _bf(N, R), _bf(R, N), _bf(K, R), wf, s, wd, s,
                                      1.0, 1.0, 1.0, 1 << 26, 0)


def _backward(wt, wx):
    s = torch.zeros(8, dtype=torch.uint8)
    forms = (_bf(2 * R, K), _bf(K, 2 * R), _bf(N, R), _bf(N, R), _bf(R, N), _bf(R, N), _bf(R, N), _bf(N, R), _bf(K, R),
             _bf(R, K))
    return _native.host().mlp_backward(_bf(T, K), _bf(T, K), _bf(T, 2 * R), _bf(T, 2 * N), forms, wt, s, wx, s, 1.0, 1.0,
                                       1.0, 128, 128, False, True, True, True, 0)


@pytest.mark.parametrize("call,what", [
    (lambda: _forward(_codes(2 * N, K), _codes(K, N + 128)), "down weight"),
    (lambda: _forward(_codes(2 * N, K), _codes(K, N - 128)), "down weight"),
    (lambda: _forward(_codes(2 * N, 2 * K), _codes(K, N)), "gate.up weight"),
    (lambda: _native.host().mlp_graph(_bf(T, K), _bf(2 * R, K), _codes(2 * N, 128), torch.zeros(8), N, 0), "gate.up weight"),
    (lambda: _backward(_codes(N, K + 128), _codes(K, 2 * N)), "down weight"),
    (lambda: _backward(_codes(N, K), _codes(K, 2 * N - 128)), "gate.up weight")])
def test_a_weight_of_other_columns_is_refused(call, what):
    with pytest.raises(RuntimeError, match=what):
        call()


def test_fitting_weights_pass_the_checks():
    for call in (lambda: _forward(_codes(2 * N, K), _codes(K, N)), lambda: _backward(_codes(N, K), _codes(K, 2 * N))):
        with pytest.raises(_native.NativeError, match="must be on the GPU"):
            call()


@pytest.mark.parametrize("cols,width,what", [((16, 32), 32, "columns 32 to 48"), ((0, 16), 16, "columns 16 to 32"),
                                             ((0,), 32, "1 to 8 layers"), ((0, 16), 32, "must be on the GPU")])
def test_group_lora_bwd_columns(cols, width, what):
    with pytest.raises(RuntimeError, match=what):
        _native.host().group_lora_bwd([_bf(T, N)] * 2, _bf(T, width), [_bf(N, R)] * 2, list(cols), [1.0, 1.0],
                                      _bf(T, width), True, 0)
