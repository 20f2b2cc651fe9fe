"""The codes of dy that the grouped backward hands to its dx GEMM (_native.host().group_lora_bwd, mxfp8_lora_bwd_batch
with q_tiled): the MX-tiled layout must hold byte for byte the row-major codes of mxfp8.lora_bwd (rearranged by
mxfp8.tile_codes; rows past T are not written), with the same scales, d(xa) and dB."""
import pytest
import torch

import _native
import mxfp8

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 16, 31, 33, 127, 129, 300, 1000])
@pytest.mark.parametrize("Ns,r", [((128,), 16), ((384, 128, 256), 16), ((256, 128), 32)])
def test_tiled_codes_of_the_grouped_backward(T, Ns, r, gpu):
    g = torch.Generator(device=gpu).manual_seed(T + sum(Ns) + r)
    dys = [(torch.randn(T, n, device=gpu, generator=g) * 1e-2).to(torch.bfloat16) for n in Ns]
    xS = torch.randn(T, 64 if r == 16 else 128, device=gpu, generator=g).to(torch.bfloat16)
    Bs = [(torch.randn(n, r, device=gpu, generator=g) * 0.02).to(torch.bfloat16) for n in Ns]
    cols, scales = [r * k for k in range(len(Ns))], [2.0 + k for k in range(len(Ns))]
    dS = torch.full_like(xS, float("nan"))
    q, s, dbs = _native.host().group_lora_bwd(dys, xS, Bs, cols, scales, dS, True, _native.stream_of(xS))
    want_q = torch.empty((T, sum(Ns)), dtype=mxfp8.F8, device=gpu)
    want_s = torch.empty(mxfp8.scale_numel(T, sum(Ns)), dtype=torch.uint8, device=gpu)
    want_dS = torch.full_like(dS, float("nan"))
    offs = [sum(Ns[:k]) // 128 for k in range(len(Ns))]
    want_db = mxfp8.lora_bwd_batch(dys, [xS[:, c:c + r] for c in cols], Bs, scales, [want_dS[:, c:c + r] for c in cols],
                                   q=want_q, s=want_s, col_tile_offs=offs)
    tiled = mxfp8.tile_codes(want_q).view(torch.uint8)
    rows = torch.zeros((mxfp8.tiled_rows(T), sum(Ns)), dtype=torch.uint8, device=gpu)
    rows[:T] = 1
    live = mxfp8.tile_codes(rows.view(mxfp8.F8)).view(torch.uint8) == 1  # the bytes of rows below T
    assert torch.equal(q.view(torch.uint8)[live], tiled[live])
    assert torch.equal(s.view(torch.uint8), want_s)
    assert torch.equal(dS.view(torch.int16), want_dS.view(torch.int16))
    for a, b in zip(dbs, want_db):
        assert torch.equal(a, b)
