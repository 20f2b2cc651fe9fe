"""The workgroup shapes of the MX GEMM (csrc/mx_gemm.hip, pick_shape): 64 x 64, 64 x 128 and 128 x 128 tiles where
256 x 128 ones would leave CUs idle (in a whole launch or in its last rows only), 256 x 256 for long launches.  An
output element adds the same products over K in the same order in every shape, so each size must give the bits of the
explicitly asked 8-wave shape run whole (MXFP8_GEMM_WIDE without a workspace), which every size takes: bit-exact, no
tolerance."""
import pytest
import torch

import _native
import mxfp8

pytestmark = pytest.mark.gpu


def _operands(M, N, K, gpu):
    g = torch.Generator(device=gpu).manual_seed(M + 3 * N + 7 * K)
    e = torch.exp2(torch.randint(-6, 6, (M, 1), device=gpu, generator=g).float())
    a = (torch.randn(M, K, device=gpu, generator=g) * e).to(torch.bfloat16)
    b = (torch.randn(N, K, device=gpu, generator=g) * 0.02).to(torch.bfloat16)
    return g, mxfp8.mx_quant_tiled(a), mxfp8.mx_quant_tiled(b), b


# (the shape, the shape of the last rows or None) that a GPU of 256 CUs takes -> sizes: edges of 64, 128 and 256 rows; N
# that is and is not a multiple of 256; an odd count of 128-wide K tiles.  test_gemm_shape_rule.py holds the sizes to
# their shapes.
SIZES = {
    ("64x64", None): [(1, 128, 128), (63, 256, 384), (64, 1024, 1024), (65, 384, 640), (129, 2048, 1152)],
    ("64x128", None): [(1000, 2048, 1024), (961, 1920, 1408)],
    ("128x128", None): [(129, 12288, 256), (1500, 2048, 2048), (1921, 1920, 1152)],
    ("256x128", None): [(321, 12288, 384), (1025, 12288, 128)],
    ("256x256", None): [(770, 12288, 3072), (2561, 4096, 3072), (5131, 2048, 3072)],
    # the rows past the last whole round of tiles: 1 to 1024 such rows, after one workgroup per CU and after two
    ("256x128", "64x128"): [(1281, 12288, 384), (1407, 6144, 256), (3840 + 257, 6272, 640), (8896, 2048, 1152),
                            (5377, 1920, 2048), (5000, 2048, 2048), (4353, 2304, 1280)],
    ("256x128", "128x128"): [(2753, 12288, 128), (3073, 6272, 640), (9217, 2048, 1152)],
}
# the same for mxfp8_gemm_nt_sum and mxfp8_gemm_nt_tn (which lose their folded work's share in the 8-wave shape)
FOLDED = {
    ("64x64", None): [(65, 384, 640)],
    ("64x128", None): [(961, 1920, 1408)],
    ("128x128", None): [(1921, 1920, 1152)],
    ("256x128", None): [(321, 12288, 384)],
    ("256x256", None): [(10497, 12288, 3072)],
    ("256x128", "64x128"): [(4097, 2048, 1152)],
    ("256x128", "128x128"): [(9217, 2048, 1152)],
}
# the same for mxfp8_gemm_nt_seg: (M, output widths, K)
SEGMENTS = {
    ("64x64", None): [(40, (256, 128, 256), 256)],
    ("64x128", None): [(700, (1024, 256, 256), 1024)],
    ("128x128", None): [(1500, (1024, 256, 256), 1024)],
    ("256x128", None): [(3073, (2048, 2048), 2048)],
    ("256x128", "64x128"): [(5377, (1280, 512, 128), 2048)],
    ("256x128", "128x128"): [(4300, (4096, 1920, 128, 128), 640)],
}


def _sizes(table):
    return [size for sizes in table.values() for size in sizes]


@pytest.mark.parametrize("M,N,K", _sizes(SIZES))
@pytest.mark.parametrize("rank", [0, 16, 48])
def test_every_shape_gives_the_same_bits(M, N, K, rank, gpu):
    g, (qa, sa), (qb, sb), b = _operands(M, N, K, gpu)
    lora = None
    if rank:
        lora = ((torch.randn(M, rank, device=gpu, generator=g) * 0.1).to(torch.bfloat16),
                (torch.randn(N, rank, device=gpu, generator=g) * 0.1).to(torch.bfloat16))
    want = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=gpu)
    _native.gemm_nt(qa, sa, K, qb, sb, K, M, N, K, want, lora=lora, alpha=0.7, split=False, layout=3 | _native.GEMM_WIDE)
    got = mxfp8.mx_mm(qa, sa, qb, sb, lora=lora, alpha=0.7, layout=3, m=M)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    # the pi_col row order of B (16-byte stores)
    qp, sp = mxfp8.mx_quant_tiled(b[mxfp8.fused_dgrad_rows(N, gpu)].contiguous())
    got = mxfp8.mx_mm(qa, sa, qp, sp, lora=lora, alpha=0.7, layout=3 | _native.GEMM_B_PI, m=M)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    # C in the fused-tile layout (rows past M are not written: both start from zeros)
    ft = [torch.zeros((mxfp8.ft_rows(M), N), dtype=torch.bfloat16, device=gpu) for _ in range(2)]
    _native.gemm_nt(qa, sa, K, qb, sb, K, M, N, K, ft[0], lora=lora, alpha=0.7, split=False,
                    layout=3 | _native.GEMM_WIDE | _native.GEMM_C_FT)
    mxfp8.mx_mm(qa, sa, qp, sp, out=ft[1], lora=lora, alpha=0.7, layout=3 | _native.GEMM_B_PI | _native.GEMM_C_FT, m=M)
    assert torch.equal(ft[0].view(torch.int16), ft[1].view(torch.int16))


@pytest.mark.parametrize("M,N,K", _sizes(FOLDED) + [(20501, 2048, 12288)])
def test_folded_launches_in_every_shape(M, N, K, gpu):
    """mxfp8_gemm_nt_sum and mxfp8_gemm_nt_tn against the separate calls, in the shapes that carry the folded work and
    in the 8-wave one, which launches it apart: bit-identical.  wait_limit 0: every tile sums its own rows of P."""
    g, (qa, sa), (qb, sb), _ = _operands(M, N, K, gpu)
    part = torch.randn(5, M, 16, device=gpu, generator=g)
    Q = (torch.randn(N, 32, device=gpu, generator=g) * 0.1).to(torch.bfloat16)
    P = torch.empty(M, 16, dtype=torch.bfloat16, device=gpu)
    _native.sum_parts(part, 5, M * 16, P)
    want = mxfp8.mx_mm(qa, sa, qb, sb, lora=(P, Q[:, :16]), alpha=0.5, layout=3, m=M)
    for wait_limit in (-1, 0):
        P2 = torch.full_like(P, float("nan"))
        got = mxfp8.mx_mm_sum(qa, sa, qb, sb, part, P2, Q[:, :16], 0.5, 3, M, wait_limit=wait_limit)
        assert torch.equal(P, P2) and torch.equal(got.view(torch.int16), want.view(torch.int16)), wait_limit
    x = torch.randn(M, 256, device=gpu, generator=g).to(torch.bfloat16)
    P3 = torch.randn(M, 32, device=gpu, generator=g).to(torch.bfloat16)
    outs = [torch.empty(32, 256, dtype=torch.bfloat16, device=gpu) for _ in range(2)]
    scratch = torch.empty(_native.lora_tn_chunks(M, 256) * 32 * 256, dtype=torch.float32, device=gpu)
    want = mxfp8.mx_mm(qa, sa, qb, sb, lora=(P3, Q), alpha=1.0, layout=3, m=M)
    _native.lora_tn_batch([(x, P3, outs[0], 1.0, False)], scratch)
    got = mxfp8.mx_mm_tn(qa, sa, qb, sb, (P3, Q), 1.0, 3, M, [(x, P3, outs[1], 1.0, False)], scratch)
    assert torch.equal(outs[0], outs[1]) and torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("M,widths,K", _sizes(SEGMENTS))
@pytest.mark.parametrize("rank,window", [(0, False), (48, False), (16, True)])
def test_separate_outputs_in_every_shape(M, widths, K, rank, window, gpu):
    """mxfp8_gemm_nt_seg against one GEMM per output in the 8-wave shape: bit-identical.  window: each output adds the
    rank-16 product over columns of its own (the others hold NaN), else all over the same 48."""
    N = sum(widths)
    g, (qa, sa), (qb, sb), _ = _operands(M, N, K, gpu)
    P = (torch.randn(M, 64, device=gpu, generator=g) * 0.1).to(torch.bfloat16)
    Q = (torch.randn(N, 64, device=gpu, generator=g) * 0.1).to(torch.bfloat16)
    cols = [16 * k for k in range(len(widths))] if window else [0] * len(widths)
    per_tile_row, c0, want = K // 128 * 512, 0, []
    for n, col in zip(widths, cols):
        lora = (P[:, col:col + rank], Q[c0:c0 + n, col:col + rank]) if rank else None
        out = torch.full((M, n), float("nan"), dtype=torch.bfloat16, device=gpu)
        scales = sb[c0 // 128 * per_tile_row:(c0 + n) // 128 * per_tile_row]
        _native.gemm_nt(qa, sa, K, qb[c0:c0 + n], scales, K, M, n, K, out, lora=lora, alpha=0.7, split=False,
                        layout=3 | _native.GEMM_WIDE)
        want.append(out)
        if window:
            keep = Q[c0:c0 + n, col:col + rank].clone()
            Q[c0:c0 + n] = float("nan")
            Q[c0:c0 + n, col:col + rank] = keep
        c0 += n
    outs = [torch.full((M, n), float("nan"), dtype=torch.bfloat16, device=gpu) for n in widths]
    lora = (P if window else P[:, :rank], Q if window else Q[:, :rank]) if rank else None
    kw = dict(lora_cols=cols, r=rank) if window else {}
    mxfp8.mx_mm_seg(qa, sa, qb, sb, outs, lora=lora, alpha=0.7, layout=3, m=M, **kw)
    for k, (a, b) in enumerate(zip(outs, want)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16)), k


@pytest.mark.parametrize("rank", [0, 16])
@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("M,N,K", [(300, 384, 256), (257, 128, 512)])
def test_the_8_wave_shape_past_the_last_column(M, N, K, split, rank, gpu):
    """MXFP8_GEMM_WIDE | MXFP8_GEMM_B_PI with N % 256 == 128: the half of the last 256-column tile that lies past N is
    not stored.  C row-major with guard columns (a tile's width of them) and guard rows, and in the fused-tile layout;
    the same bits as without MXFP8_GEMM_B_PI, split along K or not."""
    g, (qa, sa), (qb, sb), b = _operands(M, N, K, gpu)
    qp, sp = mxfp8.mx_quant_tiled(b[mxfp8.fused_dgrad_rows(N, gpu)].contiguous())
    lora = None
    if rank:
        lora = ((torch.randn(M, rank, device=gpu, generator=g) * 0.1).to(torch.bfloat16),
                (torch.randn(N, rank, device=gpu, generator=g) * 0.1).to(torch.bfloat16))
    got, want = (torch.full((M + 8, N + 256), 3.0, dtype=torch.bfloat16, device=gpu) for _ in range(2))
    kw = dict(lora=lora, alpha=0.7, split=split)
    _native.gemm_nt(qa, sa, K, qb, sb, K, M, N, K, want[:M, :N], layout=3 | _native.GEMM_WIDE, **kw)
    _native.gemm_nt(qa, sa, K, qp, sp, K, M, N, K, got[:M, :N], layout=3 | _native.GEMM_WIDE | _native.GEMM_B_PI, **kw)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    assert bool((got[:, N:] == 3.0).all()) and bool((got[M:] == 3.0).all())
    ft = [torch.full((mxfp8.ft_rows(M) + 32, N), 3.0, dtype=torch.bfloat16, device=gpu) for _ in range(2)]
    for c, q, s, bit in ((ft[0], qb, sb, 0), (ft[1], qp, sp, _native.GEMM_B_PI)):
        _native.gemm_nt(qa, sa, K, q, s, K, M, N, K, c, layout=3 | _native.GEMM_WIDE | _native.GEMM_C_FT | bit, **kw)
    assert torch.equal(ft[0].view(torch.int16), ft[1].view(torch.int16))
    assert bool((ft[1][mxfp8.ft_rows(M):] == 3.0).all())
