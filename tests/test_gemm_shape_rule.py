"""The workgroup shape that each size of test_gpu_shapes.py takes (csrc/gemm_shape.h, host code): a test of a shape's bits
means something only where that shape runs."""
import pytest

import _native
from test_gpu_shapes import FOLDED, SEGMENTS, SIZES

ALL = [("256x128", None), ("256x256", None), ("128x128", None), ("64x128", None), ("64x64", None), ("256x128", "64x128"),
       ("256x128", "128x128")]


def _cases():
    for kind, table in (("plain", SIZES), ("sum", FOLDED), ("tn", FOLDED)):
        for shape, sizes in table.items():
            for size in sizes:
                yield kind, size, shape
    for shape, sizes in SEGMENTS.items():
        for M, widths, K in sizes:
            yield "seg", (M, sum(widths), K), shape


@pytest.mark.parametrize("kind,size,shape", list(_cases()))
def test_size_takes_its_shape(kind, size, shape):
    got = _native.gemm_shape(*size, kind=kind, cus=256)
    assert got[:2] == shape
    assert got[2] % 256 == 0 and 0 <= got[2] < size[0] and bool(got[2]) == (shape[1] is not None)


def test_every_shape_has_a_size():
    assert set(SIZES) == set(FOLDED) == set(ALL)
    assert set(SEGMENTS) == set(ALL) - {("256x256", None)}  # several outputs: 4 waves only


def test_the_longest_step_takes_the_8_wave_shape():
    """One layer of a 16 x 8896 batch: down with its sum and dx with its reductions."""
    assert _native.gemm_shape(142336, 2048, 6144, "sum", 256)[0] == "256x256"
    assert _native.gemm_shape(142336, 2048, 12288, "tn", 256)[0] == "256x256"


def test_bad_sizes_are_refused():
    for M, N, K, kind in ((0, 128, 128, "plain"), (64, 100, 128, "plain"), (64, 128, 64, "tn")):
        with pytest.raises(RuntimeError, match="gemm_shape"):
            _native.gemm_shape(M, N, K, kind, 256)
