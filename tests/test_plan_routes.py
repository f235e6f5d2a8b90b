"""Which grids the LDS path takes (no device needed): mixed-radix axes up to the 16
points per thread of the largest workgroup, FP64 512 threads, FP32 1024."""
import pytest

from curig_amd import _lib as L


def _lds(nx, ny, precision):
    info = L.plan_info(1000, nx, ny, 1.0, 1e9, 1e-6, 2.0, -1, -5.0, 5.0, precision)
    return info["fft_lds"], info["nf2"], info["nf1"]


@pytest.mark.parametrize("precision,last,beyond", [(0, 8100, 8640), (1, 16200, 17280)])
def test_longest_mixed_radix_axes(precision, last, beyond):
    for n, on in ((last, 1), (beyond, 0)):
        assert _lds(n // 2, 300, precision) == (on, n, 600)
        assert _lds(300, n // 2, precision) == (on, 600, n)
