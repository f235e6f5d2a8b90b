"""GPU parity of the plan's layouts: every layout that the plan chooses by size,
density and direction against the full-plane rocFFT path on the same problem,
both directions, at sizes where the choice or its index arithmetic changes.
Bars as for the other path comparisons: 1e-11 (FP64), 2e-6 (FP32-mixed, both
sides rounding in FP32)."""
import numpy as np
import pytest

from tests import oracle_helpers as O
from tests.test_gpu_parity import C, _lib, gpu_dirty2ms, gpu_f32, gpu_ms2dirty, say

pytestmark = pytest.mark.gpu


def _case(nrow, nx, ny, fov, wmax, seed, span=0.98, f0=1e9):
    """u, v over `span` of the grid's band, w in +-wmax metres."""
    rng = np.random.default_rng(seed)
    uvw = np.empty((nrow, 3))
    for axis, n in ((0, nx), (1, ny)):
        uvw[:, axis] = (rng.random(nrow) - 0.5) * span / (fov * np.pi / 180 / n) * C / f0
    uvw[:, 2] = rng.uniform(-1, 1, nrow) * wmax
    vis = rng.standard_normal(nrow) + 1j * rng.standard_normal(nrow)
    wgt = rng.uniform(0.5, 1.0, nrow)
    img = rng.standard_normal((nx, ny)) + 1j * rng.standard_normal((nx, ny))
    return uvw, vis, wgt, img, f0


def _both_paths(precision, uvw, vis, wgt, img, nx, ny, fov, f0, eps, sigma=2.0):
    """(ms2dirty, dirty2ms) relative differences of the plan's path from the rocFFT path."""
    lib = _lib()

    def run():
        if precision == "fp64":
            return (gpu_ms2dirty(uvw, vis, wgt, nx, ny, fov, f0, eps, sigma),
                    gpu_dirty2ms(uvw, img, wgt, nx, ny, fov, f0, eps, sigma))
        return (gpu_f32(True, uvw, vis, wgt, nx, ny, fov, f0, eps, sigma=sigma),
                gpu_f32(False, uvw, img, wgt, nx, ny, fov, f0, eps, sigma=sigma))

    d, v = run()
    assert lib.curig_set_fft_path(1) == 0
    try:
        d_roc, v_roc = run()
    finally:
        lib.curig_set_fft_path(0)
    return O.l2error(d_roc, d), O.l2error(v_roc, v)


# FP32 rows of 8192: halves; odd and short image widths; kernels of 7 and 11;
# 40,000 rows on a few planes are dense enough for whole rows in dirty2ms
@pytest.mark.parametrize("nx,ny,nrow,eps", [(64, 4096, 3000, 1e-6), (64, 4095, 3000, 1e-6), (63, 4051, 3000, 1e-10),
                                            (128, 4096, 40000, 1e-6)])
def test_rows_of_8192_in_halves(nx, ny, nrow, eps):
    fov = 1.0
    uvw, vis, wgt, img, f0 = _case(nrow, nx, ny, fov, 30.0, nx + ny)
    e1, e2 = _both_paths("fp32", uvw, vis, wgt, img, nx, ny, fov, f0, eps)
    say(f"[rows of 8192] {nx}x{ny} rows {nrow} eps {eps}: ms2dirty {e1:.2e}, dirty2ms {e2:.2e}")
    assert e1 < 2e-6 and e2 < 2e-6


# power-of-two columns (grid size along u) of every length the column kernels
# are built for, few planes (several plane chunks per batch) and more than one
# batch of planes; image rows at and below half the grid
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,ny,wmax", [(32, 64, 400.0), (63, 64, 4000.0), (128, 63, 400.0), (256, 64, 3000.0),
                                        (509, 64, 400.0), (1024, 64, 400.0), (2048, 64, 400.0), (4096, 64, 400.0)])
def test_columns_of_every_length(precision, nx, ny, wmax):
    fov, eps = 2.0 if nx > 100 else 10.0, 1e-6
    uvw, vis, wgt, img, f0 = _case(2000, nx, ny, fov, wmax, nx * 3 + ny)
    e1, e2 = _both_paths(precision, uvw, vis, wgt, img, nx, ny, fov, f0, eps)
    say(f"[columns] {precision} {nx}x{ny} wmax {wmax}: ms2dirty {e1:.2e}, dirty2ms {e2:.2e}")
    tol = 1e-11 if precision == "fp64" else 2e-6
    assert e1 < tol and e2 < tol
