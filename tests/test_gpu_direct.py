"""GPU: routes that the full-plane path shares or that only some densities take,
against FP64 direct sums at sampled pixels and rows (the last rows among them), both
directions.  Bars: 3 epsilon + 1e-11 (FP64), + 3e-6 (FP32-mixed) more; against the
full-plane path 1e-11 and 2e-6."""
import numpy as np
import pytest

from curig_amd import _lib as L
from tests import oracle_helpers as O
from tests.test_gpu_layouts import _both_paths, _case
from tests.test_gpu_parity import gpu_dirty2ms, gpu_f32, gpu_ms2dirty, say

pytestmark = pytest.mark.gpu


def _direct(precision, uvw, vis, wgt, img, nx, ny, fov, f0, eps):
    """Relative errors of both directions against direct sums at 48 pixels and 100 rows."""
    rng = np.random.default_rng(nx + ny)
    f64 = precision == "fp64"
    d = (gpu_ms2dirty if f64 else (lambda *a: gpu_f32(True, *a)))(uvw, vis, wgt, nx, ny, fov, f0, eps)
    v = (gpu_dirty2ms if f64 else (lambda *a: gpu_f32(False, *a)))(uvw, img, wgt, nx, ny, fov, f0, eps)
    pix = rng.choice(nx * ny, 48, replace=False)
    rows = np.unique(np.r_[:20, rng.choice(len(uvw), 50, replace=False), len(uvw) - 30:len(uvw)])
    e1 = O.l2error(O.dft_ms2dirty_pixels(uvw, vis, wgt, nx, ny, fov, f0, pix, -1), d.reshape(-1)[pix])
    e2 = O.l2error(O.dft_dirty2ms(uvw[rows], img, wgt[rows], nx, ny, fov, f0, -1), v[rows])
    return e1, e2, 3 * eps + (1e-11 if f64 else 3e-6)


# the rows counted in LDS by chunks: a thread counts one row or several (512 x 32:
# 131 chunks of 2,062 rows)
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,ny,nrow", [(32, 64, 40001), (64, 64, 300007), (512, 32, 270000)])
def test_many_rows_to_a_bin(precision, nx, ny, nrow):
    fov, eps = 2.0, 1e-6
    uvw, vis, wgt, img, f0 = _case(nrow, nx, ny, fov, 2.0, nx + nrow)
    e1, e2, bar = _direct(precision, uvw, vis, wgt, img, nx, ny, fov, f0, eps)
    say(f"[direct: many rows to a bin] {precision} {nx}x{ny} rows {nrow}: ms2dirty {e1:.2e}, dirty2ms {e2:.2e}")
    assert e1 < bar and e2 < bar


@pytest.mark.parametrize("nx,ny,wmax", [(8, 64, 5.0), (600, 64, 500.0), (4096, 32, 60.0), (4096, 32, 300.0)])
def test_bin_offsets(nx, ny, wmax):
    fov, eps = 2.0, 1e-6
    uvw, vis, wgt, img, f0 = _case(5000, nx, ny, fov, wmax, nx + ny)
    e1, e2, bar = _direct("fp64", uvw, vis, wgt, img, nx, ny, fov, f0, eps)
    say(f"[direct: bin offsets] {nx}x{ny} wmax {wmax}: ms2dirty {e1:.2e}, dirty2ms {e2:.2e}")
    assert e1 < bar and e2 < bar


# FP32 rows of 8192 by record visits per row and plane: halves up to 1,000, then
# whole with the fused interpolation (up to 0.3 visits per cell, 2,458), then gathered
@pytest.mark.parametrize("nx,ny,nrow,eps,visits,rsplit", [
    (128, 4096, 40_000, 1e-6, 478, 2), (128, 4096, 120_000, 1e-6, 1435, 0), (127, 4051, 70_000, 1e-9, 1367, 0),
    (128, 4096, 240_000, 1e-6, 2871, 0)])
def test_rows_of_8192_by_density(nx, ny, nrow, eps, visits, rsplit):
    fov, wmax = 1.0, 30.0
    uvw, vis, wgt, img, f0 = _case(nrow, nx, ny, fov, wmax, nx + ny)
    info = L.plan_info(nrow, nx, ny, fov, f0, eps, 2.0, -1, float(uvw[:, 2].min()), float(uvw[:, 2].max()), 1)
    assert info["nf1"] == 8192 and info["rsplit"] == rsplit
    assert nrow * info["kw"] ** 2 / (info["nf3"] * info["nf2"]) == pytest.approx(visits, rel=0.01)
    e1, e2, bar = _direct("fp32", uvw, vis, wgt, img, nx, ny, fov, f0, eps)
    p1, p2 = _both_paths("fp32", uvw, vis, wgt, img, nx, ny, fov, f0, eps)
    say(f"[direct: rows of 8192] {nx}x{ny} rows {nrow}: ms2dirty {e1:.2e} ({p1:.2e}), dirty2ms {e2:.2e} ({p2:.2e})")
    assert e1 < bar and e2 < bar and p1 < 2e-6 and p2 < 2e-6


def test_mixed_radix_rows_without_records_in_fp64():
    """Five visibilities and mixed-radix grids of an upsampling of 2, at FP64's own bar."""
    eps = 1e-6
    for nx, ny, nrow, wmax in ((300, 250, 5, 2000.0), (75, 1125, 3000, 300.0), (3000, 40, 3000, 200.0),
                               (100, 100, 3000, 9000.0)):
        uvw, vis, wgt, img, f0 = _case(nrow, nx, ny, 2.0, wmax, 3)
        e1, e2 = _both_paths("fp64", uvw, vis, wgt, img, nx, ny, 2.0, f0, eps)
        say(f"[mixed radix, FP64] {nx}x{ny} rows {nrow}: ms2dirty {e1:.2e}, dirty2ms {e2:.2e}")
        assert e1 < 1e-11 and e2 < 1e-11
