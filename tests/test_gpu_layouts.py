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


# mixed-radix grids (axes 2^a 3^b 5^c, not both powers of two, or an image wider
# than half the grid): rows sharing a workgroup with a short last one, column
# tiles with a short last one, one and several stages, a kernel that wraps past
# a last block of fewer than 16 cells, long axes near the LDS limit, kernels of
# up to 16, upsampling 1.25, more than one batch of planes
MIXED = [
    # precision, nx, ny, eps, sigma, wmax
    ("fp64", 25, 31, 1e-6, 2.0, 400.0), ("fp32", 25, 31, 1e-6, 2.0, 400.0),
    ("fp64", 75, 1125, 1e-6, 2.0, 300.0), ("fp32", 75, 1125, 1e-6, 2.0, 300.0),
    ("fp32", 1500, 75, 1e-5, 2.0, 300.0), ("fp64", 1499, 77, 1e-12, 2.0, 300.0),
    ("fp64", 3000, 40, 1e-6, 2.0, 200.0), ("fp64", 40, 3000, 1e-6, 2.0, 200.0),
    ("fp32", 6000, 48, 1e-6, 2.0, 100.0), ("fp32", 48, 6000, 1e-6, 2.0, 100.0),
    ("fp32", 90, 7300, 1e-6, 2.0, 100.0), ("fp32", 7300, 90, 1e-6, 2.0, 100.0),
    ("fp64", 512, 512, 1e-6, 1.25, 500.0), ("fp64", 500, 819, 1e-4, 1.25, 500.0),
    ("fp64", 100, 100, 1e-6, 2.0, 9000.0), ("fp32", 1024, 100, 1e-6, 2.0, 900.0),
]


@pytest.mark.parametrize("case", MIXED, ids=[f"{c[0]}-{c[1]}x{c[2]}-{c[3]:g}-{c[4]:g}" for c in MIXED])
def test_mixed_radix_grids(case):
    from curig_amd import _lib as L

    precision, nx, ny, eps, sigma, wmax = case
    fov = 2.0
    uvw, vis, wgt, img, f0 = _case(3000, nx, ny, fov, wmax, nx + 7 * ny, span=1.4)
    info = L.plan_info(len(uvw), nx, ny, fov, f0, eps, sigma, -1, float(uvw[:, 2].min()), float(uvw[:, 2].max()),
                       0 if precision == "fp64" else 1)
    assert info["fft_lds"] == 1
    e1, e2 = _both_paths(precision, uvw, vis, wgt, img, nx, ny, fov, f0, eps, sigma)
    say(f"[mixed radix] {case} grid {info['nf2']}x{info['nf1']}x{info['nf3']}: ms2dirty {e1:.2e}, dirty2ms {e2:.2e}")
    tol = 1e-10 if precision == "fp64" else 2e-6
    assert e1 < tol and e2 < tol


def test_fp32_beyond_half_the_grid_keeps_full_planes():
    """FP32 at upsampling 1.25: the corrections amplify rounding to 1e-5 of the
    result and more, so the plan keeps the full-plane path there."""
    from curig_amd import _lib as L

    for nx, ny in ((500, 819), (512, 512)):
        assert L.plan_info(3000, nx, ny, 2.0, 1e9, 1e-4, 1.25, -1, -500.0, 500.0, 1)["fft_lds"] == 0
        assert L.plan_info(3000, nx, ny, 2.0, 1e9, 1e-4, 2.0, -1, -500.0, 500.0, 1)["fft_lds"] == 1


def test_mixed_radix_empty_rows_and_non_finite_values():
    """A few visibilities (most rows of most planes empty), and an infinite one:
    the image is then not finite, as on the rocFFT path."""
    nx, ny, fov, eps = 300, 250, 2.0, 1e-6
    for precision in ("fp64", "fp32"):
        uvw, vis, wgt, img, f0 = _case(5, nx, ny, fov, 2000.0, 3)
        e1, e2 = _both_paths(precision, uvw, vis, wgt, img, nx, ny, fov, f0, eps)
        assert e1 < 2e-6 and e2 < 2e-6
        vis[2] = np.inf
        d = (gpu_ms2dirty if precision == "fp64" else (lambda *a: gpu_f32(True, *a)))(uvw, vis, wgt, nx, ny, fov, f0, eps)
        assert not np.isfinite(d).any()


# whole power-of-two rows (grid size along v) of every length the row kernels are
# built for, one and several rows per workgroup; few records (fused
# interpolation) and records dense on the grid (full planes and the gather),
# kernels of 7 and 13
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("ny", [32, 63, 128, 256, 509, 1024, 2048])
def test_rows_of_every_length(precision, ny):
    nx, fov = 128, 2.0
    for nrow, eps in ((300, 1e-6), (300, 1e-12), (30000, 1e-6)):
        uvw, vis, wgt, img, f0 = _case(nrow, nx, ny, fov, 300.0, nrow + ny)
        e1, e2 = _both_paths(precision, uvw, vis, wgt, img, nx, ny, fov, f0, eps)
        say(f"[rows] {precision} {nx}x{ny} rows {nrow} eps {eps}: ms2dirty {e1:.2e}, dirty2ms {e2:.2e}")
        tol = 1e-11 if precision == "fp64" else 2e-6
        assert e1 < tol and e2 < tol


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_gather_over_plane_batches(precision):
    """Dense records gathered over several batches of planes, on mixed-radix and
    power-of-two grids, with w planes that wrap around a batch's ends."""
    lib = _lib()
    assert lib.curig_set_tuning(0, 0, 5, 0) == 0
    try:
        for nx, ny in ((45, 50), (64, 64)):
            uvw, vis, wgt, img, f0 = _case(20000, nx, ny, 10.0, 400.0, nx)
            e1, e2 = _both_paths(precision, uvw, vis, wgt, img, nx, ny, 10.0, f0, 1e-6)
            tol = 1e-11 if precision == "fp64" else 2e-6
            assert e1 < tol and e2 < tol
    finally:
        lib.curig_set_tuning(0, 0, 0, 0)


# records dense on the rows in ms2dirty (FP64 row sums in FP32; row groups shared
# by several workgroups on small grids), power-of-two and mixed-radix grids,
# whole rows of 8192 and 4096
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,ny,nrow", [(64, 64, 200000), (50, 45, 200000), (40, 150, 100000), (32, 4096, 60000),
                                        (32, 2048, 60000)])
def test_dense_records(precision, nx, ny, nrow):
    fov, eps = 2.0, 1e-6
    uvw, vis, wgt, img, f0 = _case(nrow, nx, ny, fov, 5.0, nx + nrow)
    e1, e2 = _both_paths(precision, uvw, vis, wgt, img, nx, ny, fov, f0, eps)
    say(f"[dense] {precision} {nx}x{ny} rows {nrow}: ms2dirty {e1:.2e}, dirty2ms {e2:.2e}")
    tol = 1e-11 if precision == "fp64" else 2e-6
    assert e1 < tol and e2 < tol


# the corrections' w factor by its series, kernels of 5 to 14, against the direct sum
@pytest.mark.parametrize("eps", [1e-4, 1e-11, 1e-13])
def test_w_correction_against_direct_sum(eps):
    nx, ny, fov, sigma = 60, 44, 20.0, 2.0
    uvw, vis, wgt, img, f0 = _case(2000, nx, ny, fov, 60.0, 31)
    d = gpu_ms2dirty(uvw, vis, wgt, nx, ny, fov, f0, eps, sigma)
    v = gpu_dirty2ms(uvw, img, wgt, nx, ny, fov, f0, eps, sigma)
    e1 = O.l2error(O.dft_ms2dirty(uvw, vis, wgt, nx, ny, fov, f0, -1), d)
    e2 = O.l2error(O.dft_dirty2ms(uvw, img, wgt, nx, ny, fov, f0, -1), v)
    say(f"[w correction] eps {eps}: ms2dirty {e1:.2e}, dirty2ms {e2:.2e}")
    tol = max(3 * eps, 1e-12)
    assert e1 < tol and e2 < tol


# records in few rows and planes: the other rows are neither written to nor read
# from the intermediate planes, which a call on non-finite values fills first.
# Blocks of 64 and more rows, grids below one block, records across row 0 and
# across the last plane, batches of more planes than one mask word holds
OCCUPIED = [("fp64", 64, 64), ("fp32", 64, 64), ("fp64", 1024, 64), ("fp32", 2048, 64), ("fp64", 64, 2048),
            ("fp32", 64, 2048), ("fp32", 64, 4096), ("fp64", 64, 4096), ("fp32", 64, 8192), ("fp32", 8192, 64),
            ("fp64", 8192, 64), ("fp64", 600, 90), ("fp32", 1500, 75)]


@pytest.mark.parametrize("precision,nx,ny", OCCUPIED)
@pytest.mark.parametrize("planes", [0, 70])
def test_rows_without_records(precision, nx, ny, planes):
    lib = _lib()
    fov, eps, wmax = 2.0, 1e-6, 3000.0
    uvw, vis, wgt, img, f0 = _case(400, nx, ny, fov, wmax, nx + ny)
    uvw[:, 0] = np.where(np.arange(400) % 2, 0.02, 0.3) * uvw[:, 0]
    uvw[:, 2] = np.where(np.arange(400) % 2, uvw[:, 2], 0.9 * wmax + 0.1 * uvw[:, 2])
    image = gpu_ms2dirty if precision == "fp64" else (lambda *a: gpu_f32(True, *a))
    predict = gpu_dirty2ms if precision == "fp64" else (lambda *a: gpu_f32(False, *a))
    assert lib.curig_set_tuning(0, 0, planes, 0) == 0
    try:
        full = _case(400, nx, ny, fov, wmax, 5)[0]
        image(full, np.full(400, np.inf + 0j), wgt, nx, ny, fov, f0, eps)
        d = image(uvw, vis, wgt, nx, ny, fov, f0, eps)
        predict(full, np.full((nx, ny), np.inf + 0j), wgt, nx, ny, fov, f0, eps)
        v = predict(uvw, img, wgt, nx, ny, fov, f0, eps)
        lib.curig_set_fft_path(1)
        e1 = O.l2error(image(uvw, vis, wgt, nx, ny, fov, f0, eps), d)
        e2 = O.l2error(predict(uvw, img, wgt, nx, ny, fov, f0, eps), v)
    finally:
        lib.curig_set_fft_path(0)
        lib.curig_set_tuning(0, 0, 0, 0)
    say(f"[rows without records] {precision} {nx}x{ny} planes {planes}: ms2dirty {e1:.2e}, dirty2ms {e2:.2e}")
    tol = 1e-11 if precision == "fp64" else 2e-6
    assert e1 < tol and e2 < tol


# rows counted in LDS by chunks: several and many rows to a bin, a short last chunk
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,ny,nrow", [(32, 64, 40001), (64, 64, 300007), (512, 32, 270000)])
def test_many_rows_to_a_bin(precision, nx, ny, nrow):
    fov, eps = 2.0, 1e-5
    uvw, vis, wgt, img, f0 = _case(nrow, nx, ny, fov, 2.0, nx + nrow)
    e1, e2 = _both_paths(precision, uvw, vis, wgt, img, nx, ny, fov, f0, eps)
    say(f"[many rows to a bin] {precision} {nx}x{ny} rows {nrow}: ms2dirty {e1:.2e}, dirty2ms {e2:.2e}")
    tol = 1e-11 if precision == "fp64" else 2e-6
    assert e1 < tol and e2 < tol


# bin offsets in one workgroup and in three passes: a bin or a few, 1024 of them and
# more (several to a thread), and about the most that one workgroup scans (4096
# strips times three to eight layers)
@pytest.mark.parametrize("nx,ny,wmax", [(8, 64, 5.0), (512, 64, 200.0), (600, 64, 500.0), (4096, 32, 10.0),
                                        (4096, 32, 60.0), (4096, 32, 150.0), (4096, 32, 300.0)])
def test_bin_offsets(nx, ny, wmax):
    fov, eps = 2.0, 1e-6
    uvw, vis, wgt, img, f0 = _case(5000, nx, ny, fov, wmax, nx + ny)
    e1, e2 = _both_paths("fp64", uvw, vis, wgt, img, nx, ny, fov, f0, eps)
    say(f"[bin offsets] {nx}x{ny} wmax {wmax}: ms2dirty {e1:.2e}, dirty2ms {e2:.2e}")
    assert e1 < 1e-11 and e2 < 1e-11
