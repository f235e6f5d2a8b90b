"""GPU: FP32 images of uv data that crowd a few grid cells, against the FP64 call
on the same (FP32) visibilities, for every way an FP32 row is summed: thousands of
noise visibilities share each cell, where the rounding of a sum in FP32 or in
scaled integers grows with their number.

Bar 5e-7: summed in FP64, a cell keeps the roundings of FP32 values alone (the
record, three taps and their products, and log2 n transform levels: about 25
independent ones of 2^-25 on average, 1.5e-7), three times that.  Sums in FP32 reach
1e-6 to 7e-6 on these cases, 30-bit integers 1e-5 to 4e-4."""
import numpy as np
import pytest

from tests import oracle_helpers as O
from tests.test_gpu_parity import C, gpu_f32, gpu_ms2dirty, say

pytestmark = pytest.mark.gpu
BAR = 5e-7


def _crowded(nrow, cells, fov, seed, wmax=0.5, f0=1e9):
    """u, v within `cells` cells of the centre of a grid of upsampling 2, noise rounded to FP32."""
    rng = np.random.default_rng(seed)
    uvw = (rng.random((nrow, 3)) * 2 - 1) * cells * C / f0 / (fov * np.pi / 180 * 2)
    uvw[:, 2] = (rng.random(nrow) * 2 - 1) * wmax
    vis = (rng.standard_normal(nrow) + 1j * rng.standard_normal(nrow)).astype(np.complex64)
    return uvw, vis, f0


# rows of 64 to 2048 cells (one and several per workgroup; complex cells, and
# components from 2048 on), mixed radix in components (few records a row) and in
# complex cells, rows of 8192 in halves; kernels of 7 and 11
@pytest.mark.parametrize("nx,ny,nrow,eps", [
    (48, 32, 20_000, 1e-6), (64, 64, 60_000, 1e-9), (256, 256, 30_000, 1e-6), (512, 512, 60_000, 1e-6),
    (200, 1024, 80_000, 1e-6), (200, 1023, 40_000, 1e-9), (1024, 1024, 380_000, 1e-6),
    (75, 300, 60_000, 1e-6), (300, 75, 20_000, 1e-9), (300, 600, 40_000, 1e-6), (300, 601, 300_000, 1e-6),
    (40, 3000, 4_000, 1e-6), (128, 4096, 60_000, 1e-6), (127, 4051, 60_000, 1e-9)])
def test_crowded_uv_data(nx, ny, nrow, eps):
    fov = 2.0
    uvw, vis, f0 = _crowded(nrow, 4, fov, nx + ny)
    want = gpu_ms2dirty(uvw, vis, None, nx, ny, fov, f0, eps)
    err = O.l2error(want, gpu_f32(True, uvw, vis, None, nx, ny, fov, f0, eps))
    say(f"[crowded uv data] {nx}x{ny} rows {nrow} eps {eps}: {err:.2e}")
    assert err < BAR


# integer sums (rows of 4096, row parts of 16384), whose crowded blocks of rows run in
# FP64: all rows crowded, or a crowd among rows that are not; strips and layers of bins
# of other sizes, several batches of planes
@pytest.mark.parametrize("nx,ny,nrow,crowd,eps,tuning", [
    (128, 2048, 60_000, 60_000, 1e-6, (0, 0, 0, 0)), (127, 2047, 40_000, 40_000, 1e-9, (0, 0, 0, 0)),
    (64, 8192, 30_000, 30_000, 1e-6, (0, 0, 0, 0)), (63, 8191, 30_000, 30_000, 1e-9, (0, 0, 0, 0)),
    (256, 2048, 60_000, 40_000, 1e-6, (0, 3, 5, 1)), (256, 8192, 60_000, 40_000, 1e-6, (0, 5, 0, 3)),
    (2048, 2048, 200_000, 50_000, 1e-6, (0, 0, 0, 0))])
def test_crowded_blocks_of_integer_rows(nx, ny, nrow, crowd, eps, tuning):
    from curig_amd import _lib as L

    fov = 2.0
    uvw, vis, f0 = _crowded(nrow, 4, fov, nx + ny)
    uvw[crowd:, :2] *= np.array([nx, ny]) / 4 * 0.95
    order = np.random.default_rng(1).permutation(nrow)
    uvw, vis = uvw[order], vis[order]
    want = gpu_ms2dirty(uvw, vis, None, nx, ny, fov, f0, eps)
    lib = L.load()
    assert lib.curig_set_tuning(*tuning) == 0
    try:
        err = O.l2error(want, gpu_f32(True, uvw, vis, None, nx, ny, fov, f0, eps))
    finally:
        lib.curig_set_tuning(0, 0, 0, 0)
    say(f"[crowded blocks] {nx}x{ny} rows {nrow} crowd {crowd} eps {eps} tuning {tuning}: {err:.2e}")
    assert err < BAR


def test_crowded_channels_replayed():
    """One channel of two crowded (the other's rows flagged), replayed as a graph."""
    import torch

    from curig_amd import _lib as L

    nx, ny, nrow, fov, eps = 128, 2048, 60_000, 2.0, 1e-6
    uvw, vis, f0 = _crowded(nrow, 4, fov, 5)
    uvw[50_000:, :2] *= np.array([nx, ny]) / 4 * 0.9
    freq, ms = np.array([f0, 1.02 * f0]), np.stack([vis, vis[::-1]], axis=1)
    flag = np.zeros((nrow, 2), dtype=np.uint8)
    flag[:50_000, 1] = 1
    d_uvw, d_ms, d_flag = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (uvw, ms, flag))
    want = [gpu_ms2dirty(uvw[flag[:, c] == 0], ms[flag[:, c] == 0, c], None, nx, ny, fov, freq[c], eps) for c in range(2)]
    for _ in range(3):
        out = torch.full((2, nx, ny), float("nan"), dtype=torch.complex64, device="cuda")
        L.check(L.load().curig_ms2dirty_multi_dev(nrow, 2, nx, ny, fov, freq, d_uvw.data_ptr(), d_ms.data_ptr(), None,
                                                  d_flag.data_ptr(), out.data_ptr(), 1, eps, 2.0, -1, 1,
                                                  torch.cuda.current_stream().cuda_stream))
        errs = [O.l2error(w, g) for w, g in zip(want, out.cpu().numpy())]
        say(f"[crowded channels] {errs}")
        assert max(errs) < BAR


def test_crowded_uv_data_without_allocation():
    """Whole rows of 8192 in components: the entry point of the smallest working set only."""
    import torch

    from curig_amd import _lib as L

    nx, ny, nrow, fov, eps = 64, 4096, 40_000, 2.0, 1e-6
    uvw, vis, f0 = _crowded(nrow, 4, fov, 9)
    want = gpu_ms2dirty(uvw, vis, None, nx, ny, fov, f0, eps)
    d_uvw, d_vis = torch.from_numpy(uvw).cuda(), torch.from_numpy(vis).cuda()
    out = torch.full((nx, ny), float("nan"), dtype=torch.complex64, device="cuda")
    L.check(L.load().curig_ms2dirty_dev_noalloc(nrow, nx, ny, fov, f0, d_uvw.data_ptr(), d_vis.data_ptr(), None,
                                                out.data_ptr(), eps, 2.0, -1, 1, torch.cuda.current_stream().cuda_stream))
    err = O.l2error(want, out.cpu().numpy())
    say(f"[crowded uv data, no allocation] {nx}x{ny} rows {nrow}: {err:.2e}")
    assert err < BAR
