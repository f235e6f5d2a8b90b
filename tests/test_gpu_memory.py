"""GPU: calls whose usual plan does not fit the device memory left for the
workspace (CURIG_WORKSPACE_LIMIT) run on a plan that does, with the same results:
dense dirty2ms without its full planes, mixed-radix grids on the full-plane path.
A limit below any plan is refused with code 7, and the next call runs."""
import contextlib
import os

import numpy as np
import pytest

from curig_amd import _lib as L
from tests import oracle_helpers as O
from tests.test_gpu_layouts import _case
from tests.test_gpu_parity import gpu_dirty2ms, gpu_f32, gpu_ms2dirty, say

pytestmark = pytest.mark.gpu
MB = 1 << 20


@contextlib.contextmanager
def _limit(nbytes):
    lib = L.load()
    lib.curig_release()
    os.environ["CURIG_WORKSPACE_LIMIT"] = str(nbytes)
    try:
        yield
    finally:
        del os.environ["CURIG_WORKSPACE_LIMIT"]


# buffers at 256^2 (grid 512^2, 16 planes), 60,000 rows: records, taps and sums 16
# MB (FP64), planes of the columns 36 MB, full planes 64 MB; FP32 9, 20 and 32
@pytest.mark.parametrize("precision,limit", [("fp64", 90), ("fp32", 50)])
def test_dense_prediction_without_full_planes(precision, limit):
    n, fov, eps = 256, 2.0, 1e-6
    uvw, vis, wgt, img, f0 = _case(60_000, n, n, fov, 2.0, 11)
    predict = gpu_dirty2ms if precision == "fp64" else (lambda *a: gpu_f32(False, *a))
    want = predict(uvw, img, wgt, n, n, fov, f0, eps)
    with _limit(limit * MB):
        # twice: the second call finds the buffers of the first
        got = [predict(uvw, img, wgt, n, n, fov, f0, eps) for _ in range(2)]
    errs = [O.l2error(want, g) for g in got]
    say(f"[memory] {precision} dense prediction in {limit} MB: {errs}")
    assert max(errs) < (1e-11 if precision == "fp64" else 2e-6)


def test_dense_prediction_of_channels_without_full_planes():
    """The multi-channel form, whose launches replay as one graph."""
    import torch

    n, fov, eps, nchan = 256, 2.0, 1e-6, 2
    uvw, _, _, img, f0 = _case(60_000, n, n, fov, 2.0, 12)
    freq = np.array([f0, 1.1 * f0])
    lib = L.load()
    d_uvw = torch.from_numpy(uvw).cuda()
    d_img = torch.from_numpy(np.stack([img, 1j * img])).cuda()

    def predict():
        out = torch.zeros((len(uvw), nchan), dtype=torch.complex128, device="cuda")
        L.check(lib.curig_dirty2ms_multi_dev(len(uvw), nchan, n, n, fov, freq, d_uvw.data_ptr(), out.data_ptr(), None,
                                             None, d_img.data_ptr(), 0, eps, 2.0, -1, 0,
                                             torch.cuda.current_stream().cuda_stream))
        return out.cpu().numpy()

    want = predict()
    with _limit(90 * MB):
        errs = [O.l2error(want, predict()) for _ in range(3)]
    say(f"[memory] channels in 90 MB: {errs}")
    assert max(errs) < 1e-11


def test_dense_points_without_full_planes():
    """The generic NUFFT, whose packed coordinates stay through the second plan."""
    import torch

    n, m, eps = 256, 100_000, 1e-6
    rng = np.random.default_rng(13)
    u, v = (torch.from_numpy(rng.uniform(-np.pi, np.pi, m)).cuda() for _ in range(2))
    f = torch.from_numpy(rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))).cuda()
    lib = L.load()

    def type2():
        c = torch.zeros(m, dtype=torch.complex128, device="cuda")
        L.check(lib.curig_nufft_dev(2, 2, n, n, 1, m, u.data_ptr(), v.data_ptr(), None, c.data_ptr(), f.data_ptr(), 1,
                                    eps, 2.0, 0, torch.cuda.current_stream().cuda_stream))
        return c.cpu().numpy()

    want = type2()
    # records and taps 26.0e6 bytes, coordinates 2.4e6, sums 1.6e6, image and column plane 3.4e6, full plane 4.2e6
    with _limit(36_000_000):
        err = O.l2error(want, type2())
    say(f"[memory] points in 36 MB: {err:.2e}")
    assert err < 1e-11


# 200,000 rows at kernel width 13: taps 77 MB, everything else below 25 MB
@pytest.mark.parametrize("direction", ["image", "predict"])
def test_mixed_radix_grid_on_full_planes(direction):
    n, fov, eps = 40, 2.0, 1e-12
    uvw, vis, wgt, img, f0 = _case(200_000, n, n, fov, 2.0, 14)
    assert L.plan_info(len(uvw), n, n, fov, f0, eps, 2.0, -1, -2.0, 2.0, 0)["fft_lds"] == 1
    call = ((lambda: gpu_ms2dirty(uvw, vis, wgt, n, n, fov, f0, eps)) if direction == "image"
            else (lambda: gpu_dirty2ms(uvw, img, wgt, n, n, fov, f0, eps)))
    want = call()
    with _limit(60 * MB):
        errs = [O.l2error(want, call()) for _ in range(2)]
    say(f"[memory] {direction} of a mixed-radix grid in 60 MB: {errs}")
    assert max(errs) < 1e-10


def test_a_limit_below_any_plan_is_refused():
    n, fov, eps = 64, 2.0, 1e-6
    uvw, vis, wgt, img, f0 = _case(5_000, n, n, fov, 2.0, 15)
    want = gpu_ms2dirty(uvw, vis, wgt, n, n, fov, f0, eps)
    lib = L.load()
    with _limit(1 << 16):
        out = np.zeros((n, n), dtype=np.complex128)
        code = lib.ms2dirty_2(len(uvw), n, n, fov, f0, np.ascontiguousarray(uvw), np.ascontiguousarray(vis),
                              np.ascontiguousarray(wgt), out, eps, 2.0, -1)
    assert code == 7 and b"allocation" in lib.curig_last_error()
    assert O.l2error(want, gpu_ms2dirty(uvw, vis, wgt, n, n, fov, f0, eps)) < 1e-11
