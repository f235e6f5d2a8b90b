"""bench.py names the kernels that a plan runs: the benchmark workloads' plans and
dense ones, by what gridder.hip's plan_geometry chooses for them."""
import pytest

from bench import kernel_bytes, plan_kernels


def _plan(nx, ny, nf1, nf2, nf3, nvis, rsplit=0, kw=7, fft_lds=1):
    return dict(nx=nx, ny=ny, nf1=nf1, nf2=nf2, nf3=nf3, nvis=nvis, rsplit=rsplit, kw=kw, fft_lds=fft_lds, nbatch=1)


@pytest.mark.parametrize("plan,precision,spread,interp,cols", [
    # 8192^2 and 2048^2: row parts and rows of 4096 on the plane-loop kernels
    (_plan(8192, 8192, 16384, 16384, 1280, 25067520, 4), "fp32", "spread_row_part_planes_kernel",
     "row_ifft_interp_part_planes_kernel", "_reg"),
    (_plan(2048, 2048, 4096, 4096, 180, 2080768), "fp64", "spread_row_part_planes_kernel",
     "row_ifft_interp_part_planes_kernel", ""),
    (_plan(4096, 4096, 8192, 8192, 90, 2080768, 4), "fp64", "spread_row_part_planes_kernel",
     "row_ifft_interp_part_kernel", ""),
    # 256^2, 31,744 rows on 16 planes: dense, the rows formed and gathered from
    (_plan(256, 256, 512, 512, 16, 31744), "fp64", "spread_row_reg_kernel", "row_planes_reg_kernel + interp_gather_kernel",
     ""),
    (_plan(256, 256, 512, 512, 64, 2000), "fp32", "spread_row_reg_kernel", "row_interp_reg_kernel", ""),
    # dense FP32 rows of 4096 leave the plane-loop kernel
    (_plan(2048, 2048, 4096, 4096, 16, 2000000), "fp32", "spread_row_reg_kernel",
     "row_planes_reg_kernel + interp_gather_kernel", ""),
    (_plan(2048, 2048, 4096, 4096, 16, 2000000), "fp64", "spread_row_part_planes_kernel",
     "row_planes_reg_kernel + interp_gather_kernel", ""),
    # mixed radix, also powers of two under an image beyond half the grid
    (_plan(1500, 1100, 2250, 3000, 144, 516096, kw=6), "fp32", "spread_row_mix_kernel", "row_interp_mix_kernel", "_mix"),
    (_plan(800, 800, 1024, 1024, 144, 2000), "fp64", "spread_row_mix_kernel", "row_interp_mix_kernel", "_mix"),
])
def test_kernel_names(plan, precision, spread, interp, cols):
    names = plan_kernels(plan, precision)
    assert names == {"grid": spread, "row_interp": interp, "col_fwd": f"col_fwd{cols}_kernel",
                     "col_inv": f"col_inv{cols}_kernel"}


def test_full_planes_and_gathered_bytes():
    assert plan_kernels(_plan(500, 500, 625, 625, 20, 1000, fft_lds=0), "fp32") == {"grid": "spread_tile_kernel"}
    plan = _plan(256, 256, 512, 512, 16, 31744)
    grid = 16 * 16 * 512 * 512
    assert kernel_bytes([plan], 31744, "fp64", 256, 256)["row_interp"] == grid // 2 + 64 * 31744 + 2 * grid
