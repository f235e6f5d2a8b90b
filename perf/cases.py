"""The work that users of the gridder have it do, as timed cases.

A case is one pass through a public entry point: imaging (ms2dirty: visibilities
to a dirty image), prediction (dirty2ms: an image to visibilities), a gradient
of the imaging loss, a host-array major cycle through the Python binding, a
NIFTY-style call, or a generic NUFFT.  Observations are synthetic arrays as in
the benchmark: antennas uniform in a disk, all baselines rotated through a range
of hour angles at declination -30 degrees; visibilities of a few dozen point
sources plus noise; weights U[0.5, 1]; flags i.i.d. at a fraction per channel.
Everything is made from the seed, on the GPU where the entry point takes device
memory."""
import ctypes
import math

import numpy as np
import torch

from curig_amd import _lib, autograd, cursl
from curig_amd.curagridder import dirty2vis, vis2dirty

C_LIGHT = 299792458.0
DEC = math.radians(-30.0)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _case(name, form, precision, nx, ny, fov, eps, nant, radius, nsnap, hours, nchan=1, f0=1.0e9, f1=1.4e9, sigma=2.0,
          flags=0.0):
    c = dict(form=form, precision=precision, nx=nx, ny=ny, fov=fov, eps=eps, nant=nant, radius=radius, nsnap=nsnap,
             hours=hours, nchan=nchan, f0=f0, f1=f1, sigma=sigma, flags=flags)
    if name:
        c["name"] = name
    return c


def _nufft(name, dim, n1, n2, n3, m, eps, precision):
    c = dict(form="nufft", dim=dim, n1=n1, n2=n2, n3=n3, m=m, eps=eps, precision=precision)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest calls: a 32-antenna, 1 km array, 31,744 rows on a 256^2
        # image.  Quick-look imaging in FP64, and the model prediction of a
        # calibration loop in FP32: launches and host work count here.
        _case("image_256_fp64", "image", "fp64", 256, 256, 2.0, 1e-6, 32, 1000.0, 64, 2.0, f0=1.4e9),
        _case("predict_256_fp32", "predict", "fp32", 256, 256, 2.0, 1e-6, 32, 1000.0, 64, 2.0, f0=1.4e9),
        # The Python binding as a script uses it: host arrays, its default
        # upsampling factor 1.25 and epsilon, one major cycle (prediction of the
        # model, then the image of the residual).  The grid (640^2) is no power of two.
        _case("host_cycle_512_fp64", "host_cycle", "fp64", 512, 512, 2.0, 1e-6, 32, 1500.0, 128, 3.0, f0=1.4e9,
              sigma=1.25),
        # Gradient-based imaging: one evaluation of the loss and its gradient
        # (dirty2ms forward, ms2dirty backward) on a 64-antenna, 3 km array.
        _case("gradient_1024_fp32", "gradient", "fp32", 1024, 1024, 2.0, 1e-6, 64, 3000.0, 512, 4.0, f0=1.4e9),
        # The drop-in double-precision path on a 128-antenna, 5 km array, four
        # channels with an image each.
        _case("image_2048_4ch_fp64", "image", "fp64", 2048, 2048, 4.0, 1e-6, 128, 5000.0, 256, 3.0, nchan=4),
        # The same observation predicted in FP32-mixed precision.
        _case("predict_2048_4ch_fp32", "predict", "fp32", 2048, 2048, 4.0, 1e-6, 128, 5000.0, 256, 3.0, nchan=4),
        # A few channels of a flagged spectral-line observation, an image per channel.
        _case("image_4096_4ch_flagged_fp32", "image", "fp32", 4096, 4096, 3.0, 1e-5, 128, 5000.0, 256, 3.0, nchan=4,
              f0=1.0e9, f1=1.5e9, flags=0.2),
        # Images whose padded sizes are no powers of two, as most pixel counts
        # chosen by hand: a wide FP32 image and an FP64 prediction.
        _case("image_1500x1100_fp32", "image", "fp32", 1500, 1100, 4.0, 1e-5, 64, 5000.0, 256, 3.0),
        _case("predict_3000x2500_fp64", "predict", "fp64", 3000, 2500, 3.0, 1e-6, 64, 5000.0, 256, 3.0),
        # The largest image: 8192^2 over a 6 degree field, 2.08 million rows.
        _case("image_8192_fp32", "image", "fp32", 8192, 8192, 6.0, 1e-6, 128, 5000.0, 256, 3.0),
        _case("predict_8192_fp32", "predict", "fp32", 8192, 8192, 6.0, 1e-6, 128, 5000.0, 256, 3.0),
        # The generic 2-D NUFFT: 20 million points, type 1 then type 2.
        _nufft("nufft_2d_4096_20m_fp32", 2, 4096, 4096, 1, 20000000, 1e-5, "fp32"),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi):
    """An image side: half of the draws powers of two, the others any number."""
    n = _log_uniform(rng, lo, hi)
    if rng.random() < 0.5:
        return 1 << int(round(math.log2(n)))
    return int(n)


def draw(rng):
    form = rng.choice(["image", "image", "predict", "predict", "gradient", "host_cycle", "nifty", "nufft"])
    precision = rng.choice(["fp32", "fp64"])
    eps = rng.choice([1e-4, 1e-5, 1e-6] if precision == "fp32" else [1e-5, 1e-6, 1e-8, 1e-10])
    if form == "nufft":
        dim = rng.choice([1, 2, 2, 2, 3])
        m = int(_log_uniform(rng, 2e4, 1e7))
        if dim == 1:
            return _nufft(None, 1, int(_log_uniform(rng, 256, 65536)), 1, 1, m, eps, precision)
        if dim == 2:
            return _nufft(None, 2, _size(rng, 64, 4096), _size(rng, 64, 4096), 1, m, eps, precision)
        return _nufft(None, 3, _size(rng, 16, 128), _size(rng, 16, 128), rng.randint(4, 32), min(m, 1000000), eps,
                      precision)
    host = form in ("host_cycle", "nifty")
    top = 1024 if host else 8192
    nx = _size(rng, 100, top)
    ny = nx if rng.random() < 0.5 else min(top, max(100, int(nx * rng.uniform(0.6, 1.4))))
    nant = rng.randint(16, 48 if host else 128)
    nsnap = int(_log_uniform(rng, 8, 128 if host else 256))
    nchan = rng.choice([1, 2, 3, 4]) if form in ("image", "predict", "nifty") else 1
    flags = rng.choice([0.0, rng.uniform(0.05, 0.4)]) if nchan > 1 else 0.0
    sigma = 1.25 if form == "host_cycle" and rng.random() < 0.5 else 2.0
    c = _case(None, form, precision, nx, ny, round(rng.uniform(1.0, 6.0), 2), eps, nant,
              round(_log_uniform(rng, 500.0, 6000.0), 1), nsnap, round(rng.uniform(1.0, 4.0), 2), nchan=nchan,
              f0=1.0e9, f1=1.4e9, sigma=sigma, flags=round(flags, 3))
    # no more than the largest listed case: shorter baselines need fewer w planes
    limit = 0.5 * _cells(listed()[9])
    weight = (2.0 if precision == "fp64" else 1.0) * (1.0 if form in ("image", "predict") else 2.0)
    while weight * _cells(c) > limit and c["radius"] > 50.0:
        c["radius"] = round(0.7 * c["radius"], 1)
        if c["nchan"] > 1:
            c["nchan"] -= 1
            c["flags"] = c["flags"] if c["nchan"] > 1 else 0.0
    return c


# ---------------------------------------------------------------------------
# sizes and the work a pass cannot do without
# ---------------------------------------------------------------------------
def _freqs(c):
    return np.linspace(c["f0"], c["f1"], c["nchan"]) if c["nchan"] > 1 else np.array([c["f0"]])


def _rows(c):
    return c["nant"] * (c["nant"] - 1) // 2 * c["nsnap"]


def _width(eps, sigma):
    """The kernel width that epsilon and the upsampling factor select."""
    if sigma == 2.0:
        return max(2, math.ceil(-math.log10(eps / 10.0)))
    return max(2, math.ceil(-math.log(eps) / (math.pi * math.sqrt(1.0 - 1.0 / sigma))))


def _planes(c, f):
    """About the number of w planes of a channel (the array's longest w from its
    radius; half the range of n - 1 from the field)."""
    half = math.radians(c["fov"]) / 2.0
    s = (1.0 - math.sqrt(1.0 - 2.0 * half * half)) / 2.0
    x = 2 * math.pi * f / C_LIGHT * 1.7 * c["radius"] * math.cos(DEC)
    return 2.0 * c["sigma"] * s * x / math.pi + _width(c["eps"], c["sigma"]) + 1


def _cells(c):
    return sum(_planes(c, f) for f in _freqs(c)) * c["sigma"] ** 2 * c["nx"] * c["ny"]


def work(case):
    """Bytes: rows, visibilities, weights, flags and images once each.
    Operations: the kernel's taps (4 each: two multiply-adds), and per w plane
    the FFTs along one axis of the whole plane and along the other of the image's
    columns, and the plane's phase and sum at each pixel (8 operations)."""
    c = case
    cs, rs = (16, 8) if c["precision"] == "fp64" else (8, 4)
    if c["form"] == "nufft":
        n = c["n1"] * c["n2"] * c["n3"]
        kw = _width(c["eps"], 2.0)
        grid = n * 2 ** c["dim"]
        return {"bytes": 2.0 * (c["m"] * (8 * c["dim"] + cs) + n * cs),
                "flops": 2.0 * (4.0 * c["m"] * kw ** c["dim"] + 5.0 * grid * math.log2(grid))}
    rows, nchan, npix, s = _rows(c), c["nchan"], c["nx"] * c["ny"], c["sigma"]
    keep = rows * nchan * (1.0 - c["flags"])
    images = nchan if c["form"] in ("image", "predict") else 1
    kw = _width(c["eps"], s)
    bytes_ = 24.0 * rows + rows * nchan * (cs + rs + (1 if c["flags"] else 0)) + images * npix * cs
    flops = 4.0 * keep * kw ** 3
    n1, n2 = s * c["ny"], s * c["nx"]
    for f in _freqs(c):
        per_plane = 5.0 * n1 * n2 * math.log2(n1) + 5.0 * c["ny"] * n2 * math.log2(n2) + 8.0 * npix
        flops += _planes(c, f) * per_plane
    passes = 2 if c["form"] in ("gradient", "host_cycle") else 1
    return {"bytes": passes * bytes_, "flops": passes * flops}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _uvw(c, rng):
    """[rows, 3] metres, FP64, on the GPU: all baselines at each snapshot."""
    n = c["nant"]
    r = c["radius"] * np.sqrt(rng.random(n))
    th = 2 * np.pi * rng.random(n)
    xyz = np.stack([r * np.cos(th), r * np.sin(th), rng.uniform(-20, 20, n)], axis=1)
    i, j = np.triu_indices(n, 1)
    x, y, z = torch.from_numpy((xyz[j] - xyz[i]).T.copy()).cuda()
    ha = torch.from_numpy(np.deg2rad(np.linspace(-c["hours"], c["hours"], c["nsnap"]) * 15.0)).cuda()[:, None]
    sh, ch, sd, cd = torch.sin(ha), torch.cos(ha), math.sin(DEC), math.cos(DEC)
    u = sh * x + ch * y
    v = -sd * ch * x + sd * sh * y + cd * z
    w = cd * ch * x - cd * sh * y + sd * z
    return torch.stack([u, v, w], dim=-1).reshape(-1, 3).contiguous()


def _sources(c, rng, count=30):
    half = math.radians(c["fov"]) / 2.0
    return (rng.uniform(-half, half, count), rng.uniform(-half, half, count),
            np.exp(rng.uniform(np.log(0.01), np.log(1.0), count)))


def _visibilities(c, uvw, sources, gen, cdtype):
    """[rows, nchan]: the sources' visibilities plus noise of sigma 0.1."""
    rows = uvw.shape[0]
    vis = torch.randn((rows, c["nchan"], 2), generator=gen, device="cuda", dtype=torch.float32).to(torch.float64) * 0.1
    u, v, w = uvw[:, 0], uvw[:, 1], uvw[:, 2]
    for k, f in enumerate(_freqs(c)):
        t = 2 * math.pi * f / C_LIGHT
        for l, m, flux in zip(*sources):
            nm1 = math.sqrt(1.0 - l * l - m * m) - 1.0
            ph = t * (u * l + v * m - w * nm1)
            vis[:, k, 0] += flux * torch.cos(ph)
            vis[:, k, 1] -= flux * torch.sin(ph)
    return torch.view_as_complex(vis).to(cdtype).contiguous()


def _image(c, sources, gen, images, cdtype):
    """[images, nx, ny]: a model sky, the sources on their pixels over faint noise."""
    sky = torch.randn((images, c["nx"], c["ny"]), generator=gen, device="cuda", dtype=torch.float32) * 0.01
    half = math.radians(c["fov"]) / 2.0
    for l, m, flux in zip(*sources):
        i = min(c["nx"] - 1, int((l / half + 1) / 2 * c["nx"]))
        j = min(c["ny"] - 1, int((m / half + 1) / 2 * c["ny"]))
        sky[:, i, j] += flux
    return sky.to(cdtype)


def prepare(case, seed):
    c = dict(case)
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    fp64 = c["precision"] == "fp64"
    cd, rd = (torch.complex128, torch.float64) if fp64 else (torch.complex64, torch.float32)
    s = {"case": c, "lib": _lib.load(), "prec": 0 if fp64 else 1}
    if c["form"] == "nufft":
        m = c["m"]
        x = (torch.rand((c["dim"], m), generator=gen, device="cuda", dtype=torch.float64) * 2 - 1) * math.pi
        s["x"] = [x[i].contiguous() for i in range(c["dim"])]
        s["c"] = torch.randn((m, 2), generator=gen, device="cuda", dtype=rd)
        s["c"] = torch.view_as_complex(s["c"])
        s["fk"] = torch.empty((c["n3"], c["n2"], c["n1"]), dtype=cd, device="cuda")
        s["back"] = torch.empty(m, dtype=cd, device="cuda")
        return s
    uvw = _uvw(c, rng)
    sources = _sources(c, rng)
    nchan, rows = c["nchan"], uvw.shape[0]
    wgt = torch.rand((rows, nchan), generator=gen, device="cuda", dtype=torch.float32).to(rd) * 0.5 + 0.5
    flag = None
    if c["flags"]:
        flag = (torch.rand((rows, nchan), generator=gen, device="cuda") < c["flags"]).to(torch.uint8)
    s["freqs"] = _freqs(c)
    needs_vis = c["form"] != "predict"
    needs_image = c["form"] != "image"
    vis = _visibilities(c, uvw, sources, gen, cd) if needs_vis else None
    image = _image(c, sources, gen, nchan if c["form"] == "predict" else 1, cd) if needs_image else None
    if c["form"] in ("host_cycle", "nifty"):
        s["uvw"] = uvw.cpu().numpy()
        s["wgt"] = wgt.cpu().numpy()
        s["vis"] = vis.cpu().numpy()
        s["image"] = np.ascontiguousarray(image[0].cpu().numpy())
        s["mask"] = None if flag is None else 1 - flag.cpu().numpy()
        return s
    s.update(uvw=uvw, wgt=wgt, vis=vis, image=image, flag=flag)
    if nchan == 1 and flag is None:
        s["geo"] = autograd.GridderGeometry(uvw, float(s["freqs"][0]), c["nx"], c["ny"], c["fov"], epsilon=c["eps"],
                                            wgt=wgt.reshape(-1), sigma=c["sigma"])
    elif c["form"] == "image":
        s["image"] = torch.empty((nchan, c["nx"], c["ny"]), dtype=cd, device="cuda")
    else:
        s["vis"] = torch.empty((rows, nchan), dtype=cd, device="cuda")
    if c["form"] == "gradient":
        s["image"] = image[0].real.contiguous().requires_grad_()
        s["vis"] = vis[:, 0].contiguous()
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _ptr(t):
    return None if t is None else t.data_ptr()


def _multi(s, fn):
    """Every channel of a device-resident observation, an image per channel."""
    c = s["case"]
    _lib.check(fn(s["uvw"].shape[0], c["nchan"], c["nx"], c["ny"], c["fov"], s["freqs"], _ptr(s["uvw"]),
                  _ptr(s["vis"]), _ptr(s["wgt"]), _ptr(s["flag"]), _ptr(s["image"]), 1, c["eps"], c["sigma"], -1,
                  s["prec"], ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))


def _run_nufft(s):
    c = s["case"]
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    x = [_ptr(t) for t in s["x"]] + [None] * (3 - c["dim"])
    for kind, data in ((1, s["c"]), (2, s["back"])):
        _lib.check(s["lib"].curig_nufft_dev(kind, c["dim"], c["n1"], c["n2"], c["n3"], c["m"], x[0], x[1], x[2],
                                            _ptr(data), _ptr(s["fk"]), 1 if kind == 1 else -1, c["eps"], 2.0,
                                            s["prec"], stream))
    return {"modes": s["fk"], "points": s["back"]}


def _run_host_cycle(s):
    c = s["case"]
    fp = c["precision"]
    freq, wgt, model = s["freqs"], s["wgt"].reshape(-1), s["image"]
    predicted = np.zeros(s["uvw"].shape[0], dtype=model.dtype)
    dirty2vis(s["uvw"], freq, predicted, None, model, c["fov"], epsilon=c["eps"], sigma=c["sigma"], precision=fp)
    residual = s["vis"].reshape(-1) - predicted
    dirty = np.zeros((c["nx"], c["ny"]), dtype=model.dtype)
    vis2dirty(s["uvw"], freq, residual, wgt, dirty, c["fov"], epsilon=c["eps"], sigma=c["sigma"], precision=fp)
    return {"predicted": predicted, "dirty": dirty}


def _run_nifty(s):
    c = s["case"]
    px, py = math.radians(c["fov"]) / c["nx"], math.radians(c["fov"]) / c["ny"]
    dirty = cursl.ms2dirty(s["uvw"], s["freqs"], s["vis"], s["wgt"], c["nx"], c["ny"], px, py, 0, 0, c["eps"], True,
                           mask=s["mask"])
    return {"dirty": dirty}


def run(state):
    s = state
    c = s["case"]
    if c["form"] == "nufft":
        return _run_nufft(s)
    if c["form"] == "host_cycle":
        return _run_host_cycle(s)
    if c["form"] == "nifty":
        return _run_nifty(s)
    if c["form"] == "gradient":
        # the loss |A x - V|^2 / 2 and its gradient
        predicted = autograd.dirty2ms(s["image"], s["geo"])
        residual = predicted - s["vis"]
        loss = 0.5 * (residual.real.square().sum() + residual.imag.square().sum())
        (grad,) = torch.autograd.grad(loss, s["image"])
        return {"predicted": predicted.detach(), "loss": loss.detach(), "grad": grad}
    if c["form"] == "image":
        if "geo" in s:
            return {"dirty": autograd.ms2dirty(s["vis"].reshape(-1), s["geo"])}
        _multi(s, s["lib"].curig_ms2dirty_multi_dev)
        return {"dirty": s["image"]}
    if "geo" in s:
        return {"vis": autograd.dirty2ms(s["image"][0], s["geo"])}
    _multi(s, s["lib"].curig_dirty2ms_multi_dev)
    return {"vis": s["vis"]}


# ---------------------------------------------------------------------------
# direct sums in FP64
# ---------------------------------------------------------------------------
TERMS = 6e10  # phase terms of a direct sum that stays within seconds


def _pixels(c, uvw):
    """l, m, n - 1 of every pixel, FP64, [nx * ny]."""
    half = math.radians(c["fov"]) / 2.0
    l = (torch.arange(c["nx"], device="cuda", dtype=torch.float64) - c["nx"] // 2) * (2 * half / c["nx"])
    m = (torch.arange(c["ny"], device="cuda", dtype=torch.float64) - c["ny"] // 2) * (2 * half / c["ny"])
    l, m = torch.meshgrid(l, m, indexing="ij")
    l, m = l.reshape(-1), m.reshape(-1)
    r2 = l * l + m * m
    return l, m, -r2 / (torch.sqrt(1.0 - r2) + 1.0)


def _blocks(count, per):
    for a in range(0, count, per):
        yield slice(a, min(count, a + per))


def _direct(a, b, val, sign):
    """out[i] = sum_j val[j] e^{i sign <a_i, b_j>}: a [p, k], b [q, k], val [q, channels]."""
    out = torch.zeros((a.shape[0], val.shape[1]), dtype=torch.complex128, device="cuda")
    pa, pb = 4096, 16384
    re, im = val.real.contiguous(), val.imag.contiguous()
    for i in _blocks(a.shape[0], pa):
        for j in _blocks(b.shape[0], pb):
            ph = a[i] @ b[j].T
            co, si = torch.cos(ph), torch.sin(ph) * sign
            out[i] += torch.complex(co @ re[j] - si @ im[j], co @ im[j] + si @ re[j])
    return out


def _sum_image(c, uvw, freq, val, wsign):
    """[nx, ny]: sum_j val_j e^{2 pi i f/c (u l + v m + wsign w (n - 1))} / n."""
    l, m, nm1 = _pixels(c, uvw)
    k = 2 * math.pi * freq / C_LIGHT
    out = _direct(torch.stack([l, m, wsign * nm1], 1) * k, uvw, val.to(torch.complex128)[:, None], 1)
    return (out[:, 0] / (1.0 + nm1)).reshape(c["nx"], c["ny"])


def _sum_vis(c, uvw, freq, image, wsign):
    """[rows]: the adjoint of _sum_image."""
    l, m, nm1 = _pixels(c, uvw)
    k = 2 * math.pi * freq / C_LIGHT
    val = image.to(torch.complex128).reshape(-1) / (1.0 + nm1)
    return _direct(uvw * k, torch.stack([l, m, wsign * nm1], 1), val[:, None], -1)[:, 0]


def _exact_nufft(s):
    """Type 1 by matrix products of the points' waves, and type 2 of those modes."""
    c = s["case"]
    dim, per = c["dim"], max(1024, int(1e8 / max(c["n1"], c["n2"])))
    ks = [torch.arange(n, device="cuda", dtype=torch.float64) - n // 2 for n in (c["n1"], c["n2"], c["n3"])]

    def wave(d, j, sign):
        ph = s["x"][d][j][:, None] * ks[d] if d < dim else torch.zeros((j.stop - j.start, 1), device="cuda",
                                                                      dtype=torch.float64)
        return torch.complex(torch.cos(ph), sign * torch.sin(ph))

    modes = torch.zeros((c["n3"], c["n2"], c["n1"]), dtype=torch.complex128, device="cuda")
    points = torch.zeros(c["m"], dtype=torch.complex128, device="cuda")
    for j in _blocks(c["m"], per):
        right = s["c"][j].to(torch.complex128)[:, None] * wave(0, j, 1.0)
        e2, e3 = wave(1, j, 1.0).T.contiguous(), wave(2, j, 1.0)
        for k in range(c["n3"]):
            modes[k] += e2 @ (e3[:, k:k + 1] * right)
    for j in _blocks(c["m"], per):
        e1, e2, e3 = wave(0, j, -1.0), wave(1, j, -1.0), wave(2, j, -1.0)
        for k in range(c["n3"]):
            points[j] += ((e2 @ modes[k]) * e1).sum(1) * e3[:, k]
    return {"modes": modes, "points": points}


def exact(case, seed):
    c = dict(case)
    if c["form"] != "nufft":
        terms = float(_rows(c)) * c["nx"] * c["ny"] * c["nchan"] * (2 if c["form"] in ("gradient", "host_cycle") else 1)
        if terms > TERMS:
            return None
    elif 8.0 * c["m"] * c["n1"] * c["n2"] * c["n3"] > 1e14:
        return None
    s = prepare(case, seed)
    if c["form"] == "nufft":
        return _exact_nufft(s)
    dev = lambda a: torch.as_tensor(a).cuda()  # noqa: E731
    uvw, wgt, freqs = dev(s["uvw"]), dev(s["wgt"]).to(torch.float64), s["freqs"]
    if c["form"] == "host_cycle":
        # the binding's sign of w is +1; the prediction carries no weights
        predicted = _sum_vis(c, uvw, freqs[0], dev(s["image"]), 1.0)
        residual = dev(s["vis"]).reshape(-1).to(torch.complex128) - predicted
        dirty = _sum_image(c, uvw, freqs[0], residual * wgt[:, 0], 1.0)
        return {"predicted": predicted.cpu().numpy(), "dirty": dirty.cpu().numpy()}
    if c["form"] == "nifty":
        keep = wgt if s["mask"] is None else wgt * dev(s["mask"])
        vis = dev(s["vis"]).to(torch.complex128) * keep
        dirty = sum(_sum_image(c, uvw, freqs[k], vis[:, k], -1.0) for k in range(c["nchan"]))
        return {"dirty": dirty.real.cpu().numpy()}
    if c["form"] == "gradient":
        image = s["image"].detach()
        predicted = _sum_vis(c, uvw, freqs[0], image, -1.0) * wgt[:, 0]
        residual = predicted - s["vis"].to(torch.complex128)
        grad = _sum_image(c, uvw, freqs[0], residual * wgt[:, 0], -1.0).real
        return {"predicted": predicted, "loss": 0.5 * residual.abs().square().sum(), "grad": grad}
    keep = wgt if s["flag"] is None else wgt * (s["flag"] == 0)
    if c["form"] == "image":
        vis = s["vis"].to(torch.complex128) * keep
        images = [_sum_image(c, uvw, freqs[k], vis[:, k], -1.0) for k in range(c["nchan"])]
        return {"dirty": images[0] if "geo" in s else torch.stack(images)}
    vis = [_sum_vis(c, uvw, freqs[k], s["image"][k], -1.0) * keep[:, k] for k in range(c["nchan"])]
    return {"vis": vis[0] if "geo" in s else torch.stack(vis, 1)}
