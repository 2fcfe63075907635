"""The work whose speed is measured: what a user of the library has it do, through its public entry points.

listed() names the cases, draw() gives more of the same ranges, prepare() makes a case's inputs and handles on the
GPU, run() is one pass, work() what a pass cannot do without, and exact() the result in 64 bits from plain torch.

Families (the `kind` of a case):

  farm       one grid through the per-sector calls (skew, kernel, deskew for each sector, then reduce): a program
             written against the reference's engine class, one engine per image
  viewshed   all sectors (or a worker's share of them) of one DEM in one call, the map back on the host
  batch      viewsheds of several DEMs of uneven sizes in one call
  radon      the Radon / filtered back-projection operator on a stack of slices
  local      the local Radon transform of one slice
  cepstrum   cepstral blur estimation of a stack of images
  fbp        standard parallel-beam projection, ramp filter and back-projection of a stack of slices
  learned    sparse-view reconstruction with the learned filter and the residual CNN
  gradient   the training pass of that model: loss and the gradient of every parameter
"""
import ctypes
import math

import numpy as np
import torch

import skewengine_amd as ske
from skewengine_amd import _lib, learned
from skewengine_amd._lib import check, lib
from skewengine_amd.fbp import FBP, IMAGE, RECON, SINO

F64 = torch.float64


# ---- the cases --------------------------------------------------------------------------------------------------------


def listed():
    return [
        # the smallest grids, call by call: a ported program's sector loop, where latency and launches count
        {"name": "farm_250", "kind": "farm", "n": 250, "observer_m": 1.5, "hurst": 0.8, "hmax_m": 1500.0},
        # one small DEM, the plain total viewshed of the first benchmark configuration
        {"name": "viewshed_500", "kind": "viewshed", "n": 500, "s0": 0, "s1": 180, "observer_m": 1.5, "hurst": 0.8,
         "hmax_m": 1500.0},
        # an ordinary DEM whose side is no multiple of anything, seen from a tower
        {"name": "viewshed_1501_tower", "kind": "viewshed", "n": 1501, "s0": 0, "s1": 180, "observer_m": 12.0,
         "hurst": 0.75, "hmax_m": 3000.0},
        # the headline workload's four sizes, one of each
        {"name": "viewshed_uneven_batch", "kind": "batch", "sides": "1000,2000,3000,4000", "observer_m": 1.5,
         "hurst": 0.8, "hmax_m": 3000.0},
        # one worker's share of the sectors of a DEM with rows past 4096 cells
        {"name": "viewshed_4600_share", "kind": "viewshed", "n": 4600, "s0": 36, "s1": 48, "observer_m": 1.5,
         "hurst": 0.8, "hmax_m": 3000.0},
        # one slice through the skew-space Radon operator (the second benchmark configuration): latency
        {"name": "radon_512", "kind": "radon", "n": 512, "count": 1},
        # a stack of slices through it
        {"name": "radon_512_x16", "kind": "radon", "n": 512, "count": 16},
        # the operator's local form on the same slice
        {"name": "local_radon_512", "kind": "local", "n": 512},
        # blur estimation over a stack of photographs (the third benchmark configuration, fewer images)
        {"name": "cepstrum_1024_x6", "kind": "cepstrum", "n": 1024, "count": 6},
        # projection and reconstruction of a stack of slices in the standard geometry
        {"name": "fbp_512_180x725_x16", "kind": "fbp", "n": 512, "angles": 180, "det": 725, "batch": 16},
        # the configured sparse-view model (32 channels, its trained weights), the benchmark's inference batch
        {"name": "learned_512_c32_x64", "kind": "learned", "n": 512, "angles": 60, "det": 725, "batch": 64,
         "channels": 32},
        # one training pass of the 16-channel model at the batch it is trained with
        {"name": "gradient_512_c16_x16", "kind": "gradient", "n": 512, "angles": 60, "det": 725, "batch": 16,
         "channels": 16},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["farm", "viewshed", "viewshed", "share", "batch", "radon", "radon", "local", "cepstrum", "fbp",
                       "fbp", "learned", "learned", "gradient"])
    dem = {"observer_m": rng.choice([1.5, 1.5, 1.7, 6.0, 12.0, 30.0]), "hurst": round(rng.uniform(0.7, 0.9), 3),
           "hmax_m": rng.choice([300.0, 1500.0, 3000.0])}
    if kind == "farm":
        return dict(dem, kind="farm", n=_log(rng, 48, 420))
    if kind == "viewshed":
        return dict(dem, kind="viewshed", n=_log(rng, 60, 2200), s0=0, s1=180)
    if kind == "share":
        n = _log(rng, 4100, 5600)
        s0 = rng.randrange(0, 168)
        return dict(dem, kind="viewshed", n=n, s0=s0, s1=s0 + max(3, int(12 * (4600.0 / n) ** 3 * rng.uniform(0.6, 1))))
    if kind == "batch":
        sides = [_log(rng, 250, 3000) for _ in range(rng.randint(2, 5))]
        return dict(dem, kind="batch", sides=",".join(str(s) for s in sides))
    if kind == "radon":
        n = _log(rng, 96, 1600)
        return {"kind": "radon", "n": n, "count": max(1, min(_log(rng, 1, 24), int(4 * (1600.0 / n) ** 2)))}
    if kind == "local":
        return {"kind": "local", "n": _log(rng, 80, 800)}
    if kind == "cepstrum":
        n = _log(rng, 120, 1200)
        return {"kind": "cepstrum", "n": n, "count": max(1, min(rng.randint(1, 8), int(6 * (1024.0 / n) ** 2)))}
    n = _log(rng, 128, 700)
    if kind == "fbp":
        return {"kind": "fbp", "n": n, "angles": _log(rng, 30, 360), "det": int(n * math.sqrt(2)) + rng.randint(1, 4),
                "batch": _log(rng, 1, 24)}
    n = 32 * max(2, round(n / 32.0)) if n < 528 else 512
    return {"kind": kind, "n": n, "angles": rng.randint(24, 90), "det": int(n * math.sqrt(2)) + rng.randint(1, 4),
            "batch": _log(rng, 1, 48 if kind == "learned" else 16), "channels": rng.choice([16, 32])}


# ---- inputs -----------------------------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=F64)


def _fbm(n, hurst, g):
    """An n x n window of a fractional Brownian surface (spectral synthesis on the next power of two), in [0, 1]."""
    m = 1 << max(5, (n - 1).bit_length())
    k = torch.hypot(torch.fft.fftfreq(m, device="cuda", dtype=F64)[:, None],
                    torch.fft.rfftfreq(m, device="cuda", dtype=F64)[None, :])
    k[0, 0] = 1.0
    amp = k ** -(hurst + 1.0)
    amp[0, 0] = 0.0
    z = torch.fft.irfft2(torch.polar(amp, 2 * math.pi * _rand(g, *amp.shape)), s=(m, m))[:n, :n]
    z = z - z.min()
    return z / z.max()


def _dem(n, case, g):
    """Heights in cells of 10 m, as the library takes them."""
    return (_fbm(n, case["hurst"], g) * (case["hmax_m"] / 10.0)).float().cpu().numpy()


def _povh(case):
    return float(np.float32(case["observer_m"] / 10.0))


def _ellipses(count, g, many=10):
    """(count, many, 6): centre in the unit disk, semi-axes U[0.05, 0.4], rotation U[0, pi), intensity U[-0.5, 1]."""
    u = _rand(g, count, many, 6)
    r, t = u[..., 0].sqrt(), 2 * math.pi * u[..., 1]
    return torch.stack([r * t.cos(), r * t.sin(), 0.05 + 0.35 * u[..., 2], 0.05 + 0.35 * u[..., 3],
                        math.pi * u[..., 4], -0.5 + 1.5 * u[..., 5]], -1)


def _phantoms(ell, n):
    """The ellipses sampled at the pixel centres of an n x n image on [-1, 1]^2, row 0 at y = +1."""
    c = (torch.arange(n, device="cuda", dtype=F64) + 0.5) / n * 2.0 - 1.0
    x, y = c[None, None, :], -c[None, :, None]
    img = torch.zeros(ell.shape[0], n, n, device="cuda", dtype=F64)
    for e in ell.unbind(1):
        x0, y0, a, b, phi, rho = (v[:, None, None] for v in e.unbind(-1))
        u = ((x - x0) * phi.cos() + (y - y0) * phi.sin()) / a
        v = (-(x - x0) * phi.sin() + (y - y0) * phi.cos()) / b
        img += rho * (u * u + v * v <= 1.0)
    return img.float()


def _sinograms(ell, n, angles, det, g, i0=1e5):
    """The ellipses' line integrals (closed form) measured with Poisson noise at i0 counts (normal approximation)."""
    th = (math.pi / angles) * torch.arange(angles, device="cuda", dtype=F64)[None, :, None]
    s = ((torch.arange(det, device="cuda", dtype=F64) - 0.5 * (det - 1)) * (2.0 / n))[None, None, :]
    p = torch.zeros(ell.shape[0], angles, det, device="cuda", dtype=F64)
    for e in ell.unbind(1):
        x0, y0, a, b, phi, rho = (v[:, None, None] for v in e.unbind(-1))
        w = (a * (th - phi).cos()) ** 2 + (b * (th - phi).sin()) ** 2
        d = s - x0 * th.cos() - y0 * th.sin()
        p += rho * 2 * a * b * (w - d * d).clamp_min(0.0).sqrt() / w
    lam = i0 * (-p).exp()
    z = torch.randn(p.shape, generator=g, device="cuda", dtype=F64)
    return (-((lam + lam.sqrt() * z).round().clamp_min(1.0) / i0).log()).float()


def _blurred(n, g):
    """A texture (fBm, Hurst 0.6) with a linear motion blur of 5 to 40 pixels and noise of sigma 0.01."""
    m = 1 << max(5, (n - 1).bit_length())
    tex = _fbm(m, 0.6, g)
    u = _rand(g, 2).tolist()
    length, ang = 5.0 + 35.0 * u[0], math.pi * u[1]
    t = (torch.arange(int(math.ceil(16 * length)), device="cuda", dtype=F64) + 0.5) / math.ceil(16 * length) - 0.5
    xs, ys = t * length * math.cos(ang), -t * length * math.sin(ang)
    x0, y0 = xs.floor(), ys.floor()
    psf = torch.zeros(m * m, device="cuda", dtype=F64)
    for dx in (0, 1):
        for dy in (0, 1):
            w = (1 - (xs - x0 - dx).abs()) * (1 - (ys - y0 - dy).abs())
            # one sample after another on the host: the sum does not depend on the order of atomic additions
            at = (((y0 + dy) % m) * m + (x0 + dx) % m).long().cpu()
            psf += torch.zeros(m * m, dtype=F64).index_add_(0, at, w.cpu()).cuda()
    psf /= psf.sum()
    img = torch.fft.irfft2(torch.fft.rfft2(tex) * torch.fft.rfft2(psf.view(m, m)), s=(m, m))[:n, :n]
    return (img + 0.01 * torch.randn(n, n, generator=g, device="cuda", dtype=F64)).float()


def _params(case, count, taps_offset, g):
    """For inference in the geometry they were trained in, the committed trained parameters; otherwise a model some way
    into its training: He-normal hidden layers, a small output layer and slightly perturbed Ram-Lak taps."""
    c = case["channels"]
    path = learned.default_weights(case["n"], case["angles"], case["det"], channels=c)
    if path and case["kind"] == "learned":
        return np.load(path, allow_pickle=False)
    p = torch.randn(count, generator=g, device="cuda", dtype=F64)
    cut = [0, 9 * c, 10 * c, 10 * c + 9 * c * c, 11 * c + 9 * c * c, 11 * c + 18 * c * c, 12 * c + 18 * c * c,
           21 * c + 18 * c * c, taps_offset]
    for (a, b), s in zip(zip(cut, cut[1:]), (math.sqrt(2 / 9), 0.05, math.sqrt(2 / 9 / c), 0.05, math.sqrt(2 / 9 / c),
                                             0.05, 0.02, 0.02)):
        p[a:b] *= s
    p[taps_offset:] = _ramlak(case["det"], case["n"]) * (1.0 + 0.05 * p[taps_offset:])
    return p.float().cpu().numpy()


def _model_data(case, seed):
    """(sinograms, targets, parameters) of a learned case."""
    g = _gen(seed)
    ell = _ellipses(case["batch"], g)
    sino = _sinograms(ell, case["n"], case["angles"], case["det"], g)
    c = case["channels"]
    off = 18 * c * c + 21 * c + 1
    return sino, _phantoms(ell, case["n"]), _params(case, off + case["det"], off, g)


# ---- handles and passes -----------------------------------------------------------------------------------------------


class _DeviceArray:
    """A float32 buffer of the library as the array interface describes it; keeps its owner alive."""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (ptr.value, False),
                                         "strides": None, "version": 2}


def _view(ptr, shape, owner):
    return torch.as_tensor(_DeviceArray(ptr, shape, owner), device="cuda")


def _batch(grids):
    """A batch handle and torch views of its output maps in device memory."""
    b = ske.SkewBatch(grids)
    outs = []
    for i, n in enumerate(b.sides):
        p = ctypes.c_void_p()
        check(lib().ske_batch_output_device(b._h, i, ctypes.byref(p)))
        outs.append(_view(p, (n, n), b))
    return b, outs


def _fbp_view(f, which, batch):
    p = ctypes.c_void_p()
    check(lib().ske_fbp_buffer(f._h, which, ctypes.byref(p)))
    return _view(p, f._shape(which, batch), f)


def _inputs(case, seed):
    """The host arrays (or device tensors) a case starts from, as exact() needs them too."""
    g, k = _gen(seed), case["kind"]
    if k in ("farm", "viewshed"):
        return [_dem(case["n"], case, g)]
    if k == "batch":
        return [_dem(int(s), case, g) for s in case["sides"].split(",")]
    if k in ("radon", "local"):
        return list(_phantoms(_ellipses(case.get("count", 1), g), case["n"]).cpu().numpy())
    if k == "cepstrum":
        return [_blurred(case["n"], g).cpu().numpy() for _ in range(case["count"])]
    return list(_phantoms(_ellipses(case["batch"], g), case["n"]).cpu().numpy())


def prepare(case, seed):
    k = case["kind"]
    s = {"case": case}
    if k == "farm":
        s["grid"] = _inputs(case, seed)[0]  # the engine belongs to the pass: one per image, as in the reference
    elif k == "viewshed":
        s["engine"] = ske.SkewEngine(_inputs(case, seed)[0])
    elif k in ("batch", "radon", "cepstrum"):
        s["batch"], s["outs"] = _batch(_inputs(case, seed))
    elif k == "local":
        e = s["engine"] = ske.SkewEngine(_inputs(case, seed)[0])
        e.set_option(_lib.OPT_RADON_LOCAL, 1)
        p = ctypes.c_void_p()
        check(lib().ske_output_device(e._h, ctypes.byref(p)))
        s["outs"] = [_view(p, (case["n"], case["n"]), e)]
    else:
        f = s["fbp"] = FBP(case["n"], case["angles"], case["det"], max_batch=case["batch"])
        if k == "fbp":
            f.upload(IMAGE, np.stack(_inputs(case, seed)))
            s["outs"] = [_fbp_view(f, SINO, case["batch"]), _fbp_view(f, RECON, case["batch"])]
        else:
            sino, target, params = _model_data(case, seed)
            s["model"] = learned.LearnedFBP(f, params=params, channels=case["channels"])
            f.upload(SINO, sino.cpu().numpy())
            f.upload(IMAGE, target.cpu().numpy())
            s["outs"] = [_fbp_view(f, RECON, case["batch"])]
    return s


def run(state):
    case = state["case"]
    k = case["kind"]
    if k == "farm":
        n = case["n"]
        with ske.SkewEngine(state["grid"]) as e:
            e.set_kernel(ske.KERNEL_SDEM, _povh(case))
            for angle in range(180):
                e.skew(angle)
                e.kernel()
                e.deskew()
            return e.reduce(np.zeros((n, n), np.float32))
    if k == "viewshed":
        return state["engine"].run(ske.KERNEL_SDEM, case["s0"], case["s1"], _povh(case))
    if k == "batch":
        state["batch"].run(ske.KERNEL_SDEM, povh=_povh(case))
    elif k == "radon":
        state["batch"].run(ske.KERNEL_RADON)
    elif k == "cepstrum":
        state["batch"].run(ske.KERNEL_CEPSTRUM)
    elif k == "local":
        state["engine"].run(ske.KERNEL_RADON, copy_out=False)
    elif k == "fbp":
        state["fbp"].project(case["batch"])
        state["fbp"].reconstruct(case["batch"])
    elif k == "learned":
        state["model"].reconstruct(case["batch"])
    else:
        loss, grad = state["model"].gradient(case["batch"])
        return {"loss": loss, "grad": grad, "rec": state["outs"][0]}
    return state["outs"]


# ---- work -------------------------------------------------------------------------------------------------------------


def _sector_cells(n, s0=0, s1=180):
    """Skewed cells that hold image data: every pixel feeds two of them at most, one at least."""
    return float(n) * n * (s1 - s0)


def work(case):
    """Inputs read once and outputs written once; operations as the definition of each path has them, where a shorter
    way to the same result is known with that one's count."""
    k = case["kind"]
    if k in ("farm", "viewshed", "batch"):
        sides = [int(s) for s in case["sides"].split(",")] if k == "batch" else [case["n"]]
        s0, s1 = case.get("s0", 0), case.get("s1", 180)
        # per cell and sector: 3 operations to skew, 4 to deskew, and in each of two directions at least one search
        # for the next higher target angle, log2 n tests of 4 operations
        return {"bytes": sum(8.0 * n * n for n in sides),
                "flops": sum(_sector_cells(n, s0, s1) * (7 + 8 * math.log2(n)) for n in sides)}
    if k == "radon":
        n, c = case["n"], case["count"]
        return {"bytes": 8.0 * n * n * c, "flops": c * _sector_cells(n) * (4 + 4)}
    if k == "local":
        n = case["n"]  # a window sum slid, a 64-point real transform of 26 bins (folded), a few output bins
        return {"bytes": 8.0 * n * n, "flops": _sector_cells(n) * (2 + 64 + 2 * 430 + 4 * 52)}
    if k == "cepstrum":
        n, c = case["n"], case["count"]  # 32 bins slid and squared, 32 logarithms, 16 cosine sums (folded)
        return {"bytes": 8.0 * n * n * c, "flops": c * _sector_cells(n) * (32 * 9 + 32 * 10 + 330)}
    n, a, d, b = case["n"], case["angles"], case["det"], case["batch"]
    image, sino = 4.0 * n * n * b, 4.0 * a * d * b
    filt = 5.0 * 2 * a * b * (2 * d) * math.log2(2 * d)
    back = 8.0 * n * n * a * b
    if k == "fbp":
        return {"bytes": 2 * image + sino, "flops": 12.0 * n * n * a * b + filt + back}
    c = case["channels"]
    conv = 2.0 * 9 * (2 * c + 2 * c * c) * n * n * b
    if k == "learned":
        return {"bytes": sino + image, "flops": filt + back + conv}
    return {"bytes": sino + 2 * image, "flops": 2 * (filt + back) + 3 * conv}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------------


def _plan(n, angle):
    """(type, folded angle, target, weight, first, last, rows) of a sector of an n x n grid, by the reference's rules."""
    t = 45 < angle < 135
    kind, new = ((1, 90 - angle) if angle <= 90 else (2, angle - 90)) if t else ((0, angle) if angle <= 90 else (3, 180 - angle))
    skew = math.tan(new * (math.pi / 180.0))
    drift = skew * np.arange(n)
    target = drift.astype(np.int64)
    off = int(skew * (n - 1))
    rows = n + off + 1 if new else n
    first, last = np.zeros(rows + 2, np.int64), np.zeros(rows + 2, np.int64)
    first[n:rows] = n
    last[off:rows] = n
    for j, r in enumerate(target.tolist()):
        for q in (r, r + 1):
            if j > last[q]:
                last[q] = j + 1
        for q in (r + n - 1, r + n):
            if j < first[q]:
                first[q] = j
    return kind, new, target, drift - target, first[:rows], last[:rows], rows


def _oriented(img):
    """The four copies whose rows the sector types read."""
    return [img, img.flip(0, 1).t().contiguous(), img.flip(0).t().contiguous(), img.flip(1)]


def _skewed(src, target, weight, rows):
    n = src.shape[1]
    r = torch.arange(rows, device="cuda")[:, None]
    i = r - target[None, :]
    j = torch.arange(n, device="cuda")[None, :]

    def tap(at):
        return torch.where((at >= 0) & (at < n), src[at.clamp(0, n - 1), j], 0.0)

    return weight * tap(i - 1) + (1 - weight) * tap(i)


def _sectors(img, s0, s1, op, is_max=False):
    """skew -> op -> deskew over the sectors, then reduce; op(sector plans, skewed blocks, live masks) -> blocks."""
    n = img.shape[0]
    copies = _oriented(img)
    acc = [None] * 4
    j = torch.arange(n, device="cuda")[None, :]
    i = torch.arange(n, device="cuda")[:, None]
    stale = None
    group = max(1, min(60, int(2e9 / (16.0 * n * n))))
    for a0 in range(s0, s1, group):
        plans, blocks, lives = [], [], []
        for a in range(a0, min(a0 + group, s1)):
            kind, new, target, weight, first, last, rows = _plan(n, a)
            target, weight, first, last = (torch.from_numpy(v).cuda() for v in (target, weight, first, last))
            plans.append((a, kind, new, target, weight, first, last, rows))
            blocks.append(_skewed(copies[kind], target, weight, rows))
            lives.append((j >= first[:, None]) & (j < last[:, None]))
        for (a, kind, new, target, weight, _, _, rows), block, live in zip(plans, op(plans, blocks, lives), lives):
            block = torch.where(live, block, 0.0)
            below = torch.zeros(1, n, device="cuda", dtype=F64)
            if is_max and new == 0 and stale is not None and stale.shape[0] > rows:
                below = stale[rows:rows + 1]  # the row the sector before left there
            stale = block
            block = torch.cat([block, below])
            u, v = block[i + target[None, :], j], block[i + target[None, :] + 1, j]
            if acc[kind] is None:
                acc[kind] = torch.zeros(n, n, device="cuda", dtype=F64)
            if is_max:
                best = torch.maximum(acc[kind], torch.maximum(u, v))
                acc[kind] = a + 1000.0 * torch.trunc(best / 1000.0)
            else:
                acc[kind] = acc[kind] + (1 - weight) * u + weight * v
    out = torch.zeros(n, n, device="cuda", dtype=F64)
    back = [lambda o: o, lambda o: o.t().flip(0, 1), lambda o: o.t().flip(0), lambda o: o.flip(1)]
    for t in range(4):
        if acc[t] is not None:
            v = back[t](acc[t])
            out = torch.maximum(out, v) if is_max else out + v
    return out


def _viewshed_op(povh):
    def op(plans, blocks, lives):
        n, top = blocks[0].shape[1], max(b.shape[0] for b in blocks)
        S = torch.zeros(len(blocks), top, n, device="cuda", dtype=F64)
        last, first = (torch.zeros(len(blocks), top, 1, device="cuda", dtype=torch.int32) for _ in range(2))
        for k, (p, b) in enumerate(zip(plans, blocks)):
            S[k, :b.shape[0]] = b
            first[k, :p[7], 0] = p[5].int()
            last[k, :p[7], 0] = p[6].int()
        col = torch.arange(n, device="cuda", dtype=torch.int32)
        h = S + povh
        cv = torch.zeros_like(S)
        for step in (1, -1):
            M, od2 = torch.full_like(S, -2000.0), torch.zeros_like(S)
            vis = torch.ones_like(S, dtype=torch.bool)
            for d in range(1, n):
                own = slice(0, n - d) if step > 0 else slice(d, n)
                other = slice(d, n) if step > 0 else slice(0, n - d)
                ang = (S[..., other] - h[..., own]) / d
                m, v = M[..., own], vis[..., own]
                above = ang > m
                inside = col[other] < last if step > 0 else col[other] >= first
                closing = v & ~above & inside
                cv[..., own] += torch.where(closing, float(d) * d - od2[..., own], 0.0)
                od2[..., own] = torch.where(above & ~v, float(d) * d, od2[..., own])
                m.copy_(torch.maximum(m, ang))
                v.copy_(above)
        return [cv[k, :b.shape[0]] / math.cos(p[2] * math.pi / 180.0) ** 2 for k, (p, b) in enumerate(zip(plans, blocks))]
    return op


def _radon_op(plans, blocks, lives):
    out = []
    for b, live in zip(blocks, lives):
        rows = b.shape[0]
        p = torch.where(live, b, 0.0).sum(1).cpu().numpy()
        h2 = 1 << max(0, (rows - 1).bit_length())
        k = np.arange(h2)
        q = np.fft.ifft(np.fft.fft(p, h2) * np.where(k <= rows // 2, k / rows, 0.0)).real[:rows]
        out.append(torch.from_numpy(q).cuda()[:, None].expand_as(b))
    return out


def _local_op(plans, blocks, lives):
    out = []
    k, f, m = np.arange(64), np.arange(26), np.arange(4, 32)
    spec = np.cos(2 * np.pi * np.outer(k, f) / 64) / 8 * np.sin(f / 24.6 * (np.pi / 2))
    back = np.exp(-2j * np.pi * np.outer(f, m) / 64) / 8
    re, im = torch.from_numpy(back.real.copy()).cuda(), torch.from_numpy(back.imag.copy()).cuda()
    for p, b, live in zip(plans, blocks, lives):
        rows, n = b.shape
        sigma = 12.8 * math.cos(p[2] * math.pi / 180.0)
        mat = torch.from_numpy(np.exp(-(k - 32.0) ** 2 / (2 * sigma * sigma))[:, None] * spec).cuda()
        run = torch.nn.functional.pad(torch.where(live, b, 0.0).cumsum(1), (1, 0))
        c = torch.arange(n, device="cuda")
        win = run[:, (c + 33).clamp_max(n)] - run[:, (c - 32).clamp_min(0)]
        win = torch.nn.functional.pad(win, (0, 0, 32, 32))
        got = []
        for r in range(0, rows, 128):
            w = win[r:min(r + 128, rows) + 63].unfold(0, 64, 1).reshape(-1, 64) @ mat
            y = (w @ re) ** 2 + (w @ im) ** 2
            rise = y[:, 1:] > y[:, :-1]
            at = rise.int().argmax(1)
            got.append(torch.where(rise.any(1), y.gather(1, at[:, None])[:, 0], 0.0).view(-1, n))
        out.append(torch.cat(got))
    return out


def _cepstrum_op(plans, blocks, lives):
    out = []
    k = np.arange(32)
    dft = np.exp(-2j * np.pi * np.outer(np.arange(64), k) / 64) / 8
    re, im = torch.from_numpy(dft.real.copy()).cuda(), torch.from_numpy(dft.imag.copy()).cuda()
    cos = torch.from_numpy(np.cos(2 * np.pi * np.outer(k, np.arange(16)) / 32) / math.sqrt(32)).cuda()
    for b, live in zip(blocks, lives):
        rows, n = b.shape
        x = torch.nn.functional.pad(torch.where(live, b, 0.0), (32, 31))
        got = []
        for r in range(0, rows, 256):
            w = x[r:r + 256].unfold(1, 64, 1).reshape(-1, 64)
            power = ((w @ re) ** 2 + (w @ im) ** 2).clamp_min(1e-300)
            v = -(power.log() @ cos).clamp_max(0.0)
            rise = v[:, 5:] > v[:, 4:-1]
            i0 = torch.where(rise.any(1), rise.int().argmax(1) + 5, 16)
            idx = torch.arange(16, device="cuda")[None, :]
            keep = (idx == i0[:, None] - 1) | (idx > i0[:, None])
            val = torch.where(keep, v, 0.0).amax(1)
            got.append((torch.where(i0 < 16, val, 0.0) * 10000).view(-1, n))
        out.append(torch.cat(got))
    return out


def _ramlak(det, n):
    """Half of the symmetric ramp filter times the bin spacing, for |m| = 0 .. det - 1."""
    delta = 2.0 / n
    m = torch.arange(det, device="cuda", dtype=F64)
    h = torch.where(m % 2 == 1, -1.0 / (math.pi * m.clamp_min(1.0) * delta) ** 2, 0.0)
    h[0] = 1.0 / (4 * delta * delta)
    return h * delta


def _project(img, angles, det):
    n = img.shape[0]
    delta = 2.0 / n
    pad = torch.nn.functional.pad(img, (1, 1, 1, 1)).reshape(-1)
    s = ((torch.arange(det, device="cuda", dtype=F64) - 0.5 * (det - 1)) * delta)[:, None]
    t = ((torch.arange(det, device="cuda", dtype=F64) - 0.5 * (det - 1)) * delta)[None, :]
    rows = []
    for a in range(angles):
        c, sn = math.cos(math.pi * a / angles), math.sin(math.pi * a / angles)
        u, v = (s * c - t * sn + 1) / delta - 0.5, (1 - s * sn - t * c) / delta - 0.5
        fu, fv = u.floor(), v.floor()
        inside = (fu >= -1) & (fu < n) & (fv >= -1) & (fv < n)
        at = ((fv.clamp(-1, n - 1) + 1) * (n + 2) + fu.clamp(-1, n - 1) + 1).long()
        wu, wv = u - fu, v - fv
        top = pad[at] * (1 - wu) + pad[at + 1] * wu
        low = pad[at + n + 2] * (1 - wu) + pad[at + n + 3] * wu
        rows.append(torch.where(inside, top * (1 - wv) + low * wv, 0.0).sum(1) * delta)
    return torch.stack(rows)


def _filtered(p, half):
    """The rows of p convolved with the symmetric taps."""
    det = p.shape[-1]
    d = torch.arange(det, device="cuda")
    return p @ half[(d[:, None] - d[None, :]).abs()]


def _backproject(q, n):
    angles, det = q.shape
    delta = 2.0 / n
    x = ((torch.arange(n, device="cuda", dtype=F64) + 0.5) * delta - 1.0)[None, :]
    y = (1.0 - (torch.arange(n, device="cuda", dtype=F64) + 0.5) * delta)[:, None]
    wide = torch.nn.functional.pad(q, (2, 2))
    out = torch.zeros(n, n, device="cuda", dtype=F64)
    for a in range(angles):
        k = (x * math.cos(math.pi * a / angles) + y * math.sin(math.pi * a / angles)) / delta + 0.5 * (det - 1)
        f = k.floor()
        at = (f.clamp(-2, det) + 2).long()
        w = k - f
        out = out + wide[a][at] * (1 - w) + wide[a][at + 1] * w
    return out * (math.pi / angles)


def _conv(x, w, b):
    """3 x 3 convolution with zero padding: x (ci, n, n), w (co, 9, ci), taps row by row."""
    n = x.shape[-1]
    p = torch.nn.functional.pad(x, (1, 1, 1, 1))
    y = 0.0
    for t in range(9):
        y = y + (w[:, t] @ p[:, t // 3:t // 3 + n, t % 3:t % 3 + n].reshape(x.shape[0], -1)).view(-1, n, n)
    return y + b[:, None, None]


def _model(params, sino, n, c):
    cut = [9 * c, c, 9 * c * c, c, 9 * c * c, c, 9 * c, 1]
    w1, b1, w2, b2, w3, b3, w4, b4, half = params.split(cut + [params.numel() - sum(cut)])
    r0 = _backproject(_filtered(sino, half), n)
    a = torch.relu(_conv(r0[None], w1.view(c, 9, 1), b1))
    a = torch.relu(_conv(a, w2.view(c, 9, c), b2))
    a = torch.relu(_conv(a, w3.view(c, 9, c), b3))
    return r0 + _conv(a, w4.view(1, 9, c), b4)[0]


def exact(case, seed):
    k = case["kind"]
    if k in ("learned", "gradient"):
        sino, target, params = _model_data(case, seed)
        n, c, b = case["n"], case["channels"], case["batch"]
        p = torch.from_numpy(params).cuda().to(F64)
        if k == "learned":
            with torch.no_grad():
                return [torch.stack([_model(p, s.to(F64), n, c) for s in sino])]
        p.requires_grad_(True)
        loss, recs = 0.0, []
        for s, t in zip(sino, target):
            rec = _model(p, s.to(F64), n, c)
            part = ((rec - t.to(F64)) ** 2).sum() / (b * n * n)
            part.backward()
            loss += float(part.detach())
            recs.append(rec.detach())
        return {"loss": loss, "grad": p.grad.cpu().numpy(), "rec": torch.stack(recs)}
    grids = [torch.from_numpy(g).cuda().to(F64) for g in _inputs(case, seed)]
    if k == "fbp":
        sinos = [_project(g, case["angles"], case["det"]) for g in grids]
        half = _ramlak(case["det"], case["n"])
        return [torch.stack(sinos), torch.stack([_backproject(_filtered(s, half), case["n"]) for s in sinos])]
    if k in ("farm", "viewshed", "batch"):
        # the scans take n steps over all cells: maps of up to about a thousand cells a side
        todo = [g.shape[0] ** 3 * (case.get("s1", 180) - case.get("s0", 0)) <= 180e9 for g in grids]
        if not any(todo):
            return None
        outs, op = [], _viewshed_op(_povh(case))
        for g, one in zip(grids, todo):
            outs.append(_sectors(g, case.get("s0", 0), case.get("s1", 180), op) if one else None)
            if one and k == "batch":
                todo[:] = [False] * len(todo)  # one grid of the batch
                outs += [None] * (len(grids) - len(outs))
                break
        return outs if k == "batch" else outs[0].cpu().numpy()
    if k == "radon":
        return [_sectors(g, 0, 180, _radon_op) if i < 4 else None for i, g in enumerate(grids)]
    if k == "local":
        return [_sectors(grids[0], 0, 180, _local_op)]
    return [_sectors(g, 0, 180, _cepstrum_op, True) if i == 0 else None for i, g in enumerate(grids)]
