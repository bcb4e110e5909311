"""The work a user of this package has it do, as cases that can be timed and compared.

``listed()`` names twelve cases over the package's public entry points, from
a bundle of a thousand rays to the 134M-ray-evaluation calibration step;
``draw()`` gives further ones of the same ranges.  ``prepare`` makes what a
program holds before the call (inputs on the GPU, the model, a workspace or
plan it keeps), ``run`` makes the call, ``exact`` states the same results in
64 bits with plain torch, and ``work`` what a pass cannot do without.

The kinds of case and what each stands for:

  rays      ``run_to_end`` / ``run_to_image``: a ray bundle through a column
            of elements, optionally counted into a detector image
  source    ``PointSource.make_rays`` and ``run_to_image`` on its rays: a new
            bundle generated and imaged, the first lines of most programs
  fit       ``STEMFitWorkspace.run``: one loss-and-gradient evaluation of the
            4D-STEM geometry calibration
  forward   ``stem_forward``: detector coordinates and sample values of every
            ray, or the simulated 4D dataset
  backproj  ``backproject``: a 4D dataset onto the sample plane, with weights
  beamlets  ``make_gaussian_image``: a field as a sum of Gaussian beamlets,
            and its gradient where ``grad`` is set
  gaussfit  ``GaussianFitBatch.loss_and_grad``: one step of many Gaussian
            decomposition fits at once
"""
import math

import numpy as np
import torch

from temgymcore_amd import stem
from temgymcore_amd.components import Deflector, Detector, Lens, Rotator
from temgymcore_amd.gauss_fit import GaussianFitBatch
from temgymcore_amd.gaussian import GaussianRay, make_gaussian_image
from temgymcore_amd.ray import Ray
from temgymcore_amd.run import run_to_end, run_to_image
from temgymcore_amd.source import PointSource

DTYPES = {"f32": torch.float32, "f64": torch.float64}


def listed():
    return [
        # interactive use: a small double-precision bundle through a lens
        dict(name="rays_small", kind="rays", n=1000, dtype="f64", elements=2, side=128, image=False),
        # the plain workload: 1,048,576 single-precision rays, lens, detector image
        dict(name="rays_image", kind="rays", n=1 << 20, dtype="f32", elements=2, side=128, image=True),
        # a whole column (lenses, scan coils, image rotations) in double
        # precision onto a full-size camera, an odd number of rays
        dict(name="rays_column", kind="rays", n=4194301, dtype="f64", elements=10, side=1024, image=True),
        # a new ring-sampled bundle, generated and imaged
        dict(name="source_image", kind="source", num=500000, elements=2, side=256),
        # the calibration step of the headline configuration: 64x64 scan,
        # 64x64 rays, 8 camera lengths
        dict(name="fit_headline", kind="fit", scan_h=64, scan_w=64, n_side=64, cams=8),
        # calibration on a small, ragged scan (every iteration of an L-BFGS loop)
        dict(name="fit_ragged", kind="fit", scan_h=13, scan_w=21, n_side=46, cams=3),
        # the forward model of the 16.7M-ray configuration
        dict(name="forward_values", kind="forward", scan_h=64, scan_w=64, n_side=64, cams=1, det_h=256, det_w=256,
             dataset=False),
        # a simulated 4D-STEM dataset: 64x64 images of 256x256 pixels
        dict(name="forward_dataset", kind="forward", scan_h=64, scan_w=64, n_side=64, cams=1, det_h=256, det_w=256,
             dataset=True),
        # mean back-projected image (values and weights) of a ragged scan
        dict(name="backproject", kind="backproj", scan_h=61, scan_w=67, n_side=62, det_h=250, det_w=256),
        # aperture diffraction: 131,072 untilted beamlets on 1024x1024 pixels, 4-sigma cut
        dict(name="beamlets_aperture", kind="beamlets", n=131072, height=1024, width=1024, cutoff=4.0, round=True,
             grad=False),
        # a decomposed wave (tilted, rotated astigmatic beamlets) through a
        # lens, with the gradient of every beamlet parameter and of the lens matrix
        dict(name="beamlets_gradient", kind="beamlets", n=2048, height=500, width=612, cutoff=0.0, round=False,
             grad=True),
        # 256 uneven fits, 3 to 2000 Gaussians on 128 to 512 pixel squares
        dict(name="gaussfit_batch", kind="gaussfit", instances=256, n_max=2000, side_max=512),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["rays", "rays", "source", "fit", "forward", "backproj", "beamlets", "beamlets", "gaussfit"])
    if kind == "rays":
        return dict(kind=kind, n=log_int(1000, 4194301), dtype=rng.choice(["f32", "f64"]),
                    elements=rng.randint(2, 10), side=log_int(100, 1024), image=rng.random() < 0.7)
    if kind == "source":
        return dict(kind=kind, num=log_int(1000, 500000), elements=rng.randint(2, 6), side=log_int(100, 512))
    scan = dict(scan_h=log_int(5, 64), scan_w=log_int(5, 64), n_side=2 * log_int(8, 32))
    if kind == "fit":
        return dict(kind=kind, **scan, cams=rng.randint(1, 8))
    if kind == "forward":
        return dict(kind=kind, **scan, cams=rng.randint(1, 3), det_h=log_int(64, 256), det_w=log_int(64, 256),
                    dataset=rng.random() < 0.5)
    if kind == "backproj":
        return dict(kind=kind, **scan, det_h=log_int(64, 256), det_w=log_int(64, 256))
    if kind == "beamlets":
        round_ = rng.random() < 0.5
        grad = (not round_) and rng.random() < 0.7
        return dict(kind=kind, n=log_int(64, 131072 if round_ else 4096), height=log_int(64, 1024 if round_ else 600),
                    width=log_int(64, 1024 if round_ else 612), cutoff=rng.choice([0.0, 4.0]) if not round_ else 4.0,
                    round=round_, grad=grad)
    return dict(kind=kind, instances=log_int(2, 200), n_max=log_int(30, 2000), side_max=log_int(140, 512))


# ---------------------------------------------------------------------------
# inputs: plain tensors made from (case, seed)
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _uniform(g, lo, hi, *shape, dtype=torch.float64):
    return torch.rand(*shape, generator=g, device="cuda", dtype=dtype) * (hi - lo) + lo


def _column(elements, seed):
    """(kind, z, value) of `elements` - 1 optical elements, 0.5 m apart, and the detector's z."""
    rng = np.random.default_rng(int(seed))
    col = []
    for i in range(elements - 1):
        kind = ("lens", "deflector", "lens", "rotator")[i % 4]
        if kind == "lens":
            v = float(rng.uniform(0.8, 1.2))
        elif kind == "deflector":
            v = tuple(float(a) for a in rng.uniform(-5e-3, 5e-3, 2))
        else:
            v = float(rng.uniform(-40.0, 40.0))
        col.append((kind, 0.5 * (i + 1), v))
    return col, 0.5 * elements


def _column_model(col, z_det, side):
    make = {"lens": lambda z, v: Lens(z=z, focal_length=v), "rotator": lambda z, v: Rotator(z=z, angle=v),
            "deflector": lambda z, v: Deflector(z=z, def_x=v[0], def_y=v[1])}
    return [make[k](z, v) for k, z, v in col] + [
        Detector(z=z_det, pixel_size=(1.28 / side, 1.28 / side), shape=(side, side))]


def _ray_arrays(case, seed):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    x, y = (_uniform(g, -0.1, 0.1, case["n"]).to(dt) for _ in range(2))
    dx, dy = (_uniform(g, -0.05, 0.05, case["n"]).to(dt) for _ in range(2))
    return x, y, dx, dy


def _source_of(seed):
    rng = np.random.default_rng(int(seed))
    return float(rng.uniform(0.03, 0.06)), tuple(float(v) for v in rng.uniform(-0.05, 0.05, 2))


STEM = dict(step=1e-10, rotation=12.0, semi_conv=0.5e-3, defocus=200e-9, pivot=1e4, det_pixel=2.5e-6,
            sample=512, sample_pixel=2e-11)


def _stem_params(cams, seed):
    """The parameter vector (descan 16, step, rotation, camera lengths) of one calibration."""
    L = [0.5] if cams == 1 else list(np.linspace(0.1, 1.0, cams))
    return np.concatenate([np.random.default_rng(int(seed)).normal(0.0, 1e-3, 16), [STEM["step"], STEM["rotation"]], L])


def _stem_model(case, p):
    cams = tuple(float(v) for v in p[18:])
    return stem.STEMModel(scan_shape=(case["scan_h"], case["scan_w"]), scan_step=float(p[16]),
                          scan_rotation=float(p[17]), n_side=case["n_side"], semi_conv=STEM["semi_conv"],
                          defocus=STEM["defocus"], pivot=STEM["pivot"], descan=p[:16].reshape(4, 4),
                          camera_lengths=cams, det_shape=(case.get("det_h", 256), case.get("det_w", 256)),
                          det_pixel=STEM["det_pixel"], sample_shape=(STEM["sample"],) * 2,
                          sample_pixel=STEM["sample_pixel"])


def _slopes(n):
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    return ((k - 0.5 * (n - 1)) * (2.0 * STEM["semi_conv"] / n)).float().double()


def _scan(case, p):
    """(spx, spy) [S] of the parameter tensor p (float64)."""
    h, w = case["scan_h"], case["scan_w"]
    i, j = torch.meshgrid(torch.arange(h, device="cuda", dtype=torch.float64),
                          torch.arange(w, device="cuda", dtype=torch.float64), indexing="ij")
    u, v = (i.reshape(-1) - 0.5 * (h - 1)) * p[16], (j.reshape(-1) - 0.5 * (w - 1)) * p[16]
    phi = p[17] * (math.pi / 180.0)
    return -torch.sin(phi) * u + torch.cos(phi) * v, -(torch.cos(phi) * u + torch.sin(phi) * v)


def _detector_axes(case, p, c):
    """x [S, n] over the slope columns and y [S, n] over the slope rows on camera c."""
    spx, spy = _scan(case, p)
    v = torch.stack([spx, spy, STEM["pivot"] * spx, STEM["pivot"] * spy])
    row = p[:16].reshape(4, 4) @ v
    d, L, t = STEM["defocus"], p[18 + c], _slopes(case["n_side"])
    bx, by = v[2] * d + row[0] + row[2] * L, v[3] * d + row[1] + row[3] * L
    return t * (d + L) + bx[:, None], t * (d + L) + by[:, None]


def _targets(case, seed):
    """Measured detector coordinates: those of slightly different parameters, f32 [C, S, J, 2]."""
    p = _stem_params(case["cams"], seed)
    p = torch.from_numpy(p * (1.0 + 1e-3 * np.random.default_rng(int(seed) + 1).normal(size=p.shape))).cuda()
    n, S = case["n_side"], case["scan_h"] * case["scan_w"]
    t = torch.empty((case["cams"], S, n, n, 2), dtype=torch.float32, device="cuda")
    for c in range(case["cams"]):
        x, y = _detector_axes(case, p, c)
        t[c, ..., 0] = x[:, None, :].float()
        t[c, ..., 1] = y[:, :, None].float()
    return t.reshape(case["cams"], S, n * n, 2)


def _sample(seed):
    return _uniform(_gen(seed), -math.pi, math.pi, STEM["sample"], STEM["sample"]).float()


def _dataset(case, seed):
    """Camera frames: low counts over the whole detector, f32 [S, H, W]."""
    S = case["scan_h"] * case["scan_w"]
    return torch.rand(S, case["det_h"], case["det_w"], generator=_gen(seed), device="cuda", dtype=torch.float32) * 20


BEAM = {True: dict(lam=1.97e-12, pix=4e-8, L=0.3), False: dict(lam=1.97e-12, pix=1e-8, L=1e-2, f=2e-2)}


def _beamlet_arrays(case, seed):
    """Beamlet parameters (f64, amplitude complex128) and the 5x5 ray-transfer matrix."""
    g, n, b = _gen(seed), case["n"], BEAM[case["round"]]
    T = torch.eye(5, dtype=torch.float64)
    if case["round"]:  # plane wave behind a round aperture, free space
        r, a = 5e-6 * torch.sqrt(_uniform(g, 0, 1, n)), _uniform(g, 0, 2 * math.pi, n)
        z = torch.zeros(n, dtype=torch.float64, device="cuda")
        q = dict(x=r * torch.cos(a), y=r * torch.sin(a), dx=z, dy=z.clone(),
                 amplitude=torch.ones(n, dtype=torch.complex128, device="cuda"),
                 waist_xy=torch.full((n, 2), 5e-8, dtype=torch.float64, device="cuda"),
                 radii_of_curv=torch.full((n, 2), math.inf, dtype=torch.float64, device="cuda"), theta=z.clone())
        T[0, 2] = T[1, 3] = b["L"]
    else:
        hx, hy = 0.4 * case["width"] * b["pix"], 0.4 * case["height"] * b["pix"]
        q = dict(x=_uniform(g, -hx, hx, n), y=_uniform(g, -hy, hy, n), dx=_uniform(g, -2e-5, 2e-5, n),
                 dy=_uniform(g, -2e-5, 2e-5, n),
                 amplitude=torch.polar(_uniform(g, 0.3, 1.5, n), _uniform(g, -math.pi, math.pi, n)),
                 waist_xy=_uniform(g, 6e-8, 1.4e-7, n, 2), radii_of_curv=_uniform(g, 0.3, 3.0, n, 2),
                 theta=_uniform(g, -1.5, 1.5, n))
        # half the drift, a lens, the other half
        half, f = 0.5 * b["L"], b["f"]
        A, B, C, D = 1 - half / f, 2 * half - half * half / f, -1 / f, 1 - half / f
        for k in (0, 1):
            T[k, k], T[k, k + 2], T[k + 2, k], T[k + 2, k + 2] = A, B, C, D
    return q, T.cuda()


def _cotangent(case, seed):
    g = _gen(seed + 1)
    return torch.complex(torch.randn(case["height"], case["width"], generator=g, device="cuda"),
                         torch.randn(case["height"], case["width"], generator=g, device="cuda"))


def _fit_tables(case):
    """Gaussian counts (log-uniform from 3) and square detector sides of the instances."""
    counts = np.rint(np.exp(np.random.default_rng(5).uniform(math.log(3), math.log(case["n_max"]), case["instances"])))
    sides = np.random.default_rng(6).integers(128, case["side_max"] + 1, case["instances"])
    return counts.astype(int).tolist(), sides.astype(int).tolist()


FIT_PIXEL, FIT_WAVELENGTH = 1e-6, 2.51e-12


def _fit_arrays(case, seed):
    """Parameter rows [G, 16] f64 and measured intensities [pixels] f32 (smooth spots and noise)."""
    counts, sides = _fit_tables(case)
    g, G = _gen(seed), sum(counts)
    half = torch.repeat_interleave(torch.tensor([0.4 * s * FIT_PIXEL for s in sides], dtype=torch.float64,
                                                device="cuda"), torch.tensor(counts, device="cuda"))
    p = torch.zeros(G, 16, dtype=torch.float64, device="cuda")
    p[:, 0:2] = _uniform(g, -1, 1, G, 2) * half[:, None]
    p[:, 2:4] = _uniform(g, -2e-3, 2e-3, G, 2)
    amp = torch.polar(_uniform(g, 0.2, 1.0, G), _uniform(g, -math.pi, math.pi, G))
    p[:, 5], p[:, 6] = amp.real, amp.imag
    p[:, 7:9] = _uniform(g, 5e-6, 25e-6, G, 2)
    p[:, 9:11] = math.inf
    p[:, 11] = FIT_WAVELENGTH
    p[:, 12] = _uniform(g, -math.pi / 2, math.pi / 2, G)
    target = torch.rand(sum(s * s for s in sides), generator=g, device="cuda") * 0.05
    spots = torch.rand(len(sides), 3, 4, generator=g, device="cuda")
    at = 0
    for i, s in enumerate(sides):
        t = torch.arange(s, device="cuda") / s
        fy = torch.exp(-((t - spots[i, 0, :, None]) / 0.12) ** 2)
        fx = torch.exp(-((t - spots[i, 1, :, None]) / 0.12) ** 2)
        target[at:at + s * s] += (3.0 * fy.T @ (spots[i, 2, :, None] * fx)).reshape(-1)
        at += s * s
    return p, target


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind == "rays":
        x, y, dx, dy = _ray_arrays(case, seed)
        s["rays"] = Ray(x=x, y=y, dx=dx, dy=dy, z=0.0, pathlength=0.0)
        s["model"] = _column_model(*_column(case["elements"], seed), case["side"])
    elif kind == "source":
        semi_conv, offset = _source_of(seed)
        s["source"] = PointSource(z=0.0, semi_conv=semi_conv, offset_xy=offset)
        s["model"] = _column_model(*_column(case["elements"], seed), case["side"])
    elif kind in ("fit", "forward", "backproj"):
        p = _stem_params(case.get("cams", 1), seed)
        s["model"] = _stem_model(case, p)
        s["params"] = torch.from_numpy(p).cuda()
        if kind == "fit":
            s["targets"] = _targets(case, seed)
            s["workspace"] = stem.STEMFitWorkspace(s["model"], s["params"].device)
        elif kind == "forward":
            s["sample"] = _sample(seed)
        else:
            s["data"] = _dataset(case, seed)
    elif kind == "beamlets":
        q, T = _beamlet_arrays(case, seed)
        b = BEAM[case["round"]]
        s["leaves"] = {}
        if case["grad"]:
            s["leaves"] = {k: v.requires_grad_() for k, v in dict(q, abcd=T).items() if k != "radii_of_curv"}
            s["cotangent"] = _cotangent(case, seed)
        s["abcd"] = T if case["grad"] else None
        s["rays"] = GaussianRay(z=0.0, pathlength=0.0, wavelength=b["lam"], **q)
        det = Detector(z=b["L"], pixel_size=(b["pix"],) * 2, shape=(case["height"], case["width"]))
        s["model"] = [det] if case["round"] else [Lens(z=0.5 * b["L"], focal_length=b["f"]), det]
    else:
        counts, sides = _fit_tables(case)
        grids = [Detector(z=0.0, pixel_size=(FIT_PIXEL,) * 2, shape=(n, n)) for n in sides]
        s["batch"] = GaussianFitBatch(grids, counts)
        s["params"], s["target"] = _fit_arrays(case, seed)
    return s


def _ray_outputs(ray, image=None):
    out = dict(x=ray.x, y=ray.y, dx=ray.dx, dy=ray.dy, pathlength=ray.pathlength)
    return out if image is None else dict(out, image=image)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "rays":
        if case["image"]:
            return _ray_outputs(*run_to_image(s["rays"], s["model"]))
        return _ray_outputs(run_to_end(s["rays"], s["model"]))
    if kind == "source":
        rays = s["source"].make_rays(case["num"])
        out, image = run_to_image(rays, s["model"])
        return dict(_ray_outputs(out, image), dx0=rays.dx, dy0=rays.dy)
    if kind == "fit":
        return s["workspace"].run(s["params"], s["targets"])
    if kind == "forward":
        return stem.stem_forward(s["model"], s["params"], s["sample"], coords=not case["dataset"],
                                 values=not case["dataset"], image4d=case["dataset"])
    if kind == "backproj":
        return list(stem.backproject(s["model"], s["data"], s["params"], weights=True))
    if kind == "beamlets":
        field = make_gaussian_image(s["rays"], s["model"], cutoff=case["cutoff"] or None, abcd=s["abcd"])
        if not case["grad"]:
            return {"field": field}
        grads = torch.autograd.grad(field, list(s["leaves"].values()), grad_outputs=s["cotangent"])
        return dict({"field": field.detach()}, **dict(zip(s["leaves"], grads)))
    loss, grad = s["batch"].loss_and_grad(s["params"], s["target"])
    return {"loss": loss, "grad": grad}


# ---------------------------------------------------------------------------
# the work of a pass: inputs read once, outputs written once, and the
# operations of the sums themselves
# ---------------------------------------------------------------------------
def _ring_counts(num):
    rings = max(1, int(math.floor((-1 + math.sqrt(1 + 4 * num / math.pi)) / 2)))
    kth = np.round(2 * np.pi * np.arange(1, rings + 1)).astype(int)
    return np.round(kth * (num / kth.sum())).astype(int)


def work(case):
    kind = case["kind"]
    if kind in ("rays", "source"):
        size = 4 if case.get("dtype") == "f32" else 8
        n = case["n"] if kind == "rays" else int(_ring_counts(case["num"]).sum())
        # a source reads nothing and writes its four fields too
        image = 4 * case["side"] ** 2 if case.get("image", True) else 0
        return {"bytes": 9 * size * n + image, "flops": 12 * n * case["elements"]}
    if kind in ("fit", "forward", "backproj"):
        evals = case["scan_h"] * case["scan_w"] * case["n_side"] ** 2
        if kind == "fit":
            return {"bytes": 8 * evals * case["cams"], "flops": 30 * evals * case["cams"]}
        det = 4 * case["scan_h"] * case["scan_w"] * case["det_h"] * case["det_w"]
        image = 4 * STEM["sample"] ** 2
        if kind == "backproj":  # one detector value a ray, two f64 images written
            return {"bytes": 4 * min(evals, det // 4) + 4 * image, "flops": 40 * evals}
        if case["dataset"]:
            return {"bytes": det + image, "flops": 40 * evals}
        return {"bytes": (8 * case["cams"] + 4) * evals + image, "flops": 30 * evals}
    if kind == "beamlets":
        # a complex multiply-add for each beamlet and each pixel inside its cut
        # (4 waists, or exp(-80) where nothing is cut), and three more for the
        # moments of the gradient
        b, npix = BEAM[case["round"]], case["height"] * case["width"]
        w0, shrink = (5e-8, 1.0) if case["round"] else (1e-7, 1 - 0.5 * b["L"] / b["f"])
        w = math.hypot(w0 * shrink, b["L"] * b["lam"] / (math.pi * w0)) / b["pix"]
        pairs = case["n"] * min(npix, math.pi * w * w * (case["cutoff"] or math.sqrt(80.0)) ** 2)
        return {"bytes": 8 * npix * (2 if case["grad"] else 1) + 8 * 13 * case["n"] * (2 if case["grad"] else 1),
                "flops": pairs * (32 if case["grad"] else 8)}
    counts, sides = _fit_tables(case)
    w = 15.0 * math.sqrt(80.0)
    pairs = sum(n * min(s * s, math.pi * w * w) for n, s in zip(counts, sides))
    return {"bytes": 4 * sum(s * s for s in sides) + 2 * 128 * sum(counts), "flops": 32 * pairs}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _exact_column(x, y, dx, dy, col, z_det):
    z, pl = 0.0, torch.zeros_like(x)
    for kind, zc, v in col + [("detector", z_det, None)]:
        x, y, pl, z = x + dx * (zc - z), y + dy * (zc - z), pl + (zc - z), zc
        if kind == "lens":
            dx, dy, pl = dx - x / v, dy - y / v, pl - (x * x + y * y) / (2 * v)
        elif kind == "deflector":
            pl, dx, dy = pl + dx * x + dy * y, dx + v[0], dy + v[1]
        elif kind == "rotator":
            c, s = math.cos(math.radians(v)), math.sin(math.radians(v))
            x, y, dx, dy = x * c - y * s, x * s + y * c, dx * c - dy * s, dx * s + dy * c
    return dict(x=x, y=y, dx=dx, dy=dy, pathlength=pl)


def _exact_rings(num, radius):
    """(r cos a, r sin a) of the ring sampling: the angle adds up its ring's
    step from one restart to the next, restart k lying k points after the
    start of ring k."""
    per = _ring_counts(num)
    n, rings = int(per.sum()), len(per)
    ring = np.repeat(np.arange(rings), per)
    total = np.cumsum((2 * np.pi / per)[ring])
    first = np.concatenate([[0], np.cumsum(per)[:-1]])
    restart = np.array([k + f for k, f in enumerate(first) if k + f < n])
    v = np.arange(n)
    angle = total - total[restart[np.searchsorted(restart, v, side="right") - 1]]
    r = radius * (ring + 1) / rings
    return torch.from_numpy(r * np.cos(angle)).cuda(), torch.from_numpy(r * np.sin(angle)).cuda()


def _exact_fit(case, seed):
    p = torch.from_numpy(_stem_params(case["cams"], seed)).cuda().requires_grad_()
    t = _targets(case, seed)
    n = case["n_side"]
    loss, grad = 0.0, 0.0
    for c in range(case["cams"]):
        x, y = _detector_axes(case, p, c)
        tc = t[c].reshape(-1, n, n, 2).double()
        part = ((x[:, None, :] - tc[..., 0]) ** 2).sum() + ((y[:, :, None] - tc[..., 1]) ** 2).sum()
        grad = grad + torch.autograd.grad(part, p)[0]
        loss = loss + part.detach()
    return torch.cat([grad, loss.reshape(1)])


def _sample_pixels(case, p):
    """Sample-plane pixel coordinates (row [S, n] over slope rows, column [S, n] over slope columns)."""
    spx, spy = _scan(case, p)
    t, d, k = _slopes(case["n_side"]), STEM["defocus"], 1 + STEM["pivot"] * STEM["defocus"]
    mid = 0.5 * (STEM["sample"] - 1)
    return mid - (k * spy[:, None] + t * d) / STEM["sample_pixel"], mid + (k * spx[:, None] + t * d) / STEM["sample_pixel"]


def _neighbours(case, p):
    """The four bilinear neighbours of every ray: (flat sample index, weight) [S, n, n] each."""
    fy, fx = _sample_pixels(case, p)
    n = STEM["sample"]
    y0, x0 = torch.floor(fy), torch.floor(fx)
    for a in (0, 1):
        for b in (0, 1):
            yy, xx = (y0 + a).long(), (x0 + b).long()
            wy, wx = (fy - y0) if a else 1 - (fy - y0), (fx - x0) if b else 1 - (fx - x0)
            wy, wx = wy * ((yy >= 0) & (yy < n)), wx * ((xx >= 0) & (xx < n))
            yield (yy.clamp(0, n - 1)[:, :, None] * n + xx.clamp(0, n - 1)[:, None, :], wy[:, :, None] * wx[:, None, :])


def _frame_pixels(case, p):
    """(flat index into [S, H, W], on the detector) [S, n, n] of every ray on camera 0."""
    x, y = _detector_axes(case, p, 0)
    H, W = case["det_h"], case["det_w"]
    py = torch.round(0.5 * (H - 1) - y / STEM["det_pixel"]).long()
    px = torch.round(0.5 * (W - 1) + x / STEM["det_pixel"]).long()
    ok = ((py >= 0) & (py < H))[:, :, None] & ((px >= 0) & (px < W))[:, None, :]
    s = torch.arange(x.shape[0], device="cuda")[:, None, None]
    return s * (H * W) + py.clamp(0, H - 1)[:, :, None] * W + px.clamp(0, W - 1)[:, None, :], ok


def _exact_forward(case, seed):
    p = torch.from_numpy(_stem_params(case["cams"], seed)).cuda()
    sample, n = _sample(seed).double().reshape(-1), case["n_side"]
    S = case["scan_h"] * case["scan_w"]
    values = sum(w * sample[i] for i, w in _neighbours(case, p))
    if case["dataset"]:
        at, ok = _frame_pixels(case, p)
        image = torch.zeros(S * case["det_h"] * case["det_w"], dtype=torch.float64, device="cuda")
        image.index_add_(0, at[ok], values[ok])
        return {"image4d": image.reshape(S, case["det_h"], case["det_w"])}
    coords = torch.empty((case["cams"], S, n, n, 2), dtype=torch.float64, device="cuda")
    for c in range(case["cams"]):
        x, y = _detector_axes(case, p, c)
        coords[c, ..., 0], coords[c, ..., 1] = x[:, None, :], y[:, :, None]
    return {"coords": coords.reshape(case["cams"], S, n * n, 2), "values": values.reshape(S, n * n)}


def _exact_backproject(case, seed):
    p = torch.from_numpy(_stem_params(1, seed)).cuda()
    at, ok = _frame_pixels(case, p)
    v = torch.where(ok, _dataset(case, seed).reshape(-1)[at].double(), 0.0)
    image, weight = (torch.zeros(STEM["sample"] ** 2, dtype=torch.float64, device="cuda") for _ in range(2))
    for i, w in _neighbours(case, p):
        image.index_add_(0, i.reshape(-1), (w * v).reshape(-1))
        weight.index_add_(0, i.reshape(-1), (w * ok).reshape(-1))
    return [image.reshape((STEM["sample"],) * 2), weight.reshape((STEM["sample"],) * 2)]


def _mat(a, b, c, d):
    return torch.stack([torch.stack([a, b], -1), torch.stack([c, d], -1)], -2)


def _det(m):
    return m[..., 0, 0] * m[..., 1, 1] - m[..., 0, 1] * m[..., 1, 0]


def _inv(m):
    return _mat(m[..., 1, 1], -m[..., 0, 1], -m[..., 1, 0], m[..., 0, 0]) / _det(m)[..., None, None]


def _mul(a, b):
    return (a[..., :, :, None] * b[..., None, :, :]).sum(-2)


def _vec(m, v):
    return (m * v[..., None, :]).sum(-1)


def _exponents(q, lam, T=None):
    """Coefficients [n, 6] over (x^2, x y, y^2, x, y, 1) of the exponent of
    every beamlet of unit amplitude and wavelength lam [n]: after the
    ray-transfer matrix T, or in its own plane."""
    k = 2 * math.pi / lam
    qi = torch.complex(-1.0 / q["radii_of_curv"], lam[:, None] / (math.pi * q["waist_xy"] ** 2))
    c, s = torch.cos(q["theta"]), torch.sin(q["theta"])
    off = (qi[:, 0] - qi[:, 1]) * c * s
    Q = _mat(qi[:, 0] * c * c + qi[:, 1] * s * s, off, off, qi[:, 0] * s * s + qi[:, 1] * c * c)
    r1 = torch.stack([q["x"], q["y"]], -1).to(torch.complex128)
    t1 = torch.stack([q["dx"], q["dy"]], -1).to(torch.complex128)
    if T is None:
        L = 2 * t1 - 2 * _vec(Q, r1)
        const = (r1 * _vec(Q, r1)).sum(-1) - 2 * (t1 * r1).sum(-1)
        log_pref = torch.zeros_like(const)
    else:
        A, B, C, D = (T[i:i + 2, j:j + 2].to(torch.complex128) for i in (0, 2) for j in (0, 2))
        M = A + _mul(B, Q)
        r2 = _vec(A, r1) + _vec(B, t1)
        Qi = _inv(Q)
        X = _mul(Qi, _inv(_mul(B, _mul(A, Qi) + B)))
        L = 2 * _vec(X.transpose(-1, -2), r2) - 2 * _vec(_inv(B).transpose(-1, -2), r1)
        const = (r1 * _vec(_mul(A, _inv(B)), r1)).sum(-1) - (r2 * _vec(X, r2)).sum(-1)
        log_pref = -torch.log(torch.sqrt(_det(M)))
        Q = _mul(_inv(M), C + _mul(D, Q))
        Q = 0.5 * (Q + Q.transpose(-1, -2))
        # the offsets of the matrix: positions count from e, and f tilts the wave
        e, f = T[0:2, 4].to(torch.complex128), T[2:4, 4].to(torch.complex128)
        L = L + 2 * f
        const = const + (e * _vec(Q, e.expand_as(r1))).sum(-1) - (L * e).sum(-1)
        L = L - 2 * _vec(Q, e.expand_as(r1))
    h = 0.5j * k
    return torch.stack([h * Q[:, 0, 0], h * (Q[:, 0, 1] + Q[:, 1, 0]), h * Q[:, 1, 1], h * L[:, 0], h * L[:, 1],
                        h * const + log_pref], -1)


def _monomials(height, width, pix):
    """[6, H W]: x^2, x y, y^2, x, y, 1 at the pixel centres (y points up)."""
    y = ((0.5 * (height - 1) - torch.arange(height, device="cuda", dtype=torch.float64)) * pix)[:, None].expand(height, width)
    x = ((torch.arange(width, device="cuda", dtype=torch.float64) - 0.5 * (width - 1)) * pix)[None, :].expand(height, width)
    return torch.stack([x * x, x * y, y * y, x, y, torch.ones_like(x)]).reshape(6, -1)


def _terms(c6, mono):
    """exp of the exponents over the pixels, a few beamlets at a time: (rows, [rows, H W])."""
    step = max(1, (1 << 25) // mono.shape[1])
    for at in range(0, c6.shape[0], step):
        c = c6[at:at + step].detach()
        yield slice(at, at + step), torch.polar(torch.exp(c.real @ mono), c.imag @ mono)


def _field_of(c6, amp, mono):
    return sum((amp[rows].detach()[:, None] * e).sum(0) for rows, e in _terms(c6, mono))


def _adjoint(c6, amp, mono, w, leaves):
    """Gradients of Re sum_p w_p u_p with respect to `leaves`, through amp and c6."""
    m = mono.to(torch.complex128) * w
    G = torch.cat([e @ m.T for _, e in _terms(c6, mono)])  # sum w E {monomials}
    real = (amp.detach()[:, None] * G * c6).real.sum() + (amp * G[:, 5]).real.sum()
    return torch.autograd.grad(real, leaves)


def _exact_aperture(case, seed):
    """Untilted round beamlets in free space: the field is a product of an x and a y factor."""
    q, _ = _beamlet_arrays(case, seed)
    b = BEAM[True]
    mono = _monomials(case["height"], case["width"], b["pix"]).reshape(6, case["height"], case["width"])
    g = 1j * b["lam"] / (math.pi * 5e-8 ** 2)
    h = 1j * math.pi / b["lam"] * g / (1 + b["L"] * g)
    ex = torch.exp(h * (mono[3, 0] - q["x"][:, None]) ** 2)
    ey = torch.exp(h * (mono[4, :, 0] - q["y"][:, None]) ** 2) * (q["amplitude"] / (1 + b["L"] * g))[:, None]
    return {"field": ey.T.contiguous() @ ex}


def _exact_beamlets(case, seed):
    if case["round"]:
        return _exact_aperture(case, seed)
    q, T = _beamlet_arrays(case, seed)
    leaves = {k: v.requires_grad_() for k, v in dict(q, abcd=T).items() if k != "radii_of_curv"}
    mono = _monomials(case["height"], case["width"], BEAM[False]["pix"])
    c6 = _exponents(q, torch.full_like(q["theta"], BEAM[False]["lam"]), T)
    out = {"field": _field_of(c6, q["amplitude"], mono).reshape(case["height"], case["width"])}
    if case["grad"]:
        w = _cotangent(case, seed).to(torch.complex128).conj().reshape(-1)
        out.update(zip(leaves, _adjoint(c6, q["amplitude"], mono, w, list(leaves.values()))))
    return out


def _exact_gaussfit(case, seed):
    p, target = _fit_arrays(case, seed)
    counts, sides = _fit_tables(case)
    if sum(n * s * s for n, s in zip(counts, sides)) > 2e10:
        return None
    losses, grads, at, g0 = [], [], 0, 0
    for n, s in zip(counts, sides):
        rows = p[g0:g0 + n].clone().requires_grad_()
        q = dict(x=rows[:, 0], y=rows[:, 1], dx=rows[:, 2], dy=rows[:, 3], waist_xy=rows[:, 7:9],
                 radii_of_curv=rows[:, 9:11], theta=rows[:, 12])
        phase = (2j * math.pi / rows[:, 11] * rows[:, 4])[:, None]  # k times the pathlength
        c6 = torch.cat([(c := _exponents(q, rows[:, 11]))[:, :5], c[:, 5:] + phase], -1)
        amp = torch.complex(rows[:, 5], rows[:, 6])
        mono = _monomials(s, s, FIT_PIXEL)
        u = _field_of(c6, amp, mono)
        r = u.abs() ** 2 - target[at:at + s * s].double()
        losses.append((r * r).mean())
        grads.append(_adjoint(c6, amp, mono, (4.0 / (s * s)) * r * u.conj(), [rows])[0])
        at, g0 = at + s * s, g0 + n
    return {"loss": torch.stack(losses), "grad": torch.cat(grads)}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("rays", "source"):
        col, z_det = _column(case["elements"], seed)
        if kind == "rays":
            out = _exact_column(*(v.double() for v in _ray_arrays(case, seed)), col, z_det)
            return dict(out, image=None) if case["image"] else out
        semi_conv, (ox, oy) = _source_of(seed)
        dx, dy = _exact_rings(case["num"], semi_conv)
        out = _exact_column(torch.full_like(dx, ox), torch.full_like(dx, oy), dx, dy, col, z_det)
        return dict(out, image=None, dx0=dx, dy0=dy)
    return {"fit": _exact_fit, "forward": _exact_forward, "backproj": _exact_backproject,
            "beamlets": _exact_beamlets, "gaussfit": _exact_gaussfit}[kind](case, seed)
