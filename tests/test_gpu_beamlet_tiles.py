"""The separable tile sum on the f16 matrix cores: tile edges, chunk and list
remainders, amplitudes that grow over many decades (the sums are rescaled),
far tails, one slice of beamlets longer than a list.

Reference: the complex128 oracle.  Bound per pixel, with A(p) the sum of the
beamlets' magnitudes there: each of a term's two factors carries the phasor
recurrence's 1.4e-5 rad and 6e-6 in magnitude (worst, from the CPU emulation)
and 1e-5 from an f32 envelope exponent down to exp(-40), so 6e-5 A(p); and
what the halves cannot hold, below 2^-38 of the largest term a beamlet."""
import numpy as np
import pytest
import torch

from oracle import beamlet_oracle as BO
from temgymcore_amd import autotune
from temgymcore_amd.components import Detector
from temgymcore_amd.gaussian import GaussianRay, make_gaussian_image
from temgymcore_amd.ray import Ray
from temgymcore_amd.transfer import ray_matrix

pytestmark = pytest.mark.gpu

PIX = 3e-8


def _case(n, shape, decades, waist):
    rng = np.random.default_rng(100 * n + shape[1])
    H, W = shape
    d = dict(x=rng.uniform(-0.55, 0.55, n) * W * PIX, y=rng.uniform(-0.55, 0.55, n) * H * PIX)
    d["dx"], d["dy"] = rng.uniform(-1e-5, 1e-5, (2, n))
    d["pathlength"] = rng.uniform(0, 1e-9, n)
    d["amplitude"] = 10.0 ** (decades * (np.arange(n) / max(n - 1, 1) - 0.5)) * np.exp(1j * rng.uniform(-3, 3, n))
    d["waist_xy"] = waist * rng.uniform(0.7, 1.3, (n, 2))
    d["radii"] = rng.uniform(0.5, 2.0, (n, 2))
    d["radii"][::3] = np.inf
    d["wavelength"], d["theta"] = np.full(n, 2e-12), np.zeros(n)
    return d


@pytest.mark.parametrize("n,shape,decades,waist", [
    (1, (1, 1), 0, 5e-8), (15, (63, 129), 0, 5e-8), (16, (127, 128), 0, 2e-7), (17, (128, 64), 4, 5e-8),
    (33, (130, 257), 0, 1e-6), (31, (129, 127), 12, 1e-6), (47, (65, 200), 30, 2e-7), (1023, (40, 70), 0, 1e-7),
    (1025, (33, 130), 12, 1e-7), (2065, (20, 129), 30, 5e-8),
])
def test_tile_sum_edges_vs_oracle(device, n, shape, decades, waist):
    d = _case(n, shape, decades, waist)
    det = Detector(z=1e-3, pixel_size=(PIX, PIX), shape=shape)
    t = {k: torch.from_numpy(np.ascontiguousarray(v)) for k, v in d.items()}
    ray = GaussianRay(x=t["x"], y=t["y"], dx=t["dx"], dy=t["dy"], z=torch.zeros(n, dtype=torch.float64),
                      pathlength=t["pathlength"], _one=torch.ones(n, dtype=torch.float64), amplitude=t["amplitude"],
                      waist_xy=t["waist_xy"], radii_of_curv=t["radii"], wavelength=t["wavelength"], theta=t["theta"])
    autotune.set_choice(autotune.BEAMLET_SPLITS, (n, *shape), 1)
    try:
        got = make_gaussian_image(ray, [det]).cpu().numpy().astype(np.complex128).ravel()
    finally:
        autotune.clear()
    abcd = ray_matrix([det], Ray(0.0, 0.0, 0.0, 0.0, 0.0, 0.0))
    r2 = BO.grid_coords(det.pixel_size, det.shape)
    ref, total = np.zeros(r2.shape[0], dtype=np.complex128), np.zeros(r2.shape[0])
    for i in range(n):
        u = BO.make_image(abcd=abcd, r2=r2, **{k: v[i:i + 1] for k, v in d.items()})
        ref += u
        total += np.abs(u)
    assert total.max() > 0
    assert (np.abs(got - ref) <= 6e-5 * total + n * 2.0**-38 * total.max()).all()
