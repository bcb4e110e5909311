"""The run enumeration of the moment kernels: every pixel inside the cutoff
ellipse counts once, on images narrower than a run, with row and run
remainders, whole and cut runs, more rows than a wavefront has lanes, ellipses
inside, across and around the image.

The gradient of the amplitude is the sum of conj(cotangent) E over the pixels
of the ellipse, |drop| <= nsigma^2 of the envelope exponent: compared with its
complex128 sum.  Bound: 16 f32 recurrence steps behind a term (136 roundings of
2^-23: 1.6e-5), its f32 start and the run's sums (1e-5): 3e-5 of the sum of the
terms' magnitudes.  No pixel lies within 1e-4 of the ellipse's edge (asserted),
and one pixel more or less would be seen (asserted)."""
import numpy as np
import pytest
import torch

from temgymcore_amd.components import Detector
from temgymcore_amd.gaussian import MODE_INPUT, beamlet_backward

pytestmark = pytest.mark.gpu

LAM = 2e-12


@pytest.mark.parametrize("shape,centre,waist,theta,nsigma", [
    ((1, 1), (0.0, 0.0), (3.0, 3.0), 0.0, 1.0), ((3, 15), (0.2, 0.1), (40.0, 40.0), 0.3, 1.2),
    ((64, 16), (3.3, -4.1), (50.0, 90.0), 0.0, 1.5), ((65, 17), (1.7, 2.2), (9.3, 4.4), 0.7, 1.1),
    ((130, 31), (-4.1, 30.3), (12.2, 31.1), -0.4, 1.3), ((129, 33), (0.3, 0.4), (500.0, 400.0), 0.2, 1.0),
    ((70, 100), (11.2, -8.6), (25.7, 19.3), 1.1, 1.4), ((20, 300), (40.4, 3.3), (75.6, 12.7), 0.1, 1.2),
    ((200, 40), (26.1, 3.2), (13.2, 50.4), 0.0, 1.0), ((100, 120), (300.0, 0.0), (20.0, 20.0), 0.0, 1.0),
])
@pytest.mark.parametrize("copies", [1, 8200])  # four wavefronts a beamlet; one
def test_every_pixel_of_the_ellipse_counts_once(device, shape, centre, waist, theta, nsigma, copies):
    rng = np.random.default_rng(shape[0] * 1000 + shape[1])
    pix = 1e-7
    p = np.zeros((1, 16))
    p[0, 0:2] = np.array(centre) * pix
    p[0, 5], p[0, 7:9], p[0, 9:11], p[0, 11], p[0, 12] = 1.0, np.array(waist) * pix, np.inf, LAM, theta
    det = Detector(z=0.0, pixel_size=(pix, pix), shape=shape)
    r = np.asarray(det.coords).reshape(-1, 2) - p[0, 0:2]
    u, v = np.cos(theta) * r[:, 0] + np.sin(theta) * r[:, 1], -np.sin(theta) * r[:, 0] + np.cos(theta) * r[:, 1]
    drop = (u / p[0, 7]) ** 2 + (v / p[0, 8]) ** 2
    assert (np.abs(drop - nsigma**2) > 1e-4 * nsigma**2).all()
    inside = drop <= nsigma**2
    g = ((1 + rng.uniform(0, 1, shape)) * np.exp(1j * rng.uniform(-0.5, 0.5, shape))).astype(np.complex64)
    grad, _ = beamlet_backward(torch.from_numpy(p).to(device).repeat(copies, 1), det, MODE_INPUT, torch.from_numpy(g).to(device),
                               cutoff=nsigma)
    terms = np.where(inside, np.conj(g.astype(np.complex128).ravel()) * np.exp(-drop), 0.0)
    total, size = terms.sum(), np.abs(terms).sum()
    if inside.any():
        assert np.abs(terms[inside]).min() > 2 * 3e-5 * size
    assert torch.equal(grad, grad[:1].expand_as(grad))
    got = grad.cpu().numpy()[0]
    assert abs(got[5] - total.real) <= 3e-5 * size and abs(-got[6] - total.imag) <= 3e-5 * size
