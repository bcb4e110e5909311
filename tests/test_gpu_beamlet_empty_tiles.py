"""The recurrence tile sum where beamlets leave tiles empty: a whole list of 256
beside a tile, and a short last list that no tile meets.

Reference: the complex128 oracle, a beamlet's terms outside its ellipse left
out.  Bound per pixel: as for the runs cut by an ellipse (3e-5 of the sum of the
terms' magnitudes for n <= 40), with n 2^-24 more for the f32 sum of n terms; a
pixel within 1e-4 of an ellipse's edge may fall on either side."""
import numpy as np
import pytest
import torch

from oracle import beamlet_oracle as BO
from temgymcore_amd import autotune
from temgymcore_amd.components import Detector
from temgymcore_amd.gauss_fit import GaussianFitBatch
from temgymcore_amd.gaussian import MODE_INPUT, beamlet_field

pytestmark = pytest.mark.gpu

PIX, SHAPE = 1e-7, (150, 270)


def _rows(n, beside, seed):
    """n rotated beamlets near the image's first pixel, the last `beside` of them off the image."""
    rng = np.random.default_rng(seed)
    det = Detector(z=0.0, pixel_size=(PIX, PIX), shape=SHAPE)
    corner = np.asarray(det.coords).reshape(-1, 2)[0]
    p = np.zeros((n, 16))
    p[:, 0:2] = corner + np.sign(-corner) * rng.uniform(2, 30, (n, 2)) * PIX
    p[n - beside:, 0:2] = -20 * corner
    p[:, 2:4] = rng.uniform(-1e-6, 1e-6, (n, 2))
    p[:, 5:7] = rng.uniform(-1, 1, (n, 2))
    p[:, 7:9] = rng.uniform(1.5, 4, (n, 2)) * PIX
    p[:, 9:11], p[:, 11], p[:, 12] = np.inf, 2e-12, rng.uniform(0.2, 1.3, n)
    return p, det


def _reference(p, det, level):
    r = np.asarray(det.coords).reshape(-1, 2)
    ref, size, loose = np.zeros(len(r), complex), np.zeros(len(r)), np.zeros(len(r))
    for q in p:
        d, c, s = r - q[0:2], np.cos(q[12]), np.sin(q[12])
        drop = ((c * d[:, 0] + s * d[:, 1]) / q[7]) ** 2 + ((c * d[:, 1] - s * d[:, 0]) / q[8]) ** 2
        inside = drop <= level
        if not inside.any():
            continue
        a = [q[k:k + 1] for k in (0, 1, 2, 3, 4)]
        u = BO.input_image(*a, q[5:6] + 1j * q[6:7], q[None, 7:9], q[None, 9:11], q[11:12], q[12:13], r)
        ref += np.where(inside, u, 0)
        size += np.where(inside, np.abs(u), 0)
        loose += np.where(np.abs(drop - level) <= 1e-4 * level, np.abs(u), 0)
    assert size.max() > 0 and (size == 0).mean() > 0.5  # tiles with nothing in them
    return ref, (3e-5 + len(p) * 2.0**-24) * size + loose


@pytest.mark.parametrize("n,beside", [(3, 0), (259, 3), (512, 256), (300, 300 - 256)])
@pytest.mark.parametrize("tile", ["64x64", "128x32", "32x128", "64x32"])
def test_lists_without_a_beamlet(device, n, beside, tile):
    p, det = _rows(n, beside, n)
    shapes = {"64x64": autotune.TILE_64x64_RUN16, "128x32": autotune.TILE_128x32_RUN16,
              "32x128": autotune.TILE_32x128_RUN16, "64x32": autotune.TILE_64x32_RUN8}
    autotune.clear()
    autotune.set_choice(autotune.TILE_SHAPE, (n, *SHAPE), shapes[tile])
    autotune.set_choice(autotune.BEAMLET_SPLITS, (n, *SHAPE), 1)
    try:
        got = beamlet_field(torch.from_numpy(p).to(device), det, MODE_INPUT, cutoff=3.0).cpu().numpy().ravel()
    finally:
        autotune.clear()
    ref, bound = _reference(p, det, 9.0)
    assert (np.abs(got - ref) <= bound).all()


def test_fit_field_with_empty_tiles(device):
    (p, det), (q, _) = _rows(259, 3, 1), _rows(3, 3, 2)
    both = torch.from_numpy(np.concatenate([p, q])).to(device)
    got = GaussianFitBatch([det, det], (259, 3)).field(both).cpu().numpy().ravel()
    ref, bound = _reference(p, det, 80.0)
    k = len(ref)
    assert (np.abs(got[:k] - ref) <= bound).all()
    assert (got[k:] == 0).all()
