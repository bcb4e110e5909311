"""The separable tile sum where what is visible is far below a beamlet's peak or
its neighbours': beamlets beside the image (before it and past it), narrow ones
between pixels, weak ones apart from strong ones, in one list or in two.

Reference: the complex128 oracle, pixel by pixel.  Bound, with A(p) the sum of
the magnitudes there of the terms that are to be kept (down to exp(-80), or the
cut): an f32 envelope exponent of up to 115 bits behind nine roundings of 2^-24
(4.3e-5), two factors' phasors at 1.4e-5 rad and 6e-6 in magnitude (4e-5), and
what the products and sums of a few terms add (1e-6); or, with a cut, an
exponent of up to 25 bits (1e-5), the phasors, and 2^-14 for what the f16 halves
round at the cut: 1.2e-4 A(p).  A term below the cut may be there or not, or each
of its factors rounded up to twice its size: three times its magnitude.  And the
smallest normal f32, 2^-126, below which results are flushed."""
import numpy as np
import pytest
import torch

from oracle import beamlet_oracle as BO
from temgymcore_amd import autotune
from temgymcore_amd.components import Detector
from temgymcore_amd.gaussian import MODE_INPUT, beamlet_field

pytestmark = pytest.mark.gpu

PIX = 1e-7


def _check(device, shape, xy, waist, amp, cutoff=None, curved=True):
    """xy: centres in pixel indices (x, y); waist in pixels."""
    n = len(xy)
    det = Detector(z=0.0, pixel_size=(PIX, PIX), shape=shape)
    r = np.asarray(det.coords).reshape(-1, 2)
    grid = r.reshape(*shape, 2)
    step = np.stack([grid[0, 1] - grid[0, 0], grid[1, 0] - grid[0, 0]])
    p = np.zeros((n, 16))
    p[:, 0:2] = grid[0, 0] + np.asarray(xy, float) @ step
    rng = np.random.default_rng(n)
    p[:, 2:4] = rng.uniform(-1e-6, 1e-6, (n, 2)) if curved else 0.0
    phase = np.exp(1j * rng.uniform(-3, 3, n))
    p[:, 5], p[:, 6] = (amp * phase).real, (amp * phase).imag
    p[:, 7:9] = np.asarray(waist, float).reshape(-1, 1) * PIX
    p[:, 9:11] = rng.uniform(0.2, 2.0, (n, 1)) if curved else np.inf
    p[:, 11] = 2e-12
    autotune.clear()
    autotune.set_choice(autotune.BEAMLET_SPLITS, (n, *shape), 1)
    try:
        got = beamlet_field(torch.from_numpy(p).to(device), det, MODE_INPUT, cutoff=cutoff).cpu().numpy().ravel()
    finally:
        autotune.clear()
    level = 80.0 if cutoff is None else cutoff**2
    ref, size, loose = np.zeros(len(r), complex), np.zeros(len(r)), np.zeros(len(r))
    for q, a in zip(p, amp * phase):
        u = BO.input_image(*[q[k:k + 1] for k in (0, 1, 2, 3, 4)], np.array([a]), q[None, 7:9], q[None, 9:11],
                           q[11:12], q[12:13], r)
        drop = (((r - q[0:2]) / q[7:9]) ** 2).sum(1)
        kept = drop <= level * (1 - 1e-4)
        ref += u
        size += np.where(kept, np.abs(u), 0)
        loose += np.where(kept, 0, np.abs(u))
    assert size.max() > 0
    bad = np.abs(got - ref) - (1.2e-4 * size + 3 * loose + 2.0**-126)
    assert (bad <= 0).all(), (bad.max(), np.abs(got - ref)[bad.argmax()], size[bad.argmax()])


# the image's first and last pixel are 37 or 42 pixels from the centre on both sides
@pytest.mark.parametrize("x", [-37, 100, -42, 105])
@pytest.mark.parametrize("axis", [0, 1])
def test_lone_beamlet_beside_the_image(device, x, axis):
    centre = (x, 30.5) if axis == 0 else (30.5, x)
    _check(device, (64, 64), [centre], 8.0, np.ones(1), curved=False)


@pytest.mark.parametrize("waist", [0.12, 0.1, 0.3])
def test_narrow_beamlet_between_pixels(device, waist):
    _check(device, (64, 64), [(31.5, 31.5)], waist, np.ones(1))


@pytest.mark.parametrize("cutoff", [None, 4.0, 6.0])
@pytest.mark.parametrize("shape", [(128, 128), (100, 190)])
def test_tails_of_one_beamlet(device, shape, cutoff):
    _check(device, shape, [(50.3, 61.2)], 8.0, np.ones(1), cutoff)


@pytest.mark.parametrize("weak", [1e-3, 1e-9, 1e-12, 1e-20])
@pytest.mark.parametrize("cutoff", [None, 4.0])
def test_weak_beamlet_apart_from_a_strong_one(device, weak, cutoff):
    _check(device, (120, 128), [(20.2, 20.7), (100.4, 99.1)], [3.0, 3.0], np.array([1.0, weak]), cutoff)


def test_strong_beamlet_past_the_edge(device):
    xy = [(95.0, 31.0), (20.0, 30.0), (40.0, 12.0)]
    _check(device, (64, 64), xy, [8.0, 6.0, 5.0], np.array([1e6, 1.0, 1e-4]))


@pytest.mark.parametrize("order", [1, -1])
def test_lists_of_unlike_strength(device, order):
    """1,024 beamlets of one list weak and apart, the next list's strong."""
    rng = np.random.default_rng(3)
    xy = np.concatenate([rng.uniform(2, 20, (1024, 2)), rng.uniform(100, 125, (9, 2))])
    amp = np.concatenate([np.full(1024, 1e-10), np.full(9, 1.0)])
    _check(device, (128, 130), xy[::order], np.full(len(xy), 2.5), amp[::order])


def test_cut_set_of_like_strength(device):
    """What the f16 halves hold: a cut of 4 and amplitudes within a few bits."""
    rng = np.random.default_rng(4)
    xy = rng.uniform(-10, 210, (300, 2))
    _check(device, (150, 200), xy, rng.uniform(6, 9, 300), np.ones(300), 4.0)


def test_wide_beamlets_uncut(device):
    rng = np.random.default_rng(5)
    _check(device, (130, 140), rng.uniform(0, 140, (40, 2)), rng.uniform(150, 300, 40), rng.uniform(0.5, 2, 40))
