"""The loss kernel's pixels and slices: the field and the loss of batches whose
images end around its pixel groups and chunks, against the same batch summed in
one slice (tuned).

Both sum the same f32 terms in another order, n of them a pixel: each sum is
within (n - 1) 2^-24 of the sum of the terms' magnitudes, and the stored field
within 2^-24 of its value.  The loss is the mean of the squared residuals of the
kernel's own field to the rounding of that field: |dr| <= 2^-22 |u|^2."""
import numpy as np
import pytest
import torch

from temgymcore_amd import autotune
from temgymcore_amd.components import Detector
from temgymcore_amd.gauss_fit import GaussianFitBatch

pytestmark = pytest.mark.gpu

PIX, LAM = 1e-7, 2e-12


@pytest.mark.parametrize("counts,shapes", [
    ((3,), ((1, 1),)), ((1, 257, 33), ((64, 64), (65, 63), (17, 241))), ((600,), ((130, 129),)),
    ((383, 0, 1100, 64), ((64, 48), (16, 16), (33, 31), (128, 70))), ((2000, 3), ((70, 66), (1, 300))),
])
def test_slices_and_pixel_groups(device, counts, shapes):
    rng = np.random.default_rng(sum(counts))
    n = sum(counts)
    p = np.zeros((n, 16))
    p[:, 0:2] = rng.uniform(-30, 30, (n, 2)) * PIX
    p[:, 2:4] = rng.uniform(-2e-6, 2e-6, (n, 2))
    p[:, 5:7] = rng.uniform(-1, 1, (n, 2))
    p[:, 7:9] = rng.uniform(4, 20, (n, 2)) * PIX
    p[:, 9:11], p[:, 11], p[:, 12] = np.inf, LAM, rng.uniform(-1, 1, n)
    grids = [Detector(z=0.0, pixel_size=(PIX, PIX), shape=s) for s in shapes]
    npix = [h * w for h, w in shapes]
    target = rng.uniform(0, 2, sum(npix)).astype(np.float32)
    P, T = torch.from_numpy(p).to(device), torch.from_numpy(target).to(device)

    def run():
        batch = GaussianFitBatch(grids, counts)
        return (batch.field(P).cpu().numpy().astype(np.complex128), batch.loss_and_grad(P, T)[0].cpu().numpy(),
                batch.plan.off_weight - batch.plan.off_partial)

    u, loss, partials = run()
    slices = [min(8, max(1, -(-c // 256))) for c in counts]
    assert partials == -(-8 * sum(s * k for s, k in zip(slices, npix)) // 256) * 256
    autotune.set_choice(autotune.FIT_SLICE, (len(counts), n, sum(npix)), 4096)
    try:
        one, _, partials = run()
        assert partials == -(-8 * sum(npix) // 256) * 256
    finally:
        autotune.clear()
    g0 = p0 = 0
    for i, (c, k) in enumerate(zip(counts, npix)):
        r = np.asarray(grids[i].coords).reshape(-1, 2)
        q = p[g0:g0 + c]
        size = np.zeros(k)
        for row in q:
            d = r - row[0:2]
            a, b = np.cos(row[12]) * d[:, 0] + np.sin(row[12]) * d[:, 1], np.cos(row[12]) * d[:, 1] - np.sin(row[12]) * d[:, 0]
            size += np.hypot(row[5], row[6]) * np.exp(-(a / row[7]) ** 2 - (b / row[8]) ** 2)
        here = u[p0:p0 + k]
        assert (np.abs(here - one[p0:p0 + k]) <= 2.0**-23 * 1.5 * max(c, 2) * (1.01 * size + 1e-30)).all()
        t = target[p0:p0 + k].astype(np.float64)
        res, dr = np.abs(np.abs(here) ** 2 - t), 2.0**-22 * np.abs(here) ** 2
        want = np.mean(res**2)
        assert abs(loss[i] - want) <= np.mean(2 * res * dr + dr**2) + 1e-12 * want
        g0, p0 = g0 + c, p0 + k
