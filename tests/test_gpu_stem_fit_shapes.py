"""The descan fit where its kernels change: pairs a lane (2, 4, 8, several
tiles), cameras (one to the most there are), positions (few; more than a lane
each in the summing block).  Both launch variants and the separate terms give
the same bits; the loss is the sum of the squared residuals of the forward's
own coordinates.

Loss bound: a residual is exact to two f32 roundings of itself (compensated
form) where the reference takes f32 coordinates, off by one rounding of the
1e-4-metre coordinate each, on residuals that are 1% of it: 2 * 2^-24 / 0.01 of
each square, 1.2e-5, and 2^-20 for the f32 sums of up to 64 pairs."""
import numpy as np
import pytest
import torch

from temgymcore_amd import autotune, stem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scan_shape,n_side,n_cam", [
    ((1, 1), 2, 1), ((3, 5), 22, 16), ((5, 5), 32, 10), ((7, 4), 34, 3), ((4, 4), 44, 4), ((4, 4), 46, 12),
    ((3, 3), 64, 16), ((3, 3), 66, 2), ((32, 32), 16, 1), ((32, 33), 30, 11), ((33, 33), 44, 5), ((25, 50), 46, 2),
])
def test_fit_variants_and_terms_agree(device, scan_shape, n_side, n_cam):
    model, _ = stem.reference_workload(n_cam=n_cam, scan_shape=scan_shape, n_side=n_side)
    params = stem.params_tensor(model, device)
    coords = stem.stem_forward(model)["coords"]
    g = torch.Generator(device=device).manual_seed(n_side)
    targets = coords * (1 + 0.02 * (torch.rand(coords.shape, generator=g, device=device) - 0.5))
    S, key = model.n_scan, (model.n_scan, n_side * n_side, n_cam)
    got = []
    for variant in (autotune.STEM_FIT_SCAN, autotune.STEM_FIT_CAMERA):
        autotune.clear()
        autotune.set_choice(autotune.STEM_FIT, key, variant)
        try:
            ws = stem.STEMFitWorkspace(model, device)
            out = ws.run(params, targets).clone()
            full = ws.partials.clone()
            terms = ws.terms(params, targets).clone()
        finally:
            autotune.clear()
        assert torch.equal(terms, full)
        got += [out, full]
    assert torch.equal(got[0], got[2]) and torch.equal(got[1], got[3])
    loss = float(((coords.double() - targets.double()) ** 2).sum())
    assert abs(float(got[0][-1]) - loss) <= 2e-5 * loss
