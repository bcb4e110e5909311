"""The dataset kernel's split of the detector: one position and thousands, bands
of one row and of a whole detector, rows of every alignment, the most slopes.

Reference: the sum (FP64) of the same call's values at the pixels of its
coordinates, within one f32 rounding of each term (a pixel's terms are added in
any order); buffers that held other numbers are overwritten."""
import pytest
import torch

from temgymcore_amd import stem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scan,det,n_side", [
    ((1, 1), (64, 64), 1024), ((1, 1), (3, 6143), 16), ((2, 3), (17, 6144), 30), ((1, 2), (4097, 3), 8),
    ((5, 5), (1, 1), 8), ((25, 25), (64, 100), 16), ((31, 33), (70, 201), 12), ((16, 20), (96, 64), 64),
    ((26, 50), (256, 256), 8), ((64, 64), (37, 35), 8), ((128, 96), (33, 31), 4),
])
def test_bands(device, scan, det, n_side):
    model, sample = stem.reference_workload(n_cam=1, scan_shape=scan, det_shape=det, n_side=n_side,
                                            det_pixel=6e-4 / min(det))
    S, (H, W) = model.n_scan, det
    sample = torch.from_numpy(sample).to(device)
    params = stem.params_tensor(model, device)
    res = stem.stem_forward(model, params, sample, coords=True, values=True)
    out = {"image4d": torch.full((S, H, W), float("nan"), device=device)}
    stem.stem_forward(model, params, sample, coords=False, values=False, image4d=True, out=out)
    got = out["image4d"].double().reshape(-1)
    x, y = res["coords"][0].double().unbind(-1)
    m = list(model.geometry().det_m)
    py = torch.round((m[0] * y + m[1] * x) + m[2]).long()
    px = torch.round((m[3] * y + m[4] * x) + m[5]).long()
    ok = (py >= 0) & (py < H) & (px >= 0) & (px < W)
    at = ((torch.arange(S, device=device)[:, None] * H + py) * W + px)[ok]
    v = res["values"].double()[ok]
    zero = torch.zeros(S * H * W, dtype=torch.float64, device=device)
    ref, size, n = (zero.index_add(0, at, t) for t in (v, v.abs(), torch.ones_like(v)))
    assert bool(ok.any())
    assert bool(((got - ref).abs() <= 2.0**-24 * n * size).all())
