"""Back-projection where rows and columns are handled on their own (grids
without rotation) against the general form, which a cross term too small to
move any sum selects: the same rays, pixels and f32 weights, FP64 sums in
another order.

Bound per pixel: 2^-40 of the sum of the terms' magnitudes (up to 2^12 terms a
pixel in FP64, 2^-52 each); infinities and NaN in the same places."""
import ctypes

import numpy as np
import pytest
import torch

from temgymcore_amd import _lib, stem

pytestmark = pytest.mark.gpu


def _run(g, params, data, cam, device, weights):
    image = torch.zeros(g.img_h, g.img_w, dtype=torch.float64, device=device)
    weight = torch.zeros_like(image) if weights else None
    st = _lib.load().tg_stem_backproject(ctypes.byref(g), params.data_ptr(), data.data_ptr(), cam, image.data_ptr(),
                                         None if weight is None else weight.data_ptr(), _lib.stream_ptr(device))
    _lib.check(st, "tg_stem_backproject")
    return image, weight


@pytest.mark.parametrize("weights", [True, False])
@pytest.mark.parametrize("scan_shape,n_side,change", [
    ((1, 1), 2, {}), ((3, 4), 6, {}), ((5, 5), 30, {}), ((4, 4), 64, {}), ((3, 3), 66, {}), ((2, 3), 70, dict(pixel=1e-5)),
    ((4, 4), 32, dict(defocus=2e-6)),   # footprints of 100 pixels: windows missed, rays one by one
    ((4, 4), 32, dict(shift=230.0)),    # half of the rays beside the sample image
    ((4, 4), 32, dict(pixel=1e-6)),     # most rays beside the detector
    ((3, 3), 16, dict(offset=float("nan"))), ((3, 3), 16, dict(offset=float("inf"))),
    ((4, 4), 20, dict(odd=True)),
])
def test_axes_form_equals_the_general_form(device, scan_shape, n_side, change, weights):
    model, _ = stem.reference_workload(n_cam=2, scan_shape=scan_shape, n_side=n_side,
                                       **({"defocus": change["defocus"]} if "defocus" in change else {}),
                                       **({"det_pixel": change["pixel"]} if "pixel" in change else {}))
    params = stem.params_tensor(model, device)
    gen = torch.Generator(device=device).manual_seed(n_side)
    data = torch.rand((model.n_scan,) + tuple(model.det_shape), generator=gen, device=device) - 0.3
    if change.get("odd"):
        data.view(-1)[::97] = float("inf")
        data.view(-1)[::89] = float("nan")
    got = []
    for cross in (0.0, 1e-290):
        g = model.geometry()
        assert g.img_m[1] == 0 and g.img_m[3] == 0 and g.det_m[1] == 0 and g.det_m[3] == 0
        g.img_m[1] = cross
        g.img_m[2] += change.get("shift", 0.0)
        g.offsets[1] += change.get("offset", 0.0)
        got.append([_run(g, params, d, cam, device, weights) for cam in (0, 1) for d in (data, data.abs())])
    for (image, weight), (ref, ref_w), size in zip(got[0], got[1], (1, 1, 3, 3)):
        scale = got[1][size][0]  # the same sums of magnitudes
        ok = torch.isfinite(scale)
        assert torch.equal(ok, torch.isfinite(got[0][size][0]))
        assert ((image - ref).abs()[ok] <= 2.0**-40 * scale[ok]).all()
        if weights:
            assert ((weight - ref_w).abs() <= 2.0**-40 * ref_w).all()
    if not change:
        assert all(float(r.abs().sum()) > 0 for r, _ in got[1])
