"""GPU parity of the 4D-STEM kernels against the float64 oracle.

Tolerances:
  detector coordinates: |d| <= 1e-6 * max(|ref|, 1e-6 m)   (f32 output)
  sample values:        |d| <= 2e-5 (values in [-pi, pi], f32 bilinear weights)
  fit gradient:         |d| <= 2e-4 * max|g| per block of parameters, vs central
                        FD of the float64 loss on the same f32 targets; on
                        larger detectors plus 2^-24 * sum|d(r^2)/dp| (one f32
                        rounding of every term, oracle.stem_oracle.grad_abs_scale)
  loss:                 relative 1e-5
"""
import dataclasses

import numpy as np
import pytest
import torch

from oracle import ray_oracle as R
from oracle import stem_oracle as SO
from temgymcore_amd import stem
from temgymcore_amd.run import run_to_end

pytestmark = pytest.mark.gpu


def _geom(m):
    return dict(scan_shape=m.scan_shape, n_side=m.n_side, semi_conv=m.semi_conv, defocus=m.defocus,
                pivot=m.pivot, offsets=tuple(m.descan_offsets))


def _small(n_cam=3, seed=5, **kw):
    model, sample = stem.reference_workload(n_cam=n_cam, **kw)
    return model, sample


def _close_pos(got, ref, floor=1e-6):
    bound = 1e-6 * np.maximum(np.abs(ref), floor)
    err = np.abs(got.astype(np.float64) - ref)
    assert np.all(err <= bound), f"max err {err.max():.3e}, worst ratio {(err / bound).max():.3f}"


@pytest.mark.parametrize("shape", [(4, 6), (64, 64)])
def test_forward_coords_vs_oracle(device, shape):
    print(f"[stem forward scan={shape}]", flush=True)
    model, _ = stem.reference_workload(n_cam=8, scan_shape=shape)
    out = stem.stem_forward(model)["coords"].cpu().numpy()
    x, y = SO.forward(_geom(model), model.params())
    _close_pos(out[..., 0], x)
    _close_pos(out[..., 1], y)


def test_forward_full_size_single_camera(device):
    print("[stem forward full 16.7M rays]", flush=True)
    model, sample = stem.reference_workload(n_cam=1)
    res = stem.stem_forward(model, sample=torch.from_numpy(sample).to(device), coords=True, values=True)
    coords = res["coords"].cpu().numpy()
    x, y = SO.forward(_geom(model), model.params())
    _close_pos(coords[..., 0], x)
    _close_pos(coords[..., 1], y)
    xs, ys = SO.sample_plane(_geom(model), model.params())
    Tinv = R.metres_to_pixels_matrix((0.0, 0.0), (model.sample_pixel,) * 2, model.sample_shape)
    ref_v = SO.bilinear(sample.astype(np.float64), Tinv, xs, ys)
    np.testing.assert_allclose(res["values"].cpu().numpy(), ref_v, rtol=0, atol=2e-5)


def test_image4d_deposit(device):
    model, sample = stem.reference_workload(n_cam=1, scan_shape=(8, 8))
    res = stem.stem_forward(model, sample=torch.from_numpy(sample).to(device), coords=True, values=True,
                            image4d=True)
    img = res["image4d"].cpu().numpy().astype(np.float64)
    coords = res["coords"].cpu().numpy()[0]
    vals = res["values"].cpu().numpy().astype(np.float64)
    Tinv = R.metres_to_pixels_matrix((0.0, 0.0), (model.det_pixel,) * 2, model.det_shape)
    ref = np.zeros_like(img)
    for s in range(model.n_scan):
        py, px = R.metres_to_pixels(coords[s, :, 0], coords[s, :, 1], Tinv)
        ok = (py >= 0) & (py < model.det_shape[0]) & (px >= 0) & (px < model.det_shape[1])
        np.add.at(ref[s], (py[ok], px[ok]), vals[s][ok])
    np.testing.assert_allclose(img, ref, rtol=1e-6, atol=1e-5)
    # a second call into the same out dict starts the deposit from zero
    again = stem.stem_forward(model, sample=torch.from_numpy(sample).to(device), coords=True, values=True,
                              image4d=True, out=res)
    assert again["image4d"] is res["image4d"]
    # (float atomics: the summation order may differ between calls)
    np.testing.assert_allclose(again["image4d"].cpu().numpy().astype(np.float64), ref, rtol=1e-6, atol=1e-5)
    # reused buffers of the wrong shape, dtype or layout are refused before the launch
    sample_t = torch.from_numpy(sample).to(device)
    bad = {
        "coords": torch.empty((1, model.n_scan, model.n_rays - 1, 2), device=device),
        "values": torch.empty((model.n_scan, model.n_rays), dtype=torch.float64, device=device),
        "image4d": torch.empty((model.n_scan,) + tuple(model.det_shape)[::-1] + (2,), device=device)[..., 0],
    }
    for name, t in bad.items():
        with pytest.raises(ValueError, match=f"out\\['{name}'\\]"):
            stem.stem_forward(model, sample=sample_t, coords=True, values=True, image4d=True, out={name: t})


def test_image4d_deposit_full_scan_vs_oracle(device):
    """The 4D deposit of the full 64 x 64 scan (1 GiB of shadow images) on 8
    sampled scan positions against the float64 oracle's own coordinates and
    bilinear values (not the kernel's).  A ray whose oracle pixel coordinate
    lies within 1e-3 pixel of a rounding boundary may land in either
    neighbour in f32, so its |value| is slack on each candidate pixel; every
    other pixel matches to the per-ray value tolerance (2e-5, as the values
    test) times the rays it holds."""
    print("[stem image4d full scan]", flush=True)
    model, sample = stem.reference_workload(n_cam=1)
    img = stem.stem_forward(model, sample=torch.from_numpy(sample).to(device), coords=False,
                            image4d=True)["image4d"]
    pick = np.sort(np.random.default_rng(5).choice(model.n_scan, 8, replace=False))
    got = img[torch.from_numpy(pick).to(device)].cpu().numpy().astype(np.float64)
    del img
    geom = _geom(model)
    x, y = SO.forward(geom, model.params(), scan_idx=pick)
    x, y = x[0], y[0]
    xs, ys = SO.sample_plane(geom, model.params())
    Timg = R.metres_to_pixels_matrix((0.0, 0.0), (model.sample_pixel,) * 2, model.sample_shape)
    vals = SO.bilinear(sample.astype(np.float64), Timg, xs[pick], ys[pick])
    Tdet = R.metres_to_pixels_matrix((0.0, 0.0), (model.det_pixel,) * 2, model.det_shape)
    fy, fx = R.transform(y, x, Tdet)
    py, px = R.round_to_i32(fy), R.round_to_i32(fx)
    H, W = model.det_shape
    near_y = np.abs(fy - np.floor(fy) - 0.5) < 1e-3
    near_x = np.abs(fx - np.floor(fx) - 0.5) < 1e-3
    assert (near_y | near_x).mean() < 1e-2
    for k in range(len(pick)):
        ref = np.zeros((H, W))
        cnt = np.zeros((H, W))
        slack = np.zeros((H, W))
        ok = (py[k] >= 0) & (py[k] < H) & (px[k] >= 0) & (px[k] < W)
        firm = ok & ~(near_y[k] | near_x[k])
        np.add.at(ref, (py[k][firm], px[k][firm]), vals[k][firm])
        np.add.at(cnt, (py[k][firm], px[k][firm]), 1.0)
        for j in np.nonzero(near_y[k] | near_x[k])[0]:
            cy = [int(np.floor(fy[k, j])), int(np.floor(fy[k, j])) + 1] if near_y[k, j] else [int(py[k, j])]
            cx = [int(np.floor(fx[k, j])), int(np.floor(fx[k, j])) + 1] if near_x[k, j] else [int(px[k, j])]
            for a in cy:
                for b in cx:
                    if 0 <= a < H and 0 <= b < W:
                        slack[a, b] += abs(vals[k, j]) + 2e-5
        err = np.abs(got[k] - ref)
        bound = 2e-5 * cnt + slack + 1e-6
        assert np.all(err <= bound), f"scan position {pick[k]}: worst excess {np.max(err - bound):.3e}"
        assert cnt.sum() > 0.5 * model.n_rays


def test_generic_component_path_matches_oracle_and_kernel(device):
    """The same model through run_to_end (ray programs) is bit-exact vs the
    component oracle and within tolerance of the fused STEM kernel."""
    model, _ = stem.reference_workload(n_cam=1, scan_shape=(6, 5), n_side=16)
    out = run_to_end(model.rays(device), model.components(0, device))
    spx, spy = model.scan_positions()
    spx, spy = spx.reshape(-1, 1), spy.reshape(-1, 1)
    t = model.slopes()
    ty, tx = np.meshgrid(t, t, indexing="ij")
    r = R.make_ray(0.0, 0.0, tx.reshape(1, -1), ty.reshape(1, -1))
    r = R.scanner(r, spx, spy, model.pivot * spx, model.pivot * spy)
    r = R.propagate(r, model.defocus - r["z"])
    r = SO.descanner4(r, spx, spy, model.pivot * spx, model.pivot * spy, model.descan, model.descan_offsets)
    r = R.propagate(r, model.defocus + model.camera_lengths[0] - r["z"])
    np.testing.assert_array_equal(out.x.cpu().numpy(), r["x"])
    np.testing.assert_array_equal(out.y.cpu().numpy(), r["y"])
    k = stem.stem_forward(model)["coords"].cpu().numpy()[0]
    _close_pos(k[..., 0], out.x.cpu().numpy())
    _close_pos(k[..., 1], out.y.cpu().numpy())


def _targets(model, device):
    tgt_model = stem.perturbed(model)
    return stem.stem_forward(tgt_model)["coords"]


def test_fit_gradient_vs_fd_small(device):
    model, _ = stem.reference_workload(n_cam=3, scan_shape=(6, 7), n_side=16)
    targets = _targets(model, device)
    ws = stem.STEMFitWorkspace(model, device)
    out = ws.run(stem.params_tensor(model, device), targets).cpu().numpy()
    t = targets.cpu().numpy()
    ref_loss = SO.loss(_geom(model), model.params(), t)
    ref_g = SO.fd_grad(_geom(model), model.params(), t)
    assert out[-1] == pytest.approx(ref_loss, rel=1e-5)
    g = out[:-1]
    for blk in (slice(0, 16), slice(16, 17), slice(17, 18), slice(18, None)):
        scale = np.abs(ref_g[blk]).max()
        np.testing.assert_allclose(g[blk], ref_g[blk], rtol=0, atol=2e-4 * scale, err_msg=str(blk))


def test_fit_gradient_at_zero_scan_step(device):
    """At scan step 0 every scan position is 0, but d(position)/d(step), the
    rotated pixel offset, is not: the step gradient is finite and matches FD."""
    model, _ = stem.reference_workload(n_cam=3, scan_shape=(6, 7), n_side=16, scan_step=0.0)
    targets = _targets(dataclasses.replace(model, scan_step=1e-10), device)
    ws = stem.STEMFitWorkspace(model, device)
    out = ws.run(stem.params_tensor(model, device), targets).cpu().numpy()
    assert np.all(np.isfinite(out))
    t = targets.cpu().numpy()
    steps = SO.fd_steps(model.params())
    steps[16] = 1e-10
    ref_g = SO.fd_grad(_geom(model), model.params(), t, steps=steps)
    assert abs(ref_g[16]) > 0
    g = out[:-1]
    for blk in (slice(0, 16), slice(16, 17), slice(17, 18), slice(18, None)):
        scale = np.abs(ref_g[blk]).max()
        np.testing.assert_allclose(g[blk], ref_g[blk], rtol=0, atol=2e-4 * scale, err_msg=str(blk))


def test_fit_full_size_properties(device):
    """Full 64x64 scan x 4096 rays x 8 camera lengths: zero loss/gradient at the
    generating parameters, and per-scan-position gradient rows that match the
    FD oracle on a sample of scan positions."""
    print("[stem fit full size]", flush=True)
    model, _ = stem.reference_workload(n_cam=8)
    params = stem.params_tensor(model, device)
    ws = stem.STEMFitWorkspace(model, device)
    exact = stem.stem_forward(model)["coords"]
    out0 = ws.run(params, exact).cpu().numpy()
    # targets from the same f32 forward: residuals are the f32 rounding only
    assert abs(out0[-1]) < 1e-16 * model.n_scan * model.n_rays * model.n_cam
    targets = _targets(model, device)
    out = ws.run(params, targets).cpu().numpy()
    rows = ws.partials.cpu().numpy().T  # [S, np]
    np.testing.assert_allclose(rows.sum(axis=0), out, rtol=1e-12, atol=0)
    pick = np.random.default_rng(0).choice(model.n_scan, 6, replace=False)
    t = targets.cpu().numpy()[:, pick]
    ref_g = SO.fd_grad(_geom(model), model.params(), t, scan_idx=pick)
    ref_loss = SO.loss(_geom(model), model.params(), t, scan_idx=pick)
    sub = rows[pick].sum(axis=0)
    assert sub[-1] == pytest.approx(ref_loss, rel=1e-5)
    for blk in (slice(0, 16), slice(16, 17), slice(17, 18), slice(18, 26)):
        scale = np.abs(ref_g[blk]).max()
        np.testing.assert_allclose(sub[blk], ref_g[blk], rtol=0, atol=2e-4 * scale, err_msg=str(blk))


def test_autograd_function_and_graph_replay(device):
    model, _ = stem.reference_workload(n_cam=2, scan_shape=(16, 16))
    targets = _targets(model, device)
    params = stem.params_tensor(model, device).requires_grad_(True)
    ws = stem.STEMFitWorkspace(model, device)
    loss = stem.descan_fit_loss(model, params, targets, ws)
    (3.0 * loss).backward()
    eager = ws.run(params.detach(), targets).clone()
    torch.testing.assert_close(params.grad, 3.0 * eager[:-1], rtol=0, atol=0)
    # HIP graph capture of the fused fwd+bwd; replays match eager every time
    p2 = params.detach().clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ws.run(p2, targets)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ws.run(p2, targets)
    for k in range(3):
        ws.out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        torch.testing.assert_close(ws.out, eager, rtol=0, atol=0)
        _ = (targets[0, 0, 0, 0] * 1.0).item()  # eager work between replays


def test_fit_launch_variants_are_bitwise_equal(device):
    """The per-scan and per-(scan, camera) launch variants run the same
    arithmetic in the same order."""
    from temgymcore_amd import autotune

    model, _ = stem.reference_workload(n_cam=3, scan_shape=(12, 10), n_side=32)
    params = stem.params_tensor(model, device)
    targets = stem.stem_forward(stem.perturbed(model))["coords"]
    ws = stem.STEMFitWorkspace(model, device)
    key = (model.n_scan, model.n_rays, model.n_cam)
    outs = []
    try:
        for variant in (autotune.STEM_FIT_SCAN, autotune.STEM_FIT_CAMERA):
            autotune.set_choice(autotune.STEM_FIT, key, variant)
            outs.append((ws.run(params, targets).clone(), ws.partials.clone()))
    finally:
        autotune.clear()
    assert torch.equal(outs[0][0], outs[1][0])
    assert torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("n_side, scan_shape", [
    (128, (9, 7)),    # fixed-column tile form, four full tiles per camera length
    (72, (5, 6)),     # stepped form: 36 half-columns, second tile partial
    (64, (37, 41)),   # fixed-column form, 1517 positions: several per workgroup
])
def test_fit_tile_forms_and_position_sharing(device, n_side, scan_shape):
    """Both forms of the tile sums and the sharing of scan positions among the
    scan variant's workgroups: the two launch variants agree bitwise on every
    per-position row, and sampled rows match the FD oracle."""
    from temgymcore_amd import autotune

    print(f"[stem fit tiles n_side={n_side} scan={scan_shape}]", flush=True)
    model, _ = stem.reference_workload(n_cam=2, scan_shape=scan_shape, n_side=n_side)
    params = stem.params_tensor(model, device)
    targets = _targets(model, device)
    ws = stem.STEMFitWorkspace(model, device)
    key = (model.n_scan, model.n_rays, model.n_cam)
    rows = []
    try:
        for variant in (autotune.STEM_FIT_SCAN, autotune.STEM_FIT_CAMERA):
            autotune.set_choice(autotune.STEM_FIT, key, variant)
            ws.run(params, targets)
            rows.append(ws.partials.clone())
    finally:
        autotune.clear()
    assert torch.equal(rows[0], rows[1])
    r = rows[0].cpu().numpy().T  # [S, np]
    pick = np.random.default_rng(1).choice(model.n_scan, 3, replace=False)
    t = targets.cpu().numpy()[:, pick]
    ref_g = SO.fd_grad(_geom(model), model.params(), t, scan_idx=pick)
    ref_loss = SO.loss(_geom(model), model.params(), t, scan_idx=pick)
    # f32 floor: one f32 rounding of every term of the sums (the residuals
    # cancel to ~1e-5 of their absolute sum on these detectors)
    floor = 2.0 ** -24 * SO.grad_abs_scale(_geom(model), model.params(), t, scan_idx=pick)
    sub = r[pick].sum(axis=0)
    assert sub[-1] == pytest.approx(ref_loss, rel=1e-5)
    for blk in (slice(0, 16), slice(16, 17), slice(17, 18), slice(18, 20)):
        bar = 2e-4 * np.abs(ref_g[blk]).max() + floor[blk]
        err = np.abs(sub[blk] - ref_g[blk])
        assert np.all(err <= bar), (blk, err / bar)


@pytest.mark.parametrize("scan_shape", [(12, 10), (65, 64), (1, 1)])
def test_reduction_sums_partials_and_is_repeatable(device, scan_shape):
    """The fixed-order FP64 reduction over scan positions equals the sum of
    the per-scan-position terms (small, ragged and large scans), and
    repeated calls on one workspace are bitwise equal."""
    from temgymcore_amd import autotune

    model, _ = stem.reference_workload(n_cam=2, scan_shape=scan_shape, n_side=8)
    params = stem.params_tensor(model, device)
    targets = stem.stem_forward(stem.perturbed(model))["coords"]
    ws = stem.STEMFitWorkspace(model, device)
    key = (model.n_scan, model.n_rays, model.n_cam)
    try:
        for variant in (autotune.STEM_FIT_SCAN, autotune.STEM_FIT_CAMERA):
            autotune.set_choice(autotune.STEM_FIT, key, variant)
            outs = [ws.run(params, targets).clone() for _ in range(3)]
            assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
            rows = ws.partials.double().cpu().numpy()
            ref = rows.sum(axis=1)
            scale = np.abs(rows).sum(axis=1)
            got = outs[0].cpu().numpy()
            assert np.all(np.abs(got - ref) <= 1e-13 * scale + 1e-300)
    finally:
        autotune.clear()


def test_calibration_recovers_perturbed_geometry(device):
    """The calibration loop (L-BFGS over the fused loss + gradient) drives the
    loss from the unperturbed start to the f32 noise floor of the targets.

    With everything free it recovers the camera lengths and the detector
    coordinates.  Step and rotation act on the detector only through the
    descan map times the scan position (the descanner removes the scan), so
    they are recovered when the map is held and large enough for that term
    to stand far above the f32 resolution of the targets."""
    model, _ = stem.reference_workload(n_cam=3, scan_shape=(16, 16), n_side=16)
    truth = stem.perturbed(model)
    targets = stem.stem_forward(truth)["coords"]
    ws = stem.STEMFitWorkspace(model, device)
    floor = float(ws.run(stem.params_tensor(truth, device), targets)[-1])
    res = stem.calibrate(model, targets)
    print(f"all free: loss {res.initial_loss:.3e} -> {res.loss:.3e} (floor {floor:.3e}), {res.evaluations} evals")
    assert res.loss <= max(10 * floor, 1e-7 * res.initial_loss)
    np.testing.assert_allclose(res.params[18:], truth.params()[18:], rtol=1e-6)  # camera lengths
    fitted = stem.stem_forward(res.model)["coords"]
    assert (fitted - targets).abs().max().item() <= 1e-9

    # a strongly miscalibrated descan (entries ~0.05) over a 16 nm scan
    strong = dataclasses.replace(model, scan_step=1e-9,
                                 descan=np.random.default_rng(11).normal(0.0, 0.05, (4, 4)))
    truth = stem.perturbed(strong)
    t = truth.params()
    targets = stem.stem_forward(truth)["coords"]
    floor = float(stem.STEMFitWorkspace(strong, device).run(stem.params_tensor(truth, device), targets)[-1])
    start = strong.params()
    start[:16] = t[:16]  # descan map known
    res = stem.calibrate(strong, targets, fit=("scan_step", "scan_rotation", "camera_lengths"), params0=start)
    print(f"geometry: loss {res.initial_loss:.3e} -> {res.loss:.3e} (floor {floor:.3e}), {res.evaluations} evals")
    assert res.loss <= max(10 * floor, 1e-7 * res.initial_loss)
    np.testing.assert_allclose(res.params[16:], t[16:], rtol=1e-6)
    np.testing.assert_array_equal(res.params[:16], t[:16])
    with pytest.raises(ValueError):
        stem.calibrate(model, targets, fit=("pivot",))


def _bp_oracle(model, D_host, cam=0):
    geom = dict(_geom(model), sample_shape=tuple(model.sample_shape))
    det_Tinv = R.metres_to_pixels_matrix((0.0, 0.0), (model.det_pixel,) * 2, model.det_shape)
    img_Tinv = R.metres_to_pixels_matrix((0.0, 0.0), (model.sample_pixel,) * 2, model.sample_shape)
    return SO.backproject(geom, model.params(), D_host, det_Tinv, img_Tinv, cam)


@pytest.mark.parametrize("defocus, n_side", [(200e-9, 16), (2e-6, 16), (200e-9, 74)])
def test_backproject_vs_oracle(device, defocus, n_side):
    """Constant detector images per scan position (so the detector binning of
    a ray on a pixel edge cannot matter) back-project to the oracle's sums.
    At 2 um defocus the footprints exceed the workgroup's LDS tile and the
    global-memory path carries the outer rays (and each thread's 4 x 4 ray
    block spans more than its 3 x 3 pixel window); 74 rays per side leave
    partial blocks and workgroups.  Tolerance: the kernel's bilinear weights
    are f32 products (as in the forward), 1e-6 relative."""
    model, _ = stem.reference_workload(n_cam=2, scan_shape=(8, 8), n_side=n_side, defocus=defocus, det_pixel=1e-5)
    rng = np.random.default_rng(12)
    c = rng.uniform(0.5, 2.0, model.n_scan)
    D = np.broadcast_to(c[:, None, None], (model.n_scan,) + tuple(model.det_shape)).astype(np.float32)
    for cam in (0, 1):
        img, w = stem.backproject(model, torch.from_numpy(np.ascontiguousarray(D)).to(device), cam=cam, weights=True)
        ref_img, ref_w = _bp_oracle(model, D.astype(np.float64), cam)
        assert ref_w.sum() > 0.99 * model.n_scan * model.n_rays  # every ray lands
        np.testing.assert_allclose(w.cpu().numpy(), ref_w, rtol=0, atol=1e-6 * ref_w.max())
        np.testing.assert_allclose(img.cpu().numpy(), ref_img, rtol=0, atol=1e-6 * 2.0 * ref_w.max())
    img2, none = stem.backproject(model, torch.from_numpy(np.ascontiguousarray(D)).to(device))
    assert none is None and img2.shape == tuple(model.sample_shape)


def test_backproject_is_the_adjoint_of_the_forward_deposit(device):
    """<F I, D> == <I, F^T D> with F the forward kernel's 4D deposit (camera
    0) and F^T the back-projection kernel, for random I and D (the forward
    sums in f32: 1e-5 relative)."""
    model, _ = stem.reference_workload(n_cam=1, scan_shape=(16, 16), n_side=32)
    rng = np.random.default_rng(13)
    I = torch.from_numpy(rng.normal(size=model.sample_shape).astype(np.float32)).to(device)
    D = torch.from_numpy(rng.normal(size=(model.n_scan,) + tuple(model.det_shape)).astype(np.float32)).to(device)
    FI = stem.stem_forward(model, sample=I, coords=False, image4d=True)["image4d"]
    lhs = float((FI.double() * D.double()).sum())
    B, _ = stem.backproject(model, D)
    rhs = float((I.double() * B).sum())
    scale = float((FI.double().abs() * D.double().abs()).sum())
    assert abs(lhs - rhs) <= 1e-5 * scale, (lhs, rhs, scale)


def test_fit_terms_are_the_per_scan_position_shares(device):
    """tg_stem_fit_terms writes the same per-scan-position terms as the full
    fit; their row sums are the fit's outputs, the last row a loss map."""
    model, _ = stem.reference_workload(n_cam=2, scan_shape=(10, 12), n_side=16)
    params = stem.params_tensor(model, device)
    targets = stem.stem_forward(stem.perturbed(model))["coords"]
    ws = stem.STEMFitWorkspace(model, device)
    out = ws.run(params, targets).clone()
    full = ws.partials.clone()
    ws.workspace.zero_()
    terms = ws.terms(params, targets).clone()
    assert torch.equal(terms, full)
    rows = terms.cpu().numpy()
    assert np.all(np.abs(rows.sum(axis=1) - out.cpu().numpy()) <= 1e-12 * np.abs(rows).sum(axis=1) + 1e-300)
    assert np.all(rows[-1] >= 0)


@pytest.mark.parametrize("det_shape, n_side, rot", [
    ((1, 1), 8, 0.0), ((7, 5), 30, 0.0), ((250, 253), 62, 0.0), ((64, 256), 64, 0.0), ((33, 257), 20, 0.0),
    ((3, 8192), 64, 0.0), ((2, 8193), 64, 0.0), ((97, 101), 2, 0.0), ((120, 131), 46, 33.0), ((128, 60), 64, 90.0)])
def test_dataset_bands_vs_forward_deposit(device, det_shape, n_side, rot):
    """The dataset kernel (bands of rows in LDS, written once) on detectors that
    do not divide into its bands, misaligned rows, one-row bands, the width
    past which the deposit goes through memory, and rotated detectors (whose
    rows mix both slopes): the deposit of the same call's coordinates and
    values, within one f32 rounding of each term (a pixel's terms are added in
    any order); buffers that held other numbers are overwritten."""
    import ctypes

    model, sample = stem.reference_workload(n_cam=1, scan_shape=(3, 5), det_shape=det_shape, n_side=n_side,
                                            det_pixel=6e-4 / det_shape[0])
    sample_t = torch.from_numpy(sample).to(device)
    params = stem.params_tensor(model, device)
    g = model.geometry()
    if rot:
        R_ = np.deg2rad(rot)
        rows = np.array(g.det_m).reshape(2, 3)
        c = np.array([(det_shape[0] - 1) / 2, (det_shape[1] - 1) / 2])
        lin = np.array([[np.cos(R_), np.sin(R_)], [-np.sin(R_), np.cos(R_)]]) @ rows[:, :2]
        g.det_m[:] = np.column_stack([lin, c]).reshape(-1).tolist()
    res = stem.stem_forward(model, params, sample_t, coords=True, values=True)
    img = torch.full((model.n_scan,) + det_shape, float("nan"), device=device)
    lib = stem._lib.load()
    wide = det_shape[1] > lib.tg_stem_dataset_max_width()
    st = lib.tg_stem_dataset(ctypes.byref(g), params.data_ptr(), sample_t.data_ptr(), img.data_ptr(),
                             stem._lib.stream_ptr(device))
    assert st == (-1 if wide else 0)
    if wide:
        img = stem.stem_forward(model, params, sample_t, coords=False, image4d=True)["image4d"]
    xy = res["coords"].double().cpu().numpy()[0]
    v = res["values"].double().cpu().numpy()
    m = np.array(g.det_m)
    py = np.rint((m[0] * xy[..., 1] + m[1] * xy[..., 0]) + m[2])
    px = np.rint((m[3] * xy[..., 1] + m[4] * xy[..., 0]) + m[5])
    ok = (py >= 0) & (py < det_shape[0]) & (px >= 0) & (px < det_shape[1])
    s = np.broadcast_to(np.arange(model.n_scan)[:, None], ok.shape)
    ref, size, n = np.zeros(img.shape), np.zeros(img.shape), np.zeros(img.shape)
    at = (s[ok], py[ok].astype(int), px[ok].astype(int))
    np.add.at(ref, at, v[ok])
    np.add.at(size, at, np.abs(v[ok]))
    np.add.at(n, at, 1)
    assert ok.any()
    assert np.all(np.abs(img.double().cpu().numpy() - ref) <= 2.0 ** -24 * n * size)


def test_dataset_of_undefined_parameters_bins_to_pixel_zero(device):
    """NaN detector positions cast to pixel (0, 0), as the forward's binning
    does: each position's whole sum lies there (256 values within pi, added in
    any order: 256 roundings of at most 256 pi 2^-24)."""
    model, sample = stem.reference_workload(n_cam=1, scan_shape=(1, 2), n_side=16, det_shape=(40, 300))
    params = stem.params_tensor(model, device)
    params[0] = float("nan")
    img = stem.stem_forward(model, params, torch.from_numpy(sample).to(device), coords=False, image4d=True)["image4d"]
    ref = torch.zeros_like(img)
    g = model.geometry()
    import ctypes

    sample_t = torch.from_numpy(sample).to(device)
    st = stem._lib.load().tg_stem_forward(ctypes.byref(g), params.data_ptr(), sample_t.data_ptr(), None, None,
                                          ref.data_ptr(), stem._lib.stream_ptr(device))
    assert st == 0
    torch.cuda.synchronize()
    assert img[:, 0, 0].abs().min() > 0  # every ray's value, on pixel (0, 0)
    assert (img[:, 1:].abs().sum() + img[:, 0, 1:].abs().sum()) == 0
    assert (img - ref).abs().max() <= 2 * 256 * 256 * np.pi * 2.0 ** -24
