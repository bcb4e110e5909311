"""The column kernel against the register programs of the same models (bit for
bit), and its three ways of counting rays into a detector image against the
pixels of its own positions, at the edges of its vectors, chunks, bands and
counters."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import ray_oracle as O
from temgymcore_amd import _lib, _program
from temgymcore_amd.components import Biprism, Deflector, Detector, Lens, Rotator, Scanner
from temgymcore_amd.ray import Ray
from temgymcore_amd.run import plan_run_to_end, plan_run_to_image, run_to_end, run_to_image

pytestmark = pytest.mark.gpu
FIELDS = ("x", "y", "dx", "dy", "pathlength")


def _model(shape=(64, 64)):
    return [Lens(z=0.3, focal_length=0.8), Deflector(z=0.5, def_x=3e-3, def_y=-1e-3), Rotator(z=0.5, angle=33.0),
            Scanner(z=0.7, scan_pos_x=0.01, scan_pos_y=-0.02, scan_tilt_x=1e-3), Biprism(z=0.9, def_x=2e-3),
            Lens(z=1.1, focal_length=-1.7), Detector(z=1.4, pixel_size=(1.6 / shape[0], 1.6 / shape[1]), shape=shape)]


def _arrays(n, dtype, device, offset=0, seed=0):
    g = torch.Generator(device=device).manual_seed(seed)
    big = torch.rand(5, n + offset, generator=g, device=device, dtype=torch.float64) * 0.6 - 0.3
    return [b[offset:] for b in big.to(dtype)]


def _programs_of(plan):
    """The register programs' outputs of a column plan (into the plan's buffers)."""
    stream = _lib.stream_ptr(plan.trace.device)
    for prog, spec, _ in plan.programs:
        st = _lib.load().tg_ray_program_run(ctypes.byref(prog), None if spec is None else ctypes.byref(spec), stream)
        assert st == 0
    return plan.out_ray


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 255, 1023, 1025, 2047, 2049, 300_001])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("path", [0.25, None])
def test_column_equals_its_register_programs(device, dtype, n, offset, path):
    x, y, dx, dy, p = _arrays(n, dtype, device, offset)
    x[0], dx[-1] = float("inf"), float("nan")
    if n > 2:
        x[1], y[1] = 0.0, -0.0
    ray = Ray(x=x, y=y, dx=dx, dy=dy, z=0.0, pathlength=p if path is None else path)
    plan = plan_run_to_end(ray, _model())
    assert plan.column is not None
    got = {k: getattr(plan.launch(), k).clone() for k in FIELDS}
    cached = run_to_end(ray, _model()), run_to_end(ray, _model())  # a miss (or hit) and a hit
    _programs_of(plan)
    for k in FIELDS:
        ref = getattr(plan.out_ray, k)
        for v in (got[k], *(getattr(c, k) for c in cached)):
            torch.testing.assert_close(v, ref, rtol=0, atol=0, equal_nan=True)
            assert v.shape == x.shape and v.is_contiguous()


def test_column_of_a_two_dimensional_bundle(device):
    x, y, dx, dy, p = (a.reshape(37, 11) for a in _arrays(407, torch.float64, device))
    ray = Ray(x=x, y=y, dx=dx, dy=dy, z=0.0, pathlength=p)
    out = run_to_end(ray, _model())
    flat = run_to_end(Ray(x=x.reshape(-1), y=y.reshape(-1), dx=dx.reshape(-1), dy=dy.reshape(-1), z=0.0,
                          pathlength=p.reshape(-1)), _model())
    for k in FIELDS:
        assert getattr(out, k).shape == (37, 11)
        torch.testing.assert_close(getattr(out, k).reshape(-1), getattr(flat, k), rtol=0, atol=0)


def _counts(ray, det):
    T = O.metres_to_pixels_matrix((0.0, 0.0), det.pixel_size, det.shape)
    py, px = O.metres_to_pixels(ray.x.double().cpu().numpy(), ray.y.double().cpu().numpy(), T)
    return O.into_image(py, px, det.shape)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", [(1, 1), (5, 13), (63, 65), (256, 256), (320, 256), (321, 256), (1000, 1024), (90_000, 3)])
@pytest.mark.parametrize("n, offset", [(700, 0), ((1 << 18) - 1, 0), (1 << 18, 1), (400_003, 0)])
def test_column_counts(device, dtype, shape, n, offset):
    """Private histograms (up to 81,920 bins), memory atomics (more bins, few
    rays) and bands (many rays): exactly the pixels of the final positions,
    added to what the accumulator held."""
    x, y, dx, dy, _ = _arrays(n, dtype, device, offset, seed=3)
    model = _model(shape)
    ray = Ray(x=x, y=y, dx=dx, dy=dy, z=0.0, pathlength=0.0)
    acc = torch.randint(0, 9, shape, device=device, dtype=torch.int32)
    before = acc.clone()
    out, img = run_to_image(ray, model, acc=acc)
    ref = _counts(out, model[-1])
    assert ref.sum() > 0.1 * n
    np.testing.assert_array_equal((img - before).cpu().numpy().astype(np.int64), ref)


@pytest.mark.parametrize("acc_dtype", [torch.int32, torch.int64, torch.float32, torch.float64])
@pytest.mark.parametrize("shape", [(64, 64), (700, 512)])
def test_column_counts_of_every_accumulator(device, acc_dtype, shape):
    x, y, dx, dy, _ = _arrays(300_000, torch.float32, device, seed=4)
    model = _model(shape)
    acc = torch.zeros(shape, dtype=acc_dtype, device=device)
    out, img = run_to_image(Ray(x=x, y=y, dx=dx, dy=dy, z=0.0, pathlength=0.0), model, acc=acc)
    np.testing.assert_array_equal(img.cpu().numpy().astype(np.int64), _counts(out, model[-1]))


@pytest.mark.parametrize("shape", [(64, 64), (300, 300)])
@pytest.mark.parametrize("n", [65_535, 65_536, 1_000_000])
def test_column_counters_do_not_carry(device, shape, n):
    """Every ray on one pixel: a workgroup's (or a slice's) 16-bit counter is
    never asked to hold more than 65,535."""
    one = torch.zeros(n, dtype=torch.float32, device=device)
    det = Detector(z=1.0, pixel_size=(1.0, 1.0), shape=shape)
    _, img = run_to_image(Ray(x=one, y=one.clone(), dx=one.clone(), dy=one.clone(), z=0.0, pathlength=0.0), [det])
    assert img.sum() == n and img.max() == n


def test_column_counts_of_positions_off_the_detector(device):
    """Nothing on the detector (chunks without a pixel), and NaN positions,
    which cast to pixel (0, 0)."""
    n = 300_000
    det = Detector(z=1.0, pixel_size=(1e-6, 1e-6), shape=(400, 400))
    far = torch.full((n,), 5.0, device=device)
    zero = torch.zeros(n, device=device)
    _, img = run_to_image(Ray(x=far, y=far.clone(), dx=zero, dy=zero.clone(), z=0.0, pathlength=0.0), [det])
    assert img.sum() == 0
    far[1000:3000] = float("nan")
    _, img = run_to_image(Ray(x=far, y=far.clone(), dx=zero, dy=zero.clone(), z=0.0, pathlength=0.0), [det])
    assert img.sum() == 2000 and img[0, 0] == 2000


def test_column_plan_on_a_side_stream_and_in_a_graph(device):
    """The bands' scratch memory belongs to the launch's stream, and a captured
    plan replays to the eager counts."""
    x, y, dx, dy, _ = _arrays(400_000, torch.float32, device, seed=6)
    model = _model((700, 512))
    ray = Ray(x=x, y=y, dx=dx, dy=dy, z=0.0, pathlength=0.0)
    plan = plan_run_to_image(ray, model)
    plan.launch()
    ref = _counts(plan.out_ray, model[-1])
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    plan.acc.zero_()
    torch.cuda.synchronize()
    plan.launch(side.cuda_stream)
    junk = [torch.full((1 << 20,), i, device=device) for i in range(8)]  # would land on memory given back too early
    torch.cuda.synchronize()
    np.testing.assert_array_equal(plan.acc.cpu().numpy().astype(np.int64), ref)
    assert all(int(j[0]) == i for i, j in enumerate(junk))
    with torch.cuda.stream(side):
        plan.launch()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.acc.zero_()
        plan.launch()
    for _ in range(3):
        plan.acc.fill_(7)
        plan.out_ray.x.fill_(0.0)
        graph.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(plan.acc.cpu().numpy().astype(np.int64), ref)
        np.testing.assert_array_equal(_counts(plan.out_ray, model[-1]), ref)
