"""A plan's launch takes no memory: what it needs was taken when it was built
(a stream capture that torch did not begin may not allocate)."""
import pytest
import torch

from temgymcore_amd.components import Detector, Lens
from temgymcore_amd.ray import Ray
from temgymcore_amd.run import plan_run_to_end, plan_run_to_image

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(64, 64), (256, 256), (700, 512)])  # LDS counting, its largest, two passes
@pytest.mark.parametrize("n", [1000, 300_000])
def test_launch_takes_no_memory(device, shape, n):
    g = torch.Generator(device=device).manual_seed(2)
    x, y, dx, dy, p = (torch.rand(n, generator=g, device=device) * 0.1 for _ in range(5))
    ray = Ray(x=x, y=y, dx=dx, dy=dy, z=0.0, pathlength=p)
    model = [Lens(z=0.3, focal_length=0.8), Detector(z=1.0, pixel_size=(0.001, 0.001), shape=shape)]
    for plan in (plan_run_to_image(ray, model), plan_run_to_end(ray, model)):
        assert plan.column is not None
        before = torch.cuda.memory_stats(device)["allocation.all.allocated"]
        plan.launch()
        assert torch.cuda.memory_stats(device)["allocation.all.allocated"] == before
    torch.cuda.synchronize()


def test_plan_dropped_while_another_stream_counts(device):
    """The scratch memory of a plan launched on another stream is not given
    back before that stream is done with it."""
    n, shape = 3_000_000, (700, 512)
    g = torch.Generator(device=device).manual_seed(3)
    x, y, dx, dy, p = (torch.rand(n, generator=g, device=device) * 0.2 for _ in range(5))
    ray = Ray(x=x, y=y, dx=dx, dy=dy, z=0.0, pathlength=p)
    model = [Lens(z=0.3, focal_length=0.8), Detector(z=1.0, pixel_size=(0.001, 0.001), shape=shape)]
    plan = plan_run_to_image(ray, model)
    plan.launch()
    ref = plan.acc.clone()
    size, side = plan.workspace[0].numel(), torch.cuda.Stream()
    torch.cuda.synchronize()
    plan.acc.zero_()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)  # (some ms, on that stream)
    plan.launch(side.cuda_stream)
    acc, out = plan.acc, plan.out_ray
    del plan
    junk = torch.full((size,), 1, dtype=torch.uint8, device=device)  # would land on memory given back too early
    torch.cuda.synchronize()
    assert torch.equal(acc, ref) and bool((junk == 1).all()) and out.x.numel() == n
