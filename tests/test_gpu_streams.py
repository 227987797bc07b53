"""Memory of a render on another stream than its plan's, on the GPU."""
import pytest
import torch

import iactrace_amd as ia
from iactrace_amd import configs
from iactrace_amd.render import RenderPlan

pytestmark = pytest.mark.gpu
DEV = "cuda"


def test_group_index_outlives_an_aspheric_gradient_on_another_stream():
    """The gradient is queued behind a sleep and its plan goes away.  Until it has
    run, no new tensor takes the memory of the facets' group index."""
    n = 1021
    side = torch.cuda.Stream()
    groups = [g.to(DEV) for g in ia.group_mirrors(configs.parabolic_dish(n_facets=n))]
    groups[0] = ia.MCIntegrator(8).sample_group(groups[0], 3)
    groups[0] = groups[0].replace(aspheric=torch.zeros(2))
    g = groups[0]
    tel = ia.Telescope(groups, [], [ia.SquareSensor([0, 0, 36.0], [0, 0, 0], 8, 8,
                                                    (-0.5, 0.5, -0.5, 0.5))])
    src = torch.tensor([[0.0, 0.0, 1e10]], dtype=torch.float64, device=DEV)
    args = (torch.ones(64, device=DEV), src, torch.ones(1, device=DEV), "point", g.rotations,
            g.positions, (False, False, False, False, True))
    plan = RenderPlan(tel)
    want = plan.backward(*args)["aspheric"].clone()
    at, size = plan.surface_index.data_ptr(), 4 * n
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(1 << 28)
        got = plan.backward(*args)["aspheric"]
        done = side.record_event()
    del plan  # (held by nothing else: a plan made directly is in no telescope's cache)
    new = [torch.empty(size, dtype=torch.uint8, device=DEV) for _ in range(16)]
    assert not done.query()
    assert all(t.data_ptr() != at for t in new)
    torch.cuda.synchronize()
    assert float(want.abs().max()) > 0
    assert float((got - want).abs().max()) <= 1e-6 * float(want.abs().max())
