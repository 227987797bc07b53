"""What a RenderPlan keeps between calls, on the CPU (its tables and descriptors;
nothing is launched)."""
import torch

import iactrace_amd as ia
from iactrace_amd import configs
from iactrace_amd.render import RenderPlan


def _plan(groups):
    plan = RenderPlan.__new__(RenderPlan)  # (the constructor asks for a HIP device)
    plan.tel = ia.Telescope(groups, [], [ia.SquareSensor([0, 0, 36], [0, 0, 0], 4, 4,
                                                         (-1, 1, -1, 1))])
    plan.sensor = plan.tel.sensors[0]
    plan.primary, plan.secondary = groups, []
    plan.device = torch.device("cpu")
    plan._build_static()
    return plan


def _sampled(a, b):
    g, = ia.group_mirrors(configs.parabolic_dish()[a:b])
    n = b - a
    return g.replace(points=torch.zeros(n, 2, 3), normals=torch.zeros(n, 2, 3),
                     weights=torch.ones(n, 2), perturbation_delta=torch.zeros(n, 2, 3))


def _index(plan):
    keep = []
    sc = plan.scene(keep)
    index = [t for t in keep if t.dtype == torch.int32][-1]
    assert sc.facets.surface_index == index.data_ptr()
    return sc.facets.n_facets, index.tolist()


def test_group_index_follows_groups_that_change_their_length():
    """Telescopes are immutable by convention; where a group's tensors are replaced
    all the same, each facet still has an entry, and its own group's."""
    groups = [_sampled(0, 3), _sampled(3, 5)]
    plan = _plan(groups)
    assert _index(plan) == (5, [0, 0, 0, 1, 1])
    for name, t in vars(_sampled(0, 4)).items():
        setattr(groups[0], name, t)
    assert _index(plan) == (6, [0, 0, 0, 0, 1, 1])
    for g, n in zip(groups, (2, 4)):  # the same number of facets, divided otherwise
        for name, t in vars(_sampled(0, n)).items():
            setattr(g, name, t)
    assert _index(plan) == (6, [0, 0, 1, 1, 1, 1])
