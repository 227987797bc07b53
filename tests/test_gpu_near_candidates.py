"""Obstruction candidates of sources some 100 m away, on the GPU.

The directions of a near source's rays differ over a facet by its extent as
seen from the source, a degree here.  The spot tree bounds them per run of
samples: on facets of several runs of 1024 samples, or with an aperture off its
position, a run's own extent is smaller than its distance from the facet
position, from which the sources' directions are taken.  The image is compared
with the fp64 sum of render_debug's rays (tolerances: test_gpu_tree); thin
cylinders all over the bundle make a candidate lost at its edge visible.
"""
import numpy as np
import pytest
import torch

import iactrace_amd as ia
from iactrace_amd import configs
from iactrace_amd.geometry import AsphericSurface, PolygonAperture
from iactrace_amd.mirrors import Mirror
from iactrace_amd.obstructions import Cylinder
from tests.test_gpu_tree import _sensor

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _mirrors(kind):
    if kind == "several runs":
        return configs.parabolic_dish()[:7]
    surf = AsphericSurface(1.0 / 72.0, 0.0, [])
    square = 0.15 * np.array([[1, 1], [-1, 1], [-1, -1], [1, -1]])
    return [Mirror([0, 0, 0], [0, 0, 0], surf, PolygonAperture(square + c))
            for c in ([1.5, 0.4], [-1.2, 1.0], [0.3, -1.6])]


def _cylinders(seed):
    rng = np.random.default_rng(seed)
    out = []
    for z in rng.uniform(12.0, 34.0, 200):
        p = np.append(rng.uniform(-1.4, 1.4, 2), z)
        q = p + np.append(rng.uniform(-0.3, 0.3, 2), rng.uniform(0.1, 0.3))
        out.append(Cylinder(p, q, rng.uniform(0.004, 0.015)))
    return out


@pytest.mark.parametrize("facets,samples", [("several runs", 4096), ("several runs", 2065),
                                            ("off the position", 1000),
                                            ("off the position", 3000)])
@pytest.mark.parametrize("sensor", ["hex", "square"])
def test_no_candidate_is_lost_near_by(facets, samples, sensor):
    groups = [g.to(DEV) for g in ia.group_mirrors(_mirrors(facets))]
    groups[0] = ia.MCIntegrator(samples).sample_group(groups[0], 3)
    s = _sensor(sensor)
    tel = ia.Telescope(groups, ia.group_obstructions(_cylinders(samples)), [s])
    rng = np.random.default_rng(1)
    ns = 150
    src = np.append(rng.uniform(-0.2, 0.2, (ns, 2)), rng.uniform(90.0, 120.0, (ns, 1)), 1)
    src = torch.as_tensor(src, device=DEV)
    val = torch.as_tensor(rng.lognormal(0.0, 0.5, ns).astype(np.float32), device=DEV)

    def rays(t):
        ref = torch.zeros(s.n_pixels, dtype=torch.float64, device=DEV)
        _, v, pix = ia.render_debug(t, src, val, "point", return_pixels=True)
        return ref.index_add_(0, pix[pix >= 0].long(), v[pix >= 0].double())

    img = ia.render(tel, src, val, "point").reshape(-1).double()
    ref = rays(tel)
    clear = rays(ia.Telescope(groups, [], [s]))
    assert 0.3 * float(clear.sum()) < float(ref.sum()) < 0.99 * float(clear.sum())
    err = (img - ref).abs() - 2e-5 * ref
    print(f"[near {facets} {samples} {sensor}] lit {float(ref.sum() / clear.sum()):.3f}, max "
          f"excess {float(err.max() / ref.max()):.2e} of the largest pixel", flush=True)
    assert float(err.max()) <= 1e-6 * float(ref.max())
