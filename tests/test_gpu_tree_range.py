"""The spot tree's numbers at the ends of fp32, on the GPU.

Renders are linear in the sources' values and their gradients in values and
image gradients, so powers of two come back exactly wherever no intermediate
leaves fp32's range; what is left is the order of the sums (1e-6 of the largest,
of some 10^2 fp32 additions each 2^-24).
"""
import ctypes

import pytest
import torch

import iactrace_amd as ia
from iactrace_amd import _lib
from iactrace_amd.render import LaunchConfig, RenderPlan
from tests.test_gpu_tree import _sources, _telescope

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _all(tel, src, val, st, cot, layout=0):
    g = tel.mirror_groups[0]
    leaves = [t.detach().clone().requires_grad_(True)
              for t in (g.rotations, g.positions, src, val)]
    rot, pos, s, v = leaves
    t = ia.Telescope([g.replace(rotations=rot, positions=pos)], tel.obstruction_groups,
                     tel.sensors)
    img = ia.render(t, s, v, st, launch=ia.LaunchConfig(layout=layout)).reshape(-1)
    grads = torch.autograd.grad(img, leaves, cot)
    return dict(zip(("image", "rotations", "positions", "sources", "values"),
                    [x.detach().double() for x in (img, *grads)]))


def _scene(light):
    tel = _telescope(100, "hex", "all", 0.0, 5, n_facets=7)
    src, val, st = _sources(300, light, 3)
    cot = torch.linspace(0.5, 1.5, tel.sensors[0].n_pixels, device=DEV)
    return tel, torch.as_tensor(src, device=DEV), torch.as_tensor(val, device=DEV), st, cot


@pytest.mark.parametrize("light", ["far", "near", "parallel"])
@pytest.mark.parametrize("a,b,per_metre", [(2.0 ** -60, 1.0, True), (2.0 ** -100, 1.0, False),
                                           (2.0 ** -55, 2.0 ** -55, False),
                                           (2.0 ** 60, 2.0 ** 60, True)])
def test_powers_of_two_come_back(light, a, b, per_metre):
    """a: of the values, b: of the image gradient.  per_metre: with the gradients
    per metre, which are smaller by the distance (2^33 at 1e10 m, 2^13 near by):
    ones that leave fp32's range themselves are not compared."""
    tel, src, val, st, cot = _scene(light)
    base = _all(tel, src, val, st, cot)
    got = _all(tel, src, val * a, st, cot * b)
    factor = {"image": a, "rotations": a * b, "positions": a * b, "sources": a * b, "values": b}
    for k, f in factor.items():
        if k in ("positions", "sources") and not per_metre:
            continue
        scale = float(base[k].abs().max())
        err = float((got[k] / f - base[k]).abs().max())
        print(f"[range {light} {a:.1e} {b:.1e}] {k}: {err / max(scale, 1e-300):.1e}", flush=True)
        assert err <= 1e-6 * scale, k


@pytest.mark.parametrize("light", ["far", "near", "parallel"])
@pytest.mark.parametrize("what", ["nan value", "inf value", "nan source", "inf source",
                                  "nan image gradient"])
def test_numbers_that_are_not_finite_spread_as_ray_by_ray(light, what):
    """They reach the same pixels and gradients as in the sample-major kernels, and
    no others (the rest: 1e-5 of the largest, see test_gpu_tree)."""
    tel, src, val, st, cot = _scene(light)
    bad = float(what.split()[0])
    lit = int(_all(tel, src, val, st, cot)["image"].argmax())
    {"value": val[17:18], "source": src[17], "image": cot[lit:lit + 1]}[what.split()[1]][:] = bad
    ref = _all(tel, src, val, st, cot, layout=1)
    got = _all(tel, src, val, st, cot)
    for k in ref:
        a, b = torch.isfinite(ref[k]), torch.isfinite(got[k])
        print(f"[finite {light} {what}] {k}: {int((~a).sum())} not, {int((~b).sum())} here",
              flush=True)
        assert bool((a == b).all()), k
        if bool(a.any()):
            assert float((got[k] - ref[k])[a].abs().max()) <= 1e-5 * float(ref[k][a].abs().max())


def test_tree_ends_where_its_grids_would_wrap():
    """2^24 runs of 1024 samples: the nodes' kernel would need 2^32 threads.  The
    workspace tells the kernels apart (nothing is launched): 144 bytes for each of a
    facet's three nodes beside its record, or the culling tables alone."""
    plan = RenderPlan(_telescope(1, "square", "all", 0.0, 5, n_facets=7))
    sc = plan.scene([])
    L = LaunchConfig().abi()

    def per_facet(n):
        sc.facets.n_facets = n
        return _lib.lib().iact_workspace_size(ctypes.byref(sc), 128, _lib.MODE_IMAGE,
                                              ctypes.byref(L)) / n

    assert per_facet((1 << 24) - 1) > 64 + 3 * 144
    assert 64 < per_facet(1 << 24) < 64 + 3 * 144
