"""Which kernel a launch takes, and the kernels at both sides of the spot tree's
limits, on the GPU.

The tree serves automatic launches from 128 sources behind obstructions and from
1.5e9 rays without, on cameras whose image and tables fit 64 KB of LDS; layout=2
traces every ray of the same records.  Which of the two a launch takes shows in its
workspace: the tree's holds nodes, the other culling tables.  Images are compared
with the fp64 sum of render_debug's rays, gradients with the sample-major adjoint,
with the tolerances of test_gpu_tree.
"""
import ctypes

import pytest
import torch

import iactrace_amd as ia
from iactrace_amd import _lib, configs
from iactrace_amd.render import RenderPlan
from tests.test_gpu_tree import _sources, _telescope
from tests.test_gpu_tree_range import _all

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _workspaces(tel, ns, layouts=(0, 2)):
    plan = RenderPlan(tel)
    sc = plan.scene([])
    return [_lib.lib().iact_workspace_size(ctypes.byref(sc), ns, _lib.MODE_IMAGE,
                                           ctypes.byref(ia.LaunchConfig(layout=k).abi()))
            for k in layouts]


def _takes_tree(tel, ns):
    own, rays = _workspaces(tel, ns)
    return own != rays


def _check_image(tel, s, v, st, launch=None, step=128):
    P = tel.sensors[0].n_pixels
    img = ia.render(tel, s, v, st, launch=launch).reshape(-1).double()
    ref = torch.zeros(P, dtype=torch.float64, device=DEV)
    for b in range(0, len(v), step):
        _, rv, pix = ia.render_debug(tel, s[b:b + step], v[b:b + step], st, return_pixels=True)
        ok = pix >= 0
        ref.index_add_(0, pix[ok].long(), rv[ok].double())
    err = (img - ref).abs() - 2e-5 * ref.abs()
    assert float(ref.max()) > 0
    assert float(err.max()) <= 1e-6 * float(ref.max())


def _check_gradients(tel, s, v, st, layout=0):
    gen = torch.Generator().manual_seed(3)
    cot = (0.5 + torch.rand(tel.sensors[0].n_pixels, generator=gen)).to(DEV)
    ref = _all(tel, s, v, st, cot, layout=1)
    got = _all(tel, s, v, st, cot, layout=layout)
    for k in ref:
        scale = float(ref[k].abs().max())
        assert float((got[k] - ref[k]).abs().max()) <= 1e-5 * scale, k


def _on_device(ns, light, seed):
    src, val, st = _sources(ns, light, seed)
    return torch.as_tensor(src, device=DEV), torch.as_tensor(val, device=DEV), st


@pytest.mark.parametrize("m,ns,sensor,obst,light,rough", [
    (1, 128, "hex", "all", "far", 0.0),
    (15, 130, "hex-edge", "all", "near", 20.0),
    (16, 512, "oblong-edge-tilted", "all", "mixed", 0.0),
    (17, 513, "square", "many", "wide", 0.0),
    (64, 140, "hex-edge", "all", "parallel", 0.0),
    (65, 1025, "oblong-edge-tilted", "many", "far", 30.0),
    (1025, 200, "oblong-edge-tilted", "all", "wide", 0.0),
    (2065, 150, "hex-edge", "all", "far", 0.0),
    (2048, 129, "square", "many", "near", 0.0)])
def test_obstructed_launches_walk_the_tree(m, ns, sensor, obst, light, rough):
    tel = _telescope(m, sensor, obst, rough, m + ns, n_facets=7)
    assert _takes_tree(tel, ns) and not _takes_tree(tel, 127)
    s, v, st = _on_device(ns, light, m)
    _check_image(tel, s, v, st)
    _check_gradients(tel, s, v, st)


@pytest.mark.parametrize("m,facets,light,sensor,rough", [
    (17, 91, "far", "hex-edge", 0.0), (65, 61, "parallel", "oblong-edge-tilted", 0.0),
    (1030, 19, "mixed", "hex", 20.0), (4096, 37, "far", "square", 0.0)])
def test_large_clear_launches_walk_the_tree(m, facets, light, sensor, rough):
    """1.5e9 rays and a few more.  A source's rays are summed in its flux's gradient:
    one of them in 1500 to 150000 would show there."""
    tel = _telescope(m, sensor, "none", rough, m, n_facets=facets)
    ns = -(-1500000000 // (facets * m)) + 3
    assert _takes_tree(tel, ns) and not _takes_tree(tel, ns - 4)
    s, v, st = _on_device(ns, light, m)
    cot = torch.linspace(0.5, 1.5, tel.sensors[0].n_pixels, device=DEV)
    ref = _all(tel, s, v, st, cot, layout=2)
    got = _all(tel, s, v, st, cot)
    for k in ref:
        # (2e-5: a pixel's sum, see test_gpu_tree; 1e-5: the gradients')
        tol = 2e-5 if k == "image" else 1e-5
        scale = float(ref[k].abs().max())
        err = float((got[k] - ref[k]).abs().max())
        print(f"[clear {m} x {ns} {light} {sensor}] {k}: {err / max(scale, 1e-300):.1e}", flush=True)
        assert err <= tol * scale, k


def _large_camera(kind):
    p = 0.0419
    if kind == "hex":
        return ia.HexagonalSensor([0, 0, 36.066], [0, 0, 0], configs.hex_camera(3600, 0.5 * p))
    return ia.SquareSensor([0, 0, 36.066], [0, 0, 0], 75, 70, (-16 * p, 16 * p, -15 * p, 15 * p))


@pytest.mark.parametrize("kind", ["hex", "square"])
@pytest.mark.parametrize("obst", ["all", "none"])
@pytest.mark.parametrize("ns,light,layout", [(64, "mixed", 0), (128, "far", 0), (200, "near", 2),
                                             (130, "parallel", 0)])
def test_cameras_above_the_tree_are_traced_ray_by_ray(kind, obst, ns, light, layout):
    tel = _telescope(130, "hex", obst, 0.0, ns, n_facets=7)
    tel = ia.Telescope(tel.mirror_groups, tel.obstruction_groups, [_large_camera(kind)])
    assert not _takes_tree(tel, ns)
    s, v, st = _on_device(ns, light, 4)
    _check_image(tel, s, v, st, launch=ia.LaunchConfig(layout=layout))
    _check_gradients(tel, s, v, st, layout)


@pytest.mark.parametrize("m,ns,sensor,obst,light", [
    (130, 200, "hex", "all", "mixed"), (65, 129, "hex-edge", "many", "far"),
    (70, 300, "oblong-edge-tilted", "all", "parallel"), (40, 70, "square", "all", "near"),
    (100, 150, "square", "none", "far")])
def test_layout_two_traces_every_ray(m, ns, sensor, obst, light):
    """... in scenes that the tree serves too, and in clear ones below its threshold,
    where the automatic launch does the same."""
    tel = _telescope(m, sensor, obst, 0.0, ns, n_facets=7)
    own, rays = _workspaces(tel, ns)
    assert (own != rays) == (obst != "none" and ns >= 128)
    s, v, st = _on_device(ns, light, 4)
    _check_image(tel, s, v, st, launch=ia.LaunchConfig(layout=2, sample_group=5))
    _check_gradients(tel, s, v, st, 2)


@pytest.mark.parametrize("wants", [("rotations",), ("rotations", "values"), ("positions",),
                                   ("sources",)])
@pytest.mark.parametrize("light", ["far", "near", "parallel"])
def test_gradients_whose_tables_fit_walk_the_tree_without_its_image(wants, light):
    """A camera whose fp64 image is too large for the tree, its fp32 gradient is not;
    with the sums that source gradients need it is again."""
    tel = _telescope(130, "hex", "all", 0.0, 9, n_facets=7)
    tel = ia.Telescope(tel.mirror_groups, tel.obstruction_groups, [_large_camera("hex")])
    ns = 140
    assert not _takes_tree(tel, ns)
    plan = RenderPlan(tel)
    sc = plan.scene([])
    own, rays = [_lib.lib().iact_bwd_workspace_size(
        ctypes.byref(sc), ns, ctypes.byref(ia.LaunchConfig(layout=k).abi())) for k in (0, 2)]
    assert own > rays
    s, v, st = _on_device(ns, light, 6)
    gen = torch.Generator().manual_seed(3)
    cot = (0.5 + torch.rand(tel.sensors[0].n_pixels, generator=gen)).to(DEV)

    def grads(layout):
        g = tel.mirror_groups[0]
        leaf = {"rotations": g.rotations, "positions": g.positions, "sources": s, "values": v}
        leaf = {k: t.detach().clone().requires_grad_(k in wants) for k, t in leaf.items()}
        t = ia.Telescope([g.replace(rotations=leaf["rotations"], positions=leaf["positions"])],
                         tel.obstruction_groups, tel.sensors)
        img = ia.render(t, leaf["sources"], leaf["values"], st,
                        launch=ia.LaunchConfig(layout=layout)).reshape(-1)
        return torch.autograd.grad(img, [leaf[k] for k in wants], cot, allow_unused=True)

    for k, a, b in zip(wants, grads(1), grads(0)):
        assert float((a.double() - b.double()).abs().max()) <= 1e-5 * float(a.abs().max()), k
