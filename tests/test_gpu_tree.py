"""The spot tree (images and gradients summed per run of samples) against the
per-ray kernels, on the GPU.

The image is compared with the fp64 sum of render_debug's rays -- every ray's
pixel and value -- and the gradients with the sample-major adjoint's.  Sizes
sit at the edges of the tree's runs (16, 64, 1024 samples), of its blocks of
512 sources and of its 64-lane lists; scenes cover both cameras, edge masks,
tilted and non-square sensors, rough mirrors, every obstruction kind, far, near
and parallel light, and culling off.

Tolerances: a pixel's rays are added in fp32 within a block, at most some 300
additions here, each of relative rounding 2^-24: 2e-5 of the pixel (a ray on
the wrong side of an edge moves a pixel of at most 10^4 rays by 1e-4).  The
adjoints sum the same terms in different orders: 1e-5 of the largest.
"""
import numpy as np
import pytest
import torch

import iactrace_amd as ia
from iactrace_amd import configs
from iactrace_amd.obstructions import Box, Cylinder, OrientedBox, Sphere, Triangle

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _sensor(kind):
    p = 0.0419
    if kind == "square":
        return ia.SquareSensor([0, 0, 36.066], [0, 0, 0], 32, 30,
                               (-16 * p, 16 * p, -15 * p, 15 * p))
    if kind == "oblong-edge-tilted":
        return ia.SquareSensor([0.1, -0.05, 36.0], [1.5, -2.0, 20.0], 24, 40,
                               (-16 * p, 16 * p, -15 * p, 15 * p), edge_width=0.004)
    if kind == "hex-edge":
        return ia.HexagonalSensor([0.05, 0, 36.1], [0.5, 1.0, 10.0],
                                  configs.hex_camera(613, p), edge_width=0.002)
    return ia.HexagonalSensor([0, 0, 36.066], [0, 0, 0], configs.hex_camera(1000, p))


def _obstructions(kind):
    if kind == "none":
        return []
    obs = [Box([-0.6, -0.5, 30.0], [0.4, 0.6, 31.0]),
           Cylinder([2.5, 2.0, 1.0], [0.3, 0.3, 33.0], 0.1),
           Cylinder([-2.0, 1.0, 3.0], [-1.0, -1.5, 6.0], 0.05),
           Sphere([1.0, -1.2, 9.0], 0.3),
           OrientedBox([-1.5, -1.5, 12.0], [0.3, 0.1, 0.2],
                       np.linalg.qr(np.arange(9.0).reshape(3, 3) + np.eye(3))[0]),
           Triangle([0.5, 1.5, 7.0], [1.5, 1.0, 7.5], [0.9, 2.2, 8.0])]
    if kind == "many":  # more candidates than a wave's lanes
        for k in range(90):
            a = 0.7 * k
            x, y = 0.03 * k * np.cos(a), 0.03 * k * np.sin(a)
            obs.append(Cylinder([x, y, 2.0 + 0.3 * k], [x + 0.4, y + 0.1, 2.1 + 0.3 * k], 0.01))
    return obs


def _sources(n, light, seed):
    rng = np.random.default_rng(seed)
    val = rng.lognormal(0.0, 0.5, n).astype(np.float32)
    if light == "parallel":
        d = np.stack([rng.uniform(-0.03, 0.03, n), rng.uniform(-0.03, 0.03, n), -np.ones(n)], 1)
        return d * rng.uniform(0.7, 1.3, (n, 1)), val, "parallel"
    z = np.full(n, 1e10)
    if light == "near":
        z[:] = 1.1e4
    if light == "mixed":
        z[::3] = 9e3
    a = rng.uniform(-0.03, 0.03, (n, 2))
    if light == "wide":  # a few directions far off the others
        a[::17] *= 20.0
    return np.stack([z * a[:, 0], z * a[:, 1], z], 1), val, "point"


CASES = [
    # samples, sources, sensor, obstructions, light, roughness (arcsec), culling
    (1, 64, "hex", "none", "far", 0.0, 0),
    (15, 511, "square", "none", "far", 0.0, 0),
    (16, 512, "hex", "none", "parallel", 0.0, 0),
    (17, 513, "hex-edge", "none", "far", 0.0, 0),
    (64, 200, "oblong-edge-tilted", "none", "far", 30.0, 0),
    (65, 130, "hex", "all", "far", 0.0, 0),
    (200, 600, "square", "all", "parallel", 10.0, 0),
    (256, 515, "hex", "all", "mixed", 0.0, 0),
    (100, 100, "hex-edge", "all", "near", 20.0, 0),
    (1000, 140, "hex", "all", "far", 0.0, -1),
    (1024, 300, "hex", "many", "far", 0.0, 0),
    (1025, 100, "square", "none", "wide", 0.0, 0),
    (2065, 70, "oblong-edge-tilted", "all", "far", 0.0, 0),
    (130, 1100, "hex", "many", "parallel", 0.0, 0),
]


def _telescope(m, sensor, obst, rough, seed, n_facets=19):
    wl = configs.Workload("tree", configs.parabolic_dish(n_facets=n_facets), _obstructions(obst),
                          _sensor(sensor), m, np.zeros((1, 3)), np.ones(1, np.float32), "point",
                          tilt_sigma_deg=0.02, tilt_seed=seed)
    tel = wl.telescope(DEV, key=seed)
    return tel.apply_roughness(rough) if rough else tel


@pytest.mark.parametrize("m,ns,sensor,obst,light,rough,cull", CASES)
def test_image_is_the_sum_of_the_rays(m, ns, sensor, obst, light, rough, cull):
    tel = _telescope(m, sensor, obst, rough, m + ns)
    src, val, st = _sources(ns, light, m)
    s, v = torch.as_tensor(src, device=DEV), torch.as_tensor(val, device=DEV)
    P = tel.sensors[0].n_pixels
    img = ia.render(tel, s, v, st, launch=ia.LaunchConfig(culling=cull)).reshape(-1).double()
    ref = torch.zeros(P, dtype=torch.float64, device=DEV)
    for b in range(0, ns, 128):
        _, rv, pix = ia.render_debug(tel, s[b:b + 128], v[b:b + 128], st, return_pixels=True)
        ok = pix >= 0
        ref.index_add_(0, pix[ok].long(), rv[ok].double())
    err = (img - ref).abs() - 2e-5 * ref.abs()
    print(f"[tree m={m} ns={ns} {sensor} {obst} {light}] max excess {float(err.max()):.2e} of "
          f"{float(ref.max()):.4g}", flush=True)
    assert float(ref.max()) > 0
    assert float(err.max()) <= 1e-6 * float(ref.max())


@pytest.mark.parametrize("m,ns,sensor,obst,light,rough,cull", CASES)
def test_gradients_match_the_sample_major_adjoint(m, ns, sensor, obst, light, rough, cull):
    tel = _telescope(m, sensor, obst, rough, m + ns, n_facets=7)
    src, val, st = _sources(ns, light, m)
    g = tel.mirror_groups[0]
    rng = np.random.default_rng(5)
    W = torch.as_tensor(rng.uniform(0.5, 1.5, tel.sensors[0].n_pixels), dtype=torch.float32,
                        device=DEV)

    def grads(launch, which):
        rot = g.rotations.detach().clone().requires_grad_(True)
        pos = g.positions.detach().clone().requires_grad_("positions" in which)
        s = torch.as_tensor(src, device=DEV).requires_grad_("sources" in which)
        v = torch.as_tensor(val, device=DEV).requires_grad_("values" in which)
        t = ia.Telescope([g.replace(rotations=rot, positions=pos)], tel.obstruction_groups,
                         tel.sensors)
        (ia.render(t, s, v, st, launch=launch).reshape(-1) * W).sum().backward()
        out = {"rotations": rot.grad, "positions": pos.grad, "sources": s.grad, "values": v.grad}
        return {k: x.double() for k, x in out.items() if x is not None}

    every = ("positions", "sources", "values")
    ref = grads(ia.LaunchConfig(layout=1, culling=cull), every)
    got = grads(ia.LaunchConfig(layout=2, culling=cull), every)
    got["rotations alone"] = grads(ia.LaunchConfig(layout=2, culling=cull), ())["rotations"]
    ref["rotations alone"] = ref["rotations"]
    assert float(ref["values"].abs().max()) > 0
    for k in ref:
        scale = float(ref[k].abs().max())
        err = float((got[k] - ref[k]).abs().max())
        print(f"[tree grad m={m} ns={ns} {sensor} {obst} {light}] {k}: {err / max(scale, 1e-300):.2e}",
              flush=True)
        assert err <= 1e-5 * scale, k
