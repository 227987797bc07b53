"""Response matrices from sample records, fp64 block images, the secondary's
starting root and the batched gradient adds, on the GPU.

Response rows and images are compared with the fp64 sums of render_debug's rays
(every ray's pixel and value).  A row entry is a wave's fp32 sum of 64 lanes
(six roundings), added in fp64 and rounded once (and once per part, at most 25
of them here): 2e-6 of the row's largest entry.

A secondary that is a pure conic starts its iteration from the root on its own
sheet.  The same mirror with a term of 1e-30 takes the general route, whose
converged root is the same to fp64 rounding; a hit's fp32 rounding may then move
a ray by one ulp and, at a pixel edge, to the next pixel: of some 10^5 rays at
most a few, 1e-4 of the image.
"""
import numpy as np
import pytest
import torch

import iactrace_amd as ia
from iactrace_amd import configs
from tests.test_gpu_tree import _obstructions, _sensor, _sources

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _telescope(samples, sensor, obstructions, n=7):
    groups = [g.to(DEV) for g in ia.group_mirrors(configs.parabolic_dish()[:n])]
    groups[0] = ia.MCIntegrator(samples).sample_group(groups[0], 3)
    tel = ia.Telescope(groups, ia.group_obstructions(_obstructions(obstructions)), [sensor])
    return tel.apply_roughness(20.0)


def _debug_rows(tel, src, val, light, ns, n_pixels):
    """(ns, P) fp64 sums of the rays of render_debug."""
    _, v, pix = ia.render_debug(tel, src, val, light, return_pixels=True)
    nf = len(tel.mirror_groups[0])
    row = torch.arange(ns, device=DEV)[None, :, None].expand(nf, ns, v.numel() // (nf * ns))
    at = (row.reshape(-1) * n_pixels + pix.long())[pix >= 0]
    out = torch.zeros(ns * n_pixels, dtype=torch.float64, device=DEV)
    return out.index_add_(0, at, v.double()[pix >= 0]).reshape(ns, n_pixels)


@pytest.mark.parametrize("sensor", ["square", "oblong-edge-tilted", "hex", "hex-edge"])
@pytest.mark.parametrize("samples,ns,light,obstructions", [
    (1, 1, "parallel", "none"), (63, 2, "far", "all"), (64, 3, "mixed", "all"),
    (65, 65, "parallel", "many"), (200, 129, "near", "none"), (37, 701, "far", "none")])
def test_response_rows_are_the_sums_of_their_rays(sensor, samples, ns, light, obstructions):
    s = _sensor(sensor)
    tel = _telescope(samples, s, obstructions)
    src, val, light = _sources(ns, light, 5)
    src, val = torch.as_tensor(src), torch.as_tensor(val)
    got = ia.render_response_matrix(tel, src, val, light)
    ref = _debug_rows(tel, src, val, light, ns, s.n_pixels)
    assert torch.isfinite(got).all()
    scale = ref.abs().amax(1, keepdim=True).clamp_min(1e-30)
    assert float(((got.double() - ref).abs() / scale).max()) < 2e-6


@pytest.mark.parametrize("side", [(90, 90), (91, 90), (91, 91), (128, 127), (128, 130)])
def test_images_where_fp64_entries_fill_the_block(side):
    """Around 65536 bytes: fp64, fp32 and no image in LDS; response rows too."""
    w, h = side
    s = ia.SquareSensor([0, 0, 36.066], [0, 0, 0], w, h, (-0.8, 0.8, -0.8, 0.8))
    tel = _telescope(130, s, "none")
    src, val, light = _sources(9, "far", 2)
    src, val = torch.as_tensor(src), torch.as_tensor(val)
    ref = _debug_rows(tel, src, val, light, 9, w * h)
    got = ia.render_response_matrix(tel, src, val, light).double()
    # (fp32 rows: up to some 100 further roundings)
    assert float((got - ref).abs().max() / ref.max()) < 1e-5
    img = ia.render(tel, src, val, light).double().reshape(-1)
    assert float((img - ref.sum(0)).abs().max() / ref.sum(0).max()) < 1e-5


@pytest.mark.parametrize("conic", [-16.0, -1.0, -0.6, 0.0])
@pytest.mark.parametrize("curvature,offset", [(-0.05, 0.0), (-0.05, 0.07), (0.0, 0.0)])
def test_secondary_root_on_its_own_sheet(conic, curvature, offset):
    imgs = []
    for term in (0.0, 1e-30):
        prim, sec = configs.cassegrain()[0]
        sec = ia.Mirror(sec.position, sec.rotation,
                        ia.AsphericSurface(curvature, conic, [term]), sec.aperture,
                        offset=[offset, -0.5 * offset], optical_stage=1)
        groups = [g.to(DEV) for g in ia.group_mirrors([prim, sec])]
        groups[0] = ia.MCIntegrator(500).sample_group(groups[0], 4)
        tel = ia.Telescope(groups, [], [ia.SquareSensor([0, 0, -0.45], [0, 0, 0], 64, 64,
                                                        (-0.6, 0.6, -0.6, 0.6))])
        src = torch.as_tensor(configs.parallel_grid(15, 15, 0.05))
        imgs.append(ia.render(tel, src, torch.ones(225), "parallel").double())
    a, b = imgs
    assert float(b.sum()) > 0
    assert float((a - b).abs().sum() / b.abs().sum()) < 1e-4


@pytest.mark.parametrize("ns", [1, 63, 64, 65, 130])
def test_splat_gradients_per_source(ns):
    """Value and source gradients, 64 sources at a time: dL/dvalue is the
    cotangent's sum over the unit-value image (fp32 sums of some 10^3 rays: 1e-5)."""
    p = 0.0419
    s = ia.DifferentiableSquareSensor([0, 0, 36.066], [0, 0, 0], 32, 30,
                                      (-16 * p, 16 * p, -15 * p, 15 * p), 0.7, 2)
    tel = _telescope(70, s, "none")
    src, val, light = _sources(ns, "far", 8)
    src, val = torch.as_tensor(src, device=DEV), torch.as_tensor(val, device=DEV)
    rng = torch.Generator().manual_seed(1)
    cot = torch.rand(30, 32, generator=rng).to(DEV)
    v = val.clone().requires_grad_(True)
    x = src.clone().requires_grad_(True)
    g, gx = torch.autograd.grad(ia.render(tel, x, v, light), [v, x], cot)
    rows = ia.render_response_matrix(tel, src, torch.ones(ns, device=DEV), light).double()
    ref = rows @ cot.double().reshape(-1)
    assert float((g.double() - ref).abs().max()) <= 1e-5 * float(ref.abs().max())
    one = torch.autograd.grad(ia.render(tel, x[-1:], v[-1:], light), x, cot)[0][-1]
    assert float((gx[-1] - one).abs().max()) <= 1e-4 * float(one.abs().max())


@pytest.mark.parametrize("ns", [128, 1024, 1025, 4096, 4097])
def test_sorted_sources_are_a_permutation(ns):
    """Obstructed images sort their sources, up to 4096 in one block: the image is
    the sum of the rays (2e-5: see test_gpu_tree), the gradients of the values come
    back in the caller's order."""
    tel = _telescope(16, _sensor("hex"), "all", n=3)
    src, val, light = _sources(ns, "far", ns)
    src, val = torch.as_tensor(src, device=DEV), torch.as_tensor(val, device=DEV)
    P = tel.sensors[0].n_pixels
    v = val.clone().requires_grad_(True)
    img = ia.render(tel, src, v, light)
    rows = _debug_rows(tel, src, torch.ones_like(val), light, ns, P)
    ref = val.double() @ rows
    assert float((img.detach().double() - ref).abs().max()) <= 2e-5 * float(ref.max())
    cot = torch.rand(P, generator=torch.Generator().manual_seed(2)).to(DEV)
    g = torch.autograd.grad(img, v, cot)[0].double()
    want = rows @ cot.double()
    assert float((g - want).abs().max()) <= 1e-5 * float(want.abs().max())


@pytest.mark.parametrize("sensor", ["square", "oblong-edge-tilted", "hex", "hex-edge"])
@pytest.mark.parametrize("samples,ns,light", [(1, 64, "far"), (65, 130, "parallel"),
                                              (1030, 513, "far"), (100, 70, "near")])
def test_tree_without_obstructions_by_choice(sensor, samples, ns, light):
    """Small clear scenes take the tree where the caller asks for the source-major
    layout (tolerances: test_gpu_tree)."""
    s = _sensor(sensor)
    L = ia.LaunchConfig(layout=2)
    tel = _telescope(samples, s, "none", n=5)
    src, val, light = _sources(ns, light, samples)
    src, val = torch.as_tensor(src, device=DEV), torch.as_tensor(val, device=DEV)
    v = val.clone().requires_grad_(True)
    img = ia.render(tel, src, v, light, launch=L).reshape(-1)
    rows = _debug_rows(tel, src, torch.ones_like(val), light, ns, s.n_pixels)
    ref = val.double() @ rows
    assert float((img.detach().double() - ref).abs().max()) <= 2e-5 * float(ref.max())
    cot = torch.rand(s.n_pixels, generator=torch.Generator().manual_seed(2)).to(DEV)
    g = torch.autograd.grad(img, v, cot)[0].double()
    want = rows @ cot.double()
    assert float((g - want).abs().max()) <= 1e-5 * float(want.abs().max())


def test_response_of_more_sources_than_one_grid_holds():
    """2^24 sources and some more: blocks of 512 threads for two sources each would
    be a grid of over 2^32 threads.  Every source has the same direction, so each
    row is the first source's scaled by the value (three roundings: 4e-7)."""
    groups = [g.to(DEV) for g in ia.group_mirrors(configs.parabolic_dish()[:1])]
    groups[0] = ia.MCIntegrator(1).sample_group(groups[0], 3)
    tel = ia.Telescope(groups, [], [ia.SquareSensor([0, 0, 36.0], [0, 0, 0], 2, 2,
                                                    (-0.5, 0.5, -0.5, 0.5))])
    ns = (1 << 24) + 1029
    src = torch.tensor([[0.001, 0.002, -1.0]], dtype=torch.float64, device=DEV).repeat(ns, 1)
    val = torch.linspace(0.5, 1.5, ns, dtype=torch.float32, device=DEV)
    row = ia.render_response_matrix(tel, src[:1], torch.ones(1, device=DEV), "parallel")
    assert float(row.max()) > 0
    got = ia.render_response_matrix(tel, src, val, "parallel")
    err = 0.0
    for a in range(0, ns, 1 << 22):
        want = val[a:a + (1 << 22), None] * row
        err = max(err, float((got[a:a + (1 << 22)] - want).abs().max()))
    assert err <= 4e-7 * 1.5 * float(row.max())
