"""The work that a program using iactrace_amd has it do, as measurable cases.

Each case goes through the package's public entry points (a call of the
telescope, ``render`` with autograd, ``render_response_matrix``,
``AlignmentFit``) on telescopes that the package's own generators build: the
12 m Davies-Cotton dish, the 28 m parabolic dish and the two-mirror
Cassegrain.  ``listed`` names twelve, from one point source to the full field
of a large dish; ``draw`` gives others of the same ranges (odd source and
sample counts among them).  ``exact`` restates the render in plain float64
torch: aperture sampling (Philox4x32-10), pose, shadows, reflection, secondary
mirror, sensor plane and binning, with gradients by autograd.
"""
import functools
import math

import numpy as np
import torch

import iactrace_amd as ia
from iactrace_amd import configs
from iactrace_amd.batched import AlignmentFit, render_batched

PITCH_DC = 15.0 * math.tan(math.radians(0.16))  # 0.16 degree pixels at 15 m
PITCH_PAR = 0.04193673807057477
FIELD_DEG = 2.5


def _case(name, kind, **kw):
    c = dict(kind=kind, dish="parabolic", facets=875, round=False, samples=1024, sources=1024,
             distance=1e10, sensor="hex", pixels=2048, obstructions="none", tilt_mrad=0.0,
             rough_arcsec=0.0)
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the spot of one star on axis: the smallest call, latency and launches
        _case("psf_star", "image", dish="dc", facets=382, samples=1000, sources=1,
              sensor="square", pixels=960),
        # light from a few points at shower height (12 km), rough round mirrors,
        # the sampler's default 128 samples per facet
        _case("psf_near", "image", dish="dc", facets=382, round=True, samples=128, sources=37,
              distance=1.2e4, pixels=960, rough_arcsec=24.0),
        # an ordinary star field, ragged sizes, mirrors of some roughness, masts
        _case("field_ragged", "image", samples=500, sources=1021, obstructions="masts",
              tilt_mrad=0.5, rough_arcsec=10.0),
        # a dense field on the small dish with many samples per facet
        _case("field_dc", "image", dish="dc", facets=382, samples=4096, sources=4096,
              sensor="square", pixels=960),
        # the large dish's whole field behind camera box and masts
        _case("field_hex", "image", sources=16384, obstructions="masts", tilt_mrad=0.5),
        # the same dish behind a full support truss (271 members)
        _case("field_truss", "image", sources=4096, obstructions="truss", tilt_mrad=0.5),
        # gradients of a field image in facet tilts, facet positions and fluxes
        _case("align_grad", "grad", sources=2048, obstructions="masts", tilt_mrad=0.5),
        # one iteration of the alignment fit of several pointings of unequal size
        _case("fit_batch", "fit", sources=5000, instances=5, obstructions="masts", tilt_mrad=0.5),
        # gradients through a Gaussian-splat camera (spot positions matter)
        _case("splat_grad", "splat", dish="dc", facets=382, samples=256, sources=150, pixels=960,
              tilt_mrad=0.5),
        # response matrix of the small dish over a grid of directions
        _case("response_dish", "response", dish="dc", facets=382, round=True, samples=64,
              sources=4096, distance=0.0, pixels=960, obstructions="masts", rough_arcsec=24.0),
        # response matrix through a secondary mirror
        _case("response_cassegrain", "response", dish="cassegrain", facets=1, samples=2048,
              sources=8192, distance=0.0, sensor="square", pixels=4096),
        # gradients in both mirrors' aspheric coefficients
        _case("aspheric_grad", "aspheric", dish="cassegrain", facets=1, samples=2048,
              sources=2048, distance=0.0, sensor="square", pixels=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["image", "image", "image", "image", "grad", "grad", "fit", "splat",
                       "response", "response", "aspheric"])
    if kind == "aspheric" or (kind == "response" and rng.random() < 0.4):
        m = _log_int(rng, 256, 2048)
        s = _log_int(rng, 64, 8192 if kind == "response" else 2048)
        return _case(None, kind, dish="cassegrain", facets=1, samples=m, sources=s, distance=0.0,
                     sensor="square", pixels=4096)
    dc = rng.random() < 0.4
    dish = dict(dish="dc", facets=382) if dc else dict(dish="parabolic", facets=875)
    dish["round"] = rng.random() < 0.3
    dish["sensor"], dish["pixels"] = ("square", 960) if dc and rng.random() < 0.5 else \
        ("hex", 960 if dc else 2048)
    dish["obstructions"] = rng.choice(["none", "masts"] if dc else ["none", "masts", "masts",
                                                                     "truss"])
    dish["tilt_mrad"] = rng.choice([0.0, 0.5, 0.5])
    dish["rough_arcsec"] = rng.choice([0.0, 0.0, 10.0, 24.0])
    dish["distance"] = rng.choice([1e10, 1e10, 1e10, 1.2e4, 0.0])
    if kind == "image":
        m, s = _log_int(rng, 64, 4096), _log_int(rng, 1, 16384)
        most = 14e9 if dish["obstructions"] != "truss" else 3.5e9
        while m * s * dish["facets"] > most:
            s = s // 2 + 1
    elif kind == "grad":
        m, s = _log_int(rng, 64, 1024), _log_int(rng, 16, 2048)
        if dish["obstructions"] == "truss":
            s = min(s, 765)
    elif kind == "fit":
        m, s = _log_int(rng, 128, 1024), _log_int(rng, 600, 5000)
        dish.update(instances=rng.randint(2, 6), distance=1e10, tilt_mrad=0.5, rough_arcsec=0.0,
                    obstructions="masts", round=False)
    elif kind == "splat":
        m, s = _log_int(rng, 64, 256), _log_int(rng, 8, 150)
        dish.update(obstructions="none")
    else:
        m, s = _log_int(rng, 32, 256), _log_int(rng, 50, 4096)
        dish.update(distance=0.0)
        if dish["obstructions"] == "truss":
            dish["obstructions"] = "masts"
        while m * s * dish["facets"] > 1.0e8:
            s = s // 2 + 1
    return _case(None, kind, samples=m, sources=s, **dish)


# ------------------------------------------------------------------ inputs

@functools.lru_cache(maxsize=None)
def _mirrors(dish, rnd):
    if dish == "cassegrain":
        return tuple(configs.cassegrain()[0])
    ms = configs.davies_cotton_dish() if dish == "dc" else configs.parabolic_dish()
    if rnd:
        r = 0.30 if dish == "dc" else 0.45
        ms = [ia.Mirror(m.position, m.rotation, m.surface, ia.DiskAperture(r)) for m in ms]
    return tuple(ms)


@functools.lru_cache(maxsize=None)
def _hex_centres(pixels, pitch):
    return configs.hex_camera(pixels, pitch)


def _camera(c):
    """(position, camera parameters) of a case."""
    if c["dish"] == "cassegrain":
        return (0.0, 0.0, -0.45), dict(w=64, h=64, bounds=(-0.3, 0.3, -0.3, 0.3))
    dc = c["dish"] == "dc"
    pos = (0.0, 0.0, 15.0) if dc else (0.0, 0.0, 36.066)
    p = PITCH_DC if dc else PITCH_PAR
    if c["sensor"] == "square":
        return pos, dict(w=32, h=30, bounds=(-16 * p, 16 * p, -15 * p, 15 * p))
    return pos, dict(pitch=p)


@functools.lru_cache(maxsize=None)
def _sensor(dish, sensor, pixels, splat):
    pos, k = _camera(dict(dish=dish, sensor=sensor))
    if sensor == "square":
        if splat:
            return ia.DifferentiableSquareSensor(pos, [0, 0, 0], k["w"], k["h"], k["bounds"], 0.7,
                                                 2)
        return ia.SquareSensor(pos, [0, 0, 0], k["w"], k["h"], k["bounds"])
    xy = _hex_centres(pixels, k["pitch"])
    if splat:
        return ia.DifferentiableHexagonalSensor(pos, [0, 0, 0], xy, 0.7, 1)
    return ia.HexagonalSensor(pos, [0, 0, 0], xy)


def _obstructions(c):
    """Camera box and four masts of either dish, or the truss."""
    if c["obstructions"] == "none":
        return []
    if c["obstructions"] == "truss":
        return configs.support_truss()
    rim, z0, zc, h = (6.2, 1.3, 15.1, 0.8) if c["dish"] == "dc" else (14.2, 1.4, 36.25, 1.0)
    out = [ia.Box([-h, -h, zc], [h, h, zc + 2.0 * h])]
    for k in range(4):
        a = math.radians(45.0 + 90.0 * k)
        out.append(ia.Cylinder([rim * math.cos(a), rim * math.sin(a), z0],
                               [math.copysign(h, math.cos(a)), math.copysign(h, math.sin(a)), zc],
                               0.1))
    return out


def _sources(c, seed, n):
    """(sources, values): a disk of 2.5 degrees of lognormal point sources, or
    directions of a grid with the given spacing (distance 0)."""
    rng = np.random.default_rng([seed, n])
    if c["distance"] == 0.0:
        nx = int(math.ceil(math.sqrt(2.0 * n))) if c["dish"] == "cassegrain" else \
            int(math.ceil(math.sqrt(n)))
        step = 0.01 if c["dish"] == "cassegrain" else 2.0 * FIELD_DEG / max(nx, 2)
        src = configs.parallel_grid(nx, -(-n // nx), step)[:n]
        return src, np.exp(rng.normal(0.0, 0.1, n)).astype(np.float32)
    if n == 1:
        return np.array([[0.0, 0.0, c["distance"]]]), np.ones(1, np.float32)
    return configs.point_source_field(n, FIELD_DEG, seed * 1009 + n, c["distance"])


def _tilts(c, seed, nf):
    if not c["tilt_mrad"]:
        return np.zeros((nf, 2))
    return np.random.default_rng([seed, 7]).normal(0.0, math.degrees(c["tilt_mrad"] * 1e-3),
                                                   (nf, 2))


def _sizes(c, seed):
    """Source counts of a fit's instances, uneven, summing to the case's."""
    w = np.random.default_rng([seed, 3]).uniform(0.2, 1.8, c["instances"])
    n = np.maximum((w / w.sum() * c["sources"]).astype(int), 64)
    return [int(x) for x in n]


def _telescope(c, seed, dev):
    groups = [g.to(dev) for g in ia.group_mirrors(list(_mirrors(c["dish"], c["round"])))]
    groups[0] = ia.MCIntegrator(c["samples"]).sample_group(groups[0], seed)
    rot = groups[0].rotations.clone()
    rot[:, :2] += torch.as_tensor(_tilts(c, seed, len(groups[0])), dtype=torch.float32, device=dev)
    groups[0] = groups[0].replace(rotations=rot)
    tel = ia.Telescope(groups, ia.group_obstructions(_obstructions(c)),
                       [_sensor(c["dish"], c["sensor"], c["pixels"], c["kind"] == "splat")])
    return tel.apply_roughness(c["rough_arcsec"]) if c["rough_arcsec"] else tel


def _cotangent(c, seed):
    """dL/dimage of a gradient case."""
    return np.random.default_rng([seed, 9]).uniform(0.5, 1.5, c["pixels"]).astype(np.float32)


def prepare(case, seed):
    c, dev = case, torch.device("cuda")
    tel = _telescope(c, seed, dev)
    kind = c["kind"]
    st = {"kind": kind, "type": "parallel" if c["distance"] == 0.0 else "point"}
    if kind == "fit":
        fields = [_sources(c, seed + 31 * i, n) for i, n in enumerate(_sizes(c, seed))]
        off = np.concatenate([[0], np.cumsum([len(v) for _, v in fields])]).astype(np.int64)
        src = np.concatenate([s for s, _ in fields])
        val = np.concatenate([v for _, v in fields])
        n = len(fields)
        base = tel.mirror_groups[0].rotations
        rot = base.unsqueeze(0).repeat(n, 1, 1)
        for i in range(n):
            rot[i, :, :2] += torch.as_tensor(_tilts(c, seed + 100 + i, base.shape[0]),
                                             dtype=torch.float32, device=dev)
        target = render_batched(tel, base.unsqueeze(0).repeat(n, 1, 1).contiguous(), src, val,
                                off)
        st["fit"] = AlignmentFit(tel, rot, src, val, off, target, lr=1e-4)
        return st
    src, val = _sources(c, seed, c["sources"])
    st["src"] = torch.as_tensor(src, dtype=torch.float64, device=dev)
    st["val"] = torch.as_tensor(val, device=dev)
    if kind in ("grad", "splat", "aspheric"):
        st["cot"] = torch.as_tensor(_cotangent(c, seed), device=dev)
        g = tel.mirror_groups[0]
        if kind == "aspheric":
            a0 = g.aspheric.detach().clone().requires_grad_(True)
            a1 = torch.zeros(2).requires_grad_(True)
            groups = [g.replace(aspheric=a0), tel.mirror_groups[1].replace(aspheric=a1)]
            st["wrt"] = {"primary": a0, "secondary": a1}
        else:
            rot = g.rotations.detach().clone().requires_grad_(True)
            pos = g.positions.detach().clone().requires_grad_(True)
            st["val"] = st["val"].requires_grad_(True)
            st["wrt"] = {"rotations": rot, "positions": pos, "values": st["val"]}
            groups = [g.replace(rotations=rot, positions=pos)]
        tel = ia.Telescope(groups, tel.obstruction_groups, tel.sensors)
    st["tel"] = tel
    return st


def run(state):
    kind = state["kind"]
    if kind == "fit":
        fit = state["fit"]
        fit.step()
        return {"images": fit.images, "rotations": fit.rotations, "exp_avg": fit.exp_avg}
    tel, src, val = state["tel"], state["src"], state["val"]
    if kind == "image":
        return tel(src, val, source_type=state["type"])
    if kind == "response":
        return ia.render_response_matrix(tel, src, val, state["type"])
    img = ia.render(tel, src, val, state["type"])
    wrt = state["wrt"]
    grads = torch.autograd.grad(img, list(wrt.values()), state["cot"].reshape(img.shape))
    return {"image": img.detach(), **dict(zip(wrt, grads))}


def work(case):
    """The bytes of the inputs and outputs, and the operations that no way of
    summing the rays avoids: every sample is brought to world space (63), and
    every (facet, source) pair has a direction and a spot to be placed (60; a
    secondary mirror adds its root to every ray, 300).  Rays of one facet and
    source that meet the same pixel can be summed in any order, so a count per
    ray would be no floor.  A backward counts as twice its forward."""
    c = case
    rows = c.get("instances", 1)
    samples, pairs = c["facets"] * c["samples"], c["facets"] * c["sources"]
    flops = 63.0 * samples * rows + 60.0 * pairs
    if c["dish"] == "cassegrain":
        flops += 300.0 * pairs * c["samples"]
    if c["kind"] == "splat":
        flops += 20.0 * pairs * c["samples"]
    out = c["sources"] * c["pixels"] if c["kind"] == "response" else rows * c["pixels"]
    nbytes = 40.0 * samples + 28.0 * c["sources"] + 4.0 * out
    if c["kind"] in ("grad", "splat", "fit", "aspheric"):
        flops *= 3.0
        nbytes += 24.0 * c["facets"] * rows + 4.0 * c["sources"] + 4.0 * rows * c["pixels"]
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------------ float64

def _philox(ctr, seed):
    """Philox4x32-10 of (n, 4) counters (Salmon et al., SC'11)."""
    m0, m1, mask = np.uint64(0xD2511F53), np.uint64(0xCD9E8D57), np.uint64(0xFFFFFFFF)
    x = [v.astype(np.uint64) for v in ctr]
    k0, k1 = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
    for _ in range(10):
        p0, p1 = m0 * x[0], m1 * x[2]
        x = [(p1 >> np.uint64(32)) ^ x[1] ^ np.uint64(k0), p1 & mask,
             (p0 >> np.uint64(32)) ^ x[3] ^ np.uint64(k1), p0 & mask]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return x


def _sag(x, y, curv, conic, asph):
    """Height and slopes of a conic + sum a_i (r^2)^(2 (i + 1)) surface."""
    r2 = x * x + y * y
    K = (1.0 + conic) * curv * curv
    s = torch.sqrt(1.0 - K * r2)
    z = r2 * curv / (1.0 + s)
    g = curv / (1.0 + s) + r2 * curv * K / (2.0 * s * (1.0 + s) ** 2)
    for i in range(len(asph)):
        z = z + asph[i] * r2 ** (2 * (i + 1))
        g = g + asph[i] * (2 * (i + 1)) * r2 ** (2 * i + 1)
    return z, 2.0 * x * g, 2.0 * y * g


def _dot(a, b):
    return a[..., 0] * b[..., 0] + a[..., 1] * b[..., 1] + a[..., 2] * b[..., 2]


def _unit(v):
    return v / torch.sqrt(_dot(v, v))[..., None]


def _euler(deg):
    a = torch.deg2rad(deg)
    c, s = torch.cos(a).unbind(-1), torch.sin(a).unbind(-1)
    o, z = torch.ones_like(c[0]), torch.zeros_like(c[0])

    def mat(*v):
        return torch.stack(v, -1).reshape(*v[0].shape, 3, 3)

    rx = mat(o, z, z, z, c[0], -s[0], z, s[0], c[0])
    ry = mat(c[1], z, s[1], z, o, z, -s[1], z, c[1])
    rz = mat(c[2], -s[2], z, s[2], c[2], z, z, z, o)
    return rz @ ry @ rx


def _exact_samples(c, seed, dev, asph):
    """Facet-frame points, normals, roughness displacements and weights."""
    ms, m = _mirrors(c["dish"], c["round"])[:c["facets"]], c["samples"]
    nf = len(ms)
    f, k = np.divmod(np.arange(nf * m, dtype=np.int64), m)
    zero = np.zeros_like(f)
    a = _philox([k, f, zero, zero], seed)
    b = _philox([k, f, zero, zero + 1], seed)

    def u(w, plus=0):
        return torch.as_tensor(((w >> np.uint64(8)).astype(np.float64) + plus) / 2.0 ** 24,
                               device=dev).reshape(nf, m)

    ap = ms[0].aperture
    if hasattr(ap, "radius"):
        r = torch.sqrt(u(a[0])) * float(np.float32(ap.radius))
        th = u(a[1]) * (2.0 * math.pi)
        x, y = r * torch.cos(th), r * torch.sin(th)
        area = math.pi * float(np.float32(ap.radius)) ** 2
    else:
        v = np.asarray(ap.vertices, np.float32).astype(np.float64)
        e = v[1:] - v[0]
        tri = np.abs(e[:-1, 0] * e[1:, 1] - e[:-1, 1] * e[1:, 0]) / 2.0
        cum = torch.as_tensor(np.cumsum(tri), device=dev)
        t = (u(a[0])[..., None] * cum[-1] >= cum[:-1]).sum(-1)
        q, w = torch.sqrt(u(a[1])), u(a[2])
        V = torch.as_tensor(v, device=dev)
        p = (1 - q)[..., None] * V[0] + (q * (1 - w))[..., None] * V[t + 1] \
            + (q * w)[..., None] * V[t + 2]
        x, y = p[..., 0], p[..., 1]
        area = float(tri.sum())
    su = ms[0].surface
    curv, conic = float(np.float32(su.curvature)), float(np.float32(su.conic))
    z, zx, zy = _sag(x, y, curv, conic, asph)
    n = _unit(torch.stack([-zx, -zy, torch.ones_like(zx)], -1))
    ref = torch.where((n[..., 2:].abs() > 0.9), torch.tensor([1.0, 0, 0], device=dev).double(),
                      torch.tensor([0, 0, 1.0], device=dev).double())
    t1 = _unit(torch.cross(n, ref, dim=-1))
    t2 = torch.cross(n, t1, dim=-1)
    rr, ph = torch.sqrt(-2.0 * torch.log(u(b[0], 1))), u(b[1]) * (2.0 * math.pi)
    dl = (rr * torch.cos(ph))[..., None] * t1 + (rr * torch.sin(ph))[..., None] * t2
    return torch.stack([x, y, z], -1), n, dl, n[..., 2] / area * m


def _blocked(o, d, obs):
    """Whether the ray o + t d, t > 0, meets an obstruction."""
    o, d = torch.broadcast_tensors(o, d)
    hit = torch.zeros(o.shape[:-1], dtype=torch.bool, device=o.device)
    for ob in obs:
        if isinstance(ob, ia.Box):
            lo, hi = (torch.as_tensor(np.asarray(v, np.float32), device=o.device).double()
                      for v in (ob.p1, ob.p2))
            t1, t2 = (lo - o) / (d + 1e-8), (hi - o) / (d + 1e-8)
            (ax, ay, az), (bx, by, bz) = (f(t1, t2).unbind(-1)
                                          for f in (torch.minimum, torch.maximum))
            near = torch.maximum(torch.maximum(ax, ay), az)
            far = torch.minimum(torch.minimum(bx, by), bz)
            hit |= (far >= near) & (far > 1e-8)
            continue
        p1, p2 = (np.asarray(v, np.float32).astype(np.float64) for v in (ob.p1, ob.p2))
        r, h = float(np.float32(ob.radius)), float(np.linalg.norm(p2 - p1))
        ax = torch.as_tensor((p2 - p1) / h, device=o.device)
        oc = o - torch.as_tensor(p1, device=o.device)
        da, oa = _dot(d, ax), _dot(oc, ax)
        dp, op = d - da[..., None] * ax, oc - oa[..., None] * ax
        A, B, C = _dot(dp, dp), 2.0 * _dot(op, dp), _dot(op, op) - r * r
        disc = B * B - 4.0 * A * C
        sq = torch.sqrt(disc.clamp_min(0.0))
        for t in ((-B - sq) / (2 * A + 1e-8), (-B + sq) / (2 * A + 1e-8)):
            y = oa + t * da
            hit |= (disc >= 0) & (t > 1e-8) & (y >= 0) & (y <= h)
        for t in (-oa / (da + 1e-8), (h - oa) / (da + 1e-8)):
            pt = op + t[..., None] * dp
            hit |= (t > 1e-8) & (_dot(pt, pt) <= r * r)
    return hit


def _secondary(o, d, v, asph):
    """Reflection at the Cassegrain's secondary: z = 6 m, turned by 180 deg."""
    su = _mirrors("cassegrain", False)[1].surface
    curv, conic = float(np.float32(su.curvature)), float(np.float32(su.conic))
    R = _euler(torch.tensor([180.0, 0.0, 0.0], dtype=torch.float64, device=o.device))
    pos = torch.tensor([0.0, 0.0, 6.0], dtype=torch.float64, device=o.device)
    ol, dl = (o - pos) @ R, d @ R
    with torch.no_grad():
        k1 = 1.0 + conic
        A = curv * (dl[..., 0] ** 2 + dl[..., 1] ** 2 + k1 * dl[..., 2] ** 2)
        B = 2.0 * (curv * (ol[..., 0] * dl[..., 0] + ol[..., 1] * dl[..., 1]
                           + k1 * ol[..., 2] * dl[..., 2]) - dl[..., 2])
        C = curv * (ol[..., 0] ** 2 + ol[..., 1] ** 2 + k1 * ol[..., 2] ** 2) - 2.0 * ol[..., 2]
        sq = torch.sqrt((B * B - 4 * A * C).clamp_min(0.0))
        ts = torch.stack([(-B - sq) / (2 * A + 1e-30), (-B + sq) / (2 * A + 1e-30)])
        t = torch.where(ts > 1e-8, ts, torch.inf).amin(0)

    def newton(t):
        x, y = ol[..., 0] + t * dl[..., 0], ol[..., 1] + t * dl[..., 1]
        z, zx, zy = _sag(x, y, curv, conic, asph)
        return t - (ol[..., 2] + t * dl[..., 2] - z) / (dl[..., 2] - zx * dl[..., 0]
                                                        - zy * dl[..., 1])

    with torch.no_grad():
        for _ in range(5):
            t = newton(t)
        ok = torch.isfinite(t) & (t > 1e-8)
        t = torch.where(ok, t, 0.0)
    t = torch.where(ok, newton(t), 0.0)  # one step with gradients: the root's first derivative
    x, y = ol[..., 0] + t * dl[..., 0], ol[..., 1] + t * dl[..., 1]
    z, zx, zy = _sag(x, y, curv, conic, asph)
    n = _unit(torch.stack([-zx, -zy, torch.ones_like(zx)], -1)) @ R.T
    cos = _dot(d, n)[..., None]
    ok = ok & (x * x + y * y <= 0.25)
    return torch.stack([x, y, z], -1) @ R.T + pos, d - 2.0 * cos * n, v * ok * cos[..., 0].abs()


def _axial_id(i, j, table):
    at = torch.as_tensor(table[0], device=i.device)
    n = table[1]
    ok = (i.abs() <= n) & (j.abs() <= n)
    return torch.where(ok, at[(i.clamp(-n, n) + n).long(), (j.clamp(-n, n) + n).long()], -1)


@functools.lru_cache(maxsize=None)
def _axial_table(pixels, pitch):
    xy = _hex_centres(pixels, pitch).astype(np.float64)
    j = np.rint(xy[:, 1] / (pitch * math.sqrt(3) / 2)).astype(int)
    i = np.rint(xy[:, 0] / pitch - 0.5 * j).astype(int)
    n = int(max(np.abs(i).max(), np.abs(j).max())) + 1
    t = np.full((2 * n + 1, 2 * n + 1), -1, np.int64)
    t[i + n, j + n] = np.arange(len(xy))
    return t, n


def _taps(c, x, y):
    """[(pixel, weight)] of hits (x, y): one of weight 1 unless the camera
    spreads a ray over its neighbours."""
    k, splat = _camera(c)[1], c["kind"] == "splat"
    if c["sensor"] == "square":
        x0, x1, y0, y1 = k["bounds"]
        u, v = (x - x0) / ((x1 - x0) / k["w"]), (y - y0) / ((y1 - y0) / k["h"])
        ub, vb = torch.floor(u.detach()), torch.floor(v.detach())
        offs = [(a, b) for a in range(-2, 3) for b in range(-2, 3)] if splat else [(0, 0)]

        def pix(a, b):
            i, j = ub + a, vb + b
            ok = (i >= 0) & (i < k["w"]) & (j >= 0) & (j < k["h"])
            return torch.where(ok, j * k["w"] + i, -1.0).long()

        def w(a, b):
            return torch.exp(-0.5 * ((u - ub - a) ** 2 + (v - vb - b) ** 2) / 0.7 ** 2)
    else:
        p = k["pitch"]
        v = y / (p * math.sqrt(3) / 2)
        u = x / p - 0.5 * v
        s = -u - v
        ub, vb, sb = (torch.round(t.detach()) for t in (u, v, s))
        du, dv, ds = ((a - b).abs() for a, b in ((ub, u), (vb, v), (sb, s)))
        fu = (du > dv) & (du > ds)
        fv = ~fu & (dv > ds)
        ub, vb = torch.where(fu, -vb - sb, ub), torch.where(fv, -ub - sb, vb)
        ub, vb = ub.detach(), vb.detach()
        offs = [(a, b) for a in (-1, 0, 1) for b in (-1, 0, 1) if abs(a + b) <= 1] if splat \
            else [(0, 0)]
        table = _axial_table(c["pixels"], p)

        def pix(a, b):
            return _axial_id(ub + a, vb + b, table)

        def w(a, b):
            e, f = (u - ub - a + 0.5 * (v - vb - b)).abs(), (v - vb - b).abs()
            return torch.exp(-0.5 * (torch.maximum(2 * e, e + 1.5 * f) / 0.7) ** 2)
    if not splat:
        return [(pix(0, 0), None)]
    ws = [w(a, b) for a, b in offs]
    tot = sum(ws)
    return [(pix(a, b), t / tot) for (a, b), t in zip(offs, ws)]


def _trace(c, p, n, wt, src, val, obs, asph2):
    """Rays (facets, sources, samples) to [(pixel, value)]."""
    src, val = src[None, :, None], val[None, :, None]
    p, n = p[:, None], n[:, None]
    d = src.expand(p.shape[0], -1, p.shape[2], 3) if c["distance"] == 0.0 else _unit(p - src)
    cos = _dot(d, n)
    v = val * -cos / wt[:, None]
    if obs:
        with torch.no_grad():
            lit = ~_blocked(p.detach(), -d.detach(), obs)
        v = v * lit
    r = d - 2.0 * cos[..., None] * n
    o = p
    if c["dish"] == "cassegrain":
        o, r, v = _secondary(p, r, v, asph2)
    t = (_camera(c)[0][2] - o[..., 2]) / r[..., 2]
    v = v * (t.detach() > 0)
    return [(i, v if w is None else v * w)
            for i, w in _taps(c, o[..., 0] + t * r[..., 0], o[..., 1] + t * r[..., 1])]


def _chunks(c, nf, ns):
    """(facet slice, source slice) blocks of about 2e6 rays."""
    fs = max(1, min(nf, int(2e6 / (c["samples"] * min(ns, 256)))))
    ss = max(1, min(ns, int(2e6 / (c["samples"] * fs))))
    for f in range(0, nf, fs):
        for s in range(0, ns, ss):
            yield slice(f, f + fs), slice(s, s + ss)


def _near(c, obs, pos):
    """The obstructions that can shade a facet of the block: those that come
    within the reach of rays up to the field's edge."""
    out = []
    for ob in obs:
        a, b = (np.asarray(v, float) for v in (ob.p1, ob.p2))
        e = b - a
        t = np.clip(((pos[:, None, :2] - a[:2]) * e[:2]).sum(-1) / max(e[:2] @ e[:2], 1e-9), 0, 1)
        gap = np.linalg.norm(pos[:, None, :2] - a[:2] - t[..., None] * e[:2], axis=-1).min()
        lean = max(a[2], b[2]) * math.tan(math.radians(2.0 * FIELD_DEG)) + 1.6
        if gap < lean + getattr(ob, "radius", np.linalg.norm(e[:2])):
            out.append(ob)
    return out


def _image64(c, world, src, val, obs, asph2):
    p, n, wt = world
    P, k = c["pixels"], torch.arange(512, device=p.device)
    img = torch.zeros(512 * P, dtype=torch.float64, device=p.device)  # 512 partial images
    for f, s in _chunks(c, p.shape[0], src.shape[0]):
        near = _near(c, obs, p[f].mean(1).cpu().numpy())
        for i, v in _trace(c, p[f], n[f], wt[f], src[s], val[s], near, asph2):
            i, v = i[i >= 0], v[i >= 0]
            img.index_add_(0, i + P * k.repeat(len(i) // 512 + 1)[:len(i)], v)
    return img.reshape(512, P).sum(0)


def _world(c, seed, samples, rot, pos):
    pl, nl, dl, w = samples
    R = _euler(rot)[:, None]
    nr = nl + math.radians(c["rough_arcsec"] / 3600.0) * dl if c["rough_arcsec"] else nl
    return (R @ pl[..., None])[..., 0] + pos[:, None], _unit((R @ nr[..., None])[..., 0]), w


def exact(case, seed):
    c = case
    obs = _obstructions(c)
    rays = c["facets"] * c["samples"] * c["sources"]
    grad = c["kind"] in ("grad", "splat", "fit", "aspheric")
    cost = rays * (1.0 + 0.4 * len(obs) if len(obs) < 40 else 75.0)
    if cost * (2.5 if grad and c["kind"] != "fit" else 1.0) > 1.4e10:  # some 15 seconds
        return None
    if c["kind"] == "response" and c["sources"] * c["pixels"] > 2 ** 27:
        return None
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    ms = _mirrors(c["dish"], c["round"])[:c["facets"]]
    pos = torch.stack([m.position for m in ms]).to(dev).double()
    rot = torch.stack([m.rotation for m in ms]).to(dev)
    rot[:, :2] += torch.as_tensor(_tilts(c, seed, len(ms)), dtype=torch.float32, device=dev)
    rot = rot.double()
    a0 = [float(np.float32(x)) for x in ms[0].surface.aspheric]
    a0 = torch.tensor(a0, dtype=torch.float64, device=dev)
    a1 = torch.zeros(2, dtype=torch.float64, device=dev)

    def field(sd, n):
        s, v = _sources(c, sd, n)
        return torch.as_tensor(s, device=dev).double(), torch.as_tensor(v, device=dev).double()

    if c["kind"] == "fit":
        samples = _exact_samples(c, seed, dev, a0)
        imgs = []
        for i, n in enumerate(_sizes(c, seed)):
            ri = rot.float()
            ri[:, :2] += torch.as_tensor(_tilts(c, seed + 100 + i, len(ms)), dtype=torch.float32,
                                         device=dev)
            s, v = field(seed + 31 * i, n)
            imgs.append(_image64(c, _world(c, seed, samples, ri.double(), pos), s, v, obs, a1))
        return {"images": torch.stack(imgs), "rotations": None, "exp_avg": None}
    src, val = field(seed, c["sources"])
    samples = _exact_samples(c, seed, dev, a0)
    world = _world(c, seed, samples, rot, pos)
    if c["kind"] == "response":
        P = c["pixels"]
        out = torch.zeros(c["sources"] * P, dtype=torch.float64, device=dev)
        for f, s in _chunks(c, len(ms), c["sources"]):
            near = _near(c, obs, world[0][f].mean(1).cpu().numpy())
            row = torch.arange(s.start, min(s.stop, c["sources"]), device=dev)[None, :, None]
            for i, v in _trace(c, *(x[f] for x in world), src[s], val[s], near, a1):
                out.index_add_(0, (row * P + i)[i >= 0], v[i >= 0])
        return out.reshape(c["sources"], P)
    img = _image64(c, world, src, val, obs, a1)
    if not grad:
        if c["sensor"] == "square":
            k = _camera(c)[1]
            return img.reshape(k["h"], k["w"])
        return img
    cot = torch.as_tensor(_cotangent(c, seed), device=dev).double()
    if c["kind"] == "aspheric":
        wrt = {"primary": a0.requires_grad_(True), "secondary": a1.requires_grad_(True)}
    else:
        wrt = {"rotations": rot.requires_grad_(True), "positions": pos.requires_grad_(True),
               "values": val.requires_grad_(True)}
    total = {k: torch.zeros_like(v) for k, v in wrt.items()}
    for f, s in _chunks(c, len(ms), c["sources"]):
        if c["kind"] == "aspheric":
            samples = _exact_samples(c, seed, dev, a0)
        part = tuple(x[f] for x in samples)
        w = _world(c, seed, part, rot[f], pos[f])
        near = _near(c, obs, w[0].detach().mean(1).cpu().numpy())
        loss = sum((cot[i.clamp_min(0)] * (i >= 0) * v).sum()
                   for i, v in _trace(c, *w, src[s], val[s], near, a1))
        for k, g in zip(wrt, torch.autograd.grad(loss, list(wrt.values()), allow_unused=True)):
            if g is not None:  # (parallel light does not depend on the positions)
                total[k] += g
    if c["sensor"] == "square":
        k = _camera(c)[1]
        img = img.reshape(k["h"], k["w"])
    return {"image": img.detach(), **total}
