"""Scenes with many shapes of one structure, such as facets measured one by one.

Where the lanes of a wavefront name several of them, each lane reads its own
shape; a lane alone in its wavefront reads it the way all lanes of one shape do.
Every ray must have the same bits both ways, in every kernel form: primitives,
iterative solvers, two-level composites and general polycones, lenses, rough
surfaces, FP64 and mixed, and in the schedules that hand rays to other lanes."""
import numpy as np
import pytest

from helpers import copy_soa
from robast_amd import _abi as A
from robast_amd import geometry as G
from robast_amd.manager import AOpticsManager
from robast_amd.materials import ARefractiveIndex

F64 = ("x", "y", "z", "t", "dx", "dy", "dz", "lambda_")
I32 = ("status", "npoints", "last_node")
EACH = 12  # members of a family


def _shape(kind, k):
    s = 1.0 + 0.02 * k
    n = f"{kind}{k}"
    if kind == "box":
        return G.TGeoBBox(n, 7 * s, 6 * s, 5 * s)
    if kind == "tube":
        return G.TGeoTube(n, 2 * s, 8 * s, 5 * s)
    if kind == "sphere":
        return G.TGeoSphere(n, 0, 8 * s, 0, 180)
    if kind == "pgon":
        p = G.TGeoPgon(n, 3.0 * k, 360, 6, 2)
        p.DefineSection(0, -5, 0, 6 * s)
        p.DefineSection(1, 5, 0, 8 * s)
        return p
    if kind == "cap":
        G.TGeoSphere(n + "s", 20 * s, 20 * s + 1, 140, 180)
        G.TGeoBBox(n + "b", 7, 7, 30)
        G.TGeoTranslation(n + "t", 0, 0, 18).RegisterYourself()
        return G.TGeoCompositeShape(n, f"{n}s:{n}t*{n}b")
    if kind == "disk":
        d = G.AGeoAsphericDisk(n, -2.0, 0.01 * s, 1.0, -0.01 * s, 8.0, 0.0)
        d.SetPolynomials(2, [1e-4 * s, 1e-7], 2, [1e-4, 2e-7 * s])
        return d
    if kind == "winston":
        return G.AGeoWinstonConePoly(n, 7 * s, 4 * s, 6)
    if kind == "nested":
        G.TGeoBBox(n + "a", 8 * s, 8 * s, 6)
        G.TGeoTube(n + "c", 0, 3 * s, 9)
        G.TGeoSphere(n + "d", 0, 9 * s, 0, 180)
        return G.TGeoCompositeShape(n, f"({n}a-{n}c)*{n}d")
    assert kind == "pcon"
    p = G.TGeoPcon(n, 0, 360, 3)
    p.DefineSection(0, -6, 1, 4 * s)
    p.DefineSection(1, 0, 2, 8 * s)
    p.DefineSection(2, 6, 1, 3 * s)
    return p


SCENES = {"plain": (("box", "tube", "sphere", "pgon", "cap"), "mirror"),
          "solver": (("disk", "winston", "sphere", "cap"), "mirror"),
          "deep": (("nested", "pcon", "box", "cap"), "mirror"),
          "rough": (("box", "sphere", "cap"), "rough"),
          "lens": (("sphere", "cap", "box"), "lens"),
          "deep_lens": (("nested", "sphere", "pcon"), "lens")}


def family_scene(name):
    """Every shape once, half of them half-reflecting mirrors (rough ones) or
    lenses, the others plain, on a grid in mixed order."""
    kinds, what = SCENES[name]
    mgr = AOpticsManager("manager", "families")
    world = G.AOpticalComponent("world", G.TGeoBBox("w", 300, 300, 300))
    mgr.SetTopVolume(world)
    glass = ARefractiveIndex(1.5)
    for k in range(EACH * len(kinds)):
        shape = _shape(kinds[k % len(kinds)], k // len(kinds))
        if (k // len(kinds)) % 2:
            vol = G.AOpticalComponent(f"v{k}", shape)
        elif what == "lens":
            vol = G.ALens(f"v{k}", shape)
            vol.SetRefractiveIndex(glass)
        else:
            vol = G.AMirror(f"v{k}", shape)
            vol.SetReflectance(0.4 + 0.01 * k)
        at = (32.0 * (k % 4) - 48, 32.0 * (k // 4 % 4) - 48, 32.0 * (k // 16) - 48)
        world.AddNode(vol, 1, G.TGeoCombiTrans(*at, G.TGeoRotation("", 15.0 * k, 7.0 * k, 0)))
        if what == "rough" and isinstance(vol, G.AMirror):
            G.ABorderSurfaceCondition(world, vol).SetGaussianRoughness(0.02)
    mgr.CloseGeometry()
    return mgr


def family_rays(n):
    from oracle import oracle as O
    rng = np.random.default_rng(n)
    soa = O.new_soa(n)
    for f in ("x", "y", "z"):
        soa[f][:] = rng.uniform(-70, 70, n)
    d = rng.normal(0, 1, (n, 3))
    d /= np.sqrt((d * d).sum(1))[:, None]
    soa["dx"][:], soa["dy"][:], soa["dz"][:] = d.T
    soa["lambda_"][:] = 400e-7
    return soa


def _trace(ctx, up, mgr, soa, precision, **opts):
    from robast_amd._lib import make_rays
    o = mgr.trace_opts(order=A.RB_ORDER_INPUT, **opts)
    o.precision = precision
    ctx.trace(up, make_rays(soa), len(soa["x"]), o)
    return soa


@pytest.mark.gpu
@pytest.mark.parametrize("precision", (A.RB_PRECISION_FP64, A.RB_PRECISION_MIXED))
@pytest.mark.parametrize("name", SCENES)
def test_lanes_together_equal_lanes_alone(ctx, name, precision):
    print(f"families {name} {precision}", flush=True)
    n = 2048 + 33
    mgr = family_scene(name)
    up = ctx.upload(mgr.flat())
    src = family_rays(n)
    got = _trace(ctx, up, mgr, copy_soa(src), precision, schedule=A.RB_SCHEDULE_LANE)
    assert (got["npoints"] > 3).sum() > 100
    for lane in range(64):
        alone = copy_soa(src)
        others = np.arange(n) % 64 != lane
        alone["status"][others] = A.RB_STOP
        _trace(ctx, up, mgr, alone, precision, schedule=A.RB_SCHEDULE_LANE)
        for f in F64 + I32:
            assert np.array_equal(alone[f][~others], got[f][~others]), (lane, f)


@pytest.mark.gpu
@pytest.mark.parametrize("schedule", (A.RB_SCHEDULE_PERSISTENT, A.RB_SCHEDULE_REGROUP))
@pytest.mark.parametrize("precision", (A.RB_PRECISION_FP64, A.RB_PRECISION_MIXED))
@pytest.mark.parametrize("name", SCENES)
def test_queue_schedules_equal_lanes(ctx, name, precision, schedule):
    print(f"families {name} {precision} schedule {schedule}", flush=True)
    mgr = family_scene(name)
    up = ctx.upload(mgr.flat())
    src = family_rays(5000)
    want = _trace(ctx, up, mgr, copy_soa(src), precision, schedule=A.RB_SCHEDULE_LANE)
    got = _trace(ctx, up, mgr, copy_soa(src), precision, schedule=schedule)
    for f in F64 + I32:
        assert np.array_equal(got[f], want[f]), f


@pytest.mark.gpu
@pytest.mark.parametrize("name", ("plain", "solver", "rough"))
def test_sorted_wavefronts_equal_lanes(ctx, name):
    from robast_amd._lib import make_rays
    mgr = family_scene(name)
    up = ctx.upload(mgr.flat())
    src = family_rays(20000)
    want = _trace(ctx, up, mgr, copy_soa(src), A.RB_PRECISION_FP64)
    got = copy_soa(src)
    ctx.trace(up, make_rays(got), 20000, mgr.trace_opts(order=A.RB_ORDER_COHERENT))
    for f in F64 + I32:
        assert np.array_equal(got[f], want[f]), f


@pytest.mark.gpu
def test_own_shapes_do_not_take_turns(ctx):
    """Rays in random order on 85 facets with a shape each: a turn for every
    shape of a wavefront (some 45) took 7 times as long as one shape for all."""
    import torch
    from robast_amd import configs
    from robast_amd._lib import make_rays_device
    n = 20000
    t = {f: torch.empty(n, dtype=torch.float64, device="cuda") for f in F64}
    t.update({f: torch.empty(n, dtype=torch.int32, device="cuda") for f in I32})
    ctx.generate(configs.c2_raygen(), make_rays_device(t), n)
    ms = []
    for own in (False, True):
        radii = [configs.C2_MIRROR_R + 0.1 * k for k in range(configs.C2_NFACETS)] if own else None
        mgr = configs.c2_scene(per_facet=own, facet_radius=radii)
        up = ctx.upload(mgr.flat())
        runs = []
        for _ in range(9):
            w = {k: v.clone() for k, v in t.items()}
            ctx.trace(up, make_rays_device(w), n, mgr.trace_opts(device_ptrs=1, order=A.RB_ORDER_INPUT))
            runs.append(ctx.last_kernel_ms())
        ms.append(sorted(runs)[4])
    print(f"shared {ms[0] * 1e3:.0f} us, own {ms[1] * 1e3:.0f} us", flush=True)
    assert ms[1] < 3 * ms[0], ms
