"""What sorted rays alone go through: the wavefront navigation's boolean
operations and focal efficiencies, and its reverse pass in every mode.

Scenes of unions, intersections and differences, as mirrors and as plain
components that rays cross, with turned and unturned operands, and a focal
surface whose efficiency depends on the angle of incidence: on the CPU (one
ray a wavefront, under sanitizers) against the oracle, on the GPU against the
lane form in input order, bit for bit, as every operation rounds alike in both.
The gradients of sorted rays against the dual-number reference, with the bars
of the unsorted forms' own comparisons."""
import math

import numpy as np
import pytest

from helpers import copy_soa
from oracle import oracle as O
from robast_amd import (AFocalSurface, AMirror, AOpticalComponent, AOpticsManager, TGeoBBox, TGeoCombiTrans,
                        TGeoCompositeShape, TGeoParaboloid, TGeoPgon, TGeoRotation, TGeoSphere, TGeoTranslation,
                        TGeoTube)
from robast_amd import _abi as A
from robast_amd.materials import TGraph
from test_emulation import emul_trace
from test_wave_navigation import F64, I32, emul_wave  # noqa: F401 (a fixture)

OPERANDS = ("box", "tube", "sphere", "cap", "paraboloid", "pgon")


def _operand(kind, name):
    if kind == "box":
        TGeoBBox(name, 9, 7, 6, (0.5, -0.3, 0.2))
    elif kind == "tube":
        TGeoTube(name, 2, 9, 7)
    elif kind == "sphere":
        TGeoSphere(name, 0, 9, 0, 180)
    elif kind == "cap":
        TGeoSphere(name, 5, 11, 20, 140)
    elif kind == "paraboloid":
        TGeoParaboloid(name, 1, 10, 7)
    else:
        p = TGeoPgon(name, 10, 360, 6, 2)
        p.DefineSection(0, -6, 0, 8)
        p.DefineSection(1, 7, 0, 9)


def boolean_scene(op):
    """36 composites `left op right` of all pairs of operand shapes, half of
    them half-reflecting mirrors, the others plain; the right operand is
    shifted, every second one turned as well, every third composite too."""
    mgr = AOpticsManager("manager", "booleans")
    world = AOpticalComponent("world", TGeoBBox("w", 400, 400, 400))
    mgr.SetTopVolume(world)
    rng = np.random.default_rng(11)
    for k in range(36):
        left, right = OPERANDS[k // 6], OPERANDS[k % 6]
        _operand(left, f"l{k}")
        _operand(right, f"r{k}")
        shift = rng.uniform(-4, 4, 3)
        if k % 2:
            turn = TGeoRotation("", *(float(v) for v in rng.uniform(0, 180, 3)))
            TGeoCombiTrans(f"m{k}", *(float(v) for v in shift), turn).RegisterYourself()
        else:
            TGeoTranslation(f"m{k}", *(float(v) for v in shift)).RegisterYourself()
        shape = TGeoCompositeShape(f"c{k}", f"l{k} {op} r{k}:m{k}")
        if k % 4 < 2:
            vol = AMirror(f"v{k}", shape)
            vol.SetReflectance(0.5)
        else:
            vol = AOpticalComponent(f"v{k}", shape)
        at = (35.0 * (k % 6) - 87.5, 35.0 * (k // 6) - 87.5, 12.0 * (k % 5) - 24.0)
        world.AddNode(vol, 1, TGeoCombiTrans(*at, TGeoRotation("", 20.0 * k, 10.0 * k, 0.0)) if k % 3 == 0
                      else TGeoTranslation(*at))
    mgr.CloseGeometry()
    return mgr


def boolean_rays(n):
    rng = np.random.default_rng(n)
    soa = O.new_soa(n)
    soa["x"][:], soa["y"][:] = rng.uniform(-110, 110, n), rng.uniform(-110, 110, n)
    soa["z"][:] = rng.uniform(-80, 80, n)  # some start inside a shape
    d = rng.normal(0, 1, (n, 3))
    d /= np.sqrt((d * d).sum(1))[:, None]
    soa["dx"][:], soa["dy"][:], soa["dz"][:] = d.T
    soa["lambda_"][:] = 400e-7
    return soa


def angular_scene():
    """Twenty focal tiles facing up whose efficiency falls with the angle of
    incidence and with the wavelength, one of them turned."""
    mgr = AOpticsManager("manager", "angular")
    world = AOpticalComponent("world", TGeoBBox("w", 400, 400, 400))
    mgr.SetTopVolume(world)
    tile = AFocalSurface("tile", TGeoBBox("t", 20, 24, 1))
    g = TGraph()
    g.SetPoint(0, 0.0, 0.2)
    g.SetPoint(1, math.pi / 2, 0.4)
    g.SetPoint(2, math.pi, 0.9)
    tile.SetQuantumEfficiencyAngle(g)
    w = TGraph()
    w.SetPoint(0, 300e-7, 0.5)
    w.SetPoint(1, 600e-7, 1.0)
    tile.SetQuantumEfficiency(w)
    for k in range(20):
        at = (45.0 * (k % 5) - 90.0, 50.0 * (k // 5) - 75.0, 3.0 * k)
        world.AddNode(tile, k + 1, TGeoCombiTrans(*at, TGeoRotation("", 0, 15, 0)) if k == 7 else TGeoTranslation(*at))
    mgr.CloseGeometry()
    return mgr


def angular_rays(n):
    soa = boolean_rays(n)
    soa["z"][:] += 200.0
    soa["dz"][:] = -np.abs(soa["dz"]) - 1.0
    norm = np.sqrt(soa["dx"] ** 2 + soa["dy"] ** 2 + soa["dz"] ** 2)
    for f in ("dx", "dy", "dz"):
        soa[f] /= norm
    soa["lambda_"][:] = np.random.default_rng(n + 1).uniform(300e-7, 600e-7, n)
    return soa


SCENES = {"union": (lambda: boolean_scene("+"), boolean_rays),
          "difference": (lambda: boolean_scene("-"), boolean_rays),
          "intersection": (lambda: boolean_scene("*"), boolean_rays),
          "angular": (angular_scene, angular_rays)}


@pytest.mark.parametrize("name", SCENES)
def test_wave_form_under_sanitizers_matches_oracle(emul_wave, tmp_path, name):  # noqa: F811
    """Integers equal, points within 1e-7 cm (the bar of the other per-ray
    comparisons)."""
    scene, rays = SCENES[name]
    mgr = scene()
    src = rays(2500)
    e, o = copy_soa(src), copy_soa(src)
    emul_trace(emul_wave, mgr.flat(), e, mgr.trace_opts(), str(tmp_path))
    O.trace(mgr.flat(), o, mgr.trace_opts(), nthreads=4)
    met = o["npoints"] > 2 if name != "angular" else o["status"] == A.RB_FOCUS
    assert met.sum() > 100
    for f in I32:
        assert np.array_equal(e[f], o[f]), f
    for f in ("x", "y", "z"):
        assert np.abs(e[f] - o[f]).max() <= 1e-7, f


@pytest.mark.gpu
@pytest.mark.parametrize("name", SCENES)
@pytest.mark.parametrize("n", (1, 65, 40000))
def test_sorted_rays_equal_rays_in_input_order(ctx, name, n):
    from robast_amd._lib import make_rays
    scene, rays = SCENES[name]
    mgr = scene()
    src = rays(n)
    up = ctx.upload(mgr.flat())
    out = []
    for order in (A.RB_ORDER_INPUT, A.RB_ORDER_COHERENT):
        soa = copy_soa(src)
        ctx.trace(up, make_rays(soa), n, mgr.trace_opts(order=order))
        out.append(soa)
    for f in F64 + I32:
        assert np.array_equal(out[0][f], out[1][f]), f


def _sorted_only(model):
    """The model's launches from here on trace their rays sorted."""
    plain = model.mgr.trace_opts
    model.mgr.trace_opts = lambda **k: plain(**{**k, "order": A.RB_ORDER_COHERENT})


@pytest.mark.gpu
def test_sorted_alignment_gradient_matches_dual(ctx):
    """8 angles x 25k rays, 1e-5 relative per parameter, as the unsorted form."""
    import test_c5_adjoint as T5
    from robast_amd import alignment as AL
    model = AL.DaviesCottonAlignment(ctx, rays_per_angle=25000)
    p0 = AL.c5_initial_params()
    model.loss(p0)
    _sorted_only(model)
    g = model.gradient()
    assert ctx.last_trace_launches() == 3  # key, sort, adjoint
    srcs = [{k: v.cpu().numpy().copy() for k, v in s.items()} for s in model.src]
    gd, _ = T5._dual_grad(p0, srcs, model.stats)
    nz = gd != 0
    assert np.array_equal(g != 0, nz)
    assert (np.abs(g - gd)[nz] / np.abs(gd[nz])).max() <= 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("loss", ["spot", "ee"])
def test_sorted_figure_gradient_matches_dual(ctx, loss):
    """2 angles x 20k rays, 1e-6 relative per parameter, as the unsorted form."""
    import test_aspheric_adjoint as TA
    model = TA._gpu_model(ctx, 20000, loss)
    p0 = TA.F.figure_params()
    L = model.loss(p0)
    _sorted_only(model)
    g = model.gradient()
    assert ctx.last_trace_launches() == 3
    srcs = [{k: v.cpu().numpy().copy() for k, v in s.items()} for s in model.src]
    if loss == "spot":
        per = [(A.RB_ADJ_CENTROID, cx, cy, 2.0 / n, 0.0, 0.0) for n, cx, cy in model.stats]
    else:
        per = [(A.RB_ADJ_ENCIRCLED, tx, ty, -1.0 / n, 15.0, 2.0) for (n, _, _), (tx, ty) in
               zip(model.stats, model.targets)]
        assert model.last_adjoint_loss == pytest.approx(L, rel=1e-9)
    gd, used = TA._dual(p0, srcs, per)
    assert used == sum(n for n, _, _ in model.stats)
    assert (np.abs(g - gd) / np.abs(gd)).max() <= 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("n", (1, 64, 1001, 30000))
def test_sorted_encircled_energy_of_facets(ctx, n):
    """The encircled-energy mode on spherical facets: the loss, behind the
    parameters, and the gradient of sorted and unsorted rays are the same sum
    of per-ray terms, so equal to the rounding of a sum of n terms (1e-12 of
    the largest, as for the moments), and within the FP32 chain's 1e-4 of the
    largest component of the dual reference."""
    import torch
    import test_c5_adjoint as T5
    from robast_amd import alignment as AL
    from robast_amd._lib import make_rays_device
    model = AL.DaviesCottonAlignment(ctx, angles_deg=(1.5,), rays_per_angle=n)
    p0 = AL.c5_initial_params()
    model.set_params(p0)
    P = model.n_params
    cx = 1600.0 * math.tan(math.radians(1.5))
    got = []
    for order in (A.RB_ORDER_INPUT, A.RB_ORDER_COHERENT):
        acc = torch.zeros(P + 1, dtype=torch.float64, device="cuda")
        d = AL.adjoint_desc(model.node_param, model.values, P, model.z_param, model.focal_node, cx, 0.0, -1.0 / n,
                            A.RB_ADJ_ENCIRCLED)
        d.ee_radius, d.ee_width = 3.0, 1.0
        o = model._opts()
        o.order = order
        ctx.adjoint(model.scene, make_rays_device(model.all), n, o, d, acc.data_ptr())
        got.append(acc.cpu().numpy())
    assert np.abs(got[0] - got[1]).max() <= 1e-12 * np.abs(got[0]).max()
    if n == 30000:
        assert -1.0 < got[1][P] < 0.0
        src = {k: v.cpu().numpy().copy() for k, v in model.all.items()}
        flat = AL.c5_scene(p0).flat()
        table, focal = AL.node_param_table(flat)
        h = T5._host_desc(table, np.ascontiguousarray(p0, dtype=float), focal, cx, 0.0, -1.0 / n)
        h.mode, h.ee_radius, h.ee_width = A.RB_ADJ_ENCIRCLED, 3.0, 1.0
        gd, _ = O.adjoint_dual(flat, src, model.mgr.trace_opts(), h, P)
        assert np.abs(got[1][:P] - gd).max() <= 1e-4 * np.abs(gd).max()
