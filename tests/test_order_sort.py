"""The coherence sort on either side of 2^16 rays, where it changes from a merge
sort to a radix sort: every ray has the same bits sorted and in input order,
and the gradient of rays sorted by group the same sums to the rounding of their
order (1e-12 of the largest, as in the other comparison of the two orders)."""
import math

import numpy as np
import pytest

from robast_amd import _abi as A
from robast_amd import configs

FLOATS = ("x", "y", "z", "t", "dx", "dy", "dz", "lambda_")


@pytest.mark.gpu
@pytest.mark.parametrize("n", ((1 << 16) - 1, 1 << 16, (1 << 16) + 1, 100003))
def test_order_does_not_change_results(ctx, n):
    import torch
    from robast_amd._lib import make_rays_device
    mgr = configs.c3_scene()
    scene = ctx.upload(mgr.flat())
    out = {}
    for order in (A.RB_ORDER_INPUT, A.RB_ORDER_COHERENT):
        t = {f: torch.empty(n, dtype=torch.float64, device="cuda") for f in FLOATS}
        t.update({f: torch.empty(n, dtype=torch.int32, device="cuda") for f in ("status", "npoints", "last_node")})
        ctx.generate(configs.c3_raygen(), make_rays_device(t), n)
        ctx.trace(scene, make_rays_device(t), n, mgr.trace_opts(device_ptrs=1, order=order))
        out[order] = t
    for f in out[A.RB_ORDER_INPUT]:
        assert torch.equal(out[A.RB_ORDER_INPUT][f], out[A.RB_ORDER_COHERENT][f]), f


@pytest.mark.gpu
@pytest.mark.parametrize("n", (21845, 21846, 33333))
def test_groups_on_either_side(ctx, n):
    import torch
    from robast_amd import alignment as AL
    from robast_amd._lib import make_rays_device
    angles = (0.0, 2.0, 3.5)
    model = AL.DaviesCottonAlignment(ctx, angles_deg=angles, rays_per_angle=n)
    model.set_params(AL.c5_initial_params())
    P, G = model.n_params, len(angles)
    ref = torch.tensor([[1600.0 * math.tan(math.radians(a)), 0.0] for a in angles], dtype=torch.float64, device="cuda")
    got = []
    for order in (A.RB_ORDER_INPUT, A.RB_ORDER_COHERENT):
        acc = torch.zeros((G, 3 * P + 4), dtype=torch.float64, device="cuda")
        d = AL.adjoint_desc(model.node_param, model.values, P, model.z_param, model.focal_node, 0.0, 0.0, 0.0,
                            A.RB_ADJ_MOMENTS)
        d.ref_xy, d.group_size, d.n_groups = ref.data_ptr(), n, G
        o = model._opts()
        o.order = order
        ctx.adjoint(model.scene, make_rays_device(model.all), G * n, o, d, acc.data_ptr())
        got.append(acc.cpu().numpy())
    assert np.array_equal(got[0][:, 3 * P], got[1][:, 3 * P])
    assert np.abs(got[0] - got[1]).max() <= 1e-12 * np.abs(got[0]).max()
