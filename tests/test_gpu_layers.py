"""Layered kernels (several layers a thread, columns in registers) at the layer
counts where a group of layers or the register column ends, against the oracle's
routine or, for the remapping, against one call per layer: the same sums in the
same order, so equal up to a few ulps of the largest term (1e-13, as the operator
tests) or bit for bit."""
import dataclasses

import numpy as np
import pytest

from ufemism_amd import abi, geometry
from ufemism_amd.dynamics import Step, initial_fields

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
LAYERS = (1, 2, 4, 5, 6, 10, 33)


def _oracle():
    from oracle import pyoracle
    return pyoracle


def _dev(a):
    t = torch.from_numpy(np.ascontiguousarray(a, np.float64)).cuda()
    torch.cuda.synchronize()
    return t


@pytest.fixture(scope="module", params=[60, 1021])
def pair(request, ctx):
    print(f"[layers] dome {request.param}", flush=True)
    wl = geometry.dome(request.param, seed=3, picard=1)
    Step(ctx, wl)
    return wl, _oracle().OracleMesh(wl.mesh).build()


@pytest.mark.parametrize("nz", LAYERS)
def test_layered_operators_match_oracle(ctx, pair, nz):
    wl, om = pair
    rng = np.random.default_rng(nz)
    nV, nAc = wl.mesh.nV, om.nAc
    for name, po_name, n_in, n_out in (("derivatives_Aa_3D", "get_mesh_derivatives_3D", nV, (nV, nV)),
                                       ("map_Aa_to_Ac_3D", "map_Aa_to_Ac_3D", nV, (nAc,)),
                                       ("map_Ac_to_Aa_3D", "map_Ac_to_Aa_3D", nAc, (nV,)),
                                       ("neumann_Aa_3D", "apply_Neumann_boundary_3D", nV, ())):
        h = rng.standard_normal(n_in * nz)
        d = _dev(h)
        outs = [_dev(np.full(n * nz, np.nan)) for n in n_out]
        ctx.op(name, d.data_ptr(), *(t.data_ptr() for t in outs), nz=nz)
        houts = [np.full(n * nz, np.nan) for n in n_out]
        _oracle().op(po_name, om, h, *houts, nz=nz)
        for g, o in zip(outs or [d], houts or [h]):
            g = g.cpu().numpy()
            assert np.abs(g - o).max() <= 1e-13 * np.abs(o).max(), (name, nz)


@pytest.mark.parametrize("nz", LAYERS)
def test_layered_upwind_equals_one_layer_at_a_time(ctx, pair, nz):
    """Layers with and without flow side by side; the missing points add up."""
    wl, _ = pair
    nV = wl.mesh.nV
    rng = np.random.default_rng(nz)
    u, v, d = (rng.standard_normal((nz, nV)) for _ in range(3))
    u[:, ::7] = v[:, ::7] = 0.0
    u[::2, 3::5] = v[::2, 3::5] = 1e-11
    D = [_dev(a.ravel()) for a in (u, v, d)]
    out = [_dev(np.full(nV * nz, np.nan)) for _ in range(2)]
    missing = ctx.upwind_derivatives_3D(*(t.data_ptr() for t in D + out), nz)
    one = 0
    for k in range(nz):
        L = [_dev(a[k]) for a in (u, v, d)]
        o = [_dev(np.full(nV, np.nan)) for _ in range(2)]
        one += ctx.upwind_derivatives_3D(*(t.data_ptr() for t in L + o), 1)
        for a, b in zip(out, o):
            assert torch.equal(a[k * nV:(k + 1) * nV], b), k
    assert missing == one


def test_remap_layers_and_growing_workspace():
    """One remapping with few layers, then more, then few again (the kept space
    of the second-order method grows once)."""
    wa, wb = geometry.dome(300, seed=3), geometry.dome(411, seed=4)
    ca, cb = abi.Context(0), abi.Context(0)
    try:
        ma, mb = ca.mesh_build(wa.mesh), cb.mesh_build(wb.mesh)
        for c, wl, m in ((ca, wa, ma), (cb, wb, mb)):
            c.set_params(wl.params)
            c.mesh_upload(m)
        cb.remap_build(ca, ma, mb)
        rng = np.random.default_rng(1)
        for nz in (1, 6, 11, 5):
            h = rng.standard_normal((nz, wa.mesh.nV))
            d = _dev(h.ravel())
            for method in abi.REMAP_METHODS:
                out = _dev(np.full(nz * wb.mesh.nV, np.nan))
                cb.remap_field(ca, method, d.data_ptr(), out.data_ptr(), nz)
                for k in range(nz):
                    one = _dev(np.full(wb.mesh.nV, np.nan))
                    cb.remap_field(ca, method, _dev(h[k]).data_ptr(), one.data_ptr(), 1)
                    assert torch.equal(out.view(nz, -1)[k], one), (method, nz, k)
    finally:
        ca.close()
        cb.close()


@pytest.mark.parametrize("nz", [2, 3, 15, 16, 17, 32])
def test_columns_of_every_depth_match_oracle(nz):
    """SIA, 3-D velocities and the general update on both column kernels."""
    print(f"[layers] columns nz {nz}", flush=True)
    wl = geometry.marine(1500, seed=5, picard=1)
    wl = dataclasses.replace(wl, params=dataclasses.replace(wl.params, zeta=np.linspace(0.0, 1.0, nz) ** 1.5))
    po = _oracle()
    om = po.OracleMesh(wl.mesh, nZ=nz).build()
    ice = po.OracleIce(om)
    ctx = abi.Context(0)
    try:
        ctx.set_params(wl.params)
        ctx.mesh_upload(ctx.mesh_build(wl.mesh))
        fields = initial_fields(wl, om["VAaAc"], nz)
        fields["A_flow"] = fields["A_flow"] * np.linspace(0.5, 2.0, nz)
        fields["A_flow_Ac"] = np.full((om.nAc, nz), wl.A_flow) * np.linspace(0.5, 2.0, nz)
        for k, v in fields.items():
            ctx.set(k, v)
            if k in ice.arr:
                ice[k][...] = v
        for c in (ctx, ice):
            c.update_general_ice_model_data()
        ctx.solve_SIA()
        ctx.solve_SIA_3D()
        ice.solve_SIA(wl.params)
        ice.solve_SIA_3D(wl.params)
        for k in ("mask", "mask_Ac", "mask_gl", "mask_gl_Ac", "mask_margin", "mask_cf_Ac", "mask_coast"):
            assert np.array_equal(ctx.get(k), ice[k]), k
        for k in ("Hs", "Hs_Ac", "dHs_dx", "dHi_dy", "dHs_do_Ac", "dSL_dp_Ac", "dHs_dx_shelf", "dHs_dy_shelf_Ac",
                  "D_SIA_3D_Ac", "D_SIA", "U_SIA", "V_SIA", "U_3D", "V_3D", "W_3D"):
            g, o = ctx.get(k), ice[k]
            assert np.linalg.norm(g - o) <= 1e-10 * np.linalg.norm(o), (k, nz)
    finally:
        ctx.close()
