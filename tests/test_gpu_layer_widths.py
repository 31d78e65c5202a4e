"""Layered kernels with several layers a thread (fields of many values) against
one call per layer (a thread per value): the same sums in the same order, so the
same bits.  The layer counts leave last groups of every length."""
import numpy as np
import pytest

from ufemism_amd import abi, geometry
from ufemism_amd.dynamics import Step

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
NZ = (200, 201, 202, 203, 204)       # of 1,021 vertices: above the 200,000 values from which groups of layers are taken


def _dev(a):
    t = torch.from_numpy(np.ascontiguousarray(a, np.float64)).cuda()
    torch.cuda.synchronize()
    return t


def _layer(t, nz, k):
    one = t.view(nz, -1)[k].clone()
    torch.cuda.synchronize()
    return one


@pytest.mark.parametrize("nz", NZ)
def test_operators(ctx, nz):
    print(f"[layer widths] operators nz {nz}", flush=True)
    wl = geometry.dome(1021, seed=3, picard=1)
    s = Step(ctx, wl)
    nV, nAc = wl.mesh.nV, ctx.sizes["nAc"]
    assert nV * nz > 200000
    rng = np.random.default_rng(nz)
    for name, n_in, n_out in (("derivatives_Aa_3D", nV, (nV, nV)), ("map_Aa_to_Ac_3D", nV, (nAc,)),
                              ("map_Ac_to_Aa_3D", nAc, (nV,)), ("neumann_Aa_3D", nV, ())):
        d = _dev(rng.standard_normal(n_in * nz))
        outs = [_dev(np.full(n * nz, np.nan)) for n in n_out]
        before = d.clone()
        torch.cuda.synchronize()
        ctx.op(name, d.data_ptr(), *(t.data_ptr() for t in outs), nz=nz)
        for k in (0, 1, 4, 5, nz - 5, nz - 2, nz - 1):
            x = _layer(before, nz, k)
            one = [_dev(np.full(n, np.nan)) for n in n_out]
            ctx.op(name, x.data_ptr(), *(t.data_ptr() for t in one), nz=1)
            for a, b in zip(outs or [d], one or [x]):
                assert torch.equal(a.view(nz, -1)[k], b), (name, nz, k)
    u, v, d = (rng.standard_normal((nz, nV)) for _ in range(3))
    u[:, ::7] = v[:, ::7] = 0.0
    u[::2, 3::5] = v[::2, 3::5] = 1e-11
    D = [_dev(a.ravel()) for a in (u, v, d)]
    out = [_dev(np.full(nV * nz, np.nan)) for _ in range(2)]
    missing = ctx.upwind_derivatives_3D(*(t.data_ptr() for t in D + out), nz)
    one_by_one = 0
    for k in range(nz):
        o = [_dev(np.full(nV, np.nan)) for _ in range(2)]
        x = [_layer(t, nz, k) for t in D]
        one_by_one += ctx.upwind_derivatives_3D(*(t.data_ptr() for t in x + o), 1)
        for a, b in zip(out, o):
            assert torch.equal(a.view(nz, -1)[k], b), k
    assert missing == one_by_one
    del s


def test_remapping():
    print("[layer widths] remapping", flush=True)
    wa, wb = geometry.dome(700, seed=3), geometry.dome(1021, seed=4)
    ca, cb = abi.Context(0), abi.Context(0)
    try:
        ma, mb = ca.mesh_build(wa.mesh), cb.mesh_build(wb.mesh)
        for c, wl, m in ((ca, wa, ma), (cb, wb, mb)):
            c.set_params(wl.params)
            c.mesh_upload(m)
        cb.remap_build(ca, ma, mb)
        rng = np.random.default_rng(1)
        for nz in NZ:
            d = _dev(rng.standard_normal(nz * wa.mesh.nV))
            for method in abi.REMAP_METHODS:
                out = _dev(np.full(nz * wb.mesh.nV, np.nan))
                cb.remap_field(ca, method, d.data_ptr(), out.data_ptr(), nz)
                for k in (0, 4, 5, nz - 5, nz - 2, nz - 1):
                    one = _dev(np.full(wb.mesh.nV, np.nan))
                    x = _layer(d, nz, k)
                    cb.remap_field(ca, method, x.data_ptr(), one.data_ptr(), 1)
                    assert torch.equal(out.view(nz, -1)[k], one), (method, nz, k)
    finally:
        ca.close()
        cb.close()
