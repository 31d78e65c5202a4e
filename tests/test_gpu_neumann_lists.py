"""neumann_AaAc on meshes with and without corner points."""
import numpy as np
import pytest

from ufemism_amd import abi, geometry

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("corners", [True, False])
def test_neumann_of_a_batch_with_and_without_corner_codes(corners):
    """A batch may be uploaded without the corners' codes in edge_index: its
    corners are then edge points like the others."""
    print(f"[neumann lists] corners {corners}", flush=True)
    wl = geometry.dome(300, seed=3)
    ctx = abi.Context(0)
    try:
        ctx.set_params(wl.params)
        ma = ctx.mesh_build(wl.mesh)
        if not corners:
            ma.mesh.edge_index = np.where(np.isin(ma.mesh.edge_index, (2, 4, 6, 8)), 1, ma.mesh.edge_index).astype(np.int32)
        ctx.batch_define([wl.mesh.nV], [ma.nAc])
        ctx.mesh_upload(ma)
        nA = ctx.sizes["nVAaAc"]
        d = np.random.default_rng(1).standard_normal(nA)
        t = torch.from_numpy(d.copy()).cuda()
        torch.cuda.synchronize()
        ctx.op("neumann_AaAc", t.data_ptr())
        edge = np.concatenate([ma.mesh.edge_index, ma["edge_index_Ac"]]) > 0
        C, nC = ma["CAaAc"], ma["nCAaAc"]
        ref = d.copy()
        is_corner = np.isin(np.arange(nA), np.nonzero(np.isin(ma.mesh.edge_index, (2, 4, 6, 8)))[0])
        assert is_corner.sum() == (4 if corners else 0)

        def mean(a, keep):
            s, n = 0.0, 0
            for j in C[a, :nC[a]] - 1:
                if keep(j):
                    s, n = s + ref[j], n + 1
            return s / n
        for a in np.nonzero(edge & ~is_corner)[0]:
            ref[a] = mean(a, lambda j: not edge[j])
        for a in np.nonzero(is_corner)[0]:
            ref[a] = mean(a, lambda j: True)
        assert np.array_equal(t.cpu().numpy(), ref)
    finally:
        ctx.close()
