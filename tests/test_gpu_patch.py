"""Sweeps on patches (one launch per smoothing, halo rows recomputed by every
patch that needs them) against the per-colour kernels: the same operations on
the same values, so the same bits."""
import os

import numpy as np
import pytest

from ufemism_amd import abi, batch, geometry
from ufemism_amd.dynamics import Step, frozen_ssa_system

pytestmark = pytest.mark.gpu


def _linear(wl, on, precision, nu):
    os.environ["UFE_AMG_PATCH"] = on
    ctx = abi.Context(0)
    try:
        frozen_ssa_system(ctx, wl, picard=2)
        ctx.fill("U_SSA_AaAc", 0.0)
        ctx.fill("V_SSA_AaAc", 0.0)
        st = ctx.ssa_linear_solve(1e-8, 100000, precision=precision, gmres=20, precond_sweeps=nu, orth_passes=1,
                                  precond_type=abi.UFE_PRECOND_MULTIGRID)
        return st.matvecs, st.sweeps, ctx.get("U_SSA_AaAc"), ctx.get("V_SSA_AaAc")
    finally:
        ctx.close()
        os.environ.pop("UFE_AMG_PATCH", None)


@pytest.mark.parametrize("kind,n,nu", [("dome", 300, 2), ("dome", 2000, 1), ("marine", 20000, 2), ("marine", 20000, 1),
                                       ("marine", 90000, 2)])
@pytest.mark.parametrize("precision", [abi.UFE_MIXED, abi.UFE_FP64])
def test_multigrid_smoothing_on_patches_is_bit_identical(kind, n, nu, precision):
    print(f"[patch] {kind} {n} nu {nu} precision {precision}", flush=True)
    wl = (geometry.dome if kind == "dome" else geometry.marine)(n, seed=5, picard=2)
    a, b = (_linear(wl, on, precision, nu) for on in ("0", "1"))
    assert a[:2] == b[:2], (a[:2], b[:2])
    assert np.array_equal(a[2], b[2]) and np.array_equal(a[3], b[3])
    assert np.abs(a[2]).max() > 0


def test_multigrid_patches_with_prescribed_rows():
    """The grounding-line flux holds rows of the smoother fixed."""
    print("[patch] GL flux", flush=True)
    wl = geometry.marine(20000, seed=5, picard=3)
    wl.params.use_analytical_GL_flux = True
    out = {}
    for on in ("0", "1"):
        os.environ["UFE_AMG_PATCH"] = on
        ctx = abi.Context(0)
        try:
            step = Step(ctx, wl)
            ctx.set_params(wl.params, abi.UFE_MIXED, linear_rel_tol=1e-8, precond_type=abi.UFE_PRECOND_MULTIGRID,
                           precond_sweeps=2)
            out[on] = step.run()
        finally:
            ctx.close()
            os.environ.pop("UFE_AMG_PATCH", None)
    assert out["0"]["sweeps"] == out["1"]["sweeps"]
    for k in ("U_SSA", "V_SSA", "Ux_SSA_Ac", "Uy_SSA_Ac"):
        assert np.array_equal(out["0"][k], out["1"][k]), k


def test_batch_on_patches_is_bit_identical():
    print("[patch] batch", flush=True)
    wls = batch.ensemble(n=4, nv_min=1500, nv_max=6000, seed=7, picard=2)
    out = {}
    for on in ("0", "1"):
        os.environ["UFE_AMG_PATCH"] = on
        ctx = abi.Context(0)
        try:
            b = batch.Batch(ctx, wls)
            ctx.update_general_ice_model_data()
            for _ in range(2):          # the second pass replays the captured cycle
                b.reset()
                ctx.update_general_ice_model_data()
                st, rel = ctx.batch_solve_SSA(2, rel_tol=1e-8, gmres_restart=20, precond_sweeps=2,
                                              precond_type=abi.UFE_PRECOND_MULTIGRID)
            assert st.status == 0, (st.status, rel)
            out[on] = (st.cycles, ctx.get("U_SSA"), ctx.get("V_SSA"))
        finally:
            ctx.close()
            os.environ.pop("UFE_AMG_PATCH", None)
    assert out["0"][0] == out["1"][0]
    assert np.array_equal(out["0"][1], out["1"][1]) and np.array_equal(out["0"][2], out["1"][2])


def _sor_step(wl, on, sweep_batch=0):
    os.environ["UFE_SOR_PATCH"] = on
    ctx = abi.Context(0)
    try:
        step = Step(ctx, wl, sweep_batch=sweep_batch)
        a = step.run()
        step.reset()
        b = step.run()              # the second solve starts from other counters and buffers
        assert a["sweeps"] == b["sweeps"] and np.array_equal(a["U_SSA"], b["U_SSA"])
        return b
    finally:
        ctx.close()
        os.environ.pop("UFE_SOR_PATCH", None)


def _same_step(wl, sweep_batch=0):
    a, b = _sor_step(wl, "0"), _sor_step(wl, "1", sweep_batch)
    assert a["sweeps"] == b["sweeps"], (a["sweeps"], b["sweeps"])
    assert a["stats"].status == b["stats"].status and a["stats"].resets == b["stats"].resets
    assert a["stats"].last_max_residual == b["stats"].last_max_residual
    for k in ("U_SSA", "V_SSA", "Ux_SSA_Ac", "Uy_SSA_Ac", "Hi", "eta_AaAc"):
        assert np.array_equal(a[k], b[k]), k
    return b


# sizes on both sides of each workgroup width: few patches, one per CU, and the
# widths 256, 512 and 1,024
@pytest.mark.parametrize("kind,n,picard", [("dome", 60, 3), ("dome", 300, 4), ("dome", 2000, 5), ("dome", 8000, 6),
                                           ("marine", 20000, 6), ("marine", 37000, 3), ("marine", 70000, 2),
                                           ("marine", 130000, 2)])
def test_sor_loop_on_patches_is_bit_identical(kind, n, picard):
    print(f"[sor patch] {kind} {n}", flush=True)
    wl = (geometry.dome if kind == "dome" else geometry.marine)(n, seed=5, picard=picard)
    wl.params.SSA_max_residual_UV = 1e-2     # the reference's 2.5 m/yr ends a fine mesh's first solves after one sweep
    wl.params.SSA_max_inner_loops = 300
    r = _same_step(wl)
    assert sum(r["sweeps"]) > picard


def test_sor_loop_on_patches_stops_as_the_sweeps_do():
    """The sweep limit, launches of a few sweeps, and the reset of an unstable solve."""
    print("[sor patch] limits", flush=True)
    wl = geometry.marine(12000, seed=5, picard=4)
    wl.params.SSA_max_residual_UV = 1e-3
    for limit in (1, 2, 37):
        wl.params.SSA_max_inner_loops = limit
        r = _same_step(wl)
        assert r["sweeps"] == [limit] * r["picard"] and r["stats"].status == 1
    wl.params.SSA_max_inner_loops = 200
    _same_step(wl, sweep_batch=7)
    wl = geometry.marine(12000, seed=5, picard=2)
    wl.params.use_analytical_GL_flux = True
    _same_step(wl)


# one patch width below 131,072 points and the other above, one sweep and two
@pytest.mark.parametrize("n,nu,gl", [(300, 2, False), (6000, 1, False), (6000, 2, True), (36000, 2, False)])
def test_transposed_smoothing_on_patches_is_bit_identical(n, nu, gl):
    """The adjoint's preconditioner and operator on patches against the colour passes."""
    torch = pytest.importorskip("torch")
    from ufemism_amd.adjoint import AdjointOptions, SSAProblem, ssa_velocities
    print(f"[patch] adjoint {n} nu {nu} gl {gl}", flush=True)
    wl = geometry.marine(n, seed=5, picard=2)
    wl.params.use_analytical_GL_flux = gl
    out = {}
    for on in ("0", "1"):
        os.environ["UFE_AMG_PATCH"] = on
        ctx = abi.Context(0)
        try:
            step = Step(ctx, wl)
            ctx.update_general_ice_model_data()
            prob = SSAProblem(ctx, AdjointOptions(picard_iterations=2, lin_rel_tol=1e-10, gmres_restart=20,
                                                  precond_sweeps=nu, precond_type=abi.UFE_PRECOND_MULTIGRID))
            tau = torch.tensor(wl.tau_c_override(step.ma["VAaAc"]), dtype=torch.float64, device=prob.dev)
            lt = torch.log(tau).requires_grad_(True)
            A = torch.full_like(tau, wl.A_flow).requires_grad_(True)
            U, V = ssa_velocities(lt, A, prob)
            (U * U + 2.0 * V * V).sum().backward()
            out[on] = (prob.backward_stats.adjoint_matvecs, lt.grad.clone(), A.grad.clone(), U.detach().clone())
        finally:
            ctx.close()
            os.environ.pop("UFE_AMG_PATCH", None)
    assert out["0"][0] == out["1"][0] > 0
    for a, b in zip(out["0"][1:], out["1"][1:]):
        assert torch.equal(a, b) and float(a.abs().max()) > 0
