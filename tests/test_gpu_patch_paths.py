"""Which of two ways to the same results ran: the loop and the smoothing on
patches, or the colour launches that they replace."""
import os
import subprocess
import sys

import numpy as np
import pytest

from ufemism_amd import abi, batch, geometry
from ufemism_amd.dynamics import Step, frozen_ssa_system

pytestmark = pytest.mark.gpu
FIELDS = ("U_SSA", "V_SSA", "Ux_SSA_Ac", "Uy_SSA_Ac", "Hi")


def _sor_step(wl, sweep_batch=0, **env):
    """One step; its results and the ways it took.  Environment switches are read per solve or per mesh."""
    os.environ.update(env)
    ctx = abi.Context(0)
    try:
        out = Step(ctx, wl, sweep_batch=sweep_batch).run()
        return out, ctx.path_counts()
    finally:
        ctx.close()
        for k in env:
            os.environ.pop(k, None)


def _same(a, b):
    assert a["sweeps"] == b["sweeps"], (a["sweeps"], b["sweeps"])
    for k in ("status", "resets", "last_max_residual", "last_RN"):
        assert getattr(a["stats"], k) == getattr(b["stats"], k), k
    for k in FIELDS:
        assert np.array_equal(a[k], b[k], equal_nan=True), k


@pytest.mark.parametrize("kind,n", [("dome", 300), ("marine", 12000), ("marine", 37000), ("marine", 70000)])
def test_sor_loop_that_gives_up_is_repeated_by_colour_launches(kind, n):
    """No polls at all: every workgroup gives up after its first sweep.  A few
    polls: some may give up after any sweep, and what they had written is undone."""
    print(f"[sor wait] {kind} {n}", flush=True)
    wl = (geometry.dome if kind == "dome" else geometry.marine)(n, seed=5, picard=3)
    wl.params.SSA_max_residual_UV = 1e-2
    wl.params.SSA_max_inner_loops = 60
    ref, c = _sor_step(wl, UFE_SOR_PATCH="0")
    assert c["sor_patch"] == 0 and c["sor_colour"] > 0
    out, c = _sor_step(wl, UFE_SOR_SPINS="0")
    assert c["sor_patch"] == c["sor_gave_up"] == 1 and c["sor_colour"] > 0
    _same(ref, out)
    for spins in ("1", "2", "4", "8", "12", "16", "30"):
        out, c = _sor_step(wl, sweep_batch=7, UFE_SOR_SPINS=spins)
        print(f"  spins {spins}: {c['sor_patch']} launches, {c['sor_gave_up']} gave up", flush=True)
        _same(ref, out)
    out, c = _sor_step(wl)
    assert c["sor_patch"] >= 1 and c["sor_gave_up"] == c["sor_colour"] == 0
    _same(ref, out)


def test_loop_of_a_large_mesh_beside_a_smaller_one_of_its_width():
    """Two meshes whose workgroups have 1,024 threads and whose patches take more
    than the default 64 KiB of LDS, the larger one solved before and after the smaller."""
    print("[sor paths] two meshes", flush=True)
    wls = [geometry.marine(n, seed=5, picard=2) for n in (130000, 90000)]
    ctxs = [abi.Context(0) for _ in wls]
    try:
        steps = []
        for c, wl in zip(ctxs, wls):
            wl.params.SSA_max_inner_loops = 5
            steps.append(Step(c, wl))
        first = steps[0].run()
        steps[1].run()
        steps[0].reset()
        again = steps[0].run()
        _same(first, again)
        for c in ctxs:
            p = c.path_counts()
            assert p["sor_patch"] > 0 and p["sor_colour"] == 0, p
    finally:
        for c in ctxs:
            c.close()


CHILD = r"""
import sys
sys.modules["torch"] = None          # the HIP runtime the library is linked with
sys.path.insert(0, sys.argv[1])
import numpy as np
from ufemism_amd import abi, batch, geometry
from ufemism_amd.dynamics import Step, frozen_ssa_system
for n in (300, 2000):
    ctx = abi.Context(0)
    out = Step(ctx, geometry.dome(n, seed=5, picard=3)).run()
    p = ctx.path_counts()
    print(p, flush=True)
    assert p["sor_patch"] + p["sor_colour"] > 0
    assert (p["sor_patch"] > 0) == (p["patch_sets"] > 0), p      # nothing is built that cannot run
    ctx.close()
np.save(sys.argv[2], np.stack([out["U_SSA"], out["V_SSA"]]))
"""


def test_process_beside_one_with_the_cooperative_queue(tmp_path):
    """The device has one cooperative queue: a process that does not get it takes
    the colour launches, without building the patches of the loop first."""
    print("[sor paths] second process", flush=True)
    wl = geometry.dome(2000, seed=5, picard=3)
    out, c = _sor_step(wl)
    assert c["sor_patch"] > 0
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-u", "-c", CHILD, root, str(tmp_path / "uv.npy")], capture_output=True, text=True,
                       timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0
    assert np.array_equal(np.load(tmp_path / "uv.npy"), np.stack([out["U_SSA"], out["V_SSA"]]))


def test_mesh_too_large_for_the_loop_is_not_walked():
    print("[sor paths] too large", flush=True)
    wl = geometry.marine(300000, seed=5, picard=1)
    wl.params.SSA_max_inner_loops = 2
    _, c = _sor_step(wl)
    assert c["patch_sets"] == c["sor_patch"] == 0 and c["sor_colour"] > 0, c


def test_profiled_bytes_of_a_smoothing_are_those_of_one_launch():
    """Two sweeps in one launch read the coefficients once: the bytes it is credited
    with stay below one colour sweep's and the residual's, and the rows are both sweeps'."""
    print("[patch profile]", flush=True)
    wl = geometry.marine(6000, seed=5, picard=2)
    ctx = abi.Context(0)
    try:
        frozen_ssa_system(ctx, wl, picard=2)
        ctx.profile_read()
        ctx.profile_enable(True)
        ctx.ssa_linear_solve(1e-6, 1000, precision=abi.UFE_MIXED, gmres=20, precond_sweeps=2, orth_passes=1,
                             precond_type=abi.UFE_PRECOND_MULTIGRID)
        ctx.profile_enable(False)
        p, sweep = ctx.profile_read(), ctx.sweep_bytes()
        assert ctx.path_counts()["smooth_patch"] > 0 and p.launches > 0
        per = p.algorithmic_bytes / p.launches
        assert p.rows == 2 * sweep["rows"] * p.launches
        assert 0.5 * sweep["fp32"] < per <= sweep["fp32"] + 8 * sweep["rows"], (per, sweep)
    finally:
        ctx.close()


SMOOTH = {"0": ("smooth_colour", "smooth_patch"), "1": ("smooth_patch", "smooth_colour")}


@pytest.mark.parametrize("on", ["0", "1"])
@pytest.mark.parametrize("kind,n,nu", [("dome", 300, 2), ("marine", 20000, 1), ("marine", 90000, 2)])
def test_switch_of_the_smoothing_decides_the_way(kind, n, nu, on):
    """The comparisons of the two ways compare two ways."""
    print(f"[patch ways] {kind} {n} nu {nu} {on}", flush=True)
    wl = getattr(geometry, kind)(n, seed=5, picard=2)
    os.environ["UFE_AMG_PATCH"] = on
    ctx = abi.Context(0)
    try:
        Step(ctx, wl)
        ctx.set_params(wl.params, abi.UFE_MIXED, linear_rel_tol=1e-6, precond_type=abi.UFE_PRECOND_MULTIGRID,
                       precond_sweeps=nu)
        ctx.update_general_ice_model_data()
        ctx.solve_SIA()
        ctx.solve_SSA()
        c = ctx.path_counts()
        taken, other = SMOOTH[on]
        assert c[taken] > 0 and c[other] == 0 and c["patch_sets"] == 2 * int(on), c
    finally:
        ctx.close()
        os.environ.pop("UFE_AMG_PATCH", None)


@pytest.mark.parametrize("on", ["0", "1"])
def test_switch_of_the_smoothing_decides_the_way_of_a_batch(on):
    os.environ["UFE_AMG_PATCH"] = on
    ctx = abi.Context(0)
    try:
        b = batch.Batch(ctx, batch.ensemble(n=3, nv_min=1500, nv_max=4000, seed=7, picard=2))
        ctx.update_general_ice_model_data()
        ctx.batch_solve_SSA(2, rel_tol=1e-6, gmres_restart=20, precond_sweeps=2, precond_type=abi.UFE_PRECOND_MULTIGRID)
        c = ctx.path_counts()
        taken, other = SMOOTH[on]
        assert c[taken] > 0 and c[other] == 0, c
        del b
    finally:
        ctx.close()
        os.environ.pop("UFE_AMG_PATCH", None)


@pytest.mark.parametrize("sweep_batch", [0, 3])
def test_unstable_solve_is_reset_on_both_ways(sweep_batch):
    """Over-relaxation by 2.6 diverges: the first solve resets the velocities, the
    second ends the call, with the same sweeps and the same velocities left."""
    print(f"[sor ways] divergent, sweep batch {sweep_batch}", flush=True)
    wl = geometry.marine(2000, seed=5, picard=5)
    wl.params.SSA_SOR_omega = 2.6
    wl.params.SSA_max_inner_loops = 2000
    out = {}
    for on in ("0", "1"):
        os.environ["UFE_SOR_PATCH"] = on
        ctx = abi.Context(0)
        try:
            Step(ctx, wl, sweep_batch=sweep_batch)
            ctx.update_general_ice_model_data()
            ctx.solve_SIA()
            st = ctx.solve_SSA(allow=(abi.UFE_OK, abi.UFE_SOR_NOT_CONVERGED, abi.UFE_SSA_UNSTABLE))
            assert st.resets == 2 and st.status == abi.UFE_SSA_UNSTABLE, (st.resets, st.status)
            assert st.last_max_residual > 1e6
            c = ctx.path_counts()
            assert (c["sor_patch"] > 0, c["sor_colour"] > 0) == ((False, True) if on == "0" else (True, False)), c
            out[on] = (list(st.sweeps)[:st.picard_iterations], st.last_max_residual,
                       [ctx.get(k) for k in ("U_SSA", "V_SSA", "Ux_SSA_Ac", "Uy_SSA_Ac")])
        finally:
            ctx.close()
            os.environ.pop("UFE_SOR_PATCH", None)
    assert out["0"][:2] == out["1"][:2], (out["0"][:2], out["1"][:2])
    for a, b in zip(out["0"][2], out["1"][2]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("gl", [False, True])
def test_adjoint_folds_in_one_launch_and_in_several(gl):
    """The folds of meshes with many edge points (UFE_FOLD_MAX=0) against the one
    workgroup of the others and against the colour launches: the same gradients."""
    torch = pytest.importorskip("torch")
    from ufemism_amd.adjoint import AdjointOptions, SSAProblem, ssa_velocities
    print(f"[adjoint folds] gl {gl}", flush=True)
    wl = geometry.marine(6000, seed=5, picard=2)
    wl.params.use_analytical_GL_flux = gl
    out = {}
    for name, env in (("colours", {"UFE_AMG_PATCH": "0"}), ("one", {}), ("several", {"UFE_FOLD_MAX": "0"})):
        os.environ.update(env)
        ctx = abi.Context(0)
        try:
            step = Step(ctx, wl)
            ctx.update_general_ice_model_data()
            prob = SSAProblem(ctx, AdjointOptions(picard_iterations=2, lin_rel_tol=1e-10, gmres_restart=20,
                                                  precond_sweeps=2, precond_type=abi.UFE_PRECOND_MULTIGRID))
            tau = torch.tensor(wl.tau_c_override(step.ma["VAaAc"]), dtype=torch.float64, device=prob.dev)
            lt = torch.log(tau).requires_grad_(True)
            A = torch.full_like(tau, wl.A_flow).requires_grad_(True)
            U, V = ssa_velocities(lt, A, prob)
            (U * U + 2.0 * V * V).sum().backward()
            out[name] = (lt.grad.clone(), A.grad.clone())
            c = ctx.path_counts()
            assert (c["smooth_T_patch"] > 0, c["smooth_T_colour"] > 0) == ((False, True) if name == "colours" else (True, False)), c
        finally:
            ctx.close()
            for k in env:
                os.environ.pop(k, None)
    for name in ("one", "several"):
        for a, b in zip(out["colours"], out[name]):
            assert torch.equal(a, b) and float(a.abs().max()) > 0, name


def test_profile_samples_both_smoothings():
    """The two smoothings of an application alternate and differ in bytes and time:
    the sampled mean lies between theirs."""
    print("[patch profile] both", flush=True)
    wl = geometry.marine(6000, seed=5, picard=2)
    ctx = abi.Context(0)
    try:
        frozen_ssa_system(ctx, wl, picard=2)
        ctx.profile_read()
        ctx.profile_enable(True)
        for _ in range(3):
            ctx.ssa_linear_solve(1e-8, 1000, precision=abi.UFE_MIXED, gmres=20, precond_sweeps=2, orth_passes=1,
                                 precond_type=abi.UFE_PRECOND_MULTIGRID)
        ctx.profile_enable(False)
        p, sweep = ctx.profile_read(), ctx.sweep_bytes()
        assert p.launches >= 8 and p.total_launches >= 7 * (p.launches - 1)
        pre = (10.0 * sweep["mean_degree"] + 44.0) * sweep["rows"]       # coefficients, columns, row data, z and residual
        post = pre + 8.0 * sweep["rows"]                                 # and the values it starts from
        mean = p.algorithmic_bytes / p.launches
        assert pre + 0.3 * (post - pre) < mean < pre + 0.7 * (post - pre), (pre, mean, post)
    finally:
        ctx.close()
