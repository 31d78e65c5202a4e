"""Which of two ways to the same results ran: the loop and the smoothing on
patches, or the colour launches that they replace."""
import os
import subprocess
import sys

import numpy as np
import pytest

from ufemism_amd import abi, geometry
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
from ufemism_amd import abi, geometry
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
