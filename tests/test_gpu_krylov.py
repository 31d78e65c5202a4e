"""Gram-Schmidt at the vector counts where a group of eight ends and at sizes
below, at and above one row per thread: the FP64 residual that the library
evaluates apart from the Krylov vectors has to reach the tolerance, and the
residual of a cycle never grows (GMRES minimises it over a space with zero in
it), which a wrong dot, norm or update would break."""
import pytest

from ufemism_amd import abi, geometry
from ufemism_amd.dynamics import frozen_ssa_system

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[60, 2000, 70000])
def system(request):
    print(f"[krylov] marine {request.param}", flush=True)
    ctx = abi.Context(0)
    frozen_ssa_system(ctx, geometry.marine(request.param, seed=5, picard=2), picard=2)
    yield ctx
    ctx.close()


@pytest.mark.parametrize("restart", [1, 7, 8, 9, 17, 33])
@pytest.mark.parametrize("precision,passes", [(abi.UFE_MIXED, 1), (abi.UFE_MIXED, 2), (abi.UFE_FP64, 1)])
def test_gmres_restarts(system, restart, precision, passes):
    ctx = system
    ctx.fill("U_SSA_AaAc", 0.0)
    ctx.fill("V_SSA_AaAc", 0.0)
    last = ctx.ssa_residual()
    sweeps = 4 * restart + 1                    # about one cycle a call
    for _ in range(400):
        st = ctx.ssa_linear_solve(1e-7, sweeps, precision=precision, gmres=restart, precond_sweeps=2,
                                  orth_passes=passes, precond_type=abi.UFE_PRECOND_MULTIGRID)
        r = ctx.ssa_residual()
        assert r <= last * (1 + 1e-6), (restart, r, last)
        last = r
        if st.status == 0 and r <= 1e-7 * (1 + 1e-9):
            break
    print(f"  restart {restart} precision {precision} passes {passes}: residual {last:.1e}", flush=True)
    assert last <= 1e-7 * (1 + 1e-9)
