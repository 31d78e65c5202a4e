"""The work that users of this library have it do, as timed cases.

A case is a plain dict.  ``prepare`` makes what a program holds before the
call (an uploaded mesh with its ice state, the remapping arrays, the device
buffers it passes), ``run`` makes one pass through the public entry points
of ``ufemism_amd`` and returns its outputs, ``work`` gives the bytes and
operations that pass cannot do without, and ``exact`` the 64-bit result of
the passes that have a closed form (plain numpy on the mesh arrays).

Kinds of cases:

* ``columns``   the part of a time step around the SSA: general update with
                the Arrhenius properties, SIA, 3-D velocities, mass
                continuity, critical time steps;
* ``step``      one whole dynamics step, FP64 with the reference's SOR and
                stopping rules (the drop-in use);
* ``ssa``       solve_SSA alone: the reference's SOR, or GMRES-IR with the
                multigrid preconditioner, mixed or FP64 Krylov vectors;
* ``linear``    one linearised system at fixed viscosity, from zero;
* ``adjoint``   velocities and gradients through torch.autograd;
* ``batch``     an ensemble of uneven meshes solved together;
* ``operators`` the mesh operators on a caller's device buffers;
* ``remap``     fields moved from one mesh to the next after re-meshing.

A mesh depends on the kind of ice sheet and its size only and is generated
once per process; the state (thickness, bed, friction, temperature) comes
from the seed.
"""
import dataclasses
import functools
import math

import numpy as np
import torch

from ufemism_amd import abi, batch as batching, geometry
from ufemism_amd.adjoint import AdjointOptions, SSAProblem, ssa_velocities
from ufemism_amd.dynamics import initial_fields

NZ = 15                     # the reference's default vertical grid
AT_REST = ("U_SSA", "V_SSA", "Ux_SSA_Ac", "Uy_SSA_Ac", "N_AaAc")


def listed():
    return [
        # the smallest call: a small dome between two SSA solves, bound by launches
        {"name": "columns_dome_2k", "kind": "columns", "sheet": "dome", "n": 2000},
        # the flat-bed dome benchmark: one dynamics step, 10 Picard iterations
        {"name": "step_dome_8k", "kind": "step", "sheet": "dome", "n": 8000, "picard": 10, "gl_flux": False},
        # a marine sheet with the analytical grounding-line flux
        {"name": "step_marine_20k_gl", "kind": "step", "sheet": "marine", "n": 20000, "picard": 10, "gl_flux": True},
        # the 200k-vertex marine benchmark, its first Picard iterations
        {"name": "ssa_sor_marine_200k", "kind": "ssa", "sheet": "marine", "n": 200000, "solver": "sor", "picard": 8},
        # the Picard loop with the fast linear solver, at the tolerance the tests use
        {"name": "ssa_mixed_marine_50k", "kind": "ssa", "sheet": "marine", "n": 50000, "solver": "mixed",
         "picard": 4},
        {"name": "ssa_fp64krylov_dome_30k", "kind": "ssa", "sheet": "dome", "n": 30011, "solver": "fp64_krylov",
         "picard": 4},
        # the headline benchmark: 1M vertices to 1e-6, mixed precision
        {"name": "linear_mixed_marine_1M", "kind": "linear", "sheet": "marine", "n": 1000000, "solver": "mixed",
         "tol": 1e-6},
        # friction and rate-factor inversion: a forward and its gradient
        {"name": "adjoint_marine_40k", "kind": "adjoint", "sheet": "marine", "n": 40009, "picard": 3},
        # an ensemble of uneven members
        {"name": "batch_16", "kind": "batch", "members": 16, "n_min": 5000, "n_max": 25000, "picard": 2},
        # the columns of a large sheet
        {"name": "columns_marine_400k", "kind": "columns", "sheet": "marine", "n": 400003},
        {"name": "operators_marine_200k", "kind": "operators", "sheet": "marine", "n": 200000},
        {"name": "remap_100k", "kind": "remap", "n_src": 100000, "n_dst": 125000},
    ]


def draw(rng):
    """One more case: sizes log-uniform over the ranges of the listed ones."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def sheet():
        return rng.choice(["dome", "marine"])

    kind = rng.choice(["columns", "step", "ssa", "ssa", "linear", "adjoint", "batch", "operators", "remap"])
    if kind == "columns":
        return {"kind": kind, "sheet": sheet(), "n": size(2000, 400000)}
    if kind == "step":
        s = sheet()
        return {"kind": kind, "sheet": s, "n": size(2000, 30000), "picard": rng.randint(4, 10),
                "gl_flux": s == "marine" and rng.random() < 0.5}
    if kind == "ssa":
        solver = rng.choice(["sor", "mixed", "fp64_krylov"])
        return {"kind": kind, "sheet": sheet(), "n": size(20000, 200000 if solver == "sor" else 100000),
                "solver": solver, "picard": rng.randint(2, 4)}
    if kind == "linear":
        return {"kind": kind, "sheet": "marine", "n": size(20000, 500000), "solver": rng.choice(["mixed", "fp64_krylov"]),
                "tol": rng.choice([1e-6, 1e-8, 1e-9])}
    if kind == "adjoint":
        return {"kind": kind, "sheet": "marine", "n": size(5000, 40000), "picard": rng.randint(1, 3)}
    if kind == "batch":
        return {"kind": kind, "members": rng.randint(3, 12), "n_min": 2000, "n_max": size(4000, 20000),
                "picard": rng.randint(1, 2)}
    if kind == "operators":
        return {"kind": kind, "sheet": sheet(), "n": size(2000, 200000)}
    n = size(2000, 100000)
    return {"kind": kind, "n_src": n, "n_dst": int(n * rng.uniform(0.75, 1.25)) + 1}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=24)
def _sheet(kind, n):
    return (geometry.dome if kind == "dome" else geometry.marine)(n, seed=11)


_built = {}


def _secondary(ctx, kind, n):
    """The mesh of a sheet with its secondary arrays (host), built once."""
    if (kind, n) not in _built:
        _built[kind, n] = ctx.mesh_build(_sheet(kind, n).mesh)
    return _built[kind, n]


def _workload(kind, n, seed, picard=4, gl_flux=False, physics=0):
    """A sheet with a seeded state: 2 % thickness undulations, fresh bed bumps
    on the marine sheet, log-normal friction, mass balance of a few dm/yr."""
    wl = _sheet(kind, n)
    V = wl.mesh.V
    g = geometry.gaussian_field(V, 60e3, seed + 1)
    Hb = wl.Hb
    if kind == "marine":
        Hb = -150.0 - 0.5 * np.hypot(V[:, 0], V[:, 1]) / 1e3 + 50.0 * geometry.gaussian_field(V, 20e3, seed + 2)
    p = dataclasses.replace(wl.params, SSA_max_outer_loops=picard, SSA_RN_tol=1e-6,
                            use_analytical_GL_flux=gl_flux, physical_properties=physics)
    return dataclasses.replace(wl, Hi=wl.Hi * (1.0 + 0.02 * np.clip(g, -3, 3)), Hb=Hb, params=p,
                               friction_sigma=0.5, friction_seed=seed + 3, SMB=0.3 * g, BMB=-0.1 * np.abs(g))


def _upload(ctx, wl, ma, precision=abi.UFE_FP64, **krylov):
    ctx.set_params(wl.params, precision, **krylov)
    ctx.mesh_upload(ma)
    for k, v in initial_fields(wl, ma["VAaAc"], wl.params.nZ).items():
        ctx.set(k, v)


def _dev(a):
    """A host array in the reference (column-major) layout as a device tensor."""
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a).ravel(order="F"))).to("cuda")


class _Out:
    """Device buffers that fields are copied into at the end of a pass."""

    def __init__(self, ctx, names):
        self.ctx, self.buf = ctx, {}
        for name in names:
            _, grid, dt = ctx.fields[name]
            n = math.prod(ctx._shape(grid))
            self.buf[name] = torch.empty(n, dtype=torch.float64 if dt == 0 else torch.int32, device="cuda")

    def get(self):
        for name, t in self.buf.items():
            self.ctx.get_device(name, t.data_ptr())
        return dict(self.buf)


def _general(ctx):
    ctx.update_general_ice_model_data()
    ctx.solve_SIA()


KRYLOV = {"mixed": abi.UFE_MIXED, "fp64_krylov": abi.UFE_FP64_KRYLOV}
MULTIGRID = dict(gmres_restart=20, precond_sweeps=2, precond_type=abi.UFE_PRECOND_MULTIGRID)
SSA_OUT = ("U_SSA", "V_SSA", "Ux_SSA_Ac", "Uy_SSA_Ac", "Up_SSA_Ac", "Uo_SSA_Ac", "eta_AaAc")


def prepare(case, seed):
    ctx = abi.Context(0)
    s = globals()["_prepare_" + case["kind"]](ctx, case, seed)
    s.update(ctx=ctx, kind=case["kind"], case=case)
    torch.cuda.synchronize()
    return s


def run(state):
    return globals()["_run_" + state["kind"]](state["ctx"], state)


# -- columns -----------------------------------------------------------------
def _prepare_columns(ctx, case, seed):
    wl = _workload(case["sheet"], case["n"], seed, physics=1)
    ma = _secondary(ctx, case["sheet"], case["n"])
    _upload(ctx, wl, ma)
    # sliding velocities of an earlier SSA solve
    u = 100.0 * geometry.gaussian_field(wl.mesh.V, 80e3, seed + 4)
    v = 100.0 * geometry.gaussian_field(wl.mesh.V, 80e3, seed + 5)
    ctx.set("U_SSA", u)
    ctx.set("V_SSA", v)
    out = _Out(ctx, ("Hi", "dHi_dt", "Hs", "U_SIA", "V_SIA", "D_SIA", "A_flow_mean", "U_3D", "V_3D", "W_3D", "mask"))
    return {"out": out, "Hi": _dev(wl.Hi), "Ti": _dev(wl.temperature()), "dt": 0.5}


def _run_columns(ctx, s):
    ctx.set_device("Hi", s["Hi"].data_ptr())      # thickness and temperature from the models around
    ctx.set_device("Ti", s["Ti"].data_ptr())
    ctx.update_general_ice_model_data()
    ctx.solve_SIA()
    ctx.solve_SIA_3D()
    dt = ctx.critical_timesteps()
    ctx.calculate_ice_thickness_change(s["dt"])
    return dict(s["out"].get(), dt_crit=list(dt))


# -- step ----------------------------------------------------------------------
def _prepare_step(ctx, case, seed):
    wl = _workload(case["sheet"], case["n"], seed, case["picard"], case["gl_flux"])
    _upload(ctx, wl, _secondary(ctx, case["sheet"], case["n"]))
    return {"out": _Out(ctx, ("Hi", "U_SIA", "V_SIA") + SSA_OUT), "Hi": _dev(wl.Hi), "dt": wl.dt}


def _run_step(ctx, s):
    ctx.set_device("Hi", s["Hi"].data_ptr())
    for f in AT_REST:
        ctx.fill(f, 0.0)
    _general(ctx)
    st = ctx.solve_SSA()
    ctx.calculate_ice_thickness_change(s["dt"])
    return dict(s["out"].get(), sweeps=st.total_sweeps, picard=st.picard_iterations)


# -- ssa -----------------------------------------------------------------------
def _prepare_ssa(ctx, case, seed):
    wl = _workload(case["sheet"], case["n"], seed, case["picard"])
    ma = _secondary(ctx, case["sheet"], case["n"])
    if case["solver"] == "sor":
        _upload(ctx, wl, ma)
    else:
        _upload(ctx, wl, ma, KRYLOV[case["solver"]], linear_rel_tol=1e-10, **MULTIGRID)
    _general(ctx)
    return {"out": _Out(ctx, SSA_OUT)}


def _run_ssa(ctx, s):
    for f in AT_REST:
        ctx.fill(f, 0.0)
    st = ctx.solve_SSA()
    return dict(s["out"].get(), picard=st.picard_iterations)


# -- linear --------------------------------------------------------------------
def _prepare_linear(ctx, case, seed):
    """A system frozen at a flowing state, as after some Picard iterations."""
    wl = _workload(case["sheet"], case["n"], seed, picard=2)
    p = dataclasses.replace(wl.params, SSA_RN_tol=0.0)
    _upload(ctx, dataclasses.replace(wl, params=p), _secondary(ctx, case["sheet"], case["n"]), abi.UFE_FP64_KRYLOV,
            linear_rel_tol=1e-6, **MULTIGRID)
    _general(ctx)
    ctx.solve_SSA()
    ctx.set_params(wl.params, abi.UFE_FP64)
    ctx.ssa_prepare()
    return {"out": _Out(ctx, ("U_SSA_AaAc", "V_SSA_AaAc")), "tol": case["tol"],
            "precision": abi.UFE_MIXED if case["solver"] == "mixed" else abi.UFE_FP64}


def _run_linear(ctx, s):
    ctx.fill("U_SSA_AaAc", 0.0)
    ctx.fill("V_SSA_AaAc", 0.0)
    ctx.ssa_linear_solve(s["tol"], 400000, precision=s["precision"], gmres=20, precond_sweeps=2, orth_passes=1,
                         precond_type=abi.UFE_PRECOND_MULTIGRID)
    return s["out"].get()


# -- adjoint -------------------------------------------------------------------
def _prepare_adjoint(ctx, case, seed):
    wl = _workload(case["sheet"], case["n"], seed)
    ma = _secondary(ctx, case["sheet"], case["n"])
    _upload(ctx, wl, ma)
    ctx.update_general_ice_model_data()
    prob = SSAProblem(ctx, AdjointOptions(picard_iterations=case["picard"], lin_rel_tol=1e-11, gmres_restart=20,
                                          precond_sweeps=2, precond_type=abi.UFE_PRECOND_MULTIGRID))
    log_tau = torch.log(_dev(wl.tau_c_override(ma["VAaAc"])))
    A = torch.full_like(log_tau, wl.A_flow)
    g = _dev(geometry.gaussian_field(ma["VAaAc"], 50e3, seed + 6))
    U_obs, V_obs = prob.forward(log_tau + 0.3 * g, A)
    return {"prob": prob, "log_tau": log_tau, "A": A, "U_obs": U_obs, "V_obs": V_obs}


def _run_adjoint(ctx, s):
    lt = s["log_tau"].clone().requires_grad_(True)
    A = s["A"].clone().requires_grad_(True)
    U, V = ssa_velocities(lt, A, s["prob"])
    J = 0.5 * (((U - s["U_obs"]) ** 2).sum() + ((V - s["V_obs"]) ** 2).sum())
    J.backward()
    return {"U": U.detach(), "V": V.detach(), "grad_log_tau_c": lt.grad, "grad_A": A.grad}


# -- batch ---------------------------------------------------------------------
def _member_sizes(case):
    """Uneven sizes, log-uniform between the bounds."""
    k = np.arange(case["members"])
    t = (k * 0.6180339887498949) % 1.0
    return [int(n) for n in np.exp(math.log(case["n_min"]) + t * math.log(case["n_max"] / case["n_min"]))]


def _prepare_batch(ctx, case, seed):
    rng = np.random.default_rng(seed)
    wls = []
    for i, n in enumerate(_member_sizes(case)):
        wl = _workload("marine" if i % 2 else "dome", n, seed + 10 * i)
        wls.append(dataclasses.replace(wl, A_flow=float(rng.uniform(1e-17, 1e-16))))
    b = batching.Batch(ctx, wls)
    ctx.update_general_ice_model_data()
    return {"batch": b, "out": _Out(ctx, ("U_SSA", "V_SSA", "Ux_SSA_Ac", "Uy_SSA_Ac")), "picard": case["picard"]}


def _run_batch(ctx, s):
    for f in AT_REST:
        ctx.fill(f, 0.0)
    ctx.batch_solve_SSA(s["picard"], rel_tol=1e-9, precision=abi.UFE_MIXED, **MULTIGRID)
    return s["out"].get()


# -- operators -----------------------------------------------------------------
def _points(V, rng, k=0):
    """A smooth field of ice-sheet scale plus noise."""
    return (1e3 * np.sin(V[:, 0] / 2e5 + k) * np.cos(V[:, 1] / 3e5) + 0.5 * V[:, 0] / 1e3 + rng.standard_normal(len(V)))


def _operator_inputs(case, seed, ma):
    rng = np.random.default_rng(seed)
    V = ma.mesh.V
    h = {"aa": _points(V, rng), "aa3": np.concatenate([_points(V, rng, k) for k in range(NZ)]),
         "ac": _points(ma["VAc"], rng), "bc": _points(ma["VAc"], rng, 1),
         "ac3": np.concatenate([_points(ma["VAc"], rng, k) for k in range(NZ)]), "aaac": _points(ma["VAaAc"], rng)}
    h["u3"] = 100.0 * rng.standard_normal(len(h["aa3"]))
    h["v3"] = 100.0 * rng.standard_normal(len(h["aa3"]))
    return h


# (operator, inputs, outputs as (name, grid), layers)
OPERATORS = (
    ("derivatives_Aa", ("aa",), (("dx", "Aa"), ("dy", "Aa")), None),
    ("curvatures_Aa", ("aa",), (("dxx", "Aa"), ("dxy", "Aa"), ("dyy", "Aa")), None),
    ("derivatives_Aa_3D", ("aa3",), (("dx3", "Aaz"), ("dy3", "Aaz")), NZ),
    ("derivatives_Ac", ("aa",), (("dx_Ac", "Ac"), ("dy_Ac", "Ac"), ("dp_Ac", "Ac"), ("do_Ac", "Ac")), None),
    ("derivatives_AaAc", ("aaac",), (("dx_AaAc", "AaAc"), ("dy_AaAc", "AaAc")), None),
    ("map_Aa_to_Ac_3D", ("aa3",), (("to_Ac", "Acz"),), NZ),
    ("map_Ac_to_Aa_3D", ("ac3",), (("to_Aa", "Aaz"),), NZ),
    ("rotate_xy_to_po", ("ac", "bc"), (("p", "Ac"), ("o", "Ac")), None),
)


def _prepare_operators(ctx, case, seed):
    wl = _workload(case["sheet"], case["n"], seed)
    ma = _secondary(ctx, case["sheet"], case["n"])
    ctx.set_params(wl.params)
    ctx.mesh_upload(ma)
    nV, nAc = ma.nV, ma.nAc
    size = {"Aa": nV, "Aaz": nV * NZ, "Ac": nAc, "Acz": nAc * NZ, "AaAc": nV + nAc}
    dev = {k: _dev(v) for k, v in _operator_inputs(case, seed, ma).items()}
    out = {name: torch.empty(size[g], dtype=torch.float64, device="cuda") for _, _, outs, _ in OPERATORS
           for name, g in outs}
    for name in ("upx", "upy"):
        out[name] = torch.empty(size["Aaz"], dtype=torch.float64, device="cuda")
    out["neu3"] = dev["aa3"].clone()       # filled boundary values: a second pass finds them as they are
    out["neu_AaAc"] = dev["aaac"].clone()
    return {"dev": dev, "out": out}


def _run_operators(ctx, s):
    dev, out = s["dev"], s["out"]
    for op, ins, outs, nz in OPERATORS:
        ctx.op(op, *(dev[k].data_ptr() for k in ins), *(out[k].data_ptr() for k, _ in outs), nz=nz)
    ctx.op("neumann_Aa_3D", out["neu3"].data_ptr(), nz=NZ)
    ctx.op("neumann_AaAc", out["neu_AaAc"].data_ptr())
    missing = ctx.upwind_derivatives_3D(dev["u3"].data_ptr(), dev["v3"].data_ptr(), dev["aa3"].data_ptr(),
                                        out["upx"].data_ptr(), out["upy"].data_ptr(), NZ)
    return dict(out, missing=missing)


# -- remap ---------------------------------------------------------------------
def _remap_inputs(case, seed):
    rng = np.random.default_rng(seed)
    V = _sheet("marine", case["n_src"]).mesh.V
    return np.concatenate([250.0 + _points(V, rng, k) / 100.0 for k in range(NZ)])


def _prepare_remap(ctx, case, seed):
    """Two meshes on the device with the remapping arrays between them."""
    src = abi.Context(0)
    a, b = ("marine", case["n_src"]), ("marine", case["n_dst"])
    wa, wb = _workload(*a, seed), _workload(*b, seed)
    _upload(src, wa, _secondary(src, *a))
    _upload(ctx, wb, _secondary(ctx, *b))
    ctx.remap_build(src, _built[a], _built[b])
    d = _remap_inputs(case, seed)
    src.set("Ti", d.reshape(NZ, -1).T)
    src.set("Hi_prev", wa.Hi)
    n = ctx.sizes["nV"] * NZ
    out = {m: torch.empty(n, dtype=torch.float64, device="cuda") for m in abi.REMAP_METHODS}
    return {"src": src, "d": _dev(d), "out": out, "fields": _Out(ctx, ("Hi", "Hi_prev", "Ti"))}


def _run_remap(ctx, s):
    for m, t in s["out"].items():
        ctx.remap_field(s["src"], m, s["d"].data_ptr(), t.data_ptr(), NZ)
    ctx.remap_ice_model(s["src"])
    return dict(s["out"], **s["fields"].get())


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------
def work(case):
    """Bytes of every input read once and every output written once (8-byte
    reals, 4-byte indices; six neighbours a point, three Ac points a vertex),
    and the operations of the same arithmetic done once."""
    kind = case["kind"]
    if kind == "remap":
        ns, nd = case["n_src"], case["n_dst"]
        return {"bytes": (4 + 1.2) * 8.0 * NZ * (ns + nd) + nd * (4 * 28.0 + 40.0), "flops": 40.0 * NZ * nd}
    if kind == "batch":
        n = sum(_member_sizes(case))
    else:
        n = case["n"]
    nac, na = 3 * n, 4 * n
    row = 6 * 20 + 8 + 16 + 16 + 16           # slots, cross weight, centre, right-hand side, velocities
    if kind == "columns":
        # Aa and Ac layers in and out, neighbour weights of both grids, 2-D fields
        return {"bytes": n * (8.0 * NZ * 8 + 7 * 20 + 25 * 8) + nac * (8.0 * NZ * 3 + 13 * 8 + 16 + 24 * 8 + 44),
                "flops": n * NZ * 120.0 + nac * (NZ * 40.0 + 60.0)}
    if kind == "operators":
        return {"bytes": n * (8.0 * NZ * 13 + 7 * 48 + 6 * 8) + nac * (8.0 * NZ * 2 + 13 * 8 + 8 * 8) + na * (7 * 20 + 32.0),
                "flops": n * (NZ * 70.0 + 70.0) + nac * (NZ * 2.0 + 40.0) + na * 28.0}
    per = {"ssa": case.get("picard", 1), "step": case.get("picard", 1), "linear": 1,
           "adjoint": 3 * case.get("picard", 1), "batch": case.get("picard", 1)}[kind]
    # every system assembled (weights, viscosity, friction) and its matrix read once
    asm = 0 if kind == "linear" else 6 * 20 + 20 * 8
    return {"bytes": float(na) * per * (row + asm), "flops": float(na) * per * 60.0}


# ---------------------------------------------------------------------------
# exact
# ---------------------------------------------------------------------------
def exact(case, seed):
    """The explicit passes in 64-bit numpy.  The SSA solves end at a stopping
    rule of an iteration, which has no closed form to compare with."""
    f = globals().get("_exact_" + case["kind"])
    return f(case, seed) if f else None


def _slots(n, C):
    """Per neighbour slot: the rows that use it and their neighbours, 0-based."""
    for c in range(int(n.max())):
        rows = np.nonzero(n > c)[0]
        yield c, rows, C[rows, c] - 1


def _deriv(ma, d, weights=("Nx", "Ny")):
    """Neighbour-function derivatives of d (nV, or nV x layers) on the Aa mesh."""
    n, C = ma.mesh.nC, ma.mesh.C
    every = np.arange(ma.nV)
    w = [ma[k] for k in weights]
    col = (lambda a: a) if d.ndim == 1 else (lambda a: a[:, None])
    out = [col(a[every, n]) * d for a in w]
    for c, rows, vc in _slots(n, C):
        for o, a in zip(out, w):
            o[rows] += col(a[rows, c]) * d[vc]
    return out


def _deriv_Ac(ma, d):
    Aci = ma["Aci"] - 1
    x, y, o = (sum(ma[w][:, k] * d[Aci[:, k]] for k in range(4)) for w in ("Nx_Ac", "Ny_Ac", "No_Ac"))
    return x, y, ma["Np_Ac"] * (d[Aci[:, 1]] - d[Aci[:, 0]]), o


def _to_Aa(ma, d):
    n = ma.mesh.nC
    s = np.zeros((ma.nV,) + d.shape[1:])
    for c, rows, a in _slots(n, ma["iAci"]):
        s[rows] += d[a] / (n[rows] if d.ndim == 1 else n[rows, None])
    return s


def _neumann(d, n, C, edge, corners):
    """Edge points take the mean of their interior neighbours, then the corners of all theirs."""
    s, k = np.zeros_like(d), np.zeros(len(d))
    for _, rows, vc in _slots(n, C):
        inner = edge[vc] == 0
        s[rows[inner]] += d[vc[inner]]
        k[rows[inner]] += 1
    rows = (edge > 0) & ~corners
    d[rows] = s[rows] / (k[rows] if d.ndim == 1 else k[rows, None])
    for v in np.nonzero(corners)[0]:
        d[v] = d[C[v, :n[v]] - 1].mean(0)
    return d


def _neumann_Aa(ma, d):
    return _neumann(d, ma.mesh.nC, ma.mesh.C, ma.mesh.edge_index, np.arange(ma.nV) < 4)


def _rates(T):
    return np.where(T < 263.15, 1.14e-5 * np.exp(-6.0e4 / (8.314 * T)), 5.47e10 * np.exp(-13.9e4 / (8.314 * T)))


def _integral(f, z):
    """Integral of the layers of f from the bed up to each layer (negative)."""
    I = np.zeros_like(f)
    for k in range(len(z) - 2, -1, -1):
        I[:, k] = I[:, k + 1] - 0.5 * (f[:, k + 1] + f[:, k]) * (z[k + 1] - z[k])
    return I


def _mean(f, z):
    return (0.5 * (f[:, 1:] + f[:, :-1]) * np.diff(z)).sum(1)


def _exact_columns(case, seed):
    ri, rw, grav = 910.0, 1028.0, 9.81
    wl = _workload(case["sheet"], case["n"], seed, physics=1)
    ctx = abi.Context(0)
    ma = _secondary(ctx, case["sheet"], case["n"])
    ctx.close()
    p, z, mesh = wl.params, np.asarray(wl.params.zeta), wl.mesh
    V, n, edge = mesh.V, mesh.nC, mesh.edge_index
    us = 100.0 * geometry.gaussian_field(V, 80e3, seed + 4)
    vs = 100.0 * geometry.gaussian_field(V, 80e3, seed + 5)
    H, Hb, SL, T = wl.Hi, wl.Hb, wl.SL, wl.temperature()
    vi, vj = ma["Aci"][:, 0] - 1, ma["Aci"][:, 1] - 1

    def floating(h, b, s):
        return h < (s - b) * rw / ri

    # general update and physical properties
    Hs = H + np.maximum(SL - ri / rw * H, Hb)
    ocean = floating(H, Hb, SL)
    sheet, shelf = (H > 0) & ~ocean, (H > 0) & ocean
    hx, hy = _deriv(ma, H)
    sx, sy = _deriv(ma, Hs)
    HA, HbA, SLA = (0.5 * (d[vi] + d[vj]) for d in (H, Hb, SL))
    sheetA = (HA > 0) & ~floating(HA, HbA, SLA)
    sxA, syA, spA, soA = _deriv_Ac(ma, Hs)
    A = _rates(T)
    Am = np.where(sheet, _mean(A, z), _rates((T[:, 0] + 271.15) / 2))
    AA = _rates(0.5 * (T[vi] + T[vj]))
    # SIA
    D3 = (ri * grav * HA) ** 3 * (spA ** 2 + soA ** 2)
    D3 = D3[:, None] * 2.0 * HA[:, None] * _integral(p.m_enh_sia * AA * z ** 3, z)
    Dm = np.where(sheetA, _mean(np.maximum(D3, -1e5), z), 0.0)
    U_SIA, V_SIA, D_SIA = _to_Aa(ma, Dm * sxA), _to_Aa(ma, Dm * syA), _to_Aa(ma, HA * Dm)
    # 3-D velocities
    P = (ri * grav * H) ** 3 * (sx ** 2 + sy ** 2)
    P = np.maximum(P[:, None] * 2.0 * H[:, None] * _integral(p.m_enh_sia * A * z ** 3, z), -1e5)
    P = np.where(((~shelf) & (H != 0))[:, None], P, 0.0)
    U3 = _neumann_Aa(ma, P * sx[:, None] + us[:, None])
    V3 = _neumann_Aa(ma, P * sy[:, None] + vs[:, None])
    Ux, Uy = _deriv(ma, U3)
    Vx, Vy = _deriv(ma, V3)
    W = np.zeros_like(U3)
    W[:, -1] = U3[:, -1] * (sx - hx) + V3[:, -1] * (sy - hy)
    Hc = np.maximum(0.1, H)
    for k in range(len(z) - 2, -1, -1):
        dz, zm = z[k + 1] - z[k], 0.5 * (z[k + 1] + z[k])
        div = (Ux[:, k] + Ux[:, k + 1]) / 2 + (Vy[:, k] + Vy[:, k + 1]) / 2
        div = div + (sx - zm * hx) / Hc * (U3[:, k + 1] - U3[:, k]) / dz + (sy - zm * hy) / Hc * (V3[:, k + 1] - V3[:, k]) / dz
        W[:, k] = W[:, k + 1] - H * div * dz
    W[(edge > 0) | ~sheet] = 0.0
    W = _neumann_Aa(ma, W)
    # critical time steps
    dist = np.hypot(V[vj, 0] - V[vi, 0], V[vj, 1] - V[vi, 1])
    r, speed = np.sqrt(ma["A"] / np.pi), np.abs(us) + np.abs(vs)
    dts = [np.min(dist ** 2 / (-6 * np.pi * (HA * Dm - float(np.float32(1e-9))))),
           min(np.min(dist / speed[vi]), np.min(dist / speed[vj]), np.min(r / speed)),
           np.min(r[:, None] / (np.abs(U3) + np.abs(V3)))]
    dts = [0.9 * min(1000.0, float(d)) for d in dts]
    # mass continuity: upwind fluxes over the connections, out-fluxes limited to the ice there is
    dt, area = 0.5, ma["A"]
    Up = Dm * spA
    flux = np.zeros((ma.nV, mesh.nC_mem))
    where = {}
    for c, rows, a in _slots(n, ma["iAci"]):
        from_i = vi[a] == rows
        where[c] = (rows, a, from_i)
        up = np.where(Up[a] > 0, H[vi[a]], H[vj[a]])
        # a connection's width is that of its first vertex
        first, second = np.where(from_i, rows, vi[a]), np.where(from_i, vj[a], rows)
        slot = np.argmax(mesh.C[first] == (second + 1)[:, None], axis=1)
        q = up * Up[a] * ma["Cw"][first, slot] * dt
        flux[rows, c] = np.where(from_i, -q, q)
    smb = (wl.SMB + wl.BMB) * area * dt
    have = area * H
    gone = -smb >= have
    smb = np.where(gone, -have, smb)
    out = -np.minimum(flux, 0.0).sum(1)
    scale = np.where(gone, 0.0, 1.0)
    over = out > have + smb
    scale[over] = (have[over] + smb[over]) / out[over]
    total = np.zeros(ma.nV)
    for c, (rows, a, from_i) in where.items():
        other = np.where(from_i, vj[a], vi[a])
        q = flux[rows, c]
        total[rows] += q * np.where(q < 0, np.minimum(scale[rows], 1.0), np.minimum(scale[other], 1.0))
    dH = (total + smb) / (area * dt)
    Hn = H + dH * dt
    Hn[edge > 0] = 0.0
    flat = lambda a: np.ravel(a, order="F")  # noqa: E731
    return {"Hi": Hn, "dHi_dt": dH, "Hs": Hs, "U_SIA": U_SIA, "V_SIA": V_SIA, "D_SIA": D_SIA, "A_flow_mean": Am,
            "U_3D": flat(U3), "V_3D": flat(V3), "W_3D": flat(W), "mask": None, "dt_crit": dts}


def _exact_operators(case, seed):
    ctx = abi.Context(0)
    ma = _secondary(ctx, case["sheet"], case["n"])
    ctx.close()
    h = _operator_inputs(case, seed, ma)
    layers = lambda a: a.reshape(NZ, -1).T  # noqa: E731
    flat = lambda a: np.ravel(a, order="F")  # noqa: E731
    aa3, ac3 = layers(h["aa3"]), layers(h["ac3"])
    vi, vj = ma["Aci"][:, 0] - 1, ma["Aci"][:, 1] - 1
    out = dict(zip(("dx", "dy"), _deriv(ma, h["aa"])))
    out.update(zip(("dxx", "dxy", "dyy"), _deriv(ma, h["aa"], ("Nxx", "Nxy", "Nyy"))))
    out.update((k, flat(v)) for k, v in zip(("dx3", "dy3"), _deriv(ma, aa3)))
    out.update(zip(("dx_Ac", "dy_Ac", "dp_Ac", "do_Ac"), _deriv_Ac(ma, h["aa"])))
    n, C, d = ma["nCAaAc"], ma["CAaAc"], h["aaac"]
    every = np.arange(ma.nVAaAc)
    for name, w in (("dx_AaAc", ma["Nx_AaAc"]), ("dy_AaAc", ma["Ny_AaAc"])):
        out[name] = w[every, n] * d
        for c, rows, vc in _slots(n, C):
            out[name][rows] += w[rows, c] * d[vc]
    out["to_Ac"] = flat(0.5 * (aa3[vi] + aa3[vj]))
    out["to_Aa"] = flat(_to_Aa(ma, ac3))
    e = ma.mesh.V[vj] - ma.mesh.V[vi]
    e = e / np.hypot(e[:, 0], e[:, 1])[:, None]
    out["p"] = h["ac"] * e[:, 0] + h["bc"] * e[:, 1]
    out["o"] = h["bc"] * e[:, 0] - h["ac"] * e[:, 1]
    out["upx"] = out["upy"] = None
    out["neu3"] = flat(_neumann_Aa(ma, aa3.copy()))
    edge = np.concatenate([ma.mesh.edge_index, ma["edge_index_Ac"]])
    out["neu_AaAc"] = _neumann(d.copy(), n, C, edge, every < 4)
    out["missing"] = None
    return out


def _exact_remap(case, seed):
    s = prepare(case, seed)
    w = s["ctx"].remap_export()
    d = _remap_inputs(case, seed).reshape(NZ, -1).T
    dx, dy = _deriv(_built["marine", case["n_src"]], d)
    H = _workload("marine", case["n_src"], seed).Hi

    def conservative(f, fx=None, fy=None):
        v = w["vi"] - 1
        t = f[v] * w["w0"][:, None]
        if fx is not None:
            t = t + fx[v] * w["w1x"][:, None] + fy[v] * w["w1y"][:, None]
        out = np.zeros((len(w["start"]), t.shape[1]))
        for k in range(int((w["end"] - w["start"]).max(initial=0))):
            rows = np.nonzero(w["end"] - w["start"] > k)[0]
            out[rows] += t[w["start"][rows] + k]
        return out

    flat = lambda a: np.ravel(a, order="F")  # noqa: E731
    first = conservative(d)
    Hd = conservative(H[:, None])[:, 0]
    return {"trilin": flat(sum(d[w["tvi"][:, k] - 1] * w["tw"][:, k:k + 1] for k in range(3))),
            "nearest_neighbour": flat(d[w["nn"] - 1]), "cons_1st_order": flat(first),
            "cons_2nd_order": flat(conservative(d, dx, dy)), "Hi": Hd, "Hi_prev": Hd, "Ti": flat(first)}
