"""The forms of the single-system BiCGStab (one block, fused point Jacobi, block Jacobi, two-colour and general
ILU(0)) and of GMRES, at the sizes where each changes: the row-scaled residual of the returned solution against the Jacobian on the host."""
import numpy as np
import pytest

import cases
import vfvm
from vfvm.grids import linspace, simplexgrid

pytestmark = pytest.mark.gpu

RTOL = 1e-9


def _system(name):
    """system and time step (small where the point Jacobi iteration would be long)"""
    kind, *n = name.split(":")
    n = [int(v) for v in n]
    if kind == "dd2d":
        return cases.drift_diffusion_2d(n[0], lambda2=1.0)[0], 1e-4
    g = simplexgrid(*[linspace(0, 1, v) for v in n])
    ns = 2 if kind == "exchange" else 1
    d = 1.0 / max(v - 1 for v in n) ** 2  # with a time step of 1: diagonally dominant
    data = dict(flux=vfvm.LinearFlux([d, 2 * d][:ns]), storage=vfvm.IdentityStorage())
    if ns == 2:
        data["reaction"] = vfvm.ExchangeReaction(0.5)
    return cases.pair(g, ns, data, [vfvm.Dirichlet(1, 1, 0.3)], oracle=False)[0], 1.0


@pytest.mark.parametrize("name", ["grid:2", "grid:3", "grid:65", "grid:32:32", "grid:1025", "grid:2049", "grid:45:45",
                                  "grid:9:9:9", "grid:50:50", "grid:3072", "grid:3073", "grid:70:70", "grid:6144", "grid:6145",
                                  "grid:129:129", "grid:65:65:65", "grid:70001:3", "exchange:17:9", "dd2d:9"])
@pytest.mark.parametrize("precon", ["jacobi", "blockjacobi", "ilu0"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_solution_meets_the_tolerance(name, precon, precision):
    print("bicgstab", name, precon, precision, flush=True)
    _check(name, precon, precision, krylov="bicgstab")


@pytest.mark.parametrize("name", ["grid:2", "grid:65", "grid:127:129", "grid:181:181", "grid:181:182", "exchange:17:9",
                                  "dd2d:9"])
@pytest.mark.parametrize("precon", ["jacobi", "blockjacobi", "ilu0"])
@pytest.mark.parametrize("precision,restart", [("fp64", 1), ("fp64", 7), ("fp64", 64), ("fp32", 30)])
def test_gmres_meets_the_tolerance(name, precon, precision, restart):
    """restarts after 1, 7, 30 and 64 columns; 128 blocks and more are the two ways of summing the dot products"""
    print("gmres", name, precon, precision, restart, flush=True)
    if restart == 1 and name.startswith("dd2d"):
        restart = 2
    _check(name, precon, precision, krylov="gmres", gmres_restart=restart)


def _check(name, precon, precision, **kw):
    sys, tstep = _system(name)
    if name.startswith("dd2d") and precon == "ilu0":
        precon = "ilu0_natural"  # the multicolour factor of this system is no preconditioner
    rng = np.random.default_rng(7)
    U = vfvm.unknowns(sys, inival=0.5)
    U = U + 0.1 * rng.uniform(-1, 1, np.shape(U))
    F, A = vfvm.evaluate_residual_and_jacobian(sys, U, tstep=tstep)
    b = vfvm.dofs(F) + rng.uniform(-1, 1, vfvm.dofs(F).size)
    A = A.tocsr()
    s = 1.0 / A.diagonal()
    b = b / np.abs(s)  # comparable rows, also where a Dirichlet penalty stands
    kw.update(precon=precon, precision=precision, reltol_linear=RTOL, abstol_linear=0.0, maxiters_linear=2000)
    for _ in range(2):  # the second call starts from the first one's iteration count
        x, st = vfvm.linsolve(sys, b, **kw)
        x = vfvm.dofs(x)
        res = np.linalg.norm(s * (b - A @ x))
        # the recursive residual meets RTOL; the true one differs by the rounding of the updates of x and r
        drift = 8 * (st["iters"] + 1) * np.finfo(float).eps * np.linalg.norm((abs(A) @ np.abs(x)) * np.abs(s))
        bound = RTOL * np.linalg.norm(s * b) + drift
        print("iters", st["iters"], "residual / bound", res / bound, flush=True)
        assert res <= 1.001 * bound


def test_unusable_diagonal_is_an_error():
    """a row of zeros ends the two-colour solve as a breakdown, not with a finite answer"""
    g = simplexgrid(linspace(0, 1, 9))
    sys, _ = cases.pair(g, 1, dict(flux=vfvm.LinearFlux(0.0), storage=vfvm.IdentityStorage()), [], oracle=False)
    U = vfvm.unknowns(sys, inival=0.5)
    vfvm.evaluate_residual_and_jacobian(sys, U)  # stationary: no entry of the Jacobian is left
    with pytest.raises(vfvm.LinearSolverError):
        vfvm.linsolve(sys, np.ones(g.num_nodes), precon="ilu0", reltol_linear=1e-8, maxiters_linear=50)
