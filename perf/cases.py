"""Performance cases: what users of this package have it do, through its public entry points.

Each case is a dict of plain values with a "kind":

  newton    one stationary Newton solve of the 2D nonlinear Poisson problem (vfvm.solve)
  bias      a bias continuation of the 2D bipolar drift-diffusion system (solve(embed=...))
  euler     one implicit-Euler step of 3D nonlinear diffusion (solve(times=...))
  ode       right-hand side and Jacobian of the same 3D system for an outside time
            integrator, on device memory (eval_rhs_device, eval_jacobian_device)
  batch     many independent 2D systems of uneven size solved together (Batch.solve)
  guess     a learned initial guess and the batched Newton solve that starts from it
            (Surrogate.predict_sides_device, Batch.solve_device)
  infer     the learned initial guess alone
  train     loss and gradient of the network on one minibatch (Surrogate.loss_grad)
  sweep     small-signal impedance over a range of frequencies (ImpedanceSystem.impedances)

prepare() builds what a program holds before the call (systems, batches, networks, inputs),
run() is one pass, exact() the same answer from plain torch in 64 bits.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "voronoifvm.jl_amd"))

import vfvm  # noqa: E402
from vfvm import surrogate  # noqa: E402

# ------------------------------------------------------------------------------ the cases


def listed():
    return [
        # the smallest solve: one 33 x 33 system of the uneven family with the default
        # solver (BiCGStab, point Jacobi, FP64): launches and host reads count
        dict(name="newton_33_jacobi", kind="newton", n=33, precon="jacobi", precision="fp64", krylov="bicgstab"),
        # the reference's own CPU-sized problem: 101 x 101, ILU(0)
        dict(name="newton_101_ilu0", kind="newton", n=101, precon="ilu0", precision="fp64", krylov="bicgstab"),
        # a large single 2D system, multigrid inside FP32 refinement, odd size
        dict(name="newton_513_amg", kind="newton", n=513, precon="amg", precision="fp32", krylov="bicgstab"),
        # the configured solver of the drift-diffusion sweep at test size: GMRES(30) with
        # 3 x 3 block Jacobi
        dict(name="bias_49_gmres", kind="bias", n=49, krylov="gmres", precision="fp64"),
        # three coupled species on an ordinary grid, two bias steps
        dict(name="bias_129_bicgstab", kind="bias", n=129, krylov="bicgstab", precision="fp64"),
        # the largest single system: 2.1 million unknowns, FP32 Krylov inside FP64 Newton
        dict(name="euler_129_fp32", kind="euler", n=129, precon="ilu0", precision="fp32"),
        # residual and Jacobian assembly of that system for an outside integrator
        dict(name="ode_129", kind="ode", n=129),
        # uneven members, Jacobi, FP64: the form with one launch per Krylov step
        dict(name="batch_64_uneven", kind="batch", count=64, nmax=257, precision="fp64"),
        # the headline workload: 512 systems of 129 x 129 from the learned guess
        dict(name="guess_512", kind="guess", count=512, n=129),
        # one sample through the network, as an interactive solve asks for it
        dict(name="infer_1", kind="infer", count=1, n=129),
        # one minibatch of the network's training, at the training script's batch size
        dict(name="train_16", kind="train", count=16, n=129),
        # Example150's sweep on a 2D grid: 113 frequencies over five decades
        dict(name="sweep_257_113", kind="sweep", n=257, count=113),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["newton", "newton", "bias", "euler", "ode", "batch", "guess", "infer", "train", "sweep"])
    if kind == "newton":
        n = _log_int(rng, 17, 513)
        krylov = rng.choice(["bicgstab", "bicgstab", "gmres"]) if n <= 101 else "bicgstab"
        precon = "ilu0" if krylov == "gmres" else rng.choice(["jacobi", "ilu0", "amg"] if n <= 257 else ["ilu0", "amg"])
        return dict(kind=kind, n=n, precon=precon, precision=rng.choice(["fp64", "fp32"]), krylov=krylov)
    if kind == "bias":
        krylov = rng.choice(["bicgstab", "bicgstab", "gmres"])
        return dict(kind=kind, n=_log_int(rng, 33, 65 if krylov == "gmres" else 161), krylov=krylov,
                    precision=rng.choice(["fp64", "fp32"]) if krylov == "bicgstab" else "fp64")
    if kind == "euler":
        return dict(kind=kind, n=_log_int(rng, 17, 129), precon=rng.choice(["ilu0", "jacobi"]),
                    precision=rng.choice(["fp64", "fp32"]))
    if kind == "ode":
        return dict(kind=kind, n=_log_int(rng, 17, 129))
    if kind == "batch":
        return dict(kind=kind, count=_log_int(rng, 3, 64), nmax=rng.choice([65, 129, 257]),
                    precision=rng.choice(["fp64", "fp32"]))
    if kind == "guess":
        return dict(kind=kind, count=_log_int(rng, 8, 512), n=rng.choice([65, 97, 129]))
    if kind == "infer":
        return dict(kind=kind, count=_log_int(rng, 1, 128), n=_log_int(rng, 65, 193))
    if kind == "train":
        return dict(kind=kind, count=_log_int(rng, 2, 24), n=_log_int(rng, 65, 129))
    return dict(kind=kind, n=_log_int(rng, 33, 257), count=_log_int(rng, 2, 113))


def work(case):
    """Bytes: the inputs read and the outputs written once; for a Newton solve also one Jacobian
    written, read and solved with per step (the usual number of steps of the problem), without
    the passes over vectors, whose number depends on the linear solver.  Flops: one product
    with the matrix per step, or the network's matrix products."""
    k, n = case["kind"], case["n"] if "n" in case else 0
    if k == "newton":
        N = n * n
        return dict(bytes=6 * (5 * N * 8 + 4 * N * 8) + 3 * N * 8, flops=6 * 5 * N * 2)
    if k == "bias":
        N = 3 * n * n
        return dict(bytes=3 * 5 * (13 * N * 8 + 4 * N * 8) + 4 * N * 8, flops=3 * 5 * 13 * N * 2)
    if k == "euler":
        N = n ** 3
        return dict(bytes=4 * (7 * N * 8 + 5 * N * 8) + 2 * N * 8, flops=4 * 7 * N * 2)
    if k == "ode":
        N = n ** 3
        return dict(bytes=(2 * 8 + 8) * N + 7 * N * 8, flops=2 * 7 * N * 8)
    if k == "batch":
        N = case["count"] * (case["nmax"] / 2.0) ** 2
        return dict(bytes=7 * (5 * N * 8 + 4 * N * 8) + 3 * N * 8, flops=7 * 5 * N * 2)
    if k == "guess":
        N = case["count"] * n * n
        return dict(bytes=4 * (5 * N * 8 + 4 * N * 8) + 3 * N * 8, flops=N * _NET_FLOPS)
    if k == "infer":
        N = case["count"] * n * n
        return dict(bytes=2 * N * 8, flops=N * _NET_FLOPS)
    if k == "train":
        N = case["count"] * n * n
        return dict(bytes=9 * N * 4, flops=3 * N * _NET_FLOPS)
    N = n * n
    return dict(bytes=case["count"] * N * 16 + 6 * N * 8, flops=case["count"] * N * 5 * 4)


_NET_FLOPS = 2 * (16 * 64 + 4 * 128 * 64 + 64)  # per row of the 4-layer network


def tolerance(case):
    k = case["kind"]
    if k in ("newton", "euler", "batch"):
        # Newton stops at an update of 1e-10 of the first one; its error is then the linear
        # tolerance (1e-4) times that
        return dict(rel=1e-12)
    if k == "bias":
        # the same stop, on a system whose densities and potentials differ in scale
        return dict(rel=1e-11)
    if k == "ode":
        return dict(rel=1e-14, max=1e-12)
    if k == "sweep":
        # a relative residual of 1e-12 times the condition of the scaled operator
        return dict(rel=1e-7)
    # bfloat16 operands: sums in another order move some activations to the neighbouring
    # bfloat16 value (3e-4 in the output and the gradient)
    return dict(rel=2e-3, max=0.15)


# ------------------------------------------------------------------------------ device memory


class _Device:
    """A float64 torch tensor on the GPU as the device entry points take it."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.n = tensor.numel()
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


def _device(a):
    return _Device(torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64)).cuda())


def _device_empty(n):
    return _Device(torch.zeros(int(n), dtype=torch.float64, device="cuda"))


# ------------------------------------------------------------------------------ inputs


def _square(n):
    X = vfvm.linspace(0.0, 1.0, n)
    return vfvm.simplexgrid(X, X)


_GRF = {}


def _random_field(n, rng, ell=0.1, amp=5.0):
    """Gaussian random field with squared-exponential covariance on n x n nodes (x fastest)."""
    if n not in _GRF:
        x = np.arange(n) / (n - 1)
        w, Q = np.linalg.eigh(np.exp(-((x[:, None] - x[None, :]) ** 2) / (2 * ell * ell)))
        _GRF[n] = Q * np.sqrt(np.clip(w, 0.0, None))
    L = _GRF[n]
    return (amp * (L @ rng.standard_normal((n, n)) @ L.T)).ravel(order="F")


def _newton_inputs(case, seed):
    rng = np.random.default_rng([seed, 1])
    return _random_field(case["n"], rng), rng.uniform(-1.0, 1.0, 4)


def _samples(case, seed, salt):
    rng = np.random.default_rng([seed, salt])
    F = np.stack([_random_field(case["n"], rng) for _ in range(case["count"])])
    return F, rng.uniform(-1.0, 1.0, (case["count"], 4))


def _bias_inputs(seed):
    return float(np.random.default_rng([seed, 2]).uniform(0.8, 1.2))


def _euler_inputs(case, seed):
    rng = np.random.default_rng([seed, 3])
    x = np.arange(case["n"]) / (case["n"] - 1)
    k = np.arange(1, 6)
    S = np.sin(np.pi * np.outer(x, k))
    c = rng.standard_normal((5, 5, 5)) / (k[:, None, None] ** 2 + k[None, :, None] ** 2 + k[None, None, :] ** 2)
    u = np.einsum("kji,zk,yj,xi->zyx", c, S, S, S, optimize=True)
    u[[0, -1]] = 0.0
    u[:, [0, -1]] = 0.0
    u[:, :, [0, -1]] = 0.0
    return 0.5 * u / np.abs(u).max()


def _ode_inputs(case, seed):
    u = _euler_inputs(case, seed)
    return u + 0.3 + 0.1 * np.random.default_rng([seed, 9]).standard_normal(u.shape)


def _batch_members(case, seed):
    """N from the family's sizes up to nmax, eps log-uniform in [1e-3, 1], side values in
    [-1, 1], a constant source in [-5, 5]."""
    rng = np.random.default_rng([seed, 4])
    sizes = [s for s in (33, 65, 129, 257) if s <= case["nmax"]]
    shape = np.random.default_rng([case["count"], case["nmax"]])  # the members' sizes belong to the case
    return [(int(shape.choice(sizes)), float(10.0 ** rng.uniform(-3.0, 0.0)), rng.uniform(-1.0, 1.0, 4),
             float(rng.uniform(-5.0, 5.0))) for _ in range(case["count"])]


def _sweep_inputs(case, seed):
    rng = np.random.default_rng([seed, 5])
    return float(rng.uniform(0.5, 2.0)), float(rng.uniform(0.5, 2.0)), 1e-3 * 5e4 ** (np.arange(case["count"]) / 113.0)


EPS = 1e-2  # diffusion of the Poisson family with random sources


def _poisson(grid, f, values, eps):
    return vfvm.System(grid, vfvm.Physics(
        flux=vfvm.LinearFlux(eps), reaction=vfvm.SinhReaction(), source=np.asfortranarray(f.reshape(1, -1)),
        bcondition=[vfvm.Dirichlet(species=1, region=r + 1, value=float(v)) for r, v in enumerate(values)]), species=[1])


# systems that a program builds once and keeps while its inputs (start values, sources) change
_KEPT = {}


def _diffusion3d(n, robin):
    """u_t = div((1 + u^2) grad u) on the cube: u = 0 on its faces, or a flux u through them."""
    if ("diffusion", n, robin) not in _KEPT:
        X = vfvm.linspace(0.0, 1.0, n)
        bcs = [vfvm.Robin(species=1, region=r, factor=1.0, value=0.0) if robin else
               vfvm.Dirichlet(species=1, region=r, value=0.0) for r in range(1, 7)]
        ph = vfvm.Physics(flux=vfvm.NonlinearDiffusionFlux(1.0, 1.0), storage=vfvm.IdentityStorage(), bcondition=bcs)
        s = vfvm.System(vfvm.simplexgrid(X, X, X), ph, species=[1])
        s.autotune()
        _KEPT["diffusion", n, robin] = s
    return _KEPT["diffusion", n, robin]


def _network(n, training=False):
    """The trained network on an n x n grid (its weights belong to the 129 x 129 family); a
    program that trains and one that asks for guesses each have their own."""
    if ("network", n, training) not in _KEPT:
        net = surrogate.Surrogate(_poisson(_square(n), np.zeros(n * n), np.zeros(4), EPS))
        net.load()
        _KEPT["network", n, training] = net
    return _KEPT["network", n, training]


def _family(n, count):
    key = ("family", n)
    if len(_KEPT.get(key, [])) < count:
        grid = _square(n)
        _KEPT[key] = [_poisson(grid, np.zeros(n * n), np.zeros(4), EPS) for _ in range(count)]
        for s in _KEPT[key]:
            s.handle()
    return _KEPT[key][:count]


def prepare(case, seed):
    k = case["kind"]
    if k == "newton":
        f, v = _newton_inputs(case, seed)
        s = _poisson(_square(case["n"]), f, v, EPS)
        s.handle()
        c = vfvm.SolverControl(krylov=case["krylov"], precon=case["precon"], precision=case["precision"],
                               abstol_linear=0.0, maxiters_linear=3000, gmres_restart=30,
                               inner_reltol=1e-4 if case["precon"] == "amg" else 1e-2)
        return dict(kind=k, system=s, control=c)
    if k == "bias":
        s, u0 = _drift_diffusion(case["n"], _bias_inputs(seed))
        s.handle()
        c = vfvm.SolverControl(krylov=case["krylov"], precon="blockjacobi", precision=case["precision"],
                               abstol_linear=0.0, maxiters_linear=6000, inner_reltol=1e-2, max_refinements=12,
                               gmres_restart=30, Δp=0.05, Δp_min=0.05, Δp_max=0.05, Δu_opt=10.0)
        return dict(kind=k, system=s, control=c, u0=u0)
    if k == "euler":
        s = _diffusion3d(case["n"], False)
        c = vfvm.SolverControl(krylov="bicgstab", precon=case["precon"], precision=case["precision"], abstol_linear=0.0,
                               maxiters_linear=3000, inner_reltol=1e-2, max_refinements=10)
        u0 = np.asfortranarray(_euler_inputs(case, seed).reshape(1, -1))
        return dict(kind=k, system=s, control=vfvm.fixed_timesteps(c, 1e-2), u0=u0)
    if k == "ode":
        s = _diffusion3d(case["n"], True)
        ndof, nnz, _ = s.sizes()
        return dict(kind=k, system=s, u=_device(_ode_inputs(case, seed)), du=_device_empty(ndof),
                    jac=_device_empty(nnz))
    if k == "batch":
        systems = [_poisson(_square(n), np.full(n * n, f), v, eps) for n, eps, v, f in _batch_members(case, seed)]
        c = vfvm.SolverControl(krylov="bicgstab", precon="jacobi", precision=case["precision"], abstol_linear=0.0,
                               maxiters_linear=3000, inner_reltol=1e-2, max_refinements=12, check_every=8)
        return dict(kind=k, batch=vfvm.Batch(systems), control=c)
    if k == "guess":
        F, V = _samples(case, seed, 6)
        batch = vfvm.Batch(_family(case["n"], case["count"]))
        batch.set_member_solver(1024)
        for m in range(case["count"]):
            batch.update_member(m, source=np.asfortranarray(F[m].reshape(1, -1)), bcondition=surrogate.bcs(V[m]))
        c = vfvm.SolverControl(precision="fp32", precon="amg", abstol_linear=0.0, maxiters_linear=3000,
                               inner_reltol=1e-4, max_refinements=12, check_every=1)
        return dict(kind=k, batch=batch, control=c, net=_network(case["n"]), F=_device(F), V=_device(V),
                    guess=_device_empty(F.size), u=_device_empty(F.size), count=case["count"])
    if k == "infer":
        F, V = _samples(case, seed, 7)
        return dict(kind=k, net=_network(case["n"]), F=_device(F), V=_device(V), guess=_device_empty(F.size),
                    count=case["count"])
    if k == "train":
        X, T = _train_inputs(case, seed)
        return dict(kind=k, net=_network(case["n"], training=True), X=X, T=T)
    D, R, omegas = _sweep_inputs(case, seed)
    s = vfvm.System(_square(case["n"]), vfvm.Physics(flux=vfvm.LinearFlux(D), reaction=vfvm.PowerReaction(m=1, k=R),
                                                     storage=vfvm.IdentityStorage()), species=[1])
    s.boundary_dirichlet(1, 4, 1.0)
    s.boundary_dirichlet(1, 2, 0.0)
    U0 = vfvm.solve(s, inival=0.0, control=vfvm.SolverControl(reltol_linear=1e-12, abstol_linear=0.0,
                                                              maxiters_linear=20000, precon="ilu0"))
    T = vfvm.testfunction(s, [4], [2])
    ds, dt = vfvm.measurement_derivatives(s, U0, T, 1)
    return dict(kind=k, isys=vfvm.ImpedanceSystem(s, U0, 1, 4), omegas=omegas, ds=ds, dt=dt)


def run(state):
    k = state["kind"]
    if k == "newton":
        return vfvm.solve(state["system"], inival=0.0, control=state["control"])
    if k == "bias":
        return vfvm.solve(state["system"], inival=state["u0"], control=state["control"], embed=[0.0, 0.05, 0.1]).u
    if k == "euler":
        return vfvm.solve(state["system"], inival=state["u0"], control=state["control"], times=[0.0, 1e-2],
                          store_all=False).u[-1]
    if k == "ode":
        state["system"].eval_rhs_device(state["u"], state["du"])
        state["system"].eval_jacobian_device(state["u"], state["jac"])
        return dict(rhs=state["du"].tensor, jacobian=state["jac"].tensor)
    if k == "batch":
        U = state["batch"].solve(0.0, state["control"])
        return np.concatenate([vfvm.dofs(u) for u in U])
    if k == "guess":
        state["net"].predict_sides_device(state["F"], state["V"], state["guess"], state["count"])
        state["batch"].solve_device(state["u"], state["guess"], state["control"])
        return dict(guess=state["guess"].tensor, solution=state["u"].tensor)
    if k == "infer":
        state["net"].predict_sides_device(state["F"], state["V"], state["guess"], state["count"])
        return state["guess"].tensor
    if k == "train":
        loss, grad = state["net"].loss_grad(state["X"], state["T"])
        return dict(loss=float(loss), grad=grad)
    return state["isys"].impedances(state["omegas"], state["ds"], state["dt"])


# ------------------------------------------------------------------------------ problems


def _drift_diffusion(n, doping, lambda2=1e-4):
    grid = _square(n)
    C = np.where(grid.coord[0] < 0.5, doping, -doping)
    src = np.zeros((3, grid.num_nodes), order="F")
    src[0] = C
    bcs = []
    for region, c, bias in ((4, doping, 0.0), (2, -doping, 1.0)):
        nn = 0.5 * (c + math.sqrt(c * c + 4.0))
        bcs += [vfvm.Dirichlet(species=1, region=region, value=math.asinh(c / 2.0), value_lambda=bias),
                vfvm.Dirichlet(species=2, region=region, value=nn),
                vfvm.Dirichlet(species=3, region=region, value=1.0 / nn)]
    s = vfvm.System(grid, vfvm.Physics(flux=vfvm.DriftDiffusionFlux(lambda2, -1.0, 1.0),
                                       reaction=vfvm.DriftDiffusionReaction(1.0), source=src, bcondition=bcs),
                    species=[1, 2, 3])
    return s, _equilibrium(C)


def _equilibrium(C):
    U = np.zeros((3, C.size), order="F")
    U[0] = np.arcsinh(C / 2.0)
    U[1] = 0.5 * (C + np.sqrt(C * C + 4.0))
    U[2] = 1.0 / U[1]
    return U


def _train_inputs(case, seed):
    """Features and targets of a minibatch; targets near the solutions' size and smoothness."""
    F, V = _samples(case, seed, 8)
    n = case["n"]
    X = surrogate.Features(_square(n))(F, V)
    T = np.arcsinh(F / 2.0) * 0.8
    return X, np.ascontiguousarray(T, dtype=np.float32)


# ------------------------------------------------------------------------------ 64-bit answers


def _dst(m):
    k = torch.arange(1, m + 1, dtype=torch.float64, device="cuda")
    S = math.sqrt(2.0 / (m + 1)) * torch.sin(math.pi / (m + 1) * k[:, None] * k[None, :])
    return S, 2.0 - 2.0 * torch.cos(math.pi / (m + 1) * k)


def _poisson_solution(n, eps, F, V):
    """Nodal solutions (B x n^2) of eps, sources F (B x n^2) and side values V (B x 4): Newton
    with sine-transform preconditioned CG on the interior."""
    F = torch.as_tensor(np.asarray(F, dtype=np.float64)).cuda().reshape(-1, n, n)
    V = torch.as_tensor(np.asarray(V, dtype=np.float64)).cuda().reshape(-1, 4)
    eps = torch.as_tensor(np.asarray(eps, dtype=np.float64)).cuda().reshape(-1, 1, 1)
    B, m, h2 = F.shape[0], n - 2, 1.0 / (n - 1) ** 2
    u = torch.zeros(B, n, n, dtype=torch.float64, device="cuda")
    south, east, north, west = (V[:, j, None] for j in range(4))
    u[:, 0, :], u[:, -1, :], u[:, :, -1], u[:, :, 0] = south, north, east, west
    for iy, ix, a, b in ((0, 0, 0, 3), (0, -1, 0, 1), (-1, -1, 1, 2), (-1, 0, 2, 3)):
        u[:, iy, ix] = 0.5 * (V[:, a] + V[:, b])  # a corner carries both sides' penalties
    S, lam = _dst(m)
    lam2 = lam[:, None] + lam[None, :]

    def laplace(w):
        return 4.0 * w[:, 1:-1, 1:-1] - w[:, :-2, 1:-1] - w[:, 2:, 1:-1] - w[:, 1:-1, :-2] - w[:, 1:-1, 2:]

    def dot(a, b):
        return (a * b).sum((1, 2), keepdim=True)

    f = F[:, 1:-1, 1:-1]
    for _ in range(60):
        ui = u[:, 1:-1, 1:-1]
        res = eps * laplace(u) + h2 * (torch.exp(ui) - torch.exp(-ui) - f)
        c = h2 * (torch.exp(ui) + torch.exp(-ui))
        cm = torch.exp(torch.log(c).mean((1, 2), keepdim=True))
        x = torch.zeros_like(res)
        r = res.clone()
        z = S @ ((S @ r @ S) / (eps * lam2 + cm)) @ S
        p, rz, r0 = z.clone(), dot(r, z), dot(r, r)
        for _ in range(300):
            Ap = eps * laplace(torch.nn.functional.pad(p, (1, 1, 1, 1))) + c * p
            a = torch.where(rz > 0, rz / dot(p, Ap).clamp_min(1e-300), torch.zeros_like(rz))
            x += a * p
            r -= a * Ap
            if bool((dot(r, r) <= 1e-20 * r0).all()):
                break
            z = S @ ((S @ r @ S) / (eps * lam2 + cm)) @ S
            rz, old = dot(r, z), rz
            p = z + torch.where(old > 0, rz / old.clamp_min(1e-300), torch.zeros_like(rz)) * p
        u[:, 1:-1, 1:-1] -= x
        if float(x.abs().max()) < 1e-12:
            break
    return u.reshape(B, n * n)


def _euler_solution(n, u0, dt=1e-2):
    """One implicit-Euler step of u_t = div((1 + u^2) grad u): iteration with the sine-transform
    inverse of the operator at a mean coefficient."""
    uo = torch.as_tensor(u0).cuda().reshape(n, n, n)
    u, h, m = uo.clone(), 1.0 / (n - 1), n - 2
    S, lam = _dst(m)
    lam3 = lam[:, None, None] + lam[None, :, None] + lam[None, None, :]
    mean = 1.0 + 0.5 * float(uo.abs().max()) ** 2
    for _ in range(200):
        r = torch.zeros_like(u)
        for d in range(3):
            a, b = u.narrow(d, 0, n - 1), u.narrow(d, 1, n - 1)
            g = h * (1.0 + (0.5 * (a + b)) ** 2) * (a - b)
            r.narrow(d, 0, n - 1).add_(g)
            r.narrow(d, 1, n - 1).sub_(g)
        r += h ** 3 / dt * (u - uo)
        x = r[1:-1, 1:-1, 1:-1]
        for d in range(3):
            x = torch.tensordot(S, x, dims=([1], [d])).movedim(0, d)
        x = x / (h * mean * lam3 + h ** 3 / dt)
        for d in range(3):
            x = torch.tensordot(S, x, dims=([1], [d])).movedim(0, d)
        u[1:-1, 1:-1, 1:-1] -= x
        if float(x.abs().max()) < 1e-15:
            break
    return u.reshape(1, -1)


def _ode_answer(n, u0):
    """-F and -dF/du of the 3D system at u0, the Jacobian in row-major order of the 7-point
    pattern; the boundary flux is u times the node's measure on each of the six faces."""
    u = torch.as_tensor(u0).cuda().reshape(n, n, n)
    h = 1.0 / (n - 1)
    one = torch.full((n,), h, dtype=torch.float64, device="cuda")
    one[0] = one[-1] = 0.5 * h
    F = torch.zeros_like(u)
    J = torch.zeros(n, n, n, 7, dtype=torch.float64, device="cuda")
    keep = torch.zeros(n, n, n, 7, dtype=torch.bool, device="cuda")
    keep[..., 3] = True
    for d in range(3):  # z, y, x: columns 0/6, 1/5, 2/4
        e = [one, one, one]
        e[d] = torch.ones(n - 1, dtype=torch.float64, device="cuda") / h
        fac = e[0][:, None, None] * e[1][None, :, None] * e[2][None, None, :]
        a, b = u.narrow(d, 0, n - 1), u.narrow(d, 1, n - 1)
        mid, dif = 0.5 * (a + b), a - b
        D = 1.0 + mid ** 2
        F.narrow(d, 0, n - 1).add_(fac * D * dif)
        F.narrow(d, 1, n - 1).sub_(fac * D * dif)
        J[..., 3].narrow(d, 0, n - 1).add_(fac * (D + mid * dif))
        J[..., 3].narrow(d, 1, n - 1).add_(fac * (D - mid * dif))
        J[..., 6 - d].narrow(d, 0, n - 1).copy_(fac * (-D + mid * dif))
        J[..., d].narrow(d, 1, n - 1).copy_(-fac * (D + mid * dif))
        keep[..., 6 - d].narrow(d, 0, n - 1).fill_(True)
        keep[..., d].narrow(d, 1, n - 1).fill_(True)
    face = one[:, None] * one[None, :]
    for d in range(3):
        for k in (0, n - 1):
            J[..., 3].select(d, k).add_(face)
            F.select(d, k).add_(face * u.select(d, k))
    return dict(rhs=-F.reshape(-1), jacobian=-J[keep])


def _bernoulli(x):
    """B(x) = x / (e^x - 1) and B'(x)."""
    small = x.abs() < 1e-2
    xs = torch.where(small, torch.ones_like(x), x)
    em = torch.expm1(xs)
    B = torch.where(small, 1 - x / 2 + x ** 2 / 12 - x ** 4 / 720, xs / em)
    dB = torch.where(small, -0.5 + x / 6 - x ** 3 / 180, (em - xs * (em + 1)) / em ** 2)
    return B, dB


def _bias_answer(n, doping, lambda2=1e-4, biases=(0.0, 0.05, 0.1)):
    """Newton with block elimination over the grid's columns (blocks of 3 n unknowns)."""
    dev = dict(dtype=torch.float64, device="cuda")
    h = 1.0 / (n - 1)
    x = np.tile(np.arange(n) / (n - 1), n)
    C = np.where(x < 0.5, doping, -doping)
    # u[ix, iy, species]: blocks are grid columns (fixed x), coupled to the next column only
    u = torch.as_tensor(np.ascontiguousarray(_equilibrium(C).reshape(3, n, n).transpose(2, 1, 0))).cuda()
    Cd = torch.as_tensor(C.reshape(n, n).T.copy()).cuda()
    wt = torch.ones(n, **dev)
    wt[0] = wt[-1] = 0.5
    vol = h * h * wt[:, None] * wt[None, :]
    out = []

    def flux(a, b):
        """fluxes a -> b and their 3 x 3 derivatives with respect to a and b"""
        dp = a[..., 0] - b[..., 0]
        g = torch.zeros_like(a)
        da, db = (torch.zeros(*a.shape, 3, **dev) for _ in range(2))
        g[..., 0] = lambda2 * dp
        da[..., 0, 0], db[..., 0, 0] = lambda2, -lambda2
        for i, z in ((1, -1.0), (2, 1.0)):
            bp, dbp = _bernoulli(z * dp)
            bm, dbm = _bernoulli(-z * dp)
            g[..., i] = bm * a[..., i] - bp * b[..., i]
            s = -z * dbm * a[..., i] - z * dbp * b[..., i]
            da[..., i, 0], db[..., i, 0] = s, -s
            da[..., i, i], db[..., i, i] = bm, -bp
        return g, da, db

    for bias in biases:
        for ix, c, lam in ((0, doping, 0.0), (n - 1, -doping, bias)):
            nn = 0.5 * (c + math.sqrt(c * c + 4.0))
            u[ix] = torch.tensor([math.asinh(c / 2.0) + lam, nn, 1.0 / nn], **dev)
        for _ in range(40):
            psi, ne, po = u[..., 0], u[..., 1], u[..., 2]
            den = ne + po + 2.0
            R = (ne * po - 1.0) / den
            F = torch.stack([vol * (ne - po - Cd), vol * R, vol * R], dim=-1)
            Dg = torch.zeros(n, n, 3, 3, **dev)
            Dg[..., 0, 1], Dg[..., 0, 2] = vol, -vol
            for i in (1, 2):
                Dg[..., i, 1], Dg[..., i, 2] = vol * (po - R) / den, vol * (ne - R) / den
            gx, xa, xb = flux(u[:-1], u[1:])
            w = wt[None, :, None]
            F[:-1] += w * gx
            F[1:] -= w * gx
            Dg[:-1] += w[..., None] * xa
            Dg[1:] -= w[..., None] * xb
            up, lo = w[..., None] * xb, -w[..., None] * xa
            gy, ya, yb = flux(u[:, :-1], u[:, 1:])
            w = wt[:, None, None]
            F[:, :-1] += w * gy
            F[:, 1:] -= w * gy
            Dg[:, :-1] += w[..., None] * ya
            Dg[:, 1:] -= w[..., None] * yb
            A = torch.zeros(n, n, 3, n, 3, **dev)
            k = torch.arange(n, device="cuda")
            A[:, k, :, k, :] = Dg.permute(1, 0, 2, 3)
            A[:, k[:-1], :, k[1:], :] = (w[..., None] * yb).permute(1, 0, 2, 3)
            A[:, k[1:], :, k[:-1], :] = (-w[..., None] * ya).permute(1, 0, 2, 3)
            A = A.reshape(n, 3 * n, 3 * n)
            # interior columns 1 .. n-2 (the first and last hold the contacts)
            Us = torch.zeros(n - 1, n, 3, n, 3, **dev)
            Us[:, k, :, k, :] = up.permute(1, 0, 2, 3)
            Ls = torch.zeros(n - 1, n, 3, n, 3, **dev)
            Ls[:, k, :, k, :] = lo.permute(1, 0, 2, 3)
            Us, Ls = Us.reshape(n - 1, 3 * n, 3 * n), Ls.reshape(n - 1, 3 * n, 3 * n)
            G, y = [None] * n, [None] * n
            for i in range(1, n - 1):
                M, b = A[i], F[i].reshape(-1, 1)
                if i > 1:
                    M, b = M - Ls[i - 1] @ G[i - 1], b - Ls[i - 1] @ y[i - 1]
                s = torch.linalg.solve(M, torch.cat([Us[i], b], dim=1))
                G[i], y[i] = s[:, :-1], s[:, -1:]
            d = torch.zeros_like(u)
            nxt = None
            for i in range(n - 2, 0, -1):
                nxt = y[i] if nxt is None else y[i] - G[i] @ nxt
                d[i] = nxt.reshape(n, 3)
            u = u - d
            if float(d.abs().max()) < 1e-12:
                break
        out.append(u.permute(2, 1, 0).reshape(3, n * n).clone())
    return out


def _graph_mean(y, n):
    """sum_j w_ij y_j with the edge factors (1, 1/2 along the boundary) normalised per node;
    y is ... x n x n x channels"""
    w = torch.ones(n, dtype=torch.float64, device=y.device)
    w[0] = w[-1] = 0.5
    wx, wy = w[:, None, None], w[None, :, None]  # factors of x edges by row, of y edges by column
    s, t = torch.zeros_like(y), torch.zeros(n, n, 1, dtype=torch.float64, device=y.device)
    s[..., :, :-1, :] += wx * y[..., :, 1:, :]
    s[..., :, 1:, :] += wx * y[..., :, :-1, :]
    t[:, :-1] += wx
    t[:, 1:] += wx
    s[..., :-1, :, :] += wy * y[..., 1:, :, :]
    s[..., 1:, :, :] += wy * y[..., :-1, :, :]
    t[:-1] += wy
    t[1:] += wy
    return s / t


def _net_weights():
    th = torch.as_tensor(np.load(surrogate.WEIGHTS, allow_pickle=False)["params"].astype(np.float64)).cuda()
    p, shapes = 0, [(16, 64), (64,)] + [(128, 64), (64,)] * 4 + [(64,), (1,)]
    out = []
    for s in shapes:
        q = int(np.prod(s))
        out.append(th[p:p + q].reshape(s).clone())
        p += q
    return out


def _net_inputs(n, x8):
    """The 8 features and the 8 context channels, B x n x n x 16."""
    y = torch.stack([x8[..., 1], x8[..., 0]], dim=-1)
    ctx = []
    for step in range(1, 325):
        y = 0.5 * (y + _graph_mean(y, n))
        if step in (16, 64, 160, 324):
            ctx.append(y)
    return torch.cat([x8] + [c[..., :1] for c in ctx] + [c[..., 1:] for c in ctx], dim=-1)


def _net(W, n, x16):
    h = torch.relu(x16 @ W[0] + W[1])
    for l in range(4):
        a = _graph_mean(h, n) - h
        h = h + torch.relu(torch.cat([h, a], dim=-1) @ W[2 + 2 * l] + W[3 + 2 * l])
    return h @ W[10] + W[11]


def _guess_answer(n, F, V):
    x = torch.arange(n, dtype=torch.float64, device="cuda") / (n - 1)
    X, Y = x[None, :].expand(n, n), x[:, None].expand(n, n)
    delta = math.sqrt(EPS / 2.0)
    decay = torch.stack([torch.exp(-d / delta) for d in (Y, 1.0 - X, 1.0 - Y, X)], dim=-1)
    W, out = _net_weights(), []
    for s0 in range(0, F.shape[0], 16):
        f = torch.as_tensor(F[s0:s0 + 16]).cuda().reshape(-1, n, n)
        v = torch.as_tensor(V[s0:s0 + 16]).cuda()
        x8 = torch.cat([(f / 5.0)[..., None], torch.asinh(f / 2.0)[..., None], v[:, None, None, :] * decay,
                        X.expand_as(f)[..., None], Y.expand_as(f)[..., None]], dim=-1)
        out.append(_net(W, n, _net_inputs(n, x8)).reshape(-1))
    return torch.cat(out)


def _train_answer(n, X, T):
    W = [w.requires_grad_(True) for w in _net_weights()]
    total = float(T.size)
    loss = 0.0
    for s in range(X.shape[0]):
        x8 = torch.as_tensor(X[s:s + 1]).cuda().double().reshape(1, n, n, 8)
        t = torch.as_tensor(T[s:s + 1]).cuda().double().reshape(1, n, n)
        part = ((_net(W, n, _net_inputs(n, x8)) - t) ** 2).sum() / total
        part.backward()
        loss += float(part.detach())
    return dict(loss=loss, grad=torch.cat([w.grad.reshape(-1) for w in W]))


def _sweep_answer(n, D, R, omegas):
    """The problem is constant along y: one complex tridiagonal system per frequency."""
    h = 1.0 / (n - 1)
    vol = np.full(n, h)
    vol[0] = vol[-1] = 0.5 * h
    diag = (R + 1j * omegas[:, None]) * vol[None, :]  # frequency x node
    diag[:, :-1] += D / h
    diag[:, 1:] += D / h
    off = -D / h
    # interior nodes, u = 1 at the first node and 0 at the last: elimination and back substitution
    d, r = np.empty((omegas.size, n), dtype=np.complex128), np.zeros((omegas.size, n), dtype=np.complex128)
    u = np.zeros((omegas.size, n), dtype=np.complex128)
    u[:, 0] = 1.0
    d[:, 1], r[:, 1] = diag[:, 1], -off
    for i in range(2, n - 1):
        m = off / d[:, i - 1]
        d[:, i], r[:, i] = diag[:, i] - m * off, -m * r[:, i - 1]
    for i in range(n - 2, 0, -1):
        u[:, i] = (r[:, i] - off * u[:, i + 1]) / d[:, i]
    Au = diag * u
    Au[:, :-1] += off * u[:, 1:]
    Au[:, 1:] += off * u[:, :-1]
    T = np.arange(n) / (n - 1)  # the test function: 0 on the excited side, 1 on the measured one
    return -1.0 / (Au @ T)


def exact(case, seed):
    """What run() returns, from plain torch in 64 bits."""
    k = case["kind"]
    if k == "newton":
        f, v = _newton_inputs(case, seed)
        return _poisson_solution(case["n"], [EPS], f[None], v[None]).reshape(1, -1)
    if k == "bias":
        return _bias_answer(case["n"], _bias_inputs(seed))
    if k == "euler":
        return _euler_solution(case["n"], _euler_inputs(case, seed))
    if k == "ode":
        return _ode_answer(case["n"], _ode_inputs(case, seed))
    if k == "batch":
        members = _batch_members(case, seed)
        out = [None] * len(members)
        for n in set(m[0] for m in members):
            idx = [q for q, m in enumerate(members) if m[0] == n]
            u = _poisson_solution(n, [members[q][1] for q in idx],
                                  np.stack([np.full(n * n, members[q][3]) for q in idx]),
                                  np.stack([members[q][2] for q in idx]))
            for j, q in enumerate(idx):
                out[q] = u[j]
        return torch.cat(out)
    if k == "guess":
        F, V = _samples(case, seed, 6)
        return dict(guess=_guess_answer(case["n"], F, V),
                    solution=_poisson_solution(case["n"], [EPS], F, V).reshape(-1))
    if k == "infer":
        return _guess_answer(case["n"], *_samples(case, seed, 7))
    if k == "train":
        return _train_answer(case["n"], *_train_inputs(case, seed))
    return _sweep_answer(case["n"], *_sweep_inputs(case, seed))
