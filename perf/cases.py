"""The work this framework does for its users, as measurable cases.

A case is one call of a public entry point: a batched MPC solve
(TurboMPCSolver.solve: quadrotor, obstacle avoidance, point mass), one QP
solve (ADMMSolver.solve, direct and PCG Schur solves), a differentiable solve
with its gradients (get_differentiable_solve_function), or a block-tridiagonal
linear solve (make_schur_solver).  Sizes are those of the repository's own
configurations, benchmark and tests, and odd batches and horizons around
them.  exact() restates each path in 64-bit torch from the mathematics: the
ADMM iteration on the block-tridiagonal normal equations, the SQP loop, the
merit line search and the adjoint KKT system.
"""
from __future__ import annotations

import copy
import math

import torch

# ------------------------------------------------------------------- cases ----


def listed():
    return [
        # one robot in its control loop: a single quadrotor problem, the latency of 5 x 20 iterations
        dict(name="quadrotor_one", kind="quadrotor", B=1, N=40, dtype="f32", sqp=5, iters=20, linesearch=False,
             warm=False),
        # a receding-horizon tick of a small fleet: two SQP iterations from the previous tick's solution and state
        dict(name="quadrotor_tick", kind="quadrotor", B=48, N=30, dtype="f32", sqp=2, iters=20, linesearch=False,
             warm=True),
        # a sampled set of start states planned with the merit line search, ragged batch and horizon
        dict(name="quadrotor_linesearch", kind="quadrotor", B=611, N=33, dtype="f64", sqp=4, iters=20,
             linesearch=True, warm=False),
        # the benchmark's batch: 4096 quadrotors, 5 SQP x 20 ADMM
        dict(name="quadrotor_batch", kind="quadrotor", B=4096, N=40, dtype="f32", sqp=5, iters=20, linesearch=False,
             warm=False),
        # the largest: 16384 obstacle-avoidance problems, 8 SQP x 30 ADMM
        dict(name="obstacle_batch", kind="obstacle", B=16384, N=60, dtype="f32", sqp=8, iters=30, soft=False,
             linesearch=False),
        # soft obstacle rows (slack variables), an ordinary odd batch
        dict(name="obstacle_soft", kind="obstacle", B=501, N=47, dtype="f64", sqp=4, iters=30, soft=True,
             linesearch=False),
        # the solver's default parameters (adaptive rho, termination tests, relaxation 1.6) on point masses
        dict(name="pointmass_default", kind="pointmass", B=64, N=20, dtype="f64"),
        # one QP of random stable linear systems with bounds on every variable, direct Schur solve
        dict(name="lti_direct", kind="lti", B=1024, N=50, nx=12, nu=4, dtype="f32", schur="direct", iters=100),
        # the same family on the PCG Schur solve, the batch the benchmark names
        dict(name="lti_pcg", kind="lti", B=1024, N=50, nx=12, nu=4, dtype="f32", schur="pcg", iters=100),
        # learning the weights of a rendezvous controller: forward solve and gradients
        dict(name="spacecraft_grad", kind="spacecraft_grad", B=2048, N=100, dtype="f64", iters=200),
        # learning a quadrotor's weights on a training batch: SQP and the adjoint with exact Hessians
        dict(name="quadrotor_grad", kind="quadrotor_grad", B=128, N=40, dtype="f64", sqp=5, iters=20),
        # the Schur-level solver on its own: factorize and solve block-tridiagonal systems
        dict(name="schur_direct", kind="schur", B=512, T=51, n=16, dtype="f64"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["quadrotor", "quadrotor", "quadrotor", "obstacle", "obstacle", "pointmass", "lti", "lti",
                       "spacecraft_grad", "quadrotor_grad", "schur"])
    if kind == "quadrotor":
        ls = rng.random() < 0.25
        return dict(kind=kind, B=_log(rng, 1, 4096), N=rng.randint(15, 45), sqp=rng.randint(2, 5), iters=20,
                    dtype="f64" if ls or rng.random() < 0.3 else "f32", linesearch=ls,
                    warm=not ls and rng.random() < 0.4)
    if kind == "obstacle":
        ls = rng.random() < 0.25
        return dict(kind=kind, B=_log(rng, 4, 8192), N=rng.randint(20, 60), sqp=rng.randint(2, 6), iters=30,
                    dtype="f64" if ls or rng.random() < 0.3 else "f32", soft=rng.random() < 0.4, linesearch=ls)
    if kind == "pointmass":
        return dict(kind=kind, B=_log(rng, 1, 8192), N=rng.randint(10, 40), dtype="f64")
    if kind == "lti":
        schur = rng.choice(["direct", "pcg"])
        nx, nu = (12, 4) if schur == "pcg" or rng.random() < 0.5 else (rng.randint(8, 12), rng.randint(2, 4))
        return dict(kind=kind, B=_log(rng, 8, 1024 if schur == "pcg" else 2048), N=rng.randint(20, 60), nx=nx, nu=nu,
                    dtype=rng.choice(["f32", "f64"]), schur=schur, iters=rng.randint(40, 100))
    if kind == "spacecraft_grad":
        return dict(kind=kind, B=_log(rng, 16, 2048), N=rng.randint(40, 100), dtype="f64", iters=rng.randint(100, 200))
    if kind == "quadrotor_grad":
        return dict(kind=kind, B=_log(rng, 4, 200), N=rng.randint(15, 45), dtype="f64", sqp=rng.randint(3, 5), iters=20)
    return dict(kind="schur", B=_log(rng, 16, 2048), T=rng.randint(11, 101), n=rng.choice([6, 9, 12, 16, 17]),
                dtype=rng.choice(["f32", "f64"]))


# ------------------------------------------------------------------ inputs ----
QUAD = (1.0, 0.01, 0.01, 0.02, 0.15, 0.016, 9.81)  # mass, Jxx, Jyy, Jzz, arm, yaw coefficient, g
QUAD_DT = 0.02
HOVER = QUAD[0] * QUAD[6] / 4.0


def _dtype(case):
    return torch.float64 if case["dtype"] == "f64" else torch.float32


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _inputs(case, seed):
    """The problem's data, drawn in 64 bits from the seed and rounded to the
    case's type, as 64-bit tensors on the GPU."""
    g = torch.Generator().manual_seed(int(seed))
    B, kind = case["B"], case["kind"]
    rnd = lambda *s: torch.randn(s, generator=g, dtype=torch.float64)  # noqa: E731
    uni = lambda lo, hi, *s: lo + (hi - lo) * torch.rand(s, generator=g, dtype=torch.float64)  # noqa: E731
    d = {}
    if kind in ("quadrotor", "quadrotor_grad"):
        rv = 0.1 * rnd(B, 3)
        ang = rv.norm(dim=1, keepdim=True).clamp(min=1e-12)
        q0 = torch.cat([torch.cos(ang / 2), torch.sin(ang / 2) / ang * rv], dim=1)
        d["x0"] = torch.cat([0.3 * rnd(B, 3), q0, 0.3 * rnd(B, 3), torch.zeros(B, 3, dtype=torch.float64)], dim=1)
        xg = torch.zeros(B, 13, dtype=torch.float64)
        xg[:, :3] = uni(-2.0, 2.0, B, 3)
        xg[:, 3] = 1.0
        d["goal"] = xg
        d["wx"] = torch.tensor([10.0] * 3 + [1.0] * 4 + [1.0] * 3 + [0.1] * 3, dtype=torch.float64).expand(B, 13)
        d["wu"] = torch.full((B, 4), 0.01, dtype=torch.float64)
        d["wf"] = torch.zeros(B, 13, dtype=torch.float64)
        d["x0_next"] = d["x0"] + 0.02 * rnd(B, 13)  # the measured state of the next control tick
        if kind == "quadrotor_grad":
            d["wx"] = d["wx"] * uni(0.7, 1.4, B, 13)
            d["target"] = xg[:, None] + 0.3 * rnd(B, case["N"] + 1, 13)
    elif kind == "obstacle":
        K, dt = 8, 0.05
        I3, Z3 = torch.eye(3, dtype=torch.float64), torch.zeros(3, 3, dtype=torch.float64)
        d["A"] = torch.cat([torch.cat([I3, dt * I3], 1), torch.cat([Z3, I3], 1)], 0).expand(B, 6, 6)
        d["Bm"] = torch.cat([0.5 * dt * dt * I3, dt * I3], 0).expand(B, 6, 3)
        d["centers"], d["radii"] = uni(-3.0, 3.0, B, K, 3), uni(0.3, 0.8, B, K)
        axis = torch.randint(0, 3, (B,), generator=g)
        side = 2.0 * torch.randint(0, 2, (B,), generator=g).to(torch.float64) - 1.0
        start, goal = uni(-4.0, 4.0, B, 3), uni(-4.0, 4.0, B, 3)
        start[torch.arange(B), axis], goal[torch.arange(B), axis] = -4.0 * side, 4.0 * side
        z = torch.zeros(B, 3, dtype=torch.float64)
        d["x0"], d["goal"] = torch.cat([start, z], 1), torch.cat([goal, z], 1)
        d["wx"] = torch.tensor([1.0] * 3 + [0.1] * 3, dtype=torch.float64).expand(B, 6)
        d["wu"] = torch.full((B, 3), 0.01, dtype=torch.float64)
        d["wf"] = torch.tensor([10.0] * 3 + [1.0] * 3, dtype=torch.float64).expand(B, 6)
    elif kind == "pointmass":
        dt = 0.1
        I2, Z2 = torch.eye(2, dtype=torch.float64), torch.zeros(2, 2, dtype=torch.float64)
        d["A"] = torch.cat([torch.cat([I2, dt * I2], 1), torch.cat([Z2, I2], 1)], 0).expand(B, 4, 4)
        d["Bm"] = torch.cat([0.5 * dt * dt * I2, dt * I2], 0).expand(B, 4, 2)
        d["x0"] = uni(-1.0, 1.0, B, 4)
        d["wx"], d["wu"] = torch.ones(B, 4, dtype=torch.float64), torch.full((B, 2), 0.1, dtype=torch.float64)
        d["wf"] = torch.full((B, 4), 9.0, dtype=torch.float64)
    elif kind == "lti":
        nx, nu = case["nx"], case["nu"]
        A = torch.eye(nx, dtype=torch.float64) + 0.1 * rnd(B, nx, nx) / math.sqrt(nx)
        rad = torch.linalg.eigvals(A).abs().amax(dim=1)
        d["A"] = A * (1.05 / rad).clamp(max=1.0)[:, None, None]
        d["Bm"] = 0.1 * rnd(B, nx, nu)
        d["wx"], d["wu"], d["x0"] = uni(0.1, 10.0, B, nx), uni(0.01, 1.0, B, nu), rnd(B, nx)
        d["wf"] = torch.zeros(B, nx, dtype=torch.float64)
    elif kind == "spacecraft_grad":
        # Clohessy-Wiltshire relative motion, exact zero-order-hold discretization
        n, dt = 0.0011, 10.0
        M = torch.zeros(9, 9, dtype=torch.float64)
        M[0:3, 3:6] = torch.eye(3)
        M[3, 0], M[3, 4], M[4, 3], M[5, 2] = 3 * n * n, 2 * n, -2 * n, -n * n
        M[3:6, 6:9] = torch.eye(3)
        E = torch.linalg.matrix_exp(M * dt)
        d["A"], d["Bm"] = E[:6, :6].expand(B, 6, 6), E[:6, 6:].expand(B, 6, 3)
        d["wx"], d["wu"] = uni(1.0, 10.0, B, 6), uni(0.1, 1.0, B, 3)
        d["x0"] = rnd(B, 6) * torch.tensor([100.0] * 3 + [0.1] * 3, dtype=torch.float64)
        d["wf"] = torch.zeros(B, 6, dtype=torch.float64)
        d["target"] = 10.0 * rnd(B, case["N"] + 1, 6)
    else:  # schur: S = blockdiag(theta) with off-diagonal blocks, diagonally dominant as theta is
        T, n = case["T"], case["n"]
        M = rnd(B, T, n, n)
        phi = 0.4 * rnd(B, T - 1, n, n) / math.sqrt(n)
        S = torch.zeros(B, T, n, 3 * n, dtype=torch.float64)
        S[..., n:2 * n] = M @ M.transpose(-1, -2) / n + 3.0 * torch.eye(n, dtype=torch.float64)
        S[:, 1:, :, :n] = phi
        S[:, :-1, :, 2 * n:] = phi.transpose(-1, -2)
        d["S"], d["rhs"] = S, rnd(B, T, n)
    dt_, dev = _dtype(case), _device()
    return {k: v.contiguous().to(dev).to(dt_).double() for k, v in d.items()}


def _bounds(case):
    """(state bounds, control bounds) as lists, or None."""
    kind = case["kind"]
    if kind in ("quadrotor", "quadrotor_grad"):
        return None, ([0.0] * 4, [2.0 * HOVER] * 4)
    if kind == "obstacle":
        return None, ([-3.0] * 3, [3.0] * 3)
    if kind == "pointmass":
        return None, ([-1.0] * 2, [1.0] * 2)
    if kind == "spacecraft_grad":
        return None, ([-0.01] * 3, [0.01] * 3)
    return ([-5.0] * case["nx"], [5.0] * case["nx"]), ([-1.0] * case["nu"], [1.0] * case["nu"])


SOFT_WEIGHT = 100.0


def _program(case, d):
    """The optimal control problem object a user's program keeps."""
    from turbompc_amd.problems.obstacle import ObstacleOCP
    from turbompc_amd.problems.ocp import LinearOCP
    from turbompc_amd.problems.quadrotor import QuadrotorOCP

    dt, dev, kind = _dtype(case), _device(), case["kind"]
    T = case["N"] + 1
    c = {k: v.to(dt) for k, v in d.items()}
    xb, ub = _bounds(case)
    pair = lambda b: None if b is None else tuple(torch.tensor(v, dtype=torch.float64) for v in b)  # noqa: E731
    kw = dict(horizon=case["N"], initial_state=c["x0"], weights_state=c["wx"], weights_control=c["wu"],
              weights_final=c["wf"], state_bounds=pair(xb), control_bounds=pair(ub), dtype=dt, device=dev)
    if kind in ("quadrotor", "quadrotor_grad"):
        return QuadrotorOCP(dt=QUAD_DT, reference_state=c["goal"].unsqueeze(1).expand(-1, T, 13),
                            reference_control=torch.full((case["B"], T, 4), HOVER, dtype=torch.float64),
                            penalize_control_reference=True, initial_guess_final_state=c["goal"], **kw)
    kw.update(A=c["A"], Bm=c["Bm"], num_states=c["A"].shape[1], num_controls=c["Bm"].shape[2])
    if kind == "obstacle":
        return ObstacleOCP(reference_state=c["goal"].unsqueeze(1).expand(-1, T, 6), initial_guess_final_state=c["goal"],
                           obstacles_centers=c["centers"], obstacles_radii=c["radii"], obstacles_dimension=3,
                           use_slack_variables=case["soft"],
                           slack_penalization_weight=SOFT_WEIGHT if case["soft"] else 0.0, **kw)
    return LinearOCP(**kw)


def _params(case):
    """Solver parameters: the fixed-iteration protocol of the benchmark, or
    (point masses) the defaults."""
    from turbompc_amd.solvers.turbompc_solver import DEFAULT_SOLVER_PARAMS

    p = copy.deepcopy(DEFAULT_SOLVER_PARAMS)
    if case["kind"] != "pointmass":
        p["num_sqp_iteration_max"] = case.get("sqp", 1)
        p["tol_convergence"] = 0.0
        p["linesearch"] = bool(case.get("linesearch", False))
        p["admm"].update(max_iter=case["iters"], adapt_rho_every=0, relaxation_parameter=1.0)
    return p


def prepare(case, seed):
    from turbompc_amd.solvers.linear_systems_solvers.backends import AdmmBackend, SchurSolverBackend
    from turbompc_amd.solvers.linear_systems_solvers.schur_solver import SchurComplementMatrices, make_schur_solver

    d, dt = _inputs(case, seed), _dtype(case)
    if case["kind"] == "schur":
        schur = SchurComplementMatrices(S=d["S"].to(dt), preconditioner_Phiinv=None)
        solver = make_schur_solver(backend=SchurSolverBackend.HIP_DIRECT, horizon=case["T"] - 1, num_states=case["n"] - 1,
                                   num_controls=1, pcg_params={})
        return dict(kind="schur", solver=solver, schur=schur, rhs=d["rhs"].to(dt),
                    guess=torch.zeros_like(d["rhs"], dtype=dt))
    program = _program(case, d)
    if case["kind"] == "lti":
        from turbompc_amd.solvers.admm.admm import ADMMSolver
        from turbompc_amd.solvers.qp_utils import ZShape

        solver = ADMMSolver(ZShape(case["N"], case["nx"], case["nu"]), {"max_iter": 50, "tol_epsilon": 1e-6},
                            sigma=1e-6, max_iter=case["iters"], eps_abs=1e-30, eps_rel=1e-30,
                            check_termination_every=case["iters"] + 1, adapt_rho_every=0, rho_f_factor=1000.0,
                            admm_backend=AdmmBackend.HIP_PCG if case["schur"] == "pcg" else AdmmBackend.HIP_DIRECT,
                            std_dynamics=True, diag_cost=True, const_g=True)
        qp = program.build_qp(*program.initial_guess())
        return dict(kind="lti", solver=solver, qp=qp)
    from turbompc_amd.solvers.turbompc_solver import TurboMPCSolver

    solver = TurboMPCSolver(program, _params(case))
    guess = solver.initial_guess()
    if case["kind"] in ("spacecraft_grad", "quadrotor_grad"):
        weights = {"weights_penalization_reference_state_trajectory": d["wx"].to(dt),
                   "weights_penalization_control_squared": d["wu"].to(dt),
                   "weights_penalization_final_state": d["wf"].to(dt)}
        return dict(kind="grad", fn=solver.get_differentiable_solve_function(), guess=guess, x0=d["x0"].to(dt),
                    weights=weights, target=d["target"].to(dt))
    if case.get("warm"):
        guess = solver.solve(guess)  # the previous control tick's solution
        return dict(kind="solve", solver=solver, guess=guess, params={"initial_state": d["x0_next"].to(dt)})
    return dict(kind="solve", solver=solver, guess=guess, params=None)


def run(state):
    kind = state["kind"]
    if kind == "schur":
        x, _ = state["solver"].solve(state["schur"], state["rhs"], state["guess"])
        return {"x": x}
    if kind == "lti":
        (states, controls), _, st = state["solver"].solve(state["qp"], None, 0.1, 1.0)
        return {"states": states, "controls": controls, "y_g": st.y_g, "z_g": st.z_g, "y_f_0": st.y_f_0,
                "y_f_dyn": st.y_f_dyn}
    if kind == "grad":
        x0 = state["x0"].detach().requires_grad_(True)
        w = {k: v.detach().requires_grad_(True) for k, v in state["weights"].items()}
        sol = state["fn"](state["guess"], {"initial_state": x0}, w)
        loss = ((sol.states - state["target"]) ** 2).sum()
        keys = sorted(w)
        grads = torch.autograd.grad(loss, [x0] + [w[k] for k in keys])
        out = {"states": sol.states.detach(), "controls": sol.controls.detach(), "d_x0": grads[0]}
        out.update({"d_" + k: g for k, g in zip(keys, grads[1:])})
        return out
    sol = state["solver"].solve(state["guess"], state["params"])
    st = sol.admm_state
    return {"states": sol.states, "controls": sol.controls, "slack": sol.slack, "y_g": st.y_g, "z_g": st.z_g,
            "y_f_0": st.y_f_0, "y_f_dyn": st.y_f_dyn}


# -------------------------------------------------------- work and tolerance ----


def _dims(case):
    """(B, T, n, nx, m) of the case's QPs."""
    kind = case["kind"]
    nx, nu, m = {"quadrotor": (13, 4, 4), "quadrotor_grad": (13, 4, 4), "obstacle": (6, 3, 11), "pointmass": (4, 2, 2),
                 "spacecraft_grad": (6, 3, 3)}.get(kind) or (case["nx"], case["nu"], case["nx"] + case["nu"])
    return case["B"], case["N"] + 1, nx + nu, nx, m


def work(case):
    """bytes: the call's inputs and outputs once.  flops: per ADMM iteration
    the two triangular sweeps of the block-tridiagonal solve and the
    constraint products and their transposes, per QP one factorization (and
    per adjoint one of the KKT blocks); PCG iterations are counted as 20 per
    ADMM iteration (what its tolerance takes on these systems)."""
    w = 8 if case["dtype"] == "f64" else 4
    if case["kind"] == "schur":
        B, T, n = case["B"], case["T"], case["n"]
        return {"bytes": w * B * (T * n * n + (T - 1) * n * n + 2 * T * n),
                "flops": B * T * (2 * n ** 3 / 3 + 2 * n ** 3 + n ** 3 + 8 * n * n)}
    B, T, n, nx, m = _dims(case)
    data = 3 * nx + 2 * n  # start, goal, weights
    if case["kind"] == "obstacle":
        data += 8 * 4
    if "nx" in case or case["kind"] in ("obstacle", "pointmass", "spacecraft_grad"):
        data += nx * n  # the linear system
    if case["kind"] == "lti":  # its QP is the input
        data = T * (n * n + n + m * n + 2 * m) + (T - 1) * (n * nx + nx)
    state = T * n + 3 * T * m + T * nx  # x, z, y_g, xi, y_f
    byts = w * B * (data + T * n + state)
    if case.get("warm"):
        byts += w * B * state
    sqp = case.get("sqp", 1) if case["kind"] != "pointmass" else 2
    iters = case.get("iters", 100)
    factor = T * ((nx + m) * n * n + n ** 3 + 2 * nx * n * n)
    sweeps = 4 * T * n * n + 4 * T * nx * n
    if case.get("schur") == "pcg":
        sweeps = 20 * (4 * (3 * T - 2) * n * n + 10 * T * n)
    flops = B * sqp * (factor + iters * (sweeps + 4 * T * (nx + m) * n))
    if case["kind"].endswith("grad"):
        nb = n + nx + m
        flops += B * T * (2 * nb ** 3 + 6 * 4 * nb * nb)
        byts += w * B * (T * nx + 3 * nx + n)
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    # about four times the largest distance from exact() seen per family
    kind, f32 = case["kind"], case["dtype"] == "f32"
    if kind == "schur":
        return {"rel": 3e-6 if f32 else 1e-12}
    if kind == "lti" and case["schur"] == "pcg":
        # its Schur solves stop at a relative residual of 1e-6, possibly one iteration apart
        return {"rel": 1e-4 if f32 else 2e-5}
    if kind == "pointmass":
        return {"rel": 1e-6}  # adaptive rho is a ratio of residuals that cancel
    if kind == "spacecraft_grad":
        return {"rel": 0.03}  # a KKT system of condition 1e11: d_x0 is 0.02 from exact()
    if f32:
        return {"rel": 1e-4 if kind == "quadrotor" else 3e-5}
    return {"rel": 1e-9}


# ------------------------------------------------------------------- exact ----
# Batched 64-bit reference.  Stage t holds z_t = [x_t; u_t]; the QP is
#   min sum 1/2 z'Dz + q'z  s.t.  x_0 given, x_{t+1} = A_t z_t - c_t, l <= G z (+ xi) <= u
# with D diagonal here.  The ADMM works on S = D + sigma + rho_f C'C + rho G'G.


def _mv(A, v):
    return (A * v.unsqueeze(-2)).sum(-1)


def _mtv(A, v):
    return (A * v.unsqueeze(-1)).sum(-2)


def _inv_spd(M):
    """Inverse of a batch of SPD matrices by the Gauss-Jordan exchange."""
    M = M.clone()
    for k in range(M.shape[-1]):
        p = 1.0 / M[..., k, k]
        row = M[..., k, :] * p[..., None]
        col = M[..., :, k].clone()
        M = M - col[..., :, None] * row[..., None, :]
        M[..., k, :] = row
        M[..., :, k] = -col * p[..., None]
        M[..., k, k] = p
    return 0.5 * (M + M.transpose(-1, -2))


class _QP:
    def __init__(self, D, q, x0, A, c, G, l, u, gamma=None):
        self.D, self.q, self.x0, self.A, self.c, self.G, self.l, self.u, self.gamma = D, q, x0, A, c, G, l, u, gamma


class _State:
    def __init__(self, qp, rho):
        B, T, n = qp.q.shape
        nx, m = qp.A.shape[2], qp.G.shape[2]
        z = lambda *s: torch.zeros(s, dtype=torch.float64, device=qp.q.device)  # noqa: E731
        self.x, self.yg, self.xi = z(B, T, n), z(B, T, m), z(B, T, m)
        self.z = torch.minimum(torch.maximum(z(B, T, m), qp.l), qp.u)
        self.y0, self.yf = z(B, nx), z(B, T - 1, nx)
        self.rho = torch.full((B,), float(rho), dtype=torch.float64, device=qp.q.device)
        self.it = torch.zeros(B, dtype=torch.int64, device=qp.q.device)


def _theta(qp, rho, sigma, rho_f):
    B, T, n = qp.q.shape
    nx = qp.A.shape[2]
    th = torch.diag_embed(qp.D + sigma)
    th = th + rho[:, None, None, None] * (qp.G.transpose(-1, -2) @ qp.G)
    th[:, :-1] += rho_f[:, None, None, None] * (qp.A.transpose(-1, -2) @ qp.A)
    i = torch.arange(nx, device=th.device)
    th[:, :, i, i] += rho_f[:, None, None]
    return th


def _ct(qp, y0, yf):
    """C' y for the initial rows y0 and the dynamics rows yf."""
    nx = qp.A.shape[2]
    out = torch.zeros_like(qp.q)
    out[:, :-1] += _mtv(qp.A, yf)
    out[:, 0, :nx] += y0
    out[:, 1:, :nx] -= yf
    return out


class _Direct:
    """Block LDL' of S and its solves."""

    def __init__(self, qp, rho, sigma, rho_f):
        self.A, self.rf = qp.A, rho_f
        th = _theta(qp, rho, sigma, rho_f)
        T, nx = th.shape[1], qp.A.shape[2]
        self.inv = []
        for t in range(T):
            M = th[:, t]
            if t:
                A = qp.A[:, t - 1]
                M = M.clone()
                M[:, :nx, :nx] -= (rho_f ** 2)[:, None, None] * (A @ self.inv[-1] @ A.transpose(-1, -2))
            self.inv.append(_inv_spd(M))

    def solve(self, g, guess):
        T, nx, rf = g.shape[1], self.A.shape[2], self.rf[:, None]
        w = []
        for t in range(T):
            r = g[:, t]
            if t:
                r = r.clone()
                r[:, :nx] += rf * _mv(self.A[:, t - 1], w[-1])
            w.append(_mv(self.inv[t], r))
        for t in range(T - 2, -1, -1):
            w[t] = w[t] + _mv(self.inv[t], rf * _mtv(self.A[:, t], w[t + 1][:, :nx]))
        return torch.stack(w, dim=1)


class _Pcg:
    """Preconditioned CG on S with the stair preconditioner built from the
    stage blocks; each problem stops at |eta| < 1e-12 + eps |eta_0|."""

    def __init__(self, qp, rho, sigma, rho_f, eps=1e-6, most=50):
        self.A, self.rf, self.eps, self.most = qp.A, rho_f, eps, most
        self.th = _theta(qp, rho, sigma, rho_f)
        self.inv = _inv_spd(self.th)

    def _off(self, v):
        """The off-diagonal blocks of S applied to v."""
        nx, rf = self.A.shape[2], self.rf[:, None, None]
        out = torch.zeros_like(v)
        out[:, 1:, :nx] -= rf * _mv(self.A, v[:, :-1])
        out[:, :-1] -= rf * _mtv(self.A, v[:, 1:, :nx])
        return out

    def solve(self, g, guess):
        S = lambda v: _mv(self.th, v) + self._off(v)  # noqa: E731

        def M(r):  # an approximate inverse of -S
            v = _mv(self.inv, r)
            return -v + _mv(self.inv, self._off(v))
        dot = lambda a, b: (a * b).flatten(1).sum(1)  # noqa: E731
        k = lambda a: a[:, None, None]  # noqa: E731
        x = guess.clone()
        r = g - S(x)
        rt = M(r)
        p, eta = rt, dot(r, rt)
        eta0 = eta.abs()
        run_ = eta0 > 1e-12
        for it in range(self.most):
            if it:
                run_ = run_ & ~(eta.abs() < 1e-12 + self.eps * eta0)
            if it % 4 == 0 and not bool(run_.any()):
                break
            q = S(p)
            a = torch.where(run_, eta / dot(p, q), torch.zeros_like(eta))
            x, r = x + k(a) * p, r - k(a) * q
            rt = M(r)
            new = dot(r, rt)
            p = torch.where(k(run_), rt + k(new / eta) * p, p)
            eta = torch.where(run_, new, eta)
        return x


def _amax(*ts):
    out = 0.0
    for t in ts:
        if t.numel():
            out = torch.maximum(t.abs().flatten(1).amax(1), torch.as_tensor(out, dtype=t.dtype, device=t.device))
    return out


def _admm(qp, st, iters, *, alpha=1.0, sigma=1e-6, factor=1000.0, check=0, adapt=0, eps=1e-9, schur=_Direct,
          active=None):
    """iters ADMM iterations from st (in place); with check > 0 the
    termination test, and with adapt > 0 the adaptive rho, every that many."""
    nx = qp.A.shape[2]
    k3 = lambda a: a[:, None, None]  # noqa: E731
    live = torch.ones_like(st.rho, dtype=torch.bool) if active is None else active.clone()
    rp = rd = torch.full_like(st.rho, math.inf)
    sp = sd = torch.ones_like(st.rho)
    solver = None
    for it in range(iters):
        if check and it and it % check == 0:
            live = live & ((rp > eps + eps * sp) | (rd > eps + eps * sd))
            if not bool(live.any()):
                break
        rho, rf = st.rho, st.rho * factor
        if solver is None:
            solver = schur(qp, rho, sigma, rf)
        g = sigma * st.x - qp.q + _ct(qp, rf[:, None] * qp.x0 - st.y0, k3(rf) * qp.c - st.yf)
        g = g + _mtv(qp.G, k3(rho) * st.z - st.yg)
        xt = solver.solve(g, st.x)
        x = alpha * xt + (1 - alpha) * st.x
        cx = _mv(qp.A, xt[:, :-1]) - xt[:, 1:, :nx]
        y0 = st.y0 + rf[:, None] * alpha * (xt[:, 0, :nx] - qp.x0)
        yf = st.yf + k3(rf) * alpha * (cx - qp.c)
        zr = alpha * _mv(qp.G, xt) + (1 - alpha) * st.z
        zt = zr + st.yg / k3(rho)
        pr = torch.minimum(torch.maximum(zt, qp.l), qp.u)
        if qp.gamma is None:
            z, xi = pr, torch.zeros_like(pr)
        else:
            f = qp.gamma / (qp.gamma + k3(rho))
            z, xi = (1 - f) * zt + f * pr, (1 - f) * (pr - zt)
        yg = st.yg + k3(rho) * (zr - z)
        m3 = k3(live)
        pick = lambda a, b: torch.where(m3, a, b)  # noqa: E731
        st.x, st.z, st.xi, st.yg, st.yf = pick(x, st.x), pick(z, st.z), pick(xi, st.xi), pick(yg, st.yg), pick(yf, st.yf)
        st.y0 = torch.where(live[:, None], y0, st.y0)
        st.it = torch.where(live, torch.full_like(st.it, it + 1), st.it)
        if check and it % check == 0:
            rp_, rd_, sp_, sd_ = _residuals(qp, st)
            sel = lambda a, b: torch.where(live, a, b)  # noqa: E731
            rp, rd, sp, sd = sel(rp_, rp), sel(rd_, rd), sel(sp_, sp), sel(sd_, sd)
            if adapt and it >= 2 and it % adapt == 0:
                ratio = (rp / (1e-10 + sp)) / (rd / (1e-10 + sd))
                cand = (st.rho * ratio.sqrt()).clamp(1e-6, 1e6)
                turn = live & ((rp > eps + eps * sp) | (rd > eps + eps * sd))
                turn = turn & ~(torch.maximum(cand / st.rho, st.rho / cand) < 5.0)
                st.rho = torch.where(turn, cand, st.rho)
                if bool(turn.any()):
                    solver = None
    return st


def _residuals(qp, st):
    nx = qp.A.shape[2]
    cx = _mv(qp.A, st.x[:, :-1]) - st.x[:, 1:, :nx]
    c0 = st.x[:, 0, :nx]
    gx = _mv(qp.G, st.x)
    rp = _amax(c0 - qp.x0, cx - qp.c, gx - st.z)
    px = qp.D * st.x
    aty = _ct(qp, st.y0, st.yf) + _mtv(qp.G, st.yg)
    rd = _amax(px + qp.q + aty)
    sd = _amax(px, aty, qp.q)
    if qp.gamma is not None:
        rd = torch.maximum(rd, _amax(qp.gamma * st.xi + st.yg))
        sd = torch.maximum(sd, torch.maximum(qp.gamma * _amax(st.xi), _amax(st.yg)))
    return rp, rd, _amax(c0, qp.x0, cx, qp.c, gx, st.z), sd


def _quad_step(z):
    """The RK4 step of the rotor-thrust quadrotor, z (..., 17) real or complex."""
    mass, jx, jy, jz, arm, ky, g = QUAD
    dd = arm / math.sqrt(2.0)
    f = [z[..., 13 + k] for k in range(4)]
    F = f[0] + f[1] + f[2] + f[3]
    tx, ty = dd * (f[0] + f[1] - f[2] - f[3]), dd * (f[1] + f[2] - f[0] - f[3])
    tz = ky * (f[1] + f[3] - f[0] - f[2])

    def rate(x):
        _, _, _, qw, qx, qy, qz, vx, vy, vz, wx, wy, wz = x.unbind(-1)
        return torch.stack([
            vx, vy, vz, 0.5 * (-qx * wx - qy * wy - qz * wz), 0.5 * (qw * wx + qy * wz - qz * wy),
            0.5 * (qw * wy - qx * wz + qz * wx), 0.5 * (qw * wz + qx * wy - qy * wx),
            2.0 / mass * (qx * qz + qw * qy) * F, 2.0 / mass * (qy * qz - qw * qx) * F,
            1.0 / mass * (1.0 - 2.0 * (qx * qx + qy * qy)) * F - g,
            (tx - (jz - jy) * wy * wz) / jx, (ty - (jx - jz) * wz * wx) / jy, (tz - (jy - jx) * wx * wy) / jz], dim=-1)
    x, h = z[..., :13], QUAD_DT
    k1 = rate(x)
    k2 = rate(x + 0.5 * h * k1)
    k3 = rate(x + 0.5 * h * k2)
    k4 = rate(x + h * k3)
    return x + h / 6.0 * (k1 + 2.0 * k2 + 2.0 * k3 + k4)


def _quad_blocks(z):
    """A (B,N,13,17) by complex step, c (B,N,13) = A z - f at z (B,T,17)."""
    zn = z[:, :-1].to(torch.complex128)
    cols = []
    for j in range(17):
        zj = zn.clone()
        zj[..., j] += 1e-30j
        cols.append(_quad_step(zj).imag * 1e30)
    A = torch.stack(cols, dim=-1)
    return A, _mv(A, z[:, :-1]) - _quad_step(z[:, :-1])


class _Ocp:
    """The case's problem in 64 bits: qp_at(z) and the merit terms."""

    def __init__(self, case, d, x0=None):
        self.case, self.d, kind = case, d, case["kind"]
        B, T, n, nx, m = _dims(case)
        self.B, self.T, self.n, self.nx = B, T, n, nx
        dev = d["x0"].device
        self.x0 = d["x0"] if x0 is None else x0
        w = torch.cat([d["wx"], d["wu"]], 1).unsqueeze(1).repeat(1, T, 1)
        w[:, -1, :nx] += d["wf"]
        ref = torch.zeros(B, T, n, dtype=torch.float64, device=dev)
        if "goal" in d:
            ref[..., :nx] = d["goal"][:, None]
        self.quad = kind.startswith("quadrotor")
        dt = _dtype(case)
        if self.quad:
            ref[..., nx:] = torch.tensor(HOVER, dtype=dt).double()
        self.w, self.ref = w, ref
        xb, ub = _bounds(case)
        rows = (list(range(nx)) if xb else []) + list(range(nx, n))
        self.box = torch.tensor(rows, device=dev)
        lo = torch.tensor((xb[0] if xb else []) + ub[0], dtype=torch.float64).to(dt).double()
        hi = torch.tensor((xb[1] if xb else []) + ub[1], dtype=torch.float64).to(dt).double()
        self.lo, self.hi = lo.to(dev).expand(B, T, -1), hi.to(dev).expand(B, T, -1)
        G = torch.zeros(len(rows), n, dtype=torch.float64, device=dev)
        G[torch.arange(len(rows), device=dev), self.box] = 1.0
        self.G = G.expand(B, T, len(rows), n)
        self.obs = kind == "obstacle"
        self.gamma = SOFT_WEIGHT if case.get("soft") else None
        if not self.quad:
            self.A = torch.cat([d["A"], d["Bm"]], 2).unsqueeze(1).expand(B, T - 1, nx, n)

    def guess(self):
        N = self.T - 1
        t = torch.arange(N + 1, dtype=torch.float64, device=self.x0.device).view(1, -1, 1)
        end = self.d["goal"] if "goal" in self.d else self.x0
        s = self.x0[:, None] * ((N - t) / N) + end[:, None] * (t / N) + 1e-6
        return torch.cat([s, torch.full((self.B, N + 1, self.n - self.nx), 1e-6, dtype=torch.float64,
                                        device=s.device)], -1)

    def next(self, z):
        return _quad_step(z[:, :-1]) if self.quad else _mv(self.A, z[:, :-1])

    def rows(self, z):
        """(g, l, u) of the inequality rows at z."""
        g, lo, hi = z[..., self.box], self.lo, self.hi
        if self.obs:
            d = z[..., None, :3] - self.d["centers"][:, None]
            go = 1.0 - d.norm(dim=-1) / (self.d["radii"][:, None] + 0.001)
            g = torch.cat([g, go], -1)
            lo, hi = torch.cat([lo, torch.full_like(go, -1e9)], -1), torch.cat([hi, torch.zeros_like(go)], -1)
        return g, lo, hi

    def qp_at(self, z):
        A, c = _quad_blocks(z) if self.quad else (self.A, torch.zeros(self.B, self.T - 1, self.nx, dtype=torch.float64,
                                                                      device=z.device))
        G, lo, hi = self.G, self.lo, self.hi
        if self.obs:
            p = z[..., None, :3]
            d = p - self.d["centers"][:, None]
            nrm, den = d.norm(dim=-1, keepdim=True), (self.d["radii"][:, None] + 0.001)[..., None]
            grad = -d / nrm / den
            off = 1.0 - (nrm / den)[..., 0] - (grad * p).sum(-1)
            Go = torch.zeros(*grad.shape[:3], self.n, dtype=torch.float64, device=z.device)
            Go[..., :3] = grad
            G = torch.cat([G, Go], 2)
            lo, hi = torch.cat([lo, -1e9 - off], -1), torch.cat([hi, -off], -1)
        return _QP(2.0 * self.w, -2.0 * self.w * self.ref, self.x0, A, c, G, lo, hi, self.gamma)

    def merit(self, z, sl):
        """(cost, |constraint violation|_1)."""
        cost = (self.w * (z - self.ref) ** 2).flatten(1).sum(1)
        g, lo, hi = self.rows(z)
        if self.gamma is not None:
            cost = cost + 0.5 * self.gamma * (sl * sl).flatten(1).sum(1)
            g = g + sl
        h = (z[:, 0, :self.nx] - self.x0).abs().sum(1) + (self.next(z) - z[:, 1:, :self.nx]).abs().flatten(1).sum(1)
        v = (lo - g).clamp(min=0.0) + (g - hi).clamp(min=0.0)
        return cost, h + v.flatten(1).sum(1)

    def line(self, z, sl, z_new, sl_new):
        """The step length of each problem by the Armijo test on the l1 merit."""
        dz, ds = z_new - z, sl_new - sl
        cost, cl = self.merit(z, sl)
        dc = (2.0 * self.w * (z - self.ref) * dz).flatten(1).sum(1)
        if self.gamma is not None:
            dc = dc + self.gamma * (sl * ds).flatten(1).sum(1)
        mu = torch.nan_to_num(dc / (0.5 * cl.clamp(min=1e-8)), nan=0.1, posinf=1e6, neginf=0.1).clamp(0.1, 1e6)
        base, slope = cost + mu * cl, dc - mu * cl
        alphas = [0.1, 0.3, 0.7, 1.0]
        cand = []
        for a in alphas:
            ca, va = self.merit(z + a * dz, sl + a * ds)
            cand.append(ca + mu * va)
        out = torch.full_like(cost, -1.0)
        for a, m in zip(alphas, cand):
            out = torch.where(m <= base + 0.4 * a * slope, torch.full_like(out, a), out)
        least = torch.tensor(alphas, dtype=torch.float64, device=z.device)[torch.stack(cand, 1).argmin(1)]
        return torch.where(out > 0, out, least)


def _sqp(case, ocp, z, st=None, **kw):
    """The fixed-count SQP loop; returns (z, slack, state, last QP)."""
    sl = None
    for _ in range(case.get("sqp", 1)):
        qp = ocp.qp_at(z)
        if st is None:
            st = _State(qp, 0.1)
        if sl is None:
            sl = st.xi
        _admm(qp, st, case["iters"], check=0, **kw)
        zn, sn = st.x, st.xi
        if case.get("linesearch"):
            a = ocp.line(z, sl, zn, sn)[:, None, None]
            zn, sn = z + a * (zn - z), sl + a * (sn - sl)
        z, sl = zn, sn
    return z, sl, st, qp


def _sqp_default(ocp, z):
    """The SQP loop with the default parameters (linear dynamics)."""
    qp = ocp.qp_at(z)
    st = _State(qp, 0.1)
    live = torch.ones(ocp.B, dtype=torch.bool, device=z.device)
    for _ in range(15):
        _admm(qp, st, 100, alpha=1.6, check=25, adapt=25, active=live)
        stat = qp.D * st.x + qp.q + _ct(qp, st.y0, st.yf) + _mtv(qp.G, st.yg)
        g = _mv(qp.G, st.x)
        viol = torch.maximum((qp.l - g).clamp(min=0.0), (g - qp.u).clamp(min=0.0))
        cx = _mv(qp.A, st.x[:, :-1]) - st.x[:, 1:, :ocp.nx] - qp.c
        live = live & (_amax(stat, cx, st.x[:, 0, :ocp.nx] - qp.x0, viol) > 1e-6)
        if not bool(live.any()):
            break
    return st


def _adjoint(case, ocp, qp, st, dz):
    """(v, w0): the adjoint step and the multipliers of the initial rows, from
    the KKT system of the active constraints with the Lagrangian's Hessian."""
    B, T, n, nx = ocp.B, ocp.T, ocp.n, ocp.nx
    m = qp.G.shape[2]
    H = torch.diag_embed(qp.D)
    if ocp.quad:
        f = lambda z, y: (_quad_step(z) * y).sum()  # noqa: E731
        hess = torch.func.vmap(torch.func.jacfwd(torch.func.grad(f)), chunk_size=4096)
        H[:, :-1] += hess(st.x[:, :-1].reshape(-1, n), st.yf.reshape(-1, nx)).view(B, T - 1, n, n)
    g = _mv(qp.G, st.x)
    dl, du = g - qp.l, qp.u - g
    near = torch.minimum(dl, du) <= 1e-9 + 1e-9 * torch.where(du < dl, qp.u.abs(), qp.l.abs())
    act = (st.yg.abs() > 1e-9) | near
    K = torch.zeros(B, T, n + nx + m, n + nx + m, dtype=torch.float64, device=dz.device)
    K[..., :n, :n] = H
    i, j = torch.arange(nx, device=dz.device), torch.arange(m, device=dz.device)
    sign = torch.full((T, 1), -1.0, dtype=torch.float64, device=dz.device)
    sign[0] = 1.0
    K[:, :, n + i, i] = sign
    K[:, :, i, n + i] = sign
    Ga = qp.G * act[..., None]
    K[..., n + nx:, :n] = Ga
    K[..., :n, n + nx:] = Ga.transpose(-1, -2)
    K[:, :, n + nx + j, n + nx + j] = torch.where(act, 0.0, -1.0).to(torch.float64)
    K, A, dz = K.cpu(), qp.A.cpu(), dz.cpu()
    nb = n + nx + m
    rhs = torch.zeros(B, T, nb, dtype=torch.float64)
    rhs[..., :n] = dz

    def product(w):
        out = (K @ w.unsqueeze(-1)).squeeze(-1)
        out[:, 1:, n:n + nx] += (A @ w[:, :-1, :n, None]).squeeze(-1)
        out[:, :-1, :n] += (A.transpose(-1, -2) @ w[:, 1:, n:n + nx, None]).squeeze(-1)
        return out

    inv = []
    for t in range(T):
        M = K[:, t].clone()
        if t:
            a = A[:, t - 1]
            M[:, n:n + nx, n:n + nx] -= a @ inv[-1][:, :n, :n] @ a.transpose(-1, -2)
        inv.append(torch.linalg.inv(M))

    def solve(b):
        w = []
        for t in range(T):
            r = b[:, t].clone()
            if t:
                r[:, n:n + nx] -= (A[:, t - 1] @ w[-1][:, :n, None]).squeeze(-1)
            w.append((inv[t] @ r.unsqueeze(-1)).squeeze(-1))
        for t in range(T - 2, -1, -1):
            r = torch.zeros(B, nb, dtype=torch.float64)
            r[:, :n] = (A[:, t].transpose(-1, -2) @ w[t + 1][:, n:n + nx, None]).squeeze(-1)
            w[t] = w[t] - (inv[t] @ r.unsqueeze(-1)).squeeze(-1)
        return torch.stack(w, dim=1)

    w = solve(rhs)
    for _ in range(2):
        w = w + solve(rhs - product(w))
    return w[..., :n].to(qp.D.device), w[:, 0, n:n + nx].to(qp.D.device)


def exact(case, seed):
    d, kind = _inputs(case, seed), case["kind"]
    if kind == "schur":
        S, r, n = d["S"], d["rhs"], case["n"]
        inv, w = [], []
        for t in range(case["T"]):
            M, b = S[:, t, :, n:2 * n], r[:, t]
            if t:
                phi = S[:, t, :, :n]
                M = M - phi @ inv[-1] @ phi.transpose(-1, -2)
                b = b - _mv(phi, w[-1])
            inv.append(_inv_spd(M))
            w.append(_mv(inv[-1], b))
        for t in range(case["T"] - 2, -1, -1):
            w[t] = w[t] - _mv(inv[t], _mv(S[:, t, :, 2 * n:], w[t + 1]))
        return {"x": torch.stack(w, 1)}
    ocp = _Ocp(case, d)
    nx = ocp.nx
    z = ocp.guess()
    if kind == "lti":
        qp = ocp.qp_at(z)
        st = _admm(qp, _State(qp, 0.1), case["iters"], schur=_Pcg if case["schur"] == "pcg" else _Direct)
        return {"states": st.x[..., :nx], "controls": st.x[..., nx:], "y_g": st.yg, "z_g": st.z, "y_f_0": st.y0,
                "y_f_dyn": st.yf}
    if kind == "pointmass":
        st = _sqp_default(ocp, z)
        z, sl = st.x, st.xi
    else:
        # the solver's relaxation is 1 in these cases
        z, sl, st, qp = _sqp(case, ocp, z)
        if case.get("warm"):
            ocp = _Ocp(case, d, x0=d["x0_next"])
            z, sl, st, qp = _sqp(case, ocp, z, st)
    if kind.endswith("grad"):
        dz = torch.zeros_like(z)
        dz[..., :nx] = 2.0 * (z[..., :nx] - d["target"])
        v, w0 = _adjoint(case, ocp, qp if not ocp.quad else ocp.qp_at(z), st, dz)
        e = 2.0 * (z - ocp.ref)
        return {"states": z[..., :nx], "controls": z[..., nx:], "d_x0": w0,
                "d_weights_penalization_control_squared": -(e * v)[..., nx:].sum(1),
                "d_weights_penalization_final_state": -(e * v)[:, -1, :nx],
                "d_weights_penalization_reference_state_trajectory": -(e * v)[..., :nx].sum(1)}
    return {"states": z[..., :nx], "controls": z[..., nx:], "slack": sl, "y_g": st.yg, "z_g": st.z, "y_f_0": st.y0,
            "y_f_dyn": st.yf}
