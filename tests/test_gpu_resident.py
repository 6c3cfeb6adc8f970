"""The on-chip ADMM path (csrc/resident.hpp): explicit-integrator QPs with diagonal
costs, one problem per workgroup, against the CPU oracle at the parity bars, over
the edges of its shape classes (padded and exact widths, the smallest and largest
horizons of a class, one and two stages per wavefront pass, no inequality rows)."""
import dataclasses

import numpy as np
import pytest
import torch

import oracle
from helpers import TOL, random_qp, rel_err, soften, zero_state
from test_gpu_admm import DEV, FIELDS, _assert_state_close, _run_pair, _solver, _state_to_dev
from turbompc_amd import _lib

pytestmark = pytest.mark.gpu


def _cfg(**kw):
    base = dict(max_iter=20, check_every=3, adapt_rho_every=0, sigma=1e-6, eps_abs=1e-12, eps_rel=1e-12,
                rho_f_factor=1000.0, alpha=1.6)
    base.update(kw)
    return oracle.OracleCfg(**base)


def _first(qp, k):
    """The batch's first k problems."""
    cut = lambda p: dataclasses.replace(p, **{  # noqa: E731
        f.name: getattr(p, f.name)[:k] for f in dataclasses.fields(p)
        if torch.is_tensor(getattr(p, f.name)) and getattr(p, f.name).ndim > 0})
    return dataclasses.replace(qp, **{f.name: cut(getattr(qp, f.name)) for f in dataclasses.fields(qp)
                                      if dataclasses.is_dataclass(getattr(qp, f.name))})


# (B, T, n, nx, m): n0 = nx; exact and padded classes, odd and even horizons
SHAPES = [(3, 2, 6, 4, 2), (5, 3, 6, 4, 4), (4, 64, 6, 4, 2), (3, 17, 4, 3, 1), (2, 21, 2, 1, 0),
          (3, 2, 9, 6, 3), (4, 33, 9, 6, 4), (2, 101, 9, 6, 3), (3, 13, 8, 5, 2),
          (3, 13, 9, 6, 11), (2, 61, 9, 6, 11), (3, 8, 8, 6, 12), (3, 9, 9, 6, 5),
          (3, 9, 16, 12, 16), (2, 22, 16, 12, 16), (3, 11, 13, 10, 13), (2, 10, 14, 10, 0),
          (3, 2, 17, 13, 4), (2, 33, 17, 13, 4), (2, 34, 17, 13, 3), (3, 12, 15, 13, 2)]
# horizons around the steps of the wavefront count, with more than hold the stages
SHAPES += [(2, 12, 17, 13, 4), (2, 24, 17, 13, 4), (2, 31, 17, 13, 4), (2, 41, 6, 4, 2), (2, 33, 9, 6, 11),
           (2, 57, 9, 6, 3), (2, 15, 16, 12, 16), (2, 29, 9, 6, 4)]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("shape", SHAPES)
def test_resident_matches_oracle(shape, dtype):
    B, T, n, nx, m = shape
    qp = random_qp(B, T, n, nx, m, seed=91, std=True, diag=True)
    print(shape, dtype, flush=True)
    ref, it_ref, _, out, stats = _run_pair(qp, _cfg(), dtype, std_dynamics=True, diag_cost=True)
    np.testing.assert_array_equal(stats.num_iter.cpu().numpy(), it_ref)
    assert not bool(stats.nonfinite.any())
    _assert_state_close(out, ref, TOL[dtype])
    if dtype != torch.float64:
        return
    # another kernel computes the streamed form of the same solve
    _, _, _, out_s, _ = _run_pair(qp, _cfg(), dtype, std_dynamics=True, diag_cost=True,
                                  kernel_flags=_lib.flag_stream_p(1))
    assert not torch.equal(out.x_blocks, out_s.x_blocks)
    _assert_state_close(out_s, ref, TOL[dtype])


@pytest.mark.parametrize("shape", [(7, 12, 9, 6, 11), (6, 21, 6, 4, 2), (5, 9, 17, 13, 4)])
@pytest.mark.parametrize("n0_full", [False, True])
def test_resident_slack_and_initial_controls(shape, n0_full):
    B, T, n, nx, m = shape
    qp = soften(random_qp(B, T, n, nx, m, seed=92, std=True, diag=True, n0=n if n0_full else None), 20.0, shrink=0.3)
    ref, it_ref, _, out, stats = _run_pair(qp, _cfg(check_every=4), torch.float64, use_slack=True, std_dynamics=True,
                                           diag_cost=True)
    np.testing.assert_array_equal(stats.num_iter.cpu().numpy(), it_ref)
    assert float(np.max(np.abs(ref.xi_g))) > 1e-3
    _assert_state_close(out, ref, 1e-9)


@pytest.mark.parametrize("alpha", [1.0, 1.6])
def test_resident_adaptive_rho_and_termination(alpha):
    """Chunks with refactorization between them, problems that stop early."""
    qp = random_qp(11, 9, 6, 4, 3, seed=42, std=True, diag=True)
    cfg = _cfg(max_iter=200, check_every=2, adapt_rho_every=4, eps_abs=1e-6, eps_rel=1e-6, rho_f_factor=50.0,
               alpha=alpha, adaptive_rho_tolerance=1.5)
    ref, it_ref, _, out, stats = _run_pair(qp, cfg, torch.float64, std_dynamics=True, diag_cost=True)
    np.testing.assert_array_equal(stats.num_iter.cpu().numpy(), it_ref)
    assert len(set(it_ref.tolist())) > 1 and np.any(ref.rho_bar != 0.1)
    assert rel_err(out.rho_bar, ref.rho_bar) < 1e-7
    _assert_state_close(out, ref, 1e-5)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_resident_const_g_is_the_same_solve(dtype):
    """G kept once in LDS against G per stage: the same bits."""
    qp = random_qp(5, 14, 17, 13, 4, seed=93, std=True, diag=True)
    G = qp.ineq.G[:1, :1].expand_as(qp.ineq.G).contiguous()
    qp = dataclasses.replace(qp, ineq=dataclasses.replace(qp.ineq, G=G))
    outs = [_run_pair(qp, _cfg(), dtype, std_dynamics=True, diag_cost=True, const_g=cg) for cg in (False, True)]
    ref = outs[0][0]
    for k in FIELDS:
        assert torch.equal(getattr(outs[0][3], k), getattr(outs[1][3], k)), k
    _assert_state_close(outs[1][3], ref, TOL[dtype])


@pytest.mark.parametrize("use_slack", [False, True])
@pytest.mark.parametrize("shape", [(13, 21, 6, 4, 2), (9, 11, 17, 13, 4), (7, 10, 9, 6, 11)])
def test_resident_sqp_step_check_and_activity(shape, use_slack):
    """The step's check against tmpc_sqp_first_order_*, the activity test, stopped
    problems untouched, the others as a plain solve."""
    from test_gpu_sqp import _random_state
    from turbompc_amd.solvers.sqp_hip import first_order_check

    B, T, n, nx, m = shape
    qp = random_qp(B, T, n, nx, m, seed=71, std=True, diag=True)
    if use_slack:
        qp = soften(qp, 3.0, shrink=0.5)
    rng = np.random.default_rng(9)
    st = _random_state(qp, rng, torch.float64, use_slack)
    qpd = qp.to(DEV, torch.float64)
    solver = _solver(qp, _cfg(max_iter=15, check_every=25, alpha=1.0), use_slack=use_slack, std_dynamics=True,
                     diag_cost=True)
    sw = qpd.ineq.slack_penalization_weight
    ref = first_order_check(qpd, st.x_blocks, st.y_f_0, st.y_f_dyn, st.y_g, st.xi_g if use_slack else None, float(sw),
                            std_dynamics=True, diag_cost=True)
    tol = float(ref[0].median())
    active = torch.tensor(rng.random(B) < 0.7, device=DEV)
    (_, _), stats, out, got, act = solver.sqp_step(qpd, st, active, tol, slack_weight=sw)
    (_, _), stats_g, out_g, _, act_g = solver.sqp_step(qpd, st, act, None, slack_weight=sw)
    (_, _), stats_p, out_p = solver.solve(qpd, st, slack_weight=sw)
    torch.cuda.synchronize()
    for a, b in zip(got, ref):
        assert rel_err(a, b) < 1e-12
    assert torch.equal(act, active & (ref[0] > tol)) and torch.equal(act_g, act) and 0 < int(act.sum()) < B
    on = act.cpu().numpy()
    assert np.all(stats.num_iter.cpu().numpy()[~on] == 0)
    for k in FIELDS:
        a, b0, p = (getattr(s, k).cpu().numpy() for s in (out, st, out_p))
        np.testing.assert_array_equal(a[~on], b0[~on])
        np.testing.assert_array_equal(a[on], p[on])
        np.testing.assert_array_equal(a, getattr(out_g, k).cpu().numpy())


def test_resident_nonfinite_flag():
    """A NaN in one problem's data, and in a stopped problem's state, flags it."""
    qp = random_qp(6, 9, 9, 6, 3, seed=94, std=True, diag=True).to(DEV, torch.float64)
    qp.cost.q[2, 4, 1] = float("nan")
    solver = _solver(qp, _cfg(), std_dynamics=True, diag_cost=True)
    st = _state_to_dev(zero_state(qp.to("cpu"), 0.1), torch.float64)
    _, stats, _ = solver.solve(qp, st)
    assert stats.nonfinite.cpu().tolist() == [b == 2 for b in range(6)]
    st.y_g[5, 3, 0] = float("inf")
    active = torch.tensor([True, True, False, True, True, False], device=DEV)
    _, stats, _, _, _ = solver.sqp_step(qp, st, active, None)
    assert stats.nonfinite.cpu().tolist() == [b == 5 for b in range(6)]


def test_resident_leaves_no_warm_records():
    """A streaming call that was told the workspace's records are warm, after an
    on-chip call on it (which keeps none), packs them anew."""
    from turbompc_amd.solvers.admm.admm_hip_backend import direct_workspace

    qp = random_qp(6, 9, 6, 4, 3, seed=95, std=True, diag=True)
    st0 = _state_to_dev(zero_state(qp, 0.1), torch.float64)
    qpd = qp.to(DEV, torch.float64)
    ws = direct_workspace(qpd)
    res = _solver(qp, _cfg(), std_dynamics=True, diag_cost=True)
    stream = _solver(qp, _cfg(), std_dynamics=True, diag_cost=True, kernel_flags=_lib.flag_stream_p(1))
    want = None
    for warm in (False, True):
        (_, _), _, out = res.solve(qpd, st0, workspace=ws)
        active = torch.ones(6, dtype=torch.bool, device=DEV)
        (_, _), _, out, _, _ = stream.sqp_step(qpd, out, active, None, workspace=ws, warm_records=warm)
        torch.cuda.synchronize()
        want = out if want is None else want
        for k in FIELDS:
            assert torch.equal(getattr(out, k), getattr(want, k)), (warm, k)


@pytest.mark.parametrize("form", ["problems per wavefront", "lane groups", "invariant A"])
@pytest.mark.parametrize("after", ["streaming", "on-chip", "generic"])
def test_streaming_forms_keep_their_warm_records(form, after):
    """Flags that keep a shape of the on-chip path on the streaming kernel: a warm call
    keeps the records of a streaming call before it (a q that changed against the
    caller's promise is not read) and packs them anew after a call of another path."""
    from turbompc_amd.solvers.admm.admm_hip_backend import direct_workspace

    qp = random_qp(6, 9, 17, 13, 4, seed=97, std=True, diag=True)
    G = qp.ineq.G[:1, :1].expand_as(qp.ineq.G).contiguous()
    qp = dataclasses.replace(qp, ineq=dataclasses.replace(qp.ineq, G=G))
    kw = {"problems per wavefront": dict(kernel_flags=_lib.flag_stream_p(1)),
          "lane groups": dict(kernel_flags=_lib.FLAG_FACTOR_GROUPS), "invariant A": dict(invariant_a=True)}[form]
    solver = lambda **k: _solver(qp, _cfg(max_iter=8), std_dynamics=True, diag_cost=True, const_g=True, **k)  # noqa: E731
    stream = solver(**kw)
    first = {"streaming": stream, "on-chip": solver(), "generic": solver(kernel_flags=_lib.FLAG_GENERIC_KERNEL)}[after]
    st0 = _state_to_dev(zero_state(qp, 0.1), torch.float64)
    qpd = qp.to(DEV, torch.float64)
    other = dataclasses.replace(qpd, cost=dataclasses.replace(qpd.cost, q=qpd.cost.q + 1.0))
    active = torch.ones(6, dtype=torch.bool, device=DEV)
    ws = direct_workspace(qpd)
    (_, _), _, mid = first.solve(qpd, st0, workspace=ws)
    (_, _), _, got, _, _ = stream.sqp_step(other, mid, active, None, workspace=ws, warm_records=True)
    (_, _), _, want, _, _ = stream.sqp_step(qpd if after == "streaming" else other, mid, active, None)
    torch.cuda.synchronize()
    for k in FIELDS:
        assert torch.equal(getattr(got, k), getattr(want, k)), k


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("shape", [(5, 17, 13, 4), (6, 9, 6, 11), (4, 16, 12, 9)])
def test_resident_factor_one_and_two_wavefronts(shape, dtype):
    """The factorization with a wavefront of its own for the preparation (up to 1024
    problems) and without: the same bits."""
    T, n, nx, m = shape
    qp = random_qp(1026, T, n, nx, m, seed=96, std=True, diag=True)
    part = _first(qp, 7)
    outs = []
    for q in (qp, part):
        st = _state_to_dev(zero_state(q, 0.1), dtype)
        (_, _), _, out = _solver(q, _cfg(), std_dynamics=True, diag_cost=True).solve(q.to(DEV, dtype), st)
        outs.append(out)
    torch.cuda.synchronize()
    for k in FIELDS:
        assert torch.equal(getattr(outs[0], k)[:7], getattr(outs[1], k)), k


@pytest.mark.parametrize("horizon", [50, 20])
def test_resident_is_as_near_to_64_bits_as_the_streaming_kernel(horizon):
    """fp32, 100 iterations: per output, the distance from the fp64 solve of the same
    data is no larger than the streaming kernel's, whose sums have as many roundings at
    the size of the duals (1.15: two draws of such errors over 64 problems)."""
    from turbompc_amd.problems import configs

    prob = configs.config2(B=64, seed=2)
    qp = prob.build_qp(*prob.initial_guess()).to("cpu", torch.float32).to("cpu", torch.float64)
    cut = lambda t, k: t[:, :horizon + k].contiguous()  # noqa: E731
    qp = dataclasses.replace(
        qp, cost=dataclasses.replace(qp.cost, D=cut(qp.cost.D, 1), E=cut(qp.cost.E, 0), q=cut(qp.cost.q, 1)),
        eq=dataclasses.replace(qp.eq, A_minus=cut(qp.eq.A_minus, 0), A_plus=cut(qp.eq.A_plus, 0), c=cut(qp.eq.c, 0)),
        ineq=dataclasses.replace(qp.ineq, **{k: cut(getattr(qp.ineq, k), 1) for k in ("G", "l", "u")}))
    cfg = _cfg(max_iter=100, check_every=101, alpha=1.0)
    run = lambda dtype, **kw: _solver(qp, cfg, std_dynamics=True, diag_cost=True, **kw).solve(  # noqa: E731
        qp.to(DEV, dtype), _state_to_dev(zero_state(qp, 0.1), dtype))[2]
    exact, chip, stream = run(torch.float64), run(torch.float32), run(torch.float32, kernel_flags=_lib.flag_stream_p(1))
    torch.cuda.synchronize()
    nx = 12
    parts = {"states": lambda s: s.x_blocks[..., :nx], "controls": lambda s: s.x_blocks[..., nx:], "z_g": lambda s: s.z_g,
             "y_g": lambda s: s.y_g, "y_f_0": lambda s: s.y_f_0, "y_f_dyn": lambda s: s.y_f_dyn}
    for name, f in parts.items():
        e, err = f(exact), lambda s: float((f(s).double() - e).norm() / e.norm())  # noqa: E731,B023
        a, b = err(chip), err(stream)
        print(f"  T = {horizon + 1}, {name}: on-chip {a:.2e}, streaming {b:.2e}", flush=True)
        assert a < 1.15 * b, name


# (T, n, nx, m, const_g, slack) of the fp32 form with two workgroups per CU, which more than
# 256 problems take: odd and even horizons, m below and at the class's, its largest horizons
TWO_PER_CU = [(13, 9, 6, 11, False, False), (16, 9, 6, 12, False, True), (33, 9, 6, 11, False, True),
              (64, 9, 6, 12, False, False), (12, 17, 13, 4, False, False), (25, 17, 13, 3, False, True),
              (37, 17, 13, 4, False, False), (41, 17, 13, 4, True, False)]


@pytest.mark.parametrize("case", TWO_PER_CU)
def test_resident_two_workgroups_per_cu(case):
    """fp32 against the oracle, and the first problems against a batch of their own, which
    runs one workgroup per CU: the same bits."""
    T, n, nx, m, const_g, slack = case
    B = 259
    qp = random_qp(B, T, n, nx, m, seed=98, std=True, diag=True)
    if slack:
        qp = soften(qp, 20.0, shrink=0.3)
    if const_g:
        G = qp.ineq.G[:1, :1].expand_as(qp.ineq.G).contiguous()
        qp = dataclasses.replace(qp, ineq=dataclasses.replace(qp.ineq, G=G))
    kw = dict(std_dynamics=True, diag_cost=True, const_g=const_g, use_slack=slack)
    print(case, flush=True)
    ref, it_ref, _, out, stats = _run_pair(qp, _cfg(), torch.float32, **kw)
    np.testing.assert_array_equal(stats.num_iter.cpu().numpy(), it_ref)
    _assert_state_close(out, ref, TOL[torch.float32])
    _, _, _, few, _ = _run_pair(_first(qp, 7), _cfg(), torch.float32, **kw)
    for k in FIELDS:
        assert torch.equal(getattr(out, k)[:7], getattr(few, k)), k
