"""The stage-block factorization (csrc/factor.hpp) and the Schur-level solve over the
edges of their tiles: block widths around 8, 16, 32, 48 and 64, odd and even (the last
pivot of an odd block is paired with a unit row), one problem and several."""
import numpy as np
import pytest
import torch

import oracle
from helpers import TOL, blocks_to_dense, random_qp, rel_err, zero_state
from test_gpu_admm import DEV, _assert_state_close, _run_pair
from test_gpu_resident import _cfg
from turbompc_amd import _lib
from turbompc_amd.solvers.backward.backward_kkt_hip import solve_backward_kkt_hip
from turbompc_amd.solvers.linear_systems_solvers.hip_backend import hip_blktri_solve

pytestmark = pytest.mark.gpu


def _system(B, T, n, seed):
    """SPD block-tridiagonal S = L L^T + I with a random block-bidiagonal L."""
    rng = np.random.default_rng(seed)
    Ld = rng.standard_normal((B, T, n, n)) / np.sqrt(n)
    Ls = rng.standard_normal((B, T, n, n)) / np.sqrt(n)
    Ls[:, 0] = 0
    S = np.zeros((B, T, n, 3 * n))
    S[..., n:2 * n] = Ld @ Ld.swapaxes(-1, -2) + Ls @ Ls.swapaxes(-1, -2) + np.eye(n)
    S[:, 1:, :, :n] = Ls[:, 1:] @ Ld[:, :-1].swapaxes(-1, -2)
    S[:, :-1, :, 2 * n:] = S[:, 1:, :, :n].swapaxes(-1, -2)
    return S, rng.standard_normal((B, T, n))


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [1, 2, 6, 7, 8, 9, 15, 16, 17, 31, 32, 33, 34, 47, 48, 49, 63, 64])
def test_blktri_block_widths(n, dtype):
    """Condition number of S below about 30: n eps times it is far below the bars."""
    for B, T in ((1, 2), (5, 7)):
        S, rhs = _system(B, T, n, seed=100 + n)
        x = hip_blktri_solve(torch.tensor(S, dtype=dtype, device=DEV), torch.tensor(rhs, dtype=dtype, device=DEV))
        xd = np.stack([np.linalg.solve(blocks_to_dense(S[b]), rhs[b].reshape(-1)).reshape(T, n) for b in range(B)])
        assert rel_err(x, xd) < TOL[dtype]


@pytest.mark.parametrize("dims", [(1, 1, 0), (3, 2, 1), (8, 5, 3), (9, 6, 4), (16, 12, 16), (17, 13, 4), (33, 20, 7)])
def test_qp_assembly_block_widths(dims):
    """The blocks formed from the QP's own (general dynamics, dense costs)."""
    n, nx, m = dims
    qp = random_qp(3, 6, n, nx, m, seed=7)
    ref, _, _, out, _ = _run_pair(qp, _cfg(), torch.float64, kernel_flags=_lib.FLAG_GENERIC_KERNEL)
    _assert_state_close(out, ref, TOL[torch.float64])


@pytest.mark.parametrize("dims", [(17, 13, 4), (17, 16, 1), (16, 13, 5), (12, 10, 12), (17, 14, 0)])
def test_adjoint_sweeps_of_34_rows(dims):
    """Up to 17 primal unknowns and 34 rows a stage: the sweeps and the residual that read
    the QP's blocks, against those on the assembled matrix (one factorization for both)."""
    n, nx, m = dims
    qp = random_qp(4, 8, n, nx, m, seed=17, std=False)
    G = qp.ineq.G.clone()
    G[:, :, max(n - nx - 1, 0):] = 0.0  # fewer active rows than free directions
    qp = qp.replace_ineq(G=G)
    qd = qp.to(DEV, torch.float64)
    dz_ref, mult_ref = oracle.adjoint_kkt(qp)
    for flags in (0, _lib.FLAG_GENERIC_KERNEL):
        dz, mult = solve_backward_kkt_hip(qd, refine_steps=4, kernel_flags=flags)
        assert rel_err(dz, dz_ref) < 1e-9 and rel_err(mult, mult_ref) < 1e-9


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [1, 6, 9, 16, 17, 34])
def test_blktri_infinite_pivot_pins_its_variable(n, dtype):
    """An infinite diagonal entry: its variable is zero, the others solve the system
    without its row and column."""
    B, T = 3, 5
    S, rhs = _system(B, T, n, seed=200 + n)
    pins = [(1, n - 1), (3, n // 2)]
    for t, i in pins:
        S[:, t, i, n + i] = np.inf
    x = hip_blktri_solve(torch.tensor(S, dtype=dtype, device=DEV), torch.tensor(rhs, dtype=dtype, device=DEV))
    keep = np.setdiff1d(np.arange(T * n), [t * n + i for t, i in pins])
    want = np.zeros((B, T * n))
    for b in range(B):
        want[b, keep] = np.linalg.solve(blocks_to_dense(S[b])[np.ix_(keep, keep)], rhs[b].reshape(-1)[keep])
    assert rel_err(x, want.reshape(B, T, n)) < TOL[dtype]
    for t, i in pins:
        assert bool((x[:, t, i] == 0).all())


@pytest.mark.parametrize("n", [6, 16, 34])
def test_blktri_scaled_by_powers_of_two(n):
    """S and the right-hand side scaled towards the ends of the range: the same x."""
    S, rhs = _system(2, 5, n, seed=300 + n)
    x = hip_blktri_solve(torch.tensor(S, device=DEV), torch.tensor(rhs, device=DEV))
    for e in (-1010, -700, 700, 1010):
        y = hip_blktri_solve(torch.tensor(np.ldexp(S, e), device=DEV), torch.tensor(np.ldexp(rhs, e), device=DEV))
        assert rel_err(y, x) < 1e-12, e
