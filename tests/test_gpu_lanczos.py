"""The Lanczos steps with the delayed second pass against a dense eigen-decomposition: bases that fill the space, checks
at and between the last steps, starts that end the basis early, one to many basis vectors per slice."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solver(D, chi, seed, precision="f64"):
    from carcassonne_amd import pipeline, synthetic as syn
    from carcassonne_amd.solver import GroundStateSolver
    c, s, st = syn.make_environment(D, chi, model="ising", seed=seed)
    H, N = pipeline.multipliers(*pipeline.device_environment(c, s, syn.operator_center("ising")), graph=False)
    return GroundStateSolver(H.operator, N.operator, precision=precision), H, N


def _dense(H, N):
    from scipy.linalg import eigh
    h, n = (m.formMatrix().tensor().cpu().numpy() for m in (H, N))
    return eigh(0.5 * (h + h.T), 0.5 * (n + n.T)), n


@pytest.mark.parametrize("D,chi", [(2, 6), (3, 5)])
@pytest.mark.parametrize("check_every", [1, 3, 7, 400])
def test_full_basis(gpu, D, chi, check_every):
    """As many steps as unknowns: the lowest pair to 1e-9 (the spectrum is separated; rounding alone is 1e-13)."""
    import torch
    solver, H, N = _solver(D, chi, 5)
    (values, vectors), n = _dense(H, N)
    x0 = torch.from_numpy(np.random.default_rng(1).standard_normal(solver.n)).cuda()
    x, theta, residual, iterations = solver.solve(x0, tol_residual=1e-13, tol_energy=0.0, max_iter=solver.n + 5,
                                                  check_every=check_every)
    assert iterations <= solver.n
    scale = abs(values).max()
    assert abs(theta - values[0]) <= 1e-10 * scale
    x = x.cpu().numpy()
    assert abs(abs(x @ n @ vectors[:, 0]) - 1.0) <= 1e-9


@pytest.mark.parametrize("pairs", [1, 2, 5])
def test_start_in_an_invariant_subspace(gpu, pairs):
    """A start made of a few eigenvectors: the basis ends after as many steps, up to rounding that grows from there on;
    the lowest of them is found to 1e-8 wherever the iteration stops."""
    import torch
    solver, H, N = _solver(2, 6, 9)
    (values, vectors), _ = _dense(H, N)
    x0 = torch.from_numpy(vectors[:, :pairs] @ np.arange(1.0, pairs + 1.0)).cuda()
    for steps in (pairs, pairs + 1):
        _, theta, _, _ = solver.solve(x0, max_iter=steps, check_every=1)
        assert abs(theta - values[0]) <= 1e-8 * abs(values).max()


@pytest.mark.parametrize("steps", [1, 2, 15, 16, 17, 81])
def test_basis_is_orthogonal_to_rounding(gpu, steps):
    """Ritz vector of a given number of steps: N-normalized, and its Rayleigh quotient is the Ritz value (what a loss of
    orthogonality would spoil first)."""
    import torch
    solver, _, _ = _solver(4, 8, 2)
    x0 = torch.from_numpy(np.random.default_rng(3).standard_normal(solver.n)).cuda()
    x, theta, _, iterations = solver.solve(x0, tol_residual=0.0, tol_energy=-1.0, max_iter=steps, check_every=steps)
    assert iterations == steps
    nx = torch.empty_like(x)
    solver.factor.apply_n(x, nx)
    assert abs(float((x * nx).sum()) - 1.0) <= 1e-12
    assert abs(solver.rayleigh_quotient(x) - theta) <= 1e-12 * abs(theta) + 1e-12
