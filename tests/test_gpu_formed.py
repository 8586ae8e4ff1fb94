"""The formed stage-3 operator against the slab path: application, whitened application and the whole solve, over
center bonds 2..6 and environment bonds whose squares are not multiples of the K step (16).  Tolerance: FP64 sums of
at most 2^17 products per entry in another order, a few units of 1e-16 times their square root at most; 1e-13."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operators(D, chi, model, seed, one_site=None):
    from carcassonne_amd import pipeline, synthetic as syn
    c, s, st = syn.make_environment(D, chi, model=model, seed=seed, noise=8.0)
    op = syn.operator_center(model)
    if one_site is not None:
        op[("O",)] = one_site
    H, N = pipeline.multipliers(*pipeline.device_environment(c, s, op), graph=False)
    return H.operator, N.operator, torch.from_numpy(st.ravel()).cuda()


def _rel(a, b):
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize("D,chi,model,one_site", [
    (2, 3, "ising", None), (2, 8, "heisenberg", None), (3, 5, "ising", np.array([[0.5, 0.0], [0.0, -1.5]])),
    (3, 13, "heisenberg", np.array([[0.0, 1.0], [1.0, 0.0]])), (4, 9, "ising", None), (5, 7, "heisenberg", None),
    (6, 6, "ising", np.array([[0.3, 0.2], [0.2, -0.3]])), (6, 21, "heisenberg", None)])
def test_formed_operator_matches_slab_path(gpu, D, chi, model, one_site):
    from carcassonne_amd import _lib
    from carcassonne_amd.device import ptr, stream
    from carcassonne_amd.formed import FormedOperator
    from carcassonne_amd.solver import NormalizationFactor
    H, N, x = _operators(D, chi, model, 7, one_site)
    want, got, norm_want, norm_got = (torch.empty_like(x) for _ in range(4))
    H.apply_generic_flat(x, want)
    factor = NormalizationFactor(N)
    N.apply_generic_flat(x, norm_want)
    factor.apply_n(x, norm_got)
    assert _rel(norm_got, norm_want) < 1e-13
    formed = FormedOperator.of(H, N, factor)
    assert formed is not None
    formed.apply_flat(x, got)
    assert _rel(got, want) < 1e-13
    # W H W^T x, the whitening products applied around the slab path
    t, h, w = torch.empty_like(x), torch.empty_like(x), torch.empty_like(x)
    _lib.call("cc_skinny_f64", stream(), factor.n_env, 2, ptr(factor.Wt), 2, ptr(x), ptr(t))
    H.apply_generic_flat(t, h)
    _lib.call("cc_skinny_f64", stream(), factor.n_env, 1, ptr(factor.W), 2, ptr(h), ptr(w))
    formed.whitened(factor).apply(x, got)
    assert _rel(got, w) < 1e-12                            # cond(N) of these environments is below 10


@pytest.mark.parametrize("D,chi,model", [(2, 5, "ising"), (4, 11, "heisenberg"), (6, 10, "ising")])
def test_formed_solve_matches_slab_solve(gpu, D, chi, model):
    from carcassonne_amd.solver import GroundStateSolver, NormalizationFactor
    H, N, x0 = _operators(D, chi, model, 3)
    formed = GroundStateSolver(H, N)
    before = formed.rayleigh_quotient(x0)                  # the slabs
    x, theta, _, _ = formed.solve(x0, check_every=4)
    energy = formed.rayleigh_quotient(x)
    H2, N2, _ = _operators(D, chi, model, 3)
    slabs = GroundStateSolver(H2, N2, factor=NormalizationFactor(N2))     # a factor from outside: the slab path
    assert H._formed is not None and H2._formed is None
    assert abs(before - formed.rayleigh_quotient(x0)) <= 1e-12 * abs(before)
    y, theta2, _, _ = slabs.solve(x0, check_every=4)
    assert abs(theta - theta2) <= 1e-12 * abs(theta2)
    assert abs(energy - slabs.rayleigh_quotient(y)) <= 1e-12 * abs(energy)


def test_formed_operator_follows_its_environment(gpu):
    """A factor or operator refreshed from another environment drops the matrices formed before."""
    from carcassonne_amd.solver import GroundStateSolver
    H, N, x0 = _operators(3, 6, "ising", 1)
    H2, N2, _ = _operators(3, 6, "ising", 2)
    solver = GroundStateSolver(H, N)
    solver.solve(x0)
    solver.factor.refresh(N2)
    H.refresh_fused_from(H2)
    want, got = torch.empty_like(x0), torch.empty_like(x0)
    H2.apply_generic_flat(x0, want)
    H.apply_flat(x0, got)
    assert _rel(got, want) < 1e-13
    _, theta, _, _ = solver.solve(x0)
    _, theta2, _, _ = GroundStateSolver(H2, N2).solve(x0)
    assert abs(theta - theta2) <= 1e-11 * abs(theta2)


def test_application_does_not_depend_on_solves(gpu):
    """H(x) is the same bits before and after a solve of H, and a graph that captured it after a solve still replays
    the operator once the solver is gone and the operator has been refreshed."""
    from carcassonne_amd.solver import GroundStateSolver
    H, N, x0 = _operators(3, 6, "ising", 1)
    H2, _, _ = _operators(3, 6, "ising", 2)
    before, after, y = (torch.empty_like(x0) for _ in range(3))
    H.apply_flat(x0, before)
    solver = GroundStateSolver(H, N)
    solver.solve(x0)
    H.apply_flat(x0, after)
    assert torch.equal(before, after)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        H.apply_flat(x0, y)
    del solver
    for other in (None, H2):
        if other is not None:
            H.refresh_fused_from(other)
            other.apply_flat(x0, after)
        for _ in range(2):
            graph.replay()
            assert _rel(y, after) < 1e-13


def test_formed_solvers_of_one_operator_share_nothing(gpu):
    """Two formed solvers of one operator: another environment in the factor of the first leaves the second as it was
    and is refused by the first until it is refreshed as a whole."""
    from carcassonne_amd.precision import MixedSolver
    H, N, x0 = _operators(3, 6, "ising", 1)
    H2, N2, _ = _operators(3, 6, "ising", 2)
    first, second = MixedSolver(H, N, dtype="f32"), MixedSolver(H, N, dtype="f32")
    _, want, _ = second.solve(x0)
    first.factor.refresh(N2)
    _, rho, _ = second.solve(x0)
    assert rho == want
    with pytest.raises(RuntimeError):
        first.solve(x0)
    with pytest.raises(RuntimeError):
        first.solve_fixed(x0)
    first.refresh(H2, N2)
    _, rho, _ = first.solve(x0)
    _, want, _ = MixedSolver(H2, N2, dtype="f32").solve(x0)
    assert abs(rho - want) <= 1e-11 * abs(want)
    with pytest.raises(RuntimeError):
        second.solve(x0)


@pytest.mark.parametrize("through", ["operator", "f16", "f32"])
def test_new_solver_on_a_refreshed_operator(gpu, through):
    """A solver made for an operator that was refreshed from another (by itself or through a mixed solver) solves the
    environment it was refreshed from, and the operator still applies it afterwards."""
    from carcassonne_amd.precision import MixedSolver
    from carcassonne_amd.solver import GroundStateSolver
    H, N, x0 = _operators(3, 6, "ising", 1)
    H2, N2, _ = _operators(3, 6, "ising", 2)
    if through == "operator":
        GroundStateSolver(H, N).solve(x0)
        H.refresh_fused_from(H2)
    else:
        MixedSolver(H, N, dtype=through).refresh(H2, N2)
    want, got = torch.empty_like(x0), torch.empty_like(x0)
    H2.apply_generic_flat(x0, want)
    _, theta2, _, _ = GroundStateSolver(H2, N2).solve(x0)
    solver = GroundStateSolver(H, N2)
    x, theta, _, _ = solver.solve(x0)
    assert abs(theta - theta2) <= 1e-11 * abs(theta2)
    assert abs(solver.rayleigh_quotient(x) - theta2) <= 1e-11 * abs(theta2)
    H.apply_flat(x0, got)
    assert _rel(got, want) < 1e-13
    # the FP16 slabs are converted from the operator's own channels, so this solve need not converge; its value is that
    # of its state in the new environment
    y, rho, _ = MixedSolver(H, N2, dtype="f16").solve(x0)
    hy, ny = torch.empty_like(x0), torch.empty_like(x0)
    H2.apply_generic_flat(y, hy)
    N2.apply_generic_flat(y, ny)
    assert abs(rho - float(y @ hy) / float(y @ ny)) <= 1e-11 * abs(rho)
    with pytest.raises(NotImplementedError):
        MixedSolver(H, N2, dtype="f32")


@pytest.mark.parametrize("n,count", [(1, 1), (32, 2), (33, 1), (65, 3), (513, 2), (700, 3)])
def test_whitening_products(gpu, n, count):
    """W G W^T for lower-triangular W over partial rounds of the tile order, 32- and 64-wide tiles: two sums of n products,
    each within n eps of the sum of magnitudes."""
    from carcassonne_amd import _lib
    from carcassonne_amd.device import empty, ptr, stream
    rng = np.random.default_rng(n)
    G, W = rng.standard_normal((count, n, n)), np.tril(rng.standard_normal((n, n)))
    g, wt = torch.from_numpy(G).cuda(), torch.from_numpy(np.ascontiguousarray(W.T)).cuda()
    K, work = empty((count, n, n)), empty((count, n, n))
    _lib.call("cc_whiten_f64", stream(), n, count, ptr(g), ptr(wt), ptr(K), ptr(work))
    bound = 2 * (n + 2) * np.finfo(float).eps * (abs(W) @ abs(G) @ abs(W.T))
    assert np.all(abs(K.cpu().numpy() - W @ G @ W.T) <= bound)


@pytest.mark.parametrize("beside", [False, True])
def test_factor_holds_its_matrices_alone(gpu, beside):
    """N, L, W and two transposes; the sums' parts are given back, also where the factor was made on a side stream."""
    from carcassonne_amd.device import join
    from carcassonne_amd.solver import NormalizationFactor
    _, N, _ = _operators(4, 16, "ising", 3)
    if beside:
        factor, side = NormalizationFactor.beside(N)
        join(side)
    else:
        factor = NormalizationFactor(N)
    factor.check()
    held = sum(t.numel() * t.element_size() for t in vars(factor).values() if isinstance(t, torch.Tensor))
    assert held <= 5 * 256 * 256 * 8 + 64
    used = torch.cuda.memory_allocated()
    factor.refresh(N)
    assert torch.cuda.memory_allocated() == used
    residual = factor.L @ factor.L.t() - factor.N_env
    assert float(residual.norm() / factor.N_env.norm()) < 1e-14
