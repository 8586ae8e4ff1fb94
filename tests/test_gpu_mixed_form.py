"""Which operator a mixed solve runs inside: the one its dtype names, for solves of fixed work (whose unconverged state
carries that operator's digits) as for the adaptive ones."""
import json
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
GOLDEN = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "energies.json")))


def _operators(D, chi, model, seed, noise=1.0):
    from carcassonne_amd import pipeline, synthetic as syn
    c, s, st = syn.make_environment(D, chi, model=model, seed=seed, noise=noise)
    H, N = pipeline.multipliers(*pipeline.device_environment(c, s, syn.operator_center(model)), graph=False)
    return H.operator, N.operator, torch.from_numpy(st.ravel()).cuda()


@pytest.mark.parametrize("D,chi,model", [(2, 9, "heisenberg"), (3, 8, "ising"), (4, 12, "heisenberg"), (6, 10, "ising")])
def test_fixed_work_runs_the_named_operator(gpu, D, chi, model):
    """Two refinement passes after a few Lanczos steps leave the operator's rounding in the state: FP16 and BF16 give
    what they give around a factor made outside (bit for bit, the same kernels on the same numbers), and no two of the
    three operators give the same state."""
    from carcassonne_amd.precision import MixedSolver
    from carcassonne_amd.solver import NormalizationFactor
    H, N, x0 = _operators(D, chi, model, 5)
    states = []
    for dtype in ("f16", "bf16", "f32"):
        solver = MixedSolver(H, N, dtype=dtype)
        x, _, _ = solver.solve_fixed(x0, lp_iters=6, outer=2, inner_iters=3)
        if dtype != "f32":
            assert solver.Hlp.dtype == dtype
            y, _, _ = MixedSolver(H, N, dtype=dtype, factor=NormalizationFactor(N)).solve_fixed(x0, lp_iters=6, outer=2,
                                                                                                  inner_iters=3)
            assert torch.equal(x, y)
        states.append(x / x.norm() * torch.sign(torch.dot(x, x0)))
    for i, j in ((0, 1), (0, 2), (1, 2)):
        assert float((states[i] - states[j]).norm()) > 1e-9, (i, j)


@pytest.mark.parametrize("key", ["D4_chi32_ising_seed0", "D4_chi32_heisenberg_seed0", "D6_chi64_ising_seed0",
                                 "D6_chi64_heisenberg_seed0"])
def test_formed_f32_solve_reaches_fp64_energy(gpu, key):
    from carcassonne_amd.precision import MixedSolver
    g = GOLDEN[key]
    H, N, x0 = _operators(g["D"], g["chi"], g["model"], g["seed"])
    _, rho, info = MixedSolver(H, N, dtype="f32").solve(x0)
    assert info["converged"]
    assert abs(rho - g["ground_energy"]) < 1e-10 * abs(g["ground_energy"]), info


def test_solve_mixed_returns_the_operator_it_ran(gpu):
    """lp_operator is the FP16 operator of the solve; a formed solve has none and makes none."""
    from carcassonne_amd import pipeline, synthetic as syn
    from carcassonne_amd.data import HipData
    c, s, st = syn.make_environment(3, 6, model="ising", seed=2)
    env = pipeline.device_environment(c, s, syn.operator_center("ising"))
    x0 = HipData.fromArray(st)
    r = pipeline.solve_mixed(*env, x0, graph=False)
    assert r["lp_operator"].dtype == "f16"
    f = pipeline.solve_mixed(*env, x0, dtype="f32", graph=False)
    assert f["lp_operator"] is None
    assert not any(ch.lowprec for ch in f["operator"]._A + f["operator"]._B)
    assert abs(f["energy"] - r["energy"]) <= 1e-10 * abs(r["energy"])


def test_formed_batch_in_one_graph(gpu):
    """A batch of formed solves with the setup inside the graph: replays reproduce the eager solves."""
    from carcassonne_amd.batched import BatchedSolve
    b = BatchedSolve([(2, 6, 2.5, 1), (3, 5, 3.1, 2), (4, 4, 2.9, 5)], dtype="f32")
    b.prepare()
    b.tune_work()
    ref = b.reference_energies()
    eager = [float(s["solver"].solve_fixed(s["x0"], lp_iters=b.tuning[s["key"]]["lp_iters"],
                                           outer=b.tuning[s["key"]]["outer"])[1].item()) for s in b.systems]
    b.capture()
    for _ in range(3):
        b.replay()
        assert b.energies() == eager
        b.reference_energies()          # eager work between replays
    np.testing.assert_allclose(eager, ref, rtol=1e-10)


def test_arguments_of_another_form_are_refused(gpu):
    from carcassonne_amd.precision import MixedSolver
    H, N, _ = _operators(2, 4, "ising", 1)
    with pytest.raises(KeyError):
        MixedSolver(H, N, dtype="f64")
    for kw in (dict(groups=4), dict(split="both")):
        with pytest.raises(ValueError):
            MixedSolver(H, N, dtype="f32", **kw)
