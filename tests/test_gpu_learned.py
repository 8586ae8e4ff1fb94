"""The learned warm start on the GPU: features, forward pass and gradients of the HIP kernels against
the NumPy oracle (oracle/mlp.py), one Adam step against its formula, and the gain of a trained network
over random starts on held-out environments of a family (the plain solve checks every start)."""
import numpy as np
import pytest
import torch

from oracle import mlp as OM

pytestmark = pytest.mark.gpu


def _net(K_spec=8, k=16, NO=128, H=128, seed=3):
    from carcassonne_amd.learned import WarmStartMLP
    return WarmStartMLP(K_spec, k, NO, hidden=H, seed=seed)


def _batch(net, B, seed):
    rng = np.random.default_rng(seed)
    X = rng.uniform(0, 1, (B, net.K0)).astype(np.float16)
    V = rng.standard_normal((B, net.NO)).astype(np.float32)
    return X, V


def test_features_match_oracle(gpu):
    from carcassonne_amd.learned import Family, WarmStartMLP, spectra_of_environment
    fam = Family(2, 6, sigma=0.2)
    corners, sides, opc, _ = fam.environment(7, 2.7)
    S = spectra_of_environment(corners, sides).cpu().numpy()
    from carcassonne_amd import synthetic as syn
    c, s, _ = syn.make_environment(2, 6, seed=0, perturb_seed=7, sigma=0.2)
    want = [np.linalg.svd(x[("I",)].reshape(6, 6), compute_uv=False) for x in c]
    want += [np.linalg.svd(x[("I",)].reshape(6, -1), compute_uv=False) for x in s]
    np.testing.assert_allclose(S, np.array(want), rtol=1e-10, atol=1e-12)
    net = WarmStartMLP(8, 6, 64, hidden=64)
    f = net.features(corners, sides, 2.7).float().cpu().numpy()
    np.testing.assert_allclose(f, OM.features(S, 2.7, net.K0), rtol=1e-3, atol=1e-3)


def test_forward_matches_oracle(gpu):
    net = _net()
    X, _ = _batch(net, 64, 0)
    Y, _ = net.forward(torch.from_numpy(X).cuda())
    want, _ = OM.forward(net.P32.cpu().numpy().astype(np.float64), X.astype(np.float64), net.K0, net.H, net.NO)
    err = np.linalg.norm(Y.cpu().numpy() - want) / np.linalg.norm(want)
    assert err < 1e-4, err


def test_gradients_match_oracle(gpu):
    """Backward kernels against the oracle's gradient of the same pass (the GPU's saved FP16 hidden
    activations are handed to the oracle, so only FP32-vs-FP64 accumulation differs)."""
    net = _net()
    B = 64
    X, V = _batch(net, B, 1)
    Xd, Vd = torch.from_numpy(X).cuda(), torch.from_numpy(V).cuda()
    loss, Y = net.loss_and_grad(Xd, Vd)
    Yf, (A16, A32) = net.forward(Xd)
    h = A32.cpu().numpy().reshape(2, B, net.H)
    hr = A16.float().cpu().numpy().reshape(2, B, net.H)
    saved = dict(h1=h[0], h2=h[1], h1r=hr[0], h2r=hr[1], y=Yf.cpu().numpy())
    g_want, l_want = OM.backward(net.P32.cpu().numpy().astype(np.float64), X.astype(np.float64),
                                 V.astype(np.float64), net.K0, net.H, net.NO, saved=saved)
    np.testing.assert_allclose(loss.cpu().numpy(), l_want, rtol=1e-4, atol=1e-6)
    g = net.G.cpu().numpy()
    parts = OM.split_params(np.arange(g.size), net.K0, net.H, net.NO)
    for name, idx in zip(("W1", "b1", "W2", "b2", "W3", "b3"), parts):
        a, b = g[idx.ravel()], g_want[idx.ravel()]
        assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b) + 1e-10, name


# (batch, spectra width, output, hidden): one sample, batches that leave a partial K chunk, a partial row tile or waves
# without work, input widths of one and a half column tiles, the smallest widths and unequal ones
@pytest.mark.parametrize("B,k,NO,H", [(1, 1, 64, 64), (5, 4, 64, 128), (17, 1, 192, 64), (33, 5, 128, 64), (100, 2, 64, 192),
                                      (250, 16, 128, 128)])
def test_gradients_at_ragged_sizes(gpu, B, k, NO, H):
    """As above; FP32 sums of at most 250 terms: 1e-4 is ten times 250 x 2^-24, for some cancellation."""
    net = _net(k=k, NO=NO, H=H)
    X, V = _batch(net, B, 4)
    Xd, Vd = torch.from_numpy(X).cuda(), torch.from_numpy(V).cuda()
    loss, _ = net.loss_and_grad(Xd, Vd)
    Yf, (A16, A32) = net.forward(Xd)
    h = A32.cpu().numpy().reshape(2, B, H)
    hr = A16.float().cpu().numpy().reshape(2, B, H)
    p = net.P32.cpu().numpy().astype(np.float64)
    want, _ = OM.forward(p, X.astype(np.float64), net.K0, H, NO)
    assert np.linalg.norm(Yf.cpu().numpy() - want) <= 1e-4 * np.linalg.norm(want)
    saved = dict(h1=h[0], h2=h[1], h1r=hr[0], h2r=hr[1], y=Yf.cpu().numpy())
    g_want, l_want = OM.backward(p, X.astype(np.float64), V.astype(np.float64), net.K0, H, NO, saved=saved)
    np.testing.assert_allclose(loss.cpu().numpy(), l_want, rtol=1e-4, atol=1e-6)
    g = net.G.cpu().numpy()
    parts = OM.split_params(np.arange(g.size), net.K0, H, NO)
    for name, idx in zip(("W1", "b1", "W2", "b2", "W3", "b3"), parts):
        a, b = g[idx.ravel()], g_want[idx.ravel()]
        assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b) + 1e-10, name


def test_adam_step(gpu):
    net = _net()
    X, V = _batch(net, 64, 2)
    p0 = net.P32.cpu().numpy().copy()
    net.loss_and_grad(torch.from_numpy(X).cuda(), torch.from_numpy(V).cuda())
    g = net.G.cpu().numpy()
    net.adam_step(lr=1e-3)
    m, v = 0.1 * g, 0.001 * g * g
    want = p0 - 1e-3 * (m / 0.1) / (np.sqrt(v / 0.001) + 1e-8)
    np.testing.assert_allclose(net.P32.cpu().numpy(), want, rtol=1e-5, atol=1e-7)
    p32 = net.P32.cpu().numpy()
    np.testing.assert_array_equal(net.P16.cpu().numpy(), p32.astype(np.float16))   # the mirror is the rounded master


def test_trained_network_saves_iterations(gpu):
    """A network trained on 384 converged states of a D=3, chi=8 family proposes better start vectors
    than random ones on held-out environments of the same family (on the GPU: 42.7 Lanczos iterations
    against 50.7 from random starts, 43 from the previous step's state)."""
    from carcassonne_amd.learned import Family, WarmStartMLP, evaluate_starts, generate_pairs
    fam = Family(3, 8, sigma=0.2, base_seed=11)
    net = WarmStartMLP(8, 8, 192, hidden=256, seed=0)
    rng = np.random.default_rng(0)
    n = 384
    X, T, _ = generate_pairs(fam, net, list(range(1000, 1000 + n)), rng.uniform(2.0, 4.0, n))
    hist = net.train(X, T, epochs=40, batch=64, lr=2e-3)
    assert hist[-1] < 0.5 * hist[0], hist
    hs = np.linspace(2.2, 3.8, 12)
    ev = evaluate_starts(fam, net, list(range(90000, 90012)), hs)
    assert max(ev["energy_spread"]) < 1e-9
    assert np.mean(ev["learned"]) < 0.9 * np.mean(ev["random"]), ev


def test_learned_start_at_d4_chi32(gpu):
    """The learned-start workload's shape (D=4, chi=32, TFIM family, h ~ U[2, 4]): a network trained with the
    HIP kernels on 512 plain solves proposes start vectors that take fewer Lanczos iterations than random
    starts on held-out environments (about 50 against 67 in the committed study); the previous-step start
    (the reference's own) and the Rayleigh-Ritz combination of both are reported and reach the same energies."""
    from carcassonne_amd.learned import Family, WarmStartMLP, evaluate_starts, generate_pairs, _pad64
    fam = Family(4, 32, sigma=0.05, base_seed=11)
    net = WarmStartMLP(8, 32, _pad64(fam.n), hidden=512, seed=0)
    rng = np.random.default_rng(11)
    n = 512
    X, T, _ = generate_pairs(fam, net, list(range(1000, 1000 + n)), rng.uniform(2.0, 4.0, n))
    hist = net.train(X, T, epochs=20, batch=128, lr=1e-3)
    print("train loss", hist[0], "->", hist[-1], flush=True)
    assert hist[-1] < 0.5 * hist[0]
    ev = evaluate_starts(fam, net, list(range(900000, 900010)), np.linspace(2.0, 4.0, 10))
    means = {k: float(np.mean(ev[k][1:] if k in ("random", "learned") else ev[k]))
             for k in ("random", "previous", "learned", "combined")}
    print("mean iterations", means, flush=True)
    assert max(ev["energy_spread"]) < 1e-9
    assert means["learned"] < 0.9 * means["random"], means


def test_residual_features_and_correction_start(gpu):
    """The correction network's input row is the unit residual of the previous state in the new environment
    followed by h; the learned correction start is a unit-N-norm Rayleigh-Ritz combination whose energy is
    at most the previous state's."""
    from carcassonne_amd.learned import (Family, WarmStartMLP, learned_correction_start, residual_features,
                                         solve_from, _pad64)
    from carcassonne_amd.pipeline import multipliers
    fam = Family(2, 6, sigma=0.1, base_seed=3)
    corners, sides, opc, x0 = fam.environment(5, 2.5)
    x_prev, _, _ = solve_from(corners, sides, opc, x0)
    corners, sides, opc, _ = fam.environment(6, 2.6)
    H, N = multipliers(corners, sides, opc)
    net = WarmStartMLP.for_residual(fam.n, _pad64(fam.n), hidden=64, seed=2)
    row = residual_features(net, H.operator, N.operator, x_prev, 2.6).float().cpu().numpy()
    hx, nx = torch.empty_like(x_prev), torch.empty_like(x_prev)
    H.operator.apply_flat(x_prev, hx)
    N.operator.apply_flat(x_prev, nx)
    rho = float(x_prev @ hx) / float(x_prev @ nx)
    r = (hx - rho * nx).cpu().numpy()
    np.testing.assert_allclose(row[:fam.n], r / np.linalg.norm(r), atol=2e-3)
    assert abs(row[fam.n] - 2.6) < 2e-3 and not np.any(row[fam.n + 1:])
    xs = learned_correction_start(net, H.operator, N.operator, x_prev, 2.6)
    H.operator.apply_flat(xs, hx)
    N.operator.apply_flat(xs, nx)
    assert abs(float(xs @ nx) - 1.0) < 1e-10
    assert float(xs @ hx) / float(xs @ nx) <= rho + 1e-12 * abs(rho)
