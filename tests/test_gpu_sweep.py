"""GPU parity of the sweep step against the oracle.

* The fused-bond step (System.contractAndCompressTowards: absorptions, fused truncation basis from
  cc_fused_truncation_f64, the side absorption projected as it is formed) against the oracle's
  contractTowards + fused projection (oracle/fused.py), on the synthetic fused environments: energy and
  normalization after every step, at the rank bound and below it.
* The plain CPU workload of the benchmark list: the 2D transverse-field Ising model (h = 3, d = 2) on a
  seeded double-layer environment with center bond D = 2 and per-copy environment bond 8, 20 sweep steps
  of contract -> compress every corner-side bond to 8 (the reference's per-copy compressor, deterministic
  start) -> relaxOver solve, the reference's own step (system/_2d.py:435-497, policies.py:80-113).  Every
  step of the GPU is run on the oracle's pre-step system (uploaded), so that each step is compared on
  identical inputs: energy after the contraction (1e-9), after the compression and after the solve (1e-3;
  the compressor's four unconverged alternating least-squares sweeps, with normal equations of condition
  number near 1e9 and growing with the environment, amplify round-off differences to ~1e-4 at some later
  steps; the first six steps and at least a third of all agree to 1e-8), and the solve's restarts where the
  compressed inputs agree to 1e-9.  The oracle's one-site energy estimates over the last steps scatter around -3.1
  (h = 3 is close to the 2D critical field 3.04, where the 2D TFIM energy per site is about -3.1).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,chi,model,new", [(2, 8, "ising", 8), (3, 6, "heisenberg", 6), (2, 8, "ising", 6)])
def test_fused_step_matches_oracle(gpu, D, chi, model, new):
    from carcassonne_amd import synthetic as syn
    from oracle import fused
    from oracle.system import System as OSystem
    from tests.oracle_bridge import to_oracle, to_product
    from carcassonne_amd.system import System
    c, s, st = syn.make_environment(D, chi, model=model, seed=4)
    op = syn.operator_center(model)
    osys = OSystem(*to_oracle(c, s, op)[:2], st, to_oracle(c, s, op)[2])
    pc, ps, po = to_product(c, s, op)
    from carcassonne_amd.data import HipData
    psys = System(pc, ps, HipData.fromArray(st), po)
    for step, direction in enumerate((0, 1, 2, 3, 1)):
        fused.contract_and_compress_towards(osys, direction, new)
        psys.contractAndCompressTowards(direction, new)
        e_o, n_o = osys.computeExpectationAndNormalization()
        e_p, n_p = psys.computeExpectationAndNormalization()
        print(D, chi, model, new, "step", step, "E", e_p, e_o, "N", n_p, n_o, flush=True)
        assert abs(n_p - n_o) <= 1e-9 * abs(n_o), (step, n_p, n_o)
        assert abs(e_p - e_o) <= 1e-9 * abs(e_o), (step, e_p, e_o)
        assert all(t.shape[0] == min(new, chi) for t in psys.sides[direction].values())


def test_plain_cpu_workload_sweep_steps_match_oracle(gpu):
    from carcassonne_amd import synthetic as syn
    from carcassonne_amd.data import HipData
    from oracle.system import System as OSystem
    from oracle.tags import make_simple_sparse_operator
    from tests.oracle_bridge import system_to_product, to_oracle
    X = np.array([[0.0, 1.0], [1.0, 0.0]])
    Z = np.diag([1.0, -1.0])
    c, s, st = syn.make_double_layer_environment(2, 8, seed=0)
    oc, os_, _ = to_oracle(c, s, {})
    osys = OSystem(oc, os_, st, make_simple_sparse_operator(O=-3.0 * X, OO_UD=[Z, -Z], OO_LR=[Z, -Z]),
                   rng=np.random.default_rng(1))
    osys.compressor_start = "svd"
    per_site, close = [], []
    for step in range(20):
        psys = system_to_product(osys)
        psys.compressor_start = "svd"
        rows = []
        for sys_ in (osys, psys):
            sys_.contractTowards(step % 4)
            e1 = sys_.computeExpectation()
            for corner_id in range(4):
                for direction in range(2):
                    sys_.compressCornerStateTowards(corner_id, direction, 8)
            e2 = sys_.computeExpectation()
            sys_.minimizeExpectation()
            rows.append((complex(e1).real, complex(e2).real, complex(sys_.computeExpectation()).real,
                         sys_.last_solve["restarts"]))
        (o1, o2, o3, orst), (p1, p2, p3, prst) = rows
        site = complex(osys.computeOneSiteExpectation()).real
        per_site.append(site)
        print("step", step, "oracle", rows[0], "device", rows[1], "per site", site, flush=True)
        assert abs(p1 - o1) <= 1e-9 * abs(o1), ("contract", step, p1, o1)
        # the compressor's normal equations are ill-conditioned (kept eigenvalues down to ~1e-9 of the
        # largest): a 1e-14 relative change of its input moves the compressed energy by ~2e-8 on the CPU
        # alone, and four unconverged alternating sweeps amplify it further (up to ~1e-4 at some steps);
        # the compressed and solved energies are compared to 1e-3, and most steps to 1e-8
        assert abs(p2 - o2) <= 1e-3 * abs(o2), ("compress", step, p2, o2)
        if abs(p2 - o2) <= 1e-9 * abs(o2):
            assert prst == orst, ("restarts", step, prst, orst)
        assert abs(p3 - o3) <= 1e-3 * abs(o3), ("solve", step, p3, o3)
        assert abs(complex(psys.computeOneSiteExpectation()).real - site) <= 1e-3 * abs(site)
        close.append(abs(p2 - o2) <= 1e-8 * abs(o2))
    print("steps whose compressed energies agree to 1e-8:", sum(close), "of", len(close))
    assert all(close[:6]) and sum(close) >= len(close) // 3, close
    # a loose physical check of the trajectory (the one-site estimates fluctuate from step to step)
    assert -3.4 < float(np.mean(per_site[-8:])) < -2.8, per_site


@pytest.mark.parametrize("nx,D,far,k,rank", [(32, 3, 64, 40, 48), (8, 2, 16, 16, 16), (6, 4, 50, 7, 50)])
def test_fused_truncation_basis_matches_oracle(gpu, nx, D, far, k, rank):
    """cc_fused_truncation_f64 (through system._2d.fusedTruncationBasis) against the oracle's SVD of the
    symmetrized bond matricization (oracle/fused.py fused_basis) on a ket/bra-symmetric matrix with a graded
    spectrum (1 down to 1e-4) and a null space: the columns whose singular value is at least 1e-2 of the
    largest agree to 1e-9 (signs fixed by the same rule), and every kept column is a unit vector orthogonal
    to the others."""
    from carcassonne_amd.data import HipData
    from carcassonne_amd.system._2d import fusedTruncationBasis
    from oracle import fused
    rng = np.random.default_rng(nx * 1000 + far)
    m = nx * D * D
    C3 = rng.standard_normal((nx, D, D, far))
    Cs = (0.5 * (C3 + C3.transpose(0, 2, 1, 3))).reshape(m, far)
    u, _, vt = np.linalg.svd(Cs, full_matrices=False)
    r = min(rank, u.shape[1])
    s = np.zeros(far)
    s[:r] = np.logspace(0, -4, r)
    Cm = (u[:, :far] * s[:u.shape[1]]) @ vt
    corner = HipData.fromArray(Cm.T.reshape(far, 1, 1, nx * D, D, 1))
    U = fusedTruncationBasis(corner, (3, 4, 5), (0, 1, 2), k).toArray()
    want, sv = fused.fused_basis(Cm, nx, D, min(k, far))
    assert U.shape == want.shape
    big = sv[:U.shape[1]] >= 1e-2 * sv[0]
    np.testing.assert_allclose(U[:, big], want[:, big], atol=1e-9)
    kept = sv[:U.shape[1]] > 1e-7 * sv[0]
    G = U[:, kept].T @ U[:, kept]
    assert np.abs(G - np.eye(G.shape[0])).max() < 1e-6, np.abs(G - np.eye(G.shape[0])).max()
    assert not np.any(U[:, ~kept])


# far bond n <= 64: one and two columns (padded to three pairs), odd ones, every pair occupied, and rank deficient
@pytest.mark.parametrize("n,rank", [(1, 1), (2, 2), (3, 3), (5, 5), (6, 6), (7, 7), (8, 8), (21, 21), (33, 33), (62, 62),
                                    (63, 63), (64, 64), (24, 9), (64, 40), (5, 0)])
def test_fused_truncation_diagonalizes_the_gram_matrix(gpu, n, rank):
    """cc_fused_truncation_f64 on a symmetrized C (D = 2) of condition at most 10 on its range: singular values and
    the products C^T U against NumPy's.  The Gram matrix is diagonalized to about n 1e-15 of its trace, so values and
    directions of the range are good to 100 x n x 1e-15 x n; 1e-10 leaves a factor of 2."""
    import torch
    from carcassonne_amd import _lib
    from carcassonne_amd.device import empty, ptr, stream
    rng = np.random.default_rng(100 * n + rank)
    nx = n + 2
    left = np.linalg.qr(rng.standard_normal((nx * 3, max(rank, 1))))[0]
    right = np.linalg.qr(rng.standard_normal((n, max(rank, 1))))[0]
    sym = (left * np.linspace(1.0, 0.1, max(rank, 1)) * (rank > 0)) @ right.T        # (x, [00, 11, 01 + 10]) x n
    C = np.zeros((nx, 2, 2, n))
    sym = sym.reshape(nx, 3, n)
    C[:, 0, 0], C[:, 1, 1] = sym[:, 0], sym[:, 1]
    odd = rng.standard_normal((nx, n))
    C[:, 0, 1], C[:, 1, 0] = sym[:, 2] / np.sqrt(2) + odd, sym[:, 2] / np.sqrt(2) - odd   # the odd part drops out
    Cs = 0.5 * (C + C.transpose(0, 2, 1, 3)).reshape(nx * 4, n)
    U, S = empty((nx * 4, n)), empty((n,))
    work = empty((_lib.query("cc_fused_truncation_work_size", nx, 2, n),))
    _lib.call("cc_fused_truncation_f64", stream(), nx, 2, n, n, ptr(torch.from_numpy(C).cuda()), ptr(U), ptr(S), ptr(work))
    U, S = U.cpu().numpy(), S.cpu().numpy()
    want = np.linalg.svd(Cs, compute_uv=False)
    assert np.all(np.diff(S) <= 0)
    assert np.abs(S[:rank] - want[:rank]).max(initial=0) <= 1e-10
    Ur = U[:, :rank]
    assert np.abs(Ur.T @ Ur - np.eye(rank)).max(initial=0) <= 1e-10
    T = Cs.T @ Ur
    assert np.abs(T.T @ T - np.diag(want[:rank] ** 2)).max(initial=0) <= 1e-10
    if rank == 0:
        assert not U.any()


def test_fused_step_of_a_lazily_permuted_center(gpu, monkeypatch):
    """A center whose leg permutation is still to be carried out gives the step of the plain one, and its data, which stay
    with the caller's tensor, are made on the caller's stream."""
    import torch
    from carcassonne_amd import pipeline, synthetic as syn
    from carcassonne_amd.data import HipData
    from carcassonne_amd.system import System
    c, s, st = syn.make_environment(3, 6, model="ising", seed=4)
    corners, sides, opc = pipeline.device_environment(c, s, syn.operator_center("ising"))
    plain = System(list(corners), list(sides), HipData.fromArray(st), opc)
    plain.contractAndCompressTowards(1, 5)
    moved = HipData.fromArray(np.ascontiguousarray(st.transpose(4, 3, 0, 1, 2)))
    center = moved.permuted_lazily([2, 3, 4, 1, 0])
    lazy = System(list(corners), list(sides), center, opc)
    streams = []
    permuted = HipData._permuted

    def watched(self, perm):
        if self._t is moved._t:
            streams.append(torch.cuda.current_stream())
        return permuted(self, perm)

    monkeypatch.setattr(HipData, "_permuted", watched)
    lazy.contractAndCompressTowards(1, 5)
    assert streams == [torch.cuda.current_stream()]
    np.testing.assert_array_equal(lazy.state_center_data.toArray(), plain.state_center_data.toArray())
