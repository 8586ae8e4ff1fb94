"""relaxOver's native restart (cc_relax_krylov_f64) against the loop over any multiplier, and the dense matrix of a
stage-3 operator in two contractions against the product of its terms one by one: the same operations in the same
order, so the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(1, 1), (2, 2), (7, 3), (32, 3), (65, 5), (162, 3), (300, 16), (1100, 2)])
@pytest.mark.parametrize("inverse", ["none", "cholesky", "svd"])
def test_restart_equals_the_general_loop(gpu, n, k, inverse):
    import torch
    from carcassonne_amd import _lib
    from carcassonne_amd.data import HipData
    from carcassonne_amd.device import ptr, stream
    from carcassonne_amd.solver import _DenseInverse, _FormedKrylov, _Krylov
    if inverse == "svd" and n > 256:
        pytest.skip("indefinite matrices are inverted up to n = 256")
    rng = np.random.default_rng(n + k)
    H = rng.standard_normal((n, n))
    H = HipData.fromArray(H + H.T).tensor()
    inv = None
    if inverse != "none":
        X = rng.standard_normal((n, n))
        N = X @ X.T / n + np.eye(n) if inverse == "cholesky" else X + X.T - 3.0 * np.eye(n)
        inv = _DenseInverse(HipData.fromArray(N))
        assert n == 1 or (inv.Ninv is not None) == (inverse == "svd")

    def multiply(x):
        y = torch.empty_like(x)
        _lib.call("cc_skinny_f64", stream(), n, 0, ptr(H), 1, ptr(x), ptr(y))
        return y if inv is None else inv(y)
    v = HipData.fromArray(rng.standard_normal(n)).tensor()
    native, general = _FormedKrylov(v, k, H, inv), _Krylov(v, k, multiply)
    coefficients = [1.0]
    for _ in range(3):
        a, b = native.restart(coefficients), general.restart(coefficients)
        assert a.shape == b.shape and np.array_equal(a, b)
        coefficients = rng.standard_normal(len(a))
    (x, value), (y, want) = native.finish(coefficients), general.finish(coefficients)
    assert np.array_equal(x.cpu().numpy(), y.cpu().numpy()) and value == want


def test_basis_ends_early(gpu):
    """An invariant subspace of two dimensions ends the basis after two vectors."""
    import torch
    from carcassonne_amd.solver import _FormedKrylov
    H = torch.diag(torch.tensor([1.0, 2.0, 3.0, 4.0], dtype=torch.float64)).cuda()
    v = torch.tensor([3.0, 4.0, 0.0, 0.0], dtype=torch.float64).cuda()
    native = _FormedKrylov(v, 4, H, None)
    M = native.restart([1.0])
    assert M.shape == (2, 2)
    np.testing.assert_allclose(np.linalg.eigvalsh(0.5 * (M + M.T)), [1.0, 2.0], atol=1e-14)
    assert native.restart([0.8, -0.6]).shape[0] <= 2      # an eigenvector or what rounding leaves beside it


@pytest.mark.parametrize("D,chi,model", [(2, 8, "ising"), (3, 7, "ising"), (2, 5, "heisenberg"), (1, 3, "ising")])
def test_dense_matrix_of_an_operator(gpu, D, chi, model):
    import torch
    from carcassonne_amd import pipeline, synthetic as syn
    from carcassonne_amd.tensors._2d.dense import _form_matrix
    c, s, _ = syn.make_environment(D, chi, model=model, seed=3)
    op = syn.operator_center(model)
    H, N = pipeline.multipliers(*pipeline.device_environment(c, s, op), graph=False)
    for operator in (H.operator, N.operator):
        eye = torch.eye(2, dtype=torch.float64).cuda()
        from carcassonne_amd.data import HipData
        want = None
        for a, b, o in operator.terms:
            t = _form_matrix(a, b, o if o is not None else HipData(eye))
            want = t if want is None else want + t
        assert torch.equal(operator.form_matrix().tensor(), want.tensor())
