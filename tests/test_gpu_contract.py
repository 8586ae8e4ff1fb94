"""Contractions with strided legs (cc_contract_f64 through carcassonne_amd.contraction) against NumPy in FP64: every tile
shape, both loader layouts, edges of tiles and of K steps, unit and unmergeable legs, several outputs and terms, split
sums, sums longer than the offset tables, permuted operands."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53


def _check(a, b, out, dims, terms, seed, permute=False, split=True):
    import torch
    from carcassonne_amd.contraction import contract
    from carcassonne_amd.data import HipData
    rng = np.random.default_rng(seed)
    A = [rng.standard_normal([dims[x] for x in a]) for _ in range(sum(terms))]
    B = [rng.standard_normal([dims[x] for x in b]) for _ in range(sum(terms))]

    def up(x):
        if not permute:
            return HipData.fromArray(x)
        back = np.argsort(np.arange(x.ndim)[::-1])     # stored with its legs reversed, seen through a permutation
        return HipData.fromArray(np.ascontiguousarray(x.transpose())).permuted_lazily(list(back))
    pairs = [(up(x), up(y)) for x, y in zip(A, B)]
    at = np.cumsum([0] + list(terms))
    got = contract(a, b, out, [pairs[at[o]:at[o + 1]] for o in range(len(terms))], split_long_sums=split)
    assert got is not None
    K = int(np.prod([dims[x] for x in a if x in b], dtype=np.int64))
    spec = "{},{}->{}".format(a, b, out)
    for o, t in enumerate(got):
        want = sum(np.einsum(spec, A[i], B[i], optimize=True) for i in range(at[o], at[o + 1]))
        size = sum(np.einsum(spec, abs(A[i]), abs(B[i]), optimize=True) for i in range(at[o], at[o + 1]))
        g = t.cpu().numpy()
        assert g.shape == want.shape
        # two FP64 sums of terms x K products, each within its length times EPS of the exact one
        assert np.all(abs(g - want) <= 2 * (terms[o] * K + 2) * EPS * size), (spec, o)
    torch.cuda.synchronize()


@pytest.mark.parametrize("a,b,out,dims,terms", [
    ("ik", "kj", "ij", dict(i=1, k=1, j=1), (1,)),
    ("ik", "kj", "ij", dict(i=33, k=31, j=65), (1, 2)),
    ("ik", "kj", "ji", dict(i=70, k=100, j=5), (3,)),                           # written along the first operand
    ("ki", "jk", "ij", dict(i=40, k=17, j=40), (1,)),
    ("ik", "kj", "ij", dict(i=20, k=5000, j=21), (1, 1, 1)),                    # split, longer than the tables
    ("ki", "kj", "ij", dict(i=700, k=1100, j=700), (2,)),                       # 64 x 64 tiles, two tables per term
    ("abk", "bkc", "ca", dict(a=5, b=6, k=7, c=3), (1,)),
    ("a", "b", "ba", dict(a=9, b=1), (1,)),                                     # nothing summed
    ("ab", "ab", "", dict(a=30, b=7), (1, 2)),                                  # everything summed
    ("abcdef", "ghiabcjk", "ghidjekf", dict(a=4, b=2, c=1, d=3, e=2, f=2, g=3, h=2, i=1, j=3, k=3), (2, 1)),
    ("abkyij", "iacos", "bkyjcos", dict(a=3, b=3, k=20, y=21, i=3, j=3, c=3, o=3, s=2), (1, 1)),
] + [("yxkab", "bocx", "ykaoc", dict(y=60, x=5, k=40, a=5, b=3, o=n, c=c), (1, 2, 1)) for n, c in
     ((4, 4), (5, 5), (6, 6), (7, 8), (9, 8), (9, 9))])                         # 16 to 80 columns and one past
@pytest.mark.parametrize("permute", [False, True])
def test_contract_matches_numpy(gpu, a, b, out, dims, terms, permute):
    for split in (False, True):
        _check(a, b, out, dims, terms, len(a) + 10 * len(b) + sum(dims.values()), permute, split)


@pytest.mark.parametrize("outputs", [15, 16, 17, 40])
def test_many_outputs_and_terms(gpu, outputs):
    """More outputs and terms than one launch takes (16 and 32)."""
    _check("ik", "kj", "ij", dict(i=12, k=9, j=14), tuple(1 + (o * 7) % 5 for o in range(outputs)), outputs)
    _check("ik", "kj", "ij", dict(i=12, k=40, j=14), (32, 1), outputs)


def test_what_is_left_to_the_general_path(gpu):
    """Mismatched or empty legs, mixed layouts and too many terms are not taken."""
    from carcassonne_amd.contraction import contract
    from carcassonne_amd.data import HipData
    x, y = HipData.newZeros((3, 4)), HipData.newZeros((4, 5))
    assert contract("ik", "kj", "ij", [[(x, x)]]) is None
    assert contract("ik", "kj", "ij", [[(HipData.newZeros((3, 0)), HipData.newZeros((0, 5)))]]) is None
    assert contract("ik", "kj", "ij", [[(x, y)], [(HipData.newZeros((2, 4)), y)]]) is None
    assert contract("ik", "kj", "ij", [[(x, y)] * 33]) is None
    assert contract("ik", "kj", "ij", [[(x, y)] * 32]) is not None
