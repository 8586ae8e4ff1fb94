"""How a stage-3 operator's terms are gathered into formed matrices (host side): every term is in exactly one
product with its coefficient, whatever channels the terms share."""
import numpy as np
import pytest


@pytest.mark.parametrize("seed", range(8))
def test_products_cover_every_term_once(seed):
    from carcassonne_amd.stage3 import products_of
    rng = np.random.default_rng(seed)
    pairs = {(int(rng.integers(0, 5)), int(rng.integers(0, 5))) for _ in range(12)}
    terms = [(a, b + 100, float(rng.integers(1, 9))) for a, b in sorted(pairs)]
    got = {}
    for left, right in products_of(terms):
        for a, ca in left:
            for b, cb in right:
                got[(a, b)] = got.get((a, b), 0.0) + ca * cb
    assert got == {(a, b): c for a, b, c in terms}


@pytest.mark.parametrize("same,others", [(2, 0), (8, 1), (9, 0), (17, 3)])
def test_products_add_equal_terms(same, others):
    """Terms of one pair of channels (one-site operators of one matrix under several tags) all count, past a sum's eight
    channels too."""
    from carcassonne_amd.stage3 import products_of
    terms = [(0, 100, 1.0)] * same + [(0, 101 + i, 2.0) for i in range(others)]
    got = {}
    for left, right in products_of(terms):
        for a, ca in left:
            for b, cb in right:
                got[(a, b)] = got.get((a, b), 0.0) + ca * cb
    assert got == dict([((0, 100), float(same))] + [((0, 101 + i), 2.0) for i in range(others)])


def test_star_of_terms_takes_two_products():
    from carcassonne_amd.stage3 import products_of
    # the identity channels (0 and 100) each meet several others
    terms = [(0, 101, 1.0), (0, 102, -1.0), (1, 100, 1.0), (2, 100, -1.0), (3, 100, 1.0)]
    assert len(products_of(terms)) == 2


def test_operator_groups_are_exact_multiples():
    from carcassonne_amd.stage3 import operator_groups
    values = {-1: (1.0, 0.0, 0.0, 1.0), 0: (1.0, 0.0, 0.0, -1.0), 1: (-1.0, 0.0, 0.0, 1.0), 2: (0.0, 1.0, 1.0, 0.0),
              3: (0.0, 0.0, 0.0, 0.0), 4: (0.0, 0.1, 0.1, 0.0), 5: (3.0, 0.0, 0.0, 3.0), 6: (0.0, 1.0, 0.0, 0.0)}
    groups = operator_groups(values)
    assert [sorted(k for k, _ in members) for _, members in groups] == [[-1, 5], [0, 1], [2, 4], [3], [6]]
    for first, members in groups:
        for k, c in members:
            assert tuple(c * x for x in values[first]) == values[k]
