"""The FP64 slab matvec against the generic path for every padded slab extent (K steps of 4, tiles of 16): the smallest,
full and ragged ones, equal and unequal center bonds, environment bonds that leave teams of waves without work; and for
term tables that exercise the summed channels and the common stage B (several terms per channel, operators that are
multiples of one another, more distinct operators on one channel than it takes, single terms).  Tolerance: FP64 sums of
at most 2^15 products in another order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

OPS = [None, np.diag([1.0, -1.0]), np.diag([-2.0, 2.0]), np.array([[0.0, 1.0], [1.0, 0.0]]), np.array([[0.0, 3.0], [-1.0, 0.0]]),
       np.array([[0.5, 0.25], [0.125, 2.0]]), np.array([[0.0, 0.0], [1.0, 0.0]])]
STAR = [(0, 0, 3), (0, 1, None), (1, 0, None), (2, 0, 1), (3, 0, 2), (0, 2, 1), (0, 3, 2)]
MANY = [(a, 0, o) for a, o in ((0, 0), (1, 1), (2, 3), (3, 4), (0, 5), (1, 6))] + [(2, 1, 4), (3, 2, 0), (3, 3, 5)]
ONE = [(0, 0, 5)]


def _operator(D0, D1, chi, table, seed):
    from carcassonne_amd.data import HipData
    from carcassonne_amd.stage3 import Stage3Operator
    rng = np.random.default_rng(seed)
    halves = [[HipData.fromArray(rng.standard_normal((chi, chi, D0, D1, D0, D1))) for _ in range(4)] for _ in range(2)]
    ops = [None if o is None else HipData.fromArray(o) for o in OPS]
    op = Stage3Operator([(halves[0][a], halves[1][b], None if o is None else ops[o]) for a, b, o in table],
                        physical_dimension=2)
    return op, HipData.fromArray(rng.standard_normal((D0, D1, D0, D1, 2)))._t.reshape(-1)


@pytest.mark.parametrize("D0,D1,chi", [(1, 1, 3), (1, 2, 2), (2, 1, 9), (3, 1, 5), (2, 2, 7), (1, 5, 4), (2, 3, 11), (4, 2, 6),
                                       (3, 3, 5), (5, 2, 3), (3, 4, 13), (7, 2, 3), (3, 5, 4), (4, 4, 3), (3, 6, 5), (4, 5, 7),
                                       (7, 3, 4), (6, 4, 3), (5, 5, 7), (9, 3, 2), (5, 6, 5), (8, 4, 3), (11, 3, 3), (6, 6, 5)])
@pytest.mark.parametrize("table", [STAR, MANY, ONE], ids=["star", "many", "one"])
def test_slab_matvec_matches_generic(gpu, D0, D1, chi, table):
    import torch
    op, x = _operator(D0, D1, chi, table, 100 * D0 + D1)
    assert op._use_slabs
    want, got = torch.empty_like(x), torch.full_like(x, float("nan"))
    op.apply_generic_flat(x, want)
    op.apply_flat(x, got)
    assert float((got - want).norm() / want.norm()) < 1e-13


@pytest.mark.parametrize("table", [STAR, MANY], ids=["star", "many"])
def test_slab_matvec_of_a_kept_copy(gpu, table):
    """A snapshot's joined channels give the same matvec as packing from the stage-2 tensors."""
    import torch
    op, x = _operator(3, 4, 6, table, 5)
    other, _ = _operator(3, 4, 6, table, 5)
    want, got = torch.empty_like(x), torch.empty_like(x)
    op.apply_flat(x, want)
    other.snapshot()
    other.apply_flat(x, got)
    assert torch.equal(got, want)


@pytest.mark.parametrize("D0,D1,chi", [(2, 2, 5), (3, 4, 6)])
def test_refresh_from_channels_of_other_layouts(gpu, D0, D1, chi):
    """An operator whose sums add channels of one layout is refreshed from one where a channel of each sum lies with its
    legs in another order."""
    import torch
    from carcassonne_amd.data import HipData, PermutedView
    from carcassonne_amd.stage3 import Stage3Operator
    op, x = _operator(D0, D1, chi, STAR, 5)
    assert max(len(spec) for side in op._merged()[1] for spec in side) > 1
    other, _ = _operator(D0, D1, chi, STAR, 6)
    order = [3, 0, 1, 4, 2, 5]                  # leg p of the channel is leg order[p] of the stored tensor
    moved = {}

    def view(t):
        if id(t) not in moved:
            moved[id(t)] = PermutedView(t._t.permute([order.index(k) for k in range(6)]).contiguous(), order)
        return moved[id(t)]

    a_list, b_list = ([ch.t for ch in chans] for chans in other._channels()[:2])
    terms = [(view(a) if a is a_list[1] else a, view(b) if b is b_list[2] else b, o) for a, b, o in other.terms]
    mixed = Stage3Operator(terms, physical_dimension=2)
    want, got = torch.empty_like(x), torch.empty_like(x)
    other.apply_generic_flat(x, want)
    op.apply_flat(x, got)
    op.refresh_fused_from(mixed)
    op.apply_flat(x, got)
    assert float((got - want).norm() / want.norm()) < 1e-13


def test_snapshot_of_an_applied_operator_joins_only(gpu):
    """The plan of an operator that was applied holds its packed sums: a snapshot adds the joined ones and nothing else."""
    import torch
    op, x = _operator(4, 4, 12, STAR, 5)
    op.apply_flat(x, torch.empty_like(x))
    used = torch.cuda.memory_allocated()
    op.snapshot()
    sums = sum(len(specs) for specs in op._merged()[1])
    assert op._packs == {}
    assert torch.cuda.memory_allocated() - used <= sums * (12 * 12 * 16 * 16 * 8 + 512)
