"""Tag-rule lifts of the dense contractors.  Re-implements carcassonne/tensors/_2d/sparse.py:12-161:
the same rule tables (which tag pairs combine and the result tag), applied by
carcassonne_amd.sparse.contractSparseTensors.  Stage 3 gathers every compatible
(stage2_0 tag, stage2_1 tag, operator tag) triple into one Stage3Operator, so a
matvec of the whole expectation multiplier is a single HIP call.
"""
import math

from .dense import *  # noqa: F401,F403
from .dense import (absorbDenseCenterSOSIntoSide, absorbDenseCenterSOSIntoSideProjected, absorbDenseCenterSSIntoSide,
                    absorbDenseSideIntoCornerFromLeft,
                    absorbDenseSideIntoCornerFromRight, formNormalizationStage1, formNormalizationStage2)
from ...contraction import contract
from ...data import HipData, PermutedView
from ...sparse import (Complete, Identity, OneSiteOperator, TwoSiteOperator, TwoSiteOperatorCompressed,
                       addStandardCompleteAndIdentityTerms, contractSparseTensors, getInformationFromOperatorCenter,
                       matchSparseTensors)
from ...utils import L, O, R
from ... import stage3


def _contract_channels(a, b, out, finish, rules, tensor_1, tensor_2):
    """contractSparseTensors for rules that all stand for one dense contraction (`a`, `b`, `out`: its legs, `finish`: what
    makes a channel of its result): every result channel in one launch; the pairwise loop where the channels do not
    all have one layout."""
    matched = matchSparseTensors(rules, tensor_1, tensor_2)
    results = None
    if matched and all(isinstance(x, HipData) for t in (tensor_1, tensor_2) for x in t.values()):
        results = contract(a, b, out, [[(x, y) for x, y, _ in pairs] for pairs in matched.values()])
    if results is None:
        return contractSparseTensors(rules, tensor_1, tensor_2)
    return {tag: finish(t) for tag, t in zip(matched, results)}


def _joined(*groups):
    """A result with its legs joined in groups of the given sizes."""
    def finish(t):
        shape, at = [], 0
        for n in groups:
            shape.append(math.prod(t.shape[at:at + n]))
            at += n
        return HipData(t.reshape(shape))
    return finish


def absorbSparseSideIntoCornerFromLeft(corner, side):
    """sparse.py:12-23 (handler arguments: corner tag, side tag)."""
    terms = {}
    f = absorbDenseSideIntoCornerFromLeft
    addStandardCompleteAndIdentityTerms(terms, f)
    terms.update({
        (TwoSiteOperator, Identity): lambda c, s: (c.matchesSideIdentityOnLeft(), f),
        (Identity, TwoSiteOperator): lambda c, s: (s.matchesCornerIdentityOnRight(), f),
        (TwoSiteOperator, TwoSiteOperator): lambda c, s: (s.matches(c), f),
        (TwoSiteOperatorCompressed, TwoSiteOperatorCompressed): lambda c, s: (s.matches(c), f),
    })
    return _contract_channels("abcdef", "ghiabcjk", "ghidjekf", _joined(1, 1, 1, 2, 2, 1), terms, corner, side)


def absorbSparseSideIntoCornerFromRight(corner, side):
    """sparse.py:24-35 (the compressed rule binds side.matches(corner), as written there)."""
    terms = {}
    f = absorbDenseSideIntoCornerFromRight
    addStandardCompleteAndIdentityTerms(terms, f)
    terms.update({
        (TwoSiteOperator, Identity): lambda c, s: (c.matchesSideIdentityOnRight(), f),
        (Identity, TwoSiteOperator): lambda c, s: (s.matchesCornerIdentityOnLeft(), f),
        (TwoSiteOperator, TwoSiteOperator): lambda c, s: (c.matches(s), f),
        (TwoSiteOperatorCompressed, TwoSiteOperatorCompressed): lambda c, s: (s.matches(c), f),
    })
    return _contract_channels("abcdef", "defghijk", "ajbkcghi", _joined(2, 2, 1, 1, 1, 1), terms, corner, side)


def _center_into_side_terms(direction, ss, sos):
    """The rule table of absorbSparseCenterSOSIntoSide (sparse.py:36-58): (side tag, operator tag) ->
    (result tag, dense contractor) with ss for the identity-operator pairs and sos for the others."""
    return {
        (Identity, Identity): lambda s, c: (Identity(), ss),
        (Complete, Identity): lambda s, c: (Complete(), ss),
        (Identity, OneSiteOperator): lambda s, c: (Complete(), sos),
        (TwoSiteOperator, Identity): lambda s, c: (s.matchesCenterIdentity(), ss),
        (Identity, TwoSiteOperator): lambda s, c: (c.matchesSideIdentityOutward(direction), sos),
        (TwoSiteOperator, TwoSiteOperator): lambda s, c: (s.matchesCenter(direction, c), sos),
        (TwoSiteOperatorCompressed, Identity): lambda s, c: (s, ss),
    }


def absorbSparseCenterSOSIntoSide(direction, side, state_center_data, operator_center_data, state_center_data_conj=None):
    """sparse.py:36-58 (handler arguments: side tag, operator tag)."""
    if state_center_data_conj is None:
        state_center_data_conj = state_center_data.conj()

    def ss(side_data, _):
        return absorbDenseCenterSSIntoSide(direction, side_data, state_center_data, state_center_data_conj)

    def sos(side_data, op_data):
        return absorbDenseCenterSOSIntoSide(direction, side_data, state_center_data, op_data, state_center_data_conj)
    return contractSparseTensors(_center_into_side_terms(direction, ss, sos), side, operator_center_data)


def absorbSparseCenterSOSIntoSideProjected(direction, side, state_center_data, operator_center_data, left, right,
                                           state_center_data_conj=None):
    """absorbSparseCenterSOSIntoSide with every result channel projected onto the fused truncation bases
    `left` (the bond to corner `direction`) and `right` (the bond to corner R(direction)) as it is formed
    (absorbDenseCenterSOSIntoSideProjected): the same rule table, no grown side in memory."""
    if state_center_data_conj is None:
        state_center_data_conj = state_center_data.conj()

    def ss(side_data, _):
        return absorbDenseCenterSOSIntoSideProjected(direction, side_data, state_center_data, None, left, right,
                                                     state_center_data_conj)

    def sos(side_data, op_data):
        return absorbDenseCenterSOSIntoSideProjected(direction, side_data, state_center_data, op_data, left, right,
                                                     state_center_data_conj)
    rules = _center_into_side_terms(direction, ss, sos)
    result = _project_channels(direction, matchSparseTensors(rules, side, operator_center_data), sos, state_center_data,
                               state_center_data_conj, left, right)
    return contractSparseTensors(rules, side, operator_center_data) if result is None else result


def _project_channels(direction, matched, sos, state, state_conj, left, right):
    """The result channels `matched` (matchSparseTensors) of the projected absorption, four launches for all of them: a
    side channel meets the left basis and the center once, whatever number of operators it meets after that, and the
    products that add to one channel meet the right basis once.  The operators act on the conjugate center, O[s', s]
    from its s' side.  None where the channels do not all have one layout."""
    pairs = [p for products in matched.values() for p in products]
    if not pairs or not all(isinstance(t, HipData) for p in pairs for t in p[:2] if t is not None):
        return None
    sh = pairs[0][0].shape
    if len(sh) != 8 or sh[1] * sh[2] * sh[4] * sh[5] != 1 or any(p[0].shape != sh for p in pairs):
        return None
    x, y, i = sh[0], sh[3], direction
    legs = [None] * 5
    conj = [None] * 5
    for at, ket, bra in ((i, "i", "j"), (L(i), "a", "b"), (R(i), "c", "e"), (O(i), "o", "p"), (4, "s", "s")):
        legs[at], conj[at] = ket, bra
    legs, conj = "".join(legs), "".join(conj)
    D_a, D_c = state.shape[L(i)], state.shape[R(i)]
    if left.shape[0] != x * D_a * D_a or right.shape[0] != y * D_c * D_c:
        return None
    lt, rt = left.split(x, D_a, D_a, left.shape[1]), right.split(y, D_c, D_c, right.shape[1])
    sides = {id(p[0]): p[0] for p in pairs}
    operators = {id(p[1]): p[1] for p in pairs if p[2] is sos}
    grown = contract("xabk", "xyij", "abkyij", [[(lt, t.split(x, y, sh[6], sh[7]))] for t in sides.values()],
                     together=True)
    if grown is None:
        return None
    met = contract("abkyij", legs, "bkyjcos", [[(HipData._wrap(t), state)] for t in grown], together=True)
    acted = contract("ts", conj.replace("s", "t"), conj, [[(op, state_conj)] for op in operators.values()],
                     together=True) if operators else []
    if met is None or acted is None:
        return None
    met = {key: HipData._wrap(t) for key, t in zip(sides, met)}
    acted = {key: HipData._wrap(t) for key, t in zip(operators, acted)}
    summed = contract("bkyjcos", conj, "kycoep",
                      [[(met[id(t)], acted[id(op)] if f is sos else state_conj) for t, op, f in products]
                       for products in matched.values()], together=True)
    if summed is None:
        return None
    out = contract("kycoep", "yceq", "kqop", [[(HipData._wrap(t), rt)] for t in summed], split_long_sums=True)
    if out is None:
        return None
    return {tag: HipData(t.reshape(t.shape[0], 1, 1, t.shape[1], 1, 1, t.shape[2], t.shape[3]))
            for tag, t in zip(matched, out)}


def formExpectationStage1(corner, side):
    """sparse.py:72-85 (handler arguments: corner tag, side tag)."""
    terms = {}
    f = formNormalizationStage1
    addStandardCompleteAndIdentityTerms(terms, f)
    terms.update({
        (TwoSiteOperator, Identity): lambda c, s: (c.matchesSideIdentityOnRightForStage1(), f),
        (Identity, TwoSiteOperator): lambda c, s: (s.matchesCornerIdentityOnLeftForStage1(), f),
        (TwoSiteOperator, TwoSiteOperator): lambda c, s: (c.matches(s), f),
        (TwoSiteOperatorCompressed, Identity): lambda c, s: (c.matchesSideIdentityOnRightForStage1(), f),
        (Identity, TwoSiteOperatorCompressed): lambda c, s: (s.matchesCornerIdentityOnLeftForStage1(), f),
        (TwoSiteOperatorCompressed, TwoSiteOperatorCompressed): lambda c, s: (c.matches(s), f),
    })
    return _contract_channels("abcdef", "defghijk", "abcghijk", _joined(3, 3, 1, 1), terms, corner, side)


def formExpectationStage2(right, left):
    """sparse.py:86-99 (handler arguments: right tag, left tag)."""
    terms = {}
    f = formNormalizationStage2
    addStandardCompleteAndIdentityTerms(terms, f)
    terms.update({
        (TwoSiteOperator, Identity): lambda r, l: (r.matchesStage1IdentityOnLeft(), f),
        (Identity, TwoSiteOperator): lambda r, l: (l.matchesStage1IdentityOnRight(), f),
        (TwoSiteOperator, TwoSiteOperator): lambda r, l: (l.matches(r), f),
        (TwoSiteOperatorCompressed, Identity): lambda r, l: (r.matchesStage1IdentityOnLeft(), f),
        (Identity, TwoSiteOperatorCompressed): lambda r, l: (l.matchesStage1IdentityOnRight(), f),
        (TwoSiteOperatorCompressed, TwoSiteOperatorCompressed): lambda r, l: (l.matches(r), f),
    })
    # in the product's own leg order; the packers read the slabs through strides
    return _contract_channels("abcd", "eafg", "bcdefg", lambda t: PermutedView(t, [3, 0, 1, 4, 2, 5]), terms, right, left)


STAGE3_RULES = {
    (Complete, Identity, Identity): lambda x, y, z: True,
    (Identity, Complete, Identity): lambda x, y, z: True,
    (Identity, Identity, OneSiteOperator): lambda x, y, z: True,
    (TwoSiteOperator, Identity, TwoSiteOperator): lambda x, y, z: x.matchesCenterForStage3(0, z),
    (Identity, TwoSiteOperator, TwoSiteOperator): lambda x, y, z: y.matchesCenterForStage3(1, z),
    (TwoSiteOperator, TwoSiteOperator, Identity): lambda x, y, z: x.matchesForStage3(y),
    (TwoSiteOperatorCompressed, TwoSiteOperatorCompressed, Identity): lambda x, y, z: x.matchesForStage3(y),
}


_STAGE3_BY_PAIR = {}   # (type, type) of the stage-2 tags -> type of the operator's tag -> rule
for (_x, _y, _z), _rule in STAGE3_RULES.items():
    _STAGE3_BY_PAIR.setdefault((_x, _y), {})[_z] = _rule


def stage3_terms(stage2_0, stage2_1, operator_center):
    """The compatible tag triples in the reference's enumeration order (sparse.py:116-127),
    as (stage2_0 data, stage2_1 data, operator data or None for an identity operator)."""
    terms = []
    for x, data_0 in stage2_0.items():
        for y, data_1 in stage2_1.items():
            rules = _STAGE3_BY_PAIR.get((type(x), type(y)))
            if rules is None:
                continue
            for z, op in operator_center.items():
                rule = rules.get(type(z))
                if rule is not None and rule(x, y, z):
                    terms.append((data_0, data_1, None if type(z) is Identity else op))
    return terms


def formExpectationStage3(stage2_0, stage2_1, operator_center):
    """sparse.py:100-161: (expectation multiplier, normalization multiplier)."""
    d, _, DataClass = getInformationFromOperatorCenter(operator_center)
    terms = stage3_terms(stage2_0, stage2_1, operator_center)
    normalization = stage3.Stage3Operator([(stage2_0[Identity()], stage2_1[Identity()], None)], physical_dimension=d)
    if terms:
        expectation = stage3.Stage3Operator(terms, physical_dimension=d).multiplier()
    else:
        from ...utils import Multiplier
        n = normalization.n

        def zero(v):
            return v.newZeros(v.shape)
        expectation = Multiplier((n, n), zero, 0, lambda: DataClass.newZeros((n, n)), 0)
    return expectation, normalization.multiplier()


def formExpectationAndNormalizationMultipliers(corners, sides, operator_center_data):
    """sparse.py:59-71."""
    return formExpectationStage3(
        formExpectationStage2(formExpectationStage1(corners[0], sides[0]), formExpectationStage1(corners[1], sides[1])),
        formExpectationStage2(formExpectationStage1(corners[2], sides[2]), formExpectationStage1(corners[3], sides[3])),
        operator_center_data)
