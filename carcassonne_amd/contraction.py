"""Contractions of whole sets of channels in one launch (cc_contract_f64): operands and results keep their legs where
they lie, the outputs of a call share a launch, and the products that add to one output are added in it.

Shapes, strides and the resulting leg lists are memoised; nothing is kept about the tensors themselves.
"""
import ctypes

import torch

from . import _lib
from .device import empty, ptr, stream

_PLANS = {}
MAX_TERMS = 32   # products per output and launch


def _layout(data):
    """(device tensor, what its legs' strides follow from)."""
    if data.__dict__.get("_perm") is not None and data._lazy():
        return data._base, (data._base.shape, tuple(data._perm))
    t = data._t
    return t, (t.shape, None)


def _legs(shape, perm):
    strides, acc = [], 1
    for n in reversed(shape):
        strides.append(acc)
        acc *= n
    strides.reverse()
    perm = range(len(shape)) if perm is None else perm
    return [(int(shape[p]), strides[p]) for p in perm]


class _Plan:
    """Leg lists of one contraction; `ok` is False where the kernel does not take it (mismatched or empty legs, offsets
    beyond 32 bits, more than 12 legs in a group)."""

    def __init__(self, a, b, out, la, lb, terms):
        self.ok = False
        A, B = dict(zip(a, _legs(*la))), dict(zip(b, _legs(*lb)))
        if len(A) != len(a) or len(B) != len(b) or any(A[x][0] != B[x][0] for x in a if x in B):
            return
        self.shape = [A[x][0] if x in A else B[x][0] for x in out]
        if 0 in self.shape or any(A[x][0] == 0 for x in a):
            return
        C = dict(zip(out, _legs(self.shape, None)))
        m = [A[x] + (C[x][1],) for x in a if x in C]
        n = [B[x] + (C[x][1],) for x in b if x in C]
        k = [A[x] + (B[x][1],) for x in a if x not in C]
        if any(x in B for x in a if x in C) or any(x not in A for x in b if x not in C) or any(x not in B for x in a if x not in C):
            return
        self.legs = _lib.i64_array([v for leg in m + n + k for v in leg])
        self.counts = (len(m), len(n), len(k))
        self.terms = _lib.i32_array(terms)
        try:
            self.work = _lib.query("cc_contract_work_size", *self.counts, self.legs, len(terms), self.terms)
        except NotImplementedError:
            return
        self.ok = True


def _plan(a, b, out, la, lb, terms):
    key = (a, b, out, la, lb, terms)
    plan = _PLANS.get(key)
    if plan is None:
        plan = _Plan(a, b, out, la, lb, terms)
        if len(_PLANS) < 4096:
            _PLANS[key] = plan
    return plan


def _pointers(tensors):
    return (ctypes.c_void_p * len(tensors))(*[t.data_ptr() for t in tensors])


def contract(a, b, out, outputs, split_long_sums=False, together=False):
    """One device tensor per entry of `outputs`, each the sum of A B over its pairs (A, B): `a`, `b` and `out` name the
    legs of the first operands, the second ones and the results (a leg in both operands is summed, every other is in
    `out`).  split_long_sums: long sums with small results are summed in slices (their rounding then differs from one
    sum's, so only callers that ask for it get it).  together: the results are parts of one allocation (for intermediate
    tensors).  None where the kernel does not take the contraction."""
    if any(len(pairs) > MAX_TERMS for pairs in outputs):
        return None
    A = [_layout(x) for pairs in outputs for x, _ in pairs]
    B = [_layout(y) for pairs in outputs for _, y in pairs]
    la, lb = A[0][1], B[0][1]
    if any(l != la for _, l in A) or any(l != lb for _, l in B):
        return None
    plan = _plan(a, b, out, la, lb, tuple(len(pairs) for pairs in outputs))
    if not plan.ok:
        return None
    results = empty([len(outputs)] + plan.shape).unbind(0) if together else [empty(plan.shape) for _ in outputs]
    work = empty((plan.work,)) if plan.work and split_long_sums else None
    _lib.call("cc_contract_f64", stream(), *plan.counts, plan.legs, len(outputs), plan.terms,
              _pointers([t for t, _ in A]), _pointers([t for t, _ in B]), _pointers(results),
              ptr(work) if work is not None else None)
    return results
