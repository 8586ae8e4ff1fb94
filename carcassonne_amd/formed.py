"""The stage-3 operator of one solve formed as dense matrices over the environment legs.

    H = sum_t A_t (x) B_t (x) O_t = sum_g O_g (x) G_g,    G_g = sum over the terms with operator O_g of A_t (x) B_t

with one group per distinct site operator (up to a factor) and the terms summed over shared channels first
(Stage3Operator._merged).  The reference forms the matrix of an operator when enough multiplications follow
(Multiplier.isCheaperToFormMatrix, carcassonne/utils.py:203-206; formDenseStage3_formMatrix,
carcassonne/tensors/_2d/dense.py:176-203).  Here the solvers that may form it always do: a whole solve breaks even after
4 to 8 Lanczos steps (4 at D = 4, chi = 32: 0.74 ms either way; 5 for Heisenberg at D = 5, chi = 45; 8 at D = 6, chi = 64:
2.70 formed, 2.76 through the slabs; 2.64 and 2.11 ms after the first check at 4), and 50 to 80 are usual.  The product
of the identity channels is the normalization matrix N: it is not formed again, and in whitened form (W N W^T = 1 for
N = L L^T, W = L^-1) it is the identity.
"""
import ctypes

import torch

from . import _lib
from .device import empty, ptr, stream

MAX_PRODUCTS, MAX_MATRICES = 16, 4


class FormedOperator:
    """The formed matrices of a stage-3 operator, one set per solver: apply_flat(x, y) is y = H x.  `factor`: the
    normalization factor of the same environment, whose matrix is the identity channels' product."""

    @staticmethod
    def of(h_operator, n_operator, factor):
        """Formed matrices of the operator; None where it has no such form (no fused shape, more distinct site operators
        or products than one call takes, or an operator refreshed from another: only its packed slabs hold that
        environment, its own channels are those it was built from)."""
        layout = FormedOperator._layout(h_operator, n_operator)
        h_operator._formed = FormedOperator(h_operator, factor, layout) if layout is not None else None
        return h_operator._formed

    @staticmethod
    def _layout(h_operator, n_operator):
        """([(O_g, [(A sum, B sum)...])...], identity): the matrices to form, by site operator, and the site operator
        of the identity channels' product (None: there is no such term)."""
        if not h_operator.use_fused or h_operator.d != 2 or h_operator._refreshed:
            return None
        channels, specs, ops, rows = h_operator._merged()
        values = [tuple(float(x) for x in o.toArray().reshape(-1)) for o in ops] + [(1.0, 0.0, 0.0, 1.0)]   # [-1]: 1
        groups, identity = {}, None
        for a, b, o in rows:
            left, right = specs[0][a], specs[1][b]
            if len(left) == len(right) == 1 and channels[0][left[0][0]] is n_operator._A[0] \
                    and channels[1][right[0][0]] is n_operator._B[0]:
                c = left[0][1] * right[0][1]
                identity = [x + c * y for x, y in zip(identity or (0.0,) * 4, values[o])]
            else:
                groups.setdefault(o, []).append((a, b))
        if len(groups) > MAX_MATRICES or sum(map(len, groups.values())) > MAX_PRODUCTS or (not groups and identity is None):
            return None
        return [(values[o], products) for o, products in groups.items()], identity

    def __init__(self, h_operator, factor, layout):
        self.n_env, self.d = h_operator.n // h_operator.d, h_operator.d
        self._groups, self.identity = layout
        self.ops = [O for O, _ in self._groups]
        self.factor = factor
        self._shape = (h_operator.n_alpha, h_operator.P)
        self._plan = None
        self.G = empty((len(self._groups), self.n_env, self.n_env))
        self._form(h_operator.joined)

    def _form(self, joined):
        """G from the joined sums of channels joined(half, k)."""
        self._version = self.factor.version     # counted on the host, at capture in a graph: with the refresh of all three
        if not self._groups:
            return
        na, P = self._shape
        A = [joined(0, a) for _, products in self._groups for a, _ in products]
        B = [joined(1, b) for _, products in self._groups for _, b in products]
        begin = [0]
        for _, products in self._groups:
            begin.append(begin[-1] + len(products))
        work = empty((_lib.query("cc_form_work_size", len(self._groups), max(len(p) for _, p in self._groups), na, P, P),))
        _lib.call("cc_form_f64", stream(), len(self._groups), _lib.i32_array(begin),
                  _lib.ptr_array([t.data_ptr() for t in A]), _lib.ptr_array([t.data_ptr() for t in B]), na, P, P,
                  ptr(self.G), ptr(work))

    def refresh(self, h_operator, other, factor):
        """Forms `other`, an operator of h_operator's structure from a new environment that the factor holds already,
        into these matrices; h_operator then applies it too (kernels only: capturable in a HIP graph)."""
        channels = h_operator.same_structure(other)
        if factor is not self.factor:
            self.factor, self._plan = factor, None
        h_operator.refresh_fused_from(other)
        _, specs, _, _ = h_operator._merged()
        h_operator._joined = {(side, k): h_operator.joined(side, k, channels)
                              for side in (0, 1) for k in range(len(specs[side]))}
        self._form(h_operator.joined)

    def valid(self, factor):
        """Whether `factor` is the factor formed beside and still holds that environment."""
        return factor is self.factor and factor.version == self._version

    def apply_flat(self, x, y):
        if self._plan is None:
            mats, ops = [self.G[g] for g in range(len(self.ops))], list(self.ops)
            if self.identity is not None:
                mats, ops = mats + [self.factor.N_env], ops + [self.identity]
            self._plan = FormedPlan(self.n_env, self.d, mats, ops, None)
        self._plan.apply(x, y)

    def whitened(self, factor, f32=None):
        """The plan of W H W^T with the factor's W = L^-1 (two triangular products per matrix).  f32: an FP32 array of
        G's shape that the matrices are rounded into, for inner steps that need no more."""
        K = empty(self.G.shape)
        if self.ops:
            work = empty(self.G.shape)
            _lib.call("cc_whiten_f64", stream(), self.n_env, len(self.ops), ptr(self.G), ptr(factor.Wt), ptr(K), ptr(work))
            if f32 is not None:
                _lib.call("cc_cast", stream(), K.numel(), _lib.CC_F64, ptr(K), _lib.CC_F32, ptr(f32))
        K = K if f32 is None else f32
        return FormedPlan(self.n_env, self.d, [K[g] for g in range(len(self.ops))], self.ops, self.identity)


class FormedPlan:
    """A native plan (cc_formed_plan_create) of sum_g O_g (x) M_g + identity (x) 1, holding its matrices."""

    def __init__(self, n_env, d, mats, ops, identity):
        self.mats, self.handle = mats, ctypes.c_void_p()
        _lib.call("cc_formed_plan_create_f32" if mats and mats[0].dtype == torch.float32 else "cc_formed_plan_create", ctypes.byref(self.handle), n_env, d, len(mats),
                  _lib.ptr_array([m.data_ptr() for m in mats]), _lib.f64_array([x for O in ops for x in O]),
                  _lib.f64_array(identity) if identity is not None else None)

    def apply(self, x, y):
        _lib.call("cc_formed_plan_apply", stream(), self.handle, ptr(x), ptr(y))

    def __del__(self):
        if getattr(self, "handle", None):
            try:
                _lib.load().cc_formed_plan_destroy(self.handle)
            except Exception:
                pass
