"""The center-site effective-Hamiltonian operator of one solve.

Re-implements formNormalizationStage3 / formDenseStage3 / multiplyExpectation
(carcassonne/tensors/_2d/dense.py:115-203, carcassonne/tensors/_2d/sparse.py:129-148):

    (H v)[p', q', s'] = sum_t sum_alpha sum_{p,q,s} A_t[alpha][p'][p] B_t[alpha][q'][q] O_t[s'][s] v[p, q, s]

with A_t = stage2_0.join((0,1),4,5,2,3) and B_t = stage2_1.join((1,0),4,5,2,3) -- the
alpha-major slab layout -- and O_t the center operator (identity for the
normalization contractor).  All terms of a solve are applied in one call to the
HIP library: the fused MFMA kernel for the instantiated slab shapes, the generic
GEMM path for any other shape.
"""
import ctypes
import functools
import weakref

import numpy as np
import torch

from . import _lib
from .contraction import contract
from .data import HipData
from .device import empty, ptr, stream


def cost_of_term(n_alpha, P1, P, Q1, Q, d, with_op):
    """The reference's CostTracker count (complex MACs) of one stage-3 contractor:
    [O<->v], then A<->v over (D0,D1), then B<->T over (D2,D3,alpha)."""
    c = (d * P * Q) * d if with_op else 0
    c += (n_alpha * P1 * Q * d) * P
    c += (Q1 * P1 * d) * (Q * n_alpha)
    return int(c)


def cost_of_matrix(s2_0_shape, s2_1_shape, d):
    x, y, k0, k1, b0, b1 = s2_0_shape
    _, _, k2, k3, b2, b3 = s2_1_shape
    m = k0 * k1 * b0 * b1 * k2 * k3 * b2 * b3
    return int(m * x * y + m * d * d)


MAX_SUM = 8   # channels of one sum (cc_slab_join_f64, cc_stage3_pack_sum_f64)


def operator_groups(values):
    """values: key -> matrix as a tuple of numbers.  Returns [(key, [(key', c)...])]: every matrix in the one group
    whose first matrix it is an exact multiple of, values[key'] == c * values[key]."""
    groups = []
    for key, m in values.items():
        for first, members in groups:
            o = values[first]
            k = max(range(len(o)), key=lambda i: abs(o[i]))
            c = m[k] / o[k] if o[k] != 0 else 0.0
            if c != 0 and all(c * x == y for x, y in zip(o, m)):
                members.append((key, c))
                break
        else:
            groups.append((key, [(key, 1.0)]))
    return groups


def products_of(terms):
    """The terms (a, b, c) of one site operator as products ([(a, c)...], [(b, c)...]), a sum of A channels times a sum
    of B channels: the channel with the most terms left takes them all as one product, MAX_SUM at a time.  Terms of one
    pair of channels are one term first, with their coefficients added."""
    pairs, out = {}, []
    for a, b, c in terms:
        pairs[(a, b)] = pairs.get((a, b), 0.0) + c
    left = [(a, b, c) for (a, b), c in pairs.items()]
    while left:
        count = {}
        for a, b, _ in left:
            count[(0, a)] = count.get((0, a), 0) + 1
            count[(1, b)] = count.get((1, b), 0) + 1
        side, hub = max(count, key=lambda k: count[k])
        mine = [t for t in left if t[side] == hub][:MAX_SUM]
        left = [t for t in left if t not in mine]
        if side == 0:
            out.append(([(hub, 1.0)], [(b, c) for _, b, c in mine]))
        else:
            out.append(([(a, c) for a, _, c in mine], [(hub, 1.0)]))
    return out


_MERGES = {}   # merged_terms by what it depends on


def merged_terms(d, rows, values, legs):
    """(specs, table) of Stage3Operator._merged from the term table, the numbers of the site operators and the legs and
    strides of the channels."""
    values = dict(enumerate(values))
    values[-1] = tuple(float(i == j) for i in range(d) for j in range(d))
    products = []
    for o, members in operator_groups({o: values[o] for o in (-1, *range(len(values) - 1))}):
        factor = dict(members)
        edges = [(ia, ib, factor[oo]) for ia, _, ib, oo in rows if oo in factor]
        for left, right in products_of(edges) if edges else ():
            if any(len({legs[side][i] for i, _ in part}) > 1 for side, part in ((0, left), (1, right))):
                products += [(((i, ci),), ((j, cj),), o) for i, ci in left for j, cj in right]
            else:
                products.append((tuple(left), tuple(right), o))
    specs = [list(dict.fromkeys(p[side] for p in products)) for side in (0, 1)]
    if max(map(len, specs)) > 16 or len(products) > 48:
        specs = [[((i, 1.0),) for i in range(len(legs[side]))] for side in (0, 1)]
        products = [(specs[0][ia], specs[1][ib], o) for ia, _, ib, o in rows]
    return specs, sorted((specs[0].index(left), specs[1].index(right), o) for left, right, o in products)


def _alike(channels):
    return len(channels) == 1 or len({ch.source()[1:] for ch in channels}) == 1


def join_slabs(channels, coefs):
    """sum coefs[i] * channels[i] as a contiguous (alpha, P, P) array, in one pass where the channels share their leg sizes
    and strides."""
    if not _alike(channels):
        out = join_slabs(channels[:1], coefs[:1])
        for ch, c in zip(channels[1:], coefs[1:]):
            _lib.call("cc_axpby_f64", stream(), out.numel(), 1.0, ptr(join_slabs([ch], [c])), 1.0, ptr(out))
        return out
    _, (na0, na1, d0, d1), st = channels[0].source()
    out = empty((na0 * na1, d0 * d1, d0 * d1))
    if out.numel() == 0:
        return out
    _lib.call("cc_slab_join_f64", stream(), len(channels), _lib.ptr_array([c.source()[0].data_ptr() for c in channels]),
              _lib.f64_array(coefs), na0, na1, d0, d1, _lib.i64_array(st), ptr(out))
    return out


@functools.lru_cache(maxsize=4096)
def _packed_size(n_alpha, P):
    return _lib.query("cc_stage3_packed_size", n_alpha, P)


class _Slab:
    """One slab channel of a stage-3 operator: the stage-2 tensor t read as slab[alpha][p'][p] with
    which 0: alpha = (t0, t1) (stage2_0.join((0,1),4,5,2,3)), which 1: alpha = (t1, t0)
    (stage2_1.join((1,0),4,5,2,3)); p' = (t4, t5), p = (t2, t3).  The FP64 packing for the fused kernel
    and the low-precision conversion read t in place through strides; the joined (alpha, P, P) array
    is formed only on request (generic path, normalization matrix).  One _Slab per (tensor, which),
    cached on the tensor, so operators built from the same stage-2 tensors share packed channels."""

    def __init__(self, t, which):
        # the channel is cached on t: hold t only weakly (no reference cycle, so the stage-2 tensor and
        # its packed copies are freed as soon as the last operator using them goes)
        self._tref, self.which = weakref.ref(t), which
        self._base, self._st = t.strided_source()
        self.shape = tuple(int(x) for x in t.shape)
        if len(self.shape) != 6:
            raise ValueError("a stage-2 tensor has six legs, not {}".format(len(self.shape)))
        a0, a1 = (0, 1) if which == 0 else (1, 0)
        self.na0, self.na1 = self.shape[a0], self.shape[a1]
        self.n_alpha = self.na0 * self.na1
        self.P = self.shape[2] * self.shape[3]
        self.strided = self.shape[2] == self.shape[4] and self.shape[3] == self.shape[5]
        self._joined, self._packed, self.lowprec, self._packed_f32 = None, None, {}, {}

    @staticmethod
    def of(t, which):
        cache = t.__dict__.setdefault("_stage3_slabs", {})
        if which not in cache:
            cache[which] = _Slab(t, which)
        return cache[which]

    @property
    def t(self):
        t = self._tref()
        if t is None:
            raise RuntimeError("the stage-2 tensor of this slab channel no longer exists")
        return t

    def source(self):
        """(base tensor, (na0, na1, d0, d1), six strides) of the slab map."""
        st = self._st
        a0, a1 = (0, 1) if self.which == 0 else (1, 0)
        return self._base, (self.na0, self.na1, self.shape[4], self.shape[5]), (st[a0], st[a1], st[4], st[5], st[2], st[3])

    @property
    def joined(self):
        if self._joined is None:
            if self.strided:
                self._joined = HipData(join_slabs([self], [1.0]))
            else:
                t = self.t
                self._joined = t.join((0, 1), 4, 5, 2, 3) if self.which == 0 else t.join((1, 0), 4, 5, 2, 3)
        return self._joined

    @property
    def _t(self):
        return self.joined._t

    def packed(self):
        """The channel in the fused kernel's MFMA-operand order (cc_stage3_pack_strided_f64)."""
        if self._packed is None:
            buf = empty((_lib.query("cc_stage3_packed_size", self.n_alpha, self.P),))
            base, (na0, na1, d0, d1), st = self.source()
            _lib.call("cc_stage3_pack_strided_f64", stream(), na0, na1, d0, d1, _lib.i64_array(st), ptr(base), ptr(buf))
            self._packed = buf
        return self._packed


    def packed_f32(self, role):
        """The channel in the FP32 kernel's operand order (cc_stage3_pack_strided_f32): role 0 as an A
        channel, role 1 as a B channel."""
        if role not in self._packed_f32:
            buf = torch.empty(_lib.query("cc_stage3_packed_size_f32", self.n_alpha, self.P, role), dtype=torch.float32,
                              device=self._base.device)
            base, (na0, na1, d0, d1), st = self.source()
            _lib.call("cc_stage3_pack_strided_f32", stream(), role, na0, na1, d0, d1, _lib.i64_array(st), ptr(base),
                      ptr(buf))
            self._packed_f32[role] = buf
        return self._packed_f32[role]


class Stage3Operator:
    """terms: list of (stage2_0, stage2_1, site_operator or None) with HipData tensors."""

    def __init__(self, terms, physical_dimension=None):
        self.terms = list(terms)
        if not self.terms:
            raise ValueError("a stage-3 operator needs at least one term")
        s0, s1, o = self.terms[0]
        self.d = int(physical_dimension if physical_dimension is not None else
                     next((op.shape[0] for (_, _, op) in self.terms if op is not None), None))
        self.state_shape = torch.Size((s0.shape[2], s0.shape[3], s1.shape[2], s1.shape[3], self.d))
        self.n = int(np.prod(self.state_shape))
        self.P, self.Q = s0.shape[2] * s0.shape[3], s1.shape[2] * s1.shape[3]
        self.n_alpha = s0.shape[0] * s0.shape[1]
        self._A, self._B, self._O = [], [], []
        for (a, b, op) in self.terms:
            if a.shape[0] * a.shape[1] != self.n_alpha or b.shape[0] * b.shape[1] != self.n_alpha:
                raise ValueError("stage-2 tensors of one operator must share the environment bond")
            self._A.append(self._join(a, 0))
            self._B.append(self._join(b, 1))
            self._O.append(op)
        self.cost_of_multiply = sum(cost_of_term(self.n_alpha, a.shape[4] * a.shape[5], self.P, b.shape[4] * b.shape[5],
                                                 self.Q, self.d, op is not None)
                                    for a, b, op in zip(self._A, self._B, self._O))
        self.cost_of_formMatrix = sum(cost_of_matrix(a.shape, b.shape, self.d) for (a, b, _) in self.terms)
        self._work = None
        self._fused = None
        self._formed = None     # formed.FormedOperator of the last solver that formed this operator
        self._merge, self._joined, self._packs, self._refreshed = None, {}, {}, 0
        # the slab kernels read P = Q <= 36, d = 2; the solvers, plans and low-precision forms (use_fused) serve the
        # extents D * D of equal center bonds
        self._use_slabs = (self.P == self.Q and self.P <= 36 and self.d == 2 and self.n_alpha > 0 and
                           all(x.strided for x in self._A + self._B) and self._plan_fits())
        self.use_fused = self._use_slabs and bool(_lib.load().cc_stage3_fused_supported(self.P, self.d))

    def _plan_fits(self):
        na = len({id(a) for a in self._A})
        nb = len({id(b) for b in self._B})
        nops = len({id(o) for o in self._O if o is not None})
        return na <= 16 and nb <= 16 and len(self._A) <= 48 and nops <= 16

    def _channels(self):
        """Distinct A and B channels in first-use order, the distinct site operators (HipData), and the
        term table (A index, term, B index, operator index) sorted by A channel."""
        a_ids, b_ids, o_ids = {}, {}, {}
        a_list, b_list, ops = [], [], []
        rows = []
        for k, (A, B, O) in enumerate(zip(self._A, self._B, self._O)):
            if id(A) not in a_ids:
                a_ids[id(A)] = len(a_list)
                a_list.append(A)
            if id(B) not in b_ids:
                b_ids[id(B)] = len(b_list)
                b_list.append(B)
            o = -1
            if O is not None:
                if id(O) not in o_ids:
                    o_ids[id(O)] = len(ops)
                    ops.append(O)
                o = o_ids[id(O)]
            rows.append((a_ids[id(A)], k, b_ids[id(B)], o))
        rows.sort()
        return a_list, b_list, ops, rows

    def _merged(self):
        """The operator as products of summed channels: terms whose site operators are multiples of one another and
        that share a channel are one term, c_1 A_1 (x) B (x) O + c_2 A_2 (x) B (x) O = (c_1 A_1 + c_2 A_2) (x) B (x) O.
        The transverse-field Ising operator's seven terms become five (eight channels six), Heisenberg's fourteen
        eight.  Returns (channels, specs, ops, rows): the distinct channels per half as _channels lists them, per half
        the sums as tuples of (channel, coefficient), the distinct site operators, and the term table (A sum, B sum,
        operator or -1) sorted by A sum."""
        if self._merge is None:
            a_list, b_list, ops, rows = self._channels()
            legs = tuple(tuple(ch.source()[1:] for ch in chans) for chans in (a_list, b_list))
            values = tuple(tuple(float(x) for x in op.toArray().reshape(-1)) for op in ops)
            key = (self.d, tuple(rows), values, legs)
            merge = _MERGES.get(key)
            if merge is None:
                merge = merged_terms(*key)
                if len(_MERGES) < 256:
                    _MERGES[key] = merge
            specs, table = merge
            self._merge = (a_list, b_list), specs, ops, table
        return self._merge

    def joined(self, side, k, channels=None):
        """Sum k of half `side` as a contiguous (alpha, P, P) array, kept: it stays what it was when first asked for.
        channels: of another operator of this structure (the sum over them, not kept)."""
        t = self._joined.get((side, k)) if channels is None else None
        if t is None:
            own, specs, _, _ = self._merged()
            spec = specs[side][k]
            parts = [(own if channels is None else channels)[side][i] for i, _ in spec]
            t = parts[0]._t if len(spec) == 1 and spec[0][1] == 1.0 else join_slabs(parts, [c for _, c in spec])
            if channels is None:
                self._joined[(side, k)] = t
        return t

    def same_structure(self, other):
        """The channels of `other` (per half) if it has this operator's terms, channel sharing and shapes; else
        ValueError."""
        a_list, b_list, _, rows = self._channels()
        oa, ob, _, orows = other._channels()
        if ([(r[0], r[2], r[3]) for r in rows] != [(r[0], r[2], r[3]) for r in orows] or
                [(c.n_alpha, c.P) for c in a_list + b_list] != [(c.n_alpha, c.P) for c in oa + ob]):
            raise ValueError("refresh needs an operator of the same structure")
        return oa, ob

    def snapshot(self):
        """Takes every sum of channels now (joined and packed), so that later calls do not read the stage-2 tensors."""
        self._take(True)

    def _take(self, joined):
        """The sums of channels not taken yet, packed and with `joined` joined as well, one launch per half."""
        channels, specs, _, _ = self._merged()
        for side in (0, 1):
            jobs = []
            for k, spec in enumerate(specs[side]):
                # a channel by itself is kept with the channel, for every operator built from it
                one = channels[side][spec[0][0]] if len(spec) == 1 and spec[0][1] == 1.0 else None
                need_j = joined and (one._joined is None if one else (side, k) not in self._joined)
                # packed once: into _packs until _build_fused hands them to the plan, from then on never again
                need_p = self._fused is None and (side, k) not in self._packs and (one._packed is None if one else True)
                if need_p and not need_j and (side, k) in self._joined:
                    self._packs[(side, k)] = self._pack(side, k, channels[side])     # what was taken before
                elif need_j or need_p:
                    jobs.append((k, spec, one, need_j, need_p))
            while jobs:     # channels of one leg size at a time (all of them, as a rule)
                sizes = channels[side][jobs[0][1][0][0]].source()[1]
                alike = [job for job in jobs if channels[side][job[1][0][0]].source()[1] == sizes]
                jobs = [job for job in jobs if job not in alike]
                self._take_alike(side, channels[side], sizes, alike)
            for k, spec in enumerate(specs[side]):
                if self._fused is None and (side, k) not in self._packs:
                    self._packs[(side, k)] = channels[side][spec[0][0]]._packed
                if joined and (side, k) not in self._joined:
                    self._joined[(side, k)] = channels[side][spec[0][0]]._t

    def _take_alike(self, side, channels, sizes, jobs):
        n_packed = _packed_size(self.n_alpha, self.P)
        out, sources, coefs, strides = [], [], [], []
        for k, spec, one, need_j, need_p in jobs:
            j = empty((self.n_alpha, self.P, self.P)) if need_j else None
            p = empty((n_packed,)) if need_p else None
            out.append((j, p))
            sources += [channels[i].source()[0].data_ptr() for i, _ in spec]
            coefs += [c for _, c in spec]
            strides += channels[spec[0][0]].source()[2]
        _lib.call("cc_slab_take_f64", stream(), len(jobs), _lib.i32_array([len(spec) for _, spec, _, _, _ in jobs]),
                  _lib.ptr_array(sources), _lib.f64_array(coefs), *sizes, _lib.i64_array(strides),
                  _lib.ptr_array([j.data_ptr() if j is not None else 0 for j, _ in out]),
                  _lib.ptr_array([p.data_ptr() if p is not None else 0 for _, p in out]))
        for (k, _, one, need_j, need_p), (j, p) in zip(jobs, out):
            if need_j and one:
                one._joined = HipData(j)
            elif need_j:
                self._joined[(side, k)] = j
            if need_p and one:
                one._packed = p
            elif need_p:
                self._packs[(side, k)] = p

    def _pack(self, side, k, channels, out=None):
        """Sum k of half `side` in the fused kernel's MFMA-operand order: over `channels` into `out`, or as it was joined."""
        _, specs, _, _ = self._merged()
        spec = specs[side][k]
        parts, coefs = [channels[i] for i, _ in spec], [c for _, c in spec]
        kept = self._joined[(side, k)] if out is None else None if _alike(parts) else join_slabs(parts, coefs)
        if out is None:
            out = empty((_packed_size(self.n_alpha, self.P),))
        _, (na0, na1, d0, d1), st = parts[0].source()
        if kept is not None:
            P = self.P
            _lib.call("cc_stage3_pack_strided_f64", stream(), self.n_alpha, 1, d0, d1,
                      _lib.i64_array([P * P, 0, d1 * P, P, d1, 1]), ptr(kept), ptr(out))
        else:
            _lib.call("cc_stage3_pack_sum_f64", stream(), len(spec), _lib.ptr_array([p.source()[0].data_ptr() for p in parts]),
                      _lib.f64_array(coefs), na0, na1, d0, d1, _lib.i64_array(st), ptr(out))
        return out

    def refresh_fused_from(self, other):
        """Packs the channels of `other` -- an operator of the same structure (the same terms, channel
        sharing and shapes) built from new stage-2 tensors -- into this operator's packed buffers, so that
        its fused kernel and native plan apply `other` (kernels only; capturable in a HIP graph)."""
        self._ensure_fused()
        channels = self.same_structure(other)
        self._joined = {}       # of the environment before
        self._refreshed += 1
        _, specs, _, _ = self._merged()
        for side, bufs in ((0, self._fused["A"]), (1, self._fused["B"])):
            for k in range(len(specs[side])):
                self._pack(side, k, channels[side], bufs[k])

    def _build_fused(self):
        """Pack every sum of slab channels once and build the term table (sorted by A channel)."""
        channels, specs, ops, rows = self._merged()
        self._take(False)
        A, B = ([self._packs[(side, k)] for k in range(len(specs[side]))] for side in (0, 1))
        self._packs = {}
        self._fused = dict(
            A=A, B=B, A_ptrs=_lib.ptr_array([t.data_ptr() for t in A]), B_ptrs=_lib.ptr_array([t.data_ptr() for t in B]),
            ta=_lib.i32_array([r[0] for r in rows]), tb=_lib.i32_array([r[1] for r in rows]),
            to=_lib.i32_array([r[2] for r in rows]), n_terms=len(rows), n_a=len(A), n_b=len(B),
            n_ops=len(ops), ops=_lib.f64_array([x for o in ops for x in o.toArray().reshape(-1)]),
            work=empty((max(1, _lib.query("cc_stage3_fused_work_size", self.n_alpha, self.P, self.d)),)), plan=ctypes.c_void_p())
        f = self._fused
        _lib.call("cc_stage3_slab_plan_create", ctypes.byref(f["plan"]), f["n_a"], f["A_ptrs"], f["n_b"], f["B_ptrs"],
                  f["n_terms"], f["ta"], f["tb"], f["to"], f["n_ops"], f["ops"], self.n_alpha, self.P, self.d, ptr(f["work"]))

    def _join(self, t, which):
        return _Slab.of(t, which)

    def _ensure_fused(self):
        if self._fused is None:
            self._build_fused()

    def plan_handle(self, precision="f64"):
        """A native plan (cc_stage3_plan_create) for solvers that apply this operator many times; precision
        "f32" gives the FP32-operand plan (cc_stage3_plan_create_f32) of the same operator."""
        self._ensure_fused()
        f = self._fused
        if precision == "f32":
            if f.get("plan_f32") is None:
                a_list, b_list, _, rows = self._channels()
                pa = [ch.packed_f32(0) for ch in a_list]
                pb = [ch.packed_f32(1) for ch in b_list]
                f["f32_slabs"] = pa + pb
                h = ctypes.c_void_p()
                _lib.call("cc_stage3_plan_create_f32", ctypes.byref(h), len(pa), _lib.ptr_array([t.data_ptr() for t in pa]),
                          len(pb), _lib.ptr_array([t.data_ptr() for t in pb]), len(rows), _lib.i32_array([r[0] for r in rows]),
                          _lib.i32_array([r[2] for r in rows]), _lib.i32_array([r[3] for r in rows]), f["n_ops"], f["ops"],
                          self.n_alpha, self.P, self.d, ptr(f["work"]))
                f["plan_f32"] = h
            return f["plan_f32"]
        if precision != "f64":
            raise ValueError("precision must be 'f64' or 'f32', not {!r}".format(precision))
        if not self.use_fused:
            raise NotImplementedError("the operator has no instantiated fused shape")
        return f["plan"]

    def __del__(self):
        f = getattr(self, "_fused", None)
        for key in ("plan", "plan_f32"):
            if f and f.get(key) is not None:
                try:
                    _lib.load().cc_stage3_plan_destroy(f[key])
                except Exception:
                    pass

    def apply_flat(self, x, y):
        """y = H x for flat device tensors of length n (torch float64), through the slabs whatever solves came before."""
        # also for unequal center bonds (packing may read site operators back, so not first under capture)
        if self._fused is None and self._use_slabs and (self.use_fused or not torch.cuda.is_current_stream_capturing()):
            self._build_fused()
        if self._fused is not None:
            _lib.call("cc_stage3_plan_apply", stream(), self._fused["plan"], ptr(x), ptr(y))
            return
        self.apply_generic_flat(x, y)

    def apply_generic_flat(self, x, y):
        """The reference's contraction order through the generic GEMM path (any shape)."""
        if self._work is None:
            ws = _lib.i64_array([0])
            _lib.call("cc_stage3_matvec_generic_work_size", self.n_alpha, self.P, self.Q, self.d, ws)
            self._work = empty((max(1, ws[0]),))
        _lib.call("cc_stage3_matvec_generic_f64", stream(), len(self._A),
                  _lib.ptr_array([a._t.data_ptr() for a in self._A]),
                  _lib.ptr_array([b._t.data_ptr() for b in self._B]),
                  _lib.ptr_array([o._t.data_ptr() if o is not None else 0 for o in self._O]),
                  self.n_alpha, self.P, self.Q, self.d, ptr(x), ptr(y), ptr(self._work))

    def apply(self, v):
        if v.shape != self.state_shape and v.size() != self.n:
            raise ValueError("state shape {} does not match the operator's {}".format(v.shape, self.state_shape))
        out = empty(self.state_shape)
        self.apply_flat(v._t, out)
        return HipData._wrap(out)

    def form_matrix(self):
        """The dense matrix: the environment matrices of all terms in one contraction, their products with the site
        operators, added term by term, in another."""
        from .tensors._2d.dense import _form_matrix
        eye = HipData.newIdentity(self.d)
        ops = [op if op is not None else eye for (_, _, op) in self.terms]
        G = contract("xyabcd", "yxefgh", "cdghabef", [[(a, b)] for (a, b, _) in self.terms])
        m = G and contract("cdghabef", "st", "cdghsabeft", [[(HipData(g), op) for g, op in zip(G, ops)]])
        if m:
            return HipData(m[0].reshape(self.n, self.n))
        m = None
        for (a, b, _), op in zip(self.terms, ops):
            t = _form_matrix(a, b, op)
            m = t if m is None else m + t
        return m

    def multiplier(self):
        from .utils import Multiplier
        m = Multiplier((self.n, self.n), self.apply, self.cost_of_multiply, self.form_matrix, self.cost_of_formMatrix)
        m.operator = self
        return m
