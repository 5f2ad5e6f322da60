"""Lowering of operators/BCs to libdop plans and their application on device tensors.

Replaces the reference's evaluation entry points (derivative_operator_functions.jl:18-69,
150-163, 203-802; ghost_derivative_operator.jl:15-37; composite_operators.jl:64-84):
every call becomes one fused dop_apply on the current torch stream.  Tensors must be
contiguous device tensors (float64, float32 or bfloat16); there is no CPU path.
"""
from __future__ import annotations

import collections
import ctypes as C
import os
import threading

import torch

from . import _abi
from .bcs import (AffineBC, ComposedMultiDimBC, MultiDimDirectionalBC, PeriodicAtomicBC, _LineBCs,
                  all_periodic_lines)
from .composite import DiffEqOperatorCombination, GhostDerivativeOperator
from .operators import DerivativeOperator

_STORAGE = {torch.float64: _abi.F64, torch.float32: _abi.F32, torch.bfloat16: _abi.BF16}


def storage_of(t: torch.Tensor) -> int:
    try:
        return _STORAGE[t.dtype]
    except KeyError:
        raise TypeError(f"unsupported dtype {t.dtype}: use float64, float32 or bfloat16") from None


def _check_device_tensor(t, name):
    if not isinstance(t, torch.Tensor):
        raise TypeError(f"{name} must be a torch tensor on the GPU (no CPU path)")
    if t.device.type != "cuda":
        raise TypeError(f"{name} must live on the GPU (got {t.device}); this library has no CPU path")
    if not t.is_contiguous():
        raise ValueError(f"{name} must be contiguous")


def julia_size(t: torch.Tensor):
    """Column-major size of a tensor (Julia's size(u))."""
    return tuple(int(v) for v in reversed(t.shape))


class Plan:
    """An immutable libdop plan (dop_plan_create)."""

    def __init__(self, desc: _abi.DopDesc, keep, capturing=None):
        """capturing: the raw stream that is being captured, whose graph then holds the plan."""
        self._keep = keep
        h = C.c_void_p()
        if capturing is None:
            _abi.check(_abi.lib().dop_plan_create(C.byref(desc), C.byref(h)), "dop_plan_create")
        else:
            _abi.check(_abi.lib().dop_plan_create_capturing(C.byref(desc), C.c_void_p(capturing),
                                                            C.byref(h)), "dop_plan_create_capturing")
        self.handle = h
        self.storage = desc.storage
        self.device_bytes = _abi.lib().dop_plan_device_bytes(h)
        self.in_elems = _abi.lib().dop_plan_input_elems(h)
        self.out_elems = _abi.lib().dop_plan_output_elems(h)
        self.desc = desc

    def __del__(self):
        h = getattr(self, "handle", None)
        if h is not None and h.value:
            try:
                _abi.lib().dop_plan_destroy(h)
            except Exception:
                pass
            self.handle = None

    def check(self, du: torch.Tensor, u: torch.Tensor):
        if du.numel() != self.out_elems or u.numel() != self.in_elems:
            raise AssertionError("array sizes do not match the plan")
        if storage_of(du) != self.storage or storage_of(u) != self.storage:
            raise TypeError("tensor dtype does not match the plan's storage type")
        if du.data_ptr() == u.data_ptr():
            raise ValueError("du must not alias u")

    def apply(self, du: torch.Tensor, u: torch.Tensor, accumulate: bool = False, stream=None):
        self.check(du, u)
        if stream is None:
            stream = torch.cuda.current_stream(u.device).cuda_stream
        _abi.check(_abi.lib().dop_apply(self.handle, C.c_void_p(du.data_ptr()),
                                        C.c_void_p(u.data_ptr()), int(bool(accumulate)),
                                        C.c_void_p(stream)), "dop_apply")

    def update(self, desc: _abi.DopDesc, keep, stream=None):
        """New BC values / operator tables of the same structure, in place
        (dop_plan_update): the plan's device memory is reused.  Raises DopError (EINVAL) when
        the structure differs."""
        if stream is None:
            stream = torch.cuda.current_stream().cuda_stream
        _abi.check(_abi.lib().dop_plan_update(self.handle, C.byref(desc), C.c_void_p(stream)),
                   "dop_plan_update")
        self._keep = keep
        self.desc = desc

    @property
    def variant(self):
        """(candidate launched, tuned?) -- dop_plan_variant."""
        t = C.c_int()
        v = _abi.lib().dop_plan_variant(self.handle, C.byref(t))
        return v, bool(t.value)

    def autotune(self, stream=None):
        if stream is None:
            stream = torch.cuda.current_stream().cuda_stream
        choice = C.c_int()
        _abi.check(_abi.lib().dop_plan_autotune(self.handle, C.c_void_p(stream), C.byref(choice)),
                   "dop_plan_autotune")
        return choice.value


def apply_set(terms):
    """The applies (plan, du, u, accumulate) in order, as one launch where the plans allow it
    (dop_apply_set), on u's current stream."""
    n = len(terms)
    for plan, du, u, _ in terms:
        plan.check(du, u)
    vp = C.c_void_p * n
    stream = torch.cuda.current_stream(terms[0][2].device).cuda_stream
    _abi.check(_abi.lib().dop_apply_set(n, vp(*(t[0].handle.value for t in terms)),
                                        vp(*(t[1].data_ptr() for t in terms)),
                                        vp(*(t[2].data_ptr() for t in terms)),
                                        (C.c_int * n)(*(int(bool(t[3])) for t in terms)),
                                        C.c_void_p(stream)), "dop_apply_set")


def make_desc(terms, jsize, storage, *, input_kind, semantics, bcs=None, padded=(0, 0, 0),
              transverse_view=0, accum=_abi.ACC_AUTO):
    """terms: list of DerivativeOperator; bcs: {axis0: AffineBC}."""
    ndim = len(jsize)
    if ndim < 1 or ndim > 3:
        raise ValueError("arrays of 1 to 3 dimensions are supported")
    ops = (_abi.DopOperator * len(terms))()
    keep = [ops]
    for t, L in enumerate(terms):
        if not L.N <= ndim:
            raise AssertionError(f"operator axis {L.N} > ndims {ndim}")
        ops[t] = L.c_struct(L.N - 1)
        keep.append(L)
    d = _abi.DopDesc()
    d.ndim = ndim
    d.storage = storage
    d.accum = accum
    d.input = input_kind
    d.semantics = semantics
    d.n_ops = len(terms)
    for k in range(3):
        d.size[k] = jsize[k] if k < ndim else 1
        d.padded[k] = int(padded[k]) if k < ndim else 0
    d.transverse_view = int(transverse_view)
    d.ops = ops
    for ax, bc in (bcs or {}).items():
        q = d.bc[ax]
        if isinstance(bc, _PeriodicPad):
            q.present, q.kind, q.n_l, q.n_r = 1, bc.kind, 0, 0
            continue
        if isinstance(bc, _LineBCs):
            # one BC per line: the axis entry only marks the axis as padded
            q.present, q.kind, q.n_l, q.n_r = 1, _abi.BC_AFFINE, 0, 0
            flat = bc.flat()
            arr = (_abi.DopAffineBC * len(flat))()
            for i, b in enumerate(flat):
                if isinstance(b, PeriodicAtomicBC):
                    arr[i].present, arr[i].kind = 1, _abi.BC_PERIODIC
                    continue
                if len(b.a_l) > _abi.MAX_BC_TAPS or len(b.a_r) > _abi.MAX_BC_TAPS:
                    raise ValueError("boundary condition order too high")
                e = arr[i]
                e.present, e.kind, e.n_l, e.n_r = 1, _abi.BC_AFFINE, len(b.a_l), len(b.a_r)
                for k, v in enumerate(b.a_l):
                    e.a_l[k] = float(v)
                for k, v in enumerate(b.a_r):
                    e.a_r[k] = float(v)
                e.b_l, e.b_r = float(b.b_l), float(b.b_r)
            d.line_bc[ax] = C.cast(arr, C.POINTER(_abi.DopAffineBC))
            keep.append(arr)
            continue
        if len(bc.a_l) > _abi.MAX_BC_TAPS or len(bc.a_r) > _abi.MAX_BC_TAPS:
            raise ValueError("boundary condition order too high")
        q.present = 1
        q.n_l, q.n_r = len(bc.a_l), len(bc.a_r)
        for k, v in enumerate(bc.a_l):
            q.a_l[k] = float(v)
        for k, v in enumerate(bc.a_r):
            q.a_r[k] = float(v)
        q.b_l, q.b_r = bc.b_l, bc.b_r
    return d, keep


# ------------------------------------------------------------------------------------------
# Q*u: which BC pads which axis, and which reference kernels apply

class _PeriodicPad:
    """Periodic padding of one axis: kind BC_PERIODIC (line wrap, bc_operators.jl:192) or
    BC_PERIODIC_ND (first/last planes, multi_dim_bc_operators.jl:221-252)."""

    def __init__(self, kind):
        self.kind = kind

    def key(self):
        return ("periodic", self.kind)


def _bcs_of(Q, ndim, jsize):
    """{axis0: AffineBC | _PeriodicPad} of Q applied to an array of Julia size jsize, and the
    semantics."""
    if isinstance(Q, (AffineBC, PeriodicAtomicBC)):
        # 1-D: Q*u is a BoundaryPaddedVector (bc_operators.jl:188-192);
        # N-D: BC*u = MultiDimBC{1}(BC, size(u))*u pads axis 1 (multi_dim_bc_operators.jl:210),
        # which for PeriodicBC takes the N-D periodic method (:221-228)
        if isinstance(Q, PeriodicAtomicBC):
            Q = _PeriodicPad(_abi.BC_PERIODIC if ndim == 1 else _abi.BC_PERIODIC_ND)
        return {0: Q}, (_abi.SEM_BPV if ndim == 1 else _abi.SEM_LINES)
    if ndim == 1:
        raise AssertionError("multi-dimensional BCs need arrays of 2 or more dimensions")
    if isinstance(Q, MultiDimDirectionalBC):
        _check_dir_size(Q, jsize, "Size of the BCs array in the MultiDimBC is incorrect")
        if Q.lines is not None:
            if all_periodic_lines(Q.lines):
                return {Q.D - 1: _PeriodicPad(_abi.BC_PERIODIC_ND)}, _abi.SEM_LINES
            return {Q.D - 1: _LineBCs(Q.lines)}, _abi.SEM_LINES
        bc = Q.bc
        if isinstance(bc, PeriodicAtomicBC):
            bc = _PeriodicPad(_abi.BC_PERIODIC_ND)
        return {Q.D - 1: bc}, _abi.SEM_LINES
    if isinstance(Q, ComposedMultiDimBC):
        # all atoms periodic: the N-D periodic method (:244-252); otherwise every line is
        # padded by its own atom (slice_rmul), i.e. the line wrap for periodic atoms
        all_periodic = all(all_periodic_lines(b.lines) if b.lines is not None
                           else isinstance(b.bc, PeriodicAtomicBC) for b in Q.bcs)
        out = {}
        for b in Q.bcs:
            _check_dir_size(b, jsize, f"Size of the BCs array for dimension {b.D} is incorrect")
            if b.lines is not None and not all_periodic:
                out[b.D - 1] = _LineBCs(b.lines)
                continue
            bc = b.bc
            if isinstance(bc, PeriodicAtomicBC):
                bc = _PeriodicPad(_abi.BC_PERIODIC_ND if all_periodic else _abi.BC_PERIODIC)
            out[b.D - 1] = bc
        return out, _abi.SEM_LINES
    raise TypeError(f"not a boundary condition: {type(Q)}")


def _check_dir_size(Q, jsize, msg):
    """The BC array of a MultiDimDirectionalBC must match the array's other axes
    (multi_dim_bc_operators.jl:178-192 / perpindex)."""
    if Q.lines is not None:
        other = tuple(v for k, v in enumerate(jsize) if k != Q.D - 1)
        if len(jsize) != Q.lines.ndim + 1 or tuple(Q.lines.shape) != other:
            raise AssertionError(msg)
    elif tuple(Q.s) != tuple(jsize):
        raise AssertionError(msg)


def _ghost_groups(terms, ndim, jsize):
    """Split (L, Q) terms into groups whose per-axis BCs agree (one plan per group)."""
    groups = []   # [ops, bcs{axis: bc}, keys{axis: key}, sem]
    for L, Q in terms:
        bcs, sem = _bcs_of(Q, ndim, jsize)
        ax = L.N - 1
        if ax not in bcs:
            raise AssertionError("the operator's axis is not padded by its boundary condition")
        key = bcs[ax].key()
        for g in groups:
            if g[3] == sem and g[2].get(ax, key) == key:
                g[0].append(L)
                g[1][ax] = bcs[ax]
                g[2][ax] = key
                break
        else:
            groups.append([[L], {ax: bcs[ax]}, {ax: key}, sem])
    return groups


def _plan_cache(obj):
    c = getattr(obj, "_plans", None)
    if c is None:
        c = {}
        try:
            obj._plans = c
        except AttributeError:
            pass
    return c


def _op_structure(L):
    return (L.N, int(L.wind), L.derivative_order, L.approximation_order, L.len,
            L.stencil_length, L.boundary_stencil_length, L.boundary_point_count, L.offside,
            int(L.uniform_grid), L.coeff_kind)


def _bc_structure(bc):
    if isinstance(bc, _PeriodicPad):
        return bc.key()
    if isinstance(bc, _LineBCs):
        return ("lines", hash(tuple(("p",) if isinstance(b, PeriodicAtomicBC) else
                                    (len(b.a_l), len(b.a_r)) for b in bc.flat())))
    return ("affine", len(bc.a_l), len(bc.a_r))


# The implicit `A*u` / `mul_` paths keep a plan set per live owner (an L*Q object or a sum of
# them) and kind of array.  When an owner goes, its plans go to a pool, and an owner of the same
# structure (operators' kinds and sizes, BC kinds and tap counts) takes them over with one
# dop_plan_update: a method-of-lines RHS that builds a new BC at every call (heat_equation.jl:38-43,
# KdV.jl:26-30) keeps using one plan, and owners that live side by side never replace each
# other's values.  (One plan per structure, rebound to whichever owner was applied last, cost two
# operators of one structure used in turn a table rebuild and upload per call: 460 us on the
# 4096^2 FP64 Laplacian whose apply takes 50, 10 ms on a 1-D line of 2^18 points.)  The pool holds
# at most _POOL_MAX sets and, beside the newest, _POOL_BYTES of device memory (tables of long
# non-uniform lines take hundreds of MB a plan); the oldest are dropped first.  A lock guards it,
# and every step of a search leaves it whole: an owner may go, and leave its plans, in any of them.
# Plans that a captured graph reads keep their values: they are never handed on, and the graph
# holds them (dop_plan_hold), so a replay does not depend on the owner or on what was applied since.
_POOL = collections.deque()   # (structure, plans, the stream they were applied on, bytes), oldest first
_POOL_MAX = 64
_POOL_BYTES = 256 << 20
_POOL_LOCK = threading.RLock()
_pool_held = 0                # bytes of the sets in the pool


def _pool_put(skey, plans, stream):
    global _pool_held
    nbytes = sum(p.device_bytes for p in plans)
    with _POOL_LOCK:
        _POOL.append((skey, plans, stream, nbytes))
        _pool_held += nbytes
        _pool_trim()


def _pool_trim():
    global _pool_held
    while len(_POOL) > 1 and (len(_POOL) > _POOL_MAX or _pool_held > _POOL_BYTES):
        old = _POOL.popleft()
        _pool_held -= old[3]


def _pool_take(skey, stream):
    """The newest set of the structure that was applied on the stream, or None."""
    global _pool_held
    newer, found = 0, None        # sets moved to the old end, newest first
    for _ in range(len(_POOL)):
        e = _POOL.pop()
        if e[0] == skey and e[2] == stream:
            _pool_held -= e[3]
            found = e[1]
            break
        _POOL.appendleft(e)
        newer += 1
    _POOL.rotate(-newer)
    _pool_trim()
    return found


class _Bound:
    """The plans of one owner for one kind of array, the descriptors of its values, and the
    streams that they have been applied on.  updated: the stream that set the values of plans from
    the pool, which others wait for before their first apply (None: plans made for the owner,
    complete from the start).  graph: the plans that graphs read (the same ones, or others made in
    a capture)."""

    __slots__ = ("skey", "descs", "plans", "streams", "updated", "graph", "__weakref__")

    def __init__(self, skey, descs):
        self.skey, self.descs, self.plans, self.streams = skey, descs, None, set()
        self.updated, self.graph = None, None

    def __del__(self):
        # plans applied on several streams are not reused: an update on one of them would not
        # wait for applies still queued on another
        try:
            if self.plans is not None and self.plans is not self.graph and len(self.streams) == 1:
                _pool_put(self.skey, self.plans, *self.streams)
        except Exception:   # interpreter shutdown
            pass


def ghost_plans(owner, terms, u: torch.Tensor, accum=_abi.ACC_AUTO):
    """Plans evaluating sum_t L_t*Q_t*u, cached on owner: the owner's own plans, for callers who
    keep them (in a batch, a server, an integrator)."""
    jsize = julia_size(u)
    storage = storage_of(u)
    key = ("own", jsize, storage, accum, u.device.index)
    cache = _plan_cache(owner)
    own = cache.get(key)
    if own is None:
        with torch.cuda.device(u.device):
            own = [Plan(d, keep) for d, keep, _ in _ghost_descs(terms, u, accum)]
        cache[key] = own
    return own


def _ghost_descs(terms, u, accum):
    """(descriptor, what it points to, structure) per plan of sum_t L_t*Q_t*u."""
    jsize = julia_size(u)
    storage = storage_of(u)
    out = []
    for ops, bcs, _, sem in _ghost_groups(terms, len(jsize), jsize):
        d, keep = make_desc(ops, jsize, storage, input_kind=_abi.INPUT_GHOST, semantics=sem,
                            bcs=bcs, accum=accum)
        out.append((d, keep + [bcs], (sem, tuple(_op_structure(L) for L in ops),
                                      tuple(sorted((ax, _bc_structure(bc)) for ax, bc in bcs.items())))))
    return out


def _wait_for(stream):
    """The current stream waits for what is queued on the raw `stream`; False where it cannot (a
    stream that is being captured now, or is gone).  Only an owner's first apply on a second stream
    comes here: an event at every update cost a temporary owner's apply 7 us of 48."""
    if _abi.lib().dop_capturing(stream):
        return False
    try:
        event = torch.cuda.Event()
        event.record(torch.cuda.ExternalStream(stream))
        torch.cuda.current_stream().wait_event(event)
    except RuntimeError:
        return False
    return True


def _bound_of(owner, key, u, accum):
    """The owner's _Bound for arrays like u (under the lock)."""
    bound = _plan_cache(owner).get(key)
    if bound is None:
        descs = _ghost_descs(_ghost_terms(owner), u, accum)
        # plans are created with the kernel selection the environment asks for
        skey = (julia_size(u), u.dtype, accum, u.device.index,
                os.environ.get("DOP_FORCE_GENERIC"), os.environ.get("DOP_TILE_VARIANT"),
                tuple(d[2] for d in descs))
        bound = _plan_cache(owner)[key] = _Bound(skey, descs)
    return bound


def _bind(owner, key, u, accum, stream):
    """The owner's _Bound for arrays like u, with plans holding its values on `stream`, u's
    current one."""
    with _POOL_LOCK, torch.cuda.device(u.device):
        bound = _bound_of(owner, key, u, accum)
        if bound.plans is None:
            plans = bound.graph
            if plans is None:
                plans = _pool_take(bound.skey, stream)
                if plans is None:
                    plans = [Plan(d, keep) for d, keep, _ in bound.descs]
                else:
                    for i, (d, keep, _) in enumerate(bound.descs):
                        try:
                            plans[i].update(d, keep, stream)
                        except _abi.DopError:
                            # same kinds and sizes but a different row structure (e.g. coefficients
                            # that are no longer uniform): a plan of its own
                            plans[i] = Plan(d, keep)
                    bound.updated = stream
            bound.plans = plans
        elif bound.updated is not None and stream not in bound.streams and not _wait_for(bound.updated):
            bound.plans = [Plan(d, keep) for d, keep, _ in bound.descs]
            bound.updated = None
        bound.streams.add(stream)
    return bound


def _graph_plans(owner, key, u, accum, stream):
    """The owner's plans for the graph that is being captured on `stream`, which holds them: its
    plans if their values have been there since they were made, else plans made now."""
    with _POOL_LOCK, torch.cuda.device(u.device):
        bound = _bound_of(owner, key, u, accum)
        if bound.graph is None:
            if bound.plans is not None and bound.updated is None:
                bound.graph = bound.plans
            else:
                bound.graph = [Plan(d, keep, stream) for d, keep, _ in bound.descs]
        for p in bound.graph:
            _abi.check(_abi.lib().dop_plan_hold(p.handle, C.c_void_p(stream)), "dop_plan_hold")
        return bound.graph


_raw_stream = torch._C._cuda_getCurrentRawStream if hasattr(
    torch._C, "_cuda_getCurrentRawStream") else lambda i: torch.cuda.current_stream(i).cuda_stream


def _apply_bound(owner, du, u, accum=_abi.ACC_AUTO, accumulate=False):
    """du (+)= owner * u; du and u are contiguous device tensors of one shape."""
    if du.dtype is not u.dtype:
        raise TypeError("tensor dtype does not match the plan's storage type")
    dp, up = du.data_ptr(), u.data_ptr()
    if dp == up:
        raise ValueError("du must not alias u")
    dev = u.device
    stream = _raw_stream(dev.index)
    key = (u.shape, u.dtype, dev, accum)
    lib = _abi.lib()
    if stream and lib.dop_capturing(stream):   # (the default stream cannot be captured)
        plans = _graph_plans(owner, key, u, accum, stream)
    else:
        bound = owner._plans.get(key)
        if bound is None or stream not in bound.streams:
            bound = _bind(owner, key, u, accum, stream)
        plans = bound.plans
    apply = lib.dop_apply
    for p in plans:
        rc = apply(p.handle, dp, up, 1 if accumulate else 0, stream)
        if rc:
            _abi.check(rc, "dop_apply")
        accumulate = True


def _ghost_terms(A):
    if isinstance(A, GhostDerivativeOperator):
        return [(A.L, A.Q)]
    if isinstance(A, DiffEqOperatorCombination) and all(
            isinstance(op, GhostDerivativeOperator) for op in A.ops):
        return [(op.L, op.Q) for op in A.ops]
    return None


def ghost_times(G, u):
    _check_device_tensor(u, "u")
    out = torch.empty_like(u)
    _apply_bound(G, out, u)
    return out


# ------------------------------------------------------------------------------------------
# operators on padded arrays

def _padded_plan(owner, ops, du, M, transverse_view=0, accum=_abi.ACC_AUTO):
    osz, msz = julia_size(du), julia_size(M)
    if len(osz) != len(msz):
        raise AssertionError("du and M must have the same number of dimensions")
    padded = []
    for k in range(len(osz)):
        if msz[k] == osz[k]:
            padded.append(0)
        elif msz[k] == osz[k] + 2:
            padded.append(1)
        else:
            raise AssertionError("M must equal du in size or be padded by 2 along each axis")
    for L in ops:
        if not L.N <= len(osz) or not padded[L.N - 1]:
            raise AssertionError("differentiated dimension must be padded")
    storage = storage_of(M)
    key = ("padded", tuple(id(L) for L in ops), osz, msz, storage, transverse_view, accum)
    cache = _plan_cache(owner)
    if key not in cache:
        with torch.cuda.device(M.device):
            d, keep = make_desc(list(ops), osz, storage, input_kind=_abi.INPUT_PADDED,
                                semantics=_abi.SEM_LINES, padded=padded + [0] * (3 - len(padded)),
                                transverse_view=transverse_view, accum=accum)
            cache[key] = Plan(d, keep)
    return cache[key]


def derivative_times_array(L: DerivativeOperator, M):
    """L * M (derivative_operator_functions.jl:150-163): M is padded along L's axis."""
    _check_device_tensor(M, "M")
    shape = list(M.shape)
    shape[len(shape) - L.N] -= 2
    out = torch.empty(shape, dtype=M.dtype, device=M.device)
    _padded_plan(L, [L], out, M).apply(out, M)
    return out


def combination_times(A: DiffEqOperatorCombination, x):
    """(L1 + L2 + ...) * x = sum(op * x) (composite_operators.jl:64-65)."""
    _check_device_tensor(x, "x")
    terms = _ghost_terms(A)
    if terms is not None:
        out = torch.empty_like(x)
        _apply_bound(A, out, x)
        return out
    if all(isinstance(op, DerivativeOperator) for op in A.ops):
        shapes = set()
        for L in A.ops:
            s = list(x.shape)
            s[len(s) - L.N] -= 2
            shapes.add(tuple(s))
        if len(shapes) != 1:
            raise ValueError("DimensionMismatch: the operators' results have different sizes")
        out = torch.empty(shapes.pop(), dtype=x.dtype, device=x.device)
        _padded_plan(A, A.ops, out, x).apply(out, x)
        return out
    parts = [op * x for op in A.ops]
    out = parts[0]
    for p in parts[1:]:
        out = out + p
    return out


def mul_(du, A, u, overwrite=True, accum=_abi.ACC_AUTO):
    """mul!(du, A, u): writes A*u into du (adds into du when overwrite=False)."""
    from .bcs import BoundaryPadded
    if isinstance(u, BoundaryPadded):
        # mul!(du, L, Q*u) = mul!(du, L*Q, u)
        return mul_(du, A * u.Q, u.u, overwrite=overwrite, accum=accum)
    _check_device_tensor(du, "du")
    _check_device_tensor(u, "u")
    accumulate = not overwrite
    terms = _ghost_terms(A)
    if terms is not None:
        if tuple(du.shape) != tuple(u.shape):
            raise AssertionError("du must have the unpadded size of u")
        _apply_bound(A, du, u, accum, accumulate)
        return du
    if isinstance(A, DerivativeOperator):
        # derivative_operator_functions.jl:18-69
        _padded_plan(A, [A], du, u, accum=accum).apply(du, u, accumulate=accumulate)
        return du
    if isinstance(A, DiffEqOperatorCombination) and all(
            isinstance(op, DerivativeOperator) for op in A.ops):
        nd = du.dim()
        if nd == 1:
            tv = 0   # composite_operators.jl:76-84: plain per-op mul! and sum
        elif nd == 2:
            axes = {op.N for op in A.ops}
            tv = 1 if len(axes) > 1 else 0   # derivative_operator_functions.jl:414-461
        else:
            tv = 1                           # derivative_operator_functions.jl:768-801
        _padded_plan(A, A.ops, du, u, transverse_view=tv, accum=accum).apply(
            du, u, accumulate=accumulate)
        return du
    raise TypeError(f"mul_ does not support {type(A)}")


def plans_for(A, u, accum=_abi.ACC_AUTO):
    """The libdop plans that `A * u` runs (for benchmarking and batching)."""
    terms = _ghost_terms(A)
    if terms is None:
        raise TypeError("plans_for needs L*Q or a sum of L*Q")
    return ghost_plans(A, terms, u, accum)


def plan_for_shape(A, shape, dtype=torch.float32, device="cuda", accum=_abi.ACC_AUTO):
    """The single fused plan of L*Q (or a sum of them) for an array of the given tensor
    shape and dtype, without needing the array itself."""
    u = torch.empty(1, dtype=dtype, device=device).as_strided(tuple(shape), (0,) * len(shape))
    terms = _ghost_terms(A)
    if terms is None:
        raise TypeError("plan_for_shape needs L*Q or a sum of L*Q")
    plans = ghost_plans(A, terms, u, accum)
    if len(plans) != 1:
        raise ValueError("the operator needs one BC per axis to fuse into one plan")
    return plans[0]
