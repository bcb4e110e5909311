"""Recognition of columns of standard elements in a traced model.

The traced instructions of a model made of drifts, lenses, deflectors,
rotators, scanner / descanner offsets and biprisms are matched, in order and
without remainder, against the instruction sequences those elements emit.  The
result is a list of steps that ``tg_ray_column_run`` applies with the state in
named registers: the same operations with the same immediates, so the same
bits.  Anything else (other elements, per-ray parameters, mixed dtypes,
broadcast shapes, tangents) does not match and stays a register program.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from . import _lib

FIELDS = ("x", "y", "dx", "dy", "pathlength")


class _NoMatch(Exception):
    pass


class _Cursor:
    """Walks a trace's instructions."""

    def __init__(self, instrs):
        self.instrs, self.i = instrs, 0

    def peek(self, k: int = 0):
        return self.instrs[self.i + k] if self.i + k < len(self.instrs) else None

    def take(self, op: str, a: int, b: int | None = None, imm=None):
        """The next instruction, which has to be `op` on values a (and b), with
        the immediate `imm` if one is given: (its value, its immediate)."""
        ins = self.peek()
        if ins is None or ins.op != op or ins.a != a or ins.b != (a if b is None else b) or (
                imm is not None and not _same(ins.imm, imm)):
            raise _NoMatch
        self.i += 1
        return ins.dst, ins.imm


def _same(a, b) -> bool:
    return float(a) == float(b) and np.signbit(a) == np.signbit(b)


class _State:
    """The values holding the ray; `path` is None while the pathlength is uniform."""

    __slots__ = ("x", "y", "dx", "dy", "path", "path0")


def _add_path(c: _Cursor, s: _State, v: int):
    """path + v: an addition, or (uniform pathlength) an immediate one."""
    if s.path is not None:
        return c.take("add", s.path, v)[0]
    out, s.path0 = c.take("addi", v)
    return out


def _lens(c: _Cursor, s: _State):
    nx, _ = c.take("neg", s.x)
    qx, f = c.take("divi", nx)
    dx, _ = c.take("add", qx, s.dx)
    ny, _ = c.take("neg", s.y)
    qy, _ = c.take("divi", ny, imm=f)
    dy, _ = c.take("add", qy, s.dy)
    xx, _ = c.take("mul", s.x, s.x)
    yy, _ = c.take("mul", s.y, s.y)
    r2, _ = c.take("add", xx, yy)
    q, f2 = c.take("divi", r2)
    if s.path is not None:
        s.path, _ = c.take("sub", s.path, q)
    else:
        s.path, s.path0 = c.take("rsubi", q)
    s.dx, s.dy = dx, dy
    return _lib.STEP_LENS, (f, f2)


def _slope_path(c: _Cursor, s: _State):
    """path + dx x + dy y with the incoming slopes."""
    px, _ = c.take("mul", s.dx, s.x)
    s.path = _add_path(c, s, px)
    py, _ = c.take("mul", s.dy, s.y)
    s.path, _ = c.take("add", s.path, py)


def _deflector(c: _Cursor, s: _State):
    dx, ax = c.take("addi", s.dx)
    dy, ay = c.take("addi", s.dy)
    _slope_path(c, s)
    s.dx, s.dy = dx, dy
    return _lib.STEP_DEFLECT, (ax, ay)


def _shift(c: _Cursor, s: _State):
    s.x, px = c.take("addi", s.x)
    s.y, py = c.take("addi", s.y)
    s.dx, tx = c.take("addi", s.dx)
    s.dy, ty = c.take("addi", s.dy)
    return _lib.STEP_SHIFT, (px, py, tx, ty)


def _rotated(c: _Cursor, u: int, v: int, cs=None, sn=None):
    a, cs = c.take("muli", u, imm=cs)
    b, sn = c.take("muli", v, imm=sn)
    new_u, _ = c.take("sub", a, b)
    a, _ = c.take("muli", u, imm=sn)
    b, _ = c.take("muli", v, imm=cs)
    new_v, _ = c.take("add", a, b)
    return new_u, new_v, cs, sn


def _rotator(c: _Cursor, s: _State):
    x, y, cs, sn = _rotated(c, s.x, s.y)
    dx, dy, _, _ = _rotated(c, s.dx, s.dy, cs, sn)
    s.x, s.y, s.dx, s.dy = x, y, dx, dy
    return _lib.STEP_ROTATE, (cs, sn)


def _biprism(c: _Cursor, s: _State):
    sg, _ = c.take("sign", s.x)
    t, amount = c.take("muli", sg)
    dx, _ = c.take("add", s.dx, t)
    _slope_path(c, s)
    s.dx = dx
    return _lib.STEP_BIPRISM, (amount,)


def _drift(c: _Cursor, s: _State):
    tx, d = c.take("muli", s.dx)
    s.x, _ = c.take("add", s.x, tx)
    ty, _ = c.take("muli", s.dy, imm=d)
    s.y, _ = c.take("add", s.y, ty)
    flags = _lib.STEP_DRIFT
    if s.path is not None:
        s.path, _ = c.take("addi", s.path, imm=d)
        flags |= _lib.STEP_DRIFT_PATH
    return flags, d


def _element(c: _Cursor, s: _State):
    """The element at the cursor, told by its first instruction; None: a drift."""
    ins = c.peek()
    if ins.op == "neg":
        return _lens(c, s)
    if ins.op == "sign":
        return _biprism(c, s)
    if ins.op == "addi" and ins.a == s.x:
        return _shift(c, s)
    if ins.op == "addi" and ins.a == s.dx:
        return _deflector(c, s)
    if ins.op == "muli" and ins.a == s.x:
        return _rotator(c, s)
    return None


def match_steps(trace, start: dict):
    """([(kind, flags, d, params)], final state, uniform start pathlength) of a
    trace whose ray starts as the value ids `start` (pathlength None: uniform),
    or None where it is not a column of standard elements."""
    c, s = _Cursor(trace.instrs), _State()
    s.x, s.y, s.dx, s.dy, s.path, s.path0 = (*(start[k] for k in FIELDS), 0.0)
    steps = []
    try:
        while c.peek() is not None:
            flags, d = 0, 0.0
            element = _element(c, s)
            if element is None:
                flags, d = _drift(c, s)
                element = (_element(c, s) if c.peek() is not None else None) or (_lib.STEP_NONE, ())
            steps.append((element[0], flags, d, element[1]))
    except _NoMatch:
        return None
    return steps, s, s.path0


class ColumnMatch:
    """A matched model: its steps, the input slot of each field (None: uniform
    pathlength) and the value id each output field is stored from (None: not
    stored)."""

    def __init__(self, shape, dtype, steps, slots, out_vids, path0):
        self.shape, self.dtype = shape, dtype
        self.slots, self.out_vids = slots, out_vids
        self.n_out = sum(v is not None for v in out_vids)
        col = _lib.Column()
        f32 = dtype == torch.float32
        col.dtype = _lib.TG_F32 if f32 else _lib.TG_F64
        col.n = math.prod(shape)
        # a cached call's outputs share one allocation, each on a 16-byte boundary
        size = 4 if f32 else 8
        self.row = -(-col.n // (16 // size)) * (16 // size)
        # immediates rounded once to the ray dtype, as in register programs
        num = (lambda v: float(np.float32(v))) if f32 else float
        col.pathlength = num(path0)
        col.n_step = len(steps)
        for st, (kind, flags, d, params) in zip(col.step, steps):
            st.kind, st.flags, st.d = kind, flags, num(d)
            for k, v in enumerate(params):
                st.p[k] = num(v)
        self.struct = col


def match(trace, sym_in, sym_out, bin_request=None) -> ColumnMatch | None:
    """The column a traced model is, or None.  sym_in and sym_out are the
    symbolic rays before and after; every array has to be contiguous, of one
    shape and one dtype."""
    from ._program import Sym

    start = {}
    for k in FIELDS:
        v = getattr(sym_in, k, None)
        if isinstance(v, Sym):
            start[k] = v.vid
        elif k == "pathlength":
            start[k] = None
        else:
            return None
    slots = [None if start[k] is None else trace.value_slot.get(start[k]) for k in FIELDS]
    used = [trace.slot_tensors[s] for s in slots if s is not None]
    if len(used) != len([k for k in FIELDS if start[k] is not None]):
        return None
    shape, dtype = tuple(used[0].shape), used[0].dtype
    if any(tuple(t.shape) != shape or t.dtype != dtype or not t.is_contiguous() for t in used):
        return None
    got = match_steps(trace, start)
    if got is None or not got[0] or len(got[0]) > _lib.TG_MAX_STEP:
        return None
    steps, s, path0 = got
    end = dict(x=s.x, y=s.y, dx=s.dx, dy=s.dy, pathlength=s.path)
    out_vids = []
    for k in FIELDS:
        v = getattr(sym_out, k)
        if isinstance(v, Sym):
            if v.vid != end[k]:
                return None
            out_vids.append(None if v.vid in trace.value_slot else v.vid)
        elif end[k] is not None:
            return None
        else:
            out_vids.append(None)
    # the remaining fields are uniform or unchanged inputs
    for k in ("z", "_one"):
        v = getattr(sym_out, k)
        if isinstance(v, Sym) and v.vid not in trace.value_slot:
            return None
    if bin_request is not None:
        _, bx, by = bin_request
        if not (isinstance(bx, Sym) and isinstance(by, Sym) and bx.vid == s.x and by.vid == s.y):
            return None
    if bin_request is None and not any(v is not None for v in out_vids):
        return None
    return ColumnMatch(shape, dtype, steps, slots, out_vids, path0)
