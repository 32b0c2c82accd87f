"""Device-side vector expressions over packed complex vectors (vector_arithm.hpp:450-1130).

Mirrors the reference's expression operators: vector (+ - * /) vector for any two pack sizes,
vector (+ - * /) scalar and scalar (+ - * /) vector for a real (float) or complex scalar, and
conj().  An expression is lazy; `store(expr, dst)` (the reference's pcxo::store,
vector_arithm.hpp:405-447) flattens it into a program for pcx_vexpr_eval, which evaluates the
whole tree in one fused kernel on the GPU.

Register allocation: Sethi-Ullman numbering.  A node needs max(need(l), need(r)) registers when
the two differ and need + 1 when they are equal; the operand that needs more is evaluated first.
The machine has four registers, so any expression whose tree needs at most four evaluates.
"""
from __future__ import annotations

import numbers
import struct

from . import _lib
from ._lib import PcxError, check, lib, stream_ptr

_BIN = {"+": "ADD", "-": "SUB", "*": "MUL", "/": "DIV"}
# scalar ops: (op with scalar on the right, op with scalar on the left); real and complex forms
_SCA = {"+": ("ADD", "ADD"), "-": ("SUB", "RSUB"), "*": ("MUL", "MUL"), "/": ("DIV", "RDIV")}


class Expr:
    """A lazy element-wise expression over packed device vectors."""

    __slots__ = ()

    def __add__(self, o):
        return _combine("+", self, o)

    def __radd__(self, o):
        return _combine("+", o, self)

    def __sub__(self, o):
        return _combine("-", self, o)

    def __rsub__(self, o):
        return _combine("-", o, self)

    def __mul__(self, o):
        return _combine("*", self, o)

    def __rmul__(self, o):
        return _combine("*", o, self)

    def __truediv__(self, o):
        return _combine("/", self, o)

    def __rtruediv__(self, o):
        return _combine("/", o, self)

    # n: elements; regs: registers its evaluation needs (set when a node is built)
    def size(self) -> int:
        return self.n

    def need(self) -> int:
        return self.regs


class Leaf(Expr):
    __slots__ = ("vec", "n", "regs")

    def __init__(self, vec):
        self.vec = vec
        self.n, self.regs = vec.size(), 1


class Bin(Expr):
    __slots__ = ("op", "lhs", "rhs", "n", "regs")

    def __init__(self, op, lhs, rhs):
        if lhs.n != rhs.n:
            raise PcxError(_lib.ERR_SIZE_MISMATCH, f"vector sizes {lhs.n} and {rhs.n} differ")
        self.op, self.lhs, self.rhs = op, lhs, rhs
        self.n = lhs.n
        self.regs = max(lhs.regs, rhs.regs) if lhs.regs != rhs.regs else lhs.regs + 1


class Scalar(Expr):
    __slots__ = ("op", "expr", "scalar", "left", "n", "regs")

    def __init__(self, op, expr, scalar, scalar_left):
        self.op, self.expr, self.scalar, self.left = op, expr, scalar, scalar_left
        self.n, self.regs = expr.n, expr.regs


class Conj(Expr):
    __slots__ = ("expr", "n", "regs")

    def __init__(self, expr):
        self.expr = expr
        self.n, self.regs = expr.n, expr.regs


def as_expr(x) -> Expr:
    if isinstance(x, Expr):
        return x
    if hasattr(x, "pack") and hasattr(x, "data_ptr"):
        return Leaf(x)
    raise TypeError(f"not a vector expression: {type(x).__name__}")


def _is_number(x):
    return type(x) in (float, complex, int) or (not isinstance(x, Expr) and isinstance(x, numbers.Number))


def _combine(op, a, b):
    a_s, b_s = _is_number(a), _is_number(b)
    if a_s and b_s:
        raise TypeError("an expression needs at least one vector")
    if b_s:
        return Scalar(op, as_expr(a), b, False)
    if a_s:
        return Scalar(op, as_expr(b), a, True)
    return Bin(op, as_expr(a), as_expr(b))


def conj(x):
    """vector_arithm.hpp:495 conj(expression); the conjugate of a scalar is the scalar's."""
    if _is_number(x):
        return complex(x).conjugate() if isinstance(x, complex) else x
    return Conj(as_expr(x))


_LOAD, _CONJ = _lib.VOP["LOAD"], _lib.VOP["CONJ"]
_BIN_OP = {op: _lib.VOP[name] for op, name in _BIN.items()}
# (operation, scalar on the left, real scalar) -> op
_SCA_OP = {(op, left, real): _lib.VOP[names[left] + ("R" if real else "S")]
           for op, names in _SCA.items() for left in (False, True) for real in (False, True)}


def compile_expr(expr: Expr):
    """Program (list of VInstr fields) and source list for pcx_vexpr_eval."""
    expr = as_expr(expr)
    if expr.regs > _lib.VEXPR_REGS:
        raise PcxError(_lib.ERR_UNSUPPORTED, f"expression needs {expr.regs} registers (at most 4)")
    srcs, index, prog = [], {}, []

    def gen(e, r):
        kind = type(e)
        if kind is Leaf:
            vec = e.vec
            key = (vec.data_ptr(), vec.pack)
            at = index.get(key)
            if at is None:
                at = index[key] = len(srcs)
                srcs.append(vec)
            prog.append((_LOAD, r, at, 0, 0.0, 0.0))
        elif kind is Conj:
            gen(e.expr, r)
            prog.append((_CONJ, r, r, 0, 0.0, 0.0))
        elif kind is Scalar:
            gen(e.expr, r)
            s = e.scalar
            real = type(s) in (float, int) or isinstance(s, numbers.Real)
            z = complex(s)
            prog.append((_SCA_OP[e.op, e.left, real], r, r, 0, z.real, z.imag))
        elif e.lhs.regs >= e.rhs.regs:
            gen(e.lhs, r)
            gen(e.rhs, r + 1)
            prog.append((_BIN_OP[e.op], r, r, r + 1, 0.0, 0.0))
        else:
            gen(e.rhs, r)
            gen(e.lhs, r + 1)
            prog.append((_BIN_OP[e.op], r, r + 1, r, 0.0, 0.0))

    gen(expr, 0)
    if len(prog) > _lib.VEXPR_MAX_PROG or len(srcs) > _lib.VEXPR_MAX_SRC:
        raise PcxError(_lib.ERR_UNSUPPORTED, "expression exceeds 64 instructions or 16 sources")
    return prog, srcs


# the C structs, packed straight into bytes (VSource / VSource64, VInstr, VInstr64; native mode: a
# scalar beyond FLT_MAX becomes infinite, as in ctypes)
_PACK_SRC, _PACK_F32, _PACK_F64 = struct.Struct("@Pq").pack, struct.Struct("@iiiiff").pack, struct.Struct("@iiiidd").pack


def _common_dtype(*vs) -> str:
    """The element type shared by every vector of an evaluation (float32 or float64)."""
    kinds = {getattr(v, "dtype", "float32") for v in vs}
    if len(kinds) != 1:
        raise PcxError(_lib.ERR_INVALID_ARGUMENT, "an expression mixes float and double vectors")
    return kinds.pop()


def store(expr, dst, stream=None) -> None:
    """pcxo::store(expr, dst) (vector_arithm.hpp:405-447): evaluate into dst in its pack size."""
    expr = as_expr(expr)
    if expr.n != dst.size():
        raise PcxError(_lib.ERR_SIZE_MISMATCH,
                       f"expression size (which is {expr.n}) differs from destination size (which is {dst.size()})")
    prog, srcs = compile_expr(expr)
    f64 = _common_dtype(dst, *srcs) == "float64"
    pack = _PACK_F64 if f64 else _PACK_F32
    S = b"".join([_PACK_SRC(v.data_ptr(), v.pack) for v in srcs])
    P = b"".join([pack(*i) for i in prog])
    ev = lib().pcx_vexpr_eval_f64 if f64 else lib().pcx_vexpr_eval
    check(ev(S, len(srcs), P, len(prog), dst.data_ptr(), dst.pack, dst.size(), stream_ptr(stream)))


def repack(dst, src, stream=None) -> None:
    """Pack conversion dst <- src (same size, any two pack sizes)."""
    if src.size() != dst.size():
        raise PcxError(_lib.ERR_SIZE_MISMATCH, "repack needs equal sizes")
    rp = lib().pcx_repack_f64 if _common_dtype(dst, src) == "float64" else lib().pcx_repack
    check(rp(dst.data_ptr(), dst.pack, src.data_ptr(), src.pack, dst.size(), stream_ptr(stream)))
