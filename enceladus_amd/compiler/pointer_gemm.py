"""Matmul loops written with pointer tiles and masks, rewritten to tensor descriptors.

The usual way to write a product is

    for k in range(0, K, BK):
        a = tl.load(a_ptrs, mask=(rm[:, None] < M) & (rk[None, :] + k < K), other=0.0)
        b = tl.load(b_ptrs, mask=(rk[:, None] + k < K) & (rn[None, :] < N), other=0.0)
        acc = tl.dot(a, b, acc)
        a_ptrs += BK * stride_ak
        b_ptrs += BK * stride_bk

(or with a trip-count loop, `for k in range(0, cdiv(K, BK))` and masks `rk < K - k * BK`).
Lowered as written, every step computes a pointer and a mask per element, loads through
registers with a branch per vector, and moves both tiles to the MFMA layouts through LDS with
two barriers each and no overlap. `lift_pointer_gemm` proves that such a loop reads two
row-major blocks, zero outside a box, and replaces the loads with descriptor loads, which the
emitter's block GEMM loops take: bf16 1000 x 3000 x 2000 at 64x64x32 takes 30.6 us so, and 86 as
written. Row strides may be anything: 0, shorter than the row, negative. The caller undoes the
rewrite where it does not fit or does not pay (`build_module`).

The proof works on index tiles as polynomials: `sum_d coef_d * i_d + offset`, where i_d is the
tile coordinate along dimension d and the coefficients and the offset are integer polynomials in
the program's scalar values. A load qualifies when

- its pointers are one scalar base plus such a tile with unit stride along the row (A: along k,
  B: along n), and each step moves them by the block's extent along k: carried pointers
  incremented at the end of the body, or an offset linear in the loop variable;
- its mask is a conjunction of upper bounds `i_d + offset < bound`, the one along k shrinking by
  the block's extent per step, and its `other` is zero (no mask: everything is selected).

A tile whose origin is a program id times a constant, counted from one base for all of them,
becomes an offset into the whole operand; any other one gets a descriptor based at its own first
element, whose shape is the number of rows (A) or columns (B) the mask selects, so the rewritten
loop reads exactly the selected elements whatever the sign of the offsets. Kernels with arrays
past 2^31 elements (64-bit index math) are left alone, as descriptors cannot address them.
"""

from __future__ import annotations

from enceladus_amd.compiler import ir
from enceladus_amd.language import core

_DTYPES = (core.float16, core.bfloat16, core.float32)
_BODY_OPS = ir.PURE_OPS | {"load", "dot", "yield"}
_MAX_TERMS = 16


class _Poly:
    """An integer polynomial over scalar values: {sorted atom ids: coefficient}."""

    def __init__(self, terms=None):
        self.t = {k: c for k, c in (terms or {}).items() if c}

    @staticmethod
    def const(c: int) -> "_Poly":
        return _Poly({(): int(c)})

    def __add__(self, o):
        t = dict(self.t)
        for k, c in o.t.items():
            t[k] = t.get(k, 0) + c
        return _Poly(t)

    def __neg__(self):
        return _Poly({k: -c for k, c in self.t.items()})

    def __sub__(self, o):
        return self + (-o)

    def __mul__(self, o):
        t: dict = {}
        for a, x in self.t.items():
            for b, y in o.t.items():
                k = tuple(sorted(a + b))
                t[k] = t.get(k, 0) + x * y
        return _Poly(t)

    def __eq__(self, o):
        return self.t == o.t

    def value(self):
        """The constant this is, or None."""
        if not self.t:
            return 0
        return self.t[()] if set(self.t) == {()} else None

    def split(self, atom: int):
        """(coefficient of `atom`, the rest), or None when `atom` occurs otherwise than
        linearly."""
        lin, rest = {}, {}
        for k, c in self.t.items():
            n = k.count(atom)
            if n > 1:
                return None
            if n:
                i = k.index(atom)
                lin[k[:i] + k[i + 1:]] = c
            else:
                rest[k] = c
        return _Poly(lin), _Poly(rest)

    def atoms(self) -> set:
        return {a for k in self.t for a in k}


class _Affine:
    """`sum_d dims[d] * i_d + off` over a tile's coordinates."""

    def __init__(self, off, dims=None):
        self.off = off
        self.dims = {d: p for d, p in (dims or {}).items() if p.t}


class _Analysis:
    def __init__(self):
        self.atom: dict[int, ir.Value] = {}

    def scalar(self, v: ir.Value, depth=0) -> _Poly:
        op = v.op
        if op is not None and depth < 12 and v.type.dtype is core.int32:
            if op.name == "const":
                return _Poly.const(op.attrs["value"])
            if op.name == "binary" and op.attrs["op"] in ("add", "sub", "mul"):
                a, b = (self.scalar(o, depth + 1) for o in op.operands)
                k = op.attrs["op"]
                p = a + b if k == "add" else a - b if k == "sub" else a * b
                if len(p.t) <= _MAX_TERMS:
                    return p
        self.atom[v.id] = v
        return _Poly({(v.id,): 1})

    def tile(self, v: ir.Value, depth=0):
        """The `_Affine` of an int32 scalar or tile, or None."""
        t = v.type
        if depth > 32 or not isinstance(t, ir.TType) or t.ptr or t.dtype is not core.int32:
            return None
        if t.is_scalar:
            return _Affine(self.scalar(v))
        op = v.op
        if op is None:
            return None
        n = op.name
        if n == "const":
            return _Affine(_Poly.const(op.attrs["value"]))
        if n == "splat":
            return _Affine(self.scalar(op.operands[0]))
        if n == "arange":
            return _Affine(_Poly.const(op.attrs["start"]), {0: _Poly.const(1)})
        if n in ("expand_dims", "broadcast"):
            return self._view(op, self.tile(op.operands[0], depth + 1))
        if n == "binary" and op.attrs["op"] in ("add", "sub", "mul"):
            a, b = (self.tile(o, depth + 1) for o in op.operands)
            if a is None or b is None:
                return None
            k = op.attrs["op"]
            zero = _Poly()
            if k == "mul":
                if a.dims and b.dims:
                    return None
                if b.dims:
                    a, b = b, a
                return _Affine(a.off * b.off, {d: p * b.off for d, p in a.dims.items()})
            sign = (lambda p: p) if k == "add" else (lambda p: -p)
            return _Affine(a.off + sign(b.off),
                           {d: a.dims.get(d, zero) + sign(b.dims.get(d, zero))
                            for d in set(a.dims) | set(b.dims)})
        return None

    @staticmethod
    def _view(op, a):
        if a is None:
            return None
        src = op.operands[0].type.shape
        if op.name == "expand_dims":
            ax = op.attrs["axis"]
            return _Affine(a.off, {d + (d >= ax): p for d, p in a.dims.items()})
        return _Affine(a.off, {d: p for d, p in a.dims.items() if src[d] != 1})

    def pointer(self, v: ir.Value, depth=0):
        """(scalar base pointer, `_Affine`) of a pointer scalar or tile, or None."""
        if depth > 32 or not v.type.ptr:
            return None
        op = v.op
        if op is not None:
            if op.name == "ptr_add":
                p, o = self.pointer(op.operands[0], depth + 1), self.tile(op.operands[1])
                if p is None or o is None:
                    return None
                zero = _Poly()
                return p[0], _Affine(p[1].off + o.off,
                                     {d: p[1].dims.get(d, zero) + o.dims.get(d, zero)
                                      for d in set(p[1].dims) | set(o.dims)})
            if op.name == "splat":
                return self.pointer(op.operands[0], depth + 1)
            if op.name in ("expand_dims", "broadcast"):
                p = self.pointer(op.operands[0], depth + 1)
                a = self._view(op, p[1]) if p is not None else None
                return None if a is None else (p[0], a)
        return (v, _Affine(_Poly())) if v.type.is_scalar else None


def _and_terms(v: ir.Value, out: list):
    op = v.op
    if op is not None and op.name == "binary" and op.attrs["op"] == "and":
        for o in op.operands:
            _and_terms(o, out)
    elif op is not None and op.name == "broadcast" and \
            len(op.operands[0].type.shape) == len(v.type.shape):
        _and_terms(op.operands[0], out)
    else:
        out.append(v)


def _is_zero(v: ir.Value) -> bool:
    while v.op is not None and v.op.name in ("splat", "broadcast", "expand_dims"):
        v = v.op.operands[0]
    return v.op is not None and v.op.name == "const" and v.op.attrs["value"] == 0 and \
        str(float(v.op.attrs["value"])) == "0.0"


class _Loop:
    """One candidate loop, its analysis and its rewrite."""

    def __init__(self, fn: ir.Func, block: ir.Block, op: ir.Op, uses: dict):
        self.fn, self.block, self.op, self.uses = fn, block, op, uses
        self.body = op.regions[0]
        self.iv = self.body.args[0]
        self.an = _Analysis()
        self.inner = {self.iv.id, *(a.id for a in self.body.args)}
        for o in ir.walk(self.body):
            self.inner.update(r.id for r in o.results)

    @staticmethod
    def _const(v: ir.Value):
        return v.op.attrs["value"] if v.op is not None and v.op.name == "const" else None

    def invariant(self, p: _Poly) -> bool:
        return not (p.atoms() & self.inner)

    def match(self) -> bool:
        op, body = self.op, self.body
        lo, self.step = self._const(op.operands[0]), self._const(op.operands[2])
        if lo != 0 or not isinstance(self.step, int) or self.step <= 0 or \
                self.iv.type.dtype is not core.int32:
            return False
        if any(o.name not in _BODY_OPS or o.regions for o in body.ops):
            return False
        loads = [o for o in body.ops if o.name == "load"]
        dots = [o for o in body.ops if o.name == "dot"]
        if len(loads) != 2 or len(dots) != 1:
            return False
        dot = dots[0]
        la, lb = (x.op for x in dot.operands[:2])
        if la not in loads or lb not in loads or la is lb:
            return False
        if any(len(self.uses.get(x.result.id, [])) != 1 for x in loads):
            return False
        dt = la.result.type.dtype
        if dt not in _DTYPES or lb.result.type.dtype is not dt or \
                dot.result.type.dtype is not core.float32:
            return False
        (bm, bk), bn = la.result.type.shape, lb.result.type.shape[1]
        if bm < 32 or bn < 32 or bk % 16 or bk % self.step:
            return False
        self.bk = bk
        # the accumulator and (perhaps) the two carried pointer tiles, nothing else
        y = body.ops[-1].operands
        carried = body.args[1:]
        acc = dot.operands[2]
        if acc not in carried or y[carried.index(acc)] is not dot.result or \
                len(self.uses.get(acc.id, [])) != 1:
            return False
        self.plans = []
        ptrs = []
        for ld, kdim in ((la, 1), (lb, 0)):
            p = self.load_plan(ld, kdim, carried, y)
            if p is None:
                return False
            self.plans.append(p)
            if p["carried"] is not None:
                ptrs.append(p["carried"])
        if len(carried) != 1 + len(set(ptrs)) or len(set(ptrs)) != len(ptrs):
            return False
        # both operands end at the same k: the block loops take one
        ka, kb = ([lim - off + _Poly.const(extra) for lim, off, extra in p["bounds"][p["kdim"]]]
                  for p in self.plans)
        if len(ka) != len(kb) or any(x not in kb for x in ka) or any(x not in ka for x in kb):
            return False
        self.acc, self.dot = acc, dot
        # the loop variable may feed only what the rewrite removes: nothing but the dot and the
        # accumulator's yield stays
        return True

    def load_plan(self, ld, kdim: int, carried, y):
        ptr = ld.operands[0]
        shape = ld.result.type.shape
        index = None
        step = _Poly.const(self.step)
        if ptr in carried:
            index = carried.index(ptr)
            users = self.uses.get(ptr.id, [])
            inc = y[index].op
            if len(users) != 2 or inc is None or inc.name != "ptr_add" or \
                    inc.operands[0] is not ptr or set(users) != {ld, inc} or \
                    len(self.uses.get(inc.result.id, [])) != 1 or \
                    self.uses.get(self.op.results[index].id):
                return None
            adv = self.an.tile(inc.operands[1])
            got = self.an.pointer(self.op.operands[3 + index])
            if adv is None or adv.dims or got is None:
                return None
            base, aff = got
            off, per_step = aff.off, adv.off
        else:
            got = self.an.pointer(ptr)
            if got is None:
                return None
            base, aff = got
            cut = aff.off.split(self.iv.id)
            if cut is None:
                return None
            per_step, off = cut[0] * step, cut[1]
        if base.id in self.inner or set(aff.dims) - {0, 1}:
            return None
        one = _Poly.const(1)
        if aff.dims.get(1) != one or 0 not in aff.dims:
            return None
        stride = aff.dims[0]
        along = stride if kdim == 0 else one
        if not all(map(self.invariant, (off, stride, per_step))) or \
                per_step != along * _Poly.const(self.bk):
            return None
        bounds = {0: [], 1: []}
        if len(ld.operands) > 1:
            if not _is_zero(ld.operands[2]):
                return None
            terms: list = []
            _and_terms(ld.operands[1], terms)
            for t in terms:
                b = self.bound(t, len(shape), kdim)
                if b is None:
                    return None
                bounds[b[0]].append(b[1:])
        return {"load": ld, "kdim": kdim, "base": base, "off": off, "stride": stride,
                "bounds": bounds, "shape": shape,
                "carried": index, "dtype": ld.result.type.dtype}

    def bound(self, t: ir.Value, rank: int, kdim: int):
        """(dim, limit polynomial, offset polynomial, extra): the term selects coordinates
        i < limit - offset + extra along `dim` at the first step (and BK fewer per step along
        k); None when it has another form."""
        o = t.op
        if o is None or o.name != "binary" or o.attrs["op"] not in ("lt", "le", "gt", "ge") or \
                len(t.type.shape) != rank:
            return None
        x, lim = o.operands if o.attrs["op"] in ("lt", "le") else o.operands[::-1]
        ax, al = self.an.tile(x), self.an.tile(lim)
        if ax is None or al is None or al.dims or len(ax.dims) != 1:
            return None
        (d, coef), = ax.dims.items()
        if coef != _Poly.const(1):
            return None
        cx, cl = ax.off.split(self.iv.id), al.off.split(self.iv.id)
        if cx is None or cl is None:
            return None
        moves = cx[0] - cl[0]               # per unit of the loop variable
        if moves != _Poly.const(self.bk // self.step if d == kdim else 0):
            return None
        if not (self.invariant(cx[1]) and self.invariant(cl[1])):
            return None
        return d, cl[1], cx[1], int(o.attrs["op"] in ("le", "ge"))

    # -- rewriting ---------------------------------------------------------------------
    def emit(self, name, operands, types, attrs=None) -> ir.Value:
        o = ir.Op(name, operands, types, attrs or {}, loc=self.op.loc)
        self.new.append(o)
        return o.result

    def iconst(self, c: int, dt=core.int32) -> ir.Value:
        return self.emit("const", [], [ir.TType((), dt)], {"value": int(c)})

    def arith(self, k, a, b) -> ir.Value:
        return self.emit("binary", [a, b], [a.type], {"op": k})

    def poly(self, p: _Poly) -> ir.Value:
        """Scalar ops computing `p` in int32 (wrapping, as the source's arithmetic does)."""
        total = None
        for k, c in sorted(p.t.items()):
            v = None
            for a in k:
                x = self.an.atom[a]
                v = x if v is None else self.arith("mul", v, x)
            if v is None:
                v = self.iconst((c + (1 << 31)) % (1 << 32) - (1 << 31))
            elif c != 1:
                v = self.arith("mul", v, self.iconst((c + (1 << 31)) % (1 << 32) - (1 << 31)))
            total = v if total is None else self.arith("add", total, v)
        return total if total is not None else self.iconst(0)

    def from_pids(self, p: _Poly) -> bool:
        """Whether `p` is a sum of non-negative constants and of program ids (or their counts)
        with positive factors."""
        return all(c > 0 and all(self.an.atom[a].op is not None and self.an.atom[a].op.name in
                                 ("program_id", "num_programs") for a in k)
                   for k, c in p.t.items())

    def same_base(self, base: ir.Value, rest: _Poly, first: _Poly) -> bool:
        """Whether programs that differ only in the program ids of `first` address their tiles
        from one place: the base is an argument, and nothing in `rest`, the offset less the
        tile's origin, depends on those ids (nor on a value whose origin is not in sight).
        Operands stored tile by tile, or behind a pointer per tile, fail this: the rows
        and columns before such a tile are not the operand's."""
        pids = {self.an.atom[a].op.attrs.get("axis", 0) for a in first.atoms()
                if self.an.atom[a].op.name == "program_id"}
        todo, seen = [base, *(self.an.atom[a] for a in rest.atoms())], set()
        while todo:
            v = todo.pop()
            if v.id in seen or v in self.fn.args:
                continue
            seen.add(v.id)
            if v.op is None or v.op.regions or \
                    (v.op.name == "program_id" and v.op.attrs.get("axis", 0) in pids):
                return False
            todo.extend(v.op.operands)
        return True

    def extent(self, bounds, most: int) -> ir.Value:
        """min(most, limits), at least 0: how many leading coordinates are selected. Computed
        in 64 bits, where `limit - offset` cannot wrap."""
        i64 = ir.TType((), core.int64)
        total = self.iconst(most, core.int64)
        for lim, off, extra in bounds:
            a, b = (self.emit("cast", [self.poly(p)], [i64]) for p in (lim, off))
            e = self.arith("sub", a, b)
            if extra:
                e = self.arith("add", e, self.iconst(extra, core.int64))
            total = self.arith("min", total, e)
        total = self.arith("max", total, self.iconst(0, core.int64))
        return self.emit("cast", [total], [ir.TType((), core.int32)])

    def k_extent(self, bounds, hi: ir.Value) -> ir.Value:
        """The selected extent along k from the loop's start. Without a mask along k it is
        the whole blocks of the loop's trips."""
        if not bounds:
            bk = self.iconst(self.bk)
            if self.step == self.bk:
                up = self.arith("floordiv", self.arith("add", hi, self.iconst(self.bk - 1)), bk)
                return self.arith("mul", up, bk)
            f = self.bk // self.step
            if self.step == 1:
                return self.arith("mul", hi, bk)
            up = self.arith("floordiv", self.arith("add", hi, self.iconst(self.step - 1)),
                            self.iconst(self.step))
            return self.arith("mul", self.arith("mul", up, self.iconst(self.step)),
                              self.iconst(f))
        out = None
        for lim, off, extra in bounds:
            p = lim - off + _Poly.const(extra)
            v = self.poly(p)
            # the loop runs only while 0 < hi: a bound that is hi itself is positive in it
            if v is not hi:
                v = self.arith("max", v, self.iconst(0))
            out = v if out is None else self.arith("min", out, v)
        return out

    def rewrite(self) -> None:
        op, body = self.op, self.body
        self.new: list[ir.Op] = []
        hi = op.operands[1]
        zero = self.iconst(0)
        repl = {}
        for p in self.plans:
            base = p["base"]
            root = base
            while root.op is not None and root.op.name in ("ptr_add", "hint"):
                root = root.op.operands[0]
            kd, od = p["kdim"], 1 - p["kdim"]
            off, shape, offs = p["off"], [None, None], [zero, zero]
            shape[kd] = self.k_extent(p["bounds"][kd], hi)
            offs[kd] = self.iv
            first = p["bounds"][od][0][1] if p["bounds"][od] else None
            rest = None if first is None else \
                off - first * (p["stride"] if od == 0 else _Poly.const(1))
            if rest is not None and self.from_pids(first) and \
                    all(b[1] == first for b in p["bounds"][od]) and \
                    self.same_base(base, rest, first):
                # a tile at `first` = program id x tile size, never before the operand: the
                # whole operand is described and the tile's origin is an offset into it
                offs[od] = self.poly(first)
                off = rest
                shape[od] = self.k_extent([(lim, _Poly(), extra) for lim, _, extra in
                                           p["bounds"][od]], None)
            else:
                shape[od] = self.extent(p["bounds"][od], p["shape"][od])
            if off.value() != 0:
                base = self.emit("ptr_add", [base, self.poly(off)], [base.type])
            if root not in self.fn.args or root.facts.get("span2g"):
                base.facts["span2g"] = True       # (a base of unknown origin may span as much)
            strides = [self.poly(p["stride"]), self.iconst(1)]
            d = self.emit("make_desc", [base, *shape, *strides],
                          [ir.DescType(p["dtype"], tuple(p["shape"]))],
                          {"any_row_stride": True})
            ld = p["load"]
            new = ir.Op("desc_load", [d, *offs], [ld.result.type], loc=ld.loc)
            repl[id(ld)] = new
            self.dot.operands = [new.result if x is ld.result else x for x in self.dot.operands]
        f = self.bk // self.step
        if f != 1:
            # the loop variable becomes the position along k
            op.operands[1] = self.arith("mul", hi, self.iconst(f))
            op.operands[2] = self.iconst(self.bk)
        i = self.block.ops.index(op)
        self.block.ops[i:i] = self.new
        # only the loads, the dot and the accumulator's yield remain of the body
        keep = body.args.index(self.acc)
        body.ops = [*repl.values(), self.dot, body.ops[-1]]
        body.ops[-1].operands = [self.dot.result]
        body.args = [self.iv, self.acc]
        op.operands = [*op.operands[:3], op.operands[2 + keep]]
        op.attrs["lifted"] = True
        res = op.results[keep - 1]
        res.index = 0
        op.results = [res]


def _uses(fn: ir.Func) -> dict:
    out: dict[int, list] = {}
    for op in ir.walk(fn.body):
        for o in op.operands:
            out.setdefault(o.id, []).append(op)
    return out


def lift_pointer_gemm(fn: ir.Func) -> int:
    """Rewrites every loop that qualifies; returns how many."""
    if any(a.facts.get("idx64") for a in fn.args):
        return 0
    done = 0

    def visit(b: ir.Block):
        nonlocal done
        for op in list(b.ops):
            if op.name == "for":
                lp = _Loop(fn, b, op, _uses(fn))
                if lp.match():
                    lp.rewrite()
                    done += 1
                    continue
            for r in op.regions:
                visit(r)
    visit(fn.body)
    return done
