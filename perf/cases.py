"""Performance cases: the work a program has this backend do, through `Context.compile` (what `runN f`
does at partial application) and `Program.execute` (one application to device arrays).

A state is what such a program keeps between calls: the compiled program and its device arrays.
A pass is one `execute`; its results come back as tensors over the result's own device buffers.
The arrays of a case are drawn on the GPU from the seed alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from accelerate_amd import hip, ir as A, programs as P, workloads as W

Int = A.Int
TORCH = {"i32": torch.int32, "i64": torch.int64, "f32": torch.float32, "f64": torch.float64}
TYPESTR = {"i32": "<i4", "i64": "<i8", "f32": "<f4", "f64": "<f8"}
SIZE = {"i32": 4, "i64": 8, "f32": 4, "f64": 8}

SCANS = ("scanl1", "scanl", "scanl'", "scanr1", "scanr", "scanr'")
SPECTRAL_COEFF = (0.31938153, -0.356563782, 1.781477937, -1.821255978, 1.330274429)


# ---- the programs that accelerate_amd.programs does not hold -----------------------------------

def _binop(op, ty):
    return A.lam([ty, ty], lambda x, y: op(ty, x, y))


def _row_fold(op, ty):
    """fold of the innermost dimension: row sums, or row maxima (fold1 max)."""
    if op == "sum":
        return P.fold_sum(ty, 2)
    return P.fold1_op(A.max_, ty, 2)


def _scan(kind, ty):
    d = kind[4]
    if kind.endswith("1"):
        return P.scan1_sum(d, ty)
    return P.scan_prime_sum(d, ty) if kind.endswith("'") else P.scan_sum(d, ty)


def _smvm(ty):
    """Sparse matrix times vector: foldSeg (+) 0 (zipWith (*) vals (gather inds vec)) segd; product
    and gather are fused into the segmented fold, the offsets scan is let-bound."""
    sh1 = A.tshape(1)

    def body(segd, inds, vals, vec):
        src = A.delayed(
            A.tarray(1, ty), A.shape(vals),
            A.lam([sh1], lambda ix: A.mul(ty, A.index(vals, A.vexp(ix)), A.index(vec, A.sh(A.index(inds, A.vexp(ix)))))),
            A.lam([Int], lambda i: A.mul(ty, A.linearindex(vals, i), A.index(vec, A.sh(A.linearindex(inds, i))))))
        return A.alet(A.tarray(1, Int), A.scan("l", _binop(A.add, Int), A.constI(0), segd),
                      lambda offs: A.foldseg(Int, _binop(A.add, ty), A.const(ty, 0), src, offs))

    return A.alam([A.tarray(1, Int), A.tarray(1, Int), A.tarray(1, ty), A.tarray(1, ty)], body)


def _jacobi_loop(sweeps, ty):
    """awhile (\\(_, k) -> k < sweeps) (\\(g, k) -> (jacobi g, k + 1)) (g0, 0), then the grid."""
    grid, cnt = A.tarray(2, ty), A.tarray(0, Int)
    state = A.tpair(A.tpair(A.unit, grid), cnt)

    def cond(st):
        return A.unit_(A.u8, A.lt(Int, A.index(st[1], A.nil), A.constI(sweeps)))

    def body(st):
        (_, g), k = st
        return A.apair(A.apair(A.anil, A.apply(P.jacobi_step(ty), g)),
                       A.unit_(Int, A.add(Int, A.index(k, A.nil), A.constI(1))))

    return A.alam([grid], lambda g0: A.alet(
        state, A.awhile(state, cond, body, A.apair(A.apair(A.anil, g0), A.unit_(Int, A.constI(0)))),
        lambda st: st[0][1]))


def _smooth3(ty, boundary):
    """3x3x3 binomial smoothing of a volume, the weights 1 2 1 along each axis."""
    row = A.sunit(3, ty)
    sr = A.stup(*[A.stup(row, row, row)] * 3)

    def f(st):
        acc = None
        for z, plane in enumerate(A.untup(st)):
            for y, r in enumerate(A.untup(plane)):
                for x, t in enumerate(A.untup(r)):
                    w = (1 + (z == 1)) * (1 + (y == 1)) * (1 + (x == 1)) / 64.0
                    term = A.mul(ty, A.const(ty, w), t)
                    acc = term if acc is None else A.add(ty, acc, term)
        return acc

    return A.alam([A.tarray(3, ty)], lambda g: A.stencil(
        sr, ty, A.lam([A.stencil_type(sr)], f), {"clamp": A.clamp, "mirror": A.mirror, "wrap": A.wrap}[boundary], g))


def _radix_sort(bits):
    """Least-significant-digit radix sort of Int keys, a bit a pass: two exclusive scans give the
    places of the keys whose bit is 0 and 1, a permute moves them."""
    V1, S0, sh1 = A.tarray(1, Int), A.tarray(0, Int), A.tshape(1)

    def one_pass(keys, b, rest):
        def bit(k):
            return A.band(Int, A.shr(Int, k, A.constI(b)), A.constI(1))

        def scan_of(flag, k):
            flags = A.delayed(V1, A.shape(keys), A.lam([sh1], lambda ix: flag(A.index(keys, A.vexp(ix)))),
                              A.lam([Int], lambda i: flag(A.linearindex(keys, i))))
            return A.alet(A.tpair(V1, S0), A.scan_("l", _binop(A.add, Int), A.constI(0), flags), k)

        def with_both(zs, os_):
            (zpos, nz), (opos, _) = zs, os_

            def dest(ix):
                k = A.index(keys, A.vexp(ix))
                return A.just(A.sh(A.cond(A.eq(Int, bit(k), A.constI(0)), A.index(zpos, A.vexp(ix)),
                                          A.add(Int, A.index(nz, A.nil), A.index(opos, A.vexp(ix))))))
            return A.alet(V1, A.permute(
                A.lam([Int, A.wild(Int)], lambda x, _: x),
                A.generate(V1, A.shape(keys), A.lam([sh1], lambda ix: A.constI(0))),
                A.lam([sh1], dest), keys), rest)

        return scan_of(lambda k: A.sub(Int, A.constI(1), bit(k)),
                       lambda zs: scan_of(bit, lambda os_: with_both(zs, os_)))

    def build(keys, b):
        return keys if b == bits else one_pass(keys, b, lambda moved: build(moved, b + 1))

    return A.alam([V1], lambda keys: build(keys, 0))


def _blackscholes(ty):
    """map over (price, strike, years): the call and the put price of European options."""
    t3, t2 = A.ttup(ty, ty, ty), A.ttup(ty, ty)
    c = lambda x: A.const(ty, x)
    mul, add = (lambda a, b: A.mul(ty, a, b)), (lambda a, b: A.add(ty, a, b))
    sub, div = (lambda a, b: A.sub(ty, a, b)), (lambda a, b: A.fdiv(ty, a, b))

    def cnd(d, k):
        """cumulative normal distribution of d, bound for k"""
        def tail(t):
            acc = c(SPECTRAL_COEFF[-1])
            for a in SPECTRAL_COEFF[-2::-1]:
                acc = add(c(a), mul(t, acc))
            v = mul(mul(c(0.3989422804014327), A.exp(ty, mul(mul(c(-0.5), d), d))), mul(t, acc))
            return A.let(ty, v, lambda cv: A.let(ty, A.cond(A.gt(ty, d, c(0)), sub(c(1.0), cv), cv), k))
        return A.let(ty, div(c(1.0), add(c(1.0), mul(c(0.2316419), A.abs_(ty, d)))), tail)

    def go(v):
        price, strike, years = A.untup(v)
        r, vol = c(0.02), c(0.30)
        d1_of = lambda vs: div(add(A.log(ty, div(price, strike)), mul(add(r, mul(mul(c(0.5), vol), vol)), years)), vs)

        def prices(n1, n2, xe):
            return A.tup(sub(mul(price, n1), mul(xe, n2)),
                         sub(mul(xe, sub(c(1.0), n2)), mul(price, sub(c(1.0), n1))))

        return A.let(ty, mul(vol, A.sqrt(ty, years)), lambda vs: A.let(ty, d1_of(vs), lambda d1: A.let(
            ty, sub(d1, vs), lambda d2: cnd(d1, lambda n1: cnd(d2, lambda n2: A.let(
                ty, mul(strike, A.exp(ty, mul(A.neg(ty, r), years))), lambda xe: prices(n1, n2, xe)))))))

    return A.alam([A.tarray(1, t3)], lambda xs: A.map_(t2, A.lam([t3], go), xs))


# ---- the cases ---------------------------------------------------------------------------------

def listed():
    return [
        # The smallest call: a dot product of two short vectors, as in the inner loop of a host-side
        # algorithm.  One launch, one scalar back; what counts is the way from the call to the kernel.
        {"name": "dotp_f32_1k", "kind": "dotp", "type": "f32", "n": 1000},
        # fold (+) 0 (zipWith (*) xs ys) at the size of the benchmark's dotp.
        {"name": "dotp_f32_16m", "kind": "dotp", "type": "f32", "n": 1 << 24},
        # Reduction of the rows of a matrix: many results, rows of odd length.
        {"name": "row_sums_f64", "kind": "rows", "type": "f64", "op": "sum", "rows": 20011, "cols": 1003},
        # An ordinary prefix sum, of a length that is no multiple of anything.
        {"name": "scanl_f32_1m", "kind": "scan", "type": "f32", "scan": "scanl", "n": 1000003},
        # The benchmark's headline: the largest prefix sum.
        {"name": "scanl1_i64_256m", "kind": "scan", "type": "i64", "scan": "scanl1", "n": 1 << 28},
        # The benchmark's segmented sum: short segments with a tenth of long ones, offsets scan included.
        {"name": "foldseg_i32_128m", "kind": "foldseg", "type": "i32", "segments": 1 << 20, "n": 1 << 27},
        # Sparse matrix-vector product, 24 non-zeros a row on average, a banded matrix: a gather and a
        # product fused into a segmented fold.
        {"name": "smvm_f32_6m", "kind": "smvm", "type": "f32", "rows": 262147, "n": 6291457, "band": 2048},
        # The benchmark's histogram: popular bins, a destination of 256 KiB.
        {"name": "histogram_i32_64m", "kind": "histogram", "type": "i32", "n": 1 << 26, "bins": 1 << 16, "zipf": True},
        # The benchmark's stencil: 100 Jacobi sweeps, iterated by the program itself (awhile).
        {"name": "jacobi_f32_8192_x100", "kind": "jacobi", "type": "f32", "rows": 8192, "cols": 8192, "sweeps": 100},
        # A stencil of 27 points over a volume with odd extents: image and field smoothing.
        {"name": "smooth3_f32_393", "kind": "smooth3", "type": "f32", "depth": 401, "rows": 387, "cols": 393,
         "boundary": "clamp"},
        # A whole program of many small launches: scans and permutes in turn, 16-bit keys.
        {"name": "radix_sort_1m_16b", "kind": "radix", "n": 1 << 20, "bits": 16},
        # An elementwise program with arithmetic in it, over and into arrays of tuples.
        {"name": "blackscholes_f32_4m", "kind": "blackscholes", "type": "f32", "n": 4000037},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("dotp", "rows", "scan", "scan", "foldseg", "smvm", "histogram", "jacobi", "smooth3", "radix",
                       "blackscholes"))
    fl = rng.choice(("f32", "f64"))
    if kind == "dotp":
        return {"kind": kind, "type": fl, "n": _log(rng, 1 << 9, 1 << 26)}
    if kind == "rows":
        cols = _log(rng, 8, 1 << 16)
        return {"kind": kind, "type": rng.choice(("i64", "f32", "f64")), "op": rng.choice(("sum", "max")),
                "rows": _log(rng, 4, (1 << 26) // cols), "cols": cols}
    if kind == "scan":
        return {"kind": kind, "type": rng.choice(("i32", "i64", "f32", "f64")), "scan": rng.choice(SCANS),
                "n": _log(rng, 1 << 10, 1 << 27)}
    if kind == "foldseg":
        segs = _log(rng, 1 << 6, 1 << 20)
        return {"kind": kind, "type": rng.choice(("i32", "i64", "f32", "f64")), "segments": segs,
                "n": min(1 << 26, segs * _log(rng, 4, 1000))}
    if kind == "smvm":
        rows = _log(rng, 1 << 10, 1 << 20)
        return {"kind": kind, "type": fl, "rows": rows, "n": rows * rng.randint(4, 48) + rng.randint(0, 63),
                "band": rng.choice((64, 2048, 0))}
    if kind == "histogram":
        return {"kind": kind, "type": rng.choice(("i32", "i64")), "n": _log(rng, 1 << 12, 1 << 26),
                "bins": _log(rng, 1 << 8, 1 << 17), "zipf": rng.random() < 0.5}
    if kind == "jacobi":
        return {"kind": kind, "type": fl, "rows": _log(rng, 100, 6000), "cols": _log(rng, 100, 6000),
                "sweeps": rng.choice((1, 10, 33, 100))}
    if kind == "smooth3":
        return {"kind": kind, "type": fl, "depth": rng.randint(20, 400), "rows": rng.randint(20, 400),
                "cols": rng.randint(20, 400), "boundary": rng.choice(("clamp", "mirror", "wrap"))}
    if kind == "radix":
        return {"kind": kind, "n": _log(rng, 1 << 10, 1 << 22), "bits": rng.choice((8, 16))}
    return {"kind": kind, "type": fl, "n": _log(rng, 1 << 10, 1 << 25)}


# ---- inputs ------------------------------------------------------------------------------------

class _Buffer:
    """A leaf buffer of a device array as an array-interface object; keeps the array alive."""

    def __init__(self, array, leaf, shape, ty):
        self.array = array
        self.__cuda_array_interface__ = {
            "shape": shape, "typestr": TYPESTR[ty], "version": 2,
            "data": (hip.lib().acchip_array_buffer(array._h, leaf), False)}


def _view(array, types):
    """The tensors over a device array's leaves (one tensor where there is one leaf)."""
    shape = array.shape
    if 0 in shape:
        out = [torch.empty(shape, dtype=TORCH[t], device="cuda") for t in types]
    else:
        out = [torch.as_tensor(_Buffer(array, k, shape, t), device="cuda") for k, t in enumerate(types)]
    return out[0] if len(out) == 1 else out


class _Inputs:
    """Device arrays of the default context, filled from one seeded generator."""

    def __init__(self, seed):
        self.ctx = hip.default_context()
        self.gen = torch.Generator("cuda").manual_seed(seed)

    def array(self, shape, ty, *fill):
        """fill: one function per leaf from the leaf's tensor (to be written in place)."""
        d = self.ctx.empty(shape, A.tarray(len(shape), ty))
        leaves = A.tleaves(ty)
        views = _view(d, leaves)
        for v, f in zip(views if len(leaves) > 1 else [views], fill):
            f(v)
        return d

    def ints(self, lo, hi):
        return lambda v: v.random_(lo, hi + 1, generator=self.gen)

    def reals(self, lo, hi):
        return lambda v: v.uniform_(lo, hi, generator=self.gen)

    def numbers(self, ty, lo=0.0, hi=1.0):
        return self.reals(lo, hi) if ty[0] == "f" else self.ints(-1000, 1000)

    def copy(self, t):
        return lambda v: v.copy_(t)


def _programs(case):
    k = case["kind"]
    if k == "dotp":
        return P.dotp(case["type"])
    if k == "rows":
        return _row_fold(case["op"], case["type"])
    if k == "scan":
        return _scan(case["scan"], case["type"])
    if k == "foldseg":
        return P.foldseg_sum(case["type"])
    if k == "smvm":
        return _smvm(case["type"])
    if k == "histogram":
        return P.histogram(case["bins"], A.i32, case["type"])
    if k == "jacobi":
        return _jacobi_loop(case["sweeps"], case["type"])
    if k == "smooth3":
        return _smooth3(case["type"], case["boundary"])
    if k == "radix":
        return _radix_sort(case["bits"])
    return _blackscholes(case["type"])


class State:
    def __init__(self, case, program, args):
        k, ty = case["kind"], case.get("type", "i64")
        self.program, self.args = program, args
        self.types = [ty, ty] if k == "blackscholes" else [ty]
        self.pair = k == "scan" and case["scan"].endswith("'")


def prepare(case, seed):
    k, ty, n = case["kind"], case.get("type"), case.get("n")
    x = _Inputs(seed)
    if k == "dotp":
        args = [x.array((n,), ty, x.reals(0, 1)), x.array((n,), ty, x.reals(0, 1))]
    elif k == "rows":
        args = [x.array((case["rows"], case["cols"]), ty, x.numbers(ty))]
    elif k == "scan":
        args = [x.array((n,), ty, x.numbers(ty))]
    elif k == "foldseg":
        lens = torch.from_numpy(W.segment_lengths(case["segments"], n, seed)).cuda()
        args = [x.array((n,), ty, x.numbers(ty)), x.array((case["segments"],), "i32", x.copy(lens))]
    elif k == "smvm":
        rows, band = case["rows"], case["band"]
        lens = torch.from_numpy(_row_lengths(rows, n, seed)).cuda()
        # columns within `band` of the diagonal, or anywhere (0)
        cols = torch.randint(0, band or rows, (n,), generator=x.gen, device="cuda")
        if band:
            cols += torch.repeat_interleave(torch.arange(rows, device="cuda"), lens, output_size=n) - band // 2
            cols.clamp_(0, rows - 1)
        args = [x.array((rows,), "i64", x.copy(lens)), x.array((n,), "i64", x.copy(cols)),
                x.array((n,), ty, x.reals(-1, 1)), x.array((rows,), ty, x.reals(-1, 1))]
    elif k == "histogram":
        args = [x.array((n,), "i32", _keys(x, n, case["bins"], case["zipf"]))]
    elif k == "jacobi":
        args = [x.array((case["rows"], case["cols"]), ty, x.reals(0, 1))]
    elif k == "smooth3":
        args = [x.array((case["depth"], case["rows"], case["cols"]), ty, x.reals(0, 1))]
    elif k == "radix":
        args = [x.array((n,), "i64", x.ints(0, (1 << case["bits"]) - 1))]
    else:
        args = [x.array((n,), A.ttup(ty, ty, ty), x.reals(5, 30), x.reals(1, 100), x.reals(0.25, 10))]
    program = x.ctx.compile(_programs(case))
    torch.cuda.synchronize()   # the library's stream does not wait for torch's
    return State(case, program, args)


def _row_lengths(rows, n, seed):
    """Non-zeros per row: uniform in [0, 2 n / rows], corrected to sum to n."""
    rng = np.random.default_rng(seed)
    lens = rng.integers(0, 2 * (n // rows) + 1, rows)
    off = n - int(lens.sum())
    while off:
        at = rng.integers(0, rows, min(abs(off), rows))
        step = 1 if off > 0 else -1
        at = np.unique(at if off > 0 else at[lens[at] > 0])
        lens[at] += step
        off -= step * len(at)
    return lens


def _keys(x, n, bins, zipf):
    if not zipf:
        return x.ints(0, bins - 1)
    # Zipf(1.1) over the bins by inverse CDF: rank r is bin r
    w = torch.arange(1, bins + 1, dtype=torch.float64, device="cuda") ** -1.1
    cdf = torch.cumsum(w, 0) / w.sum()

    def fill(v):
        u = torch.rand(v.shape, dtype=torch.float64, device="cuda", generator=x.gen)
        v.copy_(torch.searchsorted(cdf, u, right=True).clamp_(max=bins - 1))
    return fill


def run(state):
    r = state.program.execute(*state.args)
    if state.pair:
        values, total = r.parts()
        return _view(values, state.types), _view(total, state.types)
    return _view(r, state.types)


# ---- what a pass cannot do without, and how far results may be apart -----------------------------

def work(case):
    """Every input read once, every result written once; the operations of the program's text."""
    k, n = case["kind"], case.get("n", 0)
    s = SIZE[case.get("type", "i64")]
    if k == "dotp":
        return {"bytes": 2 * s * n + s, "flops": 2 * n}
    if k == "rows":
        return {"bytes": s * case["rows"] * (case["cols"] + 1), "flops": case["rows"] * case["cols"]}
    if k == "scan":
        return {"bytes": 2 * s * n, "flops": n}
    if k == "foldseg":
        return {"bytes": s * n + (4 + s) * case["segments"], "flops": n}
    if k == "smvm":
        return {"bytes": (8 + s) * n + (8 + 2 * s) * case["rows"], "flops": 2 * n}
    if k == "histogram":
        return {"bytes": 4 * n + s * case["bins"], "flops": n}
    if k == "jacobi":
        cells = case["rows"] * case["cols"]
        return {"bytes": 2 * s * cells, "flops": 4 * cells * case["sweeps"]}
    if k == "smooth3":
        cells = case["depth"] * case["rows"] * case["cols"]
        return {"bytes": 2 * s * cells, "flops": 53 * cells}
    if k == "radix":
        return {"bytes": 16 * n, "flops": 4 * n * case["bits"]}
    return {"bytes": 5 * s * n, "flops": 60 * n}


def tolerance(case):
    """Whole numbers and stencils (whose function fixes the order of its sums) are exact.  Sums of
    floating-point numbers differ by their order, elementary functions by their last places: about
    four times the largest difference seen from the same program in 64 bits (Float32 prefix sums of
    2^27 numbers 3.3e-7 / 8e-7, option prices 1.6e-7 / 1.8e-6; Float64 against another order of the
    sums 4.5e-15 / 1.6e-14)."""
    k, ty = case["kind"], case.get("type", "i64")
    if ty[0] == "i" or k in ("jacobi", "smooth3") or (k == "rows" and case["op"] == "max"):
        return "exact"
    return {"rel": 1.5e-6, "max": 7e-6} if ty == "f32" else {"rel": 2e-14, "max": 6e-14}


# ---- the same in 64 bits ------------------------------------------------------------------------

def _wide(t):
    """A vector on the host for sums of it: the whole numbers in 64 bits; the others in extended
    precision, so that these sums' own rounding does not count."""
    v = t.cpu().numpy()
    return v.astype(np.int64 if v.dtype.kind == "i" else np.longdouble)


def _narrow(v, like):
    v = np.ascontiguousarray(v)
    return torch.from_numpy(v.astype(np.float64 if v.dtype.kind == "f" else like))


def _segment_sums(v, lens):
    lens = lens.cpu().numpy().astype(np.int64)
    starts = np.cumsum(lens) - lens
    out = np.zeros(len(lens), v.dtype)
    some = lens > 0
    if some.any():
        out[some] = np.add.reduceat(v, starts[some])
    return out


def exact(case, seed):
    """What `run` returns for the inputs of `prepare(case, seed)`, from torch and numpy alone: whole
    numbers as they are, the others in 64 bits."""
    k, ty = case["kind"], case.get("type", "i64")
    args = prepare(case, seed).args
    types = [ty] * 3 if k == "blackscholes" else None
    xs = [_view(a, types or [ty]) for a in args] if k in ("dotp", "rows", "scan", "jacobi", "smooth3", "radix",
                                                          "blackscholes") else None
    whole = np.int32 if ty == "i32" else np.int64
    if k == "dotp":
        return _narrow(np.sum(_wide(xs[0]) * _wide(xs[1])), whole)
    if k == "rows":
        x = xs[0]
        if case["op"] == "max":
            return x.amax(1)
        return x.sum(1) if ty == "i64" else _narrow(_wide(x).sum(1), whole)
    if k == "scan":
        kind, x = case["scan"], xs[0]
        right = kind[4] == "r"
        if ty[0] == "i":
            s = torch.cumsum(x.flip(0) if right else x, 0, dtype=TORCH[ty])
        else:
            v = _wide(x)
            s = _narrow(np.cumsum(v[::-1] if right else v), whole)
        turn = (lambda t: t.flip(0)) if right else (lambda t: t)
        if kind.endswith("1"):
            return turn(s)
        from0 = torch.cat([torch.zeros(1, dtype=s.dtype, device=s.device), s])
        return (turn(from0[:-1]), from0[-1]) if kind.endswith("'") else turn(from0)
    if k == "foldseg":
        return _narrow(_segment_sums(_wide(_view(args[0], [ty])), _view(args[1], ["i32"])), whole)
    if k == "smvm":
        lens, cols = _view(args[0], ["i64"]), _view(args[1], ["i64"]).cpu().numpy()
        vals, vec = (_wide(_view(a, [ty])) for a in args[2:])
        return _narrow(_segment_sums(vals * vec[cols], lens), whole)
    if k == "histogram":
        return torch.bincount(_view(args[0], ["i32"]), minlength=case["bins"]).to(TORCH[ty])
    if k == "jacobi":
        g = xs[0].double()
        for _ in range(case["sweeps"]):
            p = torch.nn.functional.pad(g[None, None], (1, 1, 1, 1), mode="replicate")[0, 0]
            g = 0.25 * (p[:-2, 1:-1] + p[1:-1, :-2] + p[1:-1, 2:] + p[2:, 1:-1])
        return g
    if k == "smooth3":
        g = xs[0].double()
        mode = {"clamp": "replicate", "mirror": "reflect", "wrap": "circular"}[case["boundary"]]
        p = torch.nn.functional.pad(g[None, None], (1,) * 6, mode=mode)[0, 0]
        for d in range(3):   # 1 2 1 along each axis
            n = p.shape[d] - 2
            p = (p.narrow(d, 0, n) + 2 * p.narrow(d, 1, n) + p.narrow(d, 2, n)) / 4
        return p
    if k == "radix":
        return torch.sort(xs[0]).values
    price, strike, years = (x.double() for x in xs[0])
    a1, a2, a3, a4, a5 = SPECTRAL_COEFF

    def cnd(d):
        t = 1 / (1 + 0.2316419 * d.abs())
        v = 0.3989422804014327 * torch.exp(-0.5 * d * d) * (t * (a1 + t * (a2 + t * (a3 + t * (a4 + t * a5)))))
        return torch.where(d > 0, 1 - v, v)

    vs = 0.30 * torch.sqrt(years)
    d1 = (torch.log(price / strike) + (0.02 + 0.5 * 0.30 * 0.30) * years) / vs
    n1, n2, xe = cnd(d1), cnd(d1 - vs), strike * torch.exp(-0.02 * years)
    return [price * n1 - xe * n2, xe * (1 - n2) - price * (1 - n1)]
